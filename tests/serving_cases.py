"""The serving layer: the scheduler driving a gptfast (Aria) decoder, Duguzen and Kozipel alike, the command line, the trace runner.  Shared by
tests/test_emu_serving.py (CPU) and tests/test_gpu_serving.py (hardware)."""
import io
import json
import os

import pytest
import torch

from tests import kozipel_cases as K
from tests import latent_cases as L

bf16, f32 = torch.bfloat16, torch.float32


def gptfast_toy(dev, head_dim=64):
    from aria_amd import gptfast as G

    args = G.ModelArgs(block_size=64, vocab_size=136, n_layer=2, n_head=2, dim=2 * head_dim, intermediate_size=40, n_local_heads=2, rope_base=10000.0,
                       norm_eps=1e-5, num_experts=8, router_topk=3, num_shared_experts=2)
    m, g = G.Transformer(args), L.gen(5)
    with torch.no_grad():
        for n, p in m.named_parameters():
            p.copy_((1 + 0.1 * torch.randn(p.shape, generator=g)).to(bf16) if "norm" in n else (torch.randn(p.shape, generator=g) * 0.08).to(bf16))
    return m.to(dev).eval()


def case_gptfast_batch(dev, engine=True):
    """At sizes that no one-call step serves, unequal requests of one batch give each request's own logits bit for bit (its sequence runs by itself on its slot),
    with the decode engine and with the tile path; the tile path also equals one prefill of the whole prefix.  Slots are used again by a second
    batch."""
    from aria_amd.serving import Scheduler

    m = gptfast_toy(dev)
    m.use_decode_engine = engine
    toks = [torch.randint(0, 136, (n,), generator=L.gen(n)).tolist() for n in (7, 3, 5)]

    def alone(t):
        s = Scheduler(m, 16)
        return torch.cat([s.step(["x"], [t[:-2]], [[0, len(t) - 3]])] + [s.step(["x"], [[i]]) for i in t[-2:]]).cpu()

    want = [alone(t) for t in toks]
    if not engine:
        for t, x in zip(toks, want):
            m.setup_caches(1, 16)
            with torch.no_grad():
                whole = m(torch.tensor([t], device=dev))[0].float().cpu()
            assert L.rel(x, whole[[0, len(t) - 3, len(t) - 2, len(t) - 1]]) < 2e-2
    sched = Scheduler(m, 16)
    for _ in range(2):
        got = sched.step(["a", "b", "c"], [t[:-2] for t in toks], [[0, len(t) - 3] for t in toks]).cpu()
        assert torch.equal(got, torch.cat([x[:2] for x in want]))
        for back in (2, 1):
            got = sched.step(["c", "a", "b"], [[toks[i][-back]] for i in (2, 0, 1)]).cpu()
            assert torch.equal(got, torch.stack([want[i][4 - back] for i in (2, 0, 1)]))
        for r in "bca":
            sched.finish(r)


def gptfast_routed(dev, dim, head_dim, inter, block, vocab=264, top=3):
    """Embeddings carry the directions of their experts, so that no choice is a close call."""
    from aria_amd import gptfast as G

    E, k, V = 16, top, vocab
    args = G.ModelArgs(block_size=block, vocab_size=V, n_layer=2, n_head=dim // head_dim, dim=dim, intermediate_size=inter, rope_base=10000.0, norm_eps=1e-5,
                       num_experts=E, router_topk=k, num_shared_experts=2)
    m, g = G.Transformer(args), L.gen(5)
    unit = torch.nn.functional.normalize(torch.randn(E, dim, generator=g), dim=-1)
    chosen = torch.zeros(V, E).scatter_(1, torch.rand(V, E, generator=g).topk(k, -1).indices, 1.0)
    with torch.no_grad():
        for n, p in m.named_parameters():
            p.copy_((1 + 0.1 * torch.randn(p.shape, generator=g)).to(bf16) if "norm" in n else (torch.randn(p.shape, generator=g) * p.shape[-1] ** -0.5).to(bf16))
        m.tok_embeddings.weight.copy_((torch.randn(V, dim, generator=g) + 8.0 * chosen @ unit).to(bf16))
        for b in m.layers:
            b.feed_forward.gate.weight.copy_(unit[torch.randperm(E, generator=g)].to(bf16))
    return m.to(dev).eval()


def case_gptfast_decode_batch(dev, dim, head_dim, inter, requests, longest=9):
    """Steps of several requests in one call (every weight read once) against each request alone, one token at a time: requests of unequal lengths on any
    slots, experts that one, several and all of them chose.  Embeddings carry the directions of their experts, so that no choice is a close call.  Both
    sides round the same tensors to bf16; a logit differs by the order of fp32 sums and by roundings that then fall the other way, about 2^-9 a layer's
    residual step, four of them."""
    from aria_amd.serving import Scheduler

    m = gptfast_routed(dev, dim, head_dim, inter, longest + 16)
    toks = [torch.randint(0, 264, (max(3, longest - 5 * i),), generator=L.gen(i)).tolist() for i in range(requests)]

    def alone(t):
        s = Scheduler(m, longest + 1)
        s.step(["x"], [t[:-2]], [[]])
        return torch.cat([s.step(["x"], [[i]]) for i in t[-2:]]).cpu().double()

    want = [alone(t) for t in toks]
    sched = Scheduler(m, longest + 1)
    for i, t in enumerate(toks):      # (prompts as in the single runs: the caches then hold the same rows)
        if i == 0:
            m.setup_caches(requests, longest + 1)
            sched.slots, sched.free = requests, list(range(requests))[::-1]
        sched.step([i], [t[:-2]], [[]])
    for step in range(2):
        order = list(range(requests))[::-1] if step else list(range(requests))
        got = sched.step(order, [[toks[i][len(toks[i]) - 2 + step]] for i in order])
        assert L.logit_err(got, torch.stack([want[i][step] for i in order])) < 4 * 2 ** -8


def gptfast_moved_weights(dev, names):
    """(name, model, what changes its weights, a model that has had them from the beginning), each change by another way in"""
    from torch import nn

    def copies():
        return gptfast_routed(dev, 128, 64, 128, 32), gptfast_routed(dev, 128, 64, 128, 32)

    def assign(m):
        m.load_state_dict({k: v.clone() for k, v in m.state_dict().items()}, assign=True)

    def parameter(m):
        m.output.weight = nn.Parameter(m.output.weight.detach() * 2, requires_grad=False)

    def data(m):
        m.layers[1].attention.wo.weight.data = m.layers[1].attention.wo.weight.data.T.contiguous()

    def module(m):
        other = gptfast_routed(dev, 128, 64, 128, 32).layers[0].feed_forward
        with torch.no_grad():
            other.shared_ffn.w2.weight.mul_(-1)
        m.layers[0].feed_forward = other

    for change in (c for c in (assign, parameter, data, module) if c.__name__ in names):
        m, want = copies()
        change(want)
        yield change.__name__, m, change, want


def case_gptfast_moved_weights(dev, names=("assign", "parameter", "data", "module")):
    """Weights that are assigned, exchanged or re-homed between steps (by the caller, and by the packed prompts' own pairing of gate and up): every later step
    runs on the new ones, to the bit as a model that was made with them."""
    from aria_amd.serving import Scheduler

    prompts = [torch.randint(0, 264, (n,), generator=L.gen(n)).tolist() for n in (5, 3)]

    def session(s):
        out = [s.step(["a", "b"], prompts), s.step(["a", "b"], [[7], [8]])]
        s.finish("a"), s.finish("b")
        return torch.cat(out).cpu()

    for name, m, change, other in gptfast_moved_weights(dev, names):
        want = session(Scheduler(other, 16))
        sched = Scheduler(m, 16)
        for first in (False, True):
            if first:
                session(sched)                                # (tables exist when the weights change)
            else:
                m.setup_caches(2, 16)
                sched.slots, sched.free = 2, [0, 1]
            if first or name == "assign":
                change(m)
                assert torch.equal(session(sched), want), name
    m.layers[1].attention.wo.weight.data = m.layers[1].attention.wo.weight.data.T      # (refused by every path)
    with pytest.raises(ValueError):
        sched.step(["a", "b"], prompts)


def case_gptfast_weights_given_up(dev):
    """A step's tables keep no weights alive that a load has replaced."""
    import weakref

    from aria_amd.serving import Scheduler

    m = gptfast_routed(dev, 128, 64, 128, 32)
    Scheduler(m, 8).step("ab", [[5], [9]])
    kept = [weakref.ref(t) for t in m._tables.tensors]
    m.load_state_dict({k: v.clone() for k, v in m.state_dict().items()}, assign=True)
    assert kept and not any(r() is not None for r in kept)


def toy(design, dev):
    """A small decoder whose steps of several requests are one call."""
    if design == "gptfast":
        return gptfast_routed(dev, 128, 64, 128, 32)
    cases, name = DESIGNS[design]
    cfg = cases.CONFIGS[name]
    return cases.build(cfg, cases.checkpoint(cfg, seed=3), dev, bf16)


def case_wanted_rows(dev, design):
    """Wanted places named twice, none of a request's, all but not in order: the rows of the step that asks for each once."""
    from aria_amd.serving import Scheduler

    m, prompts = toy(design, dev), [[5, 3, 7], [4, 9]]

    def session(prompt_places, places):
        s = Scheduler(m, 8)
        out = [s.step("ab", prompts, prompt_places), s.step("ab", [[11], [12]], places)]
        s.finish("a"), s.finish("b")
        return [t.cpu() for t in out]

    one, two = session([[0, 1, 2], [0, 1]], [[0], [0]])
    got = session([[2, 0, 0, 1], [0]], [[0, 0], []])
    assert torch.equal(got[0], one[[2, 0, 0, 1, 3]]) and torch.equal(got[1], two[[0, 0]])
    got = session([[], [1, 0]], [[], [0, 0]])
    assert torch.equal(got[0], one[[4, 3]]) and torch.equal(got[1], two[[1, 1]])


def case_gptfast_ids(dev, dim=128, inter=128):
    """Steps take the ids of any integer type and stride on the device, and refuse on the CPU, where that can be looked at, the same ids as a model's embedding:
    outside the vocabulary, in prompts of one call, packed prompts and decoded tokens."""
    from aria_amd.serving import Scheduler

    m = gptfast_routed(dev, dim, 64, inter, 32)

    def session(second, prompts=([5, 3, 7], [4, 9])):
        s = Scheduler(m, 8)
        out = [s.step("ab", list(prompts)), s.step("ab", second)]
        s.finish("a"), s.finish("b")
        return torch.cat(out).cpu()

    want = session([[11], [12]])
    ids = torch.tensor([11, 12], device=dev)
    strided = torch.stack([ids, ids + 1], 1)[:, 0]
    for second in (ids, ids.int(), ids.short(), strided, strided.int(), ids.view(2, 1)):
        assert torch.equal(session(second), want), (second.dtype, second.shape, second.stride())
    if str(dev) == "cpu":
        for bad in ([[264], [12]], [[11], [-1]], ids + 256):
            with pytest.raises(IndexError):
                session(bad)
        with pytest.raises(IndexError):
            session([[11], [12]], ([5, 264, 7], [4, 9]))


def case_gptfast_slot_twice(dev, dim=128, inter=128):
    """A batch that names a slot twice runs its parts in order, the second one on the rows of the first; slots and positions before the first are refused."""
    from aria_amd.serving import StepBatch

    m = gptfast_routed(dev, dim, 64, inter, 32)
    m.setup_caches(2, 8)

    def step(tokens, slots, starts):
        return m.step(StepBatch.build(tokens, slots, starts, None, dev)).cpu()

    step([[5, 3], [9, 9]], [0, 1], [0, 0])
    want = [step([[t]], [0], [2 + i]) for i, t in enumerate((7, 4))]
    for c in m.layers[0].attention.kv_cache.k, m.layers[1].attention.kv_cache.v:
        c[0, 2:].fill_(float("nan"))
    assert torch.equal(step([[7], [4]], [0, 0], [2, 3]), torch.cat(want))
    for slots, starts in (([0, -1], [2, 2]), ([0, 1], [2, -1]), ([0, 2], [2, 2]), ([0, 1], [2, 8])):
        with pytest.raises(ValueError):
            step([[7], [4]], slots, starts)


def case_gptfast_hooks(dev, dim=128, inter=128):
    """Hooks on the modules see every prompt by itself, as do replaced forwards and layers of other classes; logits as without them."""
    from aria_amd import gptfast as G
    from aria_amd.serving import Scheduler

    m, prompts = gptfast_routed(dev, dim, 64, inter, 32), [[5, 3, 7], [4, 9]]

    def prompt():
        s = Scheduler(m, 8)
        out = s.step("ab", prompts).cpu().double()
        s.finish("a"), s.finish("b")
        return out

    want, seen = prompt(), []
    block = m.layers[1]
    for part in (block, block.attention, block.feed_forward):
        for register in (part.register_forward_hook, part.register_forward_pre_hook):
            hook = register(lambda m, a, *out: seen.append(a[0].shape[0]))
            assert L.logit_err(prompt(), want) < 4 * 2 ** -8 and seen == [3, 2]
            hook.remove()
            seen.clear()
    plain = block.feed_forward.forward
    block.feed_forward.forward = lambda x: seen.append(x.shape[0]) or plain(x)
    assert L.logit_err(prompt(), want) < 4 * 2 ** -8 and seen == [3, 2]
    del block.feed_forward.forward

    class Other(G.MOEFeedForward):
        def forward(self, x):
            seen.append(-x.shape[0])
            return super().forward(x)

    block.feed_forward.__class__ = Other
    for again in (1, 2):      # (on tables that were made before, and on new ones)
        assert L.logit_err(prompt(), want) < 4 * 2 ** -8 and seen == [3, 2] + [-3, -2] * again
        m._tables = None


def case_build(dev):
    """Ids as lists, ranges, arrays, tensors on any device and tensors of one element make the same tables; what 32 bits do not hold is refused; no sequences
    make an empty batch, which Aria answers with no rows."""
    import numpy as np

    from aria_amd.serving import StepBatch

    def tables(tokens, slots=(1, 0), starts=(3, 0), wanted=(2, 0)):
        b = StepBatch.build(tokens, slots, starts, wanted, dev)
        return [t.tolist() for t in (b.ids, b.slot, b.pos, b.cu, b.wanted, b.seq)]

    want = [[5, 6, 9], [1, 1, 0], [3, 4, 0], [0, 2, 3], [2, 0], [0, 0, 1]]
    t = torch.tensor([5, 6, 9], device=dev)
    for tokens in ([[5, 6], [9]], [range(5, 7), (9,)], [np.array([5, 6]), np.array([9], dtype=np.uint8)], [t[:2], t[2:]], [[t[0], t[1]], [t[2]]], [t[:2].view(2, 1), [9]]):
        assert tables(tokens) == want
    assert tables([[5], [9]], wanted=t[:0]) == tables([t[:1], [t[2]]], wanted=()) and tables([[5], [9]], torch.tensor([1, 0]), np.array([3, 0])) == tables([[5], [9]])
    for tokens, slots, starts in (([[2 ** 31]], [0], [0]), ([np.array([2 ** 40])], [0], [0]), ([torch.tensor([2 ** 40])], [0], [0]), ([[1]], [2 ** 32], [0]), ([[1]], [0], [2 ** 31])):
        with pytest.raises((RuntimeError, OverflowError)):
            tables(tokens, slots, starts, [0])
    empty = StepBatch.build([], [], [], None, dev)
    assert empty.ids.numel() == 0 and empty.cu.tolist() == [0]
    m = gptfast_routed(dev, 128, 64, 128, 32)
    m.setup_caches(1, 8)
    assert m.step(empty).shape == (0, 264)


def case_decode_splits(dev, monkeypatch, run=True):
    """ARIA_DECODE_SPLIT_KV decides over the splits of serving steps as over the decode engine's (seen in the scratch that they ask for); the logits stay those of
    the step's own choice (another order of sums: ``case_gptfast_decode_batch``)."""
    import ctypes

    import numpy as np

    from aria_amd import hip
    from aria_amd.serving import StepBatch

    def scratch(T, slots):
        dims = np.array([2, 2560, 20, 128, 64, 6, 1664, 3328, 1000, slots], dtype=np.int64)
        return int(hip.get_lib().cdll.aria_decode_step_scratch(dims.ctypes.data_as(ctypes.c_void_p), T, slots - 8))

    one = 4 * 8 * 20 * 130       # floats of one split: 8 tokens, 20 heads
    monkeypatch.setenv("ARIA_DECODE_SPLIT_KV", "0")
    none = scratch(8, 4096)
    for value, slots, splits in (("1", 4096, 4), ("7", 4096, 7), ("99", 4096, 32), ("7", 2048, 1)):
        monkeypatch.setenv("ARIA_DECODE_SPLIT_KV", value)
        assert scratch(8, slots) - none == (splits - 1) * one, value
    if not run:
        return
    m = gptfast_routed(dev, 128, 64, 128, 2600)
    m.setup_caches(3, 2600)
    for b in m.layers:
        for c in (b.attention.kv_cache.k, b.attention.kv_cache.v):
            c.copy_(torch.randn(c.shape, generator=L.gen(1)))

    def step(n):
        return m.step(StepBatch.build([[5], [9], [77]][:n], list(range(n)), [2590, 3, 1500][:n], None, dev))

    monkeypatch.delenv("ARIA_DECODE_SPLIT_KV")
    want = [step(n).cpu().double() for n in (1, 3)]
    for value in "0", "1", "5":
        monkeypatch.setenv("ARIA_DECODE_SPLIT_KV", value)
        for n, w in zip((1, 3), want):
            assert L.logit_err(step(n), w) < 4 * 2 ** -8, value


def case_decode_keys_once(dev, monkeypatch, head_dim):
    """Keys and values read non-temporally (told of more keys than the Infinity Cache holds) and plainly: the same splits, the same bits."""
    from aria_amd.serving import StepBatch

    m = gptfast_routed(dev, 2560, head_dim, 64, 4104)
    m.setup_caches(3, 4104)
    for b in m.layers:
        for c in (b.attention.kv_cache.k, b.attention.kv_cache.v):
            c.copy_(torch.randn(c.shape, generator=L.gen(1)))
    monkeypatch.setenv("ARIA_DECODE_SPLIT_KV", "5")
    for n in (1, 3):
        got = []
        for most in (1300, 4100):
            assert (n * most * 2560 * 4 >= 40 << 20) == (most == 4100)
            monkeypatch.setattr(StepBatch, "max_len", property(lambda self, most=most: most))
            got.append(m.step(StepBatch.build([[5], [9], [77]][:n], list(range(n)), [1290, 3, 700][:n], None, dev)).clone())
        assert torch.equal(*got)


def case_alignment(dev):
    """Tensors that do not start at 16 bytes are refused in front of every launch, as the tile products refuse them."""
    from aria_amd import gptfast as G
    from aria_amd import hip, ops
    from aria_amd.serving import Scheduler

    def off(t):
        return torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)

    T, H, hd, S = 3, 2, 64, 8
    slot, pos = torch.zeros(T, dtype=torch.int32, device=dev), torch.arange(T, dtype=torch.int32, device=dev)
    tensors = [L.rnd(T, 3 * H * hd, seed=1).to(dev), G.precompute_freqs_cis(S, hd).to(dev), L.rnd(1, S, H * hd, seed=2).to(dev), L.rnd(1, S, H * hd, seed=3).to(dev)]
    for bad in range(4):
        qkv, fc, k, v = (off(t) if i == bad else t for i, t in enumerate(tensors))
        with pytest.raises(hip.AriaHipError):
            ops.rope_cache_rows_(qkv, fc, slot, pos, k, v, H, hd)
    m = gptfast_routed(dev, 128, 64, 128, 32)
    m.layers[1].attention.wo.weight.data = off(m.layers[1].attention.wo.weight.data)
    with pytest.raises(hip.AriaHipError):
        Scheduler(m, 8).step("ab", [[5, 9], [5, 3, 7]])


def case_gptfast_portion_order(dev, engine=False):
    """A portion of a prompt: logits in the order in which its places are named."""
    from aria_amd.serving import Scheduler

    m = gptfast_toy(dev)
    m.use_decode_engine = engine

    def portion(places):
        s = Scheduler(m, 8)
        s.step(["a"], [[5, 3]], [[]])
        return s.step(["a"], [[9, 2, 77]], [places]).cpu()

    assert torch.equal(portion([2, 0, 2]), portion([0, 1, 2])[[2, 0, 2]])


def case_gptfast_wanted_outside(dev, dim=128, inter=128):
    """Places that a request does not have are left out, in single steps as in packed prompts and in the prompts' one call."""
    from aria_amd.serving import StepBatch

    m = gptfast_routed(dev, dim, 64, inter, 32)
    m.setup_caches(2, 8)

    def step(tokens, starts, rows):
        return m.step(StepBatch.build(tokens, [0, 1], starts, rows, dev)).cpu()

    for tokens, starts in (([[5, 3, 7], [4, 9]], [0, 0]), ([[11], [12]], [3, 2])):
        last = sum(map(len, tokens)) - 1
        both, n = step(tokens, starts, [0, last]), 4 * 2 ** -8
        assert L.logit_err(step(tokens, starts, [-1, 0]), both[:1]) < n and L.logit_err(step(tokens, starts, [last, last + 1]), both[1:]) < n


def case_rows_products(dev, M, N, K, E=3):
    """The weight-streaming products at edges of their token tiles, row groups and windows of the reduction against float64; bf16 results: half an ulp, 2^-9,
    and twice that behind the rounded gate and up of SwiGLU."""
    from aria_amd import ops

    x, w, u = (L.rnd(n, K, seed=i, scale=K ** -0.5 if i else 1.0) for i, n in enumerate((M, N, N)))
    xd, wd, ud = (t.to(dev) for t in (x, w, u))
    want, up = x.double() @ w.double().T, x.double() @ u.double().T
    assert L.rel(ops.rows_gemm(xd, wd, f32), want) < 2e-6 and L.rel(ops.rows_gemm(xd, wd), want) < 2 ** -8
    assert L.rel(ops.rows_swiglu(xd, wd, ud), torch.nn.functional.silu(want) * up) < 2 ** -7
    if K > 2560:
        return
    cuts = sorted([0, 0, M // 3, M])          # the first expert has no rows
    off = torch.tensor(cuts, dtype=torch.int32, device=dev)
    rows = torch.randperm(M, generator=L.gen(M)).to(torch.int32)
    we, ue = (L.rnd(E, N, K, seed=5 + i, scale=K ** -0.5) for i in range(2))
    for idx in (None, rows):
        xs = x if idx is None else x[idx.long()]
        y, z = (torch.cat([xs[a:b].double() @ m[e].double().T for e, (a, b) in enumerate(zip(cuts, cuts[1:]))]) for m in (we, ue))
        kw = {} if idx is None else dict(rows=idx.to(dev))
        assert L.rel(ops.rows_experts(xd, we.to(dev), off, **kw), y) < 2 ** -8
        assert L.rel(ops.rows_experts(xd, we.to(dev), off, w_up=ue.to(dev), **kw), torch.nn.functional.silu(y) * z) < 2 ** -7


def case_rows_experts_uneven(dev, counts, N, K):
    """Experts of no rows, one row, whole token tiles and a row more, among more than 64 experts too: the bits of each expert's product by itself."""
    from aria_amd import ops

    E, M = len(counts), sum(counts)
    x, w, u = (L.rnd(*n, K, seed=i, scale=K ** -0.5 if i else 1.0).to(dev) for i, n in enumerate(((M,), (E, N), (E, N))))
    cuts = [sum(counts[:e]) for e in range(E + 1)]
    rows = torch.randperm(M, generator=L.gen(M)).to(torch.int32)
    xs = x[rows.long().to(dev)]
    each = [(xs[a:b], w[e], u[e]) for e, (a, b) in enumerate(zip(cuts, cuts[1:])) if b > a]
    args = x, w, torch.tensor(cuts, dtype=torch.int32, device=dev), rows.to(dev)
    assert torch.equal(ops.rows_experts(*args), torch.cat([ops.rows_gemm(t, a) for t, a, _ in each]))
    assert torch.equal(ops.rows_experts(*args, w_up=u), torch.cat([ops.rows_swiglu(t, a, b) for t, a, b in each]))


def case_rows_whole_lines(dev, M, N, K):
    """Weights that come by whole lines against their first rows by half lines (too few for whole ones): the same bits, and float64."""
    from aria_amd import ops

    x, w = (L.rnd(n, K, seed=i, scale=K ** -0.5 if i else 1.0) for i, n in enumerate((M, N)))
    xd, wd = x.to(dev), w.to(dev)
    assert N * K >= 3 << 20 > 48 * K and K % 64 == 0
    got = ops.rows_gemm(xd, wd, f32)
    assert L.rel(got, x.double() @ w.double().T) < 2e-6
    for at in (0, N // 2, N - 48):
        assert torch.equal(got[:, at:at + 48], ops.rows_gemm(xd, wd[at:at + 48].contiguous(), f32))


# sixteen, 32 and 64 rows a tile
UNEVEN = [[0] * 65 + [40, 0, 16, 1, 17], [33, 0, 1, 24, 0, 2, 0, 0, 4], [0, 65, 1, 129, 0, 64, 2]]


def case_experts_whole_lines(dev, E, N, K, pair, counts=(0, 1, 2, 17, 5, 70, 16, 3)):
    """Sorted rows whose experts' weights come by whole lines, some with several tiles, against one expert after the other by half lines (too few weights for whole ones): the same bits."""
    from aria_amd import ops

    assert E * N * (1 + pair) * K >= 16 << 20 > 2 * N * K and K % 64 == 0
    counts = [counts[e % len(counts)] for e in range(E)]
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    x = L.rnd(sum(counts), K, seed=1).to(dev)
    w, u = (L.rnd(E, N, K, seed=s, scale=K ** -0.5).to(dev) for s in (2, 3))
    got = ops.rows_experts(x, w, off.to(dev), w_up=u if pair else None)
    for e, (a, n) in enumerate(zip(off.tolist(), counts)):
        if n == 0:
            continue
        one = ops.rows_experts(x[a:a + n], w[e:e + 1], torch.tensor([0, n], dtype=torch.int32, device=dev), w_up=u[e:e + 1] if pair else None)
        assert torch.equal(got[a:a + n], one), e


def case_rows_qkv(dev, M, D, hd, S):
    """Projection, rotation and cache write in one launch against the separate ones on the same product, bit for bit: positions 0 .. and any slots."""
    from aria_amd import gptfast as G
    from aria_amd import ops

    x, w = L.rnd(M, D, seed=1).to(dev), L.rnd(3 * D, D, seed=2, scale=D ** -0.5).to(dev)
    fc = G.precompute_freqs_cis(S, hd, 10000.0).to(dev).contiguous()
    for slots in (1, 3):
        slot = torch.arange(M, dtype=torch.int32) % slots
        pos = torch.arange(M, dtype=torch.int32) // slots
        k, v = (torch.zeros(slots, S, D, dtype=bf16, device=dev) for _ in range(2))
        k2, v2 = torch.zeros_like(k), torch.zeros_like(v)
        where = dict(slot=slot.to(dev), pos=pos.to(dev)) if slots > 1 else {}
        q = ops.rows_qkv_rope_cache(x, w, fc, k, v, hd, **where)
        qkv = ops.rope_cache_rows_(ops.rows_gemm(x, w), fc, slot.to(dev), pos.to(dev), k2, v2, D // hd, hd)
        assert torch.equal(q, qkv[:, :D]) and torch.equal(k, k2) and torch.equal(v, v2)


def gptfast_oracle(m, toks, r=lambda t: t):
    """A whole sequence through a gptfast decoder in float64, in plain torch: (logits [n, vocab], [(rotated keys, values) of a layer, [n, dim] each]).  ``r`` is
    applied to what the kernels keep in 16 bits."""
    c, n = m.config, len(toks)
    w = {name: p.detach().double() for name, p in m.named_parameters()}
    dev, D, H, hd = m.device, c.dim, c.n_head, c.head_dim
    angle = torch.arange(n, dtype=torch.float64, device=dev)[:, None] * c.rope_base ** (-torch.arange(0, hd, 2, dtype=torch.float64, device=dev) / hd)
    cos, sin = r(angle.cos())[:, None], r(angle.sin())[:, None]
    future = torch.ones(n, n, dtype=torch.bool, device=dev).triu(1)

    def norm(x, name):
        return r(x * (x.pow(2).mean(-1, keepdim=True) + c.norm_eps).rsqrt() * w[name + ".weight"])

    def rotate(x):
        a, b = x.view(n, H, hd // 2, 2).unbind(-1)
        return r(torch.stack([a * cos - b * sin, b * cos + a * sin], -1).view(n, D))

    def glu(h, up, gate, down):      # (w1 goes through silu)
        return r(r(torch.nn.functional.silu(r(h @ up.T)) * r(h @ gate.T)) @ down.T)

    x, cache = w["tok_embeddings.weight"][torch.as_tensor(toks, device=dev)], []
    for i in range(c.n_layer):
        p = f"layers.{i}."
        q, k, v = r(norm(x, p + "attention_norm") @ w[p + "attention.wqkv.weight"].T).split(D, -1)
        q, k = rotate(q), rotate(k)
        cache.append((k, v))
        heads = [t.view(n, H, hd).transpose(0, 1).contiguous() for t in (q, k, v)]
        prob = (heads[0] @ heads[1].mT.contiguous() * hd ** -0.5).masked_fill(future, -float("inf")).softmax(-1)
        x = r(x + r(r((prob @ heads[2]).transpose(0, 1).reshape(n, D)) @ w[p + "attention.wo.weight"].T))
        h, f = norm(x, p + "ffn_norm"), p + "feed_forward."
        top, chosen = r(h @ w[f + "gate.weight"].T).topk(c.router_topk, -1)
        score, routed = r(top.softmax(-1)), torch.zeros_like(x)
        for e in range(c.num_experts):
            t, place = (chosen == e).nonzero(as_tuple=True)
            if len(t):
                routed[t] += score[t, place, None] * glu(h[t], *(w[f + "cond_ffn." + name][e] for name in ("w1", "w3", "w2")))
        shared = glu(h, *(w[f + f"shared_ffn.{name}.weight"] for name in ("w1", "w3", "w2")))
        x = r(x + r(r(routed) + shared))
    return norm(x, "norm") @ w["output.weight"].T, cache


def case_gptfast_steps_oracle(dev, monkeypatch, dim, inter, lens, steps=2, vocab=264, top=3):
    """Prompts of several requests, tokens of all of them and a token of one against float64: logits and cache rows, each step seen to be one library call.  Bound:
    three times what 16-bit tensors between exact operations make of the same sequence."""
    from aria_amd import gptfast as G
    from aria_amd.serving import Scheduler

    m, served = gptfast_routed(dev, dim, 64, inter, max(lens) + 8, vocab, top), []
    for name in ("prompts", "run"):
        def seen(self, *a, plain=getattr(G._StepTables, name), name=name):
            out = plain(self, *a)
            served.append((name, out is not None))
            return out
        monkeypatch.setattr(G._StepTables, name, seen)
    toks = [torch.randint(0, 264, (n + steps,), generator=L.gen(n)).tolist() for n in lens]
    exact = [gptfast_oracle(m, t) for t in toks]
    rounded = [gptfast_oracle(m, t, lambda x: x.to(bf16).double()) for t in toks]
    tol = 3 * max(L.logit_err(b[0], a[0].cpu()) for a, b in zip(exact, rounded))
    # a row of keys or values of one head, the worst one
    rows = [[t.reshape(-1, 64) for a in one for pair in a[1] for t in pair] for one in (exact, rounded)]
    cache_tol = 3 * max(L.logit_err(b, a.cpu()) for a, b in zip(*rows))
    assert tol < 0.06 and cache_tol < 0.12, (tol, cache_tol)      # (far below what a step that leaves something out gives, about 1)
    sched, ids = Scheduler(m, max(lens) + steps + 1), list(range(len(lens)))
    got = sched.step(ids, [t[:n] for t, n in zip(toks, lens)], [list(range(n)) for n in lens])
    assert L.logit_err(got, torch.cat([x[0][:n] for x, n in zip(exact, lens)]).cpu()) < tol
    for s in range(steps):
        who = ids[::-1] if s == 0 else ids[:1]
        got = sched.step(who, [[toks[i][lens[i] + s]] for i in who])
        assert L.logit_err(got, torch.stack([exact[i][0][lens[i] + s] for i in who]).cpu()) < tol
    for i in ids:
        n = lens[i] + (steps if i == 0 else 1)
        for layer, pair in enumerate(exact[i][1]):
            kv = m.layers[layer].attention.kv_cache
            for got, want in zip((kv.k, kv.v), pair):
                assert L.logit_err(got[sched.live[i][0], :n].reshape(-1, 64), want[:n].reshape(-1, 64).cpu()) < cache_tol
    assert served == [("prompts", True)] + [("run", True)] * steps


def case_rows_rule():
    """The line between products by rows and by tiles: its points on both sides as measured, and beyond it nothing comes back."""
    from aria_amd import ops

    for M, K, N in ((320, 2560, 7680), (192, 2560, 13312), (320, 1536, 8192), (64, 1024, 32000), (16, 2560, 100352), (96, 4096, 7680), (320, 3328, 2560)):
        assert ops.rows_take(M, K, N), (M, K, N)
    for M, K, N in ((256, 2560, 13312), (128, 1024, 32000), (64, 2560, 100352), (128, 4096, 7680), (320, 4096, 2664), (321, 2560, 2560), (16, 504, 2560), (0, 2560, 64)):
        assert not ops.rows_take(M, K, N), (M, K, N)
    for K in (512, 2560, 4096):
        for N in (64, 7680, 20000, 50000):
            taken = [ops.rows_take(M, K, N) for M in range(1, 400)]
            assert taken == sorted(taken, reverse=True)


def case_experts_line():
    """Rows or tiles by expert: Aria's prompts of 86 .. 288 tokens have gate and up by tiles, of 43 .. 288 the down-projections, as their outputs' bits want it; small
    experts stay by rows; one line for the modules and the prompt step."""
    from aria_amd import ops

    E, K, N = 64, 2560, 1664
    for tokens, pair_tiles, down_rows in ((42, False, True), (43, False, False), (85, False, False), (86, True, False), (280, True, False), (288, True, False)):
        assert ops.rows_experts_take(6 * tokens, E, K, N) and ops.experts_tiles_ahead(6 * tokens, E, K, N) == pair_tiles, tokens
        assert ops.rows_experts_take(6 * tokens, E, N, K, down=True) == down_rows, tokens
    assert not ops.rows_experts_take(6 * 289, E, K, N)
    for M, taken in ((8 * 32, False), (8 * 32 + 1, True)):      # 32 of 1024 x 1536
        assert ops.experts_tiles_ahead(M, 32, 1536, 1024) == taken
    assert not ops.experts_tiles_ahead(27 * 16, 16, 1024, 768) and ops.rows_experts_take(27 * 16, 16, 1024, 768)
    assert not ops.rows_experts_take(27 * 16 + 1, 16, 1024, 768)


def case_gptfast_packed_prompts(dev, dim=256, lens=(9, 1, 40, 17), inter=128):
    """Prompts of several requests packed into one step against each prompt alone, logits at places inside and at the end, and a step on the caches that they
    left; rounding as in ``case_gptfast_decode_batch`` (the flash kernel's probabilities included)."""
    from aria_amd.serving import Scheduler

    m = gptfast_routed(dev, dim, 64, inter, max(lens) + 8)
    toks = [torch.randint(0, 264, (n + 1,), generator=L.gen(n)).tolist() for n in lens]
    places = [sorted({0, n // 2, n - 1}) for n in lens]
    want = []
    for t, p in zip(toks, places):
        s = Scheduler(m, max(lens) + 2)
        want.append((s.step(["x"], [t[:-1]], [p]).cpu().double(), s.step(["x"], [t[-1:]]).cpu().double()))
    sched = Scheduler(m, max(lens) + 2)
    ids = list(range(len(lens)))
    got = sched.step(ids, [t[:-1] for t in toks], places)
    assert L.logit_err(got, torch.cat([w[0] for w in want])) < 4 * 2 ** -8
    got = sched.step(ids, [t[-1:] for t in toks])
    assert L.logit_err(got, torch.cat([w[1] for w in want])) < 4 * 2 ** -8
    assert sched.step(ids[:1], [[1]], [[]]) is None


def case_gptfast_generate(dev):
    """serving.generate on the gptfast decoder: greedy continuation equals arg-max over full prefills wherever that is not a tie."""
    from aria_amd import serving

    m = gptfast_toy(dev)
    m.use_decode_engine = False       # (a bf16 router's close calls may fall either way between the engine and the tile path)
    prompts = [[5, 9, 77], [100, 3, 8, 20, 1]]
    for p, g in zip(prompts, serving.generate(m, prompts, 3, temperature=0)):
        m.setup_caches(1, 16)
        with torch.no_grad():
            lg = m(torch.tensor([p + g], device=dev))[0].float().cpu()
        for i, t in enumerate(g):
            row = lg[len(p) + i - 1]
            assert float(row.max() - row[t]) <= 0.05 * float(row.std())


DESIGNS = {"duguzen": (L, "equal"), "kozipel": (K, "last")}   # cases module, configuration


def write_model(tmp, design="duguzen", seed=12):
    from safetensors.torch import save_file

    cases, name = DESIGNS[design]
    cfg = cases.CONFIGS[name]
    w = cases.checkpoint(cfg, seed=seed)
    (tmp / "config.json").write_text(json.dumps(cfg))
    save_file(w, str(tmp / "model.safetensors"))
    return cfg, w


def case_command_line(dev, tmp, design="duguzen"):
    from aria_amd import inference as I
    from aria_amd import registry, serving

    cfg, _ = write_model(tmp, design)
    a = I.parse_arguments(["--base_model_path", str(tmp), "--prompt_ids", "5,17,3", "--prompt_ids", "9", "--max_new_tokens", "3", "--temperature", "0",
                           "--dtype", "float32"])
    got = I.generate_ids(a, dev)
    m = registry.load_model(str(tmp), dev, f32)
    assert got == serving.generate(m, [[5, 17, 3], [9]], 3, temperature=0) and all(0 <= t < cfg["vocab"] for g in got for t in g)


def case_trace_run(dev, tmp, dtype="float32", design="duguzen"):
    """Steps in, logits out: the files, the order of rows, ``done`` lines, requests that end, a second batch, and the values against the oracle."""
    import numpy as np

    from aria_amd import trace_run

    cases = DESIGNS[design][0]
    O = cases.O
    cfg, w = write_model(tmp, design)
    out = tmp / "out"
    out.mkdir()
    draw = L.clear_tokens if cases is L else (lambda cfg, w, n, seed: L.tokens(cfg, n, seed))
    a, b, c = ([int(t) for t in draw(cfg, w, n, seed=n)] for n in (6, 4, 3))
    steps = [dict(step=0, entries=[dict(id="a", tokens=a[:5], want=[0, 4]), dict(id="b", tokens=b[:2], want=[])], end=[]),
             dict(step=1, entries=[dict(id="b", tokens=[b[2]], want=[]), dict(id="a", tokens=[a[5]], want=[])], end=["a"]),
             dict(step=2, entries=[dict(id="b", tokens=[b[3]], want=[0])], end=["b"]),
             dict(step=3, entries=[dict(id="a", tokens=c, want=[2, 1])], end=["a"])]
    said = io.StringIO()
    rc = trace_run.main(["--model", str(tmp), "--dtype", dtype, "--out", str(out), "--max-tokens", "12"], io.StringIO("".join(json.dumps(s) + "\n" for s in steps)),
                        said, dev)
    assert rc == 0 and said.getvalue().split("\n")[:-1] == [f"done {i}" for i in range(4)]
    assert sorted(os.listdir(out)) == ["0.f32", "2.f32", "3.f32"]
    want = {0: O.forward(cfg, w, a)[[0, 4]], 2: O.forward(cfg, w, b)[[3]], 3: O.forward(cfg, w, c)[[2, 1]]}
    for n, x in want.items():
        got = torch.from_numpy(np.fromfile(out / f"{n}.f32", dtype="<f4").reshape(x.shape).copy())
        assert L.logit_err(got, x) < (5e-5 if dtype == "float32" else cases.model_tol(cfg, w, [a, b, c], bf16)), n


def case_registry():
    from aria_amd import registry

    assert registry.architecture({"architecture": "Duguzen"}) == "Duguzen"
    assert registry.architecture({"architectures": ["AriaForConditionalGeneration"]}) == registry.architecture({"model_type": "aria"})
    assert registry.resolve({"architecture": "Duguzen"})[1].__name__ == "DuguzenForCausalLM"
    assert registry.resolve({"architecture": "Kozipel"})[1].__name__ == "KozipelForCausalLM"
    with pytest.raises(ValueError):
        registry.architecture({"architecture": "nothing"})


# what is done to a float32 model whose steps run by a table of addresses
MODULES_CHANGED = ["subclass", "class", "instance", "wrapped", "global hook", "global pre hook", "config", "runs", "geometry", "attribute", "weight view", "call", "config class"]


def case_float32_step_asks_the_modules(dev, monkeypatch, cases, what):
    """A float32 step's table of addresses stands in for modules: whatever is done to them, the step's logits are those of the step run sublayer by sublayer (as it is
    with a trace).  ``cases``: the model family's cases."""
    from aria_amd.serving import StepBatch

    cfg = cases.CONFIGS["mixed"]
    w, toks = cases.checkpoint(cfg, seed=3), cases.tokens(cfg, 12, seed=1)
    models = [cases.build(cfg, w, dev, torch.float32) for _ in range(2)]

    def layers(m):
        return list(m.weights.values()) if hasattr(m, "weights") else list(m.layers)

    plain = type(layers(models[0])[0].mixer).forward

    def twice_of(y):
        return dict(y, y=2.0 * y["y"]) if isinstance(y, dict) else 2.0 * y

    def twice(self, *a):
        return twice_of(plain(self, *a))

    class Wrap(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, h):
            return twice_of(self.inner(h))

    later, call = [], torch.nn.Module.__call__

    def change(m):
        mixer = layers(m)[0].mixer
        if what == "call":
            monkeypatch.setattr(torch.nn.Module, "__call__", lambda mod, *a: twice_of(call(mod, *a)) if any(mod is layers(m)[0].mixer for m in models) else call(mod, *a))
        elif what == "subclass":
            mixer.__class__ = type("Twice", (type(mixer),), dict(forward=twice))
        elif what == "class":
            monkeypatch.setattr(type(mixer), "forward", twice)
        elif what == "instance":
            mixer.forward = lambda *a: twice(mixer, *a)
        elif what == "wrapped":
            owner = next(L for L in layers(m) if L.mlp is not None)
            owner.mlp = Wrap(owner.mlp)
        elif what == "config":
            for name in ("residual_mult", "embedding_scale", "logit_softcap"):   # (Duguzen's has none of them: a layer run less)
                if hasattr(m.config, name):
                    setattr(m.config, name, 0.25 * getattr(m.config, name))
            if hasattr(m, "weights"):
                m.config.layers.pop()
        elif what == "runs":
            if hasattr(m, "weights"):
                m.caches[0], m.caches[1] = type(m.caches[0])(*m.caches[0].rows.shape, f32, dev), type(m.caches[0])(*m.caches[1].rows.shape, f32, dev)
                m.ropes[0] = m.ropes[0].flip(1).contiguous()
            else:
                m.config.runs[3].again = not m.config.runs[3].again
        elif what == "geometry":
            for part in getattr(mixer, "parts", [mixer]):
                for name in ("scale", "q_scale"):
                    if name in part.geometry:
                        part.geometry[name] = 0.25 * part.geometry[name]
        elif what == "attribute":
            for part in m.modules():
                for name, new in (("top", lambda k: 1), ("norm_n", lambda n: n - 1), ("eps", lambda e: 0.5), ("ff", lambda n: n + 8)):
                    if name in part.__dict__:
                        setattr(part, name, new(getattr(part, name)))
        elif what == "weight view":
            m.head.data = m.head.data.flip(0)
        elif what == "config class":   # (a constant that no entry of the object holds)
            name = "residual_mult" if hasattr(m.config, "residual_mult") else "layers"
            now, was = [2], getattr(m.config, name)
            whole = property(lambda c: was[:now[0]] if name == "layers" else was * now[0], lambda c, v: None)
            m.config.__class__ = type("Config", (type(m.config),), {name: whole})
            later.append(lambda: now.__setitem__(0, 3))

    def hook(mod, args, out=None):   # (everything that a first mixer returns, or is given, doubled)
        if any(mod is layers(m)[0].mixer for m in models):
            return twice_of(out) if out is not None else (2.0 * args[0],) + tuple(args[1:])

    def both(a, b):
        got, want = (m.step(StepBatch.build([toks[a:b]], [0], [a], None, dev), t) for m, t in zip(models, (None, [])))
        assert torch.equal(got.cpu(), want.cpu())
        return got.cpu()

    for m in models:
        m.setup_caches(1, 12)
    before = both(0, 5)
    for m in models:
        change(m)
    everywhere, handle = torch.nn.modules.module, None
    if what == "global hook":
        handle = everywhere.register_module_forward_hook(hook)
    elif what == "global pre hook":
        handle = everywhere.register_module_forward_pre_hook(hook)
    try:
        first = both(0, 5)
        assert not torch.equal(first, before)
        for f in later:
            f()
        assert not later or not torch.equal(both(0, 5), first)
        both(5, 8), both(8, 9)
    finally:
        if handle is not None:
            handle.remove()


def case_stepped_model_copied(dev, cases, dtype):
    """A model that has made a step's tables is copied and pickled like any other; the copy's steps read its own weights and caches."""
    import copy
    import pickle

    from aria_amd.serving import StepBatch

    cfg = cases.CONFIGS["mixed"]
    m = cases.build(cfg, cases.checkpoint(cfg, seed=3), dev, dtype)
    toks = cases.tokens(cfg, 12, seed=1)
    m.setup_caches(1, 12)

    def steps(m):
        return [m.step(StepBatch.build([toks[a:b]], [0], [a], None, dev)).cpu() for a, b in ((0, 5), (5, 6))]

    want = steps(m)
    copies = copy.deepcopy(m), pickle.loads(pickle.dumps(m))
    with torch.no_grad():
        for t in m.parameters():
            t.zero_()
    assert not torch.equal(steps(m)[1], want[1])
    for c in copies:
        assert all(torch.equal(x, y) for x, y in zip(steps(c), want))


def case_stepped_model_released(dev, cases, dtype):
    """A model that has made a step's tables is given back with its last reference, its memory with it, not when cycles are next collected."""
    import gc
    import weakref

    from aria_amd.serving import StepBatch

    cfg = cases.CONFIGS["mixed"]
    m = cases.build(cfg, cases.checkpoint(cfg, seed=3), dev, dtype)
    toks = cases.tokens(cfg, 12, seed=1)
    m.setup_caches(1, 12)
    for a, b in ((0, 5), (5, 6)):
        m.step(StepBatch.build([toks[a:b]], [0], [a], None, dev))
    held = [weakref.ref(t) for t in (m, *m.parameters())]
    gc.collect()
    gc.disable()
    try:
        del m
        assert not any(r() is not None for r in held)
    finally:
        gc.enable()
