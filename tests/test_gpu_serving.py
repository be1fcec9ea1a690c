"""Scheduler, command line and trace runner on hardware (-m gpu)."""
import json
import os
import subprocess
import sys

import pytest
import torch

from tests import serving_cases as C

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def real_library():
    from aria_amd import hip

    assert not hip.is_emulated() and hip.get_lib().path.endswith("libaria_hip.so") and torch.cuda.is_available()
    yield


@pytest.mark.parametrize("dim,head_dim,inter,requests,longest", [(128, 64, 128, 2, 9), (512, 128, 1024, 16, 30), (2560, 128, 1664, 5, 400),
                                                                    (640, 64, 264, 3, 9), (1920, 64, 1800, 16, 300)])
def test_gptfast_decode_batch(dim, head_dim, inter, requests, longest):
    C.case_gptfast_decode_batch(DEV, dim, head_dim, inter, requests, longest)


@pytest.mark.parametrize("design", ["duguzen", "gptfast", "kozipel"])
def test_wanted_rows(design):
    C.case_wanted_rows(DEV, design)


def test_gptfast_wanted_outside():
    C.case_gptfast_wanted_outside(DEV)
    C.case_gptfast_wanted_outside(DEV, 512, 512)


@pytest.mark.parametrize("engine", [False, True])
def test_gptfast_portion_order(engine):
    C.case_gptfast_portion_order(DEV, engine)


def test_gptfast_ids():
    C.case_gptfast_ids(DEV)


def test_gptfast_slot_twice():
    C.case_gptfast_slot_twice(DEV)


def test_gptfast_hooks():
    C.case_gptfast_hooks(DEV)
    C.case_gptfast_hooks(DEV, 512, 512)


def test_build():
    C.case_build(DEV)


def test_decode_splits(monkeypatch):
    C.case_decode_splits(DEV, monkeypatch)


@pytest.mark.parametrize("head_dim", [64, 128])
def test_decode_keys_once(monkeypatch, head_dim):
    C.case_decode_keys_once(DEV, monkeypatch, head_dim)


def test_alignment():
    C.case_alignment(DEV)


def test_gptfast_weights_given_up():
    C.case_gptfast_weights_given_up(DEV)


def test_gptfast_moved_weights():
    C.case_gptfast_moved_weights(DEV)


@pytest.mark.parametrize("M,N,K", [(1, 100, 128), (16, 33, 1024), (17, 264, 1032), (33, 16, 1800), (64, 1000, 2560), (65, 7, 1792), (320, 40, 2568), (40, 130, 3336), (15, 24, 4096)])
def test_rows_products(M, N, K):
    C.case_rows_products(DEV, M, N, K)


@pytest.mark.parametrize("M,N,K", [(1, 3072, 1024), (16, 2050, 1536), (64, 2049, 1536), (33, 1900, 1664), (17, 1777, 1792), (16, 2000, 1728), (64, 1300, 2496), (9, 100352, 2560), (20, 1000, 3328),
                                   (16, 990, 3264), (30, 800, 4096)])
def test_rows_whole_lines(M, N, K):
    C.case_rows_whole_lines(DEV, M, N, K)


@pytest.mark.parametrize("E,N,K,pair", [(8, 512, 2048, True), (8, 1024, 2048, False), (16, 600, 1024, True), (9, 1250, 1536, False), (16, 300, 1792, True), (64, 1664, 2560, True)])
def test_experts_whole_lines(E, N, K, pair):
    C.case_experts_whole_lines(DEV, E, N, K, pair)


@pytest.mark.parametrize("N,K", [(33, 1024), (1664, 2560), (24, 1672)])
@pytest.mark.parametrize("counts", C.UNEVEN)
def test_rows_experts_uneven(counts, N, K):
    C.case_rows_experts_uneven(DEV, counts, N, K)


@pytest.mark.parametrize("M,D,hd,S", [(5, 512, 64, 8), (100, 2560, 128, 104), (37, 768, 64, 40)])
def test_rows_qkv(M, D, hd, S):
    C.case_rows_qkv(DEV, M, D, hd, S)


@pytest.mark.parametrize("dim,inter,lens", [(512, 512, (9, 1, 20, 7)), (1024, 1664, (20,)), (1536, 1024, (2, 3, 5, 2, 17, 1)), (2560, 1664, (33, 30, 8))])
def test_gptfast_packed_prompts_in_one_call(dim, inter, lens):
    C.case_gptfast_packed_prompts(DEV, dim, lens, inter)


@pytest.mark.parametrize("dim,inter,lens,vocab", [(512, 512, (9, 1, 20, 7), 264), (1024, 1664, (20,), 264), (2560, 1664, (33, 30, 8), 264), (2560, 1664, (140, 1), 264),
                                                  (512, 512, (9, 10), 52002), (512, 512, (9, 10), 52003)])   # (heads by tiles; of odd size)
def test_gptfast_steps_oracle(monkeypatch, dim, inter, lens, vocab):
    C.case_gptfast_steps_oracle(DEV, monkeypatch, dim, inter, lens, vocab=vocab)


def test_gptfast_steps_oracle_by_tiles(monkeypatch):
    """more tokens than the projections take by rows"""
    C.case_gptfast_steps_oracle(DEV, monkeypatch, 2560, 640, (200, 8), top=2)


def test_gptfast_packed_prompts():
    C.case_gptfast_packed_prompts(DEV)
    C.case_gptfast_packed_prompts(DEV, 1024, (300, 64, 65, 2, 129))


@pytest.mark.parametrize("engine", [False, True])
def test_gptfast_batch(engine):
    C.case_gptfast_batch(DEV, engine)


def test_gptfast_generate():
    C.case_gptfast_generate(DEV)


designs = pytest.mark.parametrize("design", sorted(C.DESIGNS))


@designs
def test_command_line(tmp_path, design):
    C.case_command_line(DEV, tmp_path, design)


@designs
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_trace_run(tmp_path, dtype, design):
    C.case_trace_run(DEV, tmp_path, dtype, design)


@designs
def test_trace_run_program(tmp_path, design):
    """bin/trace_run as a program: a step a line, an answer before the next."""
    cfg, _ = C.write_model(tmp_path, design)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.Popen([sys.executable, os.path.join(root, "bin", "trace_run"), "--model", str(tmp_path), "--dtype", "bfloat16", "--out", str(tmp_path),
                          "--max-tokens", "8"], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    try:
        for n, toks in enumerate(([1, 2, 3], [4], [5])):
            p.stdin.write(json.dumps(dict(step=n, entries=[dict(id="x", tokens=toks, want=[0])], end=["x"] if n == 2 else [])) + "\n")
            p.stdin.flush()
            assert p.stdout.readline().strip() == f"done {n}"
            assert os.path.getsize(tmp_path / f"{n}.f32") == 4 * cfg["vocab"]
        p.stdin.close()
        assert p.wait(timeout=60) == 0
    finally:
        p.kill()
