"""Latent-attention family and Duguzen through the SIMT emulator (CPU): tests/latent_cases.py at small sizes."""
import pytest
import torch

from tests import latent_cases as C
from tests import serving_cases as S

bf16, f32 = torch.bfloat16, torch.float32
DEV = "cpu"
both = pytest.mark.parametrize("dtype", [bf16, f32], ids=["bf16", "f32"])


@pytest.fixture(scope="module", autouse=True)
def emu():
    from tests.emu import emu_lib

    emu_lib.install()
    yield
    emu_lib.uninstall()


@both
def test_dyt_stream(dtype):
    C.case_dyt_stream(DEV, dtype)


@both
def test_dyt_stream_parts(dtype):
    C.case_dyt_stream_parts(DEV, dtype, 5, 136, 5, 1)


@pytest.mark.parametrize("dtype,T,D,k,offset", [(bf16, 530, 520, 5, 3), (bf16, 5000, 72, 2, 0), (f32, 4097, 176, 3, 1), (f32, 1400, 520, 5, 2)])
def test_dyt_stream_eight_columns(dtype, T, D, k, offset):
    """Beyond the lines at which a lane takes eight columns, and a wave several tokens, in either type."""
    C.case_dyt_stream_parts(DEV, dtype, T, D, k, offset)


@both
def test_activations(dtype):
    C.case_activations(DEV, dtype)


@pytest.mark.parametrize("M,N,K", [(5, 24, 16), (70, 136, 72)])
def test_gemm_relu_squared(M, N, K):
    C.case_gemm_relu_squared(DEV, M, N, K)


def test_gemm_thin():
    C.case_gemm_thin(DEV, 33, 520, 8)
    C.case_gemm_thin(DEV, 5, 512, 16)


@pytest.mark.parametrize("M,N,K", [(5, 9, 4), (70, 66, 20)])
def test_gemm_f32(M, N, K):
    C.case_gemm_f32(DEV, M, N, K)


def test_gemm_f32_whole_lines():
    C.case_gemm_f32_whole_lines(DEV, 3, 400, 3936)


@pytest.mark.parametrize("M,N,K", [(560, 481, 20), (560, 484, 100)])
def test_gemm_f32_tiles(M, N, K):
    C.case_gemm_f32_tiles(DEV, M, N, K)


@pytest.mark.parametrize("E,groups,keep,k", [(8, 2, 1, 2), (12, 4, 2, 3), (6, 1, 1, 1), (8, 8, 3, 3), (100, 10, 4, 12)])
def test_route_groups(E, groups, keep, k):
    C.case_route_groups(DEV, 9, E, groups, keep, k)


def test_sort_wide():
    C.case_sort_wide(DEV, T=12)


@both
@pytest.mark.parametrize("m,lens", [(C.mixer(), (7, 1, 12)), (C.mixer(heads=2, dim=13, rot_dim=6, vdim=11, kv_rank=21), (3, 2)),
                                    (C.mixer(heads=1, dim=100, rot_dim=60, vdim=70, kv_rank=72), (5,))])
def test_latent_attention(dtype, m, lens):
    C.case_latent_attention(DEV, dtype, m, lens, tail=2)


@pytest.mark.parametrize("heads,R", [(17, 140), (2, 600)])
def test_latent_attention_kernel_classes(heads, R):
    C.case_latent_attention(DEV, bf16, C.mixer(heads=heads, dim=8, rot_dim=8, vdim=8, kv_rank=R), (3,), tail=1)


@both
def test_one_key_stands_out(dtype):
    C.case_one_key_stands_out(DEV, dtype, [0, 1, 63, 64, 65], 68)


@pytest.mark.parametrize("dtype,name", [(bf16, "odd"), (f32, "odd"), (f32, "mixed"), (bf16, "broad"), (bf16, "vocabulary")])
def test_model(dtype, name):
    C.case_model(DEV, dtype, name, lens=(4, 1, 2), tail=2)


@pytest.mark.parametrize("width,ff,requests", [(136, 120, 3), (264, 128, 16), (1032, 136, 2)])
def test_decode_batch(width, ff, requests):
    C.case_decode_batch(DEV, width, ff, requests)


def test_portions():
    C.case_portions(DEV, f32, "equal", n=15)


@both
def test_continuation_beside_decode(dtype):
    C.case_continuation_beside_decode(DEV, dtype)


def test_borrowed_layers_keep_their_own_cache():
    C.case_borrowed_layers_keep_their_own_cache(DEV, bf16)


@both
def test_stream_after_every_layer(dtype):
    C.case_stream_after_every_layer(DEV, dtype, n=3)


@both
def test_greedy_generation(dtype, tmp_path):
    C.case_greedy_generation(DEV, dtype, n_new=4, tmp=tmp_path)


def test_bad_inputs():
    C.case_bad_inputs(DEV)


@pytest.mark.parametrize("T,n", [(1, 200), (70, 80)])
def test_latent_partials_anywhere(T, n):
    C.case_latent_partials_anywhere(DEV, T, n)


@both
@pytest.mark.parametrize("H,R,dr", [(3, 40, 6), (2, 300, 64), (16, 512, 64)])
def test_latent_cache_rows(dtype, H, R, dr):
    C.case_latent_cache_rows(DEV, dtype, H, R, dr)


@pytest.mark.parametrize("name", ["ends", "stream"])
def test_float32_step_beyond_a_round(monkeypatch, name):
    cfg, counts = C.WIDE_STEPS[name]
    C.case_float32_step_beyond_a_round(DEV, monkeypatch, C.build, cfg, C.checkpoint(cfg, seed=3), counts, every_row=False)


@pytest.mark.parametrize("name", ["mixed", "odd"])
def test_float32_step_as_one_call(monkeypatch, name):
    C.case_float32_step_as_one_call(DEV, monkeypatch, name)


@pytest.mark.parametrize("H,R,dr,dv", [(3, 36, 8, 20), (20, 52, 10, 16), (5, 21, 6, 11)])
@pytest.mark.parametrize("runs", [[(0, 0, 41), (2, 3, 30)], [(0, 20, 3), (1, 0, 1), (0, 5, 2), (2, 60, 35)], [(1, 70, 1), (0, 4, 1), (2, 0, 1)]])
def test_latent_attention_f32(H, R, dr, dv, runs):
    C.case_latent_attention_f32(DEV, H, R, dr, dv, runs)


@pytest.mark.parametrize("what", S.MODULES_CHANGED)
def test_float32_step_asks_the_modules(monkeypatch, what):
    S.case_float32_step_asks_the_modules(DEV, monkeypatch, C, what)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_stepped_model_copied(dtype):
    S.case_stepped_model_copied(DEV, C, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_stepped_model_released(dtype):
    S.case_stepped_model_released(DEV, C, dtype)
