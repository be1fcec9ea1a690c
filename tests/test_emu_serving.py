"""Scheduler, command line and trace runner on CPU through the SIMT emulator."""
import pytest

from tests import serving_cases as C

DEV = "cpu"


@pytest.fixture(scope="module", autouse=True)
def emu():
    from tests.emu import emu_lib

    emu_lib.install()
    yield
    emu_lib.uninstall()


def test_gptfast_decode_batch():
    C.case_gptfast_decode_batch(DEV, 128, 64, 128, 3)


@pytest.mark.parametrize("design", ["duguzen", "gptfast", "kozipel"])
def test_wanted_rows(design):
    C.case_wanted_rows(DEV, design)


def test_gptfast_wanted_outside():
    C.case_gptfast_wanted_outside(DEV)


@pytest.mark.parametrize("engine", [False, True])
def test_gptfast_portion_order(engine):
    C.case_gptfast_portion_order(DEV, engine)


def test_gptfast_ids():
    C.case_gptfast_ids(DEV)


def test_gptfast_slot_twice():
    C.case_gptfast_slot_twice(DEV)


def test_gptfast_hooks():
    C.case_gptfast_hooks(DEV)


def test_build():
    C.case_build(DEV)


def test_decode_splits(monkeypatch):
    C.case_decode_splits(DEV, monkeypatch, run=False)


def test_alignment():
    C.case_alignment(DEV)


def test_gptfast_weights_given_up():
    C.case_gptfast_weights_given_up(DEV)


def test_gptfast_moved_weights():
    C.case_gptfast_moved_weights(DEV, ("assign", "module"))


@pytest.mark.parametrize("M,N,K", [(5, 20, 136), (70, 9, 520)])
def test_rows_products(M, N, K):
    C.case_rows_products(DEV, M, N, K)


def test_rows_whole_lines():
    C.case_rows_whole_lines(DEV, 2, 1894, 1664)


def test_experts_whole_lines():
    C.case_experts_whole_lines(DEV, 16, 512, 1024, True, (1, 0, 0, 18, 0, 0, 0, 0))


@pytest.mark.parametrize("counts", C.UNEVEN)
def test_rows_experts_uneven(counts):
    C.case_rows_experts_uneven(DEV, counts, 20, 136)


def test_rows_qkv():
    C.case_rows_qkv(DEV, 37, 128, 64, 40)


def test_gptfast_packed_prompts():
    C.case_gptfast_packed_prompts(DEV, 128, (5, 1, 9))


def test_rows_rule():
    C.case_rows_rule()


def test_experts_line():
    C.case_experts_line()


def test_gptfast_steps_oracle(monkeypatch):
    C.case_gptfast_steps_oracle(DEV, monkeypatch, 512, 512, (3, 1, 5))


def test_gptfast_batch():
    C.case_gptfast_batch(DEV, engine=False)   # (the engine's emulated form takes a minute: on hardware only)


def test_gptfast_generate():
    C.case_gptfast_generate(DEV)


designs = pytest.mark.parametrize("design", sorted(C.DESIGNS))


@designs
def test_command_line(tmp_path, design):
    C.case_command_line(DEV, tmp_path, design)


@designs
def test_trace_run(tmp_path, design):
    C.case_trace_run(DEV, tmp_path, design=design)


def test_registry():
    C.case_registry()


def test_trace_run_refuses_a_dtype_the_model_does_not_have(tmp_path):
    import io
    import json

    from aria_amd import trace_run

    (tmp_path / "config.json").write_text(json.dumps({"architectures": ["AriaForConditionalGeneration"]}))
    assert trace_run.main(["--model", str(tmp_path), "--dtype", "float32", "--out", str(tmp_path), "--max-tokens", "4"], io.StringIO(""), io.StringIO(), DEV) == 3
