"""The size rules that choose between two kernels: every form the newer kernel does not take stays with
the general one, the environment's split counts are obeyed, and calls on both sides of a line that was
measured go where they were faster."""

import math

import pytest
import torch

from lsa_rocm_lab.port import pipeline
from lsa_rocm_lab.port.read_kernel_tiled import _sweep_pays

PREFILL = dict(dtype=torch.bfloat16, B=1, Tq=16384, Tk=16384, Hq=32, Hkv=8, D=128, width=4612, token_stride=1024,
               scale=128 ** -0.5)


@pytest.fixture(autouse=True)
def _no_split_counts(monkeypatch):
    for name in ("LSA_READ_SPLITS", "LSA_SELECT_SPLITS"):
        monkeypatch.delenv(name, raising=False)


def test_a_split_count_from_the_environment_is_for_the_gather(monkeypatch):
    assert _sweep_pays(**PREFILL)
    monkeypatch.setenv("LSA_READ_SPLITS", "4")
    assert not _sweep_pays(**PREFILL)
    monkeypatch.setenv("LSA_READ_SPLITS", "")  # as unset
    assert _sweep_pays(**PREFILL)


@pytest.mark.parametrize("form", [
    dict(dtype=torch.float32), dict(D=32), dict(D=256), dict(Hq=24), dict(Hq=128), dict(token_stride=1 << 24),
    dict(width=0), dict(Tk=0), dict(scale=0.0), dict(scale=-0.1), dict(scale=math.inf), dict(scale=math.nan),
])
def test_forms_the_sweep_does_not_take(form):
    assert not _sweep_pays(**{**PREFILL, **form})


@pytest.mark.parametrize("sizes,sweep", [
    (dict(Tq=1, Tk=32768), False),              # a decode step
    (dict(B=32, Tq=1, Tk=131072), False),
    (dict(Tq=1024, Tk=1024), True),             # gather / sweep 301 / 68 us
    (dict(Tq=2048, Tk=32768), True),            # 2590 / 1280 us
    (dict(Tq=512, Tk=32768), False),            # one workgroup crosses 512 tiles: 1.3 ms against 660 us
    (dict(Tq=2048, Tk=2048, Hq=1, Hkv=1, D=64, token_stride=64), False),  # 37 / 106 us
    (dict(Tq=32768, Tk=32768), True),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sweep_by_size(sizes, sweep, dtype):
    assert _sweep_pays(**{**PREFILL, **sizes, "dtype": dtype}) is sweep


@pytest.mark.parametrize("R,G,rows,tiles", [
    (63, 64, 4096, False), (64, 8, 1024, True),  # 51 / 28 us
    (255, 1, 4096, False), (256, 1, 2048, True),
    (600, 1, 64, False),                         # 21 / 26 us
    (2048, 1, 255, False), (2048, 1, 256, True),  # 46 / 36 us at 2^19 scores
    (1, 8, 4096, False),                         # a decode step
])
def test_rows_select_by_size(monkeypatch, R, G, rows, tiles):
    assert pipeline._rows_pay(R, G, rows) is tiles
    monkeypatch.setenv("LSA_SELECT_SPLITS", "1")
    assert not pipeline._rows_pay(R, G, rows)
