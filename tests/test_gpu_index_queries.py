"""The index queries at the sizes where their kernel changes form, equal to the oracle (the fp32
order of the sum is the definition, tolerance 0): 4 / 2 / 1 dims a thread by size, alignment and
head dim, batches longer and shorter than the rows, groups that divide a batch and one that does
not, chunks that end inside a batch."""

import numpy as np
import pytest
import torch

import oracle
from lsa_rocm_lab.port import pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,chunk,Hq,Hkv,D,offset", [
    (2200, 1, 32, 8, 128, 0),    # 4 dims a thread, 4 rows
    (1100, 4, 32, 4, 128, 0),    # 4 dims, 32 rows, whole batches of a group of 8
    (4200, 5, 8, 4, 128, 0),     # 4 dims, 10 rows, a group of 2
    (2100, 9, 16, 16, 64, 0),    # one head a group
    (4100, 17, 32, 4, 64, 0),    # 2 dims a thread, 136 rows
    (300, 64, 16, 4, 64, 0),     # 1 dim a thread
    (130, 65, 12, 2, 64, 0),     # a group of 6
    (50, 7, 4, 2, 33, 0),        # odd head dim
    (50, 3, 4, 2, 64, 1),        # rows off a 4-byte boundary, a short batch
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_index_queries(T, chunk, Hq, Hkv, D, offset, dtype):
    g = torch.Generator().manual_seed(T + chunk)
    flat = torch.randn(2 * T * Hq * D + offset, generator=g).to(dtype)
    q = flat[offset:].view(2, T, Hq, D)
    got = pipeline.index_queries(flat.cuda()[offset:].view(2, T, Hq, D), Hkv, chunk).cpu().numpy()
    want = oracle.index_queries(q[:, :T // chunk * chunk].float().numpy(), Hkv, chunk)
    assert np.array_equal(got, want)
