"""The segment build and the centroids at the sizes where their kernels change form.

Starts bit for bit against the CPU oracle: dims a lane holds 1 / 2 / 4 / any (D 65, 256, 320),
the two LDS sizes (512 / 513 pools), and segments past the reciprocals kept in LDS (counts of
2048 and more are divided), keys that are not finite (their pairs never merge). Centroids in all
three modes, equal (the fp32 order is the definition, tolerance 0): odd and even D, unaligned
pairs, more members than a batch and than one load of ids, holes and empty buckets.
"""

import numpy as np
import pytest
import torch

import oracle
from oracle import lsa_oracle
from lsa_rocm_lab.port import pipeline

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _keys(T, H, D, seed):
    g = torch.Generator().manual_seed(seed)
    centers = torch.randn(16, D, generator=g)
    return centers[torch.randint(0, 16, (H, T // 9 + 1), generator=g).repeat_interleave(9, 1)[:, :T]].transpose(0, 1) \
        + 0.3 * torch.randn(T, H, D, generator=g)


@pytest.mark.parametrize("D,pool,T,target,max_size", [
    (65, 2, 300, 9, 64),
    (256, 4, 2048, 500, 64),   # 512 pools
    (320, 4, 2050, 470, 64),   # 513 pools
    (16, 64, 9000, 3, 8192),   # counts past 2048
    (128, 1, 64, 1, 64),
])
def test_segment_starts(D, pool, T, target, max_size):
    keys = _keys(T, 2, D, seed=T + D)
    got = pipeline.segment_starts(keys[None].to(DEV), target, pool, max_size).cpu().numpy()
    for h in range(2):
        assert np.array_equal(got[0, h], oracle.ward_segments_keys(keys[:, h].numpy(), pool, target, max_size))


def test_infinite_keys_never_merge():
    keys = _keys(256, 1, 64, seed=5)
    keys[100, 0, 7] = float("inf")
    keys[180, 0, 3] = float("nan")
    got = pipeline.segment_starts(keys[None].to(DEV), 12, 4, 128).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = _starts_without_nan(keys[:, 0].numpy(), 4, 12, 128)
    assert np.array_equal(got[0, 0], want)


def _starts_without_nan(keys, pool, target, max_size):
    """The oracle's merge with an inadmissible pair written as infinity (argmin takes a NaN)."""
    sums, size = lsa_oracle.ward_pool_sums(keys, pool)
    cost = lambda i: lsa_oracle.ward_pair_cost(sums[i], sums[i + 1], int(size[i]), int(size[i + 1]), max_size)
    starts, sums, size = list(range(0, len(keys), pool)), list(sums), list(size)
    while len(starts) > target:
        c = np.array([cost(i) for i in range(len(starts) - 1)])
        i = int(np.argmin(np.where(np.isfinite(c), c, np.inf)))
        sums[i:i + 2] = [sums[i] + sums[i + 1]]
        size[i:i + 2] = [size[i] + size[i + 1]]
        del starts[i + 1]
    return np.array(starts + [len(keys)])


@pytest.mark.parametrize("D,cap,offset", [(128, 70, 0), (128, 9, 1), (66, 130, 0), (63, 64, 0), (64, 1, 0), (512, 20, 0)])
@pytest.mark.parametrize("mode", ["mean", "normalized", "sum"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_centroids(D, cap, offset, mode, dtype):
    g = torch.Generator().manual_seed(D + cap)
    flat = torch.randn(200 * D + offset, generator=g).to(dtype)
    members = torch.randint(-60, 200, (11, cap), generator=g).clamp(min=-1).to(torch.int32)
    members[4] = -1
    members[5] = torch.arange(cap) % 200  # no holes
    keys = flat.to(DEV)[offset:].view(200, D)
    c32, c16 = pipeline.bucket_centroids(keys, members.to(DEV), mode)
    want = oracle.bucket_centroids(flat[offset:].view(200, D).float().numpy(), members.numpy(), mode)
    assert np.array_equal(c32.cpu().numpy(), want)
    assert torch.equal(c16.cpu(), torch.from_numpy(want).to(torch.bfloat16))
