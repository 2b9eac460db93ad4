"""The per-row read as a masked sweep on the matrix cores (lsa_read_rows) vs the fp64 oracle.

Cases at the kernel's edges: row counts and caches around its tiles (32-row blocks, 64-key
tiles, 256 columns), both 16-bit types, head dims 64 and 128, query groups 1, 2, 4 and 8,
shared and per-kv-head lists, several batch rows and one pool for all of them, skipped ids,
ids listed twice (those rows go to the gather), rows with nothing to read under both
contracts, K/V values that are not finite (listed and not), lists too sparse for the sweep,
caches long enough for several bitmap segments and several slabs of rows.

Bound: the output's own rounding (2^-9 of it in bf16, 2^-12 in fp16, doubled), plus 2^-13 of
the largest |v| for the split weights (2^-16) and the fp32 scores of up to 128 products.
"""

import numpy as np
import pytest
import torch

import oracle
from lsa_rocm_lab import _abi
from lsa_rocm_lab.port import pipeline
from lsa_rocm_lab.port.read_kernel_tiled import _sparse_read, _sweep_pays

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def make(dtype, B, Tq, Tk, Hq, Hkv, D, W, per_head=False, seed=0, short=1.0, pool=False):
    """q, k, v and distinct ids in a random order, -1 and out-of-range ids among them, every
    17th list empty."""
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Tq, Hq, D, generator=g).to(dtype)
    k = torch.randn(1 if pool else B, Tk, Hkv, D, generator=g).to(dtype)
    v = torch.randn(1 if pool else B, Tk, Hkv, D, generator=g).to(dtype)
    shape = (B, Tq, Hkv) if per_head else (B, Tq)
    n = int(np.prod(shape))
    rng = np.random.default_rng(seed)
    ids = np.full((n, W), -1, np.int32)
    for i in range(n):
        m = min(W, Tk)
        ids[i, :m] = rng.permutation(Tk)[:m]
    ids[:, 5::13] = -1
    ids[::7, 0] = Tk + 3
    lengths = rng.integers(0, max(1, int(W * short)) + 1, n).astype(np.int32)
    lengths[::17] = 0
    return q, k, v, torch.from_numpy(ids.reshape(*shape, W)), torch.from_numpy(lengths.reshape(shape))


def sweep(q, k, v, ids, lengths, empty_nan=False, scale=None):
    B, Tq, Hq, D = q.shape
    Tk, Hkv = k.shape[1:3]
    per_head = ids.dim() == 4
    args = [t.to(DEV).contiguous() for t in (q, k, v, ids, lengths)]
    dt, W = _abi.dtype_code(q.dtype), ids.shape[-1]
    nbytes = _abi.size("lsa_read_rows_scratch_bytes", dt, B, Tq, Tk, Hq, Hkv, D, W, int(per_head))
    assert nbytes > 0
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=DEV)  # needs no initialisation
    out = torch.full_like(args[0], float("nan"))
    sb = args[1].stride(0) if k.shape[0] == B else 0
    print(f"rows sweep q={tuple(q.shape)} {q.dtype} Tk={Tk} Hkv={Hkv} W={W} per_head={per_head}", flush=True)
    _abi.call("lsa_read_rows", args[0].data_ptr(), args[1].data_ptr(), args[2].data_ptr(), dt, B, Tq, Tk, Hq, Hkv, D,
              sb, args[1].stride(1), args[1].stride(2), args[3].data_ptr(), args[4].data_ptr(), W, int(per_head),
              float(D ** -0.5 if scale is None else scale), int(empty_nan), ws.data_ptr(), nbytes, out.data_ptr(),
              _abi.stream(out.device))
    torch.cuda.synchronize()
    return out


def check(q, k, v, ids, lengths, empty_nan=False, rows=None):
    got = sweep(q, k, v, ids, lengths, empty_nan).float().cpu().numpy()
    kk, vv = (t.expand(q.shape[0], *t.shape[1:]).float().numpy() for t in (k, v))
    idn = ids.numpy().copy()
    idn[idn >= k.shape[1]] = -1  # the oracle indexes rows; out-of-range ids are skipped like -1
    pick = slice(None) if rows is None else rows
    want = oracle.sparse_read(q[:, pick].float().numpy(), kk, vv, idn[:, pick], lengths.numpy()[:, pick],
                              empty="nan" if empty_nan else "zero")
    got = got[:, pick]
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    ok = np.isfinite(want)
    bound = RTOL[q.dtype] * np.abs(want[ok]) + 2.0 ** -13 * float(np.nanmax(np.abs(vv[np.isfinite(vv)])))
    err = np.abs(got[ok] - want[ok])
    assert (err <= bound).all(), (err.max(), (err - bound).max())


@pytest.mark.parametrize("dtype,B,Tq,Tk,Hq,Hkv,D,W,per_head", [
    (torch.bfloat16, 1, 1, 1, 8, 2, 128, 4, False),        # one row, one key
    (torch.bfloat16, 1, 31, 63, 4, 1, 64, 63, False),      # one key short of a tile, a row short of a block
    (torch.float16, 1, 33, 65, 8, 1, 128, 65, False),      # one past
    (torch.bfloat16, 2, 64, 256, 8, 8, 128, 200, False),   # query group 1: 256 rows a workgroup
    (torch.float16, 2, 129, 321, 4, 2, 64, 321, True),     # group 2, a list a kv-head
    (torch.bfloat16, 1, 300, 517, 32, 8, 128, 517, False),  # group 4
    (torch.bfloat16, 1, 70, 640, 8, 1, 64, 600, False),    # group 8: 32 rows a workgroup
    (torch.float16, 1, 97, 130, 2, 2, 64, 130, True),
])
def test_edges_vs_oracle(dtype, B, Tq, Tk, Hq, Hkv, D, W, per_head):
    check(*make(dtype, B, Tq, Tk, Hq, Hkv, D, W, per_head, seed=Tq))


@pytest.mark.parametrize("empty_nan", [False, True])
def test_duplicates_and_empty_rows(empty_nan):
    q, k, v, ids, lengths = make(torch.bfloat16, 1, 96, 300, 8, 2, 128, 300, seed=3)
    ids[:, ::5, 1:3] = ids[:, ::5, 3:4]  # counted per occurrence
    check(q, k, v, ids, lengths, empty_nan)


def test_values_that_are_not_finite():
    """A NaN K row and an infinite V row: rows that list the NaN row as the gather reads them,
    every other row untouched by either (the tile's workgroups go to the gather)."""
    q, k, v, ids, lengths = make(torch.bfloat16, 1, 96, 400, 8, 2, 64, 200, seed=4)
    k[0, 130, 0] = float("nan")
    v[0, 390, 1] = float("inf")
    lists = ids.numpy()[0]
    hit = np.array([(lists[t, : int(lengths[0, t])] == 130).any() for t in range(96)])
    got = sweep(q, k, v, ids, lengths)
    dev = [t.to(DEV) for t in (q, k, v, ids, lengths)]
    gathered = _sparse_read(*dev, None, False, splits=1)
    assert hit.any() and torch.equal(got[0, torch.from_numpy(hit)], gathered[0, torch.from_numpy(hit)])
    clean = np.nonzero(~hit & ~np.array([(lists[t, : int(lengths[0, t])] == 390).any() for t in range(96)]))[0]
    want = oracle.sparse_read(q[:, clean].float().numpy(), np.nan_to_num(k.float().numpy()),
                              np.nan_to_num(v.float().numpy(), posinf=0.0), np.where(lists >= 400, -1, lists)[None][:, clean],
                              lengths.numpy()[:, clean])
    assert np.abs(got[:, clean].float().cpu().numpy() - want).max() <= 2.0 ** -8 * np.abs(want).max() + 2.0 ** -11


def test_sparse_lists_and_one_pool():
    """A few keys a row over a long cache (left to the gather), K/V one pool of both rows."""
    check(*make(torch.bfloat16, 2, 80, 5000, 8, 1, 128, 40, seed=5, short=0.2, pool=True))


@pytest.mark.parametrize("Hq,Hkv,per_head", [(4, 1, False), (12, 3, True), (64, 16, False), (8, 8, True)])
@pytest.mark.parametrize("some", [False, True])
def test_rows_left_to_the_gather(Hq, Hkv, per_head, some):
    """Rows that list a key twice, all or a few, with an empty one among them, at kv-head counts that fill the
    gather's lists evenly and not; some: the K of one kv-head not finite, which leaves all its rows."""
    q, k, v, ids, lengths = make(torch.float16, 2, 200, 300, Hq, Hkv, 64, 300, per_head, seed=Hkv)
    ids[..., 0] = ids[..., 2]
    lengths.clamp_(min=3)
    if some:
        ids[:, ::3, ..., 0] = -1
        k[:, 7, 0, 3] = float("inf")
    lengths[0, 5] = 0
    got = sweep(q, k, v, ids, lengths)
    dev = [t.to(DEV) for t in (q, k, v, ids, lengths)]
    want = _sparse_read(*dev, None, False, splits=1)
    torch.cuda.synchronize()
    # the gather is compiled twice (its sums may be contracted differently): a step of the output, and
    # for rows that were swept the weights and scores of both reads
    swept = 2.0 ** -12 * v.abs().max().item() if some else 2.0 ** -20
    if some:
        assert torch.equal(got[:, :, : Hq // Hkv].isnan(), want[:, :, : Hq // Hkv].isnan())
    err, ref = (got.float() - want.float()).abs(), want.float().abs()
    assert (err <= 2 * RTOL[q.dtype] * ref + swept).all(), err.max()


def test_dense_rows_among_thin_ones():
    """One row tile of sixteen lists enough for the sweep: the slab goes to the gather altogether."""
    q, k, v, ids, lengths = make(torch.bfloat16, 1, 1024, 4096, 8, 2, 128, 640, seed=8)
    lengths[:, 64:] = 40
    ids[:, :64, :512] = torch.arange(512, dtype=torch.int32)
    lengths[:, :64] = 512
    got = sweep(q, k, v, ids, lengths)
    want = _sparse_read(*(t.to(DEV) for t in (q, k, v, ids, lengths)), None, False, splits=1)
    torch.cuda.synchronize()
    # as gathered: of 65536 outputs of the dense rows the sweep rounds ~160 otherwise, the same gather
    # compiled again under one
    assert (got[:, :64] != want[:, :64]).sum() <= 20
    err, ref = (got.float() - want.float()).abs(), want.float().abs()
    assert (err <= 2 * RTOL[q.dtype] * ref + 2.0 ** -20).all(), err.max()
    dense = sweep(q[:, :64], k, v, ids[:, :64], lengths[:, :64])
    torch.cuda.synchronize()
    assert (dense != want[:, :64]).sum() > 20  # alone they are swept


def test_rows_left_to_the_gather_fill_the_chip():
    """1024 rows that all list a key twice cost about what the gather costs (measured 1.1 times it; twelve
    times when a workgroup read the units of four rows by itself)."""
    q, k, v, ids, lengths = make(torch.bfloat16, 1, 1024, 1024, 32, 8, 128, 1024, seed=9)
    ids[:, :, 0] = ids[:, :, 2]
    lengths.fill_(1024)
    dev = [t.to(DEV) for t in (q, k, v, ids, lengths)]
    nbytes = _abi.size("lsa_read_rows_scratch_bytes", _abi.LSA_BF16, 1, 1024, 1024, 32, 8, 128, 1024, 0)
    ws, out = torch.empty(nbytes, dtype=torch.uint8, device=DEV), torch.empty_like(dev[0])

    def rows():
        _abi.call("lsa_read_rows", *(t.data_ptr() for t in dev[:3]), _abi.LSA_BF16, 1, 1024, 1024, 32, 8, 128,
                  *dev[1].stride()[:3], dev[3].data_ptr(), dev[4].data_ptr(), 1024, 0, 128 ** -0.5, 0, ws.data_ptr(),
                  nbytes, out.data_ptr(), _abi.stream(out.device))

    def best(fn):
        times = []
        for _ in range(8):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            fn()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    gather = best(lambda: _sparse_read(*dev, None, False, splits=1))
    assert best(rows) < 3 * gather


def test_large_scores():
    """Scores of a wide spread: the running maximum moves in steps, weights of 2^-100 beside 1."""
    q, k, v, ids, lengths = make(torch.float16, 1, 64, 500, 4, 1, 128, 500, seed=6)
    check(q * 6, k * 4, v, ids, lengths)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
def test_a_swept_row_does_not_depend_on_its_neighbours(dtype, D):
    """The same rows beside others whose scores are 30 times as large and whose lists are other
    keys: bit for bit the same."""
    q, k, v, ids, lengths = make(dtype, 1, 64, 1024, 8, 2, D, 1024, seed=11)
    ids[:] = torch.stack([torch.randperm(1024, generator=torch.Generator().manual_seed(t)) for t in range(64)])
    lengths[:] = 700
    alone = sweep(q, k, v, ids, lengths)
    q[:, 1::2] *= 30
    ids[:, 1::2] = ids[:, 1::2].flip(-1)
    other = sweep(q, k, v, ids, lengths)
    torch.cuda.synchronize()
    assert torch.equal(alone[:, ::2], other[:, ::2])
    assert not torch.equal(alone[:, 1::2], other[:, 1::2])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [4611, 40000])
def test_small_weights_beside_a_large_one(dtype, n):
    """A row of one key of weight 1 (V 0) and n of weight 2^-x (V 1): what is read is the small
    ones' share, about n 2^-x.

    Bound: the output's rounding (its smallest step in fp16 2^-24); 2^-9 of the share for bf16's
    split weights, the exponent's rounding (x 2^-24 of it) and fp32 sums of n / 8 terms; and in
    fp16 2^-37 a weight."""
    D, half = 64, dtype == torch.float16
    q = torch.zeros(1, 64, 4, D, dtype=dtype)
    q[..., 0] = 1
    k = torch.zeros(1, n + 1, 1, D, dtype=dtype)
    v = torch.ones(1, n + 1, 1, D, dtype=dtype)
    v[0, 0] = 0
    ids = torch.arange(n + 1, dtype=torch.int32).expand(1, 64, n + 1).contiguous()
    lengths = torch.full((1, 64), n + 1, dtype=torch.int32)
    scale = float(np.float32(np.log(2.0)))
    for x in (8, 16, 20, 23.5, 24.5, 25.25, 27.25, 30.25, 33, 36):
        k[0, :, 0, 0], k[0, 0, 0, 0] = -x / 2, x / 2  # exact in both types
        w = np.exp(-x * scale)
        want = n * w / (1 + n * w)
        got = sweep(q, k, v, ids, lengths, scale=scale).double().cpu().numpy()
        bound = (RTOL[dtype] + 2.0 ** -9) * want + (n * 2.0 ** -37 + 2.0 ** -25 if half else 0.0)
        err = np.abs(got - want).max()
        assert err <= bound, (x, got.flat[0], want, err, bound)


def test_segments_and_slabs():
    """A 262144-row cache (eight bitmap segments, a slab of 64 row tiles) under 2080 rows: both
    slabs' rows against the oracle, keys of every segment."""
    B, Tq, Tk, Hq, Hkv, D, W = 1, 2080, 262144, 8, 1, 64, 200
    g = torch.Generator().manual_seed(7)
    q = torch.randn(B, Tq, Hq, D, generator=g).half()
    k, v = (torch.randn(B, Tk, Hkv, D, generator=g).half() for _ in range(2))
    # dense at the end (dense enough for the sweep), a key in every segment
    pick = torch.stack([torch.randperm(512, generator=g)[:192] for _ in range(Tq)])
    ids = torch.cat([pick + (Tk - 512), torch.arange(8).expand(Tq, 8) * 32768 + 5], 1).int()[None]
    lengths = torch.full((B, Tq), W, dtype=torch.int32)
    rows = [0, 31, 32, 1000, 2047, 2048, 2079]
    check(q, k, v, ids, lengths, rows=rows)


def _views(kind, B, Tk, Hkv, D, dtype, g):
    """K and V as a program may hold them: strides of a longer cache, of heads before tokens, of a
    fused projection's rows, of one pool."""
    draw = lambda *shape: torch.randn(*shape, device=DEV, generator=g).to(dtype)
    if kind == "longer":  # the first Tk rows of a cache
        return draw(B, Tk + 300, Hkv, D)[:, :Tk], draw(B, Tk + 300, Hkv, D)[:, :Tk]
    if kind == "heads first":
        return draw(B, Hkv, Tk, D).transpose(1, 2), draw(B, Hkv, Tk, D).transpose(1, 2)
    if kind == "fused":  # q, k and v of a token side by side
        rows = draw(B, Tk, 6 * Hkv, D)
        return rows[:, :, 4 * Hkv:5 * Hkv], rows[:, :, 5 * Hkv:]
    assert kind == "pool"
    return draw(1, Tk, Hkv, D), draw(1, Tk, Hkv, D)


@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("kind,dtype", [("longer", torch.bfloat16), ("heads first", torch.float16),
                                        ("fused", torch.bfloat16), ("pool", torch.float16)])
def test_public_reads_of_cache_views(monkeypatch, kind, dtype, per_head):
    """``lsa_read`` over views of a cache: read in place by the sweep, against the gather."""
    B, Tq, Tk, Hq, Hkv, D, W = 2, 768, 1000, 32, 8, 128, 1000
    g = torch.Generator(device=DEV).manual_seed(13)
    q = torch.randn(B, Tq, Hq, D, device=DEV, generator=g).to(dtype)
    k, v = _views(kind, B, Tk, Hkv, D, dtype, g)
    lead = (B, Tq, Hkv) if per_head else (B, Tq)
    ids = torch.rand(*lead, W, device=DEV, generator=g).argsort(-1).to(torch.int32)
    lengths = torch.randint(500, W + 1, lead, device=DEV, generator=g).to(torch.int32)
    called, call = [], _abi.call
    monkeypatch.setattr(_abi, "call", lambda name, *a: (called.append((name, a)), call(name, *a))[1])
    got = pipeline.lsa_read(q, k, v, ids, lengths, D ** -0.5)
    name, args = called[0]
    assert name == "lsa_read_rows" and args[1] == k.data_ptr()  # no copy
    want = _sparse_read(q, k, v, ids, lengths, None, False, splits=1)
    assert called[1][0] == "lsa_read"
    torch.cuda.synchronize()
    err, ref = (got.float() - want.float()).abs(), want.float().abs()
    # the two reads' own rounding, and the weights and scores of both
    assert (err <= 2 * RTOL[dtype] * ref + 2.0 ** -12 * v.abs().max().item()).all(), err.max()


def test_the_widest_token_stride():
    """Tokens 2^24 - 8 elements apart, the widest the sweep takes: 63 rows of a tile are 2 GB."""
    D, Tk, stride = 64, 130, (1 << 24) - 8
    g = torch.Generator(device=DEV).manual_seed(14)
    store = torch.empty((Tk - 1) * stride + 2 * D, device=DEV, dtype=torch.bfloat16)
    k, v = (torch.as_strided(store, (1, Tk, 1, D), (0, stride, D, 1), off) for off in (0, D))
    for t in (k, v):
        t.copy_(torch.randn(1, Tk, 1, D, device=DEV, generator=g))
    q = torch.randn(1, 64, 4, D, device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.rand(1, 64, Tk, device=DEV, generator=g).argsort(-1).to(torch.int32)
    lengths = torch.full((1, 64), Tk, device=DEV, dtype=torch.int32)
    nbytes = _abi.size("lsa_read_rows_scratch_bytes", _abi.LSA_BF16, 1, 64, Tk, 4, 1, D, Tk, 0)
    ws, out = torch.empty(nbytes, dtype=torch.uint8, device=DEV), torch.empty_like(q)
    print(f"rows sweep token stride {stride}", flush=True)
    _abi.call("lsa_read_rows", q.data_ptr(), k.data_ptr(), v.data_ptr(), _abi.LSA_BF16, 1, 64, Tk, 4, 1, D, 0, stride, D,
              ids.data_ptr(), lengths.data_ptr(), Tk, 0, D ** -0.5, 0, ws.data_ptr(), nbytes, out.data_ptr(),
              _abi.stream(out.device))
    dense = sweep(*(t.cpu() for t in (q, k, v, ids, lengths)))
    torch.cuda.synchronize()
    assert torch.equal(out, dense)


def test_the_sweep_in_a_captured_graph():
    """A read that goes to the sweep as a replayed graph, over new queries, lists and caches, some rows
    left to the gather, with eager work between the replays."""
    Tq, Hq, Hkv, D, W = 1024, 32, 8, 128, 1024
    g = torch.Generator(device=DEV).manual_seed(15)
    q, k, v = (torch.randn(1, Tq, h, D, device=DEV, generator=g).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    assert _sweep_pays(q.dtype, 1, Tq, Tq, Hq, Hkv, D, W, k.stride(1), D ** -0.5)
    ids = torch.empty(1, Tq, W, device=DEV, dtype=torch.int32)
    lengths = torch.empty(1, Tq, device=DEV, dtype=torch.int32)

    def inputs():
        for t in (q, k, v):
            t.copy_(torch.randn(t.shape, device=DEV, generator=g))
        ids.copy_(torch.rand(ids.shape, device=DEV, generator=g).argsort(-1))
        ids[:, ::9, 0] = ids[:, ::9, 1]  # for the gather
        lengths.copy_(torch.randint(300, W + 1, lengths.shape, device=DEV, generator=g))

    def step():
        return pipeline.lsa_read(q, k, v, ids, lengths, D ** -0.5)

    inputs()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = step()
    for _ in range(4):
        inputs()
        want = step().clone()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
