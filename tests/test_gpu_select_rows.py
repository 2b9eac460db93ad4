"""The flat select of many rows (scores as fp64 matrix tiles) against the general fused select,
a workgroup a row: lists and lengths bit-exact at tile, slab and exponent-range edges. And the default chain's pick
counts against the chain that packs and lists its keys."""

import pytest
import torch

from lsa_rocm_lab.port import pipeline
from lsa_rocm_lab.port.pipeline import Buckets, PortConfig

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _table(G, rows, D, gen, block_visible, spans=True):
    """Spans of 1 to 8 keys a bucket, a table a group (G 0: one table)."""
    lead = (G,) if G else ()
    sizes = torch.randint(1, 9, (*lead, rows), device=DEV, generator=gen, dtype=torch.int32)
    ends = sizes.cumsum(-1).to(torch.int32).contiguous()
    slot = torch.arange(8, device=DEV, dtype=torch.int32)
    members = torch.where(slot < sizes[..., None], (ends - sizes)[..., None] + slot, -1).to(torch.int32).contiguous()
    c32 = torch.randn(*lead, rows, D, device=DEV, generator=gen)
    return Buckets(c32.to(torch.bfloat16), members, sizes, centroids_f32=c32, ends=ends, spans=spans,
                   block_visible=block_visible)


def _both(monkeypatch, q, pos, table, config):
    got = []
    for tiles in (True, False):
        monkeypatch.setattr(pipeline, "_rows_pay", lambda *a, tiles=tiles: tiles)
        got.append(pipeline._fused_select(q, pos, table, config, config.top_k, "bf16"))
    torch.cuda.synchronize()
    (lists, lengths), (want_lists, want_lengths) = got
    assert torch.equal(lengths, want_lengths)
    assert torch.equal(lists, want_lists)


def _config(top_p, **kw):
    base = dict(cluster_block_size=64, bucket_size=4, bucket_cap=8, top_p=top_p, top_k=256, window_size=12, sink_size=4)
    return PortConfig(**{**base, **kw})


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("R,G,rows,top_p,block_visible,spans,dtype", [
    (1, 0, 1, 4, False, True, torch.float32),
    (16, 0, 16, 4, True, True, torch.bfloat16),
    (17, 2, 15, 8, False, True, torch.float16),
    (257, 1, 517, 32, False, True, torch.float32),
    (300, 3, 1041, 130, True, True, torch.float32),
    (67, 4, 65, 64, False, False, torch.bfloat16),
    (129, 0, 4096, 1024, True, True, torch.float32),
])
def test_rows_select_equals_the_general_select(monkeypatch, D, R, G, rows, top_p, block_visible, spans, dtype):
    print(f"case D={D} R={R} G={G} rows={rows} top_p={top_p} {block_visible} {spans} {dtype}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(R + rows + D)
    table = _table(G, rows, D, gen, block_visible, spans)
    q = torch.randn(*((R, G) if G else (R,)), D, device=DEV, generator=gen).to(dtype)
    # a negative position (nothing visible), block edges, the whole table
    pos = torch.randint(-1, 5 * rows + 64, (R,), device=DEV, generator=gen).to(torch.int32)
    pos[0], pos[-1] = -1, 8 * rows + 64
    _both(monkeypatch, q, pos, table, _config(top_p))


@pytest.mark.parametrize("D", [64, 128])
def test_rows_select_exponents_ties_and_special_values(monkeypatch, D):
    """Exponent ranges on both sides of what fp64 holds exactly, zeros, subnormals, infinities,
    NaN, equal buckets: the lists are the canonical scores' all the same."""
    gen = torch.Generator(device=DEV).manual_seed(D)
    R, rows = 96, 200
    table = _table(0, rows, D, gen, False)
    q = torch.randn(R, D, device=DEV, generator=gen)
    c = table.centroids_f32
    for i in range(40):  # one element 2^-i down: ranges from a few to about 45 bits
        c[i, i] = 1.5 * 2.0 ** -i
        q[i, 3 * i % D] = -1.25 * 2.0 ** -i
    c[40], q[40] = 0.0, 0.0
    c[41] = torch.where(torch.arange(D, device=DEV) % 2 == 0, 1e-40, 3.0)
    c[42, 5], c[43, 6], c[44, 7] = float("inf"), float("-inf"), float("nan")
    q[41, 5], q[42, 6], q[43, 7] = float("inf"), float("-inf"), float("nan")
    q[44] *= 1e-38
    c[45], c[46] = 1e38, -1e38
    c[50:90] = c[49]
    # scores that a rounded sum decides: large terms cancel and leave what small ones add
    c[90:200, 0], c[90:200, 1] = 2.0 ** 60, 2.0 ** 60
    q[50:, 0], q[50:, 1] = 1.0, -1.0
    table.centroids.copy_(c.to(torch.bfloat16))
    pos = torch.full((R,), 8 * rows, device=DEV, dtype=torch.int32)
    for top_p in (16, 100):
        _both(monkeypatch, q, pos, table, _config(top_p))


def test_rows_select_more_rows_than_a_slab(monkeypatch):
    """8213 rows of 4096 buckets: 8192 fit the scores of a slab."""
    gen = torch.Generator(device=DEV).manual_seed(5)
    table = _table(0, 4096, 64, gen, True)
    q = torch.randn(8213, 64, device=DEV, generator=gen)
    pos = torch.arange(8213, device=DEV, dtype=torch.int32) * 3
    _both(monkeypatch, q, pos, table, _config(100))


@pytest.mark.parametrize("G", [0, 3])
@pytest.mark.parametrize("rows,top_p", [(1, 1), (200, 1), (200, 33), (33, 64), (300, 257), (5000, 64), (1200, 4096)])
def test_default_chain_equals_the_listing(monkeypatch, G, rows, top_p):
    print(f"case chain G={G} rows={rows} top_p={top_p}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(rows + top_p)
    table = _table(G, rows, 64, gen, False)
    R = 21
    q = torch.randn(*((R, G) if G else (R,)), 64, device=DEV, generator=gen)
    q[3] = float("nan")
    pos = torch.randint(-1, 5 * rows + 64, (R,), device=DEV, generator=gen).to(torch.int32)
    got = pipeline.flat_select_reference(q, pos, table, _config(top_p))
    monkeypatch.setenv("LSA_SELECT_IMPL", "fused_unpack")
    want = pipeline.flat_select(q, pos, table, _config(top_p))
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_rows_select_and_read_in_a_captured_graph():
    """The many-row select, and a read of its lists (by the gather at this size), as a replayed graph, over
    new inputs, with eager work between."""
    gen = torch.Generator(device=DEV).manual_seed(9)
    R, rows, Hq, Hkv, D = 2048, 300, 8, 2, 64
    table, config = _table(0, rows, D, gen, False), _config(64)
    idx = torch.randn(R, D, device=DEV, generator=gen)
    q, k, v = (torch.randn(1, n, h, D, device=DEV, generator=gen).to(torch.bfloat16)
               for n, h in ((R, Hq), (3000, Hkv), (3000, Hkv)))
    pos = torch.arange(R, device=DEV, dtype=torch.int32)
    assert pipeline._rows_pay(R, 1, rows)

    def step():
        lists, lengths = pipeline._fused_select(idx, pos, table, config, config.top_k, "bf16")
        return pipeline.lsa_read(q, k, v, lists[None], lengths[None], D ** -0.5), lists, lengths

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = step()
    for _ in range(3):
        idx.copy_(torch.randn(R, D, device=DEV, generator=gen))
        q.copy_(torch.randn(1, R, Hq, D, device=DEV, generator=gen))
        want = [t.clone() for t in step()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for got, w in zip(out, want):
            assert torch.equal(got, w)


@pytest.mark.parametrize("G", [0, 2])
@pytest.mark.parametrize("spans", [False, True])
def test_rows_select_of_a_paged_cache(monkeypatch, G, spans):
    """Listed ids through a slot table, every query row by its own table row, some ids past the
    table's width: as the general select maps them."""
    gen = torch.Generator(device=DEV).manual_seed(21 + G)
    R, rows, D = 311, 700, 64
    table = _table(G, rows, D, gen, False, spans)
    q = torch.randn(*((R, G) if G else (R,)), D, device=DEV, generator=gen)
    pos = torch.randint(-1, 5 * rows, (R,), device=DEV, generator=gen).to(torch.int32)
    slots = torch.stack([torch.randperm(4000, device=DEV, generator=gen)[:2500] for _ in range(5)]).to(torch.int32)
    slots[:, ::50] = -1  # pages not there
    which = torch.randint(0, 5, (R,), device=DEV, generator=gen).to(torch.int32)
    config, got, called, call = _config(64), [], [], pipeline._abi.call
    monkeypatch.setattr(pipeline._abi, "call", lambda name, *a: (called.append(name), call(name, *a))[1])
    for tiles in (True, False):
        monkeypatch.setattr(pipeline, "_rows_pay", lambda *a, tiles=tiles: tiles)
        got.append(pipeline._fused_select(q, pos, table, config, config.top_k, "bf16", slots, which))
    torch.cuda.synchronize()
    assert called == ["lsa_select_rows", "lsa_select_flat"]
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
