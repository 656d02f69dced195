"""Bulk-prefill tiles through the matrix-instruction attention kernel (head dims
128 and 256) against the oracle, which runs the tile's rows as causal lanes with
the decode step's reduction order: every layer's K/V bit for bit, and the final
rows, whose logits through the oracle's own final norm and head have to be the
bits of the logits that its step reports.

Sizes are where the kernel can go wrong: row groups of every GQA width (16/G
rows per workgroup) with a remainder, splits that start and end
inside 16-token chunks, chunks and pages, windows that open inside a split, a
route start other than 0, and infinities in V that some rows of a wave see and
others do not.
"""
import time

import numpy as np
import pytest

import oracle as O
from rstr import configs, hip
from test_prefill import prefill_lane_descriptors

SEED = 4

# (head dim, q heads, kv heads, split, window, page size, rows, rows before the tile, route start)
CASES = [
    (128, 4, 1, 256, 0, 16, 70, 530, 0),
    (128, 4, 2, 64, 0, 16, 33, 0, 0),
    (128, 2, 2, 20, 0, 32, 65, 37, 3),
    (128, 8, 1, 1024, 0, 16, 9, 1100, 0),
    (256, 4, 1, 32, 24, 16, 50, 61, 0),
    (256, 2, 1, 48, 40, 16, 19, 100, 5),
    (256, 2, 2, 512, 0, 64, 17, 700, 0),
    (256, 8, 1, 100, 70, 16, 5, 333, 0),
    (128, 4, 1, 1028, 0, 16, 21, 1900, 0),   # more than the kernel holds: the work-list kernel
    (128, 4, 2, 32, 0, 8, 21, 50, 0),       # chunks that cross pages: the work-list kernel
    (128, 4, 1, 64, 0, 16, 1, 300, 0),      # one row: the work-list kernel
    (256, 4, 1, 32, 24, 16, 1, 61, 2),
    (256, 4, 1, 32, 24, 16, 2, 60, 0),
]


def _tile(cfg, rows, before, start, ps, split, poison=None, pps=None):
    n = before + rows
    pages = -(-n // ps) + 4
    pps = pps or -(-n // ps) + 1
    rng = np.random.default_rng(rows * 1000 + before)
    route = rng.permutation(pages).astype(np.int32)[:-(-n // ps)]
    table = np.full(pps, -1, np.int32)
    table[:route.size] = route
    at = np.arange(before, n)
    slots = (route[at // ps] * ps + at % ps).astype(np.int32)
    tokens = rng.integers(0, cfg["vocab"], rows).astype(np.int32)
    positions = (start + at).astype(np.int32)
    desc = dict(tokens=tokens, slots=slots, positions=positions, page_table=table, start_positions=[start])
    maxpos = start + n + 1
    om = O.Model(cfg, seed=SEED)
    od = O.Decoder(om, rows, ps, pages, pps, maxpos, kv_f16=True, split=split)
    with hip.Session(0) as s:
        m = hip.Model(s, cfg, seed=SEED)
        p = hip.Pool(m, ps, pages)
        pf = hip.Prefill(m, p, rows, pps, maxpos, split)
        for page in route:
            p.fill_synthetic([int(page)], seed=9)
            od.fill_synthetic(int(page), 9)
        for t, value in (poison or {}).items():  # V of a cached token of every layer, one dim each head
            e = (int(route[t // ps]) * ps + t % ps) * cfg["n_kv"] * cfg["head_dim"]
            for layer in range(cfg["n_layers"]):
                v = p.download(1, layer, e, cfg["n_kv"] * cfg["head_dim"]).view(np.float16)
                v[7::cfg["head_dim"]] = value
                p.upload(1, layer, e, v)
                od.slab(1, layer).view(np.float16).reshape(-1)[e:e + v.size] = v
        d = prefill_lane_descriptors(desc, rows)
        od.prime_lanes(d["lanes"], d["tokens"])
        od.step_lanes(**{k: d[k] for k in ("slots", "row_offsets", "positions", "page_table", "lengths",
                                           "start_positions")})
        out = []
        for _ in range(2):  # captured, then replayed
            pf.prefill_range(tokens, slots, positions, table, n, start)
            out.append((pf.rows_out(), [p.pages(k, layer).view(np.uint16).ravel() for layer in range(cfg["n_layers"])
                                        for k in (0, 1)]))
    want = [od.slab(k, layer).view(np.uint16).ravel().copy() for layer in range(cfg["n_layers"]) for k in (0, 1)]
    if poison is None:
        want.append(od.logits().view(np.uint32))
        for rows_out, pages in out:
            assert np.isfinite(rows_out).all()
            h = O.rmsnorm(rows_out, om.norm(-1, "final_norm"), float(cfg["gain_offset"]), cfg["eps"])
            pages.append(O.qlinear(cfg["weight_bits"], *om.tensor(-1, "embed"), *O.quant_act(h)).view(np.uint32))
    od.close()
    om.close()
    return out, want


def _cfg(hd, n_q, n_kv, window):
    return dict(configs.TINY_QWEN, n_layers=3, d_model=256, d_ff=256, vocab=512, head_dim=hd, n_q=n_q, n_kv=n_kv,
                attn_scale=hd ** -0.5, sliding_window=window, global_pattern=2 if window else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("hd,n_q,n_kv,split,window,ps,rows,before,start", CASES)
def test_tiles_match_the_oracle(hd, n_q, n_kv, split, window, ps, rows, before, start):
    print("case tile", hd, n_q, n_kv, split, window, ps, rows, before, start, flush=True)
    out, want = _tile(_cfg(hd, n_q, n_kv, window), rows, before, start, ps, split)
    for _, pages in out:
        for i, (a, b) in enumerate(zip(pages, want, strict=True)):
            assert np.array_equal(a, b), i


# (head dim, q heads, kv heads, split, window, rows, rows before the tile, pages a route may have):
# 2048 (head dim 256: 1024) workgroups a split and a limit of 16384, so a workgroup takes several of the route's
# splits, which begin at 0 or at the window; and a capacity of more splits than a launch has grid planes
@pytest.mark.gpu
@pytest.mark.parametrize("hd,n_q,n_kv,split,window,rows,before,pps", [
    (128, 64, 8, 32, 0, 512, 100, None), (256, 32, 4, 8, 300, 512, 40, None), (128, 4, 2, 4, 0, 9, 30, 16400)])
def test_more_splits_than_the_launch_holds(hd, n_q, n_kv, split, window, rows, before, pps):
    print("case tile splits", hd, n_q, n_kv, split, window, rows, before, pps, flush=True)
    out, want = _tile(_cfg(hd, n_q, n_kv, window), rows, before, 0, 16, split, pps=pps)
    for _, pages in out:
        for i, (a, b) in enumerate(zip(pages, want, strict=True)):
            assert np.array_equal(a, b), i


@pytest.mark.gpu
def test_a_short_route_takes_as_long_in_a_large_decoder():
    """Routes of 256 tokens, one decoder for 2 k and one for 128 k of context:
    with a workgroup for every split of the capacity, the second took several
    times as long."""
    print("case tile capacity", flush=True)
    cfg, ps, rows = _cfg(128, 32, 8, 0), 256, 256
    best = {}
    with hip.Session(0) as s:
        m = hip.Model(s, cfg, seed=SEED)
        p = hip.Pool(m, ps, 4)
        at = np.arange(rows, dtype=np.int32)
        for tokens in (2048, 131072):
            pf = hip.Prefill(m, p, rows, tokens // ps, tokens, 64)
            table = np.full(tokens // ps, -1, np.int32)
            table[0] = 1
            took = []
            for _ in range(12):
                t = time.perf_counter()
                pf.prefill_range(at, ps + at, at, table, rows, 0)
                took.append(time.perf_counter() - t)
            best[tokens] = min(took)
            pf.close()
    assert best[131072] < 2 * best[2048], best


@pytest.mark.gpu
@pytest.mark.parametrize("hd,window", [(128, 0), (128, 24), (256, 24)])
def test_infinite_values_reach_only_the_rows_that_see_them(hd, window):
    """V = inf (and NaN) at cached tokens: with a window, rows of one wave see
    them or not, and the K/V each row appends follows the oracle's."""
    print("case tile infinities", hd, window, flush=True)
    cfg = _cfg(hd, 4, 1, window)
    out, want = _tile(cfg, 40, 45, 0, 16, 32, poison={3: np.inf, 30: np.inf, 41: -np.inf, 44: np.nan})
    for _, pages in out:
        for i, (a, b) in enumerate(zip(pages, want)):
            x, y = a.view(np.float16), b.view(np.float16)
            assert np.array_equal(np.isnan(x), np.isnan(y)), i
            assert np.array_equal(a[~np.isnan(x)], b[~np.isnan(x)]), i


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("d_model,d_ff,n_q,n_kv", [(640, 256, 16, 8), (4096, 512, 4, 2)])
def test_large_tiles_in_two_slices_match_the_oracle(d_model, d_ff, n_q, n_kv, bits):
    """At 449 rows a 4096-wide projection runs in two K slices: the qkv
    projection over K = 640 (quarters of five blocks), or o and down (the last
    layer's through the logits)."""
    print("case two slices", d_model, bits, flush=True)
    cfg = dict(_cfg(128, n_q, n_kv, 0), n_layers=2, d_model=d_model, d_ff=d_ff, weight_bits=bits)
    out, want = _tile(cfg, 449, 20, 0, 16, 256)
    for _, pages in out:
        for i, (a, b) in enumerate(zip(pages, want, strict=True)):
            assert np.array_equal(a, b), i
