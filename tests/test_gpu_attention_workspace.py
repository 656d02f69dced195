"""The isolated attention keeps one device block and one pinned block per pool:
calls that grow, fit in and exceed what is kept give the same bits, on two pools
of one session in turn.  The reference of each lane is the same lane in a call
of its own through the allocation-free entry."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from rstr import configs, hip


@pytest.mark.gpu
def test_calls_of_any_size_share_the_kept_blocks():
    print("case attention workspace", flush=True)
    cfg = dict(configs.TINY_QWEN, n_layers=1, n_q=8, n_kv=1, head_dim=128, vocab=512)
    ps, pages = 16, 256
    rng = np.random.default_rng(2)
    # (lanes, split): 41 lanes of 4096 tokens at split 4 have 41984 partials, 177 MB
    calls = [(3, 64), (41, 256), (2, 256), (41, 4), (7, 32)]
    with hip.Session(0) as s:
        m = hip.Model(s, cfg, seed=1)
        pools = [hip.Pool(m, ps, pages) for _ in range(2)]
        for i, p in enumerate(pools):
            p.fill_synthetic(np.arange(pages), seed=3 + i)
        for lanes, split in calls:
            q = rng.standard_normal((lanes, 8, 128)).astype(np.float32)
            table = np.stack([rng.permutation(pages) for _ in range(lanes)]).astype(np.int32)
            lengths = rng.integers(0, pages * ps + 1, lanes).astype(np.int32)
            lengths[0] = pages * ps
            for p in pools:
                got = p.attention(0, q, table, lengths, split=split)
                for b in (0, lanes // 2, lanes - 1):
                    want = p.attention(0, q[b:b + 1], table[b:b + 1], lengths[b:b + 1], split=split, static=True)
                    assert np.array_equal(got[b].view(np.uint32), want[0].view(np.uint32)), (lanes, split, b)


@pytest.mark.gpu
def test_large_arrays_go_without_the_staging_block():
    """Page tables on both sides of the 16 MB that are staged, in turn on one pool;
    the entries past a route are not read."""
    print("case attention large arrays", flush=True)
    cfg = dict(configs.TINY_QWEN, n_layers=1, n_q=8, n_kv=1, head_dim=128, vocab=512)
    ps, pages, lanes = 16, 64, 9
    rng = np.random.default_rng(6)
    with hip.Session(0) as s:
        p = hip.Pool(hip.Model(s, cfg, seed=1), ps, pages)
        p.fill_synthetic(np.arange(pages), seed=3)
        q = rng.standard_normal((lanes, 8, 128)).astype(np.float32)
        table = np.stack([rng.permutation(pages) for _ in range(lanes)]).astype(np.int32)
        lengths = rng.integers(1, pages * ps + 1, lanes).astype(np.int32)
        want = p.attention(0, q, table, lengths, split=64, static=True)
        for width in (pages, 600_000, 400_000, pages, 465_000):
            wide = np.full((lanes, width), -1, np.int32)
            wide[:, :pages] = table
            got = p.attention(0, q, wide, lengths, split=64)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), width


@pytest.mark.gpu
def test_a_call_beside_another_takes_its_own_blocks():
    print("case attention beside attention", flush=True)
    cfg = dict(configs.TINY_QWEN, n_layers=1, n_q=8, n_kv=1, head_dim=128, vocab=512)
    ps, pages = 16, 64
    rng = np.random.default_rng(4)
    with hip.Session(0) as s:
        p = hip.Pool(hip.Model(s, cfg, seed=1), ps, pages)
        p.fill_synthetic(np.arange(pages), seed=3)
        args = []
        for lanes in (5, 9):
            q = rng.standard_normal((lanes, 8, 128)).astype(np.float32)
            table = np.stack([rng.permutation(pages) for _ in range(lanes)]).astype(np.int32)
            args.append((q, table, rng.integers(1, pages * ps + 1, lanes).astype(np.int32)))
        want = [p.attention(0, *a, split=64, static=True) for a in args]
        with ThreadPoolExecutor(2) as threads:
            calls = [(i, threads.submit(p.attention, 0, *args[i], split=64)) for _ in range(20) for i in (0, 1)]
            for i, c in calls:
                assert np.array_equal(c.result().view(np.uint32), want[i].view(np.uint32)), i
