"""Decoders whose routes fit one attention split: one item a lane and kv head, at
the longest route the decoder takes too, against the oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from rstr import configs, hip


# (head dim, q heads, kv heads, window, lanes, split, maxpos): 130 lanes of 8 kv heads are one round more
# than the workgroups that fit, the last one's head dim has no few-item kernel
@pytest.mark.gpu
@pytest.mark.parametrize("hd,n_q,n_kv,window,lanes,split,maxpos", [
    (128, 16, 8, 0, 130, 64, 64), (256, 4, 1, 20, 33, 32, 32), (128, 8, 2, 24, 5, 64, 60), (64, 8, 2, 0, 9, 32, 32)])
def test_routes_of_one_split_match_the_oracle(hd, n_q, n_kv, window, lanes, split, maxpos):
    print("case single split", hd, n_q, n_kv, window, lanes, split, maxpos, flush=True)
    cfg = dict(configs.TINY_QWEN, n_layers=2, d_model=256, d_ff=256, vocab=512, head_dim=hd, n_q=n_q, n_kv=n_kv,
               attn_scale=hd ** -0.5, sliding_window=window, global_pattern=2 if window else 0)
    ps, pps = 16, split // 16 + 2
    rng = np.random.default_rng(lanes)
    lengths = rng.integers(1, maxpos + 1, lanes).astype(np.int32)
    lengths[0], lengths[1], lengths[2] = maxpos, 0, 1
    pages = lanes * pps
    table = rng.permutation(pages).astype(np.int32).reshape(lanes, pps)
    last = np.maximum(lengths - 1, 0)
    slots = np.where(lengths > 0, table[np.arange(lanes), last // ps] * ps + last % ps, -1).astype(np.int32)
    desc = dict(slots=slots, row_offsets=np.arange(lanes + 1, dtype=np.int32), positions=last.astype(np.int32),
                page_table=table, lengths=lengths, start_positions=np.zeros(lanes, np.int32))
    tokens = rng.integers(0, cfg["vocab"], lanes).astype(np.int32)
    om = O.Model(cfg, seed=5)
    od = O.Decoder(om, lanes, ps, pages, pps, maxpos, kv_f16=True, split=split)
    with hip.Session(0) as s:
        m = hip.Model(s, cfg, seed=5)
        p = hip.Pool(m, ps, pages)
        d = hip.Decoder(m, p, lanes, pps, maxpos, split)
        p.fill_synthetic(np.arange(pages), seed=9)
        for page in range(pages):
            od.fill_synthetic(page, 9)
        od.prime_lanes(np.arange(lanes), tokens)
        want = od.step_lanes(**desc)
        active = lengths > 0
        for graph in (True, True, False):  # captured, replayed, launched one by one
            d.set_graph(graph)
            d.prime_lanes(np.arange(lanes), tokens)
            got = d.step_lanes(**desc)
            assert np.array_equal(got[active], want[active])
            assert np.array_equal(d.logits()[active].view(np.uint32), od.logits()[active].view(np.uint32))
    od.close()
    om.close()
