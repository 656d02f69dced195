"""Projections whose launches leave CUs idle, against the oracle bit for bit.

- Two to sixteen rows against a long K (weights streamed past resident
  activations): the smallest K it takes and every chunk-group width it has, the
  largest K (20480: 160 KB of LDS) and width (4096 columns), column tiles that do
  and do not fill a workgroup, row counts at both ends, and the shapes next to
  its limits, which other forms serve.
- The LM head in four K slices that the tail adds: vocabularies on both sides of
  the line, where the next token's row and the logits read back come from the
  added slices.
"""
import numpy as np
import pytest

import oracle as O
from rstr import configs, hip

SEED = 6


def _cfg(bits, **kw):
    return configs.with_bits(dict(configs.TINY_QWEN, n_layers=1, **kw), bits)


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("k,n", [(7168, 256), (8192, 128), (9216, 384), (6656, 128), (14336, 128),
                                 (20480, 128), (21504, 128), (7168, 4096), (7168, 4224)])
def test_few_rows_over_a_long_k(bits, k, n):
    print("case long k", bits, k, n, flush=True)
    cfg = _cfg(bits, d_model=n, d_ff=k, vocab=512)
    om = O.Model(cfg, seed=SEED)
    rng = np.random.default_rng(k + n)
    wq, ws = om.tensor(0, "down")
    with hip.Session(0) as s:
        m = hip.Model(s, cfg, seed=SEED)
        for rows in (1, 2, 3, 16, 17):
            x = (rng.standard_normal((rows, k)) * rng.uniform(0.1, 3.0, (rows, 1))).astype(np.float32)
            xq, xs = O.quant_act(x)
            got, want = m.linear(0, "down", xq, xs, 4), O.qlinear(bits, wq, ws, xq, xs)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), rows
    om.close()


def _step_matches(cfg, lanes):
    """Two decode steps of one token over one-token routes: tokens, logits and the next rows."""
    vocab = cfg["vocab"]
    ps, pages, pps, maxpos, split = 16, lanes + 2, 1, 16, 16
    rng = np.random.default_rng(vocab)
    table = rng.permutation(pages).astype(np.int32)[:lanes].reshape(lanes, 1)
    lengths = np.ones(lanes, np.int32)
    desc = dict(slots=table[:, 0] * ps, row_offsets=np.arange(lanes + 1, dtype=np.int32),
                positions=np.zeros(lanes, np.int32), page_table=table, lengths=lengths,
                start_positions=np.zeros(lanes, np.int32))
    tokens = rng.integers(0, vocab, lanes).astype(np.int32)
    om = O.Model(cfg, seed=SEED)
    od = O.Decoder(om, lanes, ps, pages, pps, maxpos, kv_f16=True, split=split)
    od.prime_lanes(np.arange(lanes), tokens)
    want = od.step_lanes(**desc)
    with hip.Session(0) as s:
        m = hip.Model(s, cfg, seed=SEED)
        p = hip.Pool(m, ps, pages)
        dec = hip.Decoder(m, p, lanes, pps, maxpos, split)
        for _ in range(2):
            dec.prime_lanes(np.arange(lanes), tokens)
            got = dec.step_lanes(**desc)
            assert np.array_equal(got, want)
            assert np.array_equal(dec.logits().view(np.uint32), od.logits().view(np.uint32))
            assert np.array_equal(dec.rows().view(np.uint32), od.r0().view(np.uint32))
    od.close()
    om.close()


# two rows over K = 7168: under 2048 columns the down projection computes its own activation
@pytest.mark.gpu
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("d", [256, 2048])
def test_two_lanes_over_a_long_down_projection(bits, d):
    print("case two lanes", bits, d, flush=True)
    _step_matches(_cfg(bits, d_model=d, d_ff=7168, vocab=512), 2)


# rows, vocabulary: one row is the GEMV; three rows of d_model 256 are 128-column
# workgroups (four slices up to 191 of them), of d_model 1024 256-column ones (255);
# 64 rows of d_model 512 stay at one slice from 524 288 logits on, of 2048 from 256
# 64-column workgroups on
@pytest.mark.gpu
@pytest.mark.parametrize("lanes,d,vocab", [(1, 512, 48), (2, 256, 16), (3, 256, 24448), (3, 256, 24464), (3, 256, 32768),
                                           (3, 1024, 65280), (3, 1024, 65296), (2, 512, 1040), (64, 512, 8192),
                                           (64, 512, 8208), (64, 512, 16384), (64, 2048, 16320), (64, 2048, 16336),
                                           (130, 256, 528)])
def test_head_slices(lanes, d, vocab):
    print("case head", lanes, d, vocab, flush=True)
    _step_matches(_cfg(4, d_model=d, d_ff=128, vocab=vocab), lanes)
