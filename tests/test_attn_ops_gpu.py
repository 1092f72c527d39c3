"""The single-query attention operators away from the GPT-2 shapes: head dims
that no block of 16 loads divides, lengths on both sides of a block of
positions, caches whose stride or address rules out 16-byte loads, and fused
calls on both sides of one, two and four chunks, in a row, so that the shared
partials hold an earlier call's; against a 64-bit softmax attention."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


def reference(q, kc, vc, T, NH, DH, scale):
    s = (q.astype(np.float64).reshape(NH, DH, 1) * kc.reshape(NH, DH, -1)[:, :, :T]).sum(1) * scale
    p = np.exp(s - s.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    return s, p, np.einsum("ht,thd->hd", p, vc[:T].astype(np.float64).reshape(T, NH, DH)).ravel()


@pytest.mark.parametrize("NH,DH,S,T", [(3, 5, 70, 64), (2, 17, 65, 65), (1, 64, 1024, 1), (5, 80, 257, 257), (4, 130, 1000, 999),
                                       (12, 64, 1024, 1024)])
def test_reference_operators(g2, NH, DH, S, T):
    D = NH * DH
    r = np.random.default_rng(NH * DH + T)
    q, kc, vc = (r.standard_normal(n).astype(np.float32) for n in (D, D * S, S * D))
    scale = float(np.float32(1 / np.sqrt(DH)))
    s, p, o = reference(q, kc, vc.reshape(S, D), T, NH, DH, scale)
    dk, dv, dO = g2.to_device(kc), g2.to_device(vc), g2.to_device(np.full(D + 1, 7.0, np.float32))
    # scores are written with stride S and read by the softmax with stride 1024
    dS = g2.to_device(np.zeros(NH * 1024, np.float32))
    g2.attn_scores_1q(g2.to_device(q), dk, dS, 0, T, D, DH, NH, S, scale)
    got = dS.download(np.float32, NH * S).reshape(NH, S)[:, :T]
    np.testing.assert_allclose(got, s, rtol=1e-5, atol=2e-6 * np.sqrt(DH))
    rows = np.zeros((NH, 1024), np.float32)
    rows[:, :T] = s
    dS = g2.to_device(rows)
    g2.attn_softmax_1q(dS, T, NH)
    got = dS.download(np.float32, NH * 1024).reshape(NH, 1024)
    np.testing.assert_allclose(got[:, :T], p, rtol=2e-5, atol=1e-7)
    assert (got[:, T:] == 0).all()  # nothing past the row
    g2.attn_out_1q(dS, dv, dO, T, D, DH, 0)
    got = dO.download(np.float32, D + 1)
    np.testing.assert_allclose(got[:D], o, rtol=1e-4, atol=2e-5)
    assert got[D] == 7.0


@pytest.mark.parametrize("NH,S,shift", [(1, 1024, 0), (25, 1024, 0), (7, 1023, 0), (12, 1024, 1), (64, 1000, 0)])
def test_fused_lengths_in_a_row(g2, NH, S, shift):
    D = NH * 64
    r = np.random.default_rng(NH + S)
    q, kc, vc = (r.standard_normal(n).astype(np.float32) for n in (D, D * S, S * D))
    pad = np.zeros(shift, np.float32)
    dq, dk, dv = g2.to_device(q), g2.to_device(np.concatenate([pad, kc])), g2.to_device(np.concatenate([pad, vc]))
    for fn in (g2.attn_1q, g2.attn_1q_noalloc):
        for T in (S, 64, 65, 1, 128, 129, 256, 257, 63, S - 1):
            dO = g2.DevBuf(D * 4)
            for _ in range(2):
                fn(dq, dk.offset(4 * shift), dv.offset(4 * shift), dO, 0, T, D, NH, S, 0, 0.125)
            o = reference(q, kc, vc.reshape(S, D), T, NH, 64, 0.125)[2]
            np.testing.assert_allclose(dO.download(np.float32, D), o, rtol=1e-4, atol=2e-5, err_msg=f"T {T}")


@pytest.mark.parametrize("T", [1, 64, 200, 256, 300])
def test_fused_output_in_its_operands(g2, T):
    """An output over the queries (in place, and a head further), over keys
    and over values in use: everything is read before it is written."""
    NH, S = 20, 512
    D = NH * 64
    r = np.random.default_rng(T)
    q, kc, vc = (r.standard_normal(n).astype(np.float32) for n in (2 * D, D * S, S * D))
    o = reference(q[:D], kc, vc.reshape(S, D), T, NH, 64, 0.125)[2]
    for fn in (g2.attn_1q, g2.attn_1q_noalloc):
        for which, at in ((0, 0), (0, 64), (1, 0), (1, 5 * S + 3), (2, 0), (2, (T - 1) * D)):
            bufs = [g2.to_device(x) for x in (q, kc, vc)]
            fn(*bufs, bufs[which], 0, T, D, NH, S, at, 0.125)
            got = bufs[which].download(np.float32, at + D)[at:]
            np.testing.assert_allclose(got, o, rtol=1e-4, atol=2e-5, err_msg=f"operand {which} + {at}")


@pytest.mark.parametrize("D,DH,T", [(64, 64, 300), (64, 16, 1), (50, 25, 1024), (7, 7, 65)])
def test_weighted_sum_over_its_operands(g2, D, DH, T):
    """Up to 64 dims over the scores or the values that they are summed from."""
    NH = D // DH
    r = np.random.default_rng(D + T)
    p, v = r.random((NH, 1024), np.float32), r.standard_normal((T, D)).astype(np.float32)
    ref = np.einsum("ht,thd->hd", p[:, :T].astype(np.float64), v.astype(np.float64).reshape(T, NH, DH)).ravel()
    for which, at in ((0, 0), (0, max(T - D, 0)), (1, 0), (1, (T - 1) * D)):
        bufs = [g2.to_device(p), g2.to_device(v)]
        g2.attn_out_1q(bufs[0], bufs[1], bufs[which], T, D, DH, at)
        got = bufs[which].download(np.float32, at + D)[at:]
        np.testing.assert_allclose(got, ref, rtol=1e-5, atol=2e-5 * np.sqrt(T), err_msg=f"operand {which} + {at}")


def test_weighted_sum_wider_than_a_launch_of_16_dims(g2):
    """2^26 + 20 dims, 64 threads each were 2^32."""
    D = (1 << 26) + 20
    v = (np.arange(D) % 1000).astype(np.float32)
    p = np.zeros((1, 1024), np.float32)
    p[0, 0] = 0.5
    dO = g2.to_device(np.full(D + 1, 7.0, np.float32))
    g2.attn_out_1q(g2.to_device(p), g2.to_device(v), dO, 1, D, D, 0)
    got = dO.download(np.float32, D + 1)
    assert (got[:D] == v / 2).all() and got[D] == 7.0


@pytest.mark.parametrize("E,NH,P", [(128, 2, 1), (96, 6, 64), (160, 2, 65), (30, 2, 257), (256, 4, 1000)])
def test_reference_prefill_attention(g2, E, NH, P):
    """The reference path's prompt attention (all rows in one launch) at head
    dims 64, 16, 80 and 15: every logit of the prompt's last row, and of a
    decode step behind it, within 2e-4 of the oracle's (measured below 1e-5)."""
    cfg = g2.make_config(2, E, NH, vocab_size=512)
    w = g2.synth_weights(cfg, 11, affine=True)
    ids = np.random.default_rng(P).integers(0, cfg.vocab_size, P + 1).astype(np.int32)
    m = g2.Model.from_host(cfg, w, g2.F32, g2.PATH_REFERENCE)
    om = oracle.Model(cfg, w)
    m.prefill(ids[:P])
    np.testing.assert_allclose(m.logits(), om.generate(ids[:P], 1, logit_steps=1)[2][0], rtol=2e-4, atol=2e-4)
    m.decode(int(ids[P]), P)
    np.testing.assert_allclose(m.logits(), om.generate(ids, 1, logit_steps=1)[2][0], rtol=2e-4, atol=2e-4)
    m.free()
