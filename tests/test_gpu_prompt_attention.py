"""GPU checks of the prompt chunk's causal attention, q4_prompt_attention_dev
(on the matrix cores with two-term fp16 operands), against the reference's sdpa with causal=True
(hetero/cpu_model.py:233-252) evaluated in float64 here: query row i of a
chunk at positions [pos0, pos0 + rows) sees the cache positions
[0, pos0 + i], query head h reads kv head h / (nh / nkv),
o = softmax((q . k) * scale) v.

The kernel evaluates the softmax online (tile by tile) and sum in fp32, so
the bar is fp32 rounding, not bit equality: normwise relative error (max
|diff| / max |ref|) below ATTN_TOL = 2e-6, stated here.  A planted
mistake -- one position too many or too few, the wrong kv head, a missing
scale -- moves the output by far more (checked on the reference below).
"""
import ctypes

import numpy as np
import pytest

import oracle
from hetero import q4

ATTN_TOL = 2e-6


def sdpa_causal(q, kc, vc, pos0, nh, nkv, scale, extra=0, head_shift=0):
    """float64 reference; `extra` / `head_shift` plant mistakes."""
    rows, d = q.shape[0], kc.shape[2]
    qh = q.reshape(rows, nh, d).astype(np.float64)
    out = np.empty((rows, nh, d))
    g = nh // nkv
    for h in range(nh):
        kvh = (h // g + head_shift) % nkv
        n = pos0 + rows + extra
        k = kc[kvh, :n].astype(np.float64)
        v = vc[kvh, :n].astype(np.float64)
        s = qh[:, h] @ k.T * scale
        mask = np.arange(n)[None, :] <= (pos0 + np.arange(rows) + extra)[:, None]
        s = np.where(mask, s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = (p / p.sum(1, keepdims=True)) @ v
    return out.reshape(rows, nh * d)


# (heads, kv heads, head_dim, rows, pos0, cap): a 512-token Qwen2.5-7B chunk
# (7 heads per kv head, 8 tiles); a chunk after a context; a single row;
# 1 and 8 heads per kv head; head_dim 64 and 32; ragged row
# blocks and tiles throughout
CASES = [(28, 4, 128, 512, 0, 512), (28, 4, 128, 70, 64, 200), (28, 4, 128, 1, 300, 301),
         (8, 8, 128, 33, 100, 140), (16, 2, 128, 40, 5, 45), (4, 2, 128, 24, 0, 24),
         (8, 2, 64, 50, 10, 64), (4, 4, 32, 17, 3, 20)]


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,d,rows,pos0,cap", CASES, ids=lambda v: str(v))
def test_prompt_attention_vs_float64(nh, nkv, d, rows, pos0, cap):
    import torch
    print(f"prompt attention nh={nh} nkv={nkv} d={d} rows={rows} pos0={pos0} cap={cap}", flush=True)
    rng = np.random.default_rng(nh * 1000 + rows + pos0)
    q = rng.normal(0, 2, (rows, nh * d)).astype(np.float32)
    kc = rng.normal(0, 1, (nkv, cap, d)).astype(np.float16)
    vc = rng.normal(0, 1, (nkv, cap, d)).astype(np.float16)
    scale = ctypes.c_float(d ** -0.5).value
    lib = q4.load()
    tq, tk, tv = (torch.from_numpy(a).cuda() for a in (q, kc, vc))
    out = torch.full((rows, nh * d), float("nan"), device="cuda")
    rc = lib.q4_prompt_attention_dev(tq.data_ptr(), tk.data_ptr(), tv.data_ptr(), out.data_ptr(), rows, pos0, nh,
                                     nkv, d, cap, scale, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, q4.last_error(lib)
    got = out.cpu().numpy()
    ref = sdpa_causal(q, kc, vc, pos0, nh, nkv, scale)
    err = oracle.normwise_rel(got, ref)
    print(f"normwise error vs float64: {err:.2e}", flush=True)
    assert np.isfinite(got).all()
    assert err < ATTN_TOL
    again = torch.empty_like(out)
    lib.q4_prompt_attention_dev(tq.data_ptr(), tk.data_ptr(), tv.data_ptr(), again.data_ptr(), rows, pos0, nh, nkv,
                                d, cap, scale, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(out, again)


def test_planted_mistakes_exceed_the_bar():
    """The reference with a mistake planted differs from the true one by far
    more than ATTN_TOL (so the bar above can see such a mistake)."""
    rng = np.random.default_rng(3)
    nh, nkv, d, rows, pos0, cap = 8, 2, 128, 20, 7, 40
    q = rng.normal(0, 2, (rows, nh * d)).astype(np.float32)
    kc = rng.normal(0, 1, (nkv, cap, d)).astype(np.float16)
    vc = rng.normal(0, 1, (nkv, cap, d)).astype(np.float16)
    scale = d ** -0.5
    ref = sdpa_causal(q, kc, vc, pos0, nh, nkv, scale)
    for bad in (sdpa_causal(q, kc, vc, pos0, nh, nkv, scale, extra=1),
                sdpa_causal(q, kc, vc, pos0, nh, nkv, scale, extra=-1),
                sdpa_causal(q, kc, vc, pos0, nh, nkv, scale, head_shift=1),
                sdpa_causal(q, kc, vc, pos0, nh, nkv, 1.0)):
        assert oracle.normwise_rel(bad, ref) > 1e3 * ATTN_TOL


# The tiles of a row block go to 2 or 4 groups of waves and its heads to
# workgroups of 2 or 4: fewer tiles than groups, a last round of some groups
# only, rows that see none of a group's positions, heads that leave a
# workgroup's last waves idle, few and many workgroups; and every form that
# launch_prompt_heads picks by tiles, heads and workgroups per CU (256).  The bar is the one above: the groups' sums are
# merged by one more rescaling, 2 fp32 roundings against the up to 40 of the
# tiles' running ones.
@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,d,rows,pos0", [
    (7, 1, 128, 5, 62), (7, 1, 64, 16, 112), (5, 1, 128, 20, 250), (10, 2, 64, 700, 0), (12, 2, 32, 700, 60),
    (28, 4, 128, 330, 15), (16, 8, 64, 17, 600), (3, 3, 128, 40, 127), (24, 3, 64, 48, 300), (15, 5, 128, 2, 2500),
    (28, 4, 128, 37, 0), (8, 4, 128, 17, 110), (4, 4, 64, 30, 120), (4, 4, 32, 30, 270), (6, 3, 128, 40, 330),
    (5, 5, 64, 17, 500), (8, 8, 64, 520, 0), (16, 8, 128, 520, 0), (8, 8, 128, 530, 800), (8, 8, 32, 540, 1600), (64, 8, 128, 300, 0),
    (64, 8, 64, 512, 100), (9, 3, 32, 700, 0), (15, 3, 64, 600, 0), (8, 1, 128, 16, 0)],
    ids=lambda v: str(v))
def test_prompt_attention_groups_and_heads(nh, nkv, d, rows, pos0):
    import torch
    rng = np.random.default_rng(nh * 100 + rows + pos0)
    cap = pos0 + rows + 3
    q = rng.normal(0, 2, (rows, nh * d)).astype(np.float32)
    kc = rng.normal(0, 1, (nkv, cap, d)).astype(np.float16)
    vc = rng.normal(0, 1, (nkv, cap, d)).astype(np.float16)
    kc[:, pos0 + rows:] = np.nan                              # no row sees these
    vc[:, pos0 + rows:] = np.nan
    scale = ctypes.c_float(d ** -0.5).value
    lib = q4.load()
    tq, tk, tv = (torch.from_numpy(a).cuda() for a in (q, kc, vc))
    out = torch.full((rows + 1, nh * d), -7.0, device="cuda")
    rc = lib.q4_prompt_attention_dev(tq.data_ptr(), tk.data_ptr(), tv.data_ptr(), out.data_ptr(), rows, pos0, nh,
                                     nkv, d, cap, scale, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, q4.last_error(lib)
    got = out.cpu().numpy()
    assert (got[rows] == -7.0).all()
    err = oracle.normwise_rel(got[:rows], sdpa_causal(q, kc, vc, pos0, nh, nkv, scale))
    assert err < ATTN_TOL, err


def _one_head(q, k, v, scale):
    """One query row over every position of one head."""
    import torch
    lib, (n, d) = q4.load(), k.shape
    tq, tk, tv = (torch.from_numpy(a).cuda() for a in (q, k, v))
    out = torch.zeros((1, d), device="cuda")
    rc = lib.q4_prompt_attention_dev(tq.data_ptr(), tk.data_ptr(), tv.data_ptr(), out.data_ptr(), 1, n - 1, 1, 1, d,
                                     n, scale, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, q4.last_error(lib)
    return out.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 128])
def test_prompt_attention_scores_of_minus_infinity(d):
    """Scores of -inf over a whole tile leave the others' softmax alone; a row
    whose every score is -inf is 0 / 0."""
    n = 400
    q = np.full((1, d), 1e38, np.float32)
    k = np.full((n, d), -1.0, np.float16)                     # q . k = -1e38 d: -inf in fp32
    v = np.random.default_rng(d).normal(0, 1, (n, d)).astype(np.float16)
    assert np.isnan(_one_head(q, k, v, 1.0)).all()
    for seen in (3, 70, 399):
        k1 = k.copy()
        k1[seen] = 0.0
        np.testing.assert_array_equal(_one_head(q, k1, v, 1.0)[0], v[seen].astype(np.float32))
    q[0, 5] = np.inf
    assert np.isnan(_one_head(q, k, v, 1.0)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 128])
def test_prompt_attention_queries_past_fp16(d):
    """Queries beyond fp16's range: scores of q = 2^17 and k of about 2^-14,
    |s| up to 16, each to 2^-21 of its value (the two-term operands), so
    probabilities to 16 x 2^-21 besides the fp32 rounding of ATTN_TOL."""
    rng = np.random.default_rng(d)
    n = 300
    q = np.zeros((1, d), np.float32)
    q[0, 3] = 2.0 ** 17
    k = np.zeros((n, d), np.float16)
    k[:, 3] = rng.choice([-1, 1], n) * (1 + rng.random(n)) * 2.0 ** -14
    v = rng.normal(0, 1, (n, d)).astype(np.float16)
    ref = sdpa_causal(q, k[None], v[None], n - 1, 1, 1, 1.0)
    assert oracle.normwise_rel(_one_head(q, k, v, 1.0), ref) < ATTN_TOL + 2 * 16 * 2.0 ** -21


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,d,rows", [(1, 1, 32, 1), (1, 1, 64, 1), (1, 1, 128, 1), (7, 1, 64, 20),
                                           (32, 8, 32, 280), (32, 8, 64, 280), (32, 8, 128, 280)],
                         ids=lambda v: str(v))
def test_prompt_attention_one_dominant_key(nh, nkv, d, rows):
    """One key far above the others whose value is 0, so that the output is
    made of the others' small probabilities, 10 to 19 nats below (positive
    values: nothing averages out).  Scores of one product each, to 2^-22 (q's
    two terms) + 2^-23 (fp32) of their value, one sign in a row, so
    probabilities to that times the largest score, besides ATTN_TOL."""
    rng = np.random.default_rng(d + rows)
    pos0, worst = 4000, 0.0
    for nats in (10.0, 14.0, 18.0):
        q = np.zeros((rows, nh * d), np.float32)
        q.reshape(rows, nh, d)[:, :, 3] = 1.0
        kc = np.zeros((nkv, pos0 + rows, d), np.float16)
        kc[:, :, 3] = -nats * (1 + rng.random(kc.shape[:2]) / 16)
        vc = rng.uniform(0.5, 1.5, kc.shape).astype(np.float16)
        kc[:, 1000] = vc[:, 1000] = 0.0
        import torch
        lib = q4.load()
        tq, tk, tv = (torch.from_numpy(a).cuda() for a in (q, kc, vc))
        out = torch.zeros((rows, nh * d), device="cuda")
        rc = lib.q4_prompt_attention_dev(tq.data_ptr(), tk.data_ptr(), tv.data_ptr(), out.data_ptr(), rows, pos0, nh,
                                         nkv, d, pos0 + rows, 1.0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, q4.last_error(lib)
        err = oracle.normwise_rel(out.cpu().numpy(), sdpa_causal(q, kc, vc, pos0, nh, nkv, 1.0))
        print(f"{nats} nats: {err:.2e}", flush=True)
        worst = max(worst, err)
    assert worst < ATTN_TOL + 18 * 17 / 16 * (2.0 ** -22 + 2.0 ** -23)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 128])
def test_prompt_attention_small_queries_large_keys(d):
    """Queries below fp16's range against keys near its end."""
    rng = np.random.default_rng(d)
    q = (rng.normal(0, 1, (1, d)) * 2.0 ** -17).astype(np.float32)
    k = (rng.uniform(-1, 1, (300, d)) * 2.0 ** 15).astype(np.float16)
    v = rng.normal(0, 1, (300, d)).astype(np.float16)
    assert oracle.normwise_rel(_one_head(q, k, v, 1.0), sdpa_causal(q, k[None], v[None], 299, 1, 1, 1.0)) < ATTN_TOL


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 128])
def test_prompt_attention_infinite_keys(d):
    """A key of -inf times the query's sign (an overflow of the cache) has a
    score of -inf and is left out, whatever bits the query has there (1.5 is
    exact in one fp16 value)."""
    rng = np.random.default_rng(d)
    n, scale = 200, ctypes.c_float(np.log(2)).value          # times log2(e): the kernel's q is this one
    for value in (1.5, -1.25, 2.0 ** -13):
        q = rng.normal(0, 1, (1, d)).astype(np.float32)
        q[0, 5] = value
        k = rng.normal(0, 1, (n, d)).astype(np.float16)
        k[77, 5] = -np.inf * value
        v = rng.normal(0, 1, (n, d)).astype(np.float16)
        got = _one_head(q, k, v, scale)
        assert oracle.normwise_rel(got, sdpa_causal(q, k[None], v[None], n - 1, 1, 1, scale)) < ATTN_TOL


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nkv,d,rows", [(8, 4, 128, 6), (7, 1, 64, 40), (1, 1, 32, 300), (32, 8, 128, 300)])
def test_prompt_attention_one_visible_key(nh, nkv, d, rows):
    """The first row of an empty cache sees one key: its output is that key's
    value, exactly, and so its bf16 rounding (an eighth of the fp16 values are
    ties between two bf16 ones)."""
    import torch
    rng = np.random.default_rng(d + rows)
    lib, scale = q4.load(), ctypes.c_float(d ** -0.5).value
    tq = torch.from_numpy((2 * rng.normal(0, 1, (rows, nh * d))).astype(np.float32)).cuda()
    tk, tv = (torch.from_numpy(rng.normal(0, 1, (nkv, rows, d)).astype(np.float16)).cuda() for _ in range(2))
    want = tv[:, 0].float().repeat_interleave(nh // nkv, dim=0).reshape(-1)
    for fn, dt in ((lib.q4_prompt_attention_dev, torch.float32), (lib.q4_prompt_attention_bf16_dev, torch.bfloat16)):
        out = torch.zeros((rows, nh * d), dtype=dt, device="cuda")
        rc = fn(tq.data_ptr(), tk.data_ptr(), tv.data_ptr(), out.data_ptr(), rows, 0, nh, nkv, d, rows, scale,
                torch.cuda.current_stream().cuda_stream)
        assert rc == 0, q4.last_error(lib)
        assert torch.equal(out[0], want.to(dt)), dt


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 128])
def test_prompt_attention_one_overwhelming_key(d):
    """A key 400 nats above all others (scores that are no whole numbers): its
    value, exactly in the first tile, elsewhere to four fp32 roundings of p, o,
    l and their quotient and p's two terms (2^-23)."""
    rng = np.random.default_rng(d)
    n = 400
    q = rng.normal(0, 1, (1, d)).astype(np.float32)
    q[0, 3] = 37.3
    v = rng.normal(0, 1, (n, d)).astype(np.float16)
    for best in (0, 3, 63, 70, 200, 399):
        k = rng.normal(0, 0.1, (n, d)).astype(np.float16)
        k[best, 3] = 13.7
        got, want = _one_head(q, k, v, 1.0)[0].astype(np.float64), v[best].astype(np.float64)
        assert (np.abs(got - want) <= (0.0 if best < 64 else 6 * 2.0 ** -24) * np.abs(want)).all(), best


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 128])
def test_prompt_attention_scores_far_apart(d):
    """Scores of up to 2^30, every two at least 2^18 apart: the output is the
    value of the largest, whichever tile and group it is in, exactly."""
    rng = np.random.default_rng(d)
    n = 400
    q = np.zeros((1, d), np.float32)
    q[0, 3] = 2.0 ** 14
    v = rng.normal(0, 1, (n, d)).astype(np.float16)
    for sign in (1, -1):
        for best in (3, 70, 399):
            k = np.zeros((n, d), np.float16)
            k[:, 3] = sign * 32768.0 - 16.0 * (2 + rng.permutation(n))
            k[best, 3] = sign * 32768.0 - 16.0
            np.testing.assert_array_equal(_one_head(q, k, v, 1.0)[0], v[best].astype(np.float32))
