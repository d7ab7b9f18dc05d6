"""GPU checks of the prefill contraction q4_gemm_bf16_dev (bf16 MFMA GEMM with
the group-64 dequantisation fused into the weight-tile load).

Two references:
  * exact-operand: x and the dequantised weights rounded to bf16 (round to
    nearest even, the rule of q4_dequant_bf16_dev) and multiplied in fp64 --
    the kernel may differ only by its fp32 accumulation order (tolerance
    1e-5 norm-wise, stated here);
  * the reference's own contraction, fp32 dequant-matmul
    (hetero/cpu_model.py:119-136), computed here in fp64: the bf16 rounding
    of both operands sets the error; the maximum relative error is reported
    and bounded at 1e-2 norm-wise.
"""
import numpy as np
import pytest

from hetero import q4, synth
import oracle

pytestmark = pytest.mark.gpu

EXACT_OPERAND_TOL = 1e-5
BF16_TOL = 1e-2


def bf16_round(a):
    b = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    b = (b + 0x7FFF + ((b >> 16) & 1)) & 0xFFFF0000
    return b.astype(np.uint32).view(np.float32)


# Shapes that take each tile height and split: (37, 200, 512) and
# (130, 96, 1024) partial 128-row and 256-column tiles; (512, 3584, 3584) and
# (512, 512, 3584) split along K; (500, 16600, 1024) a partial last tile of
# both kinds; (512, 18944, 3584) gate/up of a 512-token prompt unsplit;
# (512, 3584, 18944) and (64, 3584, 18944) down_proj, split along K
@pytest.mark.parametrize("m,n_out,n_in", [(37, 200, 512), (130, 96, 1024), (512, 3584, 3584),
                                          (512, 512, 3584), (64, 3584, 18944), (500, 16600, 1024),
                                          (512, 18944, 3584), (512, 3584, 18944)])
def test_gemm_bf16(m, n_out, n_in):
    import torch
    print(f"gemm m={m} n={n_out} k={n_in}", flush=True)
    w, s, b = synth.qlinear(700 + n_out, n_out, n_in, 64)
    x = synth.activations(701, m, n_in)
    tw, ts, tb, tx = (torch.from_numpy(a).cuda() for a in (w, s.view(np.int16), b.view(np.int16), x))
    got = q4.gemm_bf16_dev(tw, ts, tb, tx)
    torch.cuda.synchronize()
    got = got.cpu().numpy()
    wd = oracle.dequant_np(w, s, b, 64)
    exact = bf16_round(x).astype(np.float64) @ bf16_round(wd).astype(np.float64).T
    assert oracle.normwise_rel(got, exact) < EXACT_OPERAND_TOL
    ref = x.astype(np.float64) @ wd.astype(np.float64).T
    rel = oracle.normwise_rel(got, ref)
    print(f"max relative error vs fp32 dequant-matmul: {rel:.3e}")
    assert rel < BF16_TOL


def test_gemm_bf16_dequant_matches_bf16_dequant_kernel():
    """The weights the GEMM multiplies are exactly q4_dequant_bf16_dev's: with x
    a one-hot row selector the product returns dequantised columns."""
    import torch
    n_out, n_in = 64, 512
    w, s, b = synth.qlinear(710, n_out, n_in, 64)
    x = np.zeros((n_in, n_in), np.float32)
    x[np.arange(n_in), np.arange(n_in)] = 1.0
    tw, ts, tb, tx = (torch.from_numpy(a).cuda() for a in (w, s.view(np.int16), b.view(np.int16), x))
    got = q4.gemm_bf16_dev(tw, ts, tb, tx)             # [n_in, n_out] = W^T in bf16
    deq = q4.dequant_dev(tw, ts, tb, bf16=True).float()
    torch.cuda.synchronize()
    assert torch.equal(got.t().contiguous(), deq)


def _plan(monkeypatch, plan):
    if plan is None:
        monkeypatch.delenv("Q4_GEMM_PLAN", raising=False)
    else:
        monkeypatch.setenv("Q4_GEMM_PLAN", plan)


def _operands(seed, m, n_out, n_in):
    import torch
    w, s, b = synth.qlinear(seed, n_out, n_in, 64)
    x = synth.activations(seed + 1, m, n_in)
    dev = [torch.from_numpy(a).cuda() for a in (w, s.view(np.int16), b.view(np.int16), x)]
    exact = bf16_round(x).astype(np.float64) @ bf16_round(oracle.dequant_np(w, s, b, 64)).astype(np.float64).T
    return dev, exact


@pytest.mark.parametrize("m,n_out,n_in,splits", [(190, 8768, 3392, 5), (434, 8768, 3392, 3), (512, 8768, 3392, 3),
                                                 (512, 3584, 3584, 4)])
def test_gemm_bf16_default_plan(monkeypatch, m, n_out, n_in, splits):
    """The splits the call itself takes, told by the order of its sums: with
    an odd group count (53; scales copied a group at a time) a few splits of
    high tiles, as two 64-row workgroups to a CU took twice as long."""
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("plans of 256 CUs")
    print(f"default plan m={m} n={n_out} k={n_in}", flush=True)
    (tw, ts, tb, tx), _ = _operands(705, m, n_out, n_in)
    got = {}
    for s in (None, *range(1, 7)):
        _plan(monkeypatch, s and f"rows:192:{s}")
        got[s] = q4.gemm_bf16_dev(tw, ts, tb, tx)
    torch.cuda.synchronize()
    assert [s for s in range(1, 7) if torch.equal(got[None], got[s])] == [splits]


# Stream-K plans: P workgroups over tiles x G iterations, in 8 XCD groups
# when P is a multiple of 8 and there are at least 8 tiles (one group
# otherwise).  P = tiles gives every workgroup one whole tile (no partials);
# P = tiles + 1 cuts every range across two tiles (a partial and an owner
# segment each); the largest P gives ranges of one or two K steps, so an
# owner adds many partials (up to G - 1 of them).  (300, 600, 1024) and
# (500, 16600, 1024): ragged last tiles in both dimensions; the latter's 130
# tiles split 16/17 over the groups.  (512, 3584, 18944): 37-step ranges in
# 296-step tiles, 8 partials per owner.
@pytest.mark.parametrize("m,n_out,n_in,ps", [(37, 200, 512, (1, 3, 8)),
                                             (300, 600, 1024, (6, 7, 50, 96)),
                                             (512, 3584, 3584, (28, 29, 200, 256)),
                                             (500, 16600, 1024, (136, 256)),
                                             (512, 3584, 18944, (224,)),
                                             (512, 18944, 3584, (148, 256))])
def test_gemm_bf16_stream_k(monkeypatch, m, n_out, n_in, ps):
    import torch
    (tw, ts, tb, tx), exact = _operands(720 + m, m, n_out, n_in)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for p in ps:
        p = min(p, cus)
        print(f"stream-K m={m} n={n_out} k={n_in} P={p}", flush=True)
        _plan(monkeypatch, f"sk:{p}")
        a = q4.gemm_bf16_dev(tw, ts, tb, tx)
        b2 = q4.gemm_bf16_dev(tw, ts, tb, tx)
        torch.cuda.synchronize()
        got = a.cpu().numpy()
        assert np.isfinite(got).all(), "a tile's partials did not arrive"
        assert oracle.normwise_rel(got, exact) < EXACT_OPERAND_TOL
        assert torch.equal(a, b2), "stream-K sums in a fixed order: runs agree bit for bit"
        assert q4.prefill_errors() == 0, "a partial missed its wait"
    _plan(monkeypatch, None)


def test_gemm_bf16_stream_k_graph_replays(monkeypatch):
    """Each launch waits for flags carrying its own epoch, which the launch
    before it advanced, so a captured stream-K launch replays correctly:
    every replay equals the eager result bit for bit, and no partial ever
    misses its wait."""
    import torch
    m, n_out, n_in = 512, 3584, 3584
    (tw, ts, tb, tx), exact = _operands(760, m, n_out, n_in)
    _plan(monkeypatch, "sk:200")
    eager = q4.gemm_bf16_dev(tw, ts, tb, tx)            # workspace sized before capture
    torch.cuda.synchronize()
    out = torch.full_like(eager, float("nan"))
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        q4.gemm_bf16_dev(tw, ts, tb, tx, out=out, stream=s)   # this stream's workspace
        s.synchronize()
        with torch.cuda.graph(g, stream=s):
            q4.gemm_bf16_dev(tw, ts, tb, tx, out=out, stream=s)
    for r in range(4):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {r}"
        q4.gemm_bf16_dev(tw, ts, tb, tx)                # eager work between replays
    assert q4.prefill_errors(stream=s) == 0 and q4.prefill_errors() == 0
    assert oracle.normwise_rel(eager.cpu().numpy(), exact) < EXACT_OPERAND_TOL
    _plan(monkeypatch, None)


@pytest.mark.parametrize("plan", ["sk:0", "sk:100000", "dp:64:1", "dp:256:3", "splitk"])
def test_gemm_bf16_plan_override_rejected(monkeypatch, plan):
    """A plan the shape cannot take is an error, not a silent fallback."""
    import torch
    (tw, ts, tb, tx), _ = _operands(770, 64, 512, 512)   # one tile of G = 8 K steps
    _plan(monkeypatch, plan)
    if plan == "dp:256:3":
        q4.gemm_bf16_dev(tw, ts, tb, tx)                # splits of 3, 3 and 2 steps: valid
        torch.cuda.synchronize()
    else:
        with pytest.raises(RuntimeError, match="Q4_GEMM_PLAN"):
            q4.gemm_bf16_dev(tw, ts, tb, tx)
    _plan(monkeypatch, None)


# Several matrices sharing x in one launch: q/k/v and gate/up of the Qwen
# shapes at M=512, and a ragged set -- 300 rows (a partial block), a matrix
# of no rows and 700 rows -- at M=200, under the default plan and forced
# data-parallel, split-K and stream-K plans.  Each output against its own
# exact-operand product; two runs agree bit for bit.
@pytest.mark.parametrize("m,n_in,n_outs,plans", [
    (512, 3584, (3584, 512, 512), (None, "dp:128:4", "sk:40")),
    (512, 3584, (18944, 18944), (None, "dp:256:1")),
    (200, 1024, (300, 0, 700), (None, "dp:256:3", "sk:8", "sk:5")),
])
def test_gemm_bf16_multi(monkeypatch, m, n_in, n_outs, plans):
    import torch
    mats, exacts = [], []
    x = synth.activations(780 + m, m, n_in)
    xr = bf16_round(x).astype(np.float64)
    for i, n in enumerate(n_outs):
        w, s, b = synth.qlinear(781 + i + n, max(n, 1), n_in, 64)
        w, s, b = w[:n], s[:n], b[:n]
        mats.append(tuple(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (w, s.view(np.int16), b.view(np.int16))))
        exacts.append(xr @ bf16_round(oracle.dequant_np(w, s, b, 64)).astype(np.float64).T if n else None)
    tx = torch.from_numpy(x).cuda()
    for plan in plans:
        print(f"multi m={m} k={n_in} n={n_outs} plan={plan}", flush=True)
        _plan(monkeypatch, plan)
        a = q4.gemm_bf16_multi_dev(mats, tx)
        b2 = q4.gemm_bf16_multi_dev(mats, tx)
        torch.cuda.synchronize()
        for n, got, again, exact in zip(n_outs, a, b2, exacts):
            assert got.shape == (m, n)
            if n == 0:
                continue
            g = got.cpu().numpy()
            assert np.isfinite(g).all()
            assert oracle.normwise_rel(g, exact) < EXACT_OPERAND_TOL, (plan, n)
            assert torch.equal(got, again), (plan, n)
    _plan(monkeypatch, None)


# Group counts that take each way of copying scales and biases (8 groups a
# copy: G a multiple of 8; 2: even; 1: odd, or pointers off a 4-byte
# boundary) and each start of a K range (even, odd, across an 8-group
# boundary) in splits, stream-K ranges and whole tiles; the copies' two-step
# and one-step tails; one row and a ragged last tile.
@pytest.mark.parametrize("groups,plans", [(1, (None,)), (2, (None, "dp:256:2")), (3, ("dp:128:3", "dp:256:1")),
                                          (7, ("dp:128:2", "sk:5")), (8, ("dp:256:2", "dp:128:3", "sk:5")),
                                          (14, ("dp:256:3", "dp:128:2", "sk:9")), (17, ("dp:128:4", "sk:7")),
                                          (24, ("dp:256:5", "dp:128:1", "sk:11"))])
def test_gemm_bf16_group_copies(monkeypatch, groups, plans):
    import torch
    n_out, n_in = 300, 64 * groups
    for m in (1, 70, 257):
        (tw, ts, tb, tx), exact = _operands(900 + groups + m, m, n_out, n_in)
        odd = []
        for t in (ts, tb):                                     # the same values 2 bytes past a 4-byte boundary
            o = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
            o[1:] = t.reshape(-1)
            odd.append(o[1:].reshape(t.shape))
        for plan in plans:
            print(f"group copies G={groups} m={m} plan={plan}", flush=True)
            _plan(monkeypatch, plan)
            got = q4.gemm_bf16_dev(tw, ts, tb, tx)
            one = q4.gemm_bf16_dev(tw, odd[0], odd[1], tx)
            torch.cuda.synchronize()
            assert oracle.normwise_rel(got.cpu().numpy(), exact) < EXACT_OPERAND_TOL
            assert torch.equal(got, one), "the copies' width changed the result"
    _plan(monkeypatch, None)
    assert q4.prefill_errors() == 0


@pytest.mark.parametrize("m", [1, 33, 64, 65, 129, 200, 257])
def test_gemm_bf16_tile_heights(monkeypatch, m):
    """Every tile height and split of it, rows at and past its edges: within
    the bar of the exact-operand product, unsplit sums the same bits whatever
    the height; the paired gate/up tiles the same bits at every height too."""
    import torch
    n_out, n_in = 520, 64 * 9
    (tw, ts, tb, tx), exact = _operands(940 + m, m, n_out, n_in)
    (uw, us, ub, _), _ = _operands(960 + m, m, n_out, n_in)
    first = pair = None
    for bm in (64, 128, 192, 256):
        for split in (1, 2, 9):                                # 9: one K step each
            print(f"tile heights m={m} rows:{bm}:{split}", flush=True)
            _plan(monkeypatch, f"rows:{bm}:{split}")
            got = q4.gemm_bf16_dev(tw, ts, tb, tx)
            torch.cuda.synchronize()
            assert oracle.normwise_rel(got.cpu().numpy(), exact) < EXACT_OPERAND_TOL
            if split == 1:
                first = got if first is None else first
                assert torch.equal(got, first), bm
        monkeypatch.setenv("Q4_PAIR_PLAN", f"rows:{bm}")
        h = q4.gemm_bf16_gate_up_silu_dev((tw, ts, tb), (uw, us, ub), tx.bfloat16())
        torch.cuda.synchronize()
        pair = h if pair is None else pair
        assert torch.equal(h, pair), bm
    _plan(monkeypatch, "rows:256:1")
    monkeypatch.delenv("Q4_PAIR_PLAN")
    g, u = q4.gemm_bf16_multi_dev([(tw, ts, tb), (uw, us, ub)], tx.bfloat16())
    want = torch.nn.functional.silu(g.double()) * u.double()
    torch.cuda.synchronize()
    err = (pair.double() - want).abs() / want.abs().clamp_min(1e-30)
    assert float(err.max()) < 2.0 ** -8                          # one rounding to bf16 of an fp32 expression
    _plan(monkeypatch, None)


@pytest.mark.gpu
@pytest.mark.parametrize("n_out,n_in,warm", [(512, 3584, 300), (3584, 3584, 520), (9000, 1024, 512)])
def test_smaller_calls_under_capture_after_the_largest(n_out, n_in, warm):
    """Plans and their scratch are not monotonic in the rows: after one call of
    the most rows, every smaller one can be captured on the stream, and its
    replays equal the eager result."""
    import torch
    s = torch.cuda.Stream()
    (tw, ts, tb, tx), _ = _operands(911, warm, n_out, n_in)
    eager = [q4.gemm_bf16_dev(tw, ts, tb, tx[:m]) for m in (17, 64, 130, 200, 257)]
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        q4.gemm_bf16_dev(tw, ts, tb, tx, stream=s)
    s.synchronize()
    for e in eager:
        m, out, g = e.shape[0], torch.full_like(e, float("nan")), torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            q4.gemm_bf16_dev(tw, ts, tb, tx[:m], out=out, stream=s)
        for _ in range(2):
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, e), m


@pytest.mark.gpu
def test_partials_reserved_by_the_call():
    """A stream holds the partial sums that its calls can take, not those of
    the largest plan there is: a 17-row call of a small matrix under 2 MiB, and
    five streams not five times 128 MiB."""
    import torch
    n_out, n_in = 512, 3584
    (tw, ts, tb, tx), exact = _operands(977, 17, n_out, n_in)
    q4.gemm_bf16_dev(tw, ts, tb, tx)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(5)]
    outs = [torch.empty((17, n_out), device="cuda") for _ in streams]
    free = torch.cuda.mem_get_info()[0]
    for s, o in zip(streams, outs):
        q4.gemm_bf16_dev(tw, ts, tb, tx, out=o, stream=s)
    torch.cuda.synchronize()
    # a split of 64 rows takes at most 32 planes of 64 x 512 floats, 4 MiB, x and flags less than one more
    assert free - torch.cuda.mem_get_info()[0] <= 5 * (6 << 20)
    for o in outs:
        assert oracle.normwise_rel(o.cpu().numpy(), exact) < EXACT_OPERAND_TOL


@pytest.mark.gpu
@pytest.mark.parametrize("m", [17, 300, 512])
def test_captured_calls_without_room_for_their_plan(monkeypatch, m):
    """A captured call of a shape that the stream has not run (bf16 x: no copy
    of it): the tiling that fits the stream's workspace, the result within the
    bar; the paired gate/up form, which would take stream-K at 512 rows, equal to
    its unsplit form bit for bit."""
    import torch
    n_out, n_in = 18944, 5120
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    mats = []
    for _ in range(2):
        w = torch.randint(-2 ** 31, 2 ** 31, (n_out, n_in // 8), dtype=torch.int64, device="cuda", generator=g)
        s = (torch.randn((n_out, n_in // 64), device="cuda", generator=g) * 0.01).abs().half()
        mats.append((w.to(torch.int32), s, (-7.5 * s.float()).half()))
    x = torch.randn((m, n_in), device="cuda", generator=g).bfloat16()
    small = [t[:64].contiguous() for t in mats[0]]
    want_h = torch.empty((m, n_out), dtype=torch.bfloat16, device="cuda")
    monkeypatch.setenv("Q4_PAIR_PLAN", "dp")
    q4.gemm_bf16_gate_up_silu_dev(*mats, x, h=want_h)
    monkeypatch.delenv("Q4_PAIR_PLAN")
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        q4.gemm_bf16_multi_dev([small], x[:1], stream=stream)      # the stream's first call, a small one
    torch.cuda.synchronize()
    out, h = torch.empty((m, 512), device="cuda"), torch.zeros_like(want_h)
    part = [t[:512].contiguous() for t in mats[0]]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        q4.gemm_bf16_multi_dev([part], x, outs=[out], stream=stream)
        q4.gemm_bf16_gate_up_silu_dev(*mats, x, h=h, stream=stream)
    eager = q4.gemm_bf16_multi_dev([part], x)[0]
    for _ in range(2):
        out.fill_(float("nan"))
        h.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert oracle.normwise_rel(out.cpu().numpy(), eager.cpu().numpy()) < 2 * EXACT_OPERAND_TOL
        assert torch.equal(h, want_h)
    assert q4.prefill_errors() == 0
