"""The few-row kernels (the SO(2) convolution pair fu_so2_pair_fwd / _bwd, fu_linear_short, and
fu_linear_dgrad_ln_silu_bwd with a pre-split weight) against float64, at the
edges of their 32-row tiles, for every lmax and several widths (K ranges that do not divide evenly
over the waves), and where the fp16 window rule sends a segment to the two-loop products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pair(cuda, M, C, L, ramp=0.0, runs=0):
    """A pair on the GPU; with ramp > 0 the operands' columns carry 2^t and the weights' 2^-t, t
    ramping over [-ramp, ramp] along K: the same products, opposite magnitudes.  runs > 0: t is -runs
    on every other run of 4 columns of the m = 1, 2 operands, and 0 on the others."""
    from ops import gating
    from ops.linear import complex_weight_split, linear_weight_split
    g = torch.Generator().manual_seed(M + 7 * C + L)
    r = lambda *s: torch.randn(*s, generator=g)
    n0, n1, n2 = (L + 1) * C, L * C, (L - 1) * C
    t = lambda K: torch.exp2(torch.round(torch.linspace(-ramp, ramp, K)))
    w = lambda n, k: r(n, k) / k ** 0.5
    X = [r(M, 2 * n0), r(M, 4 * n1), r(M, 4 * n2)]
    W0, b0, V0, c0 = w((2 * L + 1) * C, 2 * n0), r((2 * L + 1) * C) * 0.3, w(n0, n0), r(n0) * 0.3
    R1, I1, R2, I2 = w(n1, 2 * n1), w(n1, 2 * n1), w(n2, 2 * n2), w(n2, 2 * n2)
    S1, T1, S2, T2 = w(n1, n1), w(n1, n1), w(n2, n2), w(n2, n2)
    f0, f1, f2 = t(2 * n0), t(2 * n1), t(2 * n2)
    if runs:
        f1, f2 = (torch.exp2(-runs * (torch.arange(k) // 4 % 2).float()) for k in (2 * n1, 2 * n2))
        # the last pieces of the weights small: rough columns, against which small operands count
        for w_ in (R1, I1, R2, I2):
            w_[:, -16:] *= 2.0 ** -10
    Xs = [X[0] * f0, X[1] * torch.cat([f1, f1]), X[2] * torch.cat([f2, f2])]
    rows = gating.gate_paired_rows(C, L)
    d = lambda a: a.contiguous().to(cuda)
    A0, P1, Q1, P2, Q2 = W0[rows] / f0, R1 / f1, I1 / f1, R2 / f2, I2 / f2
    conv1 = [d(A0), d(b0[rows]), d(A0.t()), d(P1), d(Q1), d(P1.t()), d(-Q1.t()), d(P2), d(Q2), d(P2.t()), d(-Q2.t())]
    conv2 = [d(V0), d(c0), d(V0.t()), d(S1), d(T1), d(S1.t()), d(-T1.t()), d(S2), d(T2), d(S2.t()), d(-T2.t())]
    cw = [conv1[3:5], conv1[5:7], conv1[7:9], conv1[9:11], conv2[3:5], conv2[5:7], conv2[7:9], conv2[9:11]]
    sp = tuple(complex_weight_split(*p) for p in cw) + tuple(
        linear_weight_split(v) for v in (conv1[0], conv1[2], conv2[0], conv2[2]))
    cot = [r(M, n0), r(M, 2 * n1), r(M, 2 * n2)]
    from oracle import ops_ref as R

    def ref_fn(x0, x1, x2):
        y = (x0 @ W0.double().T + b0.double(), x1 @ R.pack_so2(R1.double(), I1.double()).T,
             x2 @ R.pack_so2(R2.double(), I2.double()).T)
        z0, z1, z2 = R.gating(*y, C) if L == 2 else R.gating_lmax(*y, C, L)
        return (z0 @ V0.double().T + c0.double(), z1 @ R.pack_so2(S1.double(), T1.double()).T,
                z2 @ R.pack_so2(S2.double(), T2.double()).T)

    Xd = [x.double().requires_grad_() for x in X]
    ref = ref_fn(*Xd)
    gref = torch.autograd.grad(ref, Xd, [c.double() for c in cot])
    scale = [f0, torch.cat([f1, f1]), torch.cat([f2, f2])]
    gref = [a / s.double() for a, s in zip(gref, scale)]
    return [x.to(cuda) for x in Xs], conv1, conv2, sp, [c.to(cuda) for c in cot], list(ref) + gref


def _run(X, conv1, conv2, C, sp, cot):
    from ops import gating
    Xg = [x.clone().requires_grad_() for x in X]
    z = gating.conv1_gate_conv2(*Xg, conv1, conv2, C, sp)
    return [t.detach() for t in z] + list(torch.autograd.grad(z, Xg, cot))


def _err(got, ref):
    return [((a.double().cpu() - b.detach()).norm() / b.detach().norm()).item() for a, b in zip(got, ref)]


@pytest.mark.parametrize("M,C,L,ramp", [
    (1, 128, 2, 0), (32, 128, 2, 0), (33, 128, 2, 0), (300, 128, 2, 0), (77, 64, 2, 0), (40, 256, 2, 0), (65, 64, 3, 0),
    (100, 128, 3, 0), (150, 64, 4, 0), (95, 128, 4, 0), (70, 128, 2, 4), (70, 128, 2, 12), (70, 64, 4, 12)])
def test_short_pair(cuda, monkeypatch, M, C, L, ramp):
    """Outputs and input gradients, normwise: two products in a row of 22-bit operands and fp32 sums
    (each at most 2^-21 relative, measured 2-4e-7) and no worse than 1.5x the tiled kernels' error;
    twice the same bits."""
    from ops import _lib, gating
    X, conv1, conv2, sp, cot, ref = _pair(cuda, M, C, L, ramp)
    calls = []
    real = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    got = _run(X, conv1, conv2, C, sp, cot)
    assert calls == ["fu_so2_pair_fwd", "fu_so2_pair_bwd"]
    again = _run(X, conv1, conv2, C, sp, cot)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    monkeypatch.setattr(gating, "SHORT_PAIR_MAX_EDGES", 0)
    tiled = _run(X, conv1, conv2, C, sp, cot)
    for e, t in zip(_err(got, ref), _err(tiled, ref)):
        assert e <= 1e-6 and e <= 1.5 * t + 1e-7, (e, t)


@pytest.mark.parametrize("M,C,L", [(70, 128, 2), (33, 64, 3), (40, 64, 4)])
@pytest.mark.parametrize("runs", [12, 20, 24])
def test_short_pair_runs_of_four(cuda, monkeypatch, M, C, L, runs):
    """Operands of the complex products with a run of 4 small elements in every piece of 8, against
    weights as much larger there: those runs are below the fp16 window from 2^-16 on and go to the
    two-loop products, as in the tiled kernels.  Bars of test_short_pair."""
    from ops import gating
    X, conv1, conv2, sp, cot, ref = _pair(cuda, M, C, L, runs=runs)
    got = _run(X, conv1, conv2, C, sp, cot)
    monkeypatch.setattr(gating, "SHORT_PAIR_MAX_EDGES", 0)
    tiled = _run(X, conv1, conv2, C, sp, cot)
    for e, t in zip(_err(got, ref), _err(tiled, ref)):
        assert e <= 1e-6 and e <= 1.5 * t + 1e-7, (e, t)


def test_short_pair_nonfinite_rows_stay_apart(cuda):
    """An infinite and a NaN element make their own rows non-finite and leave the others' bits."""
    X, conv1, conv2, sp, cot, _ = _pair(cuda, 64, 128, 2)
    clean = _run(X, conv1, conv2, 128, sp, cot)
    X[0][3, 40], X[1][50, 7] = float("inf"), float("nan")
    got = _run(X, conv1, conv2, 128, sp, cot)
    ok = torch.ones(64, dtype=torch.bool, device=cuda)
    ok[3] = ok[50] = False
    for a, b in zip(got, clean):
        assert torch.equal(a[ok], b[ok])
    assert not torch.isfinite(got[0][3]).all() and not torch.isfinite(got[1][50]).all()


@pytest.mark.parametrize("M,N,K,ramp", [(1, 64, 640, 0), (33, 64, 640, 0), (200, 192, 16, 0), (65, 64, 48, 0),
                                        (90, 128, 1152, 0), (70, 64, 320, 12)])
def test_linear_short(cuda, M, N, K, ramp):
    """fu_linear_short on K ranges shorter than and not divisible by its four waves, a strided output
    whose other columns keep their contents, and anti-correlated magnitudes (the two-loop products);
    bar as above."""
    from ops import _lib, linear
    g = torch.Generator().manual_seed(M + N + K)
    f = torch.exp2(torch.round(torch.linspace(-ramp, ramp, K)))
    x, W, b = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) / K ** 0.5, torch.randn(N, generator=g)
    ref = x.double() @ W.double().T + b.double()
    xd, Wd, bd = (x * f).to(cuda), (W / f).to(cuda), b.to(cuda)
    W2 = linear.linear_weight_split(Wd)
    buf = torch.full((M, N + 4), 7.0, device=cuda)
    _lib.call("fu_linear_short", xd.data_ptr(), K, W2.data_ptr(), bd.data_ptr(), buf.data_ptr(), N + 4, M, N, K,
              _lib.stream_ptr(cuda))
    tiled = linear.gemm(xd, Wd, bd)
    e, t = _err([buf[:, :N], tiled], [ref, ref])
    assert (buf[:, N:] == 7.0).all() and e <= 1e-6 and e <= 1.5 * t + 1e-7, (e, t)


@pytest.mark.parametrize("K", [64, 96, 640])
@pytest.mark.parametrize("spread", [8, 12, 14])
@pytest.mark.parametrize("seed", range(6))
def test_linear_short_runs_of_four(cuda, K, spread, seed):
    """Operands whose magnitude changes every 4 columns by powers of two up to 2^+-spread, against weights with
    the inverse: a run of the weight below the window next to larger ones in its piece of 8 meets the
    largest operands.  Every row at the tiled kernel's error and at the fp32 instructions'."""
    from ops import _lib, linear
    g = torch.Generator().manual_seed(100 * seed + K)
    t = torch.randint(-spread, spread + 1, (K // 4,), generator=g).repeat_interleave(4)
    x, W = torch.randn(65, K, generator=g) * torch.exp2(t), torch.randn(64, K, generator=g) / torch.exp2(t)
    ref, x, W = x.double() @ W.double().T, x.to(cuda), W.to(cuda)
    W2, y = linear.linear_weight_split(W), torch.empty(65, 64, device=cuda)
    _lib.call("fu_linear_short", x.data_ptr(), K, W2.data_ptr(), None, y.data_ptr(), 64, 65, 64, K, _lib.stream_ptr(cuda))
    with _lib.matmul_mode(_lib.MATMUL_FP32):
        fp32 = linear.gemm(x, W)
    e, f = (((v.double().cpu() - ref).norm(dim=1) / ref.norm(dim=1)).max().item() for v in (y, fp32))
    # 22-bit operands down to 2^-27 of the largest, in fp32 sums: as the window cases of the tiled kernels
    assert e <= 1.5 * f + 2e-7, (e, f)


@pytest.mark.parametrize("M,K", [(49152, 320), (49153, 320)])
def test_few_row_product_on_both_sides_of_its_line(cuda, monkeypatch, M, K):
    """gemm_few_rows at its last row count and past it: the two entry points, each at the bar above."""
    from ops import _lib, linear
    g = torch.Generator(device=cuda).manual_seed(M)
    x, W = torch.randn(M, K, device=cuda, generator=g), torch.randn(64, K, device=cuda, generator=g) / K ** 0.5
    calls, real = [], _lib.call
    W2 = linear.linear_weight_split(W)
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    y = linear.gemm_few_rows(x, W, W2, torch.empty(M, 64, device=cuda))
    assert calls == ["fu_linear_short" if M <= linear.FEW_ROWS_MAX else "fu_linear"]
    ref = x.double() @ W.double().T
    assert ((y.double() - ref).norm() / ref.norm()).item() <= 1e-6


@pytest.mark.parametrize("M,K,group", [(1, 1536, 0), (31, 384, 4), (33, 1536, 2), (500, 3072, 1), (70, 16, 3)])
def test_dgrad_ln_silu_short(cuda, M, K, group):
    """The radial output layer's input gradient with the LayerNorm-SiLU backward of its group, few rows
    and a pre-split weight, against float64 and the tiled kernel (no pre-split weight); the other
    groups' columns keep their contents."""
    from ops import _lib, linear
    G, C = 5, 128
    g = torch.Generator(device=cuda).manual_seed(M + K)
    r = lambda *s: torch.randn(*s, device=cuda, generator=g)
    A, W, x = r(M, K), r(C, K) / K ** 0.5, r(M, G * C)
    gm, bt = r(G * C).abs() + 0.5, r(G * C) * 0.1
    xd = x.double().view(M, G, C)
    mean, var = xd.mean(2), xd.var(2, unbiased=False)
    mu, rs = mean.float().flatten().contiguous(), (var + 1e-5).rsqrt().float().flatten().contiguous()
    W2, s = linear.linear_weight_split(W), slice(group * C, (group + 1) * C)
    outs = []
    for w2 in (W2, None):
        out = torch.full((M, G * C), 7.0, device=cuda)
        _lib.call("fu_linear_dgrad_ln_silu_bwd", A.data_ptr(), K, W.data_ptr(), K, out[:, s].data_ptr(), G * C, M, K,
                  x.data_ptr(), G * C, gm.data_ptr(), bt.data_ptr(), mu.data_ptr(), rs.data_ptr(), G, group,
                  _lib.ptr(w2), _lib.stream_ptr(cuda))
        assert (out[:, :s.start] == 7.0).all() and (out[:, s.stop:] == 7.0).all()
        outs.append(out[:, s])
    v = x[:, s].double().requires_grad_()
    xh = (v - v.mean(1, keepdim=True)) * (v.var(1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
    y = torch.nn.functional.silu(xh * gm[s].double() + bt[s].double())
    (ref,) = torch.autograd.grad(y, v, A.double() @ W.double().T)
    e, t = _err(outs, [ref.cpu()] * 2)
    assert e <= 1e-6 and e <= 1.5 * t + 1e-7, (e, t)


@pytest.mark.parametrize("M,N,K,batch", [(1, 16, 32, 3), (15, 128, 128, 9), (16, 144, 96, 1), (17, 256, 160, 2),
                                         (54, 128, 128, 25), (512, 64, 64, 5), (513, 64, 64, 5), (2049, 128, 384, 1),
                                         (4096, 256, 128, 1), (8200, 128, 32, 1)])
def test_linear_batched_few_rows(cuda, M, N, K, batch):
    """fu_linear_batched on its 16-row tiles and just past them: interleaved batches (row stride over all of
    them), a bias on the first batches only, and a residual that is the output itself, against float64
    and a plain fp32 product of torch; the columns between the batches keep their contents."""
    from ops import _lib
    g = torch.Generator().manual_seed(M + N + K)
    r = lambda *s: torch.randn(*s, generator=g)
    A, W, b, R = r(M, batch, K + 4), r(batch, N, K) / K ** 0.5, r(batch, N), r(M, batch, N + 4)
    nb = min(2, batch)
    bias = torch.cat([b[:nb], torch.zeros(batch - nb, N)])
    x64 = A[..., :K].double()
    ref = torch.stack([x64[:, i] @ W[i].double().T for i in range(batch)], 1) + bias.double() + R[..., :N].double()
    Ad, Wd, bd, Y = (t.to(cuda) for t in (A, W, b, R))
    _lib.call("fu_linear_batched", Ad.data_ptr(), batch * (K + 4), K + 4, Wd.data_ptr(), K, N * K, bd.data_ptr(), N, nb,
              Y.data_ptr(), batch * (N + 4), N + 4, Y.data_ptr(), batch * (N + 4), N + 4, M, N, K, batch,
              _lib.stream_ptr(cuda))
    plain = torch.stack([A[:, i, :K] @ W[i].T for i in range(batch)], 1) + bias + R[..., :N]
    e, t = _err([Y[..., :N], plain], [ref, ref])
    # fp32 products in sums of K / 4 terms, or 22-bit operands past the rule
    assert e <= 1e-6 and e <= 2.0 * t + 1e-7, (e, t)
    assert torch.equal(Y[..., N:].cpu(), R[..., N:])


@pytest.mark.parametrize("M,N,K,mode", [(54, 128, 128, "split_f16"), (8200, 128, 64, "split_f16"), (8200, 200, 36, "split_f16"),
                                        (8200, 128, 64, "split_bf16"), (8200, 128, 64, "fp32"), (66000, 128, 128, "split_f16")])
def test_linear_batched_residual_in_place(cuda, M, N, K, mode):
    """R = Y (16-row, 128-row and tall tiles, a K tail, the three modes): the bits of the same call with the
    residual in an array of its own."""
    from ops import _lib
    g = torch.Generator(device=cuda).manual_seed(M + K)
    r = lambda *s: torch.randn(*s, device=cuda, generator=g)
    A, W, R = r(M, K), r(N, K), r(M, N)
    Y, out = R.clone(), torch.empty_like(R)
    with _lib.matmul_mode(_lib.MATMUL_MODES[mode]):
        for res, y in ((R, out), (Y, Y)):
            _lib.call("fu_linear_batched", A.data_ptr(), K, 0, W.data_ptr(), K, 0, None, 0, 0, res.data_ptr(), N, 0,
                      y.data_ptr(), N, 0, M, N, K, 1, _lib.stream_ptr(cuda))
    assert torch.equal(Y, out)


@pytest.mark.parametrize("counts", [[3, 0, 257, 1], [1], [0, 0, 5000, 70, 0], [40] * 300])
def test_edge_shifts_batched(cuda, counts):
    """Shifts of several systems and their cells' gradients against float64, with systems of no edges;
    counts that do not describe the edges are refused; a float64 cell still works."""
    from ops.node import edge_shifts_batched
    g = torch.Generator().manual_seed(len(counts))
    n, E = torch.tensor(counts), sum(counts)
    off = torch.randint(-3, 4, (E, 3), generator=g).float()
    cell, cot = torch.randn(len(counts), 3, 3, generator=g) * 8, torch.randn(E, 3, generator=g)
    cd = cell.double().requires_grad_()
    ref = torch.einsum("ij,ijk->ik", off.double(), cd.repeat_interleave(n, dim=0))
    (gref,) = torch.autograd.grad(ref, cd, cot.double())
    cg = cell.to(cuda).requires_grad_()
    out = edge_shifts_batched(off.to(cuda), cg, n.to(cuda))
    (gc,) = torch.autograd.grad(out, cg, cot.to(cuda))
    # three fp32 products and two sums each; the gradient's sums in fp64, rounded once
    assert (out.cpu().double() - ref.detach()).abs().max() <= 3 * 2.0 ** -23 * 3 * cell.abs().max() * 3
    assert (gc.cpu().double() - gref).abs().max() <= 2.0 ** -22 * gref.abs().max()
    assert torch.equal(gc, torch.autograd.grad(edge_shifts_batched(off.to(cuda), cg, n.to(cuda)), cg, cot.to(cuda))[0])
    for bad in (n + torch.eye(len(counts), dtype=torch.long)[0], torch.cat([n[:-1], n[-1:] - 1])):
        with pytest.raises(RuntimeError):
            edge_shifts_batched(off.to(cuda), cg, bad.to(cuda))
    d = edge_shifts_batched(off.to(cuda), cell.double().to(cuda), n.to(cuda))
    assert d.dtype == torch.float64 and torch.allclose(d.cpu(), ref.detach(), atol=1e-12)
