"""Which entry point a call goes to, and which calls are refused, by shapes and alignment: on the CPU,
with the library's entry points replaced by a recorder (nothing is launched)."""
import pytest
import torch


@pytest.fixture
def calls(monkeypatch):
    """Names of the entry points called; CPU tensors pass for device ones."""
    from ops import _lib
    names = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: names.append(name))
    monkeypatch.setattr(_lib, "require", lambda t, dtype, name: t.to(dtype).contiguous())
    monkeypatch.setattr(_lib, "ptr", lambda t: None if t is None else t.data_ptr())
    monkeypatch.setattr(_lib, "stream_ptr", lambda device=None: 0)
    monkeypatch.setattr(_lib, "side_stream", lambda device: None)
    monkeypatch.setattr(_lib, "get_matmul_mode", lambda: _lib.MATMUL_SPLIT_F16)
    return names


def _pair(E=8, C=64, L=2, S=None, H=None, wide=0):
    """Operands of a pair of E edges: S input channels per degree, H output ones (both C by default),
    `wide` unused columns after X_m0's."""
    S, H = S or C, H or C
    n = (L + 1, L, L - 1)
    z = torch.zeros
    w = lambda r, k: (z(r, k), z(k, r))
    cx = lambda r, k: (z(r, k), z(r, k), z(k, r), z(k, r))
    W0, W0t = w((2 * L + 1) * C, 2 * n[0] * S)
    V0, V0t = w(n[0] * H, n[0] * C)
    conv1 = (W0, z((2 * L + 1) * C), W0t, *cx(n[1] * C, 2 * n[1] * S), *cx(n[2] * C, 2 * n[2] * S))
    conv2 = (V0, z(n[0] * H), V0t, *cx(n[1] * H, n[1] * C), *cx(n[2] * H, n[2] * C))
    X = [z(E, 2 * n[0] * S + wide), z(E, 4 * n[1] * S), z(E, 4 * n[2] * S)]
    g = [z(E, n[0] * H), z(E, 2 * n[1] * H), z(E, 2 * n[2] * H)]
    Y = (z(E, (2 * L + 1) * C), z(E, 2 * n[1] * C), z(E, 2 * n[2] * C))
    return X, g, Y, conv1, conv2, tuple(z(4) for _ in range(12))


SHORT, TILED = "fu_so2_pair_fwd", "fu_linear_gate"


@pytest.mark.parametrize("C,L", [(64, 2), (128, 3), (192, 4), (256, 2)])
def test_pair_takes_the_few_row_kernels(calls, C, L):
    from ops import gating
    X, g, Y, conv1, conv2, sp = _pair(C=C, L=L)
    gating.conv_pair_fwd(X, conv1, conv2, C, sp)
    gating.conv_pair_bwd(Y, conv1, conv2, C, sp, g)
    assert calls == ["fu_so2_pair_fwd", "fu_so2_pair_bwd"]


@pytest.mark.parametrize("form", [dict(S=32), dict(S=128), dict(H=32), dict(H=128), dict(wide=4)])
def test_pair_of_other_widths_stays_tiled(calls, form):
    """Input or output channels other than C, or rows with more columns than the weight reads: the few-row
    entry points, which are given C alone, would read and write at other strides than the arrays'."""
    from ops import gating
    X, g, Y, conv1, conv2, sp = _pair(**form)
    gating.conv_pair_fwd(X, conv1, conv2, 64, sp)
    assert SHORT not in calls and TILED in calls
    if "wide" not in form:
        gating.conv_pair_bwd(Y, conv1, conv2, 64, sp, g)
        assert "fu_so2_pair_bwd" not in calls and "fu_linear_gate_bwd" in calls


def test_pair_with_an_unaligned_conv2_bias_stays_tiled(calls):
    """fu_linear reads its bias a float at a time; the few-row kernels read 16 bytes."""
    from ops import gating
    X, g, Y, conv1, conv2, sp = _pair()
    conv2 = (conv2[0], torch.zeros(conv2[1].numel() + 1)[1:], *conv2[2:])
    gating.conv_pair_fwd(X, conv1, conv2, 64, sp)
    assert SHORT not in calls and TILED in calls


def test_pair_with_rows_of_another_count_stays_tiled(calls):
    from ops import gating
    X, g, Y, conv1, conv2, sp = _pair()
    X[0] = X[0][:5]
    gating.conv_pair_fwd(X, conv1, conv2, 64, sp)
    assert SHORT not in calls


def test_scalar_gemm_refuses_other_widths(calls):
    """The scalar linear reads rows of x (N, K, Cin) at its own weight's width: a weight of another width is
    refused, forward and backward, as ops.linear.gemm refuses it, not read across coefficients."""
    from ops import _lib, node
    z = torch.zeros
    x, Wk, Wtk = z(5, 9, 64), z(9, 32, 64), z(9, 64, 32)
    ok = node.scalar_gemm_so3(x, z(96, 64), z(96), z(64, 96), Wk, Wtk, z(32))
    assert [t.shape for t in ok] == [(5, 96), (5, 9, 32)]
    with pytest.raises(_lib.FlashUMAError):
        node.scalar_gemm_so3(x, z(96, 128), z(96), z(128, 96), Wk, Wtk, z(32))
    for Wt in (z(64, 64), z(128, 96)):   # of another gradient's width, and of another x's
        xg = x.clone().requires_grad_()
        pre, h = node.scalar_gemm_so3(xg, z(96, 64), z(96), Wt, Wk, Wtk, z(32))
        with pytest.raises(_lib.FlashUMAError):
            torch.autograd.grad((pre.sum() + h.sum()), xg)


def test_few_row_product_dispatch(calls):
    """fu_linear_short takes rows of unit column stride at the weight's width; other rows are copied for
    fu_linear, and another width is refused."""
    from ops import _lib, linear
    z = torch.zeros
    W, W2, out = z(64, 320), z(4), z(7, 64)
    linear.gemm_few_rows(z(7, 320), W, W2, out)
    linear.gemm_few_rows(z(7, 324)[:, :320], W, W2, out)
    assert calls == ["fu_linear_short"] * 2
    linear.gemm_few_rows(z(7, 640)[:, ::2], W, W2, out)
    linear.gemm_few_rows(z(320, 8).t()[:7], W, W2, out)
    assert calls[2:] == ["fu_linear"] * 2
    with pytest.raises(_lib.FlashUMAError):
        linear.gemm_few_rows(z(7, 256), W, W2, out)


@pytest.mark.parametrize("C,L,most", [(64, 2, 16384), (64, 3, 14209), (64, 4, 7898), (128, 2, 7992), (128, 4, 1974),
                                      (256, 2, 1998), (256, 4, 493)])
def test_pair_on_both_sides_of_its_line(calls, C, L, most):
    """The last edge count of the few-row kernels and the first of the tiled ones, forward and backward."""
    from ops import gating
    e = lambda *s: torch.empty(*s, device="meta")
    for pair in gating._pair_shapes(C, L):
        for E in (1, most, most + 1):
            arrays, weights = [e(E, w) for w in pair[1]], [e(*s) for s in pair[2]]
            assert gating._short_pair(E, pair, (0,) * 12, arrays, weights) is (E <= most)
