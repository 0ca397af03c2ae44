"""Node segments shared by one, two or four waves (the scatters, the gather backward): node counts on
both sides of the rules' lines, segments that are empty, of one to three edges (fewer than the waves)
and of 150, against the float64 oracle, and the same bits on every run."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _edges(N, seed):
    """Both directions of random pairs, node 0 with 150 neighbours, nodes 1 to 3 with 1 to 3, and
    node 4 with none."""
    g = torch.Generator().manual_seed(seed)
    lo = 5 if N > 6 else 0
    i = torch.randint(lo, N, (3 * N + 5,), generator=g)
    j = torch.randint(lo, N, (3 * N + 5,), generator=g)
    if N > 6:
        hub, few = torch.randint(lo, N, (150,), generator=g), torch.tensor([1, 2, 2, 3, 3, 3])
        i = torch.cat([i, hub, few])
        j = torch.cat([j, torch.zeros(150, dtype=torch.long), torch.randint(lo, N, (6,), generator=g)])
    return torch.stack([torch.cat([i, j]), torch.cat([j, i])])


@pytest.mark.parametrize("N,C,L", [(1, 128, 2), (6, 64, 2), (256, 128, 2), (257, 128, 2), (1024, 64, 2), (1025, 128, 2),
                                   (1537, 64, 2), (2049, 64, 2), (30, 128, 4), (257, 64, 4), (1025, 64, 3), (12, 256, 4),
                                   (9, 256, 2)])
def test_shared_segments(cuda, N, C, L):
    from _helpers import assert_close
    from oracle import ops_ref as R
    from oracle import sh_ref as S
    from ops import gather, lmax, scatter, topology
    ei = _edges(N, N + C + L)
    E = ei.shape[1]
    g = torch.Generator().manual_seed(E + L)
    q = torch.randn(E, 4, generator=g, dtype=torch.float64)
    q = q / q.norm(dim=1, keepdim=True)
    rot = R.rotation_from_quaternion(q)
    wig = torch.cat([rot.reshape(E, 9), R.wigner_l2_from_quaternion(q).reshape(E, 25)], 1).float()
    ext = S.wigner_ext(rot, L).float() if L > 2 else torch.zeros(E, 0)
    r = lambda *s: torch.randn(*s, generator=g)
    x, rad, csd, env = r(N, (L + 1) ** 2, C), r(E, 6 * L * C), r(1, C), torch.rand(E, generator=g)
    Z = [r(E, k * C) for k in (L + 1, 2 * L, 2 * (L - 1))]
    cot = [r(E, 2 * k * C) for k in (L + 1, 2 * L, 2 * (L - 1))]
    rad0, Ws, Zn = r(E, (L + 1) * C), r(100, C), torch.randint(1, 90, (N,), generator=g)
    batch = torch.zeros(N, dtype=torch.long)
    D = [t.double() for t in (wig, ext, env, x, rad, csd, rad0, Ws)]
    xr, radr, wr = (t.requires_grad_() for t in (x.double(), rad.double(), wig.double()))
    if L == 2:
        ref_s = R.rotate_scatter(*[z.double() for z in Z], D[0], D[2], D[3], ei[1], N)
        ref_i = R.init_scatter(D[6], D[0], D[2], Zn, batch, D[7], D[5], ei[1], N)
        X = R.gather_rotate(xr, ei[0], ei[1], wr, radr, D[5], batch)
    else:
        ref_s = R.rotate_scatter_lmax(*[z.double() for z in Z], D[0], D[1], D[2], D[3], ei[1], N, L)
        ref_i = R.init_scatter_lmax(D[6], D[0], D[1], D[2], Zn, batch, D[7], D[5], ei[1], N, L)
        X = R.gather_rotate_lmax(xr, ei[0], ei[1], wr, D[1], radr, D[5], batch, L)
    ref_g = torch.autograd.grad(sum((a * c.double()).sum() for a, c in zip(X, cot)), (xr, radr, wr))

    t = lambda v: v.to(cuda)
    ij = t(ei)
    rp, ri = topology.receiver_csr(ij[1], N)

    def run():
        with torch.no_grad():
            if L == 2:
                s = scatter.rotate_scatter_split(*map(t, Z), t(wig), t(env), t(x), ij[1], rp, ri, N)
                i = scatter.init_node_scatter(t(rad0), t(wig), t(env), t(Zn), t(batch), t(Ws), t(csd), ij[1], rp, ri, N)
            else:
                s = lmax.rotate_scatter_lmax(*map(t, Z), t(wig), t(ext), t(env), t(x), ij[1], rp, ri, N, L)
                i = lmax.init_node_scatter_lmax(t(rad0), t(wig), t(ext), t(env), t(Zn), t(batch), t(Ws), t(csd), ij[1],
                                                rp, ri, N, L)
        ins = [t(v).requires_grad_() for v in (x, rad, wig)]
        if L == 2:
            out = gather.gather_wigner_split(ins[0], ij[0], ij[1], ins[2], ins[1], t(csd), t(batch))
        else:
            out = lmax.gather_rotate_lmax(ins[0], ij[0], ij[1], ins[2], t(ext), ins[1], t(csd), t(batch), None, L)
        return [s, i, *torch.autograd.grad(out, ins, [t(c) for c in cot])]

    a, b = run(), run()
    assert all(torch.equal(u, v) for u, v in zip(a, b))
    # the bar of the kernels with one wave a segment: fp32 messages, sums in fp64 where a node collects
    # its edges, relative to the largest value
    for u, v, name in zip(a, [ref_s, ref_i, *ref_g], ("scatter", "init scatter", "g_x", "g_rad", "g_wigner")):
        assert_close(u, v, 1e-5, name)
