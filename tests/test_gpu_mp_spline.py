"""Message passing with in-kernel radial spline: parity with the fp64 oracle (spline evaluation followed by the
message-passing definition, gradients by autograd) and bit-level consistency with the two-step GPU path."""
import numpy as np
import pytest
import torch

from oracle import ops as O
from tests.util import close, mp_inputs, random_graph

pytestmark = pytest.mark.gpu

CASES = [
    # nnodes, avg degree, channels, isolated fraction, seed
    (50, 6, 32, 0.2, 0),
    (200, 30, 64, 0.0, 1),
    (300, 52, 96, 0.05, 2),
    (300, 52, 128, 0.0, 3),
    (30, 160, 128, 0.0, 4),
    (120, 40, 192, 0.1, 5),
    (60, 20, 256, 0.0, 6),
    (70, 30, 160, 0.1, 7),   # 40 of 64 lanes carry channels
    (50, 90, 224, 0.0, 8),   # 56 of 64 lanes; segments longer than one 64-edge chunk
]


def _case(nnodes, avg, C, iso, seed):
    snd, rcv = random_graph(nnodes, avg, seed, isolated_frac=iso)
    E = snd.numel()
    X, v, _, G = mp_inputs(nnodes, E, C, seed)
    g = torch.Generator().manual_seed(seed + 100)
    r = torch.rand(E, generator=g, dtype=torch.float64) * 4.6 + 0.7  # a few beyond r_max = 5
    r = r.float().double()  # the kernel sees fp32 lengths
    Y = O.spherical_harmonics(v).contiguous()
    knots_np, h = np.linspace(1e-12, 6.0, 256, retstep=True)
    knots = torch.from_numpy(knots_np)
    J = 4 * C
    table = torch.sin(knots[:, None] * torch.linspace(0.5, 2.5, J, dtype=torch.float64)[None, :]) * torch.randn(
        1, J, generator=g, dtype=torch.float64)
    coeffs = O.spline_coefficients(knots, table).float().double()  # the kernel sees fp32 coefficients
    return snd, rcv, X, Y, r, knots.float().double(), coeffs, float(np.float32(h)), G


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_d%d_C%d_s%d" % (c[0], c[1], c[2], c[4]))
def test_mp_spline_forward_backward(cabi, case):
    print("mp_spline", case, flush=True)
    nnodes, C = case[0], case[2]
    snd, rcv, X, Y, r, knots, coeffs, h, G = _case(*case)
    E = snd.numel()
    Xa, Ya, ra = (t.clone().requires_grad_(True) for t in (X, Y, r))
    R = O.spline_eval(ra, knots, coeffs, h, 5.0).view(E, 4, C)
    ref = O.mp_forward(Xa, Ya, R, snd, rcv, nnodes)
    (ref * G).sum().backward()

    d = lambda t: t.float().cuda()
    fo = cabi.first_occurences(rcv.cuda(), nnodes)
    perm, off = cabi.stable_key_sort(snd.cuda(), nnodes)
    out = cabi.mp_spline_forward(d(X), d(Y), d(r), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    gX, gY, gr = cabi.mp_spline_backward(d(X), d(Y), d(r), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes)
    close(out, ref.detach(), 2e-5, 2e-6)
    close(gX, Xa.grad, 2e-5, 2e-6)
    close(gY, Ya.grad, 2e-5, 2e-6)
    close(gr, ra.grad, 3e-5, 3e-6)

    # the two-step GPU path (spline kernel, then tabulated message passing) gives the same numbers
    R32 = cabi.spline_forward(d(r), d(knots), d(coeffs), h, 5.0)
    out2 = cabi.mp_forward(d(X), d(Y), R32.view(E, 4, C), snd.cuda(), fo, nnodes)
    close(out, out2.double().cpu(), 1e-6, 1e-6)
    gX2, gY2, gR2 = cabi.mp_backward(d(X), d(Y), R32.view(E, 4, C), d(G), snd.cuda(), fo, perm, off, nnodes)
    gr2 = cabi.spline_backward(d(r), d(knots), d(coeffs), gR2.view(E, 4 * C), h, 5.0)
    close(gY, gY2.double().cpu(), 1e-5, 1e-6)
    close(gX, gX2.double().cpu(), 1e-5, 1e-6)
    bound = 4e-6 * (gR2.view(E, -1).abs().double().cpu() * O.spline_eval(r, knots, coeffs, h, 5.0, deriv=True)[1].abs()).sum(-1) + 1e-30
    assert bool(((gr.double().cpu() - gr2.double().cpu()).abs() <= bound).all())

    # edge-vector variant: harmonics and length computed in-kernel; oracle = SH + spline + MP, gradient by autograd
    g2 = torch.Generator().manual_seed(case[4] + 7)
    vec = torch.randn(E, 3, generator=g2, dtype=torch.float64)
    vec = (vec / vec.norm(dim=1, keepdim=True) * r[:, None]).float().double()  # lengths spread like r, fp32-representable
    va = vec.clone().requires_grad_(True)
    Xb = X.clone().requires_grad_(True)
    Rv = O.spline_eval(va.norm(dim=1), knots, coeffs, h, 5.0).view(E, 4, C)
    ref_e = O.mp_forward(Xb, O.spherical_harmonics(va), Rv, snd, rcv, nnodes)
    (ref_e * G).sum().backward()
    out_e = cabi.mp_edge_forward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    gX_e, gvec = cabi.mp_edge_backward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes)
    close(out_e, ref_e.detach(), 2e-5, 2e-6)
    close(gX_e, Xb.grad, 2e-5, 2e-6)
    close(gvec, va.grad, 5e-5, 5e-6)
    gX_only, none = cabi.mp_edge_backward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes,
                                          need_gvec=False)
    assert none is None and torch.equal(gX_only, gX_e)
    none, gvec_only = cabi.mp_edge_backward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes,
                                            need_gX=False)
    assert none is None and torch.equal(gvec_only, gvec)

    # subsets of gradients
    only_r = cabi.mp_spline_backward(d(X), d(Y), d(r), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes,
                                     need_gX=False, need_gY=False)
    assert only_r[0] is None and only_r[1] is None and torch.equal(only_r[2], gr)
    no_x = cabi.mp_spline_backward(d(X), d(Y), d(r), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes,
                                   need_gX=False)
    assert no_x[0] is None and torch.equal(no_x[1], gY) and torch.equal(no_x[2], gr)


@pytest.mark.parametrize("degree", [70, 200])
def test_edges_beyond_cutoff_and_invalid_senders_cost_nothing_and_contribute_nothing(cabi, degree):
    """A list with a wide skin (most edges beyond r_max) and a few out-of-range sender indices: those edges add nothing
    to the output and get exactly zero gradients; the rest matches the oracle evaluated on the live edges alone.  The
    kernels stage 64 live edges at a time out of as many raw ones as that takes: 70 raw edges per node fill one chunk from
    two reads, 200 make chunks that end in the middle of a read."""
    nnodes, C, seed = 90, 128, 11
    snd, rcv = random_graph(nnodes, degree, seed)
    E = snd.numel()
    X, _, _, G = mp_inputs(nnodes, E, C, seed)
    g = torch.Generator().manual_seed(seed)
    r = torch.rand(E, generator=g, dtype=torch.float64) * 9.0 + 0.7  # r_max = 5: about half the edges are beyond it
    vec = torch.randn(E, 3, generator=g, dtype=torch.float64)
    vec = (vec / vec.norm(dim=1, keepdim=True) * r[:, None]).float().double()
    snd = snd.clone()
    bad = torch.randperm(E, generator=g)[:40]
    snd[bad[:20]] = nnodes + 3
    snd[bad[20:]] = -1
    knots_np, h = np.linspace(1e-12, 6.0, 256, retstep=True)
    knots = torch.from_numpy(knots_np)
    table = torch.cos(knots[:, None] * torch.linspace(0.3, 2.0, 4 * C, dtype=torch.float64)[None, :])
    coeffs = O.spline_coefficients(knots, table).float().double()
    h = float(np.float32(h))
    live = (vec.norm(dim=1).float() <= 5.0) & (snd >= 0) & (snd < nnodes)
    assert 0.3 < float(live.double().mean()) < 0.7

    va = vec[live].clone().requires_grad_(True)
    Xa = X.clone().requires_grad_(True)
    Rv = O.spline_eval(va.norm(dim=1), knots.float().double(), coeffs, h, 5.0).view(-1, 4, C)
    ref = O.mp_forward(Xa, O.spherical_harmonics(va), Rv, snd[live], rcv[live], nnodes)
    (ref * G).sum().backward()

    d = lambda t: t.float().cuda()
    fo = cabi.first_occurences(rcv.cuda(), nnodes)
    perm, off = cabi.stable_key_sort(snd.cuda(), nnodes)
    out = cabi.mp_edge_forward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    gX, gvec = cabi.mp_edge_backward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes)
    close(out, ref.detach(), 2e-5, 2e-6)
    close(gX, Xa.grad, 2e-5, 2e-6)
    close(gvec[live.cuda()], va.grad, 5e-5, 5e-6)
    assert float(gvec[~live.cuda()].abs().max()) == 0.0
    gvec_only = cabi.mp_edge_backward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes,
                                      need_gX=False)[1]
    assert torch.equal(gvec_only, gvec)


# ---- many receiver nodes: the forward from edge vectors runs on the kernel that keeps its part of the table in LDS ----
def _edge_case(nnodes, avg, C, iso, seed, nknots=256, heavy=0):
    """Receiver-sorted random graph with edge vectors of lengths 0.7 .. 5.3 (r_max = 5), a few senders out of range,
    optionally one node with `heavy` extra edges (more edge blocks than the kernel's node sort tells apart)."""
    snd, rcv = random_graph(nnodes, avg, seed, isolated_frac=iso)
    if heavy:
        g0 = torch.Generator().manual_seed(seed + 5)
        node = nnodes // 3
        extra = torch.randint(0, nnodes, (heavy,), generator=g0, dtype=torch.int32)
        at = int(torch.searchsorted(rcv, torch.tensor(node, dtype=torch.int32)))
        snd = torch.cat([snd[:at], extra, snd[at:]])
        rcv = torch.cat([rcv[:at], torch.full((heavy,), node, dtype=torch.int32), rcv[at:]])
    E = snd.numel()
    g = torch.Generator().manual_seed(seed + 100)
    X = torch.randn(nnodes, C, generator=g, dtype=torch.float64)
    r = torch.rand(E, generator=g, dtype=torch.float64) * 4.6 + 0.7
    vec = torch.randn(E, 3, generator=g, dtype=torch.float64)
    vec = (vec / vec.norm(dim=1, keepdim=True) * r[:, None]).float().double()
    snd = snd.clone()
    bad = torch.randperm(E, generator=g)[:30]
    snd[bad[:15]] = nnodes + 5
    snd[bad[15:]] = -1
    knots_np, h = np.linspace(1e-12, 6.0, nknots, retstep=True)
    knots = torch.from_numpy(knots_np)
    table = torch.sin(knots[:, None] * torch.linspace(0.5, 2.5, 4 * C, dtype=torch.float64)[None, :]) * torch.randn(
        1, 4 * C, generator=g, dtype=torch.float64)
    coeffs = O.spline_coefficients(knots, table).float().double()
    return snd, rcv, X, vec, knots.float().double(), coeffs, float(np.float32(h))


MANY_NODES = [
    # nnodes, avg degree, channels, isolated fraction, seed, knots, extra edges of one node
    (2100, 14, 32, 0.1, 0, 256, 0),
    (2300, 9, 64, 0.0, 1, 256, 300),   # one node with more than 63 blocks of four edges
    (2048, 21, 96, 0.05, 2, 200, 0),
    (3000, 6, 160, 0.3, 3, 256, 0),
    (2500, 3, 256, 0.0, 4, 272, 0),    # the largest table the kernel keeps in LDS
]


@pytest.mark.parametrize("case", MANY_NODES, ids=lambda c: "N%d_d%d_C%d_k%d" % (c[0], c[1], c[2], c[5]))
def test_mp_edge_forward_many_nodes(cabi, case):
    """Parity with the fp64 oracle (harmonics, spline, message-passing definition) on the live edges; edges beyond the
    cutoff or with a sender out of range add nothing; nodes without edges come out as zeros; the result is the same
    on a second call (which wave serves a node changes from run to run, the node's result must not)."""
    print("mp_edge_forward many nodes", case, flush=True)
    nnodes, C = case[0], case[2]
    snd, rcv, X, vec, knots, coeffs, h = _edge_case(*case)
    live = (vec.norm(dim=1).float() <= 5.0) & (snd >= 0) & (snd < nnodes)
    Rv = O.spline_eval(vec[live].norm(dim=1), knots, coeffs, h, 5.0).view(-1, 4, C)
    ref = O.mp_forward(X, O.spherical_harmonics(vec[live]), Rv, snd[live], rcv[live], nnodes)
    d = lambda t: t.float().cuda()
    fo = cabi.first_occurences(rcv.cuda(), nnodes)
    out = cabi.mp_edge_forward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    close(out, ref, 2e-5, 2e-6)
    empty = torch.bincount(rcv.long(), minlength=nnodes) == 0
    assert float(out[empty.cuda()].abs().max()) == 0.0 if bool(empty.any()) else True
    again = cabi.mp_edge_forward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    assert torch.equal(out, again)


@pytest.mark.parametrize("case", [(5121, 4, 32, 0.1, 5, 256, 0), (2561, 9, 64, 0.0, 6, 256, 300), (2560, 9, 64, 0.0, 6, 256, 300),
                                  (1281, 7, 128, 0.1, 7, 272, 0), (1280, 7, 128, 0.1, 7, 272, 0), (641, 11, 256, 0.2, 8, 2, 0),
                                  (1281, 50, 128, 0.0, 7, 272, 0), (641, 20, 256, 0.0, 8, 2, 0)],
                         ids=lambda c: "N%d_d%d_C%d" % (c[0], c[1], c[2]))
def test_mp_edge_forward_on_both_sides_of_the_line(cabi, case):
    """The smallest node counts at which that kernel is taken, and the largest at which it is not."""
    test_mp_edge_forward_many_nodes(cabi, case)


@pytest.mark.parametrize("case", [(2600, 38, 64, 0.0, 1, 256, 300), (2600, 30, 64, 0.0, 1, 256, 300), (2048, 33, 96, 0.05, 2, 200, 0),
                                  (2048, 26, 96, 0.05, 2, 200, 0), (1300, 14, 160, 0.3, 3, 256, 0), (1300, 9, 160, 0.3, 3, 256, 0),
                                  (900, 13, 192, 0.0, 4, 256, 0), (900, 9, 192, 0.0, 4, 256, 0), (1000, 10, 224, 0.0, 5, 256, 0),
                                  (1000, 7, 224, 0.0, 5, 256, 0), (700, 13, 256, 0.0, 6, 272, 0), (700, 9, 256, 0.0, 6, 272, 0)],
                         ids=lambda c: "N%d_d%d_C%d" % (c[0], c[1], c[2]))
def test_mp_edge_forward_on_both_sides_of_the_line_by_edges(cabi, case):
    """Nodes enough for that kernel, edges just enough and not enough: its heavy node, tables and isolated nodes again."""
    test_mp_edge_forward_many_nodes(cabi, case)


@pytest.mark.parametrize("case", [(2048, 36, 96, 0.05, 2, 200, 0), (1300, 25, 160, 0.3, 3, 256, 0), (900, 22, 192, 0.0, 4, 256, 0),
                                  (1000, 12, 224, 0.0, 5, 256, 0), (700, 17, 256, 0.0, 6, 272, 0), (9000, 9, 128, 0.1, 7, 128, 300),
                                  (3841, 3, 32, 0.3, 8, 256, 0), (2433, 11, 64, 0.0, 9, 256, 70), (1217, 23, 128, 0.0, 10, 256, 0), (769, 9, 160, 0.0, 11, 256, 0),
                                  (609, 53, 256, 0.0, 12, 256, 0)],
                         ids=lambda c: "N%d_d%d_C%d" % (c[0], c[1], c[2]))
def test_mp_edge_forward_just_above_the_line_by_edges(cabi, case):
    """As above, with the edges that the line asks for at these widths, and many nodes with few edges."""
    test_mp_edge_forward_many_nodes(cabi, case)


@pytest.mark.parametrize("nnodes,avg,C", [(40000, 13, 256), (40000, 18, 256), (23500, 15, 256), (46000, 10, 128), (33000, 12, 256), (33000, 14, 256)])
def test_mp_edge_forward_sorts_the_nodes_of_a_workgroup_in_batches(cabi, nnodes, avg, C):
    """More receiver nodes per workgroup than the 2 816 that are sorted at a time (40 000 at 256 channels: 5 000), with edges enough
    for that kernel where the output is beyond the last-level cache, and with fewer (12 per node at 40 000 and 33 000
    nodes).  Against the kernel that takes harmonics and lengths, and the oracle on a sample of nodes."""
    snd, rcv, X, vec, knots, coeffs, h = _edge_case(nnodes, avg, C, 0.1 if avg == 13 else 0.0, 9)
    assert rcv.numel() > 9 * nnodes
    d = lambda t: t.float().cuda()
    fo = cabi.first_occurences(rcv.cuda(), nnodes)
    out = cabi.mp_edge_forward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    other = cabi.mp_spline_forward(d(X), cabi.sh_forward(d(vec)), d(vec).norm(dim=1), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    # fp32 rounding of length, harmonics and about a dozen terms per sum, against the largest component
    assert float((out - other).abs().max()) <= 1e-5 * float(other.abs().max())
    nodes = torch.arange(0, nnodes, 997)
    pick = torch.isin(rcv.long(), nodes)
    live = pick & (vec.norm(dim=1).float() <= 5.0) & (snd >= 0) & (snd < nnodes)
    Rv = O.spline_eval(vec[live].norm(dim=1), knots, coeffs, h, 5.0).view(-1, 4, C)
    ref = O.mp_forward(X, O.spherical_harmonics(vec[live]), Rv, snd[live], rcv[live], nnodes)
    close(out[nodes.cuda()], ref[nodes], 2e-5, 2e-6)


def test_mp_edge_forward_many_nodes_agrees_with_harmonics_and_lengths_path(cabi):
    """40 000 receiver nodes at 256 channels: a workgroup of the LDS-table kernel sorts and serves its nodes in more than
    one batch.  Checked against the kernel that takes harmonics and lengths (same radial table, same per-edge
    arithmetic, another summation order), and against the oracle on a sample of nodes."""
    nnodes, C = 40000, 256
    snd, rcv, X, vec, knots, coeffs, h = _edge_case(nnodes, 3, C, 0.1, 9)
    d = lambda t: t.float().cuda()
    fo = cabi.first_occurences(rcv.cuda(), nnodes)
    out = cabi.mp_edge_forward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    Y = cabi.sh_forward(d(vec))
    length = d(vec).norm(dim=1)  # rounding of the length may differ from the kernel's in the last bit
    other = cabi.mp_spline_forward(d(X), Y, length, d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    close(out, other.double().cpu(), 1e-4, 1e-5)
    nodes = torch.arange(0, nnodes, 997)
    pick = torch.isin(rcv.long(), nodes)
    live = pick & (vec.norm(dim=1).float() <= 5.0) & (snd >= 0) & (snd < nnodes)
    Rv = O.spline_eval(vec[live].norm(dim=1), knots, coeffs, h, 5.0).view(-1, 4, C)
    ref = O.mp_forward(X, O.spherical_harmonics(vec[live]), Rv, snd[live], rcv[live], nnodes)
    close(out[nodes.cuda()], ref[nodes], 2e-5, 2e-6)


@pytest.mark.parametrize("case", [(1024, 6, 160, 0.2, 21, 256, 0), (1100, 13, 160, 0.0, 22, 600, 150), (1024, 5, 192, 0.2, 23, 256, 0), (1024, 15, 192, 0.2, 25, 256, 0),
                                  (1060, 17, 192, 0.0, 24, 2, 129)], ids=lambda c: "N%d_d%d_C%d_k%d" % (c[0], c[1], c[2], c[5]))
def test_mp_edge_backward_of_four_edges_per_step(cabi, case):
    """The kernel with a row of 16 lanes per edge (and, at five edges per node and 192 channels, the one with an edge per wave):
    nodes with every remainder of a group of four edges, one with more than one and more than two chunks of 64, dead edges in
    between, knots in LDS and in memory, a table of one interval."""
    nnodes, C = case[0], case[2]
    snd, rcv, X, vec, knots, coeffs, h = _edge_case(*case)
    degrees = torch.bincount(rcv.long(), minlength=nnodes)
    assert set((degrees % 4).tolist()) == {0, 1, 2, 3}
    G = torch.randn(nnodes, 16, C, generator=torch.Generator().manual_seed(case[4]), dtype=torch.float64)
    live = (vec.norm(dim=1).float() <= 5.0) & (snd >= 0) & (snd < nnodes)
    va, Xa = vec[live].clone().requires_grad_(True), X.clone().requires_grad_(True)
    Rv = O.spline_eval(va.norm(dim=1), knots, coeffs, h, 5.0).view(-1, 4, C)
    (O.mp_forward(Xa, O.spherical_harmonics(va), Rv, snd[live], rcv[live], nnodes) * G).sum().backward()
    d = lambda t: t.float().cuda()
    fo = cabi.first_occurences(rcv.cuda(), nnodes)
    perm, off = cabi.stable_key_sort(snd.cuda(), nnodes)
    args = (d(X), d(vec), d(knots), d(coeffs), h, 5.0, d(G), snd.cuda(), fo, perm, off, nnodes)
    gX, gvec = cabi.mp_edge_backward(*args)
    close(gX, Xa.grad, 2e-5, 2e-6)
    close(gvec[live.cuda()], va.grad, 5e-5, 5e-6)
    assert float(gvec[~live.cuda()].abs().max()) == 0.0
    assert torch.equal(cabi.mp_edge_backward(*args, need_gvec=False)[0], gX)
    assert torch.equal(cabi.mp_edge_backward(*args, need_gX=False)[1], gvec)


@pytest.mark.parametrize("case", [(120, 9, 64, 0.1, 51, 256, 0), (409, 20, 32, 0.0, 52, 256, 0), (513, 16, 32, 0.1, 53, 256, 0), (1024, 9, 64, 0.0, 54, 256, 0), (1025, 33, 64, 0.0, 55, 256, 0),
                                  (1536, 33, 32, 0.2, 56, 256, 0), (1537, 33, 32, 0.0, 57, 256, 150), (40, 9, 160, 0.0, 31, 3, 0), (90, 21, 192, 0.0, 32, 257, 150), (300, 19, 224, 0.1, 33, 600, 150),
                                  (1100, 13, 224, 0.0, 34, 256, 129), (40, 7, 64, 0.0, 35, 4, 0), (300, 13, 64, 0.1, 36, 512, 150),
                                  (1100, 9, 32, 0.1, 37, 5, 150), (2100, 6, 128, 0.1, 38, 513, 70), (300, 17, 96, 0.0, 39, 256, 130)],
                         ids=lambda c: "N%d_d%d_C%d_k%d" % (c[0], c[1], c[2], c[5]))
def test_mp_edge_backward_few_and_many_nodes(cabi, case):
    """Few nodes (an edge range cut into parts) and many, every width class, partly filled groups, trips and chunks, and tables on
    both sides of what the copy of the knots takes (four knots at a time, up to 256 or 512)."""
    test_mp_edge_backward_of_four_edges_per_step(cabi, case)


@pytest.mark.parametrize("case", [(1023, 9, 160, 0.1, 71, 256, 0), (1025, 9, 192, 0.0, 72, 256, 0), (2049, 7, 224, 0.1, 73, 256, 70), (2047, 1, 160, 0.0, 74, 256, 0),
                                  (511, 9, 160, 0.1, 75, 256, 0), (512, 9, 160, 0.0, 76, 256, 0), (513, 9, 160, 0.1, 77, 256, 0), (341, 9, 160, 0.0, 78, 256, 0),
                                  (343, 9, 160, 0.1, 79, 256, 0)],
                         ids=lambda c: "N%d_d%d_C%d_k%d" % (c[0], c[1], c[2], c[5]))
def test_mp_edge_backward_of_nodes_beyond_whole_runs(cabi, case):
    """Workgroups, a node's parts in order, are dealt to the eight XCDs in runs of 128, those behind the last 1 024 one at a time.
    Just below and above a multiple of 1 024 workgroups with one part per node (1 025, 2 047, 2 049 nodes), with two (1 022, 1 024, 1 026 and
    2 046 workgroups) and with three (1 023 and 1 029), where a run begins and ends inside a node."""
    test_mp_edge_backward_of_four_edges_per_step(cabi, case)


@pytest.mark.parametrize("case", [(600, 4, 192, 0.0, 41, 256, 70), (600, 6, 192, 0.0, 42, 256, 70), (700, 2, 224, 0.0, 43, 256, 66),
                                  (700, 4, 224, 0.0, 44, 300, 66), (1537, 9, 224, 0.0, 45, 256, 0), (1536, 9, 224, 0.0, 46, 256, 0),
                                  (2048, 6, 224, 0.1, 47, 512, 130), (2049, 4, 224, 0.0, 48, 256, 0), (2049, 6, 224, 0.0, 49, 256, 0),
                                  (500, 51, 224, 0.0, 50, 256, 0)],
                         ids=lambda c: "N%d_d%d_C%d_k%d" % (c[0], c[1], c[2], c[5]))
def test_mp_edge_backward_on_both_sides_of_the_line(cabi, case):
    """The sizes between which 192 and 224 channels change from groups of four edges to an edge per wave: edges per node, and at 224
    a round of waves, whole or in parts."""
    nnodes, C, E = case[0], case[2], _edge_case(*case)[0].numel()
    per_node = {(600, 4): 5, (600, 6): 5, (700, 2): 2.5, (700, 4): 2.5, (2049, 4): 5, (2049, 6): 5}.get(case[:2])
    assert per_node is None or (E < per_node * nnodes) == (case[1] < per_node)
    test_mp_edge_backward_of_four_edges_per_step(cabi, case)


@pytest.mark.parametrize("nnodes,C", [(1750, 96), (1400, 128), (1000, 160), (900, 192), (700, 256)])
def test_forward_from_vectors_is_no_less_precise_than_from_harmonics_and_lengths(cabi, nnodes, C):
    """From vectors these sizes run on the kernel that forms length and direction from one reciprocal square root; given
    harmonics and lengths they run with one wave per node.  The lengths handed over are those the other kernels form from
    fp32 vectors: squares added up by fma, a correctly rounded square root.  Over the two million components of the message
    the relative error against fp64 is a number with three firm digits, so two per cent are allowed."""
    snd, rcv, X, vec, knots, coeffs, h = _edge_case(nnodes, 52, C, 0.0, 31)
    X = X.float().double()
    r2 = torch.zeros(vec.shape[0], dtype=torch.float64)
    for k in range(3):
        r2 = (r2 + vec[:, k] ** 2).float().double()  # the product is exact in fp64: one rounding, as in an fma
    r = r2.sqrt().float()
    live = (r <= 5.0) & (snd >= 0) & (snd < nnodes)
    R = O.spline_eval(vec[live].norm(dim=1), knots, coeffs, h, 5.0).view(-1, 4, C)
    ref = O.mp_forward(X, O.spherical_harmonics(vec[live]), R, snd[live], rcv[live], nnodes)
    d = lambda t: t.float().cuda()
    fo = cabi.first_occurences(rcv.cuda(), nnodes)
    a = cabi.mp_edge_forward(d(X), d(vec), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    b = cabi.mp_spline_forward(d(X), cabi.sh_forward(d(vec)), r.cuda(), d(knots), d(coeffs), h, 5.0, snd.cuda(), fo, nnodes)
    error_a, error_b = (float((t.double().cpu() - ref).norm() / ref.norm()) for t in (a, b))
    print("C=%d from vectors %.3e, from harmonics and lengths %.3e" % (C, error_a, error_b), flush=True)
    assert error_a <= 1.02 * error_b


@pytest.mark.parametrize("case", [(1, 3, 160, 0.0, 61, 256, 0), (40, 1, 160, 0.3, 62, 200, 0), (60, 3, 160, 0.0, 63, 256, 70), (60, 4, 160, 0.0, 64, 256, 0), (200, 13, 160, 0.1, 65, 600, 130),
                                  (1024, 6, 160, 0.0, 66, 256, 0), (2048, 2, 160, 0.2, 67, 256, 0), (2049, 2, 160, 0.2, 68, 256, 0)],
                         ids=lambda c: "N%d_d%d_k%d" % (c[0], c[1], c[5]))
def test_mp_forward_of_five_channels_per_lane(cabi, case):
    """160 channels with few nodes: one part and several, parts without an edge, one round of waves and one node more; from vectors and from
    lengths and harmonics."""
    test_mp_edge_forward_many_nodes(cabi, case)
    test_mp_spline_forward_backward(cabi, case[:5])
