"""Device neighbour list (cm_neighbour_list_count / _fill) against the brute-force oracle: identical integer output."""
import numpy as np
import pytest
import torch

from oracle import ops as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _device_list(pos, cell, pbc, cutoff, max_cells=0):
    from cuda_mace import _cabi as cabi

    p = torch.tensor(pos, dtype=torch.float64, device=DEV).reshape(-1, 3)
    c = None if cell is None else torch.tensor(cell, dtype=torch.float64, device=DEV)
    ri, rj, S = cabi.neighbour_list(p, c, pbc, cutoff, max_cells)
    return np.stack([ri.cpu().numpy(), rj.cpu().numpy()]).astype(np.int64), S.cpu().numpy().astype(np.int64)


def _check(pos, cell, pbc, cutoff, max_cells=0):
    ei, S = _device_list(pos, cell, pbc, cutoff, max_cells)
    ei_ref, S_ref = O.neighbour_list(pos, cell, pbc, cutoff)
    assert ei.shape == ei_ref.shape, (ei.shape, ei_ref.shape)
    assert np.array_equal(ei, ei_ref)
    assert np.array_equal(S, S_ref)
    return ei, S


CASES = {
    "cluster": dict(n=60, lo=0.0, hi=9.0, cell=None, pbc=(0, 0, 0), cutoff=5.0),
    "cluster_with_unused_cell": dict(n=40, lo=-4.0, hi=7.0, cell=np.eye(3) * 30.0, pbc=(0, 0, 0), cutoff=4.0),
    "cubic": dict(n=300, lo=0.0, hi=14.0, cell=np.eye(3) * 14.0, pbc=(1, 1, 1), cutoff=5.0),
    "cubic_unwrapped": dict(n=200, lo=-40.0, hi=55.0, cell=np.eye(3) * 13.0, pbc=(1, 1, 1), cutoff=5.0),
    "orthorhombic_slab": dict(n=150, lo=0.0, hi=11.0, cell=np.diag([11.0, 16.0, 40.0]), pbc=(1, 1, 0), cutoff=5.0),
    "triclinic": dict(n=120, lo=-2.0, hi=15.0, cell=np.array([[12.0, 0, 0], [3.0, 11.0, 0], [-2.0, 4.0, 13.0]]),
                      pbc=(1, 1, 1), cutoff=5.0),
    "small_cell_many_images": dict(n=7, lo=-3.0, hi=8.0, cell=np.array([[4.0, 0, 0], [1.0, 3.5, 0], [0.5, 0.7, 4.2]]),
                                   pbc=(1, 1, 1), cutoff=5.0),
    "wire": dict(n=25, lo=0.0, hi=6.0, cell=np.array([[0.0, 0, 3.1], [7.0, 0.0, 0], [0.0, 9.0, 0.0]]), pbc=(1, 0, 0),
                 cutoff=4.5),
    "left_handed_cell": dict(n=50, lo=0.0, hi=12.0, cell=np.array([[0, 12.0, 0], [12.5, 0, 0], [0, 0, 13.0]]),
                             pbc=(1, 1, 1), cutoff=5.0),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_neighbour_list_matches_brute_force(cabi, name):
    k = CASES[name]
    rng = np.random.default_rng(sorted(CASES).index(name))
    pos = rng.uniform(k["lo"], k["hi"], (k["n"], 3))
    ei, S = _check(pos, k["cell"], k["pbc"], k["cutoff"])
    assert ei.shape[1] > 0
    assert np.all(np.diff(ei[0]) >= 0)
    # every pair appears with its reverse
    fwd = {tuple(r) for r in np.concatenate([ei.T, S], axis=1)}
    assert fwd == {(j, i, -a, -b, -c) for (i, j, a, b, c) in fwd}


def test_bin_cap_does_not_change_the_list(cabi):
    rng = np.random.default_rng(5)
    pos = rng.uniform(0, 30.0, (400, 3))
    cell = np.eye(3) * 30.0
    base = _device_list(pos, cell, (1, 1, 1), 4.0)
    for cap in (1, 2, 7, 50):
        got = _device_list(pos, cell, (1, 1, 1), 4.0, max_cells=cap)
        assert np.array_equal(got[0], base[0]) and np.array_equal(got[1], base[1])
    ref = O.neighbour_list(pos, cell, (1, 1, 1), 4.0)
    assert np.array_equal(base[0], ref[0]) and np.array_equal(base[1], ref[1])


def test_degenerate_inputs(cabi):
    from cuda_mace import _cabi as cabi_mod

    # no atoms, one atom without and with self-images, two atoms out of range, coincident coordinates along an axis
    ei, S = _device_list(np.zeros((0, 3)), None, (0, 0, 0), 5.0)
    assert ei.shape == (2, 0) and S.shape == (0, 3)
    ei, S = _device_list(np.array([[1.0, 2.0, 3.0]]), None, (0, 0, 0), 5.0)
    assert ei.shape == (2, 0)
    _check(np.array([[1.0, 2.0, 3.0]]), np.eye(3) * 3.0, (1, 1, 1), 5.0)
    ei, _ = _device_list(np.array([[0.0, 0, 0], [9.0, 0, 0]]), None, (0, 0, 0), 5.0)
    assert ei.shape == (2, 0)
    planar = np.random.default_rng(3).uniform(0, 8.0, (30, 3))
    planar[:, 2] = 1.25
    _check(planar, None, (0, 0, 0), 3.0)
    with pytest.raises(cabi_mod.CudaMaceError, match="singular"):
        _device_list(planar, np.zeros((3, 3)), (1, 1, 1), 3.0)
    with pytest.raises(cabi_mod.CudaMaceError):
        _device_list(planar, None, (0, 0, 0), -1.0)


GRAPH_CASES = {
    # atoms, box edge (None: no cell), periodic axes, cutoff
    "one_atom": (1, None, (0, 0, 0), 5.0),
    "no_pairs": (5, None, (0, 0, 0), 0.01),
    "one_atom_images": (1, 3.0, (1, 1, 1), 5.0),
    "few_atoms_many_images": (7, 3.7, (1, 1, 1), 6.0),
    "wave_edges": (65, 9.0, (1, 0, 1), 5.0),
    "box": (1000, 21.5, (1, 1, 1), 5.0),
    "dense": (900, 9.0, (1, 1, 1), 5.5),          # more than 512 neighbours: one wave per workgroup
    "denser": (400, 3.0, (0, 0, 0), 6.0),
    "about_two_per_lane": (260, 8.6, (1, 1, 1), 4.4),  # 128 neighbours and a few less or more: in order through LDS, or by rank
    "thinner_than_the_reach": (3, 1.3, (1, 1, 1), 6.0),
    "one_workgroup_most": (4096, 34.5, (1, 1, 1), 4.0),
    "several_launches": (4097, 34.5, (1, 1, 0), 4.0),
    "many_32768": (32768, 69.0, (1, 1, 1), 4.0),
    "many_32769": (32769, 69.0, (1, 1, 0), 4.0),
    "bins_halved": (40000, 126.0, (1, 1, 1), 5.0),  # 45 bins in reach, about 58 candidates: one set of 64 of each
    "bins_halved_dense": (3000, 60.0, (1, 1, 1), 10.0),
}


def _search(cabi_mod, p, c, pbc, cutoff):
    """cm_neighbour_list_search as the header has it: the workspace, offsets [N + 1], status [1] and max_degree [1], left on the device."""
    n = p.shape[0]
    max_cells = max(1, n)
    size = cabi_mod.lib.cm_neighbour_list_workspace(n, max_cells)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    offsets, numbers = torch.full((n + 1,), -7, dtype=torch.int32, device=DEV), torch.full((2,), -7, dtype=torch.int32, device=DEV)
    cabi_mod._check(cabi_mod.lib.cm_neighbour_list_search(p.data_ptr(), c.data_ptr() if c is not None else None, *(int(b) for b in pbc), cutoff, n, max_cells,
                                                          ws.data_ptr(), size, offsets.data_ptr(), numbers.data_ptr(), numbers.data_ptr() + 4,
                                                          cabi_mod._stream()))
    return ws, max_cells, offsets, numbers


@pytest.mark.parametrize("name", list(GRAPH_CASES))
def test_graph_of_a_list(cabi, name):
    """cm_neighbour_list_search_counts / _graph: the pairs of cm_neighbour_list_count / _fill (held against the oracle above; against
    the oracle here too where it is quick), the same in int64 and fp64, shifts, CSR offsets, batch and ptr;
    cm_neighbour_list_search, which leaves the same numbers on the device; and cm_symmetric_sender_view against the stable sort by sender."""
    from cuda_mace import _cabi as cabi_mod
    from cuda_mace.utils.neighbour_list import shifts_from_unit_shifts

    n, box, pbc, cutoff = GRAPH_CASES[name]
    rng = np.random.default_rng(len(name))
    pos = rng.uniform(-1.0, (box or 6.0) * 1.1, (n, 3))
    cell = None if box is None else np.eye(3) * box + np.array([[0, 0, 0], [0.3, 0, 0], [0.1, -0.2, 0]])
    p = torch.tensor(pos, dtype=torch.float64, device=DEV)
    c = None if cell is None else torch.tensor(cell, dtype=torch.float64, device=DEV)
    if name in ("one_atom_images", "few_atoms_many_images", "wave_edges", "thinner_than_the_reach"):
        _check(pos, cell, pbc, cutoff)
    ri, rj, S = cabi_mod.neighbour_list(p, c, pbc, cutoff)
    g = cabi_mod.neighbour_graph(p, c, pbc, cutoff)
    print(name, "pairs", ri.numel(), flush=True)
    assert torch.equal(g["row_i"], ri) and torch.equal(g["row_j"], rj)
    assert torch.equal(g["edge_index"], torch.stack([ri, rj]).long())
    assert torch.equal(g["unit_shifts"], S.double())
    assert torch.equal(g["shifts"], shifts_from_unit_shifts(S, c))
    assert torch.equal(g["first_occ"], cabi_mod.first_occurences(ri, n))
    assert g["batch"].tolist() == [0] * n and g["ptr"].tolist() == [0, n] and g["ptr32"].tolist() == [0, n]
    perm, off = cabi_mod.stable_key_sort(rj, n)
    assert torch.equal(g["offsets"], off)
    _, _, offsets, numbers = _search(cabi_mod, p, c, pbc, cutoff)
    assert torch.equal(offsets, off) and numbers.tolist() == [0, int((off[1:] - off[:-1]).max())]
    assert torch.equal(cabi_mod.symmetric_sender_view(g["row_i"], g["row_j"], g["unit_shifts"], g["first_occ"], n), perm)


@pytest.mark.parametrize("n,box,cutoff", [(300, 12.0, 4.0), (700, 9.0, 5.5), (4097, 34.5, 4.0)])
def test_graph_into_fewer_places_than_pairs(cabi, n, box, cutoff):
    """cm_neighbour_list_graph with `nedges` below the number of pairs: the segments that end before it come out whole, nothing is written
    behind it, and segments that begin behind it (their room is negative) touch nothing."""
    from cuda_mace import _cabi as cabi_mod

    p = torch.tensor(np.random.default_rng(n).uniform(0.0, box, (n, 3)), dtype=torch.float64, device=DEV)
    c = torch.eye(3, dtype=torch.float64, device=DEV) * box
    whole = cabi_mod.neighbour_graph(p, c, (True,) * 3, cutoff)
    ws, max_cells, offsets, numbers = _search(cabi_mod, p, c, (True,) * 3, cutoff)
    pairs = whole["row_i"].numel()
    for nedges in (pairs - 1, pairs // 2 + 1, 3):
        guard = 64
        ri, rj = (torch.full((nedges + guard,), -5, dtype=torch.int32, device=DEV) for _ in range(2))
        index = torch.full((2 * nedges + guard,), -5, dtype=torch.int64, device=DEV)
        S, shifts = (torch.full((nedges + guard, 3), -5.0, dtype=torch.float64, device=DEV) for _ in range(2))
        fo = torch.empty(2 * n, dtype=torch.int32, device=DEV)
        cabi_mod._check(cabi_mod.lib.cm_neighbour_list_graph(cutoff, n, max_cells, ws.data_ptr(), offsets.data_ptr(), nedges, int(numbers[1]), ri.data_ptr(),
                                                             rj.data_ptr(), index.data_ptr(), S.data_ptr(), shifts.data_ptr(), fo.data_ptr(), None, None, None,
                                                             cabi_mod._stream()))
        inside = int(offsets[offsets <= nedges].max())  # pairs of segments that fit
        assert torch.equal(ri[:inside], whole["row_i"][:inside]) and torch.equal(rj[:inside], whole["row_j"][:inside])
        assert torch.equal(index[:inside], whole["edge_index"][0, :inside]) and torch.equal(index[nedges:nedges + inside], whole["edge_index"][1, :inside])
        assert torch.equal(S[:inside], whole["unit_shifts"][:inside]) and torch.equal(shifts[:inside], whole["shifts"][:inside])
        assert bool((ri[nedges:] == -5).all()) and bool((rj[nedges:] == -5).all()) and bool((index[2 * nedges:] == -5).all())
        assert bool((S[nedges:] == -5).all()) and bool((shifts[nedges:] == -5).all())
        assert torch.equal(fo, whole["first_occ"])


@pytest.mark.parametrize("n", [0, 1, 300, 4097])
@pytest.mark.parametrize("fills", [0, 60])
def test_counts_reach_a_waiting_host(cabi, n, fills):
    """The numbers the host polls for: with the stream idle, and with some ten milliseconds of fills of 1 GiB ahead of the
    search (the host then gives up polling and waits for the stream), against the entry that leaves them on the device."""
    from cuda_mace import _cabi as cabi_mod

    rng = np.random.default_rng(n)
    p = torch.tensor(rng.uniform(0.0, 1.0 + 3.0 * n ** (1.0 / 3.0), (n, 3)), dtype=torch.float64, device=DEV)
    ri, rj, _ = cabi_mod.neighbour_list(p, None, (False,) * 3, 4.0)
    ahead = torch.empty(1 << 28 if fills else 0, device=DEV)
    torch.cuda.synchronize()
    for _ in range(fills):
        ahead.fill_(1.0)
    g = cabi_mod.neighbour_graph(p, None, (False,) * 3, 4.0)
    assert torch.equal(g["row_i"], ri) and torch.equal(g["row_j"], rj)
    assert g["offsets"].shape == (n + 1,) and int(g["offsets"][-1]) == ri.numel()
    assert g["ptr"].tolist() == [0, n]


@pytest.mark.parametrize("satellites", [4097, 8191, 8192, 8300])
def test_atom_with_thousands_of_neighbours(cabi, satellites):
    """One atom in the middle of a shell of others, all within its cutoff: up to 8 192 neighbours the last pass keeps them in
    LDS (128 KB), beyond that the list comes from count and fill.  Against the accept test evaluated in numpy."""
    from cuda_mace import _cabi as cabi_mod
    from cuda_mace.utils.neighbour_list import _search

    rng = np.random.default_rng(satellites)
    v = rng.normal(size=(satellites, 3))
    pos = np.concatenate([v / np.linalg.norm(v, axis=1, keepdims=True) * rng.uniform(4.0, 4.9, (satellites, 1)), np.zeros((1, 3))])
    n, cutoff = satellites + 1, 5.0
    rows = []
    for i in range(n):
        d = pos - pos[i]
        near = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2] < cutoff * cutoff
        near[i] = False
        rows.append(np.nonzero(near)[0])
    assert len(rows[-1]) == satellites
    want = np.stack([np.repeat(np.arange(n), [len(r) for r in rows]), np.concatenate(rows)])
    p = torch.tensor(pos, dtype=torch.float64, device=DEV)
    g = cabi_mod.neighbour_graph(p, None, (0, 0, 0), cutoff)
    assert (g is None) == (satellites > 8192)
    edge_index, shifts, unit_shifts = _search(p, cutoff, None, None)[:3]
    assert np.array_equal(edge_index.cpu().numpy(), want)
    assert float(shifts.abs().max()) == 0.0 and float(unit_shifts.abs().max()) == 0.0
    if g is not None:
        assert torch.equal(g["edge_index"], edge_index)
        assert torch.equal(g["first_occ"], cabi_mod.first_occurences(g["row_i"], n))


def test_full_size_box_equals_host_list_and_feeds_the_model(cabi):
    """25 000 atoms: the device list equals the host list of the benchmark generator entry for entry, and the model gives
    bit-identical energy and forces from either."""
    from cuda_mace.models import OptimizedInvariantMACE, SyntheticInvariantMACE
    from cuda_mace.utils.neighbour_list import get_neighborhood
    from cuda_mace.utils.synthetic import make_system, to_device

    data = make_system(25000, 10, seed=0)
    dev = to_device(data, DEV)
    edge_index, shifts, unit_shifts, cell = get_neighborhood(dev["positions"], 5.0, (True, True, True), dev["cell"])
    assert torch.equal(edge_index.cpu(), data["edge_index"])
    assert torch.equal(unit_shifts.cpu(), data["unit_shifts"])
    assert torch.allclose(shifts.cpu(), data["shifts"], rtol=0, atol=1e-12)
    avg = data["edge_index"].shape[1] / 25000
    model = OptimizedInvariantMACE(SyntheticInvariantMACE(channels=32, atomic_numbers=tuple(range(1, 11)), avg_num_neighbors=avg,
                                                          seed=1), device=DEV)
    out_host = model(dict(dev))
    dev2 = dict(to_device(data, DEV))
    dev2.update(edge_index=edge_index, shifts=shifts, unit_shifts=unit_shifts)
    out_dev = model(dev2)
    assert torch.equal(out_host["energy"], out_dev["energy"])
    assert torch.equal(out_host["forces"], out_dev["forces"])


@pytest.mark.parametrize("n", [0, 1, 63, 1000, 300_001])
def test_max_displacement(cabi, n):
    """cm_max_displacement against the same maximum taken by torch in fp64 (bit-exact: squares and sums of three terms,
    left to right without fused multiply-adds, then a maximum); a NaN coordinate gives +inf."""
    g = torch.Generator(device="cuda").manual_seed(n)
    ref = 20.0 * torch.rand(n, 3, device="cuda", dtype=torch.float64, generator=g)
    pos = ref + 0.1 * torch.randn(n, 3, device="cuda", dtype=torch.float64, generator=g)
    got = cabi.max_displacement(pos, ref)
    d = pos - ref
    want = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]).max() if n else torch.zeros((), dtype=torch.float64)
    assert got.shape == (1,) and float(got[0]) == float(want)
    if n:
        pos[n // 2, 1] = float("nan")
        assert float(cabi.max_displacement(pos, ref, out=got)[0]) == float("inf")


@pytest.mark.parametrize("case", ["periodic_skin", "batch", "exact_list", "cluster", "no_edges", "headline"])
def test_graph_prepare_matches_the_host_restatement(cabi, case):
    """cm_graph_prepare (relabelled atoms, re-sorted pairs with the skin shell last, CSR offsets, sender-sorted view) entry
    for entry against a numpy restatement with library sorts, and its derived structures against the index oracles."""
    from cuda_mace.utils.synthetic import collate, make_system
    from oracle import ops as O
    from tests.util import spatial_order_reference

    r_max = 5.0
    if case == "periodic_skin":
        data = make_system(400, 4, seed=5, density=0.1, cutoff=5.6)
    elif case == "batch":
        data = collate([make_system(n, 4, seed=20 + k, density=0.1, cutoff=5.2) for k, n in enumerate((150, 230, 120))])
    elif case == "exact_list":
        data = make_system(300, 4, seed=6, density=0.1)
    elif case == "cluster":
        data = make_system(21, 4, seed=0, density=None, cluster_box=8.0)
    elif case == "no_edges":
        data = make_system(12, 4, seed=2, density=None, cluster_box=60.0, min_dist=8.0)
        assert data["edge_index"].shape[1] == 0
    else:
        data = make_system(25000, 10, seed=0, density=0.1, cutoff=5.5)
    N, E = data["positions"].shape[0], data["edge_index"].shape[1]
    ngraphs = int(data["ptr"].numel()) - 1
    print("graph_prepare", case, N, E, ngraphs, flush=True)
    dev = lambda t: t.to("cuda").contiguous()  # noqa: E731
    bins = 64 if ngraphs == 1 else 16
    got = cabi.graph_prepare(dev(data["positions"].double()), dev(data["edge_index"][0].int()), dev(data["edge_index"][1].int()),
                             dev(data["shifts"].double()), None if ngraphs == 1 else dev(data["batch"].int()), ngraphs, r_max, bins)
    perm, inverse, rcv, snd, order = spatial_order_reference(data["positions"], data["batch"], data["edge_index"], data["shifts"],
                                                             r_max, bins)
    eq = lambda name, want: np.testing.assert_array_equal(got[name].cpu().numpy(), want, err_msg=name)  # noqa: E731
    eq("node_perm", perm)
    eq("node_inverse", inverse)
    eq("receiver", rcv)
    eq("sender", snd)
    eq("edge_perm", order)
    assert torch.equal(got["shifts"].cpu(), data["shifts"].double()[torch.from_numpy(order)])
    assert torch.equal(got["first_occ"].cpu(), O.first_occurences(torch.from_numpy(rcv).int(), N))
    sperm, soff = O.stable_key_sort(torch.from_numpy(snd).int(), N)
    assert torch.equal(got["sender_perm"].cpu(), sperm) and torch.equal(got["sender_offsets"].cpu(), soff)
    if E:
        # every receiver's pairs beyond the cutoff come last
        v = data["positions"][data["edge_index"][1]] - data["positions"][data["edge_index"][0]] + data["shifts"]
        beyond = (v.norm(dim=1) > r_max)[torch.from_numpy(order)]
        fo = got["first_occ"].cpu()
        for n in (0, N // 2, N - 1):
            seg = beyond[fo[n]:fo[N + n]]
            assert bool((seg[1:] >= seg[:-1]).all())


@pytest.mark.parametrize("degrees", [(512, 513, 0, 64, 65, 1), (1500, 2), (1024, 768, 1025)])
def test_graph_prepare_long_segments(cabi, degrees):
    """cm_graph_prepare where a segment or a sender's bucket is longer than what a wave keeps on chip (512 keys, 256 pairs), on a
    list in which a pair has no reverse and names of atoms out of range occur, against the numpy restatement."""
    from oracle import ops as O
    from tests.util import spatial_order_reference

    g = torch.Generator().manual_seed(len(degrees))
    N = len(degrees) + 3  # the last three atoms receive nothing
    pos = 4.0 * torch.rand(N, 3, generator=g, dtype=torch.float64)
    rcv = torch.repeat_interleave(torch.arange(len(degrees)), torch.tensor(degrees))
    E = rcv.numel()
    snd = torch.where(torch.rand(E, generator=g) < 0.7, torch.tensor(N - 1), torch.randint(0, N, (E,), generator=g))
    shifts = 2.0 * torch.randint(-2, 3, (E, 3), generator=g).double()
    got = cabi.graph_prepare(pos.cuda(), rcv.int().cuda(), snd.int().cuda(), shifts.cuda(), None, 1, 5.0, 8)
    perm, inverse, new_rcv, new_snd, order = spatial_order_reference(pos, torch.zeros(N, dtype=torch.int64), torch.stack([rcv, snd]), shifts, 5.0, 8)
    for name, want in (("node_perm", perm), ("node_inverse", inverse), ("receiver", new_rcv), ("sender", new_snd), ("edge_perm", order)):
        np.testing.assert_array_equal(got[name].cpu().numpy(), want, err_msg=name)
    sperm, soff = O.stable_key_sort(torch.from_numpy(new_snd).int(), N)
    assert torch.equal(got["sender_perm"].cpu(), sperm) and torch.equal(got["sender_offsets"].cpu(), soff)
    # names out of range: of atom j a pair counts for no sender; the views stay a function of the pairs that count
    snd[::7] = N + 5
    got = cabi.graph_prepare(pos.cuda(), rcv.int().cuda(), snd.int().cuda(), shifts.cuda(), None, 1, 5.0, 8)
    new_snd = got["sender"].cpu()
    counted = int(((snd >= 0) & (snd < N)).sum())
    want = torch.sort(new_snd, stable=True).indices[:counted]
    assert int(got["sender_offsets"][-1]) == counted and torch.equal(got["sender_perm"].cpu()[:counted].long(), want)


@pytest.mark.parametrize("n,ngraphs,bins", [(4095, 1, 1), (4096, 1, 1), (4095, 1, 4), (4096, 1, 4), (4160, 64, 1), (4160, 65, 1), (20000, 2, 3), (70000, 1, 2)])
def test_graph_prepare_few_bins(cabi, n, ngraphs, bins):
    """Few bins of many atoms, on both sides of each line of the rule for them (64 keys, 4 096 atoms), counted and of a list that
    is known, against the numpy restatement."""
    from oracle import ops as O
    from tests.util import spatial_order_reference

    g = torch.Generator().manual_seed(n + bins)
    pos = 30.0 * torch.rand(n, 3, generator=g, dtype=torch.float64)
    batch = torch.arange(n) * ngraphs // n
    i = torch.arange(n)
    rcv = torch.cat([i, i]).sort().values  # two pairs per atom, each with its reverse
    snd = torch.stack([(i - 1) % n, (i + 1) % n], dim=1).sort(dim=1).values.reshape(-1)
    shifts = torch.zeros(2 * n, 3, dtype=torch.float64)
    perm, inverse, new_rcv, new_snd, order = spatial_order_reference(pos, batch, torch.stack([rcv, snd]), shifts, 5.0, bins)
    sperm, soff = O.stable_key_sort(torch.from_numpy(new_snd).int(), n)
    first_occ = O.first_occurences(rcv.int(), n).cuda()
    for known in (None, first_occ):
        got = cabi.graph_prepare(pos.cuda(), rcv.int().cuda(), snd.int().cuda(), shifts.cuda(), batch.int().cuda() if ngraphs > 1 else None, ngraphs, 5.0,
                                 bins, symmetric_first_occ=known)
        for name, want in (("node_perm", perm), ("node_inverse", inverse), ("receiver", new_rcv), ("sender", new_snd), ("edge_perm", order)):
            np.testing.assert_array_equal(got[name].cpu().numpy(), want, err_msg=name)
        assert torch.equal(got["sender_perm"].cpu(), sperm) and torch.equal(got["sender_offsets"].cpu(), soff)


@pytest.mark.parametrize("sent,N,degree", [(256, 40, 20), (257, 40, 20), (20000, 3000, 100)])
def test_graph_prepare_long_buckets(cabi, sent, N, degree):
    """Some atoms send exactly `sent` pairs: as many as a wave ranks on chip, one more, and more than the slots that one round of
    threads takes, against the numpy restatement; and with names out of range, whose slots no pair takes."""
    from oracle import ops as O
    from tests.util import spatial_order_reference

    g = torch.Generator().manual_seed(sent)
    pos = 15.0 * torch.rand(N, 3, generator=g, dtype=torch.float64)
    E = N * degree
    rcv = torch.arange(N).repeat_interleave(degree)
    snd = torch.randint(3, N, (E,), generator=g)
    snd[torch.randperm(E, generator=g)[:2 * sent]] = torch.tensor([0, 2]).repeat(sent)
    shifts = torch.zeros(E, 3, dtype=torch.float64)
    got = cabi.graph_prepare(pos.cuda(), rcv.int().cuda(), snd.int().cuda(), shifts.cuda(), None, 1, 5.0, 6)
    _, inverse, new_rcv, new_snd, order = spatial_order_reference(pos, torch.zeros(N, dtype=torch.int64), torch.stack([rcv, snd]), shifts, 5.0, 6)
    for name, want in (("receiver", new_rcv), ("sender", new_snd), ("edge_perm", order)):
        np.testing.assert_array_equal(got[name].cpu().numpy(), want, err_msg=name)
    sperm, soff = O.stable_key_sort(torch.from_numpy(new_snd).int(), N)
    assert torch.equal(got["sender_perm"].cpu(), sperm) and torch.equal(got["sender_offsets"].cpu(), soff)
    lost = torch.randperm(E, generator=g)[:50]
    snd[lost] = N + 1
    got = cabi.graph_prepare(pos.cuda(), rcv.int().cuda(), snd.int().cuda(), shifts.cuda(), None, 1, 5.0, 6)
    want = torch.sort(got["sender"].cpu(), stable=True).indices[:E - 50]
    assert int(got["sender_offsets"][-1]) == E - 50 and torch.equal(got["sender_perm"].cpu()[:E - 50].long(), want)


@pytest.mark.parametrize("n,ne", [(0, 3), (1, 1), (255, 2), (256, 63), (257, 10), (5000, 4)])
def test_element_groups_and_gathered_rows(cabi, n, ne):
    """Both groupings against the sorts they stand for, with rows that hold no one, two ones or other values and with types out
    of range; rows of 1 to 40 bytes gathered by a permutation against torch, all equal to the bit."""
    g = torch.Generator().manual_seed(n + ne)
    types = torch.randint(-1, ne + 1, (n,), generator=g).int().cuda()
    one_hot = torch.randint(0, 3, (n, ne), generator=g).float().cuda()
    by_type, by_column = cabi.element_groups(types, one_hot)
    mask = one_hot == 1
    column = torch.where(mask.any(dim=1), mask.to(torch.int8).argmax(dim=1), ne).int() if n else types
    for got, keys, nkeys in ((by_type, types, ne), (by_column, column, ne + 1)):
        perm, offsets = cabi.stable_key_sort(keys, nkeys)
        count = int(offsets[-1])
        assert torch.equal(got[1], offsets) and torch.equal(got[0][:count], perm[:count])
    perm = torch.randperm(n, generator=g).int().cuda()
    arrays = [torch.randint(0, 127, (n, w), generator=g, dtype=torch.int8).cuda() for w in (1, 4, 8, 16, 31, 40)] + [types, one_hot.double().T.contiguous().T]
    for got, want in zip(cabi.gather_rows(perm, *arrays), arrays):
        assert torch.equal(got, want.index_select(0, perm))
    more = [torch.cat([a, a[:1], a]) for a in arrays]  # rows behind the first n
    for got, want in zip(cabi.gather_rows(perm, *more), arrays):
        assert torch.equal(got, want.index_select(0, perm))
    if n:
        with pytest.raises(cabi.CudaMaceError):
            cabi.gather_rows(perm, types[:-1])


@pytest.mark.parametrize("n,pbc", [(1, False), (40, True), (700, True), (9000, False)])
def test_symmetric_list_is_prepared_alike(cabi, n, pbc):
    """What cm_graph_prepare_symmetric makes of a list of the device search, whose pairs it does not count, is to the bit what
    cm_graph_prepare makes of it."""
    from cuda_mace.utils.neighbour_list import neighbour_data

    g = torch.Generator().manual_seed(n)
    box = (n / 0.08) ** (1.0 / 3.0) + 2.0
    pos = (box * torch.rand(n, 3, generator=g, dtype=torch.float64)).cuda()
    cell = torch.eye(3, dtype=torch.float64, device="cuda") * box if pbc else None
    data = neighbour_data(pos, torch.ones(n, 1, dtype=torch.float64, device="cuda"), 5.5, (pbc,) * 3, cell)
    row_i, row_j = (r.contiguous() for r in data["edge_index"].int())
    first_occ = cabi.first_occurences(row_i, n)
    args = (pos, row_i, row_j, data["shifts"], None, 1, 5.0, 20)
    plain, known = cabi.graph_prepare(*args), cabi.graph_prepare(*args, symmetric_first_occ=first_occ)
    for name in plain:
        assert torch.equal(plain[name], known[name]), name


@pytest.mark.parametrize("case,known", [("rows_in_turn", True), ("rows_in_turn", False), ("all_ranges_whole", True), ("sums_beyond_32_bits", True)])
def test_graph_prepare_of_unsorted_rows_stays_within_the_list(cabi, case, known):
    """Rows that are not sorted, or a CSR whose ranges overlap, give a view that means nothing, every index of which lies within
    the list: offsets ascend to at most the number of pairs, and nothing is written behind an output."""
    N, E = {"rows_in_turn": (2, 400), "all_ranges_whole": (70, 300), "sums_beyond_32_bits": (600_000, 4096)}[case]
    print("graph_prepare", case, known, flush=True)
    g = torch.Generator().manual_seed(N)
    pos = (30.0 * torch.rand(N, 3, generator=g, dtype=torch.float64)).cuda()
    row_i = (torch.arange(E) % N).int().cuda()
    row_j = torch.randint(0, N, (E,), generator=g).int().cuda()
    shifts = torch.zeros(E, 3, dtype=torch.float64, device="cuda")
    if case == "rows_in_turn":  # what the two writers of one entry can leave: both ranges all but whole
        csr = torch.tensor([0, 1, E - 1, E], dtype=torch.int32, device="cuda")
    else:
        csr = torch.cat([torch.zeros(N), torch.full((N,), E)]).int().cuda()
    guard, word = 4096, 0x5A5A5A5A
    sizes = {"node_perm": N, "node_inverse": N, "receiver": E, "sender": E, "edge_perm": E, "shifts": 6 * E, "first_occ": 2 * N,
             "sender_perm": E, "sender_offsets": N + 1}
    out = {k: torch.full((n + guard,), word, dtype=torch.int32, device="cuda") for k, n in sizes.items()}
    ws = torch.empty(cabi.lib.cm_graph_prepare_workspace(N, E, 1, 8), dtype=torch.uint8, device="cuda")
    prepare = cabi.lib.cm_graph_prepare_symmetric if known else cabi.lib.cm_graph_prepare
    cabi._check(prepare(pos.data_ptr(), row_i.data_ptr(), row_j.data_ptr(), shifts.data_ptr(), *([csr.data_ptr()] if known else []), None, N, E, 1, 5.0, 8,
                        *[out[k].data_ptr() for k in sizes], ws.data_ptr(), ws.numel(), cabi._stream()))
    torch.cuda.synchronize()
    for k, n in sizes.items():
        assert bool((out[k][n:] == word).all()), "%s: written behind its end" % k
    offsets, first_occ = out["sender_offsets"][:N + 1].cpu(), out["first_occ"][:2 * N].cpu()
    assert int(offsets[0]) == 0 and int(offsets[-1]) <= E and bool((offsets[1:] >= offsets[:-1]).all())
    assert bool(((first_occ >= 0) & (first_occ <= E)).all()) and bool((first_occ[N:] >= first_occ[:N]).all())
    view = out["sender_perm"][:int(offsets[-1])].cpu()
    assert bool(((view >= 0) & (view < E)).all())
