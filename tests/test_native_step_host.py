"""What the binding of the library's one-call step hands to it, checked without a GPU: a stand-in for the library records
the scratch memory of every call."""
import torch

N, E, C = 40, 300, 64


class _Library:
    """cm_mace_step / cm_mace_energy that record their workspace and, while the first call is under way, make another one:
    what a second thread does while ctypes has let go of the interpreter lock, or a second stream while the first one's
    kernels have not run yet."""

    def __init__(self, real):
        self.real, self.calls, self.during = real, [], None

    def __getattr__(self, name):
        return getattr(self.real, name)

    def _call(self, kind, workspace, nbytes):
        self.calls.append((kind, workspace, nbytes))
        during, self.during = self.during, None
        if during is not None:
            during()
        return 0

    def cm_mace_step(self, weights, graph, positions, shifts, workspace, nbytes, *rest):
        return self._call("step", workspace, nbytes)

    def cm_mace_energy(self, weights, graph, positions, shifts, workspace, nbytes, *rest):
        return self._call("energy", workspace, nbytes)


def _step(monkeypatch):
    from cuda_mace import _cabi
    from cuda_mace.ops import native_step

    library = _Library(_cabi.lib)
    monkeypatch.setattr(_cabi, "lib", library)
    monkeypatch.setattr(_cabi, "_stream", lambda: 0)
    monkeypatch.setattr(native_step, "_ptr", lambda t, dtype, name: None if t is None else t.data_ptr())
    step = native_step.NativeStep.__new__(native_step.NativeStep)
    step.weights, step._keep, step.channels, step.nelements, step._streams = native_step._Weights(), [], C, 4, [0]
    graph = native_step._Graph()
    graph.nnodes, graph.nedges, graph.ngraphs = N, E, 1
    handle = native_step._GraphHandle(graph, ())
    pos, shifts = torch.zeros(N, 3, dtype=torch.float64), torch.zeros(E, 3, dtype=torch.float64)
    return library, lambda **kw: step(handle, pos, shifts, **kw)


def test_calls_under_way_at_the_same_time_share_no_scratch_memory(monkeypatch):
    library, evaluate = _step(monkeypatch)
    for outer in (True, False):
        for inner in (True, False):
            library.calls.clear()
            library.during = lambda: evaluate(want_forces=inner)
            evaluate(want_forces=outer)
            (_, a, na), (_, b, nb) = library.calls
            assert a + na <= b or b + nb <= a, "forces %s inside forces %s: both calls write the same memory" % (inner, outer)


def test_energies_alone_take_no_memory_of_the_backward_chain(monkeypatch):
    """Vectors [E, 3] and edge ranges, two [N, 16, C], five [N, C], each rounded up to 256 bytes: nothing of the E x C of
    per-edge gradients or of the gradient rows."""
    library, evaluate = _step(monkeypatch)
    evaluate(want_forces=False)
    evaluate(want_forces=True)
    (kind, _, energy), (_, _, step) = library.calls
    assert kind == "energy"
    assert energy <= 4 * (3 * E + 2 * N + (2 * 16 + 5) * N * C) + 256 * 9
    assert step >= energy + 4 * E * C


def test_forces_take_no_memory_for_edge_records():
    """Edge vectors and their gradients of both layers (9 E floats), the per-edge gradients (E C) and what the nodes need, each
    piece rounded up to 256 bytes: the 16-byte records of the forward lie where the per-edge gradients go afterwards."""
    from cuda_mace import _cabi

    up = lambda nbytes: -(-nbytes // 256) * 256
    for n, e, c in ((N, E, C), (21, 170, 32), (5000, 260574, 96), (1, 70000, 256), (7, 0, 64)):
        pieces = 3 * [12 * e] + [4 * e * c] + 3 * [64 * n * c] + 12 * [4 * n * c] + [8 * n, 48 * n]
        assert _cabi.lib.cm_mace_step_workspace(n, e, c) == sum(up(p) for p in pieces), (n, e, c)
