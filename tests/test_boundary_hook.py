"""compute_rhs calls the solver's insert_boundary_values, which a subclass may override, whatever conditions are
registered (the native library stands aside: no GPU)."""
from types import SimpleNamespace

from ablate_amd import fv


class Hooked(fv.FiniteVolumeSolver):
    def __init__(self):  # no handle
        self._h, self._ghosts, self.times = None, [], []
        self._rhs = lambda *args: 0

    def _check_tensor(self, t, name):
        pass

    def insert_boundary_values(self, time, U):
        self.times.append(time)


def test_compute_rhs_calls_an_overridden_insert_boundary_values():
    solver, t = Hooked(), SimpleNamespace(data_ptr=lambda: 0)
    solver.compute_rhs(0.25, t, t, stream=0)
    solver.compute_rhs(0.5, t, t, accumulate=True, stream=0)
    assert solver.times == [0.25, 0.5]
