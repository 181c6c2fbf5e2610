"""The multiplicative scheme's autotuner times the program that runs: several views in a launch.

Its time per view update, times the views, is then the time of an iteration: at most twice the measured one (eight views of
48^3: 0.045 ms per update with one view a launch, 0.007 with eight, an iteration 0.055).
"""
import time

import pytest
import torch  # noqa: F401  before the library is loaded: the process then has one HIP runtime, torch's

from mvr import hip
from mvr import synthetic as syn

pytestmark = pytest.mark.gpu


def test_trials_run_the_views_of_a_launch():
    shape, V = (48, 48, 48), 8
    w = syn.small_workload(shape=shape, views=V, k=9, psf_type="INDEPENDENT")
    inp = syn.make_inputs(w)
    d = hip.Decon(shape, V, "INDEPENDENT", "MUL", 6e-4)
    for v in range(V):
        d.set_view(v, inp["imgs"][v], inp["weights"][v], inp["psfs"][v])
    d.init()
    _, ms = d.autotune(1)
    d.run(5)
    t = time.perf_counter()
    d.run(50)
    iteration = (time.perf_counter() - t) * 1e3 / 50
    d.close()
    print(f"autotuner {ms:.4f} ms per view update, iteration of {V} views {iteration:.4f} ms")
    assert ms * V <= 2 * iteration
