"""Edges of how the step's work is split over launches and workgroups: lists
longer than one launch's threads, tiles smaller than the default and grids on
either side of a rule's line. Needs an MI355X."""
import numpy as np
import pytest

from method_amd import engine as eng
from method_amd import initdata as idt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 40])
def test_retry_of_every_cell_clears_its_list(n):
    """Every cell fails from a guess at |v| = 1 and is recovered by the retry
    from rest: fewer cells than one workgroup's threads, and more than all the
    threads of the launch (64 x 256). A second call finds an empty list, so it
    counts the same failures. The root is found to the Newton tolerance 1e-12,
    which the recovery divides by p's share of the energy, above 1e-2 here."""
    g = idt.kh3d_grid(n)
    p0 = idt.kh_prims(g, seed=3)
    print(f"gpu: retry of all cells, {n}^3", flush=True)
    with eng.Engine(eng.Config(n, n, n, -0.5, 0.5, -1.0, 1.0, 0.0, 1.0, quirks=0)) as e:
        e.set_prims(p0)
        true = e.download()[1]
        bad = true.copy()
        bad[1], bad[2], bad[3] = 1.0, 0.0, 0.0
        for call in range(2):
            e.upload(prims=bad)
            rc, st = e.c2p()
            got = e.download()[1]
            assert rc == n**3 and st["failures"] == n**3 and st["fallbacks"] == 0, call
            assert np.abs(got - true).max() <= 1e-10
