"""GPU kernels at the sizes where their dispatch changes, against the oracle.

Each test drives one kernel family over the edges of its size classes (lanes
per item, rows per workgroup, rounds of a loop); bars are those of the parity
tests of the same stage.
"""
import numpy as np
import pytest

from sw_reaxff_amd import systems

from .parity import harness
from .test_valence import _gpu_tor_vs_oracle, _gpu_vs_oracle


def lattice(m=8, a=1.7, seed=3):
    """m^3 C/H/O atoms on a shaken cubic lattice: every atom has a dozen or
    more bonds, so centres have up to 135 angles and bonds up to 99
    quadruples (more than one round of a 64-lane group)."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) * a
    x = g + rng.normal(scale=0.05, size=g.shape) + 20.0
    t = rng.integers(1, 4, size=len(x)).astype(np.int32)
    return systems.System(x=x, v=np.zeros_like(x), type=t, tag=np.arange(1, len(x) + 1, dtype=np.int32),
                          elements=["H", "O", "C"], lo=np.zeros(3), hi=np.full(3, 60.0), periodic=False)


GROUP_SYSTEMS = {
    "lattice": lambda: lattice(),                         # items of 1 to more than 64 evaluations
    "cluster21": lambda: systems.cluster(20, seed=1),     # 21 centres, 28 bonds: one or two waves
    "water4200": lambda: systems.water_box(1400, seed=4),   # 4,200 centres: past the 16-lane minimum
    "water30k": lambda: systems.water_box(10000, seed=5),   # 30,000 centres, ~17,600 bonds: single lanes
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(GROUP_SYSTEMS))
def test_gpu_valence_and_torsion_groups(gpu_lib, oracle_lib, ffield, case):
    s = GROUP_SYSTEMS[case]()
    for check in (_gpu_vs_oracle, _gpu_tor_vs_oracle):
        check(oracle_lib, ffield, harness(s, ffield, tol=1e-10), s.elements, s.type, s.tag)
