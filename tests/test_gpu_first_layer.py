"""GPU tests of the first interaction layer evaluated as species-resolved neighbour sums.

The layer's conv-TP input depends on the sender's species only, so the engine sums Y h3 over each
receiver's edges per species and applies the radial MLP's output layer once per node
(`blocks.py:253-274` evaluated in another order).  Rows of every length around the kernels' 16-edge
tiles and 64-edge steps (0, 1, 15, 16, 17, ..., and one longer than the 256 edges whose species the
ordering pass keeps in registers), with one species, several, the largest number the sums take and
one more (which runs the general kernels), against the float64 oracle on the same edge list.
"""

import numpy as np
import pytest

from gpu_helpers import Case
from mace_mlx_amd.systems import System, arch_config

pytestmark = pytest.mark.gpu

ZS = [1, 5, 6, 7, 8, 9, 14, 15, 16, 17]
DEGREES = [0, 1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 0, 270, 5]


def _system(n_species, seed):
    """40 atoms on a jittered 1.6 A grid; receivers 0 .. 18 have DEGREES edges from random senders
    (repeated senders allowed: the list need not be a neighbour list), the rest seven each."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3)[:40]
    pos = 10.0 + 1.6 * g + rng.normal(scale=0.1, size=(40, 3))
    z = np.array(ZS)[np.concatenate([np.arange(n_species), rng.integers(0, n_species, 40 - n_species)])]
    s = System(pos, rng.permutation(z), np.eye(3) * 60.0, np.array([False] * 3))
    snd, rcv = [], []
    for n in range(40):
        d = DEGREES[n] if n < len(DEGREES) else 7
        snd.append(rng.choice(np.delete(np.arange(40), n), size=d))
        rcv.append(np.full(d, n))
    return s, np.concatenate(snd), np.concatenate(rcv)


# float32: about a thousand roundings of 2^-24 lie between an edge's features and a force (hidden
# layers, the 270-edge sum, products over 64 x species and 128 channels); their random sum is
# ~30 x 2^-24 = 2e-6 of the largest term and a few times that of the largest force, hence 2e-5.
# float16 / bfloat16: the feature policies' bounds on the force RMS (11 and 8 significant bits).
@pytest.mark.parametrize("n_species,dtype,rms", [(1, "float32", 2e-5), (2, "float32", 2e-5), (5, "float32", 2e-5),
                                                 (8, "float32", 2e-5), (9, "float32", 2e-5), (1, "float16", 0.01),
                                                 (8, "float16", 0.01), (1, "bfloat16", 0.08), (5, "bfloat16", 0.08)])
def test_neighbour_sums_by_species(n_species, dtype, rms):
    cfg = arch_config("medium", num_elements=len(ZS), z_table=ZS, avg_num_neighbors=12.0)
    case = Case(cfg, seed=70, dtype=dtype)
    s, snd, rcv = _system(n_species, 71)
    zmap = {z: k for k, z in enumerate(ZS)}
    sp = np.array([zmap[int(z)] for z in s.numbers], np.int32)
    case.eng.set_system(sp, s.cell, s.pbc, 0.5)
    case.eng.set_edges(snd, rcv, np.zeros((len(snd), 3), np.int32))
    E, ne, F, vir = case.eng.step(s.positions, stress=True)
    ref = case.reference(s, sp, case.edges(), stress=True)
    dF = np.sqrt(np.mean((F - ref["F"]) ** 2) / np.mean(ref["F"] ** 2))
    dN = np.abs(ne - ref["ne"]).max() / np.abs(ref["ne"]).max()
    dV = np.abs(vir - ref["vir"]).max() / np.abs(ref["vir"]).max()
    print(f"{n_species} species {dtype}: force rms {dF:.2e}, node energies {dN:.2e}, virial {dV:.2e}", flush=True)
    assert dF <= rms and dN <= rms and dV <= rms
    # the same step replayed from its captured graphs, and once more after another species assignment
    E2, _, F2, _ = case.eng.step(s.positions, stress=True)
    assert E2 == E and np.array_equal(F2, F)
    if n_species > 1:
        other = np.roll(sp, 1)
        case.eng.set_system(other, s.cell, s.pbc, 0.5)
        case.eng.set_edges(snd, rcv, np.zeros((len(snd), 3), np.int32))
        case.eng.step(s.positions)
        case.eng.set_system(sp, s.cell, s.pbc, 0.5)
        case.eng.set_edges(snd, rcv, np.zeros((len(snd), 3), np.int32))
        assert np.array_equal(case.eng.step(s.positions, stress=True)[2], F)
