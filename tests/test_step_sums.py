"""The kernels of the MD entry and the batch inference that sum an atom's triplets, over the numbers of neighbours, species and
channels at which their loops take another way: against the op-by-op kernels that the host network's path takes."""
import numpy as np
import pytest

from util import nerr


def _crowd(edge, spacing, species, seed):
    """edge^3 atoms near the points of a cubic lattice, in a periodic box, and their species, dealt at random."""
    rng = np.random.Generator(np.random.Philox(seed))
    g = np.stack(np.unravel_index(np.arange(edge ** 3), (edge,) * 3), 1)
    x = spacing * g + rng.uniform(-0.1, 0.1, (edge ** 3, 3))
    L = spacing * edge
    return x, np.array([L, 0.0, 0.0, L, 0.0, L]), rng.integers(0, species, edge ** 3).astype(np.int32)


# Neighbours inside the angular cutoff: about 6, 18, 32 and 56 of at most `nr`.  A sweep of the force kernel takes 1024
# triplets (46 neighbours have 1035), the fingerprints' rows go four by four and their columns sixteen by sixteen.  125 to 1331
# centres: eight waves each up to 448 for the fingerprints and 1280 for the forces.  Four species with 40 channels: 40 to 84
# KB of LDS with eight waves, at 64 slots one workgroup per CU, which is enough for 216 centres and not for 343.
@pytest.mark.gpu
@pytest.mark.parametrize("edge,spacing,nr", [(5, 3.6, 24), (6, 2.6, 60), (6, 2.1, 64), (9, 2.1, 65), (7, 1.9, 64), (10, 1.9, 64),
                                             (11, 2.6, 60)])
@pytest.mark.parametrize("species,channels,beta", [(1, (15,), 1.0), (2, (3, 17, 40), 1.0), (2, (14, 13, 13), -12.0),
                                                   (3, (4, 3, 5, 3, 4, 3), 30.0), (4, (4,) * 10, 1.0)])
def test_sums_of_a_step(tmp_path, edge, spacing, nr, species, channels, beta):
    """float64, sums in another order: 1e-11.  beta: the largest exponent of the angular descriptor, one channel's."""
    from alphanesgpu_amd import libstaf, model_dir
    from test_oracle_pins import small_model
    ps = small_model(species, (5, 4, 6, 3)[:species], channels, seed=5, hidden=20, dense=species != 2)
    for p in ps:
        p["alpha3b"][0, 2] = beta
    x, box, types = _crowd(edge, spacing, species, seed=edge)
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=4.5, rs=1.6, radial_buffer=nr,
                              angular_buffer=nr * (nr - 1) // 2, tipos=np.bincount(types, minlength=species), precision="double")
    out = []
    for host in (True, False):
        m = libstaf.StafModel(str(tmp_path), precision=1, full_virial=True, host_mlp=host)
        out.append(m.compute(x, box, types))
        m.close()
    (e0, f0, v0), (e1, f1, v1) = out
    assert np.isfinite(e0) and np.abs(f0).max() > 0
    assert abs(e1 - e0) <= 1e-11 * max(1.0, abs(e0)) and nerr(f1, f0) <= 1e-11 and nerr(v1, v0) <= 1e-11
