"""The kernels of the MD entry and the batch inference that sum an atom's triplets, over the numbers of neighbours, species and
channels at which their loops take another way: against the op-by-op kernels that the host network's path and the layers take."""
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
# centres: eight waves each up to 448 for the fingerprints and 1280 (65 slots: 768) for the forces.  Four species with 40 channels: 40 to 84
# KB of LDS with eight waves, at 64 slots one workgroup per CU, which is enough for 216 centres and not for 343.
@pytest.mark.gpu
@pytest.mark.parametrize("edge,spacing,nr", [(5, 3.6, 24), (6, 2.6, 60), (6, 2.1, 64), (9, 2.1, 65), (10, 2.1, 65), (7, 1.9, 64),
                                             (10, 1.9, 64), (11, 2.6, 60)])
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


# The same kernels over several frames and in single precision, where the tables of the parameters are written by the call itself and not
# with the model: launches of 125 to 2662 centres, angular cutoff shorter than the radial one (about 4, 12, 30 and 41 neighbours inside).
# `exponents`: alpha1, alpha2 and beta of one channel of every class: within the rows that a table has, at their limits, beyond them.
@pytest.mark.gpu
@pytest.mark.parametrize("edge,spacing,nr,frames", [(5, 3.6, 24, 1), (6, 2.6, 60, 2), (7, 2.1, 65, 1), (9, 1.9, 64, 1), (7, 1.9, 64, 4),
                                                    (11, 2.6, 60, 2)])
@pytest.mark.parametrize("species,channels,exponents", [(1, (15,), (1.0, 0.5, 1.0)), (2, (3, 17, 40), (12.0, -12.0, -7.0)),
                                                        (2, (14, 13, 13), (-20.0, 4.0, 64.0)), (2, (20, 19, 1), (4.0, 1.0, -70.0)),
                                                        (3, (4, 3, 5, 3, 4, 3), (16.0, 20.0, 30.0)),
                                                        (4, (4,) * 10, (2.0, -5.0, -40.0))])
def test_sums_of_a_batch(tmp_path, edge, spacing, nr, frames, species, channels, exponents):
    """float64 against the layers' ops and against the MD entry, whose table is the host's: other summation orders, 1e-11.  float32
    against the float64 layers: an exponential of exponent a D carries a times the rounding of D (the sum of the three here, 6e-8
    each), a force the difference of some dozens of such terms."""
    import torch
    from alphanesgpu_amd import inference, libstaf, model_dir
    from test_oracle_pins import small_model
    ps = small_model(species, (5, 4, 6, 3)[:species], channels, seed=5, hidden=20, dense=species != 2)
    for p in ps:
        first = np.argmax(p["emb3b"] != 0, 1)
        for s, c in enumerate(first):
            p["alpha3b"][s, 3 * c:3 * c + 3] = exponents
    x, box, types = _crowd(edge, spacing, species, seed=edge)
    order = np.argsort(types, kind="stable")
    x, types = x[order], types[order]
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=4.0, rs=1.6, radial_buffer=nr,
                              angular_buffer=nr * (nr - 1) // 2, tipos=np.bincount(types, minlength=species), precision="double")
    rng = np.random.Generator(np.random.Philox(edge + 1))
    pos = np.stack([(x + rng.uniform(-0.05, 0.05, x.shape) * (f > 0)).reshape(-1) for f in range(frames)])
    boxes = np.tile(box, (frames, 1))
    inf = inference.staf_full_inference(str(tmp_path), max_batch=frames)
    T = lambda a: torch.as_tensor(a, dtype=torch.float64, device="cuda")
    N = lambda t: t.cpu().double().numpy()
    assert inf._species_of_call(T(pos), T(boxes)) is not None
    E, F, W = map(N, inf.full_test(pos, boxes))
    e, f, w = map(N, inf._full_test_by_layers(T(pos), T(boxes), False))
    scale = max(1.0, float(np.abs(e).max()))
    assert np.isfinite(e).all() and np.abs(f).max() > 0
    assert np.abs(E - e).max() <= 1e-11 * scale and nerr(F, f) <= 1e-11 and nerr(W, w) <= 1e-11
    m = libstaf.StafModel(str(tmp_path), precision=1, full_virial=True)
    me, mf, _ = m.compute(x, box, types)
    m.close()
    assert abs(E[0] - me) <= 1e-11 * scale and nerr(F[0], mf.reshape(-1)) <= 1e-11
    inf = inference.staf_full_inference(str(tmp_path), max_batch=frames, dtype=torch.float32)
    E, F, W = map(N, inf.full_test(pos, boxes))
    rel = 6e-8 * (sum(map(abs, exponents)) + 4)
    assert np.abs(E - e).max() <= 30 * rel * scale and nerr(F, f) <= 100 * rel and nerr(W, w) <= 100 * rel
