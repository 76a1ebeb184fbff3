"""The MD-facing entry (include/staf.h, include/staf_mlp.h): staf_load / staf_compute / staf_free and the MLP plug-in.

CPU tests cover the host-only parts (MLP plug-in against the numpy Dense stack, option defaults, null handling);
GPU tests call staf_compute through the C ABI and compare with the oracle pipeline, the reference's recorded
energies, and the two neighbour-list modes against each other."""
import ctypes as C
import json
import os

import numpy as np
import pytest

from util import GOLDEN, load_frame_mbpol, load_model, load_water_smoke, mlp_energy_and_grad, nerr

KNOWN = json.load(open(os.path.join(GOLDEN, "known_answers.json")))
RC = 4.5


# ----------------------------------------------------------------------------- host-only

class _Eval(C.Structure):
    _fields_ = [("n_type", C.c_int), ("n_atoms", C.POINTER(C.c_int)), ("n_af", C.POINTER(C.c_int)),
                ("af_f32", C.POINTER(C.c_float)), ("af_f64", C.POINTER(C.c_double)),
                ("energy_f32", C.POINTER(C.c_float)), ("energy_f64", C.POINTER(C.c_double)),
                ("dE_daf_f32", C.POINTER(C.c_float)), ("dE_daf_f64", C.POINTER(C.c_double))]


@pytest.mark.parametrize("prec", ["float", "double"])
def test_mlp_plugin_matches_numpy_dense_stack(prec):
    """staf_mlp_eval on the exported mlp_type*.bin against the numpy evaluation of the same weights read from the
    .npz export: energy = 1/2 sum of atomic energies, dE_daf = d(sum atomic)/d af."""
    from alphanesgpu_amd import _lib
    L = _lib.lib()
    L.staf_mlp_create.restype = C.c_void_p
    L.staf_mlp_create.argtypes = [C.c_int, C.c_char_p, C.c_int, C.c_int]
    L.staf_mlp_eval.argtypes = [C.c_void_p, C.POINTER(_Eval)]
    L.staf_mlp_destroy.argtypes = [C.c_void_p]
    L.staf_mlp_ntypes.argtypes = [C.c_void_p]
    L.staf_mlp_n_af.argtypes = [C.c_void_p, C.c_int]
    L.staf_mlp_precision.argtypes = [C.c_void_p]
    p = 0 if prec == "float" else 1
    dt, ct = (np.float32, C.c_float) if p == 0 else (np.float64, C.c_double)
    tipos, model = load_model(prec)
    h = L.staf_mlp_create(1, os.path.join(GOLDEN, f"model_{prec}").encode(), p, 0)
    assert h
    assert L.staf_mlp_ntypes(h) == 2 and L.staf_mlp_precision(h) == p
    rng = np.random.default_rng(5)
    n_atoms = np.array([7, 12], np.int32)
    n_af = np.array([L.staf_mlp_n_af(h, k) for k in range(2)], np.int32)
    assert list(n_af) == [m["mu"].size for m in model]
    afs = [rng.uniform(0.05, 3.0, (n_atoms[k], n_af[k])).astype(dt) for k in range(2)]
    flat = np.concatenate([a.reshape(-1) for a in afs])
    grad = np.zeros_like(flat)
    e = ct(0)
    ev = _Eval()
    ev.n_type = 2
    ev.n_atoms = n_atoms.ctypes.data_as(C.POINTER(C.c_int))
    ev.n_af = n_af.ctypes.data_as(C.POINTER(C.c_int))
    if p == 0:
        ev.af_f32, ev.dE_daf_f32 = (flat.ctypes.data_as(C.POINTER(C.c_float)), grad.ctypes.data_as(C.POINTER(C.c_float)))
        ev.energy_f32 = C.pointer(e)
    else:
        ev.af_f64, ev.dE_daf_f64 = (flat.ctypes.data_as(C.POINTER(C.c_double)),
                                    grad.ctypes.data_as(C.POINTER(C.c_double)))
        ev.energy_f64 = C.pointer(e)
    assert L.staf_mlp_eval(h, C.byref(ev)) == 0
    want_e, want_g = 0.0, []
    for k in range(2):
        ek, gk = mlp_energy_and_grad(afs[k].astype(np.float64), model[k]["mu"].astype(np.float64),
                                     [(W.astype(np.float64), b.astype(np.float64), a) for W, b, a in model[k]["layers"]])
        want_e += 0.5 * float(ek)
        want_g.append(gk.reshape(-1))
    want_g = np.concatenate(want_g)
    tol = 2e-5 if p == 0 else 1e-12
    assert abs(e.value - want_e) <= tol * max(1.0, abs(want_e))
    assert nerr(grad, want_g) <= tol
    # wrong fingerprint width is refused
    bad = n_af.copy()
    bad[1] += 1
    ev.n_af = bad.ctypes.data_as(C.POINTER(C.c_int))
    assert L.staf_mlp_eval(h, C.byref(ev)) == -3
    L.staf_mlp_destroy(h)
    assert L.staf_mlp_create(1, b"/nonexistent_model_dir", p, 0) is None


def test_options_default_and_null_model():
    from alphanesgpu_amd import libstaf
    o = libstaf.options_default()
    assert (o.mlp_backend, o.device_id, o.precision) == (libstaf.STAF_MLP_ORT, 0, 0)
    L = libstaf._bind()
    x = np.zeros(3)
    assert L.staf_compute(None, 1, 0, x.ctypes.data, x.ctypes.data, None, None, None, 0, None, None, None) == -1


# ----------------------------------------------------------------------------- GPU

def _wrap(pos, box6):
    """Positions folded into the primary cell of box6 = (Lx, xy, xz, Ly, yz, Lz)."""
    H = np.array([[box6[0], box6[1], box6[2]], [0, box6[3], box6[4]], [0, 0, box6[5]]])
    s = np.linalg.solve(H, pos.T).T
    s -= np.floor(s)
    return s @ H.T, H


def _ghost_configuration(pos, box6, types, rc):
    """What an MD code hands over: owned atoms plus explicit periodic images (ghosts) within rc of an owned atom,
    and per owned atom the neighbours within rc sorted by distance (indices into owned+ghost)."""
    pos, H = _wrap(pos, box6)
    n = len(pos)
    shifts = [np.array([a, b, c]) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1) if (a, b, c) != (0, 0, 0)]
    gx, gowner = [], []
    for sh in shifts:
        img = pos + H @ sh
        d2 = ((img[:, None, :] - pos[None, :, :]) ** 2).sum(-1)
        keep = np.where((d2 < rc * rc).any(axis=1))[0]
        gx.append(img[keep])
        gowner.append(keep)
    gx = np.concatenate(gx)
    gowner = np.concatenate(gowner)
    allx = np.concatenate([pos, gx])
    alltypes = np.concatenate([types, types[gowner]]).astype(np.int32)
    d2 = ((pos[:, None, :] - allx[None, :, :]) ** 2).sum(-1)
    lists = []
    for i in range(n):
        c = np.where((d2[i] < rc * rc) & (d2[i] > 1e-24))[0]
        lists.append(c[np.argsort(d2[i, c], kind="stable")])
    maxneigh = max(len(l) for l in lists)
    howmany = np.array([len(l) for l in lists], np.int32)
    neigh = np.zeros((n, maxneigh), np.int32)
    for i, l in enumerate(lists):
        neigh[i, :len(l)] = l
    return pos, allx, alltypes, gowner, howmany, neigh


def _as64(model):
    return [{k: (v.astype(np.float64) if isinstance(v, np.ndarray) else
                 [(W.astype(np.float64), b.astype(np.float64), a) for W, b, a in v]) for k, v in m.items()}
            for m in model]


@pytest.mark.gpu
def test_compute_matches_oracle_pipeline_fp64_model(oracle):
    """float64 model: energy, forces and virial diagonal of the reference frame against the oracle ops wired in the
    reference's order; tolerance 1e-10 (fp64 kernels, sums of ~1e3 terms in different orders)."""
    from alphanesgpu_amd import libstaf
    from test_oracle_pins import energy_and_forces
    tipos, model = load_model("double")
    pos, box, tp, type_map = load_frame_mbpol(np.float64)
    E, F, W, _, _ = energy_and_forces(oracle, pos, box, tp, type_map, _as64(model), virial=True)
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1, full_virial=True)
    e, f, vir = m.compute(pos.reshape(-1, 3), box[0], type_map)
    assert abs(e - float(E[0])) <= 1e-10 * abs(float(E[0]))
    assert nerr(f.reshape(-1), F[0]) <= 1e-10
    Wm = W[0].reshape(3, 3)
    want = np.array([Wm[0, 0], Wm[1, 1], Wm[2, 2], 0.5 * (Wm[0, 1] + Wm[1, 0]), 0.5 * (Wm[0, 2] + Wm[2, 0]),
                     0.5 * (Wm[1, 2] + Wm[2, 1])])
    assert nerr(vir, want) <= 1e-10
    # second call on the same handle (buffers reused) gives the same bits
    e2, f2, vir2 = m.compute(pos.reshape(-1, 3), box[0], type_map)
    assert e2 == e and np.array_equal(f2, f) and np.array_equal(vir2, vir)
    m.close()


@pytest.mark.gpu
def test_compute_6144_atom_box_matches_oracle_pipeline(oracle):
    """The large-box configuration through the MD entry: 2048 water molecules, one call, neighbour list rebuilt by the library
    (cell list: 6144 >= 4096 atoms), no tensor of the angular buffer's width on the device; energy and forces against
    the oracle ops wired in the reference's order (all-pairs neighbour search there), 1e-10."""
    from alphanesgpu_amd import libstaf, synth
    from test_oracle_pins import energy_and_forces
    tipos, model = load_model("double")
    b = synth.water_batch("water6144")
    pos, box = b["pos"].astype(np.float64), b["box"].astype(np.float64)
    E, F, W, _, _ = energy_and_forces(oracle, pos, box, b["tipos"], b["type_map"], _as64(model), virial=True)
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1, full_virial=True)
    e, f, vir = m.compute(pos.reshape(-1, 3), box[0], b["type_map"])
    assert abs(e - float(E[0])) <= 1e-10 * abs(float(E[0]))
    assert nerr(f.reshape(-1), F[0]) <= 1e-10
    Wm = W[0].reshape(3, 3)
    assert nerr(vir[:3], np.array([Wm[0, 0], Wm[1, 1], Wm[2, 2]])) <= 1e-10
    m.close()


@pytest.mark.gpu
def test_compute_is_invariant_under_periodic_replication():
    """A size-independent property at a size the oracle does not reach: the 6144-atom box replicated 2x2x2 (49152
    atoms, species-sorted, box edges doubled) has the same local environments, so the energy and the virial are
    eight times those of the single box and every replica carries the single box's forces (1e-12; the sums are
    the same, only the neighbour search runs over other cells)."""
    from alphanesgpu_amd import libstaf, synth
    b = synth.water_batch("water6144")
    x = b["pos"][0].reshape(-1, 3).astype(np.float64)
    box = b["box"][0].astype(np.float64)
    tm = b["type_map"]
    L = box[0]
    n_o = int((tm == 0).sum())
    shifts = np.array([[i, j, k] for i in range(2) for j in range(2) for k in range(2)], float) * L
    xo = np.concatenate([x[:n_o] + s for s in shifts])
    xh = np.concatenate([x[n_o:] + s for s in shifts])
    big_x = np.concatenate([xo, xh]) - L / 2
    big_tm = np.array([0] * len(xo) + [1] * len(xh), np.int32)
    big_box = box.copy()
    big_box[[0, 3, 5]] *= 2
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1)
    e, f, v = m.compute(x, box, tm)
    E, F, V = m.compute(big_x, big_box, big_tm)
    m.close()
    assert abs(E - 8 * e) <= 1e-12 * abs(8 * e)
    want = np.concatenate([np.concatenate([f[:n_o]] * 8), np.concatenate([f[n_o:]] * 8)])
    assert nerr(F.reshape(-1), want.reshape(-1)) <= 1e-12
    assert nerr(V, 8 * v) <= 1e-12


@pytest.mark.gpu
def test_compute_reproduces_recorded_energies_fp32_model(oracle):
    """float32 MLP (the reference's default build): E and rms(F) recorded by the reference for its 768-atom frame
    (test/test-lammps-STAF-inference-STAF-comp/results/frames.csv:2) and PE of data.water_smoke
    (test/B_ARCHITECTURE.md:167).  The water_smoke atoms come in file order (O H H ...), so this also covers the
    species-sorted packing and un-packing."""
    from alphanesgpu_amd import libstaf
    from test_oracle_pins import energy_and_forces
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_float"), precision=0)
    pos, box, tp, type_map = load_frame_mbpol(np.float64)
    e, f, vir = m.compute(pos.reshape(-1, 3), box[0], type_map)
    ka = KNOWN["frame0_model_float"]
    assert abs(e - ka["E_lammps"]) < 1.5e-4 and abs(e - ka["E_python"]) < 1.5e-4
    assert abs(float(np.sqrt(np.mean(f ** 2))) - ka["rms_F_python"]) < 5e-6
    assert np.all(vir[3:] == 0.0)          # diagonal only unless asked otherwise

    pos, box, types = load_water_smoke(np.float64)
    e, f, vir = m.compute(pos.reshape(-1, 3), box[0], types)
    assert abs(e - KNOWN["water_smoke_model_float"]["PE"]) < 2e-4
    # forces in the caller's order against the oracle on the species-sorted arrangement (float64 MLP there:
    # the float32 MLP's rounding is ~1e-6 of the force scale)
    tipos, model = load_model("float")
    order = np.argsort(types, kind="stable")
    ps = pos.reshape(-1, 3)[order].reshape(1, -1)
    E, F, _, _, _ = energy_and_forces(oracle, ps, box, np.bincount(types).astype(np.int32),
                                      types[order].astype(np.int32), _as64(model))
    Fo = np.zeros_like(f)
    Fo[order] = F[0].reshape(-1, 3)
    assert nerr(f, Fo) < 2e-5
    # permuting the caller's atom order permutes the forces and nothing else
    rng = np.random.default_rng(11)
    perm = rng.permutation(len(types))
    e_p, f_p, vir_p = m.compute(pos.reshape(-1, 3)[perm], box[0], types[perm])
    assert abs(e_p - e) < 1e-5 * abs(e)
    assert nerr(f_p, f[perm]) < 2e-5
    m.close()


@pytest.mark.gpu
def test_compute_with_injected_list_and_ghosts_matches_own_list():
    """The MD code's neighbour list (explicit periodic images as ghost atoms, no wrap inside the kernels) against
    the library's own minimum-image list: same energy and virial, and the ghost forces folded back onto their
    owners give the same forces.  float64 model, tolerance 1e-10."""
    from alphanesgpu_amd import libstaf
    pos, box, types = load_water_smoke(np.float64)
    pos = pos.reshape(-1, 3)
    n = len(pos)
    wrapped, allx, alltypes, gowner, howmany, neigh = _ghost_configuration(pos, box[0], types, RC)
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1, full_virial=True)
    e0, f0, v0 = m.compute(wrapped, box[0], types)
    e1, f1, v1 = m.compute(allx, box[0], alltypes, nlocal=n, howmany=howmany, neigh=neigh)
    folded = f1[:n].copy()
    np.add.at(folded, gowner, f1[n:])
    assert abs(e1 - e0) <= 1e-10 * abs(e0)
    assert nerr(folded, f0) <= 1e-10
    assert nerr(v1, v0) <= 1e-10
    # and back: the own-list mode is not left in no-wrap mode by the previous call
    e2, f2, v2 = m.compute(wrapped, box[0], types)
    assert e2 == e0 and np.array_equal(f2, f0)
    m.close()


@pytest.mark.gpu
def test_callers_list_after_own_list_after_callers_list():
    """A handle that goes from the caller's list to its own and back writes both neighbour maps to one place, and transposes
    the caller's in a block whose counters every build must find cleared.  Same bits as the first call; the own-list calls
    too."""
    from alphanesgpu_amd import libstaf
    pos, box, types = load_water_smoke(np.float64)
    pos = pos.reshape(-1, 3)
    n = len(pos)
    wrapped, allx, alltypes, _, howmany, neigh = _ghost_configuration(pos, box[0], types, RC)
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1, full_virial=True)
    theirs = lambda: m.compute(allx, box[0], alltypes, nlocal=n, howmany=howmany, neigh=neigh)
    ours = lambda: m.compute(wrapped, box[0], types)
    e0, f0, v0 = theirs()
    g0 = ours()
    for _ in range(3):
        e1, f1, v1 = theirs()
        assert e1 == e0 and np.array_equal(f1, f0) and np.array_equal(v1, v0)
        g1 = ours()
        assert g1[0] == g0[0] and np.array_equal(g1[1], g0[1])
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("width", [0, 1, 61, 200])
def test_callers_list_of_any_row_width_gives_the_same_bits(width):
    """The list reaches the device in the caller's order and row width: rows wider than the longest one (with entries
    behind the counts that are no atoms), atoms whose counts are zero or negative, counts beyond the row width, which are
    cut.  Reference: the narrowest rows that hold the same neighbours, in species order."""
    from alphanesgpu_amd import libstaf
    pos, box, types = load_water_smoke(np.float64)
    pos = pos.reshape(-1, 3)
    n = len(pos)
    _, allx, alltypes, _, howmany, neigh = _ghost_configuration(pos, box[0], types, RC)
    howmany = howmany.copy()
    howmany[::7] = -np.arange(len(howmany[::7]))
    w = neigh.shape[1] if width == 0 else width
    rows = np.full((n, w), -5, np.int32)
    for i in range(n):
        k = min(max(howmany[i], 0), w)
        rows[i, :k] = neigh[i, :k]
    order = np.argsort(alltypes[:n], kind="stable")            # species order: the library's slots
    back = np.argsort(order)
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1, full_virial=True)
    perm = np.concatenate([order, np.arange(n, len(allx))])
    slot = np.concatenate([back, np.arange(n, len(allx))]).astype(np.int32)
    cut = np.clip(howmany, 0, w)
    narrow = np.zeros((n, max(1, cut.max())), np.int32)
    for s, i in enumerate(order):
        narrow[s, :cut[i]] = slot[neigh[i, :cut[i]]]
    e0, f0, v0 = m.compute(allx[perm], box[0], alltypes[perm], nlocal=n, howmany=cut[order].astype(np.int32), neigh=narrow)
    e1, f1, v1 = m.compute(allx, box[0], alltypes, nlocal=n, howmany=howmany, neigh=rows)
    assert e1 == e0 and np.array_equal(f1[perm], f0) and np.array_equal(v1, v0)
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [("double", 1e-11), ("float", 2e-5)])
def test_device_mlp_matches_host_mlp(prec, tol):
    """The MLP evaluated on the GPU between the kernels (default) against the host evaluation of the same weights
    (reserved bit 1): energy, forces, virial.  float64 nets: 1e-11; float32 nets: the two evaluations sum in
    different orders, 2e-5 of the largest force."""
    from alphanesgpu_amd import libstaf
    pos, box, types = load_water_smoke(np.float64)
    pos = pos.reshape(-1, 3)
    p = 1 if prec == "double" else 0
    host = libstaf.StafModel(os.path.join(GOLDEN, f"model_{prec}"), precision=p, full_virial=True, host_mlp=True)
    e0, f0, v0 = host.compute(pos, box[0], types)
    host.close()
    dev = libstaf.StafModel(os.path.join(GOLDEN, f"model_{prec}"), precision=p, full_virial=True)
    e1, f1, v1 = dev.compute(pos, box[0], types)
    dev.close()
    assert abs(e1 - e0) <= max(tol, 1e-6 if p == 0 else 0) * abs(e0)
    assert nerr(f1, f0) <= tol
    assert nerr(v1, v0) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [("double", 1e-11), ("float", 2e-5)])
def test_device_mlp_on_small_widths_and_ragged_atom_counts(tmp_path, prec, tol):
    """The network kernel (matrix cores, four atoms per workgroup in launches this small) against the host evaluation on a
    written three-species model whose widths (fingerprints 9/7/11, hidden 20) are no multiples of the tile sizes and whose
    atom counts (7, 9, 3) leave a workgroup of every species partly empty: a wrong row layout of the matrix tiles or a
    padding row entering a sum shows here, not on the 256/512-atom frames."""
    from alphanesgpu_amd import libstaf, model_dir
    from test_oracle_pins import cluster, small_model
    ps = small_model(3, (5, 4, 6), (4, 3, 5, 3, 4, 3), seed=5, hidden=20, dense=True)
    pos, box, tipos, type_map = cluster([7, 9, 3], seed=9)
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=24, angular_buffer=276,
                              tipos=tipos, precision=prec)
    p = 1 if prec == "double" else 0
    host = libstaf.StafModel(str(tmp_path), precision=p, full_virial=True, host_mlp=True)
    e0, f0, v0 = host.compute(pos.reshape(-1, 3), box[0], type_map)
    host.close()
    dev = libstaf.StafModel(str(tmp_path), precision=p, full_virial=True)
    e1, f1, v1 = dev.compute(pos.reshape(-1, 3), box[0], type_map)
    dev.close()
    assert abs(e1 - e0) <= max(tol, 1e-6 if p == 0 else 0) * abs(e0)
    assert nerr(f1, f0) <= tol and nerr(v1, v0) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [("double", 1e-11), ("float", 2e-5)])
@pytest.mark.parametrize("hidden,last", [([], "linear"), ([], "tanh"), ([1], "linear"), ([16], "relu"), ([17, 15], "tanh"),
                                         ([300, 33], "linear"), ([16, 48, 16, 5], "linear")])
def test_device_mlp_stack_shapes(tmp_path, prec, tol, hidden, last):
    """The matrix-core network at the edges of its tiles: no hidden layer, one feature, exactly a tile, one more and one
    less, more tiles than waves, an output neuron with an activation; 16 and 17 atoms of a species (workgroups of four
    atoms exactly full, one atom in the next).  Against the host evaluation; float64: rounding of sums of at most 300 terms,
    float32: as the test above."""
    from alphanesgpu_amd import libstaf, model_dir, synth
    from test_oracle_pins import cluster
    rng = np.random.Generator(np.random.Philox(31))
    ps = synth.fingerprint_params(nt=2, ar_map=(5, 4), aa_map=(4, 3, 5), seed=3, dense_embedding=True)
    for p in ps:
        dims = [p["mu"].shape[0]] + hidden + [1]
        acts = ["tanh" if i % 2 == 0 else "relu" for i in range(len(hidden))] + [last]
        p["layers"] = [(rng.normal(0, 1 / np.sqrt(a), (a, b)), rng.normal(0.3, 0.1, b), act)
                       for a, b, act in zip(dims[:-1], dims[1:], acts)]
    pos, box, tipos, type_map = cluster([16, 17], seed=9, spread=4.4)
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=40, angular_buffer=780,
                              tipos=tipos, precision=prec)
    got = []
    for host in (True, False):
        m = libstaf.StafModel(str(tmp_path), precision=1 if prec == "double" else 0, full_virial=True, host_mlp=host)
        got.append(m.compute(pos.reshape(-1, 3), box[0], type_map))
        m.close()
    (e0, f0, v0), (e1, f1, v1) = got
    assert abs(e1 - e0) <= tol * max(1.0, abs(e0)) and nerr(f1, f0) <= tol and nerr(v1, v0) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol,hidden,on_gpu", [("float", 2e-5, [400] * 6, True), ("float", 2e-5, [430] * 6, True),
                                                    ("double", 1e-11, [200] * 6, True), ("double", 1e-11, [420] * 6, False)])
def test_deep_stacks_around_the_limits_of_a_workgroup(tmp_path, capfd, prec, tol, hidden, on_gpu):
    """Stacks whose activations of 16 atoms just fit a workgroup's LDS, fit it for 8 atoms only, and do not fit: the first
    two are evaluated on the GPU, the last one on the host (a line on stderr says so) and, in the batch inference, by the
    layers.  17 atoms of a species: five workgroups of four, the last one with a single atom.  Against the host evaluation;
    float64: rounding of sums of at most 420 terms, float32: as above."""
    import torch
    from alphanesgpu_amd import inference, libstaf, model_dir, synth
    from test_oracle_pins import cluster
    rng = np.random.Generator(np.random.Philox(37))
    ps = synth.fingerprint_params(nt=2, ar_map=(5, 4), aa_map=(4, 3, 5), seed=3, dense_embedding=True)
    for p, h in zip(ps, (hidden, [9])):
        dims = [p["mu"].shape[0]] + h + [1]
        acts = ["tanh"] * len(h) + ["linear"]
        p["layers"] = [(rng.normal(0, 1 / np.sqrt(a), (a, b)), rng.normal(0, 0.1, b), act)
                       for a, b, act in zip(dims[:-1], dims[1:], acts)]
    pos, box, tipos, type_map = cluster([17, 16], seed=9, spread=4.4)
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=40, angular_buffer=780,
                              tipos=tipos, precision=prec)
    p = 1 if prec == "double" else 0
    m = libstaf.StafModel(str(tmp_path), precision=p, full_virial=True, host_mlp=True)
    e0, f0, v0 = m.compute(pos.reshape(-1, 3), box[0], type_map)
    m.close()
    capfd.readouterr()
    m = libstaf.StafModel(str(tmp_path), precision=p, full_virial=True)
    assert ("on the host" not in capfd.readouterr().err) == on_gpu
    e1, f1, v1 = m.compute(pos.reshape(-1, 3), box[0], type_map)
    m.close()
    assert abs(e1 - e0) <= tol * max(1.0, abs(e0)) and nerr(f1, f0) <= tol and nerr(v1, v0) <= tol
    inf = inference.staf_full_inference(str(tmp_path), dtype=torch.float64 if p else torch.float32)
    e2, f2, _ = inf.full_test(pos, box)
    tol2 = tol if p else 5e-5       # (everything in float32)
    assert abs(float(e2[0]) - e0) <= tol2 * max(1.0, abs(e0)) and nerr(f2.cpu().numpy().reshape(-1, 3), f0) <= tol2


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [("double", 1e-11), ("float", 2e-5)])
@pytest.mark.parametrize("last", ["tanh", "relu", "linear"])
def test_one_layer_network_beside_a_wide_one(tmp_path, prec, tol, last):
    """A species without hidden layers in the launch of one whose 300 features give every workgroup sixteen waves: all of
    them add up the output neuron's shares while the first of them already knows its slope.  Against the host evaluation,
    and the same bits on every call; tolerances as above."""
    from alphanesgpu_amd import libstaf, model_dir, synth
    from test_oracle_pins import cluster
    rng = np.random.Generator(np.random.Philox(33))
    ps = synth.fingerprint_params(nt=2, ar_map=(5, 4), aa_map=(4, 3, 5), seed=3, dense_embedding=True)
    for p, hidden in zip(ps, ([], [300, 33])):
        dims = [p["mu"].shape[0]] + hidden + [1]
        acts = ["tanh"] * len(hidden) + [last]
        p["layers"] = [(rng.normal(0, 1 / np.sqrt(a), (a, b)), rng.normal(0.3, 0.1, b), act)
                       for a, b, act in zip(dims[:-1], dims[1:], acts)]
    pos, box, tipos, type_map = cluster([33, 17], seed=9, spread=5.0)
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=50, angular_buffer=1225,
                              tipos=tipos, precision=prec)
    p = 1 if prec == "double" else 0
    m = libstaf.StafModel(str(tmp_path), precision=p, full_virial=True, host_mlp=True)
    e0, f0, v0 = m.compute(pos.reshape(-1, 3), box[0], type_map)
    m.close()
    m = libstaf.StafModel(str(tmp_path), precision=p, full_virial=True)
    got = [m.compute(pos.reshape(-1, 3), box[0], type_map) for _ in range(8)]
    m.close()
    e1, f1, v1 = got[0]
    assert abs(e1 - e0) <= tol * max(1.0, abs(e0)) and nerr(f1, f0) <= tol and nerr(v1, v0) <= tol
    for e, f, v in got[1:]:
        assert e == e1 and np.array_equal(f, f1) and np.array_equal(v, v1)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [("double", 1e-11), ("float", 2e-5)])
def test_infinite_activations_stay_out_of_the_padded_features(tmp_path, prec, tol):
    """A feature of a linear layer that overflows saturates the tanh layer behind it (slope 0, so that gradients are
    finite too).  Layers of 5 and 7 features leave most of their 16-feature tiles empty: infinity times the zero weights
    of the empty ones must not reach the energy.  Against the host evaluation, which has no such features."""
    from alphanesgpu_amd import libstaf, model_dir, synth
    from test_oracle_pins import cluster
    rng = np.random.Generator(np.random.Philox(35))
    ps = synth.fingerprint_params(nt=2, ar_map=(5, 4), aa_map=(4, 3, 5), seed=3, dense_embedding=True)
    for p in ps:
        n = p["mu"].shape[0]
        p["mu"][2] += 50.0     # |log(af + 1e-3) - mu| of this fingerprint is far above 2
        W = [rng.normal(0, 1 / np.sqrt(a), (a, b)) for a, b in ((n, 5), (5, 7), (7, 6), (6, 1))]
        W[0][:, 3] = 0
        W[0][2, 3] = 0.9 * (np.finfo(np.float64).max if prec == "double" else float(np.finfo(np.float32).max))
        p["layers"] = [(w, rng.normal(0.3, 0.1, w.shape[1]), a) for w, a in zip(W, ("linear", "tanh", "tanh", "linear"))]
    pos, box, tipos, type_map = cluster([16, 17], seed=9, spread=4.4)
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=40, angular_buffer=780,
                              tipos=tipos, precision=prec)
    got = []
    for host in (True, False):
        m = libstaf.StafModel(str(tmp_path), precision=1 if prec == "double" else 0, full_virial=True, host_mlp=host)
        got.append(m.compute(pos.reshape(-1, 3), box[0], type_map))
        m.close()
    (e0, f0, v0), (e1, f1, v1) = got
    assert np.isfinite(e0) and np.isfinite(f0).all()
    assert abs(e1 - e0) <= tol * max(1.0, abs(e0)) and nerr(f1, f0) <= tol and nerr(v1, v0) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("counts,nr", [([16, 17, 5], 40), ([1, 0, 9], 24), ([0, 3, 0], 60), ([40, 30, 3], 100)])
@pytest.mark.parametrize("callers_list", [False, True])
def test_all_species_in_one_launch(tmp_path, counts, nr, callers_list):
    """The stages of the device path, each one launch over all species, against the op-by-op path the host network
    takes: species without atoms, a single atom, fewer and more than 64 slots per row (one and two waves that hold
    slots), with and without the virial, repeated calls.  float64: sums in another order, 1e-11."""
    from alphanesgpu_amd import libstaf, model_dir
    from test_oracle_pins import cluster, small_model
    ps = small_model(3, (5, 4, 6), (4, 3, 5, 3, 4, 3), seed=5, hidden=20, dense=True)
    pos, box, tipos, types = cluster(counts, seed=17, spread=5.0)
    model_dir.write_model_dir(str(tmp_path), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=nr, angular_buffer=nr * (nr - 1) // 2,
                              tipos=tipos, precision="double")
    x = pos.reshape(-1, 3)
    order = np.random.default_rng(3).permutation(len(x))
    x, types = x[order], types[order]
    extra = {}
    if callers_list:
        d = np.linalg.norm(x[:, None] - x[None], axis=-1)
        rows = [[j for j in np.argsort(r, kind="stable")[1:] if r[j] < 4.5] for r in d]
        neigh = np.zeros((len(x), nr), np.int32)
        for i, r in enumerate(rows):
            neigh[i, :len(r)] = r
        extra = dict(nlocal=len(x), howmany=np.array([len(r) for r in rows], np.int32), neigh=neigh)
    m = libstaf.StafModel(str(tmp_path), precision=1, full_virial=True, host_mlp=True)
    e0, f0, v0 = m.compute(x, box[0], types, **extra)
    m.close()
    m = libstaf.StafModel(str(tmp_path), precision=1, full_virial=True)
    for want in (True, True, False, True):
        e1, f1, v1 = m.compute(x, box[0], types, want_virial=want, **extra)
        assert abs(e1 - e0) <= 1e-11 * max(1.0, abs(e0)) and nerr(f1, f0) <= 1e-11
        assert (v1 is None) if not want else nerr(v1, v0) <= 1e-11
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("callers_list", [False, True])
def test_neighbour_buffers_whose_slots_leave_no_room_for_both_bodies(tmp_path, callers_list):
    """250 slots and three species: a force workgroup holds the 3-body rows (154 of 160 KB) but not the 2-body ones beside
    them, and the forces come from an op per body.  Buffers beyond the neighbours an atom has change nothing, so the same
    model with 60 slots, whose forces come from one launch, is the reference; sums in another order, 1e-11.  The batch
    inference takes such a model through its layers."""
    import torch
    from alphanesgpu_amd import inference, libstaf, model_dir
    from test_oracle_pins import cluster, small_model
    ps = small_model(3, (5, 4, 6), (4, 3, 5, 3, 4, 3), seed=5, hidden=20, dense=True)
    pos, box, tipos, types = cluster([16, 17, 5], seed=17, spread=5.0)
    x = pos.reshape(-1, 3)
    extra = {}
    if callers_list:
        d = np.linalg.norm(x[:, None] - x[None], axis=-1)
        rows = [[j for j in np.argsort(r, kind="stable")[1:] if r[j] < 4.5] for r in d]
        neigh = np.zeros((len(x), 40), np.int32)
        for i, r in enumerate(rows):
            neigh[i, :len(r)] = r
        extra = dict(nlocal=len(x), howmany=np.array([len(r) for r in rows], np.int32), neigh=neigh)
    out = []
    for nr in (60, 250):
        d = tmp_path / str(nr)
        d.mkdir()
        model_dir.write_model_dir(str(d), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=nr, angular_buffer=780, tipos=tipos,
                                  precision="double")
        m = libstaf.StafModel(str(d), precision=1, full_virial=True)
        for want in (False, True):
            e, f, v = m.compute(x, box[0], types, want_virial=want, **extra)
        m.close()
        out.append((e, f, v))
        if not callers_list:
            g = inference.staf_full_inference(str(d), dtype=torch.float64)
            T = lambda a: torch.as_tensor(a, device="cuda")
            out.append(tuple(t.cpu().numpy() for t in g.full_test(T(pos), T(box))))
    e0, f0, v0 = out[0]
    full = lambda v: np.array([v[0], v[4], v[8], (v[1] + v[3]) / 2, (v[2] + v[6]) / 2, (v[5] + v[7]) / 2])
    for e, f, v in out[1:]:
        if np.ndim(e):
            e, f, v = e[0], f.reshape(-1, 3), full(v.reshape(-1))
        assert abs(e - e0) <= 1e-11 * max(1.0, abs(e0)) and nerr(f, f0) <= 1e-11 and nerr(v, v0) <= 1e-11


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(4, 4, 2), (8, 7, 3), (8, 8, 4), (9, 8, 4)])
def test_device_path_on_both_sides_of_the_workgroup_sizes_lines(cells):
    """96, 504, 768 and 864 centres: wider workgroups for the fingerprints of up to 512 and the slot forces of up to 768.
    Against the op-by-op path the host network takes; float64, sums in another order, 1e-11."""
    from alphanesgpu_amd import libstaf, synth
    molecules = int(np.prod(cells))
    x, box = synth.water_frame(cells, (29.9 * molecules) ** (1 / 3), 0.05, 11)
    types = np.repeat(np.arange(2, dtype=np.int32), (molecules, 2 * molecules))
    out = []
    for host in (True, False):
        m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1, full_virial=True, host_mlp=host)
        out.append(m.compute(x.reshape(-1, 3), box, types))
        m.close()
    (e0, f0, v0), (e1, f1, v1) = out
    assert abs(e1 - e0) <= 1e-11 * max(1.0, abs(e0)) and nerr(f1, f0) <= 1e-11 and nerr(v1, v0) <= 1e-11


@pytest.mark.gpu
def test_compute_without_virial_gives_the_same_energy_and_forces():
    """A null virial pointer skips the virial kernels; energy and forces keep their bits."""
    from alphanesgpu_amd import libstaf
    pos, box, tp, type_map = load_frame_mbpol(np.float64)
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1)
    e, f, vir = m.compute(pos.reshape(-1, 3), box[0], type_map)
    e2, f2, vir2 = m.compute(pos.reshape(-1, 3), box[0], type_map, want_virial=False)
    assert vir2 is None and np.all(np.isfinite(vir))
    assert e2 == e and np.array_equal(f2, f)
    m.close()


@pytest.mark.gpu
def test_a_handle_that_follows_shape_changes_gives_the_bits_of_a_fresh_one():
    """A handle walks through a sequence of configurations -- the 768-atom frame moving from call to call, then the
    water_smoke frame (other atom count and order) with the library's list and with a caller's, then the first one again,
    with and without virial -- and every call must agree bit for bit with the first call of a handle that has just been
    loaded: what a handle holds between calls (blocks of an earlier size, the species it has sent, a list's transpose)
    does not enter a result."""
    from alphanesgpu_amd import libstaf
    d = os.path.join(GOLDEN, "model_double")
    a = libstaf.StafModel(d, precision=1, full_virial=True)
    posA, boxA, _, tmA = load_frame_mbpol(np.float64)
    posB, boxB, typB = load_water_smoke(np.float64)
    rng = np.random.default_rng(17)
    plan = ([("A", True)] * 2 + [("B", True)] * 2 + [("list", True)] * 2 + [("A", True)] + [("A", False)] * 2 +
            [("list", False)] + [("B", False)] * 2 + [("list", True)] + [("A", True)])
    for step, (which, want_w) in enumerate(plan):
        pos, box, types = (posA, boxA[0], tmA) if which == "A" else (posB, boxB[0], typB)
        x = pos.reshape(-1, 3) + 0.02 * rng.standard_normal((pos.shape[1] // 3, 3))   # the atoms move every step
        extra = {}
        if which == "list":
            n = len(x)
            _, x, types, _, howmany, neigh = _ghost_configuration(x, box, types, RC)
            extra = dict(nlocal=n, howmany=howmany, neigh=neigh)
        elif step % 2:
            flip = rng.permutation(len(x))       # (another order of the same species counts)
            x, types = x[flip], np.asarray(types)[flip]
        ea, fa, wa = a.compute(x, box, types, want_virial=want_w, **extra)
        b = libstaf.StafModel(d, precision=1, full_virial=True)
        eb, fb, wb = b.compute(x, box, types, want_virial=want_w, **extra)
        b.close()
        assert ea == eb and np.array_equal(fa, fb), (step, which)
        assert (wa is None and wb is None) or np.array_equal(wa, wb), (step, which)
        assert np.isfinite(ea) and np.abs(fa).max() > 0
        if step and plan[step - 1][0] == which:
            assert ea != prev_e          # the inputs did change: a call that re-used old inputs would show here
        prev_e = ea
    a.close()


@pytest.mark.gpu
def test_release_of_the_ops_state_between_calls():
    """staf_ops_release (the op interface's call that frees the library's work areas) between calls of a handle of the MD
    entry: the next call sizes the areas again -- same bits on every call."""
    from alphanesgpu_amd import libstaf, ops
    pos, box, _, type_map = load_frame_mbpol(np.float64)
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1, full_virial=True)
    x = pos.reshape(-1, 3)
    ref = [m.compute(x, box[0], type_map) for _ in range(4)][-1]
    for _ in range(2):
        ops.release()
        for _ in range(4):
            e, f, w = m.compute(x, box[0], type_map)
            assert e == ref[0] and np.array_equal(f, ref[1]) and np.array_equal(w, ref[2])
    m.close()


@pytest.mark.gpu
def test_three_handles_on_three_host_threads():
    """Three handles, each used by a host thread of its own at the same time (every handle has a stream of its own): every
    call returns the bits a single handle returned for the same positions."""
    import threading
    from alphanesgpu_amd import libstaf
    pos, box, _, type_map = load_frame_mbpol(np.float64)
    x = pos.reshape(-1, 3)
    d = os.path.join(GOLDEN, "model_double")
    rng = np.random.default_rng(1)
    xs = [x + 0.02 * rng.standard_normal(x.shape) for _ in range(8)]
    ref = libstaf.StafModel(d, precision=1, full_virial=True)
    want = [ref.compute(xx, box[0], type_map) for xx in xs]
    ref.close()
    bad = []

    def worker(t):
        try:
            m = libstaf.StafModel(d, precision=1, full_virial=True)
            for rep in range(2):
                for i, xx in enumerate(xs):
                    e, f, w = m.compute(xx, box[0], type_map)
                    if e != want[i][0] or not np.array_equal(f, want[i][1]) or not np.array_equal(w, want[i][2]):
                        bad.append((t, rep, i))
            m.close()
        except Exception as ex:   # a thread's exception would otherwise be lost
            bad.append((t, repr(ex)))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad, bad[:10]


@pytest.mark.gpu
@pytest.mark.parametrize("host_mlp", [False, True])
def test_more_handles_on_threads_than_maps_are_remembered(host_mlp):
    """Twelve handles on twelve host threads, every other one with a caller's list: more than the neighbour maps the ops
    remember by address, so a call may rely only on what its own handle holds between its launches.  Every call returns the
    bits a single handle returned for the same frame."""
    import threading
    from alphanesgpu_amd import libstaf
    pos, box, types = load_water_smoke(np.float64)
    pos = pos.reshape(-1, 3)
    x, allx, alltypes, _, howmany, neigh = _ghost_configuration(pos, box[0], types, RC)
    d = os.path.join(GOLDEN, "model_double")
    frames = [((pos, box[0], types), {}), ((allx, box[0], alltypes), dict(nlocal=len(x), howmany=howmany, neigh=neigh))]
    make = lambda: libstaf.StafModel(d, precision=1, full_virial=True, host_mlp=host_mlp)
    m = make()
    want = [m.compute(*a, **kw) for a, kw in frames]
    m.close()
    bad = []

    def worker(t):
        try:
            m = make()
            for rep in range(4 if host_mlp else 25):
                which = (t + rep // 3) % 2
                a, kw = frames[which]
                got = m.compute(*a, **kw)
                if not all(np.array_equal(g, w) for g, w in zip(got, want[which])):
                    bad.append((t, rep))
            m.close()
        except Exception as ex:   # a thread's exception would otherwise be lost
            bad.append((t, repr(ex)))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(12)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad, bad[:10]


@pytest.mark.gpu
def test_compute_return_codes():
    """Validation order and codes of libstaf/src/staf_api.cpp:196-337."""
    from alphanesgpu_amd import libstaf
    m = libstaf.StafModel(os.path.join(GOLDEN, "model_float"), precision=0)
    pos, box, types = load_water_smoke(np.float64)
    pos = pos.reshape(-1, 3)
    code = lambda **kw: pytest.raises(libstaf.StafComputeError, m.compute, **kw).value.code
    assert code(x=pos[:0], box=box[0], types=types[:0]) == -3
    zb = box[0].copy()
    zb[3] = 0.0
    assert code(x=pos, box=zb, types=types) == -7
    bt = types.copy()
    bt[5] = 2
    assert code(x=pos, box=box[0], types=bt) == -8
    hm = np.ones(len(pos), np.int32)
    w = np.zeros((len(pos), 4), np.int32)
    w[3, 0] = len(pos)
    assert code(x=pos, box=box[0], types=types, howmany=hm, neigh=w) == -9
    # one atom named by more centres than the force gather holds keys for (4 x the radial buffer): every other atom
    # of the frame lists atom 0.  Detected on the device, returned by the host; every kernel runs to its end.
    w[:] = 0
    w[0, 0] = 1
    assert len(pos) - 1 > 4 * 60
    assert code(x=pos, box=box[0], types=types, howmany=hm, neigh=w) == -11
    # a valid call still works afterwards
    e, f, v = m.compute(pos, box[0], types)
    assert abs(e - KNOWN["water_smoke_model_float"]["PE"]) < 2e-4
    m.close()
    with pytest.raises(RuntimeError):
        libstaf.StafModel("/nonexistent_model_dir")


# ----------------------------------------------------------------------------- a caller written in C

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MD_STEP = os.path.join(ROOT, "tests", "c_consumer", "md_step")


def test_headers_are_plain_c_and_the_c_caller_is_built():
    """include/*.h compile as C99 and as C++11 with -pedantic (they are what a C or C++ host includes), and the C
    caller built against include/staf.h alone links the library and reports a usage error without touching a GPU."""
    import subprocess
    for h in ("staf.h", "staf_mlp.h", "staf_ops.h"):
        path = os.path.join(ROOT, "include", h)
        for cc, std, lang in (("gcc", "-std=c99", "c"), ("g++", "-std=c++11", "c++")):
            r = subprocess.run([cc, std, "-Wall", "-Wextra", "-pedantic", "-Werror", "-fsyntax-only", "-x", lang, path],
                               capture_output=True, text=True)
            assert r.returncode == 0, (h, cc, r.stderr)
    assert os.path.exists(MD_STEP), "run __graft_entry__.build() first"
    r = subprocess.run([MD_STEP], capture_output=True, text=True)
    assert r.returncode == 100 and "usage" in r.stderr


@pytest.mark.gpu
def test_c_caller_reproduces_recorded_energy():
    """The plain-C program (tests/c_consumer/md_step.c: staf_load, staf_compute with the library's own neighbour
    list, staf_free) on the reference's 768-atom frame with its float32 model: E and rms(F) recorded by the
    reference (test/test-lammps-STAF-inference-STAF-comp/results/frames.csv:2); a second step on rigidly shifted
    coordinates gives the same energy and forces to rounding."""
    import subprocess
    d = os.path.join(GOLDEN, "frame_mbpol")
    r = subprocess.run([MD_STEP, os.path.join(GOLDEN, "model_float"), os.path.join(d, "pos_0"),
                        os.path.join(d, "box_0"), os.path.join(d, "type.dat"), "0", "2"],
                       capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, (r.stdout, r.stderr)
    lines = [l.split() for l in r.stdout.splitlines() if l.startswith("step")]
    assert len(lines) == 2 and all(l[3] == "0" for l in lines)
    e = [float(l[5]) for l in lines]
    rms = [float(l[7]) for l in lines]
    ka = KNOWN["frame0_model_float"]
    assert abs(e[0] - ka["E_lammps"]) < 1.5e-4 and abs(rms[0] - ka["rms_F_python"]) < 5e-6
    # float32 network: the shifted coordinates round differently (same bounds as the permutation check above)
    assert abs(e[1] - e[0]) < 1e-5 * abs(e[0]) and abs(rms[1] - rms[0]) < 2e-5
    vir = [float(x) for x in lines[0][9:15]]
    assert vir[3] == vir[4] == vir[5] == 0.0 and all(v != 0.0 for v in vir[:3])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 3, 170, 171, 10922, 10925])
def test_every_atom_of_a_call_arrives_and_returns(n):
    """Input and results are copied by kernels in pieces of two doubles, 256 to a workgroup and 64 workgroups to a round of
    results: pairs of atoms in a row, each the same to the last bit (offsets are whole numbers, box edges a power of two), have
    the first pair's forces to the last bit wherever they lie in the blocks, and the energies add up (n 2^-53 of the sum of n
    equal terms)."""
    from alphanesgpu_amd import libstaf
    model = libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1)
    x = np.zeros((n, 3))
    x[:, 0] = 16.0 * (np.arange(n) // 2) + 2.5 * (np.arange(n) % 2)
    howmany = np.array([min(1, n - 1 - i) if i % 2 == 0 else 1 for i in range(n)], np.int32)
    neigh = (np.arange(n) ^ 1).reshape(-1, 1).astype(np.int32)
    neigh[howmany == 0] = 0
    types = (np.arange(n) % 2).astype(np.int32)
    box = 2.0 ** 20 * np.array([1.0, 0.0, 0.0, 1.0, 0.0, 1.0])   # (a power of two: fractions of it are exact)
    for _ in range(2):
        e, f, _ = model.compute(x, box, types, nlocal=n, howmany=howmany, neigh=neigh)
        pairs = n // 2
        if pairs:
            e2, f2, _ = model.compute(x[:2], box, types[:2], nlocal=2, howmany=howmany[:2], neigh=neigh[:2])
            assert np.abs(f2).max() > 0
            assert np.array_equal(f[:2 * pairs], np.tile(f[:2], (pairs, 1)))
            assert np.abs(f[:2] - f2).max() <= 1e-13 * np.abs(f2).max()   # (other workgroup sizes: sums of 140 terms in another order)
        else:
            e2 = 0.0
        e1 = 0.0
        if n % 2:
            e1, f1, _ = model.compute(x[:1], box, types[:1], nlocal=1, howmany=np.zeros(1, np.int32), neigh=np.zeros((1, 1), np.int32))
            assert np.array_equal(f[-1:], f1) and np.abs(f1).max() == 0
        want = pairs * e2 + e1
        assert abs(e - want) <= (n + 2) * 2.0 ** -53 * (pairs * abs(e2) + abs(e1)) * 4
    model.close()


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [("double", 1e-11), ("float", 2e-5)])
@pytest.mark.parametrize("n", [1021, 1027, 2043, 2053])
def test_network_on_both_sides_of_the_atoms_per_workgroup_lines(prec, tol, n):
    """256 workgroups of four atoms, 256 of eight, 512 of four (n atoms of two species, ragged last tiles): device network
    against the host's, tolerances of test_device_mlp_matches_host_mlp."""
    from alphanesgpu_amd import libstaf
    rng = np.random.Generator(np.random.Philox(n))
    edge = 4 * round(n ** (1 / 3) + 1)
    cells = rng.permutation((edge // 4) ** 3)[:n]
    x = 4.0 * np.stack(np.unravel_index(cells, (edge // 4,) * 3), 1) + rng.uniform(0, 1.5, (n, 3))
    types = rng.integers(0, 2, n).astype(np.int32)
    box = edge * np.array([1.0, 0.0, 0.0, 1.0, 0.0, 1.0])
    d = os.path.join(GOLDEN, f"model_{prec}")
    out = []
    for host in (False, True):
        m = libstaf.StafModel(d, precision=1 if prec == "double" else 0, full_virial=True, host_mlp=host)
        out.append(m.compute(x, box, types))
        m.close()
    (e, f, w), (eh, fh, wh) = out
    assert abs(e - eh) <= tol * abs(eh)
    assert nerr(f, fh) <= tol and nerr(w, wh) <= tol


@pytest.mark.gpu
def test_a_handle_keeps_the_order_of_the_types_it_was_last_given():
    """The slots of the atoms are worked out for the types of a call and kept for calls with the same ones: after other types,
    other ghosts' types, no types at all and a refused call the results are those of a fresh handle, to the last bit."""
    from alphanesgpu_amd import libstaf, synth
    pos, box = synth.water_frame((4, 4, 2), 9.86, 0.05, 5)
    pos, H = _wrap(pos.reshape(-1, 3), box)
    water = np.repeat(np.arange(2, dtype=np.int32), (32, 64))
    rng = np.random.Generator(np.random.Philox(8))
    own = [(pos, t) for t in (water, water[::-1].copy(), rng.permutation(water), np.zeros(96, np.int32), None, water, None)]
    listed = []
    for t in (water, rng.permutation(water)):
        x, allx, alltypes, _, howmany, neigh = _ghost_configuration(pos, box, t, RC)
        listed += [(allx, alltypes, 96, howmany, neigh), (allx, np.concatenate([t, rng.permutation(alltypes[96:])]), 96, howmany, neigh)]
    calls = own[:3] + listed[:2] + own[3:5] + ["refused"] + own[5:] + listed[2:] + own[:1]
    make = lambda: libstaf.StafModel(os.path.join(GOLDEN, "model_double"), precision=1)
    used = make()
    for c in calls:
        if c == "refused":
            bad = water.copy()
            bad[50] = 2
            with pytest.raises(libstaf.StafComputeError):
                used.compute(pos, box, bad)
            continue
        args = (c[0], box, c[1]) if len(c) == 2 else (c[0], box, c[1], *c[2:])
        fresh = make()
        want, got = fresh.compute(*args), used.compute(*args)
        fresh.close()
        assert got[0] == want[0] and np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2])
    used.close()


def _gas(counts, seed):
    """So many atoms of each species, one anywhere in the middle of a 4 A cell: at least 2.5 A apart, few neighbours."""
    rng = np.random.Generator(np.random.Philox(seed))
    n = sum(counts)
    edge = int(np.ceil(n ** (1 / 3))) + 1
    x = 4.0 * np.stack(np.unravel_index(rng.permutation(edge ** 3)[:n], (edge,) * 3), 1) + rng.uniform(0, 1.5, (n, 3))
    return x, 4.0 * edge * np.array([1.0, 0.0, 0.0, 1.0, 0.0, 1.0]), np.repeat(np.arange(len(counts), dtype=np.int32), counts)


def _device_and_host_network(folder, prec, tol, hidden, last, counts, seed, change=None):
    """A model of two species with these hidden layers, evaluated on the GPU and by the host.  Forces and virials to tol;
    energies to tol and, in single precision, what the host's running sum of n atoms may lose (n 2^-24), of the energy or of a
    sixteenth per atom where they cancel."""
    from alphanesgpu_amd import libstaf, model_dir, synth
    rng = np.random.Generator(np.random.Philox(seed))
    ps = synth.fingerprint_params(nt=2, ar_map=(5, 4), aa_map=(4, 3, 5), seed=3, dense_embedding=True)
    for p, h in zip(ps, hidden):
        dims = [p["mu"].shape[0]] + h + [1]
        acts = ["tanh" if i % 2 == 0 or len(h) > 4 else "relu" for i in range(len(h))] + [last]
        p["layers"] = [(rng.normal(0, 1 / np.sqrt(a), (a, b)), rng.normal(0.3, 0.1, b), act)
                       for a, b, act in zip(dims[:-1], dims[1:], acts)]
        if change is not None:
            change(p, rng)
    x, box, types = _gas(counts, seed)
    model_dir.write_model_dir(str(folder), ps, rc=4.5, rc_ang=3.2, rs=1.6, radial_buffer=40, angular_buffer=780, tipos=counts,
                              precision=prec)
    got = []
    for host in (True, False):
        m = libstaf.StafModel(str(folder), precision=1 if prec == "double" else 0, full_virial=True, host_mlp=host)
        got.append(m.compute(x, box, types))
        m.close()
    (e0, f0, v0), (e1, f1, v1) = got
    assert np.isfinite(e0) and np.isfinite(f0).all() and (change is not None or np.abs(f0).max() > 0)
    assert abs(e1 - e0) <= (tol + (len(x) * 2.0 ** -24 if prec == "float" else 0.0)) * max(abs(e0), len(x) / 16)
    assert nerr(f1, f0) <= tol and nerr(v1, v0) <= tol


# Launches of more than 1024 atoms in double precision and of more than 2048 in single take more than four to a workgroup:
# eight (double, up to 2048; stacks that fit no more) or sixteen.  The species' last workgroups are ragged.
LARGER = [("double", 1e-11, (1004, 521)), ("double", 1e-11, (1506, 601)), ("float", 2e-5, (1506, 601))]


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol,counts", LARGER)
@pytest.mark.parametrize("hidden,last", [([], "linear"), ([], "tanh"), ([1], "linear"), ([16], "relu"), ([17, 15], "tanh"),
                                         ([300, 33], "linear"), ([16, 48, 16, 5], "linear")])
def test_network_stack_shapes_with_more_atoms_per_workgroup(tmp_path, prec, tol, counts, hidden, last):
    """The stacks of test_device_mlp_stack_shapes, beside one without and one with another number of hidden layers in the same launch, by
    eight and by sixteen atoms."""
    _device_and_host_network(tmp_path, prec, tol, (hidden, [] if hidden else [300, 33]), last, counts, seed=41)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol,hidden,counts", [("float", 2e-5, [400] * 6, (705, 1401)), ("float", 2e-5, [430] * 6, (705, 1401)),
                                                    ("double", 1e-11, [192] * 6, (705, 1401)), ("double", 1e-11, [200] * 6, (705, 1401)),
                                                    ("double", 1e-11, [400] * 6, (405, 701))])
def test_deep_stacks_with_more_atoms_per_workgroup(tmp_path, prec, tol, hidden, counts):
    """Sixteen atoms where their activations fit (2400 of 2496 features in single, 1152 of 1216 in double precision), eight
    where they do not (2592; 1248, 2400 of 2432: 160 KB of LDS).  float64: sums of at most 400 terms through seven layers."""
    _device_and_host_network(tmp_path, prec, tol, (hidden, [9]), "linear", counts, seed=43)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol,counts", LARGER)
def test_infinite_activations_with_more_atoms_per_workgroup(tmp_path, prec, tol, counts):
    """As test_infinite_activations_stay_out_of_the_padded_features, by eight and by sixteen atoms.  (The infinite feature
    saturates the whole tanh layer behind it: forces are zero.)"""
    def overflow(p, rng):
        n = p["mu"].shape[0]
        p["mu"][2] += 50.0
        W = [rng.normal(0, 1 / np.sqrt(a), (a, b)) for a, b in ((n, 5), (5, 7), (7, 6), (6, 1))]
        W[0][:, 3] = 0
        W[0][2, 3] = 0.9 * (np.finfo(np.float64).max if prec == "double" else float(np.finfo(np.float32).max))
        p["layers"] = [(w, rng.normal(0.3, 0.1, w.shape[1]), a) for w, a in zip(W, ("linear", "tanh", "tanh", "linear"))]
    _device_and_host_network(tmp_path, prec, tol, ([5], [5]), "linear", counts, seed=45, change=overflow)
