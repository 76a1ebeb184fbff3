"""PyTorch layer shells (alphanesgpu_amd/layers.py) with the reference's gradient routing.

A small two-species model is assembled from the layers the way the reference's training step assembles its TF
modules (STAF/staf_models/staf_model.py:168-208: descriptor tensors split per species -> physics layer, lognorm,
Dense stack -> dE/dAF by differentiation of the network -> force layer), a loss
L = sum_b cE_b E_b + sum Q.F (+ sum Qw.W) is back-propagated with torch.autograd, and every kind of trainable parameter is checked against central finite
differences of the same loss evaluated through the CPU oracle pipeline.  That pins the routing (which gradient op
feeds which input, the second-order path through the network, the squared embeddings), not the ops themselves,
which have their own parity tests."""
import numpy as np
import pytest


def _two_frames():
    from test_oracle_pins import cluster
    a = cluster([4, 5], seed=21)
    b = cluster([4, 5], seed=22)
    return np.concatenate([a[0], b[0]]), np.concatenate([a[1], b[1]]), a[2], a[3]


def _oracle_loss(oracle, frames, model, cE, Q, Qw, nr, na, rc, ra, rs):
    from test_oracle_pins import energy_and_forces
    pos, box, tipos, type_map = frames
    E, F, W, _, _ = energy_and_forces(oracle, pos, box, tipos, type_map, model, nr=nr, na=na, rc=rc, ra=ra, rs=rs,
                                      virial=Qw is not None)
    L = float(np.dot(cE, E) + np.sum(Q * F))
    if Qw is not None:
        L += float(np.sum(Qw * W))
    return L


@pytest.mark.gpu
@pytest.mark.parametrize("virial", [False, True])
def test_autograd_through_the_layers_matches_finite_differences_of_the_oracle(oracle, virial):
    import torch
    from alphanesgpu_amd import layers
    from test_oracle_pins import small_model
    dev = torch.device("cuda:0")
    nr, na, rc, ra, rs = 16, 45, 4.5, 3.4, 1.6
    frames = _two_frames()
    pos, box, tipos, type_map = frames
    nf, nt = pos.shape[0], len(tipos)
    model = small_model(nt, (3, 2), (2, 2, 3), seed=13, hidden=5, dense=True)
    rng = np.random.default_rng(4)
    cE = rng.standard_normal(nf)
    Q = rng.standard_normal((nf, pos.shape[1]))
    Qw = rng.standard_normal((nf, 9)) if virial else None

    T = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(dev)
    tpos, tbox, ttm, ttp = T(pos), T(box), T(type_map), T(tipos)
    desc = layers.descriptor_layer(rc, nr, ra, na, pos.shape[1] // 3, tbox, rs, nf)
    rad, ang, sup, im2, im3, d2, d3, d3s, ntr = desc(tpos, tbox)
    flayer = layers.force_virial_layer(nr, na) if virial else layers.force_layer(nr, na)
    phys, logn, dense = [], [], []
    for m in model:
        phys.append(layers.physics_layer(T(m["alpha2b"]), T(m["alpha3b"]),
                                         [T(np.sqrt(m["emb2b"])), T(np.sqrt(m["emb3b"]))]))
        logn.append(layers.lognorm_layer(T(m["mu"])))
        dense.append([(torch.nn.Parameter(T(W)), torch.nn.Parameter(T(b)), act) for W, b, act in m["layers"]])

    E = torch.zeros(nf, dtype=torch.float64, device=dev)
    F = torch.zeros((nf, pos.shape[1]), dtype=torch.float64, device=dev)
    Wv = torch.zeros((nf, 9), dtype=torch.float64, device=dev)
    o = 0
    for k, n in enumerate(tipos):
        s = slice(o, o + int(n))
        o += int(n)
        c = lambda a: a[:, s]
        af = phys[k](c(rad), c(sup), c(im2), c(ang), c(im3), c(ntr), ttm)
        x = logn[k](af)
        for W, b, act in dense[k]:
            x = x @ W + b
            if act == "tanh":
                x = torch.tanh(x)
        e_atoms = x[..., 0]
        E = E + 0.5 * e_atoms.sum(dim=1)
        net_der, = torch.autograd.grad(e_atoms.sum(), af, create_graph=True)
        Ar = phys[k].nalpha_r
        args = (net_der[..., :Ar].contiguous(), c(rad), c(d2), c(im2), phys[k].alpha2b,
                net_der[..., Ar:].contiguous(), c(ang), c(sup), c(d3), c(d3s), c(im3), c(ntr), phys[k].alpha3b,
                phys[k].type_emb_2b, phys[k].type_emb_3b, ttm, ttp, k)
        if virial:
            f, w = flayer(*args, tpos, tbox)
            Wv = Wv + w
        else:
            f = flayer(*args)
        F = F + f
    L = (T(cE) * E).sum() + (T(Q) * F).sum()
    if virial:
        L = L + (T(Qw) * Wv).sum()
    L.backward()

    L0 = _oracle_loss(oracle, frames, model, cE, Q, Qw, nr, na, rc, ra, rs)
    assert abs(L.item() - L0) <= 1e-10 * max(1.0, abs(L0))

    def fd(k, key, idx, layer=None, h=1e-5):
        """central difference of the oracle loss in one entry of one parameter array"""
        vals = []
        for sgn in (+1, -1):
            mm = [dict(m, layers=[(W.copy(), b.copy(), a) for W, b, a in m["layers"]]) for m in model]
            if layer is None:
                arr = mm[k][key].copy()
                if key in ("emb2b", "emb3b"):        # the trainable quantity is the unsquared embedding
                    r = np.sqrt(arr)
                    r[idx] += sgn * h
                    arr = r * r
                else:
                    arr[idx] += sgn * h
                mm[k][key] = arr
            else:
                mm[k]["layers"][layer][key][idx] += sgn * h
            vals.append(_oracle_loss(oracle, frames, mm, cE, Q, Qw, nr, na, rc, ra, rs))
        return (vals[0] - vals[1]) / (2 * h)

    g = lambda p: p.grad.detach().cpu().numpy()
    checks = []
    for k in range(nt):
        Aa = phys[k].nalpha_a
        checks += [(g(phys[k].alpha2b)[1, 0], fd(k, "alpha2b", (1, 0))),
                   (g(phys[k].alpha2b)[0, 1], fd(k, "alpha2b", (0, 1))),
                   (g(phys[k].alpha3b)[0, 1], fd(k, "alpha3b", (0, 1))),               # alpha1
                   (g(phys[k].alpha3b)[1, Aa], fd(k, "alpha3b", (1, Aa))),             # alpha2
                   (g(phys[k].alpha3b)[2, 2 * Aa + 1], fd(k, "alpha3b", (2, 2 * Aa + 1))),   # beta
                   (g(phys[k].type_emb_2b)[1, 1], fd(k, "emb2b", (1, 1))),
                   (g(logn[k].mu)[2], fd(k, "mu", (2,))),
                   (g(dense[k][0][0])[1, 2], fd(k, 0, (1, 2), layer=0)),
                   (g(dense[k][1][1])[3], fd(k, 1, (3,), layer=1))]
        # the reference's gradient ops return zeros for the 3-body embedding (its kernels never fill that output):
        # the routing hands exactly that on
        assert not g(phys[k].type_emb_3b).any()
    got = np.array([a for a, _ in checks])
    want = np.array([b for _, b in checks])
    scale = np.abs(want).max()
    # finite differences with h = 1e-5 on a smooth function of O(1) curvature: ~1e-9 absolute
    assert np.all(np.abs(got - want) <= 2e-7 * scale), (got, want)
    assert np.count_nonzero(np.abs(want) > 1e-6 * scale) >= len(want) - 4


def test_layer_classes_have_the_reference_signatures():
    """Names and argument lists of STAF/source_routine/*.py (descriptor_builder.py:16,31, physics_layer_mod.py:10,33,
    55,59, force_layer_mod.py:9,25-27,78,90-92)."""
    import inspect
    from alphanesgpu_amd import layers
    sig = lambda f: [p for p in inspect.signature(f).parameters if p != "self"]
    assert sig(layers.descriptor_layer.__init__)[:8] == ["rc", "rad_buff", "rc_ang", "ang_buff", "N", "box_example",
                                                         "Rs", "maxbatch"]
    assert sig(layers.descriptor_layer.forward) == ["pos", "box"]
    assert sig(layers.physics_layer.__init__) == ["init_alpha2b", "init_alpha3b", "initial_type_emb"]
    assert sig(layers.physics_layer.forward) == ["x2b", "x3bsupp", "intmap2b", "x3b", "intmap3b", "numtriplet",
                                                 "type_map"]
    assert sig(layers.lognorm_layer.__init__) == ["mu"] and sig(layers.lognorm_layer.forward) == ["restot"]
    call = ["net_der_r", "x2b", "intder2b", "int2b", "alpha2b", "net_der_a", "x3b", "x3bsupp", "intder3b",
            "intder3bsupp", "int3b", "numtriplet", "alpha3b", "type_emb_2b", "type_emb_3b", "type_map", "tipos",
            "type_now"]
    assert sig(layers.force_layer.__init__) == ["radbuff", "angbuff"] and sig(layers.force_layer.forward) == call
    assert sig(layers.force_virial_layer.__init__) == ["radbuff", "angbuff", "with_grad"]
    assert sig(layers.force_virial_layer.forward) == call + ["pos", "box"]


@pytest.mark.parametrize("two,three,want", [
    ("float64", "float64", ["staf_op_forces_f64"]), ("float32", "float32", ["staf_op_forces_f32"]),
    ("float32", "float64", ["staf_op_force_doublets_f32", "staf_op_force_tripl_f64"]),
    ("float64", "float32", ["staf_op_force_doublets_f64", "staf_op_force_tripl_f32"])])
def test_force_layer_takes_the_bodies_in_precisions_of_their_own(monkeypatch, two, three, want):
    """2-body and 3-body tensors of different precisions go to the two force ops, each in its own (one op for both would
    read one body's memory as the other's); the forces are their sum in the wider one, and its gradient goes back to each
    body in the body's precision.  Which library calls are made, on host tensors with the calls themselves replaced."""
    import torch
    from alphanesgpu_amd import layers, ops
    d2, d3 = getattr(torch, two), getattr(torch, three)
    nf, N, nr, na, Ar, Aa = 1, 3, 4, 6, 2, 3
    z = lambda dt, *sh: torch.ones(sh, dtype=dt)
    zi = lambda *sh: torch.zeros(sh, dtype=torch.int32)
    layer = layers.force_layer(nr, na)
    made = []
    monkeypatch.setattr(ops, "call", lambda name, *args: made.append(name))
    monkeypatch.setattr(ops, "_stream", lambda: None)
    g2, g3 = z(d2, nf, N, Ar).requires_grad_(True), z(d3, nf, N, Aa).requires_grad_(True)
    f = layer(g2, z(d2, nf, N, nr), z(d2, nf, N, 3 * nr), zi(nf, N, nr + 1), z(d2, 1, Ar), g3, z(d3, nf, N, na),
              z(d3, nf, N, nr), z(d3, nf, N, 3 * na * 2), z(d3, nf, N, 3 * nr), zi(nf, N, na * 2), zi(nf, N), z(d3, 1, 3 * Aa),
              z(d2, 1, Ar), z(d3, 1, Aa), zi(N), zi(1), 0)
    assert made == want
    came = {}
    monkeypatch.setattr(ops, "compute_force_radial_grad", lambda q, g, *a: came.update(two=q.dtype) or (g, a[3], a[4]))
    monkeypatch.setattr(ops, "compute_force_tripl_grad", lambda q, g, *a: came.update(three=q.dtype) or (g, a[6], a[7]))
    torch.autograd.grad(f.sum(), [g2, g3])
    assert came == dict(two=d2, three=d3)
    assert f.dtype == torch.promote_types(d2, d3) and f.shape == (nf, 3 * N)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("nr,na,counts,own_map", [(60, 1770, (32, 64), True), (60, 1770, (32, 64), False),
                                                  (64, 2016, (96, 0), True), (65, 2080, (1, 95), False),
                                                  (130, 2080, (50, 46), True)])
def test_forces_in_one_op_agree_with_the_two_force_ops(dtype, nr, na, counts, own_map):
    """ops.compute_forces against ComputeForceRadial + ComputeForceTripl of the same centres, with the virial: slot
    counts around a wave, an empty and a one-atom species, the descriptor op's map and a copy of it (a caller's map)."""
    import torch
    from alphanesgpu_amd import ops, synth
    dev, dt = torch.device("cuda:0"), getattr(torch, dtype)
    frames = [synth.water_frame((4, 4, 2), 9.86, 0.05, seed) for seed in (3, 4)]
    N = 96
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(dev)
    tpos, tbox = (T(np.stack(a)).to(dt) for a in zip(*frames))
    tm, tp = T(np.repeat(np.arange(2, dtype=np.int32), counts)), T(np.array(counts, np.int32))
    ops.construct_descriptors_light(synth.RC, nr, na, N, tbox, synth.RS, synth.RA, 2, dtype=dt)
    rad, ang, sup, im2, im3, d2, d3, d3s, ntr = ops.compute_descriptors_light(tpos, tbox)
    if not own_map:
        im2 = im2.clone()
    g = torch.Generator(device=dev)
    g.manual_seed(5)
    o = 0
    for k, (p, n) in enumerate(zip(synth.fingerprint_params(2, dtype=getattr(np, dtype)), counts)):
        c = lambda t: t[:, o:o + n]
        P = {q: T(v) for q, v in p.items()}
        G2 = torch.randn((2, n, P["emb2b"].shape[1]), dtype=dt, device=dev, generator=g)
        G3 = torch.randn((2, n, P["emb3b"].shape[1]), dtype=dt, device=dev, generator=g)
        tn = T(np.array([k], np.int32))
        for virial in [(), (tpos, tbox)]:
            a = ops.compute_force_radial(G2, c(d2), c(im2), c(rad), P["alpha2b"], P["emb2b"], tm, tp, tn, *virial)
            b = ops.compute_force_tripl(G3, c(sup), c(ang), c(d3s), c(d3), c(im2), c(im3), P["alpha3b"], P["emb3b"], tm, tp,
                                        tn, c(ntr), *virial)
            f = ops.compute_forces(G3, G2, c(sup), c(ang), c(d3s), c(d3), c(rad), c(d2), c(im2), c(im3), P["alpha3b"],
                                   P["emb3b"], P["alpha2b"], P["emb2b"], tm, tp, tn, c(ntr), *virial)
            for x, y, z, terms in zip(*([(v,) for v in (a, b, f)] if not virial else (a, b, f)), (128, 8 * N)):
                assert z.shape == x.shape
                # the same terms, added in another order: a force is a sum of at most 2 x 60 slot terms per body, a
                # virial of 2 x 60 terms per atom in a tree; each of `terms` additions rounds a partial sum that is at
                # most a few times the largest result
                bound = terms * torch.finfo(dt).eps * (x.abs().max() + y.abs().max())
                assert (z - (x + y)).abs().max() <= bound, (k, virial != (), (z - (x + y)).abs().max(), bound)
        o += n


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_forces_in_one_op_do_not_read_the_padding_of_the_rows(dtype):
    """Descriptor rows of another origin may hold anything beyond an atom's neighbours (the force ops take the counts from
    the map): with NaN there, ops.compute_forces and the force layers give the same bits as with the descriptor op's
    zeros, as the two ops do."""
    import torch
    from alphanesgpu_amd import layers, ops, synth
    dev, dt = torch.device("cuda:0"), getattr(torch, dtype)
    b = synth.water_batch("water96")
    counts, nr, na, N = [int(c) for c in b["tipos"]], 60, 1770, len(b["type_map"])
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(dev)
    tpos, tbox = (T(np.tile(b[q][:1], (2, 1))).to(dt) for q in ("pos", "box"))
    tm, tp = T(b["type_map"].astype(np.int32)), T(np.array(counts, np.int32))
    ops.construct_descriptors_light(synth.RC, nr, na, N, tbox, synth.RS, synth.RA, 2, dtype=dt)
    rad, ang, sup, im2, im3, d2, d3, d3s, ntr = ops.compute_descriptors_light(tpos, tbox)
    pad = torch.arange(nr, device=dev) >= im2[..., :1]
    assert bool(pad.any())
    nan = lambda t: t.masked_fill(pad.unsqueeze(2) if t.dim() == 4 else pad, float("nan"))
    P = {q: T(v) for q, v in synth.fingerprint_params(2, dtype=getattr(np, dtype))[0].items()}
    g = torch.Generator(device=dev)
    g.manual_seed(5)
    n = counts[0]
    G2 = torch.randn((2, n, P["emb2b"].shape[1]), dtype=dt, device=dev, generator=g)
    G3 = torch.randn((2, n, P["emb3b"].shape[1]), dtype=dt, device=dev, generator=g)
    layer = layers.force_virial_layer(nr, na)
    out = []
    for f in (lambda t: t, nan):
        c = lambda t: t[:, :n]
        R, S, D2, D3s = (c(f(t)) for t in (rad, sup, d2.reshape(2, N, 3, nr), d3s.reshape(2, N, 3, nr)))
        D2, D3s = D2.reshape(c(d2).shape), D3s.reshape(c(d3s).shape)
        out.append(ops.compute_forces(G3, G2, S, c(ang), D3s, c(d3), R, D2, c(im2), c(im3), P["alpha3b"], P["emb3b"],
                                      P["alpha2b"], P["emb2b"], tm, tp, 0, c(ntr), tpos, tbox) +
                   layer(G2, R, D2, c(im2), P["alpha2b"], G3, c(ang), S, c(d3), D3s, c(im3), c(ntr), P["alpha3b"],
                         P["emb2b"].sqrt(), P["emb3b"].sqrt(), tm, tp, 0, tpos, tbox))
    for x, y in zip(*out):
        assert bool(torch.isfinite(x).all()) and torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("counts", [(32, 64), (96, 0), (1, 95)])
@pytest.mark.parametrize("virial", [False, True])
def test_layers_as_single_calls_give_the_bits_of_the_ops_on_squared_embeddings(dtype, counts, virial):
    """physics_layer, force_layer and force_virial_layer square the embeddings where the kernels read them and write the
    gradients of the unsquared ones; the values and gradients of the op-by-op route on torch's squares, to the last bit
    (the same sums, and g (2 e) is one rounding either way), with a species without atoms and one of a single atom."""
    import torch
    from alphanesgpu_amd import layers, ops, synth
    dev, dt = torch.device("cuda:0"), getattr(torch, dtype)
    nr, na, N = 60, 1770, 96
    frames = [synth.water_frame((4, 4, 2), 9.86, 0.05, seed) for seed in (3, 4)]
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(dev)
    tpos, tbox = (T(np.stack(a)).to(dt) for a in zip(*frames))
    tm, tp = T(np.repeat(np.arange(2, dtype=np.int32), counts)), T(np.array(counts, np.int32))
    ops.construct_descriptors_light(synth.RC, nr, na, N, tbox, synth.RS, synth.RA, 2, dtype=dt)
    rad, ang, sup, im2, im3, d2, d3, d3s, ntr = ops.compute_descriptors_light(tpos, tbox)
    g = torch.Generator(device=dev)
    g.manual_seed(5)
    rand = lambda *sh: torch.randn(sh, dtype=dt, device=dev, generator=g)
    o = 0
    for k, (p, n) in enumerate(zip(synth.fingerprint_params(2, dtype=getattr(np, dtype)), counts)):
        c = lambda t: t[:, o:o + n]
        ph = layers.physics_layer(T(p["alpha2b"]), T(p["alpha3b"]), [0.5 + rand(*p["emb2b"].shape).abs(),
                                                                      T(p["emb3b"]) * (0.5 + rand(*p["emb3b"].shape).abs())])
        par = list(ph.parameters())
        U, Q, Qw = rand(2, n, ph.output_dim), rand(2, 3 * N), rand(2, 9)
        G = [rand(2, n, w).requires_grad_(True) for w in (ph.nalpha_r, ph.nalpha_a)]
        af = ph(c(rad), c(sup), c(im2), c(ang), c(im3), c(ntr), tm)
        af_ops = torch.cat([layers._SortProj.apply(c(rad), c(im2), ph.alpha2b, torch.square(ph.type_emb_2b), tm),
                            layers._SortProj3body.apply(c(ang), c(sup), c(im3), c(im2), ph.alpha3b,
                                                        torch.square(ph.type_emb_3b), tm, c(ntr))], dim=2)
        assert torch.equal(af, af_ops)
        for x, y in zip(torch.autograd.grad(af, par, U), torch.autograd.grad(af_ops, par, U)):
            assert torch.equal(x, y)
        layer = layers.force_virial_layer(nr, na) if virial else layers.force_layer(nr, na)
        box = (tpos, tbox) if virial else (None, None)
        F = layer(G[0], c(rad), c(d2), c(im2), ph.alpha2b, G[1], c(ang), c(sup), c(d3), c(d3s), c(im3), c(ntr), ph.alpha3b,
                  ph.type_emb_2b, ph.type_emb_3b, tm, tp, k, *(box if virial else ()))
        tn = T(np.array([k], np.int32))
        F_ops = layers._Forces.apply(G[0], G[1], c(rad), c(d2), c(im2), ph.alpha2b, torch.square(ph.type_emb_2b), c(ang), c(sup),
                                     c(d3), c(d3s), c(im3), c(ntr), ph.alpha3b, torch.square(ph.type_emb_3b), tm, tp, tn, *box)
        F, F_ops = ([t] if not virial else list(t) for t in (F, F_ops))
        assert all(torch.equal(x, y) for x, y in zip(F, F_ops))
        up = [Q, Qw][:len(F)]
        wanted = G + [ph.alpha2b, ph.alpha3b, ph.type_emb_2b, ph.type_emb_3b]
        for x, y in zip(torch.autograd.grad(F, wanted, up, retain_graph=True), torch.autograd.grad(F_ops, wanted, up)):
            assert torch.equal(x, y)
        x, = torch.autograd.grad(F, G[1:], up)   # (one body alone, one output alone)
        if n:
            assert bool(x.abs().max() > 0)
        o += n


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["layer_forces", "compute_forces", "force_total"])
def test_arguments_that_are_not_dense_are_copied_to_places_of_their_own(entry):
    """Halves of one tensor and strided parameters: every one is copied for the call, and the copies live until it is made."""
    import torch
    from alphanesgpu_amd import ops, synth
    dev, dt = torch.device("cuda:0"), torch.float64
    pos, box = synth.water_frame((4, 4, 2), 9.86, 0.05, 3)
    N, n = 96, 32
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(dev)
    tpos, tbox = T(pos[None]), T(box[None])
    tm, tp, tn = T(np.repeat(np.arange(2, dtype=np.int32), (32, 64))), T(np.array([32, 64], np.int32)), T(np.zeros(1, np.int32))
    ops.construct_descriptors_light(synth.RC, 60, 1770, N, tbox, synth.RS, synth.RA, 1, dtype=dt)
    rad, ang, sup, im2, im3, d2, d3, d3s, ntr = ops.compute_descriptors_light(tpos, tbox)
    c = lambda t: t[:, :n]
    P = {q: T(v) for q, v in synth.fingerprint_params(2, dtype=np.float64)[0].items()}
    g = torch.Generator(device=dev)
    g.manual_seed(5)
    Ar, Aa = P["emb2b"].shape[1], P["emb3b"].shape[1]
    G = torch.randn((1, n, Ar + Aa), dtype=dt, device=dev, generator=g)
    strided = lambda t: torch.stack([t, torch.full_like(t, float("nan"))], -1)[..., 0]
    forms = []
    for form in (lambda t: t.contiguous(), strided):
        G2, G3 = form(G[..., :Ar]), form(G[..., Ar:])
        Q = {k: form(P[k]) for k in ("alpha2b", "alpha3b", "emb2b", "emb3b")}
        if entry == "layer_forces":
            f = ops.layer_forces(G2, G3, c(rad), c(d2), c(im2), Q["alpha2b"], Q["emb2b"], c(ang), c(sup), c(d3), c(d3s), c(ntr),
                                 Q["alpha3b"], Q["emb3b"], tm, tp, tn)
        else:
            args = (G3, G2, c(sup), c(ang), c(d3s), c(d3), c(rad), c(d2), c(im2), c(im3), Q["alpha3b"], Q["emb3b"],
                    Q["alpha2b"], Q["emb2b"], tm, tp, tn, c(ntr))
            if entry == "compute_forces":
                f = ops.compute_forces(*args)
            else:
                slots, own = ops.compute_forces_slots(*args)
                none = [torch.zeros((1, 64, *slots.shape[2:]), dtype=dt, device=dev), torch.zeros((1, 64, *own.shape[2:]), dtype=dt, device=dev)]
                f = ops.force_total(im2, [32, 64], [form(slots), form(none[0])], [form(own), form(none[1])])
        forms.append(f)
    assert torch.equal(*forms)


@pytest.mark.gpu
@pytest.mark.parametrize("frozen", ["2", "3"])
def test_gradients_beside_a_frozen_body_have_the_bits_of_both(frozen):
    """physics_layer with the parameters of one body frozen: the other body's gradients, to the last bit."""
    import torch
    from alphanesgpu_amd import layers, ops, synth
    dev, dt = torch.device("cuda:0"), torch.float64
    pos, box = synth.water_frame((4, 4, 2), 9.86, 0.05, 3)
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(dev)
    ops.construct_descriptors_light(synth.RC, 60, 1770, 96, T(box[None]), synth.RS, synth.RA, 1, dtype=dt)
    rad, ang, sup, im2, im3, _, _, _, ntr = ops.compute_descriptors_light(T(pos[None]), T(box[None]))
    tm = T(np.repeat(np.arange(2, dtype=np.int32), (32, 64)))
    p = synth.fingerprint_params(2, dtype=np.float64)[0]
    ph = layers.physics_layer(T(p["alpha2b"]), T(p["alpha3b"]), [T(p["emb2b"]), T(p["emb3b"])])
    c = lambda t: t[:, :32]
    g = torch.Generator(device=dev)
    g.manual_seed(5)
    U = torch.randn((1, 32, ph.output_dim), dtype=dt, device=dev, generator=g)
    got = []
    for freeze in (False, True):
        ph.zero_grad()
        for name, q in ph.named_parameters():
            q.requires_grad_(not freeze or frozen not in name)
        ph(c(rad), c(sup), c(im2), c(ang), c(im3), c(ntr), tm).backward(U)
        got.append({name: q.grad for name, q in ph.named_parameters()})
    for name, x in got[1].items():
        assert x is None if frozen in name else torch.equal(x, got[0][name])
