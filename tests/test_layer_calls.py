"""What ops.layer_* and the layers hand to the library, looked at without a GPU: the library's entries are replaced by ones that
take note of their arguments."""
import pytest
import torch

from alphanesgpu_amd import layers, ops

NF, NL, N, NR, NA, AR, AA = 2, 3, 5, 8, 28, 4, 6


class Calls(list):
    """(entry, arguments) of every call."""

    def entry(self, name, dtype, kinds):
        def fn(*args):
            assert len(args) == len(kinds.replace(" ", ""))
            self.append((name, args))
            return 0
        return fn

    def by_name(self, name, *args):
        self.append((name, args))


@pytest.fixture
def calls(monkeypatch):
    seen = Calls()
    monkeypatch.setattr(ops, "_entry", seen.entry)
    monkeypatch.setattr(ops, "call", seen.by_name)
    monkeypatch.setattr(ops, "_stream_addr", lambda: 0)
    monkeypatch.setattr(ops, "_stream", lambda: None)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda t: True), raising=False)
    return seen


def made(nt, rows3=None, rows2=None):
    """Arguments of ops.layer_forces of a species among nt."""
    ntc = nt * (nt + 1) // 2
    z = lambda *sh: torch.zeros(sh, dtype=torch.float64)
    i = lambda *sh: torch.zeros(sh, dtype=torch.int32)
    a = dict(netderiv2b=z(NF, NL, AR), netderiv3b=z(NF, NL, AA), x2b=z(NF, NL, NR), intder2b=z(NF, NL, 3, NR),
             intmap2b=i(NF, NL, NR + 1), alpha2b=z(nt, AR), emb2b=z(nt, AR), x3b=z(NF, NL, NA), x3bsupp=z(NF, NL, NR),
             intder3b=z(NF, NL, 3, 2 * NA), intder3bsupp=z(NF, NL, 3, NR), numtriplet=i(NF, NL), alpha3b=z(ntc, 3 * AA),
             emb3b=z(ntc, AA), type_map=i(N), tipos=i(nt), type_now=i(1))
    a["intmap3b"] = i(NF, NL, 2 * NA)
    return a


FORCES = ("netderiv2b", "netderiv3b", "x2b", "intder2b", "intmap2b", "alpha2b", "emb2b", "x3b", "x3bsupp", "intder3b",
          "intder3bsupp", "numtriplet", "alpha3b", "emb3b", "type_map", "tipos", "type_now")
FINGERPRINTS = ("x2b", "intmap2b", "alpha2b", "emb2b", "x3b", "x3bsupp", "alpha3b", "emb3b", "type_map", "numtriplet")
# a parameter of a species among three with fewer rows than the gradient has (2-body: 3, 3-body: 6), or more, or other columns
OTHER = [("emb2b", (2, AR)), ("alpha2b", (2, AR)), ("alpha3b", (5, 3 * AA)), ("emb3b", (5, AA)), ("emb3b", (7, AA)),
         ("emb3b", (6, AA - 1)), ("emb2b", (3 * AR,))]


@pytest.mark.parametrize("name,shape", OTHER)
def test_gradients_of_other_shapes_than_the_library_writes_are_refused(calls, name, shape):
    a = made(3)
    a[name] = torch.zeros(shape, dtype=torch.float64)
    with pytest.raises(ValueError):
        ops.layer_forces_grad(torch.zeros(NF, 3 * N, dtype=torch.float64), *[a[k] for k in FORCES])
    with pytest.raises(ValueError):
        ops.layer_fingerprints_grad(torch.zeros(NF, NL, AR + AA, dtype=torch.float64), *[a[k] for k in FINGERPRINTS])
    assert not calls


@pytest.mark.parametrize("nt", [1, 2, 3])
def test_gradients_have_the_shapes_that_the_library_writes(calls, nt):
    a = made(nt)
    ntc = nt * (nt + 1) // 2
    got = ops.layer_forces_grad(torch.zeros(NF, 3 * N, dtype=torch.float64), *[a[k] for k in FORCES])
    assert [tuple(t.shape) for t in got] == [(NF, NL, AR), (nt, AR), (nt, AR), (NF, NL, AA), (ntc, 3 * AA), (ntc, AA)]
    got = ops.layer_fingerprints_grad(torch.zeros(NF, NL, AR + AA, dtype=torch.float64), *[a[k] for k in FINGERPRINTS])
    assert [tuple(t.shape) for t in got] == [(nt, AR), (nt, AR), (ntc, 3 * AA), (ntc, AA)]
    assert [c[0] for c in calls] == ["staf_op_layer_forces_grad", "staf_op_layer_fingerprints_grad"]


def forward(a):
    """A physics_layer's and a force_layer's call."""
    ph = layers.physics_layer(torch.zeros(1, AR, dtype=torch.float64), torch.zeros(1, 3 * AA, dtype=torch.float64),
                              [torch.zeros(1, AR, dtype=torch.float64), torch.zeros(1, AA, dtype=torch.float64)])
    for own, k in (("alpha2b", "alpha2b"), ("type_emb_2b", "emb2b"), ("alpha3b", "alpha3b"), ("type_emb_3b", "emb3b")):
        setattr(ph, own, torch.nn.Parameter(a[k]))
    yield lambda: ph(a["x2b"], a["x3bsupp"], a["intmap2b"], a["x3b"], a["intmap3b"], a["numtriplet"], a["type_map"])
    fl = layers.force_layer.__new__(layers.force_layer)
    torch.nn.Module.__init__(fl)
    yield lambda: fl(a["netderiv2b"], a["x2b"], a["intder2b"], a["intmap2b"], a["alpha2b"], a["netderiv3b"], a["x3b"], a["x3bsupp"],
                     a["intder3b"], a["intder3bsupp"], a["intmap3b"], a["numtriplet"], a["alpha3b"], a["emb2b"], a["emb3b"],
                     a["type_map"], a["tipos"], a["type_now"])


def test_layers_take_the_single_calls(calls):
    for layer in forward(made(3)):
        layer()
    assert [c[0] for c in calls] == ["staf_op_layer_fingerprints", "staf_op_layer_forces"]


@pytest.mark.parametrize("name,shape", [("alpha3b", (5, 3 * AA)), ("emb3b", (5, AA)), ("emb3b", (7, AA))])
def test_layers_of_parameters_with_other_rows_take_the_ops(calls, name, shape):
    """The forward ops read 2 nt - 1 rows and take such parameters; autograd refuses their gradients by the shapes."""
    a = made(3)
    a[name] = torch.zeros(shape, dtype=torch.float64)
    for layer in forward(a):
        try:
            layer()
        except ValueError as e:   # (rows of alpha3b that are those of no number of species)
            assert name == "alpha3b" and "is not nt(nt+1)/2" in str(e)
    assert calls and not any("layer" in c[0] for c in calls)


@pytest.mark.parametrize("what,error", [(lambda m: m.long(), TypeError), (lambda m: m.transpose(0, 1).contiguous().transpose(0, 1), ValueError),
                                        (lambda m: torch.stack([m, m], -1)[..., 0], ValueError), (lambda m: None, AttributeError)])
def test_layers_refuse_a_map_of_the_triplets_that_the_ops_refuse(calls, what, error):
    """Another type, rows that lie otherwise and no map at all: no kernel reads it, and the ops refuse it all the same."""
    a = made(2)
    a["intmap3b"] = what(a["intmap3b"])
    for layer in forward(a):
        with pytest.raises(error):
            layer()
    assert not calls


@pytest.mark.parametrize("rows", [slice(0, NL), slice(2, N), slice(1, 1), slice(1, 2)])
@pytest.mark.parametrize("frames", [1, 2])
def test_a_map_of_the_triplets_is_taken_where_the_whole_test_takes_it(rows, frames):
    """check_rows knows a map by its strides beside x3b's: the same verdict as of the test of every dimension, for slices of a
    descriptor output, copies of them and maps of other widths."""
    def verdict(f, *args):
        try:
            f(*args)
        except (TypeError, ValueError) as e:
            return type(e), str(e)

    def whole(x3b, intmap3b):
        v = ops._Views()
        v(x3b), v(ops._i32(intmap3b))
    out = {w: torch.zeros(frames, N, w, dtype=torch.int32 if w > NA else torch.float64)[:, rows] for w in (NA, 2 * NA, 2 * NA + 1)}
    maps = [out[2 * NA], out[2 * NA].clone(), out[2 * NA + 1], out[2 * NA + 1][..., :2 * NA], out[2 * NA].flip(1), out[2 * NA].long()]
    for x3b in (out[NA], out[NA].clone()):
        for m in maps:
            assert verdict(ops.check_rows, x3b, m) == verdict(whole, x3b, m)
        assert verdict(ops.check_rows, x3b, maps[x3b.is_contiguous() and frames > 1]) is None


@pytest.mark.parametrize("frozen", ["2", "3"])
def test_a_body_whose_parameters_are_frozen_gets_no_gradient_kernels(calls, frozen):
    """The library is handed null for the gradients of a body that needs none, and makes no launches for it."""
    a = made(2)
    ph = layers.physics_layer(a["alpha2b"], a["alpha3b"], [a["emb2b"], a["emb3b"]])
    for name, p in ph.named_parameters():
        p.requires_grad_(frozen not in name)
    out = ph(a["x2b"], a["x3bsupp"], a["intmap2b"], a["x3b"], a["intmap3b"], a["numtriplet"], a["type_map"])
    out.backward(torch.zeros_like(out))
    name, args = calls[-1]
    assert name == "staf_op_layer_fingerprints_grad"
    assert [v is None for v in args[-6:-2]] == [frozen == "2"] * 2 + [frozen == "3"] * 2
    assert [p.grad is None for _, p in ph.named_parameters()] == [frozen in n for n, _ in ph.named_parameters()]
