"""Which kernel form a launch of fingerprints takes, and the table that a loaded model's launches read (csrc/staf_step.hpp): host
code, compiled for the host alone."""
import math
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "%s/alphanesgpu_amd/csrc/staf_step.hpp"
#include <stdio.h>
#include <stdlib.h>
using namespace staf;
template <typename real>
static void line(int nr, int nt, int Ar, int Aa, int centres) {
  RowsLaunch<real> L;
  for (int k = 0; k < nt; k++) L.add(nr, nr * (nr - 1) / 2, nt, Ar, Aa, (centres + k) / nt);
  printf("%%d %%zu %%zu\n", L.waves(), rows_lds<real, 4>(nr, nt, Ar, Aa), rows_lds<real, 8>(nr, nt, Ar, Aa));
}
int main(int argc, char** argv) {
  if (argc > 1) {   // argv[1] species, argv[2] channels, then alpha3b and emb3b on stdin: the table
    const int nt = atoi(argv[1]), Aa = atoi(argv[2]), nsig = 2 * nt - 1;
    std::vector<double> al((size_t)nsig * Aa * 3), emb((size_t)nsig * Aa);
    for (double& v : al) if (scanf("%%lf", &v) != 1) return 1;
    for (double& v : emb) if (scanf("%%lf", &v) != 1) return 1;
    for (double v : step_table_host(al.data(), emb.data(), nt, Aa)) printf("%%.17g\n", v);
    return 0;
  }
  int f64, nr, nt, Ar, Aa, centres;
  while (scanf("%%d %%d %%d %%d %%d %%d", &f64, &nr, &nt, &Ar, &Aa, &centres) == 6)
    if (f64) line<double>(nr, nt, Ar, Aa, centres);
    else line<float>(nr, nt, Ar, Aa, centres);
}
""" % ROOT


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("step_form")
    src, exe = str(d / "rule.hip"), str(d / "rule")
    open(src, "w").write(SOURCE)
    subprocess.check_call(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-x", "hip", "--offload-host-only", src, "-o", exe])

    def ask(*case, args=()):
        r = subprocess.run([exe, *map(str, args)], input=" ".join(map(repr, case)), stdout=subprocess.PIPE, text=True, check=True)
        return tuple(map(float if args else int, r.stdout.split()))
    return ask


def test_the_lds_is_that_of_the_workgroups_that_are_launched(rule):
    """Three species in double precision: the 2-body workgroups' LDS lies in the same allocation as the 3-body ones' and does not
    count on top of it, and every number of waves has a size of its own."""
    for nr in (60, 64):
        for Ar, Aa in ((20, 40), (24, 44), (1000, 60)):
            got = rule(1, nr, 3, Ar, Aa, 100)
            rows = nr + 9
            for waves, lds in zip((4, 8), got[1:]):
                three = (3 * rows * 32 + 5 * rows + waves * Aa) * 8 + (rows + 9) * 4
                two = 2 * 3 * Ar * 8 + waves * nr * 12
                assert lds == max(-(-three // 16) * 16, two)


@pytest.mark.parametrize("f64,nr,nt,centres,waves", [
    # few centres: eight waves
    (1, 60, 2, 96, 8), (1, 60, 2, 448, 8), (1, 60, 2, 449, 4), (1, 60, 3, 448, 8), (0, 60, 4, 448, 8), (1, 64, 3, 100, 8),
    # four workgroups per CU in double, three in single precision: any number of centres
    (1, 60, 1, 24576, 4), (1, 60, 2, 24576, 4), (1, 64, 2, 24576, 4), (1, 32, 3, 24576, 4), (0, 60, 2, 24576, 4), (0, 64, 5, 24576, 4),
    # fewer: launches whose centres are resident at once, two (45 of 128 pieces of 1280 bytes each) and three per CU
    (1, 60, 3, 512, 4), (1, 60, 3, 513, 0), (1, 48, 3, 768, 4), (1, 48, 3, 769, 0), (1, 60, 3, 24576, 0), (0, 60, 6, 512, 4),
    (0, 60, 6, 513, 0),
    # one workgroup per CU, none
    (1, 64, 5, 256, 8), (1, 64, 5, 257, 0), (1, 64, 8, 64, 0)])
def test_a_launch_whose_tables_leave_few_waves_takes_the_staged_form(rule, f64, nr, nt, centres, waves):
    assert rule(f64, nr, nt, 20, 40, centres)[0] == waves


@pytest.mark.parametrize("active,largest,rows", [((14, 13, 13), 2.0, (128, 64)), ((3, 17, 0), 16.0, (1024, 1024)),
                                                 ((1, 0, 5), 16.5, (2048, 0)), ((20, 1, 5), 64.0, (4096, 0)), ((1, 0, 5), 64.5, (0, 0)),
                                                 ((40, 40, 40), 0.01, (1, 1)), ((0, 0, 0), 2.0, (1, 1))])
def test_a_table_is_as_wide_as_the_channels_in_use(rule, active, largest, rows):
    """Two species, forty channels of which a class has `active`: the pitch is the largest number in whole sixteens, the rows those
    that the largest exponent needs, and every entry lies where the layout says."""
    rng = np.random.Generator(np.random.Philox(3))
    al = rng.uniform(-0.009, 0.009, (3, 40, 3))
    emb = np.zeros((3, 40))
    for s, n in enumerate(active):
        emb[s, np.sort(rng.permutation(40)[:n])] = rng.uniform(0.1, 1.0, n)
    for s in range(3):   # (the largest exponents are those of channels in use)
        if active[s]:
            c = int(np.flatnonzero(emb[s])[-1])
            al[s, c] = largest / 2, -largest if rows[1] != 64 else -1.0, largest
    t = np.array(rule(*al.reshape(-1).tolist(), *emb.reshape(-1).tolist(), args=(2, 40)))
    pitch = max(16, -(-max(active) // 16) * 16)
    N, Np = rows
    assert t[:4].tolist() == [N, max(active), Np, pitch] and t[8:11].tolist() == list(active)
    par = t[32:32 + 3 * pitch * 4].reshape(3, pitch, 4)
    o = 32 + 3 * pitch * 4
    beta = t[o:o + 3 * pitch].reshape(3, pitch)
    o += 3 * pitch
    n = 3 * (N + 1) * pitch if N else 0
    row = t[o:o + n].reshape(3, -1, pitch)
    o += n
    n = 3 * (Np + 1) * pitch * 2 if Np else 0
    pair = t[o:o + n].reshape(3, -1, pitch, 2)
    assert o + n == len(t)
    # the roundings of the entry, of math.exp and of its argument
    close = lambda v, a, i, n: abs(v / math.exp(a * i / n) - 1) <= (4 + abs(a)) * 2.0 ** -53
    for s in range(3):
        on = np.flatnonzero(emb[s])
        assert np.array_equal(par[s, :len(on)], np.column_stack([al[s, on, 0], al[s, on, 1], emb[s, on], on]))
        assert np.array_equal(beta[s, :len(on)], al[s, on, 2])
        assert not par[s, len(on):].any() and not beta[s, len(on):].any()
        for c, a in enumerate(on):
            for i in range(0, N + 1, max(1, N // 7)) if N else ():
                assert close(row[s, i, c], al[s, a, 2], i, N)
            for i in range(0, Np + 1, max(1, Np // 7)) if Np else ():
                for k in range(2):
                    assert close(pair[s, i, c, k], al[s, a, k], i, Np)
