"""Which kernel form a launch of fingerprints takes (csrc/staf_step.hpp): the rule is host code and is compiled for the host alone."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "%s/alphanesgpu_amd/csrc/staf_step.hpp"
#include <stdio.h>
using namespace staf;
template <typename real>
static void line(int nr, int nt, int Ar, int Aa, int centres) {
  RowsLaunch<real> L;
  for (int k = 0; k < nt; k++) L.add(nr, nr * (nr - 1) / 2, nt, Ar, Aa, (centres + k) / nt);
  printf("%%d %%zu %%zu\n", L.waves(), rows_lds<real, 4>(nr, nt, Ar, Aa), rows_lds<real, 8>(nr, nt, Ar, Aa));
}
int main() {
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

    def ask(*case):
        r = subprocess.run([exe], input=" ".join(map(str, case)), stdout=subprocess.PIPE, text=True, check=True)
        return tuple(map(int, r.stdout.split()))
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
