"""The FP64 Coulomb table (csrc/coulomb_table.hpp, the code the pair kernel
inlines) against erfc and its derivative in 40 digits, over the kappa and r_off
a caller may give.

Bars, with x = kappa r and eps = 2^-53: rounding r changes erfc and f by up to
2 x^2 of themselves per relative error of r; the table corrects r to the last
bit, so one eps of r^2 is left, which is x^2 eps.  The polynomials add a few eps:
(8 + 4 x^2) eps of the value.  Beyond x = 5, where f is below 1e-10, the fit's
own error may reach 2e-13 of it.  Systems beyond x = 12 have no table."""
import os
import shutil
import subprocess

import numpy as np
import pytest

mp = pytest.importorskip("mpmath")
HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
EPS = 2.0 ** -53


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("table") / "coulomb_table")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wno-unknown-pragmas", "-I",
                    os.path.join(HERE, "..", "apocharmm_amd", "csrc"),
                    os.path.join(HERE, "cpp", "coulomb_table.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("kappa,roff", [
    (k, r) for k in (1e-8, 1e-4, 0.1, 0.3, 0.34, 0.4, 0.5, 0.77, 1.0, 3.0)
    for r in (1.9, 9.0, 12.0, 14.0, 24.0, 35.0) if k * r <= 12.0])
def test_table_against_mpmath(program, kappa, roff):
    rng = np.random.default_rng(int(100 * kappa + roff))
    r = np.concatenate([roff * rng.random(150), 1e-3 * roff * rng.random(10),
                        min(roff, 5.0 / kappa) * rng.random(40), [roff, np.nextafter(roff, 0)]])
    r2 = r * r
    text = "".join("%s %s %s\n" % (float(kappa).hex(), float(roff).hex(), float(v).hex())
                   for v in r2)
    out = subprocess.run([program], input=text, capture_output=True, text=True, check=True).stdout
    rows = [line.split() for line in out.splitlines()]
    assert len(rows) == len(r2) and int(rows[0][3]) <= 384
    with mp.workdps(40):
        for v, (g, f, ge, _) in zip(r2, rows):
            x = mp.mpf(kappa) * mp.sqrt(mp.mpf(float(v)))
            G = mp.erfc(x)
            F = G + 2 * x / mp.sqrt(mp.pi) * mp.exp(-x * x)
            bar = (8 + 4 * float(x) ** 2) * EPS + (2e-13 if x > 5 else 0.0)
            for name, got, want in (("g", g, G), ("f", f, F), ("energy g", ge, G)):
                err = abs(mp.mpf(float.fromhex(got)) - want)
                assert err <= bar * want, (name, float(x), got)
