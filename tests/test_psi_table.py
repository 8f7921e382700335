"""The piecewise polynomials of the stability functions (ne_psi_table.h, written by gen_psi_table.py):
the header is the generator's output, and its coefficients, evaluated as the kernel evaluates them
(interval from the bits of the shifted argument, fused Horner steps), hold ψ_m and ψ_s against the
closed forms at 40 digits. The fit is within 2⁻⁵⁴ (FP32 2⁻²⁵) of max(1, |ψ|); the argument's shift, the
leading coefficient and the last Horner step round, each by half an ulp of a value below
max(1, |ψ|) (the shift's rounding scaled by |t ψ'| ≤ 4·max(1, |ψ|) on the table), so the bound is 4 ulp.
The logarithm's table likewise: an absolute error below an ulp of max(1, |log x|)."""
import pathlib
import re
import subprocess
import sys

import mpmath as mp
import numpy as np
import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "numericalearth.jl_amd" / "csrc"
TEXT = (CSRC / "ne_psi_table.h").read_text()
sys.path.insert(0, str(CSRC))
import gen_psi_table as gen  # noqa: E402


def _array(name):
    body = re.search(name + r"\[[^\]]*\] = \{(.*?)\};", TEXT, re.S).group(1)
    return [float(x.rstrip("f")) for x in re.findall(r"[-+0-9.]+e[-+0-9]+f?", body)]


def test_header_is_the_generator_output():
    out = subprocess.run([sys.executable, str(CSRC / "gen_psi_table.py")], capture_output=True, text=True,
                         check=True).stdout
    assert out == TEXT


def _closed(z):
    t = gen.A - z if z < 0 else z + gen.B
    return (gen.momentum_unstable(t), gen.scalar_unstable(t)) if z < 0 else (gen.momentum_stable(t), gen.scalar_stable(t))


def _arguments():
    rng = np.random.default_rng(3)
    edges = [-float(c + s * r - gen.A) for c, r in gen.intervals(gen.A, mp.mpf(128)) for s in (-0.999, 0.999)]
    edges += [float(c + s * r - gen.B) for c, r in gen.intervals(gen.B, mp.mpf(16)) for s in (-0.999, 0.999)]
    z = [x for x in edges if -127.9 < x < 14.49]
    z += list(-np.exp(rng.uniform(np.log(1e-9), np.log(127.0), 600))) + list(np.exp(rng.uniform(np.log(1e-9), np.log(14.4), 300)))
    return z + [0.0, -5e-324, 5e-4, -5e-4]


@pytest.mark.parametrize("kind,bits,shift,ulp", [("f64", 64, 49, 2.0 ** -53), ("f32", 32, 20, 2.0 ** -24)])
def test_table_holds_the_closed_forms(kind, bits, shift, ulp):
    mp.mp.dps = 40
    real, word = (np.float64, np.uint64) if bits == 64 else (np.float32, np.uint32)
    stride, bias = (20, 1023) if bits == 64 else (12, 127)
    coefficients = _array(f"psi_table_{kind}")
    unstable = int(re.search(r"NE_PSI_UNSTABLE_BINS (\d+)", TEXT).group(1))
    bins = int(re.search(r"NE_PSI_BINS (\d+)", TEXT).group(1))
    assert len(coefficients) == bins * stride
    worst = 0.0
    for z in _arguments():
        z = real(z)
        t = real(abs(z) + real(float(gen.A) if z < 0 else 1.5))
        b = int(t.view(word))
        first = ((bias - 6) * 8 + 6) if z < 0 else (bias * 8 + 4 - unstable)
        k = (b >> shift) - first
        assert 0 <= k < bins and (k < unstable) == bool(z < 0), (z, k)
        centre = word((b >> shift << shift) | (1 << (shift - 1))).view(real)
        x = mp.mpf(float(t)) - mp.mpf(float(centre))
        row = coefficients[k * stride:(k + 1) * stride]
        for n, want in enumerate(_closed(mp.mpf(float(z)))):
            got = mp.mpf(0)
            for c in reversed(row[n::2]):
                got = mp.mpf(float(real(float(got * x + mp.mpf(c)))))
            worst = max(worst, float(abs(got - want) / max(1, abs(want))) / ulp)
    assert worst <= 8.0, worst   # 4 ulp, an ulp of [1, 2) being 2·2⁻⁵³ (2·2⁻²⁴)


def test_log_table():
    mp.mp.dps = 40
    table = _array("log_table_f64")
    worst = 0.0
    rng = np.random.default_rng(4)
    for x in list(np.exp(rng.uniform(-30, 5, 2000))) + [0.5, 1.0, 2.0, 1.0 - 2.0 ** -53, 1.0 + 2.0 ** -52]:
        m, e = np.frexp(x)
        inv, lc = table[2 * (int((m - 0.5) * 128)):][:2]
        r = float(mp.mpf(float(m)) * mp.mpf(inv) - 1)
        assert abs(r) < 0.01
        q = 1.0 / 7.0
        for c in (-1.0 / 6.0, 1.0 / 5.0, -1.0 / 4.0, 1.0 / 3.0, -0.5):
            q = float(mp.mpf(q) * r + mp.mpf(c))
        p = float(mp.mpf(r * r) * q + r)
        hi = float(mp.mpf(int(e)) * mp.mpf(0.6931471805599453) + mp.mpf(lc))
        lo = float(mp.mpf(int(e)) * mp.mpf(2.3190468138462996e-17) + mp.mpf(p))
        want = mp.log(mp.mpf(float(x)))
        worst = max(worst, float(abs(mp.mpf(hi + lo) - want) / max(1, abs(want))))
    assert worst <= 2.0 ** -52
