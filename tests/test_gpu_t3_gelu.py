"""The T3 MLP's gelu on the GPU (t3_gelu_f, chatterbox.cpp_amd/csrc/cbx_split.h)
against its value in 64 bits, g(x) = x / (1 + exp(-2 w)) with w = sqrt(2/pi) x
(1 + 0.044715 x^2): ordinary, small and large values, both ends of the range,
and no less precise than the tanh form in binary32.

Tolerance per value, with s = 1 / (1 + exp(2 |w|)): the result's own rounding,
2^-24 |g|, and |x| s times s's relative error, which is e = exp(-2 |w|)'s times
1 - s (exp2 to one ulp, 2^-23; the roundings of x^2, of its multiple and of the
constants shift the exponent 2 |w| by 4 parts in 2^24 at most) and that of the
quotient, 2^-23; e below the smallest normal number counts as 0.
"""
import numpy as np
import pytest

import debug_t3_lib as D

pytestmark = pytest.mark.gpu

F32 = np.float32
C = 0.7978845608028654


def gelu(x):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    d = torch.from_numpy(np.ascontiguousarray(x, F32)).cuda()
    out = torch.empty_like(d)
    D.gelu(d, out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def value(x):
    """g(x) and the tolerance, in 64 bits."""
    x = x.astype(np.float64)
    w2 = 2 * C * np.abs(x) * (1 + 0.044715 * x * x)
    e = np.exp(-w2)
    s = e / (1 + e)
    g = np.where(x > 0, x - np.abs(x) * s, x * s)
    tol = 2.0 ** -24 * np.abs(g) + np.abs(x) * s * ((1 - s) * (2.0 ** -23 + 2.0 ** -22 * w2) + 2.0 ** -23)
    return g, tol + np.abs(x) * 2.0 ** -125 + 2.0 ** -149


def tanh_form(x):
    """0.5 x (1 + tanh(w)), every operation rounded to binary32."""
    inner = (F32(C) * x) * (F32(1) + (F32(0.044715) * x) * x)
    return (F32(0.5) * x) * (F32(1) + np.tanh(inner.astype(np.float64)).astype(F32))


@pytest.mark.parametrize("sd", [0.02, 0.2, 0.5, 1.0, 1.5, 3.0, 6.0])
def test_ordinary_values(sd):
    rng = np.random.default_rng(int(sd * 100))
    x = (rng.standard_normal(1 << 20) * sd).astype(F32)
    print(f"[gpu-case] gelu N(0, {sd})", flush=True)
    got = gelu(x).astype(np.float64)
    g, tol = value(x)
    assert np.all(np.abs(got - g) <= tol), float((np.abs(got - g) / tol).max())
    rms = lambda y: float(np.sqrt(np.mean((y - g) ** 2)))
    assert rms(got) <= rms(tanh_form(x).astype(np.float64))


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_every_magnitude(sign):
    """Magnitudes from the smallest subnormals to the largest finite value."""
    rng = np.random.default_rng(5)
    x = np.concatenate([2.0 ** rng.uniform(-149, 128, 1 << 18), 2.0 ** rng.uniform(-3, 5, 1 << 18),
                        [9.9, 9.95, 15.99, 16.0, 16.01, 1e38, 3.4e38]])
    x = (sign * np.minimum(x, np.finfo(F32).max)).astype(F32)
    print(f"[gpu-case] gelu magnitudes, sign {sign}", flush=True)
    got = gelu(x).astype(np.float64)
    g, tol = value(x)
    # far out the value is x or 0, whatever the tolerance's |x| 2^-125
    far = np.abs(x) >= 16
    assert np.array_equal(got[far], np.where(x[far] > 0, x[far], 0.0).astype(np.float64))
    assert np.all(np.abs(got - g)[~far] <= tol[~far])


def test_ends_of_the_range():
    inf, nan = np.inf, np.nan
    print("[gpu-case] gelu inf, NaN, zeros", flush=True)
    got = gelu(np.array([inf, -inf, nan, 0.0, -0.0, 1e38, -1e38], F32))
    assert got[0] == inf and np.isnan(got[1]) and np.isnan(got[2])
    assert np.array_equal(got[3:], np.array([0.0, 0.0, 1e38, 0.0], F32))
    assert np.signbit(got[4]) and not np.signbit(got[3])
