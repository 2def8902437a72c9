"""The form of GELU in the GeGLU epilogues (gelu_sigmoid, csrc/device_math.h)
in float32 as the device evaluates it, its two hardware functions off by up to
one unit in the last place either way, against float64 and beside the rational
tanh that the other products use (gelu_tanh_ref)."""
import numpy as np
import pytest

f = np.float32


def fma(a, b, c):
    return (a.astype(np.float64) * b.astype(np.float64) + np.asarray(c, np.float64)).astype(f)


def hardware(v, r):
    v = v.astype(f)
    u = r.integers(-1, 2, v.shape)
    return np.where(u == 0, v, np.nextafter(v, np.where(u > 0, f(np.inf), f(-np.inf)))).astype(f)


def gelu_sigmoid(x, r):
    t = x * fma(x * x, f(-0.10294324), f(-2.3022082))
    s = hardware(np.exp2(np.minimum(t, f(125)).astype(np.float64)), r)
    d = f(1) + s
    dl = s - (d - f(1))
    q = hardware(1 / d.astype(np.float64), r)
    e = fma(-dl, q, fma(-d, q, f(1)))
    y = x * q
    return y + fma(y, e, fma(x, q, -y))


def gelu_tanh_ref(x):
    v = fma(x * x * x, f(0.044715), x) * f(0.7978845608028654)
    c = np.clip(v, f(-7.99881172180175781), f(7.99881172180175781))
    c2 = c * c
    p = np.full_like(x, -2.76076847742355e-16)
    for k in (2.00018790482477e-13, -8.60467152213735e-11, 5.12229709037114e-08, 1.48572235717979e-05,
              6.37261928875436e-04, 4.89352455891786e-03):
        p = fma(p, c2, f(k))
    q = np.full_like(x, 1.19825839466702e-06)
    for k in (1.18534705686654e-04, 2.26843463243900e-03, 4.89352518554385e-03):
        q = fma(q, c2, f(k))
    t = ((p * c).astype(np.float64) / q).astype(f)
    t = np.where(v >= 9, f(1), np.where(v <= -9, f(-1), np.where(np.abs(v) < f(0.0004), v, t)))
    return (t + f(1)) * x * f(0.5)


@pytest.mark.parametrize("size", [1e-3, 0.05, 0.3, 1.0, 3.0, 20.0])
def test_gelu_of_the_geglu_products(size):
    r = np.random.default_rng(3)
    x = (size * r.standard_normal(200_000)).astype(f)
    X = x.astype(np.float64)
    want = 0.5 * X * (1 + np.tanh(0.7978845608028654 * (X + 0.044715 * X ** 3)))
    got, ref = gelu_sigmoid(x, r) - want, gelu_tanh_ref(x) - want
    assert (np.abs(got) <= 1e-7 * np.abs(X)).all(), np.abs(got / X).max()
    # and in the mean no further off than the rational form, or than the
    # rounding of 1 + tanh that it is spared near 0 accounts for
    assert np.linalg.norm(got) <= 1.3 * np.linalg.norm(ref)


def test_gelu_at_the_ends():
    r = np.random.default_rng(4)
    x = np.array([0.0, -0.0, 1e30, -1e30, np.nan, -20.0, 40.0], f)
    with np.errstate(all="ignore"):
        got = gelu_sigmoid(x, r)
    assert got[0] == 0 and got[1] == 0 and got[2] == f(1e30) and abs(got[3]) < 1e-6 and np.isnan(got[4])
    assert abs(got[5]) < 1e-30 and got[6] == f(40)
