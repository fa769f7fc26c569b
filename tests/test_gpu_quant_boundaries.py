"""Codes of values within an ulp of where two codes meet, for scales of any mantissa, sign and a range of exponents: there the
quotient that the kernels form has to fall to the same side as the correctly rounded one."""
import numpy as np
import pytest

from helpers import rng

pytestmark = pytest.mark.gpu


def _middles(name, round_to_int):
    """Where two codes meet (magnitudes), and past the largest."""
    if name in ("i8", "i4", "i4p") or round_to_int:
        top = {"i8": 128, "i4": 8, "i4p": 8, "f8": 448}[name]
        return np.arange(top + 2) + 0.5
    if name == "f4p":
        codes = np.array([0, 0.5, 1, 1.5, 2, 3, 4, 6, 8])
    else:
        codes = np.unique(np.concatenate([np.arange(8) * 2.0 ** -9] + [(8 + np.arange(8)) * 2.0 ** (e - 3) for e in range(-6, 10)]))
    return (codes[1:] + codes[:-1]) / 2


CODES = [("i8", None), ("i4", None), ("i4p", None), ("f4p", None), ("f8", None), ("f8", "Q_ROUND_TO_INT"), ("f8", "F8_VIA_F16"), ("f8", "F8_REFHOST")]


def _scales(g, n, exponents=None):
    mantissas = 1 + g.integers(0, 1 << 23, n) * 2.0 ** -23
    e = g.integers(-20, 20, n) if exponents is None else np.resize(exponents, n)
    return (mantissas * 2.0 ** e * g.choice([-1.0, 1.0], n)).astype(np.float32)


def _beside(s, qname, flag):
    """[scales, values]: what lies beside the places where two codes of each scale meet."""
    m = _middles(qname, flag == "Q_ROUND_TO_INT")
    if flag == "F8_VIA_F16":                                        # and where two f16 values meet beside them
        m = np.concatenate([m * (1 - 2.0 ** -12), m * (1 + 2.0 ** -11)])
    mids = np.concatenate([m, (m + np.nextafter(m.astype(np.float32), np.float32(0)).astype(np.float64)) / 2,
                           (m + np.nextafter(m.astype(np.float32), np.float32(np.inf)).astype(np.float64)) / 2])
    x1 = (s.astype(np.float64)[:, None] * mids[None, :]).astype(np.float32)
    x = np.concatenate([np.nextafter(x1, np.float32(0)), x1, np.nextafter(x1, np.float32(np.inf)), -x1], 1)
    return np.ascontiguousarray(x[:, : x.shape[1] // 8 * 8])


def _check(pkg, orc, qname, flag, kind, x, s):
    import torch
    code = {"i8": "I8", "f8": "F8E4M3FN", "i4": "I4", "i4p": "I4_PACKED", "f4p": "F4_PACKED"}[qname]
    d0, d1 = x.shape
    nb = {"ROW": s.size, "COL": d0, "UNIFORM": 1}[kind]
    flags = getattr(pkg, flag) if flag else 0
    oflags = {"Q_ROUND_TO_INT": orc.Q_ROUND_TO_INT, "F8_VIA_F16": orc.F8_VIA_F16}.get(flag, 0)
    mode = orc.REFHOST if flag == "F8_REFHOST" else orc.IEEE
    xd, sd = torch.from_numpy(x).cuda(), torch.from_numpy(s).cuda()
    got = pkg.quantize(xd, sd, getattr(pkg, code), getattr(pkg, "SCALE_" + kind), d0, d1, nb, flags).cpu().numpy().view(np.uint8).ravel()
    ref = orc.quantize(x.ravel(), orc.F32, getattr(orc, code), s, getattr(orc, "SCALE_" + kind), d0, d1, nb, oflags, mode).view(np.uint8)
    bad = np.flatnonzero(got[: ref.size] != ref)
    assert bad.size == 0, (bad.size, bad[:5], s[:1])


@pytest.mark.parametrize("kind", ["row", "col"])
@pytest.mark.parametrize("qname,flag", CODES)
def test_codes_beside_the_middles(pkg, orc, qname, flag, kind):
    g = rng(41)
    s = _scales(g, 512)
    x = _beside(s, qname, flag)
    _check(pkg, orc, qname, flag, kind.upper(), x if kind == "row" else np.ascontiguousarray(x.T), s)


@pytest.mark.parametrize("kind", ["row", "col", "uniform"])
@pytest.mark.parametrize("qname,flag", CODES)
def test_scales_on_both_sides_of_the_divide(pkg, orc, qname, flag, kind):
    """Scales of less than 2^-60 and from 2^61 up are divided by: rows, columns and tensors on one side each, and (columns) waves with both."""
    g = rng(42)
    for exponents in ([-62.0, -61.0], [-60.0, -59.0], [59.0, 60.0], [61.0, 62.0], [-61.0, -60.0, 60.0, 61.0]):
        s = _scales(g, 64, exponents)
        x = _beside(s, qname, flag)
        if kind == "uniform":
            for i in range(0, s.size, 9):
                _check(pkg, orc, qname, flag, "UNIFORM", x[i:i + 1], s[i:i + 1])
        else:
            _check(pkg, orc, qname, flag, kind.upper(), x if kind == "row" else np.ascontiguousarray(x.T), s)
