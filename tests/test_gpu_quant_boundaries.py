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


@pytest.mark.parametrize("kind", ["row", "col"])
@pytest.mark.parametrize("qname,flag", [("i8", None), ("i4", None), ("i4p", None), ("f4p", None), ("f8", None), ("f8", "Q_ROUND_TO_INT"), ("f8", "F8_VIA_F16"), ("f8", "F8_REFHOST")])
def test_codes_beside_the_middles(pkg, orc, qname, flag, kind):
    import torch
    g = rng(41)
    code = {"i8": "I8", "f8": "F8E4M3FN", "i4": "I4", "i4p": "I4_PACKED", "f4p": "F4_PACKED"}[qname]
    p_q, o_q = getattr(pkg, code), getattr(orc, code)
    m = _middles(qname, flag == "Q_ROUND_TO_INT")
    if flag == "F8_VIA_F16":                                        # and where two f16 values meet beside them
        m = np.concatenate([m * (1 - 2.0 ** -12), m * (1 + 2.0 ** -11)])
    mids = np.concatenate([m, (m + np.nextafter(m.astype(np.float32), np.float32(0)).astype(np.float64)) / 2,
                           (m + np.nextafter(m.astype(np.float32), np.float32(np.inf)).astype(np.float64)) / 2])
    ns = 512
    s = ((1 + g.integers(0, 1 << 23, ns) * 2.0 ** -23) * 2.0 ** g.integers(-20, 20, ns) * g.choice([-1.0, 1.0], ns)).astype(np.float32)
    x1 = (s.astype(np.float64)[:, None] * mids[None, :]).astype(np.float32)
    x = np.concatenate([np.nextafter(x1, np.float32(0)), x1, np.nextafter(x1, np.float32(np.inf)), -x1], 1)
    x = np.ascontiguousarray(x[:, : x.shape[1] // 8 * 8])
    if kind == "col":
        x = np.ascontiguousarray(x.T)
    d0, d1 = x.shape
    flags = getattr(pkg, flag) if flag else 0
    oflags = {"Q_ROUND_TO_INT": orc.Q_ROUND_TO_INT, "F8_VIA_F16": orc.F8_VIA_F16}.get(flag, 0)
    mode = orc.REFHOST if flag == "F8_REFHOST" else orc.IEEE
    kinds = (pkg.SCALE_ROW, orc.SCALE_ROW, ns) if kind == "row" else (pkg.SCALE_COL, orc.SCALE_COL, d0)
    xd, sd = torch.from_numpy(x).cuda(), torch.from_numpy(s).cuda()
    got = pkg.quantize(xd, sd, p_q, kinds[0], d0, d1, kinds[2], flags).cpu().numpy().view(np.uint8).ravel()
    ref = orc.quantize(x.ravel(), orc.F32, o_q, s, kinds[1], d0, d1, kinds[2], oflags, mode).view(np.uint8)
    bad = np.flatnonzero(got[: ref.size] != ref)
    assert bad.size == 0, (bad.size, bad[:5])
