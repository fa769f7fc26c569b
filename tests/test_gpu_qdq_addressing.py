"""Where a scale is looked up and a code is formed, at the sizes where either can go wrong: row scales whose trips of 64
groups hold the ends of no, one or many rows and whose rows go through the scales more than once; column scales whose
blocks end inside a chunk of 8 rows or are one row; integer codes at ties, the ends of their range, beyond it
and at special values, with scales of either sign.  Bit-exact against the oracle."""
import numpy as np
import pytest

from helpers import rng
from test_gpu_qdq import _check_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xname,qname", [("f32", "i8"), ("bf16", "i4"), ("f16", "f8"), ("bf16", "i4p")])
@pytest.mark.parametrize("d0,d1,ns", [(7, 8, 7), (300, 8, 5), (65, 1016, 65), (33, 1024, 3), (40, 1032, 40), (9, 4096, 2), (1, 24, 1), (130, 504, 13)])
def test_row_scales(pkg, orc, xname, qname, d0, d1, ns):
    r = rng(d0 * 7 + d1)
    _check_all(pkg, orc, r.standard_normal((d0, d1), dtype=np.float32), xname, qname, pkg.SCALE_ROW, d0, d1, ns,
               r.uniform(0.01, 0.1, ns).astype(np.float32) * np.where(np.arange(ns) % 3 == 2, -1, 1).astype(np.float32))


@pytest.mark.parametrize("xname,qname", [("f32", "i8"), ("bf16", "i4"), ("f16", "f8"), ("f32", "i4p")])
@pytest.mark.parametrize("blocks,nb,d1", [(3, 1, 16), (2, 7, 520), (2, 8, 512), (1, 15, 1032), (2, 16, 504), (2, 17, 8), (1, 33, 2056), (3, 128, 64)])
def test_column_scales(pkg, orc, xname, qname, blocks, nb, d1):
    r = rng(nb * 5 + d1)
    s = r.uniform(0.01, 0.1, (blocks, d1)).astype(np.float32) * np.where(r.random((blocks, d1)) < 0.2, -1, 1).astype(np.float32)
    _check_all(pkg, orc, r.standard_normal((blocks * nb, d1), dtype=np.float32), xname, qname, pkg.SCALE_COL, blocks * nb, d1, nb, s)


@pytest.mark.parametrize("xname,qname", [("f32", "i8"), ("bf16", "i4"), ("f16", "f8"), ("f32", "i4p")])
@pytest.mark.parametrize("blocks,nb,strips,rows", [(2, 6136, 1, 4), (2, 6137, 1, 4), (2, 6145, 1, 8), (1541, 5, 1, 8), (1, 3079, 4, 8), (1539, 4, 1, 4), (1537, 3, 2, 4)])
def test_rows_of_a_wave_of_column_scales(pkg, orc, xname, qname, blocks, nb, strips, rows):
    """Four and eight rows to a wave, on both sides of the line between them on 256 compute units, ends inside a chunk, against the oracle."""
    d0, d1 = blocks * nb, 64 * strips * (4 if xname == "f32" else 8) - 8
    r = rng(nb + d0)
    k = _check_all(pkg, orc, r.standard_normal((d0, d1), dtype=np.float32), xname, qname, pkg.SCALE_COL, d0, d1, nb,
                   r.uniform(0.01, 0.1, (blocks, d1)).astype(np.float32))
    end = "r8" if rows == 8 else ""
    assert list(k) == ["mtrt_%s_col_%s_%s%s" % (mode, xname, qname, end) for mode in ("q", "dq", "qdq")]


@pytest.mark.parametrize("qname,top", [("i8", 127), ("i4", 7), ("i4p", 7)])
@pytest.mark.parametrize("kind", ["uniform", "row", "col"])
@pytest.mark.parametrize("scale", [0.37, -0.37, 1.0, 3e-18, 2.0 ** 60, 2.0 ** -60, 1e-30, 3e38, 1e-40])
def test_integer_codes_at_their_edges(pkg, orc, qname, top, kind, scale):
    s = np.float32(scale)
    q = np.arange(-top - 3, top + 3.5, 0.5, dtype=np.float32)
    with np.errstate(over="ignore", under="ignore"):
        x = np.concatenate([q * s, np.nextafter(q * s, np.float32(np.inf)), np.nextafter(q * s, np.float32(-np.inf)),
                            np.array([0.0, -0.0, np.inf, -np.inf, 3.4e38, -3.4e38, 1e-45, -1e-45, 1.2e-38], dtype=np.float32)]).astype(np.float32)
    d1 = (x.size + 7) // 8 * 8
    x = np.resize(x, (17, d1)).astype(np.float32)
    k, nb, n = {"uniform": (pkg.SCALE_UNIFORM, 1, 1), "row": (pkg.SCALE_ROW, 17, 17), "col": (pkg.SCALE_COL, 17, d1)}[kind]
    _check_all(pkg, orc, x, "f32", qname, k, 17, d1, nb, np.full(n, s, np.float32))
