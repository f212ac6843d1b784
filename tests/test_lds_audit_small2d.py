"""The small 2D images' crossing layout (Turn, conv2d.hip): entry (s, r) at
s * SH + (r ^ flip(s)), SH = H + H/8.  Brute force for every shape: a bijection
into each column's own slots, and at most one lane per bank residue on the row
side and the column side of a crossing (quarter-wavefronts, 16 residues)."""
import pytest

from tests.test_lds_audit import ilog2, quarter

SHAPES = [(h, w) for h in (8, 16, 32, 64, 128, 256, 512) for w in (8, 16, 32, 64, 128, 256, 512) if h * w <= 8192]


def slot(h, w, s, r):
    lanes = min(ilog2(w // 8), 4)
    frm, bits = (4, max(lanes - 1, 0)) if h == 8 else (3, lanes)
    to = (3 if h == 8 else 4) - bits
    return s * (h + h // 8) + (r ^ (((s >> frm) & ((1 << bits) - 1)) << to))


@pytest.mark.parametrize("h,w", SHAPES)
def test_crossing_layout(h, w):
    sh, lanes = h + h // 8, h * w // 8
    per = w * sh                                       # slots of an image
    for s in range(w):
        assert sorted(slot(h, w, s, r) for r in range(h)) == list(range(s * sh, s * sh + h))
    tw, th = w // 8, h // 8
    for k in range(8):
        # two wavefronts' worth of consecutive lanes (several images where one is smaller)
        rows = [(i // lanes) * per + slot(h, w, (i % lanes) % tw * 8 + k, (i % lanes) // tw) for i in range(128)]
        cols = [(i // lanes) * per + slot(h, w, (i % lanes) // th, (i % lanes) % th + k * th) for i in range(128)]
        for a in (0, 64):
            assert quarter(rows[a: a + 64]) == 1 and quarter(cols[a: a + 64]) == 1, (k, a)
