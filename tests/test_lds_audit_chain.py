"""The LDS audit (test_lds_audit.py) for the plans of the four-step chain in one
workgroup: a radix-16 outer level first, then the radix-16 plan of n / 16
points, so the lead pass (radix 2, 4 or 8) is the second one.  The exchanges of N =
8192 and 16384 at 16 values per lane, with the per-exchange layouts; those of
N = 32768 at 32 values per lane are in test_lds_audit_halves.py."""
import pytest

from tests import test_lds_audit as A


def chain_radices(n):
    bits = A.ilog2(n) - 4
    return [16] + ([1 << (bits % 4)] if bits % 4 else []) + [16] * (bits // 4)


def chain_plan(n, v):
    out, m = [], n
    for r in chain_radices(n):
        m //= r
        out.append((r, m))
    return out


@pytest.mark.parametrize("n", [8192, 16384])
def test_exchange_layouts(n, monkeypatch):
    monkeypatch.setattr(A, "plan", chain_plan)
    assert A.xchg_problems(n, 16, A.xchg_params) == []


@pytest.mark.parametrize("n,v,stride_lanes", [(8192, 16, 512), (16384, 16, 1024), (32768, 32, 1024)])
def test_one_base_twiddle_for_the_groups_of_the_later_passes(n, v, stride_lanes):
    """W^j of a lane's groups: j = (L + g T) mod M is the same for every group where
    M <= T, which is every pass but the first, so those passes run one chain."""
    assert n // v == stride_lanes
    for p, (r, m) in enumerate(chain_plan(n, v)):
        js = {(lane, (lane + g * stride_lanes) % m) for lane in (0, 1, 77, stride_lanes - 1) for g in range(v // r)}
        assert (len(js) == 4) == (p > 0 or v // r == 1)
