"""The LDS audit of the N = 16384 and 32768 conv's exchanges (wide.hip): whole
complex values, one half of the positions per round, a position of the upper
half in the slot of the one N / 2 below it.  Slots padded by one per 16 positions
for the exchange inside each wavefront, by 16 per 256 for the others."""
import pytest

from tests import lds_bank_model as M

V, MAIN = 32, 16
PLANS = {"16384": (16384, [4, 16, 16, 16]), "32768": (32768, [8, 16, 16, 16]), "32768 chain": (32768, [16, 8, 16, 16])}


def pad16(n, pos):
    i = pos % (n // 2)
    return i + (i >> 4)


def pad256(n, pos):
    i = pos % (n // 2)
    return i + (i >> 8 << 4)


def stride(n, radices, p):
    for r in radices[:p + 1]:
        n //= r
    return n


def taps(n, radices, p, lane, half):
    """positions of the half's groups of pass p, in the kernel's order per group"""
    r, m, t = radices[p], stride(n, radices, p), n // V
    groups = range(V // r) if p == 0 else range(half * V // r // 2, (half + 1) * V // r // 2)
    ks = range(half * r // 2, (half + 1) * r // 2) if p == 0 else range(r)
    return [[(g // m) * r * m + g % m + k * m for k in ks] for g in (lane + q * t for q in groups)]


def sides(n, radices):
    """(pass, slot layout) of both sides of every exchange"""
    for p in range(len(radices) - 1):
        private = stride(n, radices, p) <= 64 and radices[p] == radices[p + 1]
        yield from ((p, pad16 if private else pad256), (p + 1, pad16 if private else pad256))


@pytest.mark.parametrize("name", PLANS)
def test_halves(name):
    n, radices = PLANS[name]
    t, size = n // V, n // 2 + n // 32
    for p, slot in sides(n, radices):
        owner = {}
        for half in (0, 1):
            seen = set()
            for lane in range(t):
                pos = [x for g in taps(n, radices, p, lane, half) for x in g]
                seen.update(pos)
                for x in pos:
                    assert owner.setdefault(slot(n, x), lane) == lane     # both halves: the lane's own slots
            # a half is one half of the positions, each in a slot of its own
            assert seen == set(range(half * n // 2, (half + 1) * n // 2))
        assert len(owner) == n // 2 and max(owner) < size
        if stride(n, radices, p) <= 64:       # the passes that meet both layouts: the wavefront's own range
            assert all(s // 1088 == lane // 64 for s, lane in owner.items())


@pytest.mark.parametrize("name", PLANS)
def test_conflict_free_and_additive(name):
    n, radices = PLANS[name]
    for p, slot in sides(n, radices):
        m = stride(n, radices, p)
        for half in (0, 1):
            for w in (0, 3, n // V // 64 - 1):
                lanes = [taps(n, radices, p, lane, half) for lane in range(64 * w, 64 * w + 64)]
                for g in range(len(lanes[0])):
                    base = [slot(n, x[g][0]) for x in lanes]
                    for k in range(len(lanes[0][g])):
                        s = [slot(n, x[g][k]) for x in lanes]
                        assert s == [b + slot(n, k * m) for b in base]
                        assert M.conflict_cycles(s, "read_b64") == 0 and M.conflict_cycles(s, "write_b64") == 0


@pytest.mark.parametrize("name", PLANS)
def test_private_exchange_rule_matches_brute_force(name):
    """An exchange has wavefront fences in place of workgroup barriers where both
    passes run at M <= 64 with the same radix: exactly where every wavefront reads
    back, in each half, the positions that it wrote."""
    n, radices = PLANS[name]
    for p in range(len(radices) - 1):
        private = True
        for half in (0, 1):
            for w in range(n // V // 64):
                wrote, reads = ({x for lane in range(64 * w, 64 * w + 64) for g in taps(n, radices, q, lane, half)
                                 for x in g} for q in (p, p + 1))
                private &= wrote == reads
        assert private == (stride(n, radices, p) <= 64 and radices[p] == radices[p + 1]), p
