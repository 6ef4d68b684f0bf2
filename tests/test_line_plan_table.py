"""The table of line plans (PFH_FAST_ROUTE_PLANS in csrc/pfh_stage.hpp) derived
again from the rule that its comment states."""
import itertools
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# lane instructions of a butterfly; composite radices from their coprime factors
BUTTERFLY = {2: 4, 3: 16, 4: 16, 5: 36, 7: 66, 8: 56, 9: 136, 11: 150, 16: 170}
for a, b in ((2, 3), (2, 5), (4, 3), (2, 7), (3, 5)):
    BUTTERFLY[a * b] = b * BUTTERFLY[a] + a * BUTTERFLY[b]
EXCHANGE = 14  # per value and pass


def _threads(radices, em):
    m = 1
    for r in radices:
        m *= r
    return max(-(-(m // r) // max(1, em // r)) for r in radices)


def _cost(radices, em):
    m = 1
    for r in radices:
        m *= r
    threads = _threads(radices, em)
    lanes = sum(-(-(m // r) // threads) * threads * (BUTTERFLY[r] + r * EXCHANGE) for r in radices)
    return lanes * (1 + 0.002 * em) * (1.2 if threads > 64 else 1) * (1.03 if threads > 32 else 1)


def _best(m):
    plans = []
    for k in (2, 3):
        for radices in itertools.product(sorted(BUTTERFLY), repeat=k):
            p = 1
            for r in radices:
                p *= r
            if p == m:
                plans += [(_cost(radices, em), em, _threads(radices, em), radices)
                          for em in range(max(radices), (8 if m < 64 else 16) + 1)]
    return min(plans) if plans else None


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def test_table_follows_its_rule():
    text = open(os.path.join(ROOT, "pencil-rs_amd", "csrc", "pfh_stage.hpp")).read()
    start = text.index("#define PFH_FAST_ROUTE_PLANS")
    entries = re.findall(r"X\((\w+), (\d+), (\d+), (\d+), (\d+)\)", text[start:text.index("#define PFH_FAST_PLANS")])
    table = {}
    for precision, *plan in entries:
        r0, r1, r2, em = map(int, plan)
        table.setdefault(precision, set()).add(((r0, r1, r2) if r2 else (r0, r1), em))
    want = set()
    for m in [n for n in range(8, 1025) if _smooth(n)] + [385]:
        best = _best(m)
        if best is None:
            continue
        _, em, threads, radices = best
        want.add((radices, em))
        if 64 < m <= 128 and threads <= 8:  # the variant with about twice the threads
            want.add((radices, radices[0]))
    assert table["float"] == want
    assert table["double"] == want
