"""Invariants of the paged step's work split (tq_attention.hip: Segments,
item_passes, the split kernel's unit walk and attn_paged_combine_kernel),
restated in integer Python.

Every kv head has the same work: unit u holds n passes of weight w from work
position start (a per-head prefix sum), after a lead of positions that no
pass occupies (a unit's setup cost, 8 in the kernel's plan; 0 for a unit
without passes).  Each head's work is split into Gh
segments; workgroup s of a head takes the work positions [bound(s),
bound(s + 1)) with bound(s) = floor(s * total / Gh), computed as q*s +
floor(r*s / Gh) with divisions by the high word of a product with the inverse of
Gh, and a pass belongs to the segment holding its first position.  A step with
no more passes than Gh has as many segments as passes instead (weight 1, no
lead), with the inverse of Gh all the same.  Each workgroup writes one partial per (unit, segment) piece of its
head at slot (unit + segment) * H + head; the combine finds a unit's
segments from its first and last pass.  On random plans (weights 1, 3, 4,
empty units, more segments than work, steps of a pass per segment and of no
work) this checks what the kernels rely on: the bound formula equals the exact
floor, the segment lookup inverts it,
every pass of every (unit, head) lands in exactly one piece, no two pieces
share a slot, slots stay below (units + Gh) * H, and the combine visits
exactly the pieces the split kernel wrote."""
from __future__ import annotations

import numpy as np


def _inverse(Gh):
    return 0xFFFFFFFF // Gh


def _div(n, G, inv):
    """n // G as the kernel has it: the high word of n * inv, one too few at most."""
    assert 0 <= n < 1 << 31
    d = (n * inv) >> 32
    return d + (1 if n - d * G >= G else 0)


def _bound(s, total, G, inv):
    q = 1 if total == G else _div(total, G, inv)
    r = total - q * G
    return q * s + (_div(r * s, G, inv) if r else 0)


def _segment_of(x, total, G, inv):
    if total == G:
        return x
    # the kernel's float estimate, then the +-1 correction
    g = int(np.float32(np.float32(x) + np.float32(1)) * np.float32(G) / np.float32(total)) - 1
    g = max(0, min(g, G - 1))
    while g + 1 < G and _bound(g + 1, total, G, inv) <= x:
        g += 1
    while g > 0 and _bound(g, total, G, inv) > x:
        g -= 1
    return g


def _passes(S, n, w, b0, b1):
    x0 = 0 if S >= b0 else (b0 - S + w - 1) // w
    x1 = 0 if S >= b1 else min(n, (b1 - S + w - 1) // w)
    return x0, x1


def test_division_through_the_inverse():
    """Exact for every segment count a launch can have (a multiple of 8) and
    every dividend below 2^31, at the multiples and their neighbours."""
    rng = np.random.default_rng(78)
    for G in range(8, 520, 8):
        inv = _inverse(G)
        top = ((1 << 31) - 1) // G
        ks = {0, 1, 2, G - 1, G, G + 1, top // 2, top - 1, top, *rng.integers(0, top, 200).tolist()}
        for k in ks:
            for n in (k * G - 1, k * G, k * G + 1, k * G + G // 2):
                if 0 <= n < 1 << 31:
                    assert _div(n, G, inv) == n // G, (n, G)


def _plan(units, Gh, lead):
    """plan_step's records: (start, n, w) of every unit, the total and the
    segments, from (passes, weight) pairs."""
    tn = sum(n for n, _ in units)
    single = tn <= Gh
    recs, x = [], 0
    for n, w in units:
        x += lead if not single and n > 0 else 0
        w = 1 if single else w
        recs.append((x, n, w))
        x += w * n
    return recs, x, (max(tn, 1) if single else Gh)


def test_paged_plan_pieces_partition_every_item():
    rng = np.random.default_rng(77)
    singles = 0
    for trial in range(400):
        U = int(rng.integers(1, 40))
        H = int(rng.choice([1, 2, 4]))
        Gh = int(rng.choice([8, 64, 256, 512]))
        lead = int(rng.choice([0, 1, 8, 40]))
        # every third plan short enough for a pass per segment, some without work
        most = 300 if trial % 3 else int(rng.choice([1, 3, 20]))
        shapes = [(int(rng.choice([0, 1, 2, 17, 128, int(rng.integers(0, 300))])) % most,
                   int(rng.choice([3, 4]))) for _u in range(U)]
        units, total, G = _plan(shapes, Gh, lead)
        inv = _inverse(Gh)
        if total == 0:  # no piece: every segment is empty, and the combine looks for none
            assert G == 1 and _bound(0, 1, G, inv) == 0 and _bound(1, 1, G, inv) == 1
            continue
        singles += total == G
        ends = [units[k + 1][0] if k + 1 < U else total for k in range(U)]
        for s in range(G + 1):
            assert _bound(s, total, G, inv) == (s * total) // G
        for x in range(0, total, max(1, total // 97)):
            g = _segment_of(x, total, G, inv)
            assert _bound(g, total, G, inv) <= x < _bound(g + 1, total, G, inv)
        written = {}
        for h in range(H):  # the split kernel's walk: workgroup (head h, segment seg)
            for seg in range(G):  # (the workgroups past G have none)
                b0, b1 = _bound(seg, total, G, inv), _bound(seg + 1, total, G, inv)
                if b0 >= b1:
                    continue
                # (before the first unit's first pass: unit 0)
                u = next(k for k in range(U) if (k == 0 or units[k][0] <= b0) and b0 < ends[k])
                while u < U:
                    S, n, w = units[u]
                    if S >= b1:
                        break
                    x0, x1 = _passes(S, n, w, b0, b1)
                    if x0 < x1:
                        slot = (u + seg) * H + h
                        assert slot not in written
                        written[slot] = (u, h, x0, x1)
                    u += 1
        assert max(written) < (U + Gh) * H
        seen = 0
        for u, (S, n, w) in enumerate(units):  # the combine's view
            for h in range(H):
                covered = []
                if n > 0:
                    lo = _segment_of(S, total, G, inv)
                    hi = _segment_of(S + w * (n - 1), total, G, inv)
                    for g in range(lo, hi + 1):
                        x0, x1 = _passes(S, n, w, _bound(g, total, G, inv),
                                         _bound(g + 1, total, G, inv))
                        if x0 < x1:
                            assert written[(u + g) * H + h] == (u, h, x0, x1)
                            covered += range(x0, x1)
                            seen += 1
                assert covered == list(range(n))
        assert seen == len(written)
        if total == G:  # a pass of its own in every segment
            assert len(written) == H * G
            assert all(x1 == x0 + 1 for _u, _h, x0, x1 in written.values())
    assert singles > 50
