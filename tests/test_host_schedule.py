"""Host logic of the fill's LDS schedule (lcg_pair_schedule, the function
lcg_batch_create uses): every group of a row is placed once, a round of a
workgroup member holds at most `waves` groups on distinct waves, their LDS
regions are disjoint and inside the pool, and the row's round count covers
them.  And the dealing of pairs to workgroups (lcg_deal_workgroups, the function
of the band fill and of LocARNA-P): the workgroups that wait for each other are
resident together, and queued pairs have some left.  And the LDS of LocARNA-P's
regions.  Runs on the CPU."""
import collections
import random

import pytest

from locarna_amd import api, synth


def _pairs():
    pps, pairs, span = synth.workload("allpairs64", limit_pairs=6)
    out = [api.Pair(pps[a], pps[b], api.locarna_params(max_bp_span=span)) for a, b in pairs]
    pps, pairs, span = synth.workload("long500", limit_pairs=1)
    out += [api.Pair(pps[a], pps[b], api.locarna_params(max_bp_span=span, sequ_local=1)) for a, b in pairs]
    return out


@pytest.mark.parametrize("waves,pool,members", [(16, 40000, 1), (8, 20000, 1), (16, 40000, 4), (16, 40000, 64)])
def test_schedule_invariants(waves, pool, members):
    for P in _pairs():
        sched, rounds = P.schedule(waves, pool, members)
        assert len(sched) == P.num_groups
        by_slot = collections.defaultdict(list)
        for (rnd, wave, member, off, size, al, bl) in sched:
            assert 0 <= wave < waves and 0 <= member < members
            assert rnd < rounds[al]
            assert 0 <= off and off + size <= pool
            by_slot[(al, member, rnd)].append((wave, off, size))
        for key, items in by_slot.items():
            assert len(items) <= waves
            assert len({w for w, _, _ in items}) == len(items), key
            spans = sorted((o, o + s) for _, o, s in items)
            for (a0, a1), (b0, b1) in zip(spans, spans[1:]):
                assert a1 <= b0, (key, spans)
        rows = {al for (_, _, _, _, _, al, _) in sched}
        for al in range(1, P.lenA + 1):
            if al not in rows:
                assert rounds[al] == 0


def test_schedule_rejects_small_pool():
    P = _pairs()[0]
    with pytest.raises(api.LcgError):
        P.schedule(16, 64, 1)


def _works(rng, n, kind):
    if kind == "equal":
        return [1e6] * n
    if kind == "one":
        return sorted([1e3 * rng.uniform(1, 2) for _ in range(n - 1)] + [1e7], reverse=True)
    return sorted((rng.lognormvariate(10, 1.5) for _ in range(n)), reverse=True)


@pytest.mark.parametrize("kind", ["ragged", "equal", "one"])
@pytest.mark.parametrize("npairs", [1, 2, 30, 255, 256, 257, 300, 2016])
@pytest.mark.parametrize("first", [0, 1, 40, 400])
def test_dealt_workgroups_are_resident(kind, npairs, first):
    """`first` pairs of the other fill (too wide for the band fill) and as many
    that cannot be split come before those that can."""
    rng = random.Random(7 * npairs + first)
    for slots in (256, 64):
        for meet in (0.14, 0.08):
            work = _works(rng, npairs, kind)
            most = [q // first if q < 2 * first else rng.randint(2, 16) for q in range(npairs)]
            K, dealt = api.deal_workgroups(work, most, slots, meet)
            assert all(min(1, m) <= k <= m for k, m in zip(K, most))
            assert all(k <= 1 for k in K[dealt:])
            used = sum(K[:dealt])
            assert used <= slots and (sum(K[dealt:]) == 0 or used < slots)
            if sum(m > 0 for m in most) < slots:
                assert dealt == npairs
            own = [q for q in range(npairs) if most[q]]
            if not own:
                continue
            work, K, dealt = [work[q] for q in own], [K[q] for q in own], sum(q < dealt for q in own)

            def span(K, dealt):  # the dealt pairs' slowest, the others spread over the rest
                t = [w * (1 + meet * (k - 1)) / k for w, k in zip(work, K)]
                load = [0.0] * max(1, slots - sum(K[:dealt]))
                for x in t[dealt:]:
                    load[load.index(min(load))] += x
                return max(t[:dealt] + load)
            assert span(K, dealt) <= 1.2 * span([1] * len(own), 0)


def test_pf_regions_at_the_edge_of_the_pool():
    """In the outside pass and at the top level a region of the sizes that an LDS
    pool ends at (6,000 doubles for the longest pairs, up to 20,000) takes no
    more than its two matrices and one row."""
    size = api.lib().lcg_pf_region_doubles
    for rows in (20, 60, 129, 193):
        for width in (20, 64, 129, 193):
            for cols in (width, 2 * width):
                cells = rows * width
                assert size(rows, width, cols, 0) == cells + 4 * cols
                assert size(rows, width, cols, 1) >= cells + 4 * cols  # a forward fill fits too
                if 2 * cells + cols > 6000:
                    assert size(rows, width, cols, 1) <= 2 * cells + cols
