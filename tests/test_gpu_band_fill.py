"""The band fill (rows of at most 128 band columns) against the general fill
(LCG_FIXED_COLS=0): D of every arc match, score, alignment and structures,
exact, at the edges of its row widths (31 / 33 columns: two groups or one per
wave, 63 / 65, 127 / 129: not taken), for the batch sizes that deal pairs to
several workgroups, and with the options that change D or sigma."""
import pytest

from locarna_amd import api, synth

pytestmark = pytest.mark.gpu


def _texts(lens, seed, span=100):
    out = []
    for k, n in enumerate(lens):
        s = synth.sequences(seed + k, 1, n, n, 0.5, 0.5)[0]
        out.append(synth.make_pp("s%d" % k, s, span))
    return out


def _results(texts, params, monkeypatch, fixed, shape=None, prepare=None):
    if fixed is None:
        monkeypatch.delenv("LCG_FIXED_COLS", raising=False)
    else:
        monkeypatch.setenv("LCG_FIXED_COLS", fixed)
    pairs = prepare() if prepare else [api.Pair(a, b, params) for a, b in texts]
    B = api.Batch(pairs, shape=shape)
    B.run(mode=0)
    r = [(B.score(k), B.alignment(k), B.D(k)) for k in range(len(pairs))]
    B.run(mode=2)
    assert [B.score(k) for k in range(len(pairs))] == [x[0] for x in r]
    B.destroy()
    return r


@pytest.mark.parametrize("max_diff", [2, 15, 16, 31, 32, 63, 64])
@pytest.mark.parametrize("local", [0, 1])
def test_row_widths(max_diff, local, monkeypatch):
    t = _texts([150, 150, 149, 141], 500 + max_diff)
    texts = [(t[0], t[1]), (t[2], t[3])]
    pa = api.locarna_params(max_diff=max_diff, min_trace_prob=0.0, sequ_local=local)
    ref = _results(texts, pa, monkeypatch, "0")
    assert _results(texts, pa, monkeypatch, None) == ref
    assert _results(texts, pa, monkeypatch, None, dict(waves=3, wg_per_pair=1)) == ref


@pytest.mark.parametrize("kw", [dict(), dict(indel_opening=0), dict(indel_opening=120), dict(tau=50),
                                dict(no_lonely_pairs=1), dict(stacking=1), dict(free_endgaps=15)],
                         ids=["default", "linear", "opening_bonus", "tau", "nolp", "stacking", "free"])
def test_options(kw, monkeypatch):
    t = _texts([97, 64, 33, 130, 76, 12], 700)
    texts = [(t[a], t[b]) for a in range(6) for b in range(a)]
    pa = api.locarna_params(**kw)
    ref = _results(texts, pa, monkeypatch, "0")
    assert _results(texts, pa, monkeypatch, None) == ref
    assert _results(texts, pa, monkeypatch, None, dict(waves=2, wg_per_pair=3)) == ref


def test_device_prepared_and_mixed(monkeypatch):
    """Device-compacted pairs; a batch of which one pair is too wide for the
    band fill and one has no arc match."""
    t = _texts([180, 175, 20, 90], 900)
    texts = [(t[0], t[1]), (t[2], t[3]), (t[3], t[0])]
    for kw in (dict(), dict(min_trace_prob=0.0), dict(sequ_local=1)):
        pa = api.locarna_params(**kw)

        def prep():
            return api.prepare_pairs(texts, pa, device_compaction=True, device_band=True)[0]
        ref = _results(texts, pa, monkeypatch, "0", prepare=prep)
        assert _results(texts, pa, monkeypatch, None, prepare=prep) == ref


def test_profiles(monkeypatch):
    """Sigma from the column-pair table: profiles of two rows."""
    t = _texts([70, 74, 66, 81], 950)
    pa = api.locarna_params()
    B = api.Batch([api.Pair(t[0], t[1], pa), api.Pair(t[2], t[3], pa)])
    B.run()
    prof = [B.consensus_pp(0), B.consensus_pp(1)]
    B.destroy()
    texts = [(prof[0], prof[1]), (prof[1], t[0])]
    ref = _results(texts, pa, monkeypatch, "0")
    assert _results(texts, pa, monkeypatch, None) == ref


def _shared(texts, params, mode=0, shape=None):
    """Whether several workgroups share a pair: a run whose waits all expire is
    invalid then."""
    B = api.Batch([api.Pair(a, b, params) for a, b in texts], shape=shape)
    B.set_spin_limit(-1)
    B.run(mode=mode, trace=False)
    try:
        B.score(0)
        return False
    except api.LcgError:
        return True
    finally:
        B.destroy()


def test_many_pairs_dealt(monkeypatch):
    """More pairs than CUs, one of them far larger: dealt to several
    workgroups, the others queued."""
    big = _texts([230, 240], 960, span=150)
    t = _texts([30 + k for k in range(24)], 970)
    texts = [(big[0], big[1])] + [(t[a], t[b]) for a in range(24) for b in range(a)]
    pa = api.locarna_params(max_bp_span=150)
    assert len(texts) > 256 and _shared(texts, pa)
    assert _results(texts, pa, monkeypatch, None) == _results(texts, pa, monkeypatch, "0")


@pytest.mark.parametrize("short", [2, 8, 24], ids=["3", "31", "279"])
def test_mixed_batches(short, monkeypatch):
    """Pairs for both fills, which run side by side (no trace band: 134 columns
    and more are too wide for the band fill), with fewer pairs than CUs, where
    several workgroups share a pair of either, and with more, where the wide ones
    come first in the work order: eagerly, as a graph replayed between other
    runs, one pair per launch and without allocations."""
    big = _texts([140, 133, 127, 125], 980, span=150)
    t = _texts([20 + k for k in range(short)], 990)
    texts = [(big[0], big[1]), (big[1], big[0])][:1 if short == 2 else 2] + [(big[2], big[3])]
    texts += [(t[a], t[b]) for a in range(short) for b in range(a)]
    pa = api.locarna_params(max_bp_span=150, min_trace_prob=0.0)
    assert _shared(texts, pa)
    ref = _results(texts, pa, monkeypatch, "0")
    monkeypatch.delenv("LCG_FIXED_COLS")
    B = api.Batch([api.Pair(a, b, pa) for a, b in texts])
    for mode in (0, 2, 2, 0, 2, 1):
        print("mode", mode, flush=True)
        B.run(mode=mode)
        assert [(B.score(k), B.alignment(k), B.D(k)) for k in range(len(texts))] == ref, mode
    B.run_noalloc()
    assert [(B.score(k), B.alignment(k), B.D(k)) for k in range(len(texts))] == ref
    B.run(mode=0, count=True)
    assert [B.score(k) for k in range(len(texts))] == [x[0] for x in ref]
    B.destroy()


def test_one_pair_per_launch():
    """Mode 1: with fewer pairs than CUs several workgroups share the launch's
    pair, with the wanted number where one is asked for."""
    t = _texts([150, 143, 60, 64], 940)
    texts = [(t[2], t[3]), (t[0], t[1]), (t[1], t[2])]
    pa = api.locarna_params()
    assert _shared(texts, pa, mode=1) and _shared(texts, pa, mode=1, shape=dict(wg_per_pair=3))
    assert not _shared(texts, pa, mode=1, shape=dict(wg_per_pair=1))
    B = api.Batch([api.Pair(a, b, pa) for a, b in texts])
    res = []
    for mode in (0, 1, 2, 1):
        B.run(mode=mode)
        res.append([(B.score(k), B.alignment(k), B.D(k)) for k in range(3)])
    B.destroy()
    assert res[1:] == [res[0]] * 3
