"""The folding kernel at the edges of its batches and workgroups: lengths
up to 52 nt (matrices in LDS), around 64, 128 and 256 nt (1, 2, 4 chunks of
cells a batch) and above (several workgroups per sequence), spans below and above the interior-loop limit, alone
and together (with half as many sequences as CUs and more, the long ones too on
one workgroup each, with two chunks a batch where Z5 of the longest takes the
LDS), against the folding oracle (1e-10 absolute on probabilities, as sums of up
to 500 positive terms per cell in another order allow, 1e-12 relative on log Z;
above 1000 nt, where its unscaled partition function overflows, against the
sequence alone, which has several workgroups); and the probability texts against
printf's rounding."""
import numpy as np
import pytest

from locarna_amd import api, synth
from oracle import oracle

pytestmark = pytest.mark.gpu


def _seqs(lens, seed):
    return [synth.sequences(seed + k, 1, n, n, 0.5, 0.6)[0] for k, n in enumerate(lens)]


def _check(seqs, span, first=None):
    F = api.Fold(seqs, max_bp_span=span, min_prob=0.0005)
    for k, s in enumerate(seqs[:first]):
        P, P2 = F.probs(k)
        if len(s) <= 1000:
            Po, P2o, lz = oracle.fold(s, span)
        else:
            alone = api.Fold([s], max_bp_span=span, min_prob=0.0005)
            (Po, P2o), lz = alone.probs(0), alone.log_z(0)
            alone.destroy()
        assert np.abs(P - Po).max() <= 1e-10, (len(s), span)
        assert np.abs(P2 - P2o).max() <= 1e-10, (len(s), span)
        assert abs(F.log_z(k) - lz) <= 1e-12 * max(1.0, abs(lz)), (len(s), span)
    F.destroy()


@pytest.mark.parametrize("n", [5, 9, 10, 11, 30, 40, 52, 53, 63, 64, 65, 127, 128, 129, 192, 255, 256, 257, 321])
@pytest.mark.parametrize("span", [-1, 7, 36, 70])
def test_one_sequence(n, span):
    _check(_seqs([n], 40 + n), span)


@pytest.mark.parametrize("lens", [[1, 4, 64, 65, 128, 129, 250], [300, 12, 90, 64, 257], [52, 1, 4, 30, 17, 40]])
def test_together(lens):
    _check(_seqs(lens, 90), 100)


@pytest.mark.parametrize("lens,span", [([257, 300, 513, 1000], 70), ([130, 640, 1300, 3700], 40)])
def test_many_with_long(lens, span):
    short = [65 + k % 30 for k in range(140)]
    assert all(k == 1 for k, _, _ in api.fold_plan(lens + short)[0])
    seqs = _seqs(lens + short, 500)
    _check(seqs, span, len(lens) + 3)


def test_probability_digits():
    F = api.Fold(_seqs([150, 140], 7), max_bp_span=100, min_prob=1e-6)
    for k in range(2):
        P, _ = F.probs(k)
        for line in F.pp(k, "x").split("#BPCUT")[1].split("\n")[1:]:
            f = line.split()
            if len(f) != 3:
                continue
            p = P[int(f[0]), int(f[1])]
            want = "%.4g" % p
            if len(want) > 8:
                want = "%.3e" % p
            assert f[2] == want.replace("e-0", "e-"), (p, f[2])
    F.destroy()
