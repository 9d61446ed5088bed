"""LocARNA-P's fixed-column kernels (four rows at a time, one to three chunks
of 64 columns) against the oracle at the edges of their ranges: sequences of
63 to 67 and 127 to 131 nt without a band limit (one and two chunks, two and
three at the top level), 192 and 193 nt (the top level's largest and the
general kernel), narrow bands whose rows leave a chunk, gap opening cost 0
(the factor 1 - o is 0), and with the groups of a row dealt to one wave or
several workgroups.  Tolerances as for the whole path."""
import pytest

from locarna_amd import api, synth
from oracle import oracle
from test_gpu_pf import _compare

pytestmark = pytest.mark.gpu


def _texts(lens, seed, span):
    out = []
    for k, n in enumerate(lens):
        s = synth.sequences(seed + k, 1, n, n, 0.5, 0.5)[0]
        out.append(synth.make_pp("s%d" % k, s, span))
    return out


@pytest.mark.parametrize("n,m,kw", [
    (9, 12, {}), (63, 67, {}), (66, 64, {}), (65, 66, dict(indel_opening=0)), (130, 66, {}), (127, 131, {}),
    (150, 150, dict(max_diff=5)), (131, 150, dict(max_diff=31)), (192, 192, dict(max_diff=20)),
    (193, 190, dict(max_diff=20)),
])
def test_edges(n, m, kw):
    t = _texts([n, m], 40 * n + m, 190)
    kw = dict(kw, max_bp_span=190, min_trace_prob=1e-4 if "max_diff" not in kw else 0.0)
    want = oracle.pf(t[0], t[1], oracle.locarna_p_params(**kw))
    B = api.Batch([api.Pair(t[0], t[1], api.locarna_p_params(**kw))])
    for shape in ({}, dict(pf_waves=1, pf_wg_per_pair=1), dict(pf_waves=3, pf_wg_per_pair=5)):
        B.reshape(**shape)
        print(n, m, kw, shape, flush=True)
        B.pf_run()
        _compare(B, 0, want, (n, m, kw, shape))
    B.destroy()
