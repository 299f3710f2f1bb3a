"""Type groups in forms of their own (DEuler::run_groups), side by side in 3D and
one after another in 2D, against the oracle: many substeps, every group in
another form, values that send one group alone to its exact kernels, and the
same march captured on one stream.
"""

import numpy as np
import pytest

import pair
from test_lane_gpu import _defn, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('name,form', [
    ('both-0', 'f1'), ('both-0', '3:f1s,4:s1/1'), ('mixed-7', 'f2st'),
    ('mixed-7', '5:s1s/1,6:f2st,7:f2t,8:f2'),
    ('mixed-8', '5:f2,6:s1/2,7:f1,8:f2st')])
def test_groups_side_by_side(orc, monkeypatch, name, form):
    print('case: groups side by side', name, form, flush=True)
    monkeypatch.setenv('SC_EULER_FORM', form)
    ge, oe = _pair(orc, _defn(name), 1e-3)
    for steps in (1, 30):
        ge.march(steps)
        oe.march(steps)
        pair.same_euler(ge, oe)
    assert ge.exact_passes == 0
    # One group's cell leaves the fast range; then another's too.
    types = ge.mesh.cltpn.ndarray[ge.ngstcell:]
    for t in np.unique(types)[:2]:
        c = ge.ngstcell + np.nonzero(types == t)[0][-1]
        ge.so0n.ndarray[c, 0] = oe.so0n[c, 0] = 1e15
        ge.so0n.ndarray[c, -1] = oe.so0n[c, -1] = 1e16
        before = ge.exact_passes
        ge.march(2)
        oe.march(2)
        assert ge.exact_passes > before
        for a in ('so0n', 'so1n', 'cflo', 'cflc', 'so0t'):
            assert np.array_equal(getattr(ge, a).ndarray, getattr(oe, a),
                                  equal_nan=True), (t, a)


def test_groups_captured(orc, monkeypatch):
    print('case: groups captured', flush=True)
    monkeypatch.setenv('SC_EULER_FORM', '5:s1s/1,6:f2st,7:f2t,8:f2')
    a, oe = _pair(orc, _defn('mixed-7'), 1e-3)
    b, _ = _pair(orc, _defn('mixed-7'), 1e-3)
    b.use_graph = True
    for steps in (3, 4, 1):
        a.march(steps)
        b.march(steps)
        oe.march(steps)
        pair.same_euler(a, oe)
        pair.same_euler(b, oe)
