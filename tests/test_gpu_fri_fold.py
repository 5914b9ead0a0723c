"""GPU tests of the FRI fold's two forms (several lanes a group, one lane a group) at the
sizes where the launch changes between them, in and out of place, against the oracle."""
import numpy as np
import pytest

import datagen

pytestmark = pytest.mark.gpu
P = 0xFFFFFFFF00000001


@pytest.fixture(scope="module")
def pc():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a HIP device")
    import pil2_commit
    return pil2_commit


@pytest.mark.parametrize("logx", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("place", ["one", "few", "last_lanes", "first_single"])
def test_fold_forms_match_oracle(pc, oracle, logx, place):
    """2^cur groups of 2^logx values: one group, fewer than a wave's, the longest layer with
    several lanes a group and the shortest with one; words of the layer at and past p."""
    import torch
    cur = {"one": 0, "few": 2, "last_lanes": 18 - logx, "first_single": 19 - logx}[place]
    prev, nbe = cur + logx, cur + logx + 1
    pol = datagen.uniform(3 << prev, 100 * logx + cur)
    raw = pol.copy()
    raw[::7] = np.array([0, 1, P - 1, P, P + 5, 2**64 - 1], dtype=np.uint64)[np.arange(raw[::7].size) % 6]
    ch = datagen.challenges(1, 40 + logx)[0]
    want = oracle.fri_fold(np.where(raw >= np.uint64(P), raw - np.uint64(P), raw), ch, 1, nbe, prev, cur)
    d = pc.to_device(raw)
    out = pc.FRI.fold(1, d, ch, nbe, prev, cur, out=pc.empty(3 << cur))
    pc.FRI.fold(1, d, ch, nbe, prev, cur)
    torch.cuda.synchronize()
    assert (pc.to_host(out).reshape(-1) == np.asarray(want).reshape(-1)[:3 << cur]).all()
    assert (pc.to_host(d)[:3 << cur] == np.asarray(want).reshape(-1)[:3 << cur]).all()
