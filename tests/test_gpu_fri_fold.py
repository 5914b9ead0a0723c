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


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("nbe,folding", [(13, 3), (17, 4), (18, 2)])
def test_layer_sources_in_spent_buffers(pc, oracle, nbe, folding, graph):
    """Short layers whose tree source lies in what the layer's fold reads and nobody needs
    afterwards: layer 1's in the polynomial, the next ones' in the work buffer's end."""
    import torch
    pc.set_hash_family(2)
    steps = pc.FRI.steps(nbe, folding=folding)
    n = len(steps)
    pol = datagen.uniform(3 << nbe, 60 + nbe)
    ch = datagen.challenges(n, 61 + nbe)

    def run(shared):
        d, work = pc.to_device(pol), pc.empty(3 << steps[1])
        trees = [pc.MerkleTreeGL(3, 0, True, 1 << steps[k + 1], 3 << (steps[k] - steps[k + 1])) for k in range(n - 1)]
        if shared:
            trees[1].source = d[17:17 + (3 << steps[1])]
            end = work.numel()
            for k in range(2, n - 1):
                end -= 3 << steps[k]
                if end < 3 << steps[k]:  # would lie in the folded layer itself
                    break
                trees[k].source = work[end:end + (3 << steps[k])]
        pc.FRI.layers(d, work, pc.to_device(np.asarray(ch).reshape(-1)), nbe, steps, trees, arity=3, graph=graph)
        torch.cuda.synchronize()
        return trees, pc.to_host(work)[:3 << steps[-1]]

    trees, final = run(True)
    cur = pol.copy()
    for k in range(n):
        if k:
            cur = np.asarray(oracle.fri_fold(cur, np.asarray(ch)[k], k, nbe, steps[k - 1], steps[k])).reshape(-1)
            cur = cur[:3 << steps[k]]
        if k + 1 < n:
            h, w = 1 << (steps[k] - steps[k + 1]), 1 << steps[k + 1]
            rows = np.ascontiguousarray(cur.reshape(h, w, 3).transpose(1, 0, 2)).reshape(w, 3 * h)
            assert (pc.to_host(trees[k].source)[:3 << steps[k]].reshape(w, 3 * h) == rows).all(), k
            assert (pc.to_host(trees[k].nodes) == oracle.merkletree(rows, 3)).all(), k
    assert (final == cur).all()
