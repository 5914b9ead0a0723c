"""GPU tests of the transforms' rounds on the matrix cores: every number of strided bits and
short-round bits, every blowup, odd column counts, words at and past p, and the shapes next
to those that keep the rounds on the VALU, against the oracle."""
import numpy as np
import pytest

from golden_helpers import colmajor_to_rowmajor
import datagen

pytestmark = pytest.mark.gpu
P = 0xFFFFFFFF00000001


@pytest.fixture(scope="module")
def pc():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a HIP device")
    import pil2_commit
    pil2_commit.set_hash_family(2)
    return pil2_commit


def _words(n, seed):
    """n words, some of them at and past p, and the same residues below p."""
    raw = datagen.uniform(n, seed)
    raw[::5] = np.array([0, 1, P - 1, P, P + 1, 2**64 - 1, 2**32 - 1], dtype=np.uint64)[np.arange(raw[::5].size) % 7]
    return raw, np.where(raw >= np.uint64(P), raw - np.uint64(P), raw)


LDE = [(10, 0, 2), (11, 0, 3), (12, 0, 1), (14, 0, 2), (15, 0, 1), (17, 0, 2), (18, 0, 3), (19, 0, 1),
       (9, 1, 3), (10, 1, 2), (13, 1, 1), (14, 1, 3), (15, 1, 2), (16, 1, 5), (17, 1, 1), (18, 1, 2), (21, 1, 1),
       (22, 1, 1), (8, 2, 2), (9, 2, 3), (12, 2, 2), (13, 2, 5), (14, 2, 1), (15, 2, 4), (17, 2, 3), (18, 2, 2),
       (7, 3, 3), (8, 3, 2), (9, 3, 1), (11, 3, 5), (12, 3, 3), (13, 3, 2), (16, 3, 1), (17, 3, 3), (20, 3, 1),
       (10, 4, 3), (13, 4, 2)]


@pytest.mark.parametrize("nb,lb,cols", LDE)
def test_lde(pc, oracle, nb, lb, cols):
    import torch
    n, ne = 1 << nb, 1 << (nb + lb)
    raw, trace = _words(n * cols, 7000 + 40 * nb + lb)
    out = pc.empty(ne * cols)
    pc.NTT_Goldilocks(n).LDE(out, pc.to_device(raw.reshape(n, cols)), ne, n, cols)
    torch.cuda.synchronize()
    got = colmajor_to_rowmajor(pc.to_host(out), ne, cols)
    assert (got == oracle.lde(trace.reshape(n, cols), ne)).all()


@pytest.mark.parametrize("lg,cols", [(10, 2), (11, 3), (14, 1), (15, 2), (16, 3), (17, 1), (19, 2), (21, 1), (22, 1)])
@pytest.mark.parametrize("inverse", [False, True])
def test_ntt(pc, oracle, lg, cols, inverse):
    import torch
    n = 1 << lg
    raw, a = _words(n * cols, 8000 + lg)
    d = pc.to_device(raw)
    ntt = pc.NTT_Goldilocks(n)
    (ntt.INTT if inverse else ntt.NTT)(None, d, n, cols, row_major=False)
    torch.cuda.synchronize()
    f = oracle.intt if inverse else oracle.ntt
    got = pc.to_host(d).reshape(cols, n)
    for c in range(cols):
        assert (got[c] == f(a.reshape(cols, n)[c])).all()


@pytest.mark.parametrize("nb,lb,qdeg,qdim", [(11, 0, 1, 3), (13, 1, 2, 3), (16, 1, 2, 1), (17, 1, 1, 3), (12, 2, 4, 3),
                                             (14, 2, 3, 3), (18, 2, 4, 1), (8, 3, 8, 3), (12, 3, 5, 3), (16, 3, 8, 1),
                                             (9, 4, 3, 3)])
def test_compute_q(pc, oracle, nb, lb, qdeg, qdim):
    import torch
    ne = 1 << (nb + lb)
    raw, q = _words(ne * qdim, 9000 + 40 * nb + lb)
    cm, _ = pc.compute_q(pc.to_device(raw), nb, nb + lb, qdeg, q_dim=qdim, arity=3, row_major=True)
    torch.cuda.synchronize()
    got = colmajor_to_rowmajor(pc.to_host(cm), ne, qdeg * qdim)
    assert (got == oracle.compute_q(q.reshape(ne, qdim), 1 << nb, qdeg)).all()


@pytest.mark.parametrize("lg,cols", [(4, 8), (5, 1), (6, 9), (11, 8), (12, 7), (12, 64), (13, 65), (15, 50)])
@pytest.mark.parametrize("inverse", [False, True])
def test_ntt_rows(pc, oracle, lg, cols, inverse):
    """Row-major transforms: about the width of the tile that transposes and reverses, fewer
    rows than it has, one column and many; in place and not."""
    import torch
    n = 1 << lg
    raw, a = _words(n * cols, 8500 + lg * 70 + cols)
    ntt = pc.NTT_Goldilocks(n)
    run = ntt.INTT if inverse else ntt.NTT
    src = pc.to_device(raw)
    dst = pc.empty(n * cols)
    run(dst, src, n, cols, row_major=True)
    torch.cuda.synchronize()
    assert (pc.to_host(src) == raw).all()
    run(None, src, n, cols, row_major=True)
    torch.cuda.synchronize()
    f = oracle.intt if inverse else oracle.ntt
    want = np.stack([f(a.reshape(n, cols)[:, c]) for c in range(cols)], axis=1)
    assert (pc.to_host(dst).reshape(n, cols) == want).all()
    assert (pc.to_host(src).reshape(n, cols) == want).all()


@pytest.mark.parametrize("lg,cols", [(22, 4), (22, 5)])
def test_ntt_rows_long(pc, lg, cols):
    """The longest narrow rows that go through one pass, and longer: as the columns do."""
    import torch
    n = 1 << lg
    raw, _ = _words(n * cols, 8900 + cols)
    ntt = pc.NTT_Goldilocks(n)
    rows = pc.to_device(raw)
    columns = rows.reshape(n, cols).t().contiguous().reshape(-1)
    ntt.INTT(None, rows, n, cols, row_major=True)
    ntt.INTT(None, columns, n, cols, row_major=False)
    torch.cuda.synchronize()
    assert torch.equal(rows.reshape(n, cols), columns.reshape(cols, n).t())


@pytest.mark.parametrize("lg,cols", [(4, 3), (7, 40), (10, 17), (15, 5), (23, 3)])
@pytest.mark.parametrize("dst_half,src_half", [(0, None), (1, None), (None, 1), (0, 1), (1, 1)])
def test_ntt_rows_within_the_scratch(pc, lg, cols, dst_half, src_half):
    """Row-major data whose result lies in a half of the scratch, or whose source lies in the
    second half: as with buffers of their own."""
    import torch
    n = 1 << lg
    raw, _ = _words(n * cols, 8600 + lg)
    ntt = pc.NTT_Goldilocks(n)
    want = pc.empty(n * cols)
    ntt.NTT(want, pc.to_device(raw), n, cols, row_major=True)
    buffer = pc.empty(2 * n * cols)
    src, dst = pc.to_device(raw), pc.empty(n * cols)
    if src_half is not None:
        half = buffer[src_half * n * cols:(src_half + 1) * n * cols]
        half.copy_(src)
        src = half
    if dst_half is not None:
        dst = buffer[dst_half * n * cols:(dst_half + 1) * n * cols]
    ntt.NTT(dst, src, n, cols, buffer=buffer, row_major=True)
    torch.cuda.synchronize()
    assert torch.equal(dst, want)


# blocks of two columns: even pairs and an odd last column, every line of a piece its own
# (blowup 8) or shared by waves (blowup 4), and one column fewer than pairs begin with
PAIRS = [(19, 3, 32), (19, 3, 33), (19, 3, 31), (20, 3, 16), (20, 3, 17), (21, 3, 8), (21, 3, 9), (20, 2, 32), (20, 2, 33),
         (21, 2, 17), (22, 2, 9)]


@pytest.mark.parametrize("nb,lb,cols", PAIRS)
def test_lde_in_pairs(pc, oracle, nb, lb, cols):
    import torch
    n, ne = 1 << nb, 1 << (nb + lb)
    some = sorted({0, 1, cols // 2 | 1, cols - 2, cols - 1})
    trace = pc.fill_uniform(pc.empty(n * cols), 7100 + 40 * nb + cols).reshape(n, cols)
    raw = pc.to_host(trace[:, some].contiguous()).reshape(n, len(some)).copy()
    edge, _ = _words(len(some) * 1000, 7200 + cols)
    raw[:1000] = edge.reshape(1000, len(some))
    trace[:, some] = pc.to_device(raw)
    out = pc.empty(ne * cols)
    pc.NTT_Goldilocks(n).LDE(out, trace, ne, n, cols)
    torch.cuda.synchronize()
    want = oracle.lde(np.where(raw >= np.uint64(P), raw - np.uint64(P), raw), ne)
    got = out.reshape(cols, ne)
    for k, c in enumerate(some):
        assert (pc.to_host(got[c]) == want[:, k]).all(), c


@pytest.mark.parametrize("lg", [23, 24])
@pytest.mark.parametrize("inverse", [False, True])
def test_ntt_longest_strided(pc, oracle, lg, inverse):
    """The transforms with 9 and 10 bits in the strided pass."""
    import torch
    n = 1 << lg
    raw, a = _words(n, 8000 + lg)
    d = pc.to_device(raw)
    ntt = pc.NTT_Goldilocks(n)
    (ntt.INTT if inverse else ntt.NTT)(None, d, n, 1, row_major=False)
    torch.cuda.synchronize()
    assert (pc.to_host(d) == (oracle.intt if inverse else oracle.ntt)(a)).all()
