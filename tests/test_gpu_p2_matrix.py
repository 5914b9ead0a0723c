"""GPU tests of the Poseidon2 kernels whose partial rounds run on the matrix cores:
trees tall enough for one permutation per lane (above 16,384 rows and parents), at the
edges of waves and blocks, over boundary words, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P = 0xFFFFFFFF00000001
EDGE_WORDS = [0, 1, 2, 2**31, 2**32 - 1, 2**32, 2**32 + 1, 2**63 - 1, 2**63, P - 2**32, P - 2, P - 1, P, P + 1,
              P + 2**32 - 2, 2**64 - 2**33, 2**64 - 2, 2**64 - 1, 0x8080808080808080, 0x7F7F7F7F7F7F7F7F]


@pytest.fixture(scope="module")
def pc():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a HIP device")
    import pil2_commit
    pil2_commit.set_hash_family(2)
    return pil2_commit


@pytest.mark.parametrize("arity", [2, 3, 4])
@pytest.mark.parametrize("rows,extra", [(16385, 0), (16384 + 63, 1), (16384 + 257, -3), (3 * 16384 + 513, 2),
                                        (1 << 16, 9)])
def test_tall_tree_matches_oracle(pc, oracle, arity, rows, extra):
    """rows x (rate + extra) columns, column-major, half boundary words, half random."""
    import torch
    cols = max(4 * arity - 4 + extra, 1)
    rng = np.random.default_rng(rows + 10 * arity + extra)
    src = rng.integers(0, 2**64, (rows, cols), dtype=np.uint64)
    edge = np.array(EDGE_WORDS, dtype=np.uint64)[rng.integers(0, len(EDGE_WORDS), (rows, cols))]
    src[::2] = edge[::2]
    d = pc.to_device(np.ascontiguousarray(src.T))
    t = pc.MerkleTreeGL(arity, 0, True, rows, cols, source=d, row_stride=1, col_stride=rows)
    t.merkelize()
    torch.cuda.synchronize()
    assert (pc.to_host(t.nodes) == oracle.merkletree(src, arity)).all()


@pytest.mark.parametrize("arity", [2, 3, 4])
@pytest.mark.parametrize("rows", [2, 3, 4, 5, 9, 10, 16, 17, 27, 28, 32, 33, 64, 65, 82, 145, 255, 257, 1025, 6913,
                                  8193, 16384])
def test_short_tree_matches_oracle(pc, oracle, arity, rows):
    """Trees whose levels take 16 lanes a permutation and several levels a launch: one to
    three blocks of every kind, partly filled ones, pads, and the switch to single levels;
    one or two blocks of columns, boundary words in every other row."""
    import torch
    cols = 4 * arity - 4 + (rows % 3) - 1
    rng = np.random.default_rng(rows * 5 + arity)
    src = rng.integers(0, 2**64, (rows, cols), dtype=np.uint64)
    edge = np.array(EDGE_WORDS, dtype=np.uint64)[rng.integers(0, len(EDGE_WORDS), (rows, cols))]
    src[::2] = edge[::2]
    t = pc.MerkleTreeGL(arity, 0, True, rows, cols, source=pc.to_device(src))
    t.nodes = pc.empty(t.num_nodes)
    t.nodes.fill_(-1)
    t.merkelize()
    torch.cuda.synchronize()
    assert (pc.to_host(t.nodes) == oracle.merkletree(src, arity)).all()
