"""Sign-bit queries at the Hamming kernel's edges, exactly against the C oracle:
every count of 16-row blocks per pass, passes with and without whole batch
rows, sums in registers and in LDS, empty, short and long documents."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (1, 15, 16, 0, 17, 33, 0, 129, 300, 2)


@pytest.mark.parametrize("docs", [1, 9, 700])
@pytest.mark.parametrize("shape", [(1, 1), (1, 32), (2, 17), (2, 32), (5, 24), (4, 32), (3, 50), (6, 32), (8, 32),
                                   (9, 32), (7, 48), (1, 256), (2, 257), (40, 13)])
def test_hamming_scores_at_the_edges(gpu, oracle, shape, docs):
    from maxsim_amd._maxsim_hip import CudaPackedDocs

    rng = np.random.default_rng(shape[0] * 1000 + shape[1] + docs)
    lengths = np.resize(np.array(LENGTHS, np.int64), docs)
    if docs == 1:
        lengths[:] = 35
    offsets = np.concatenate(([0], np.cumsum(lengths))).astype(np.int64)
    codes = rng.integers(0, 256, (int(offsets[-1]), 16), dtype=np.uint8)
    bits = rng.integers(0, 256, (*shape, 16), dtype=np.uint8)
    h = CudaPackedDocs(codes, offsets, 128)
    exp = oracle.binary_hamming_maxsim(bits, codes, offsets, 128)
    got = h.hamming_batch(bits)
    np.testing.assert_array_equal(got, exp)
    k = min(docs, 10)
    scores, ids = h.topk_hamming(bits, k)
    np.testing.assert_array_equal(np.take_along_axis(exp, np.asarray(ids), 1), np.asarray(scores))
    np.testing.assert_array_equal(np.sort(exp, 1)[:, ::-1][:, :k], np.asarray(scores))
