"""int8 scans of several passes in one launch: batches at and past the rows of a pass, even and uneven splits, exactly
against the C oracle; a binary-prefix scan against the passes of single rows."""
import numpy as np
import pytest

from conftest import ragged_fixture

pytestmark = pytest.mark.gpu

SHAPES = [(4, 32), (5, 32), (7, 21), (9, 16), (16, 8), (17, 8), (3, 128), (2, 127), (5, 65), (40, 48), (130, 1), (300, 3)]


@pytest.mark.parametrize("granularity", ["token", "tensor"])
@pytest.mark.parametrize("shape", SHAPES)
def test_scan_passes_bit_exact(gpu, oracle, granularity, shape):
    from maxsim_amd.experimental import int4_maxsim_int8q, int4_to_device, pack_int4_symmetric

    docs, offsets = ragged_fixture(150, seed=71, hi=20)
    query = np.random.default_rng(shape[0] * 131 + shape[1]).standard_normal((*shape, 128)).astype(np.float32)
    packed = pack_int4_symmetric(docs, offsets, scale_granularity=granularity)
    exp = oracle.int4_int8q_scores(query, packed.values, packed.doc_offsets, token_scale=packed.token_scale,
                                   scale=float(packed.scale))
    np.testing.assert_array_equal(int4_maxsim_int8q(query, int4_to_device(packed)), exp)


@pytest.mark.parametrize("shape", [(5, 32), (7, 21), (3, 128), (40, 48)])
def test_prefix_scan_passes_do_not_depend_on_the_batch(gpu, shape):
    from maxsim_amd.binres import binres_cascade_topk, binres_to_device, pack_binary_residual

    docs, offsets = ragged_fixture(700, seed=11, hi=20)
    query = np.random.default_rng(shape[0] * 131 + shape[1]).standard_normal((*shape, 128)).astype(np.float32)
    dev = binres_to_device(pack_binary_residual(docs, offsets))
    got = binres_cascade_topk(query, dev, k=10, candidates=64)
    for b in (0, shape[0] // 2, shape[0] - 1):
        one = binres_cascade_topk(query[b:b + 1], dev, k=10, candidates=64)
        np.testing.assert_array_equal(np.asarray(got[0])[b], np.asarray(one[0])[0])
        np.testing.assert_array_equal(np.asarray(got[1])[b], np.asarray(one[1])[0])
