"""fp32 queries against int4 streams read as nibbles (a handle's first calls)
and from the fp6 copy made later: the same scores, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (1, 15, 16, 17, 0, 31, 32, 33, 100, 0, 129, 1)


def _corpus(rng, dim):
    lengths = np.array(LENGTHS * 3, np.int64)
    offsets = np.concatenate(([0], np.cumsum(lengths))).astype(np.int64)
    tokens = int(offsets[-1])
    codes = [rng.integers(0, 256, (tokens, dim // 2), dtype=np.uint8) for _ in range(2)]
    codes[0][:256] = np.arange(256, dtype=np.uint8)[:, None]  # every pair of nibbles
    scale = [rng.uniform(0.5, 1.5, tokens).astype(np.float32) for _ in range(2)]
    return offsets, codes, scale


@pytest.mark.parametrize("dim", [2, 8, 20, 40, 128, 136, 256, 264, 384, 512])
@pytest.mark.parametrize("shape", [(1, 1), (1, 17), (2, 32), (3, 33), (1, 65)])
def test_scores_before_and_after_the_copy(gpu, oracle, dim, shape):
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs

    rng = np.random.default_rng(dim * 100 + shape[0] * shape[1])
    offsets, codes, scale = _corpus(rng, dim)
    query = rng.standard_normal((*shape, dim)).astype(np.float32)
    ids = rng.integers(0, offsets.size - 1, 5)
    calls = [(residual, reducer) for residual in (False, True) for reducer in ("maxsim", "topk2", "topk4", "smoothsim")]

    def handle():
        h = CudaInt4PackedDocs(codes[0], offsets, dim, 0.1)
        h.set_token_scale_vector(scale[0])
        h.set_residual_int4(codes[1], 0.01, scale[1])
        return h

    copied = handle()
    for _ in range(33):
        copied.score_residual_batch(query)
    have = copied.resident_bytes
    for residual, reducer in calls:
        h = handle()
        empty = h.resident_bytes
        full = h.score_residual_batch if residual else h.score_batch
        some = h.score_residual_candidates_batch if residual else h.score_candidates_batch
        exp = (copied.score_residual_batch if residual else copied.score_batch)(query, reducer, None, 0.5)
        np.testing.assert_array_equal(some(query, ids, reducer, None, 0.5), exp[:, ids])
        np.testing.assert_array_equal(full(query, reducer, None, 0.5), exp)
        if dim % 8 == 0:
            assert h.resident_bytes == empty  # nothing is copied by a first search
        for _ in range(32):
            np.testing.assert_array_equal(full(query, reducer, None, 0.5), exp)
        chunks = -(-dim // 128) if dim <= 256 else 4
        assert h.resident_bytes - empty >= (1 + residual) * int(offsets[-1]) * 96 * chunks
        np.testing.assert_array_equal(some(query, ids, reducer, None, 0.5), exp[:, ids])
    assert copied.resident_bytes == have
    # The cascade's two passes, its first and later calls.
    h = handle()
    first = h.cascade_topk(query, 3, 8)
    for _ in range(33):
        later = h.cascade_topk(query, 3, 8)
        np.testing.assert_array_equal(first[0], later[0])
        np.testing.assert_array_equal(first[1], later[1])
    # The nibbles' order: the oracle's scores.
    values = np.empty((codes[0].shape[0], dim), np.int8)
    values[:, 0::2] = (codes[0] << 4).view(np.int8) >> 4
    values[:, 1::2] = codes[0].view(np.int8) >> 4
    exp = oracle.int4_fp32_scores(query, values, offsets, scale=np.float32(0.1), token_scale=scale[0])
    got = handle().maxsim_batch(query)
    np.testing.assert_allclose(got, exp, rtol=1e-5, atol=1e-5 * max(1.0, float(np.abs(exp).max())))


@pytest.mark.parametrize("shape", [(1, 1), (1, 17), (2, 32), (3, 33), (1, 65)])
def test_binary_residual_before_and_after_the_copy(gpu, shape):
    from maxsim_amd._maxsim_hip import CudaPackedDocs

    rng = np.random.default_rng(shape[0] * shape[1])
    offsets, codes, scale = _corpus(rng, 128)

    def handle():
        h = CudaPackedDocs(rng2.integers(0, 256, (int(offsets[-1]), 16), dtype=np.uint8), offsets, 128)
        h.set_token_scale_vector(scale[0])
        h.set_residual_int4(codes[0], 0.01, scale[1])
        h.set_rescore_limbs(3)
        return h

    query = rng.standard_normal((*shape, 128)).astype(np.float32)
    ids = rng.integers(0, offsets.size - 1, (shape[0], 4))
    results = []
    for order in (0, 1):
        rng2 = np.random.default_rng(9)
        h = handle()
        for _ in range(33 * order):
            h.binres_score_batch(query)
        results.append((h.binres_score_batch(query, True, ids), h.cascade_topk(query, 3, 8), h.binres_score_batch(query)))
    (cand, top, full), (cand2, top2, full2) = results
    np.testing.assert_array_equal(cand, cand2)
    np.testing.assert_array_equal(top[0], top2[0])
    np.testing.assert_array_equal(top[1], top2[1])
    np.testing.assert_array_equal(full, full2)
    np.testing.assert_array_equal(np.take_along_axis(full, ids, 1), cand)
