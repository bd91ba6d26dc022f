"""More documents than one launch's work units cover (2^24): the fp32-query and
sign-query scorers go over them range by range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DOCS = (1 << 24) + 3


def _documents(rng):
    """One or two tokens per document, the last ones among them."""
    lengths = np.ones(DOCS, np.int64)
    lengths[:: 1 << 20] = 2
    lengths[-1] = 2
    lengths[7] = lengths[-3] = 0
    return np.concatenate(([0], np.cumsum(lengths)))


def _max_per_document(sims, offsets):
    """[rows, tokens] -> [rows, documents]; an empty document has 0."""
    out = np.zeros((sims.shape[0], offsets.size - 1), sims.dtype)
    full = np.flatnonzero(np.diff(offsets) > 0)
    out[:, full] = np.maximum.reduceat(sims, offsets[full], axis=1)
    return out


def test_fp32_scores_of_more_than_2_24_documents(gpu):
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs

    rng = np.random.default_rng(41)
    offsets = _documents(rng)
    tokens = int(offsets[-1])
    codes = rng.integers(0, 256, (tokens, 4), dtype=np.uint8)
    values = np.empty((tokens, 8), np.int8)
    values[:, 0::2] = (codes << 4).view(np.int8) >> 4
    values[:, 1::2] = codes.view(np.int8) >> 4
    h = CudaInt4PackedDocs(codes, offsets, 8, 1.0)
    h.set_residual_int4(codes, 0.5, np.ones(tokens, np.float32))
    # Small integers: every product and sum is exact.
    query = rng.integers(-3, 4, (1, 2, 8)).astype(np.float32)
    sims = query[0] @ values.T.astype(np.float32)
    rows = _max_per_document(sims, offsets)
    exp = rows.sum(0)
    np.testing.assert_array_equal(h.maxsim_batch(query)[0], exp)
    np.testing.assert_array_equal(h.topk_score_batch(query, 3, residual=True)[0][0], np.sort(1.5 * exp)[::-1][:3])
    wide = np.concatenate([query[0]] * 40)[None]  # 80 tokens: summed by the second launch
    np.testing.assert_array_equal(h.maxsim_batch(wide)[0], 40 * exp)
    # A cascade's coarse pass; its best have the best scores (ties by document).
    best = np.lexsort((np.arange(DOCS), -exp))[:4]
    scores, ids = h.cascade_topk(query, 4, 64)
    np.testing.assert_array_equal(ids[0], best)
    np.testing.assert_array_equal(scores[0], 1.5 * exp[best])


def test_sign_scores_of_more_than_2_24_documents(gpu):
    from maxsim_amd._maxsim_hip import CudaPackedDocs

    rng = np.random.default_rng(42)
    offsets = _documents(rng)
    words = rng.integers(0, 1 << 64, (int(offsets[-1]), 2), dtype=np.uint64)
    h = CudaPackedDocs(words.view(np.uint8), offsets, 128)
    bits = rng.integers(0, 1 << 64, (2, 2), dtype=np.uint64)
    sims = np.stack([128 - 2 * np.bitwise_count(words ^ row).sum(1, dtype=np.int32) for row in bits])
    exp = _max_per_document(sims, offsets).sum(0)
    np.testing.assert_array_equal(h.hamming_batch(bits.view(np.uint8)[None])[0], exp)
    np.testing.assert_array_equal(h.hamming_batch(np.stack([bits] * 2).view(np.uint8))[1], exp)
    long = np.concatenate([bits] * 150)[None]  # 300 tokens: summed by the second launch
    np.testing.assert_array_equal(h.hamming_batch(long.view(np.uint8))[0], 150 * exp)
    # (-1 / +1 as an fp32 query: the same scores, with a scale per document)
    scale = rng.integers(1, 4, DOCS).astype(np.float32)
    h.set_scale_vector(scale)
    signs = np.unpackbits(bits.view(np.uint8), axis=1, bitorder="little").astype(np.float32)[None] * 2 - 1
    np.testing.assert_array_equal(h.maxsim_batch(signs, use_scale_vector=True)[0], exp * scale)


@pytest.mark.parametrize("kind", ["int4", "binary_int8", "binary_fp32"])
def test_more_batch_rows_than_grid_rows(gpu, kind):
    """Per-row candidate lists take a grid row per batch row, and a launch has
    at most 65,535: the results are those of the same rows a part at a time."""
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs, CudaPackedDocs

    rng = np.random.default_rng(43)
    offsets = np.array([0, 3, 3, 20, 21, 40], np.int64)
    dim = 8 if kind == "int4" else 128
    codes = rng.integers(0, 256, (40, dim // 2), dtype=np.uint8)
    scale = rng.uniform(0.5, 1.5, 40).astype(np.float32)
    if kind == "int4":
        h = CudaInt4PackedDocs(codes, offsets, dim, 1.0)
        h.set_residual_int4(rng.integers(0, 256, codes.shape, dtype=np.uint8), 0.1, scale)
    else:
        h = CudaPackedDocs(rng.integers(0, 256, (40, 16), dtype=np.uint8), offsets, dim)
        h.set_token_scale_vector(scale)
        h.set_residual_int4(codes, 0.1, scale)
        h.set_rescore_limbs(3 if kind == "binary_fp32" else 1)
    query = rng.standard_normal((66_000, 1, dim)).astype(np.float32)
    scores, ids = h.cascade_topk(query, 2, 3)
    for part in (slice(0, 1000), slice(65_000, 66_000)):
        exp_s, exp_i = h.cascade_topk(query[part], 2, 3)
        np.testing.assert_array_equal(scores[part], exp_s)
        np.testing.assert_array_equal(ids[part], exp_i)
