"""fp32 queries as five base-32 digits against the C oracle, at the tile, chunk and pass edges.

The documents are exact in fp32 (scales are powers of two), so with
e = 2^-24 the scores differ from exact ones by, per query token and at
its documents' largest sum |doc||q|: the row's fixed point (half a unit of
2^(E-24), 2^E <= 2 max|q|), one fp32 rounding per MFMA of the chain (five digits
per 128 dims, a residual's as many) and up to eight in the epilogue, weights
and the oracle; then one per addition of the query tokens.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (1, 15, 16, 17, 0, 31, 32, 33, 100, 0, 129, 1)


def _codes(rng, tokens, dim):
    v = rng.integers(-8, 8, (tokens, dim)).astype(np.int8)
    v[0] = -8
    return v, ((v[:, 0::2] & 15) | ((v[:, 1::2] & 15) << 4)).astype(np.uint8)


def _bound(query, sims_abs, row_abs, streams, chunks, temperature):
    """[batch, docs]: the error of the module's docstring, both sides together."""
    e = 2.0**-24
    per_row = sims_abs * (streams * 5 * chunks + 8) * e + row_abs * 2 * e + temperature * 16 * e + 2.0**-146
    return per_row.sum(1) + sims_abs.sum(1) * query.shape[1] * e


def _doc_max(x, offsets):
    """Largest of each document's tokens: x [tokens, rows] -> [docs, rows]."""
    return np.stack([x[s:e].max(0) if e > s else np.zeros(x.shape[1]) for s, e in zip(offsets[:-1], offsets[1:])])


@pytest.mark.parametrize("kind", ["int4", "residual", "sign", "sign_scaled"])
@pytest.mark.parametrize("dim", [8, 128, 136, 256, 264, 512])
@pytest.mark.parametrize("shape", [(1, 1), (1, 16), (3, 17), (2, 32), (5, 32), (2, 65)])
def test_digit_scores_at_the_edges(gpu, oracle, kind, dim, shape):
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs, CudaPackedDocs

    rng = np.random.default_rng(dim * 100 + shape[0] * shape[1])
    lengths = np.array(LENGTHS * 3, np.int64)
    offsets = np.concatenate(([0], np.cumsum(lengths))).astype(np.int64)
    tokens = int(offsets[-1])
    scale = np.exp2(rng.integers(-2, 3, tokens)).astype(np.float32)
    values, packed = _codes(rng, tokens, dim)
    streams = 1
    if kind in ("int4", "residual"):
        h = CudaInt4PackedDocs(packed, offsets, dim, 1.0)
        h.set_token_scale_vector(scale)
        docs = values * scale[:, None]
        score, cand_score, kw = h.score_batch, h.score_candidates_batch, {}
        if kind == "residual":
            values2, packed2 = _codes(rng, tokens, dim)
            scale2 = scale / 16
            h.set_residual_int4(packed2, 1.0, scale2)
            docs = docs + values2 * scale2[:, None]
            score, cand_score, streams = h.score_residual_batch, h.score_residual_candidates_batch, 2
    else:
        bits = rng.integers(0, 2, (tokens, dim))
        h = CudaPackedDocs(np.packbits(bits, axis=1, bitorder="little"), offsets, dim)
        docs = (2 * bits - 1).astype(np.float32)
        score, cand_score, kw = h.score_batch, h.score_candidates_batch, {}
        if kind == "sign_scaled":
            h.set_token_scale_vector(scale)
            docs = docs * scale[:, None]
            kw = {"use_token_scale": True}
    query = rng.standard_normal((*shape, dim)).astype(np.float32)
    flat = query.reshape(-1, dim)
    flat[0] = 0.0
    flat[-1, 0] = 64.0  # one element far above the rest of its row
    near = query.copy()
    if shape[0] > 1:  # whole batch rows far from the others
        query[1] *= np.float32(1e30)
        query[-1] *= np.float32(1e-41) if shape[0] > 2 else np.float32(1)
    ids = rng.integers(0, lengths.size, 37)
    chunks = {8: 1, 128: 1, 136: 2, 256: 2}.get(dim, 4)
    mag = np.abs(docs).astype(np.float64)
    if kind == "residual":
        mag = np.abs(values * scale[:, None]).astype(np.float64) + np.abs(values2 * scale2[:, None])
    for reducer, temperature in (("maxsim", 0.0), ("topk2", 0.0), ("topk4", 0.0), ("smoothsim", 0.5)):
        if reducer == "smoothsim":
            query = near  # (no exponents of rows of 1e30)
        q64 = np.abs(query.reshape(-1, dim)).astype(np.float64)
        sims = _doc_max(mag @ q64.T, offsets).T.reshape(*shape, lengths.size)
        rows = (_doc_max(mag.sum(1)[:, None], offsets).T * q64.max(1)[:, None]).reshape(*shape, lengths.size)
        args = {"temperature": temperature} if reducer == "smoothsim" else {}
        got = score(query, reducer, None, **args, **kw)
        exp = oracle.dense_scores(query, docs, offsets, reducer=reducer, **args)
        err = np.abs(got.astype(np.float64) - exp)
        # (a log-sum of up to 129 terms rounds each of them)
        bound = _bound(query, sims, rows, streams, chunks, 129 * temperature)
        assert (err <= bound).all(), (reducer, float((err / np.maximum(bound, 1e-300)).max()))
        np.testing.assert_array_equal(cand_score(query, ids, reducer, None, **args, **kw), got[:, ids])


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_rows_that_are_not_finite_leave_the_others_alone(gpu, bad):
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs

    rng = np.random.default_rng(5)
    offsets = np.arange(0, 40 * 33, 33, dtype=np.int64)
    _, packed = _codes(rng, int(offsets[-1]), 128)
    h = CudaInt4PackedDocs(packed, offsets, 128, 0.1)
    query = rng.standard_normal((4, 8, 128)).astype(np.float32)
    clean = h.score_batch(query, "maxsim")
    query[2, 3, 7] = bad
    got = h.score_batch(query, "maxsim")
    np.testing.assert_array_equal(got[[0, 1, 3]], clean[[0, 1, 3]])
    if np.isinf(bad):
        assert np.isnan(got[2]).all()


@pytest.mark.parametrize("tau", [0.5, 3.0])
@pytest.mark.parametrize("shape", [(1, 8), (2, 16), (1, 32), (3, 17), (2, 32), (1, 64), (2, 65)])
def test_smoothsim_at_document_scales_that_are_zero_or_negative(gpu, oracle, shape, tau):
    """Documents of whole tiles and with masked rows, first in their wave (every
    document of a candidate call is) and later ones; a zero scale's score is
    tau ln(tokens) per query token."""
    from maxsim_amd._maxsim_hip import CudaPackedDocs

    rng = np.random.default_rng(shape[0] * 100 + shape[1])
    lengths = np.array((16, 32, 5, 48, 17, 0, 160, 1) * 50, np.int64)
    offsets = np.concatenate(([0], np.cumsum(lengths))).astype(np.int64)
    bits = rng.integers(0, 2, (int(offsets[-1]), 128))
    scale = np.resize(np.array([0.0, 0.25, -0.5, 0.0, 0.0, -1.0, -0.25, -0.125, 0.5], np.float32), lengths.size)
    h = CudaPackedDocs(np.packbits(bits, axis=1, bitorder="little"), offsets, 128)
    h.set_scale_vector(scale)
    docs = (2 * bits - 1).astype(np.float32) * np.repeat(scale, lengths)[:, None]
    query = rng.standard_normal((*shape, 128)).astype(np.float32)
    args = {"temperature": tau}
    got = h.score_batch(query, "smoothsim", None, use_scale_vector=True, **args)
    exp = oracle.dense_scores(query, docs, offsets, reducer="smoothsim", **args)
    q64 = np.abs(query.reshape(-1, 128)).astype(np.float64)
    mag = np.abs(docs).astype(np.float64)
    sims = _doc_max(mag @ q64.T, offsets).T.reshape(*shape, lengths.size)
    rows = (_doc_max(mag.sum(1)[:, None], offsets).T * q64.max(1)[:, None]).reshape(*shape, lengths.size)
    assert (np.abs(got.astype(np.float64) - exp) <= _bound(query, sims, rows, 1, 1, 160 * tau)).all()
    ids = rng.integers(0, lengths.size, 61)
    np.testing.assert_array_equal(
        h.score_candidates_batch(query, ids, "smoothsim", None, use_scale_vector=True, **args), got[:, ids])


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3e38])
@pytest.mark.parametrize("reducer", ["maxsim", "topk2", "topk4", "smoothsim"])
def test_token_scales_of_one_document_leave_the_others_alone(gpu, reducer, bad):
    """A token scale that is not finite (or whose products are not): only its
    own document's scores may differ, not those of the document before it,
    whose last tile holds that token among its masked rows."""
    from maxsim_amd._maxsim_hip import CudaPackedDocs

    rng = np.random.default_rng(6)
    offsets = np.concatenate(([0], np.cumsum(np.resize([10, 16, 1, 33, 47], 200)))).astype(np.int64)
    h = CudaPackedDocs(rng.integers(0, 256, (int(offsets[-1]), 16), dtype=np.uint8), offsets, 128)
    scale = rng.uniform(0.5, 1.5, int(offsets[-1])).astype(np.float32)
    ids = np.arange(offsets.size - 1)
    for shape in ((1, 8), (2, 32), (3, 17)):
        query = rng.standard_normal((*shape, 128)).astype(np.float32)
        h.set_token_scale_vector(scale)
        clean = h.score_batch(query, reducer, use_token_scale=True)
        marked = ids[1::4]
        scale2 = scale.copy()
        scale2[offsets[marked]] = bad
        h.set_token_scale_vector(scale2)
        others = np.setdiff1d(ids, marked)
        np.testing.assert_array_equal(h.score_batch(query, reducer, use_token_scale=True)[:, others], clean[:, others])
        got = h.score_candidates_batch(query, ids, reducer, use_token_scale=True)
        np.testing.assert_array_equal(got[:, others], clean[:, others])


@pytest.mark.parametrize("dim, shapes", [(128, [(3, 33), (4, 40), (5, 50), (16, 33)]), (256, [(8, 17), (3, 20)]),
                                         (512, [(8, 17), (3, 20)])])
def test_batch_rows_cut_at_the_ends_of_passes(gpu, dim, shapes):
    """Corpora large enough that badly filled passes are not taken: the scores
    are bit for bit those of each query by itself."""
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs

    rng = np.random.default_rng(dim)
    lengths = rng.integers(0, 130, 4000)
    offsets = np.concatenate(([0], np.cumsum(lengths))).astype(np.int64)
    _, packed = _codes(rng, int(offsets[-1]), dim)
    h = CudaInt4PackedDocs(packed, offsets, dim, 0.1)
    h.set_residual_int4(_codes(rng, int(offsets[-1]), dim)[1], 0.01, np.ones(int(offsets[-1]), np.float32))
    ids = rng.integers(0, 4000, 3500)
    for shape in shapes:
        query = rng.standard_normal((*shape, dim)).astype(np.float32)
        weights = rng.uniform(0.5, 1.5, shape).astype(np.float32)
        for reducer, w in (("weighted_maxsim", weights), ("smoothsim", None)):
            each = [h.score_batch(query[b : b + 1], reducer, None if w is None else w[b])[0] for b in range(shape[0])]
            np.testing.assert_array_equal(h.score_batch(query, reducer, w), np.stack(each))
            got = h.score_candidates_batch(query, ids, reducer, w)
            np.testing.assert_array_equal(got, np.stack(each)[:, ids])
        each = [h.score_residual_batch(query[b : b + 1])[0] for b in range(shape[0])]
        np.testing.assert_array_equal(h.score_residual_batch(query), np.stack(each))


@pytest.mark.parametrize("scale, row, token", [(1e-7, -117, 10), (1.0, 127, -20), (1e5, 120, -30)])
def test_factors_whose_product_alone_leaves_the_floats_range(gpu, scale, row, token):
    """Query rows, token scales and a tensor scale far from 1 whose similarities
    are ordinary floats (rows of up to 2^row, token scales of 2^token)."""
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs

    rng = np.random.default_rng(8)
    offsets = np.arange(0, 33 * 40, 33, dtype=np.int64)
    tokens = int(offsets[-1])
    values, packed = _codes(rng, tokens, 128)
    h = CudaInt4PackedDocs(packed, offsets, 128, scale)
    h.set_token_scale_vector(np.full(tokens, 2.0**token, np.float32))
    query = rng.uniform(-1, 1, (2, 32, 128)).astype(np.float32) * np.float32(2.0**row)
    docs = values * (2.0**token * float(np.float32(scale)))
    sims = docs @ query.reshape(-1, 128).T.astype(np.float64)
    mag = np.abs(docs) @ np.abs(query.reshape(-1, 128).T.astype(np.float64))
    rows = _doc_max(np.abs(docs).sum(1)[:, None], offsets).T * np.abs(query.reshape(-1, 128)).max(1).astype(np.float64)[:, None]
    shape = (2, 32, offsets.size - 1)
    bound = _bound(query, _doc_max(mag, offsets).T.reshape(shape), rows.reshape(shape), 1, 1, 0.0)
    ordered = np.sort(sims.reshape(offsets.size - 1, 33, 64), axis=1)[:, ::-1]
    for reducer, k in (("maxsim", 1), ("topk2", 2), ("topk4", 4)):
        exp = ordered[:, :k].mean(1).T.reshape(shape).sum(1)
        got = h.score_batch(query, reducer)
        assert np.isfinite(got).all()
        assert (np.abs(got.astype(np.float64) - exp) <= bound).all(), reducer
