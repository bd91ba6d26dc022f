"""Device top-k (msim_topk_async) against the oracle's stable order for every
selector: threshold filter (n <= 4096, k <= 32), row threshold (k <= 1024),
radix (larger k)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 100, 1000, 4096, 4097, 10000, 16384, 20000])
@pytest.mark.parametrize("k", [1, 10, 32, 33, 500])
def test_topk_matches_oracle_with_ties(gpu, oracle, n, k):
    import torch

    from maxsim_amd._maxsim_hip import _stream_ptr
    from maxsim_amd._native import check, ptr

    if k > n:
        pytest.skip("k must not exceed n")
    rng = np.random.default_rng(n * 131 + k)
    scores = rng.integers(-50, 50, size=(3, n)).astype(np.float32) * np.float32(0.25)  # many ties
    scores[1, : n // 2] = -np.inf
    scores[2, 0] = -0.0
    d = torch.from_numpy(scores).cuda()
    s = torch.empty((3, k), dtype=torch.float32, device="cuda")
    i = torch.empty((3, k), dtype=torch.int64, device="cuda")
    check(gpu.msim_topk_async(ptr(d), 3, n, n, k, ptr(s), ptr(i), _stream_ptr(None)))
    torch.cuda.synchronize()
    es, ei = oracle.topk(scores, k)
    np.testing.assert_array_equal(i.cpu().numpy(), ei)
    np.testing.assert_array_equal(s.cpu().numpy(), es)


@pytest.mark.parametrize("n", [16385, 24577, 65536])
@pytest.mark.parametrize("k", [1, 32, 100, 1024, 1025])
def test_long_rows_of_a_handle_are_selected_chunk_by_chunk(gpu, n, k):
    """Rows longer than a workgroup's registers (16,384 scores) go through the
    handle's scratch memory, k <= 1024, else through the radix form.  Documents
    of one token, every third one a copy of its neighbour (ties across chunk
    borders), the best ones adjacent."""
    from maxsim_amd._maxsim_hip import CudaInt4PackedDocs

    rng = np.random.default_rng(n + k)
    codes = rng.integers(0, 256, size=(n, 64), dtype=np.uint8)
    codes[2::3] = codes[1::3][: len(codes[2::3])]
    codes[n // 2 : n // 2 + 700] = codes[n // 2]
    h = CudaInt4PackedDocs(codes, np.arange(n + 1, dtype=np.int64), 128, 1.0)
    query = rng.standard_normal((2, 3, 128)).astype(np.float32)
    scores = h.maxsim_batch_int8q(query)
    order = np.stack([np.lexsort((np.arange(n), -row)) for row in scores])[:, :k]
    top_s, top_i = h.topk_batch_int8q(query, k)
    np.testing.assert_array_equal(top_i, order)
    np.testing.assert_array_equal(top_s, np.take_along_axis(scores, order, axis=1))


@pytest.mark.parametrize("n", [5000, 16384, 40000])
def test_rows_whose_best_scores_share_threads_or_tie(gpu, oracle, n):
    """More than 4,096 scores reach the threshold: rows of one value (every
    score ties) and rows whose larger half is one value take the radix form;
    -0 ties +0 at the threshold."""
    import torch

    from maxsim_amd._maxsim_hip import _stream_ptr
    from maxsim_amd._native import check, ptr

    k = 100
    scores = np.zeros((3, n), np.float32)
    scores[1, : n // 2 - 200] = -3.0
    scores[2] = -1.0
    scores[2, 7::50] = 0.0
    scores[2, 8::50] = -0.0
    d = torch.from_numpy(scores).cuda()
    s = torch.empty((3, k), dtype=torch.float32, device="cuda")
    i = torch.empty((3, k), dtype=torch.int64, device="cuda")
    check(gpu.msim_topk_async(ptr(d), 3, n, n, k, ptr(s), ptr(i), _stream_ptr(None)))
    torch.cuda.synchronize()
    es, ei = oracle.topk(scores, k)
    np.testing.assert_array_equal(i.cpu().numpy(), ei)
    np.testing.assert_array_equal(s.cpu().numpy(), es)
