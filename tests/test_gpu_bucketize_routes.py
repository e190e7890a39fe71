"""block_bucketize_sparse_features at the sizes where it changes its kernels, exactly
against the CPU oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _compare(oracle, gpu, lengths, indices, block_sizes, my, lists=None, weighted=True):
    w = np.random.default_rng(1).uniform(-1, 1, indices.size).astype(np.float32) if weighted else None
    print(f"[gpu] bucketize routes L={lengths.size} N={indices.size} F={block_sizes.size} my={my}", flush=True)
    want = oracle.block_bucketize_sparse_features(lengths, indices, True, True, block_sizes, my, weights=w,
                                                  block_bucketize_pos=lists)
    d = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    got = torch.ops.fbgemm.block_bucketize_sparse_features(
        d(lengths), d(indices), True, True, d(block_sizes), my, weights=d(w),
        block_bucketize_pos=None if lists is None else [d(p) for p in lists])
    for name, g, e in zip(("lengths", "indices", "weights", "pos", "unbucketize"), got, want):
        assert (g is None) == (e is None), name
        if e is not None:
            assert np.array_equal(g.cpu().numpy(), e), name


@pytest.mark.parametrize("F,my,dtype", [(1, 2, np.int64), (120, 16, np.int32), (121, 17, np.int64), (250, 64, np.int32)])
def test_position_lists(pkg, oracle, gpu, F, my, dtype):
    # the lists' addresses travel 120 a launch; every row takes the general map
    rng = np.random.default_rng(F)
    lengths = rng.integers(0, 90, F * 3).astype(dtype)
    lists = [np.concatenate([[0], rng.integers(1, 50, my).cumsum()]).astype(dtype) for _ in range(F)]
    indices = rng.integers(0, 60 * my, int(lengths.sum())).astype(dtype)
    _compare(oracle, gpu, lengths, indices, np.full(F, 30, dtype), my, lists)


@pytest.mark.parametrize("L", [5, 4096, 270_000])
def test_rows_past_their_blocks(pkg, oracle, gpu, L):
    # every other row holds an index past its blocks: the general pass rewrites them, and
    # from 2^18 rows a wave of it walks more than one batch of flags
    rng = np.random.default_rng(L)
    lengths = rng.integers(1, 4, L).astype(np.int32)
    indices = rng.integers(0, 64 * 3, int(lengths.sum())).astype(np.int32)
    starts = np.cumsum(lengths) - lengths
    indices[starts[::2]] += 64 * 3
    _compare(oracle, gpu, lengths, indices, np.array([64], np.int32), 3)
