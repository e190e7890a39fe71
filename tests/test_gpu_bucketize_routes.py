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


# the two-launch path: 4, 8 and 16 rows a work-group, cut last groups, the last sizes it
# takes and the first it does not, the smallest calls
@pytest.mark.parametrize("F,B,my,dtype", [
    (1, 1, 1, np.int32), (1, 1, 33, np.int64), (1, 1, 64, np.int64), (3, 1, 2, np.int64), (7, 9, 64, np.int32),
    (1, 2048, 16, np.int64), (1, 2049, 16, np.int64), (2, 2047, 32, np.int64), (1, 4097, 32, np.int64),
    (1, 16384, 16, np.int32), (1, 16385, 16, np.int32), (5, 1639, 64, np.int64), (1, 300, 65, np.int64)])
@pytest.mark.parametrize("lists", [False, True])
def test_few_rows(pkg, oracle, gpu, F, B, my, dtype, lists):
    rng = np.random.default_rng(F * B + my)
    lengths = rng.integers(0, 12, F * B).astype(dtype)
    lengths[:: max(1, F * B // 3)] = 700  # rows of more than one chunk
    pos = [np.concatenate([[0], rng.integers(1, 50, my).cumsum()]).astype(dtype) for _ in range(F)] if lists else None
    indices = rng.integers(0, 40 * my, int(lengths.sum())).astype(dtype)  # some past the blocks of 25
    _compare(oracle, gpu, lengths, indices, np.full(F, 25, dtype), my, pos)


# a wave per row in groups of 4, 8 and 16 rows: the lines between them, and the last rows
# taken without and with lists (8192 of int64, 12288)
@pytest.mark.parametrize("F,B,my,dtype", [
    (1, 2048, 2, np.int64), (1, 2049, 2, np.int64), (1, 4095, 16, np.int32), (1, 4096, 17, np.int64),
    (1, 4097, 2, np.int64), (3, 5, 40, np.int64), (2, 4096, 32, np.int64), (1, 8192, 33, np.int64),
    (1, 8193, 8, np.int64), (4, 3072, 8, np.int32), (1, 12289, 8, np.int32), (3, 4095, 21, np.int64)])
@pytest.mark.parametrize("lists", [False, True])
def test_few_rows_groups(pkg, oracle, gpu, F, B, my, dtype, lists):
    test_few_rows(pkg, oracle, gpu, F, B, my, dtype, lists)


@pytest.mark.parametrize("L", [1, 5, 4099])
def test_few_rows_c_abi(pkg, oracle, gpu, L):
    # offsets given or formed, scratch of the caller or the library's own; new_offsets is an output
    rng = np.random.default_rng(L)
    lengths = rng.integers(0, 9, L).astype(np.int64)
    indices = rng.integers(0, 12, int(lengths.sum())).astype(np.int64)
    want = oracle.block_bucketize_sparse_features(lengths, indices, False, True, np.array([4]), 3)
    d = lambda a: torch.from_numpy(a).to(gpu)  # noqa: E731
    for noalloc in (False, True):
        for pass_offsets in (False, True):
            got, offs = pkg.capi.block_bucketize_sparse_features(d(lengths), d(indices), False, True,
                                                                 d(np.array([4])), 3, noalloc=noalloc,
                                                                 pass_offsets=pass_offsets)
            for g, e in zip(got, want):
                if e is not None:
                    assert np.array_equal(g.cpu().numpy(), e)
            assert np.array_equal(offs.cpu().numpy(), np.concatenate([[0], want[0].cumsum()]))
