"""permute_pooled_embs around the sizes where its launch changes, bit-exact against the
oracle: vectors of every width and alignment, rows of one work-group from 1 to 64, row blocks
either side of the number of XCDs, many segments, lists that leave columns out."""
import numpy as np
import pytest
import torch

from test_gpu_pooled_ops import _run_and_check
from test_pooled_ops import lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("B", [1, 2, 3, 5, 64, 1031])
@pytest.mark.parametrize("dims", [[1280], [1281], [640, 1, 640], [2047, 3, 8], [3] * 500, [1, 2, 5, 7, 9, 31] * 40,
                                  [16, 0, 1300, 0, 0, 8], [7] * 2048, [2] * 2049])
def test_permute_chunks(pkg, oracle, gpu, dims, B, dtype):
    rng = np.random.default_rng(len(dims) + B)
    permute = rng.permutation(len(dims)).tolist()
    x = torch.from_numpy(rng.integers(0, 2 ** 11, (B, sum(dims)))).to(dtype)
    _run_and_check(oracle, gpu, dims, permute, x, via="fbgemm")


def test_permute_lists_out_of_order(pkg, oracle, gpu):
    # destination segments that go back or leave the row: the ones that lie in the row are written
    x = torch.arange(2 * 3000, dtype=torch.float32).view(2, 3000)
    off = np.array([0, 1000, 2000, 3000], np.int64)
    perm = np.array([1, 0, 2], np.int64)
    inv = np.array([2000, 3000, 1000, 3500], np.int64)  # the second has no width it may write, the third leaves
    out = torch.full_like(x, -1.0).to(gpu)
    pkg.capi.permute_pooled_embs(x.to(gpu), *(torch.from_numpy(a).to(gpu) for a in (off, perm, inv)), out=out)
    torch.cuda.synchronize()
    want = torch.full_like(x, -1.0)
    want[:, 2000:3000] = x[:, 1000:2000]
    assert torch.equal(out.cpu(), want)


def _by_lists(x, off, perm, inv, out):
    """The columns each destination segment takes, in list order (x, out: [B, D, inner])."""
    D, T = x.shape[1], len(perm)
    for t in range(T):
        a, b = int(inv[t]), int(inv[t + 1])
        if a < 0 or b < a or b > D:
            continue
        src = int(off[perm[t]]) if 0 <= perm[t] < T else -1
        out[:, a:b] = x[:, src:src + b - a] if 0 <= src <= D - (b - a) else 0
    return out


@pytest.mark.parametrize("elem", [2, 4])
@pytest.mark.parametrize("inner", [1, 3])
@pytest.mark.parametrize("dims", [[700, 1, 9, 400], [4096, 8], [4200] * 3, [64] * 40, [5, 7, 2] * 30])
@pytest.mark.parametrize("B", [1, 7, 8, 9, 63, 65, 448, 449, 513])
def test_permute_lists(pkg, gpu, dims, B, inner, elem):
    # columns before the first segment and after the last are not written, a segment without
    # a source is zero, one whose source leaves the row is zero
    T, gap = len(dims), 3
    D = sum(dims) + gap + 2
    rng = np.random.default_rng(T + B)
    perm = rng.permutation(T)
    off = np.concatenate([[0], np.cumsum(dims)])
    inv = gap + np.concatenate([[0], np.cumsum([dims[p] for p in perm])])
    perm[rng.integers(T)] = -1
    perm[rng.integers(T)] = T
    off[rng.integers(T)] = D - 1
    x = rng.integers(-2 ** 15, 2 ** 15, (B, D, inner)).astype(np.int16 if elem == 2 else np.int32)
    want = _by_lists(x, off, perm, inv, np.full_like(x, 77))
    as_float = torch.float16 if elem == 2 else torch.float32  # bits are copied
    out = torch.full((B, D, inner), 77, dtype=torch.int16 if elem == 2 else torch.int32, device=gpu)
    print(f"[gpu] permute lists T={T} D={D} B={B} inner={inner} elem={elem}", flush=True)
    pkg.capi.permute_pooled_embs(torch.from_numpy(x).to(gpu).view(as_float),
                                 *(torch.from_numpy(a.astype(np.int64)).to(gpu) for a in (off, perm, inv)),
                                 out=out.view(as_float))
    assert np.array_equal(out.cpu().numpy(), want)
