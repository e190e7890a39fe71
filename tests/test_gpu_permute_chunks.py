"""permute_pooled_embs around the sizes where its kernels change, bit-exact against the
oracle: chunks of one, two and more source runs, row ends inside a chunk, the first and last
rows, rows either side of the narrow-row line and of one work-group, many segments."""
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
