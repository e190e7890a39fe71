"""The kernel a table group takes by its bags, rows per bag and row width: one call on each
side of every line of the rule, against the CPU oracle with the tolerance of tests/_parity.py."""
import pytest
import torch

from test_gpu_parity import BF16, FP8, FP16, FP32, INT2, INT4, INT8, _check_module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("types,D,T,B,rows,weighted", [
    ((FP32,), 128, 2, 4095, 2, False), ((FP32,), 128, 2, 4096, 2, True),      # 8192 bags: row streams of plain rows
    ((FP16,), 130, 2, 4096, 2, False),                                         # an odd word count: no row stream
    ((BF16,), 128, 1, 8192, 17, False),                                        # past 16 rows a bag
    ((BF16,), 128, 1, 32768, 17, True),                                        # until 32768 bags
    ((INT8,), 256, 1, 32767, 12, False), ((INT8,), 256, 1, 32768, 12, False),
    ((INT8,), 512, 1, 64, 40, False), ((INT8,), 256, 1, 64, 23, False), ((INT8,), 256, 1, 64, 24, True),
    ((INT4,), 512, 1, 64, 24, False), ((INT4,), 512, 1, 64, 24, True), ((INT2,), 1024, 1, 64, 24, False),
    ((FP8,), 1024, 2, 64, 5, True), ((FP8,), 1028, 1, 300, 40, False),         # rows past 128 words
    ((FP32,), 512, 1, 32768, 1, False), ((FP32,), 514, 1, 32768, 1, True),
    ((INT8,), 64, 1, 49151, 1, False), ((INT4,), 64, 1, 49152, 1, True),       # 49152 bags per row of a bag
    ((INT8, FP16, FP32), 128, 3, 43690, 1, False), ((INT8, FP16, FP32), 128, 3, 43691, 1, False),  # 2^17 bags in all
    ((INT2, BF16), 64, 2, 65537, 2, True),
    ((INT8, FP16, FP32), 128, 3, 26624, 2, True), ((INT8, FP16, FP32), 128, 3, 26625, 2, True),  # short bags, 3 groups
    ((INT8, FP16, FP32), 128, 3, 43690, 24, False),                            # long bags: 2^17 in all
    ((INT2, FP8), 1024, 2, 65537, 9, True),    # past both: the any-type kernel for the second group alone
])
def test_dispatch_lines(pkg, oracle, gpu, types, D, T, B, rows, weighted):
    specs = [(500 + 30 * t, D, pkg.SparseType(types[t % len(types)])) for t in range(T)]
    m = pkg.IntNBitTableBatchedEmbeddingBagsCodegen(specs, device=gpu, pooling_mode=1, output_dtype=FP32)
    m.fill_random_weights(3)
    g = torch.Generator(device=gpu)
    g.manual_seed(B)
    L = torch.full((T * B,), rows, device=gpu)
    L[::7] -= 1   # empty or shorter bags, made up for by longer ones: the mean stays `rows`
    L[3::7] += 1
    L[-1] += T * B * rows - int(L.sum())
    assert int(L.sum()) == T * B * rows and int(L.min()) >= 0
    idx = torch.randint(0, 500, (int(L.sum()),), device=gpu, generator=g).to(torch.int32)
    off = torch.cat([torch.zeros(1, dtype=torch.int64, device=gpu), L.cumsum(0)]).to(torch.int32)
    psw = torch.rand(idx.numel(), device=gpu, generator=g) if weighted else None
    b_sel = torch.unique(torch.cat([torch.arange(0, min(B, 40)), torch.arange(max(0, B - 70), B)]))
    _check_module(oracle, m, idx, off, psw, f"{types} D={D} T={T} B={B} rows={rows}", b_sel=b_sel)
