"""The one-launch pooled kernel (calls of several table groups): rows at the edges of its
words per lane and column tiles, bags at the edges of its row steps, both waves per bag,
against the CPU oracle with the tolerance of tests/_parity.py."""
import pytest
import torch

from test_gpu_parity import BF16, FP8, FP16, FP32, INT2, INT4, INT8, _check_module

pytestmark = pytest.mark.gpu

PER_WORD = {FP32: 1, FP16: 2, BF16: 2, FP8: 4, INT8: 4, INT4: 8, INT2: 16}
# payload words: 1-4 lanes, INT4's half rows, a full tile and one past it, two and four
# words per lane with a cut last lane, more than one tile of four
WORDS = (1, 3, 5, 16, 17, 32, 33, 63, 64, 65, 127, 129, 131, 257)


@pytest.mark.parametrize("lengths", ["short", "long"])
@pytest.mark.parametrize("weighted,index,pm,out", [(False, torch.int32, 0, FP32), (True, torch.int64, 1, FP32),
                                                   (False, torch.int64, 1, FP16), (True, torch.int32, 0, BF16)])
@pytest.mark.parametrize("ty", sorted(PER_WORD))
def test_any_kernel_edges(pkg, oracle, gpu, ty, weighted, index, pm, out, lengths, fp8=(4, 7)):
    specs = [(40 + 7 * i, w * PER_WORD[ty], pkg.SparseType(ty)) for i, w in enumerate(WORDS)]
    m = pkg.IntNBitTableBatchedEmbeddingBagsCodegen(specs, device=gpu, pooling_mode=pm, output_dtype=out,
                                                    indices_dtype=index, fp8_exponent_bits=fp8[0],
                                                    fp8_exponent_bias=fp8[1])
    m.fill_random_weights(11)
    # "long" bags average over 32 rows, so four waves share one; "short" ones take a wave
    lens = [0, 1, 2, 7, 8, 9, 16, 33] if lengths == "short" else [0, 1, 3, 31, 64, 65, 129, 200]
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    L = torch.tensor([lens[(i + t) % len(lens)] for t in range(len(specs)) for i in range(len(lens))], device=gpu)
    per = len(lens)
    idx = torch.cat([torch.randint(-1, E + 1, (int(L[t * per:(t + 1) * per].sum()),), device=gpu, generator=g)
                     for t, (E, _, _) in enumerate(specs)]).to(index)  # -1 and E: skipped rows
    off = torch.cat([torch.zeros(1, dtype=torch.int64, device=gpu), L.cumsum(0)]).to(index)
    psw = torch.rand(idx.numel(), device=gpu, generator=g) if weighted else None
    _check_module(oracle, m, idx, off, psw, f"any ty={ty} {lengths}")


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("bits,bias", [(1, 3), (2, 5), (3, 0), (5, 15), (7, 60)])
def test_any_kernel_fp8_formats(pkg, oracle, gpu, bits, bias, weighted):
    # up to 4 exponent bits codes are read as shifted fp16 halves, above through fp32
    test_any_kernel_edges(pkg, oracle, gpu, FP8, weighted, torch.int32, 0, FP32, "short", fp8=(bits, bias))


@pytest.mark.parametrize("out,D", [(FP32, 16), (FP16, 64), (BF16, 128), (FP16, 144), (FP32, 1040), (FP16, 2064)])
@pytest.mark.parametrize("ty", sorted(PER_WORD))
def test_nobag_batches(pkg, oracle, gpu, ty, out, D):
    # sequence rows: segments cut inside and at the edges of the 8-load batches and 64-index
    # chunks, widths of one load, of a cut last lane and of several column tiles
    specs = [(60 + 9 * t, D, pkg.SparseType(ty)) for t in range(3)]
    m = pkg.IntNBitTableBatchedEmbeddingBagsCodegen(specs, device=gpu, pooling_mode=2, output_dtype=out)
    m.fill_random_weights(4)
    g = torch.Generator(device=gpu)
    g.manual_seed(D)
    L = torch.tensor([1, 63, 0, 64, 7, 130, 8, 9, 0, 15, 31, 1], device=gpu)
    idx = torch.cat([torch.randint(-1, E + 1, (int(L[t * 4:t * 4 + 4].sum()),), device=gpu, generator=g)
                     for t, (E, _, _) in enumerate(specs)]).to(torch.int32)
    off = torch.cat([torch.zeros(1, dtype=torch.int64, device=gpu), L.cumsum(0)]).to(torch.int32)
    _check_module(oracle, m, idx, off, None, f"nobag ty={ty} D={D} out={out}")


@pytest.mark.parametrize("ty,out", [(INT8, FP32), (FP16, FP16), (INT4, BF16)])
def test_nobag_far_output_rows(pkg, gpu, ty, out):
    # output rows so far apart that 64 of them span more than 4 GiB
    D = 16 * PER_WORD[ty] if ty != INT4 else 32 * PER_WORD[ty]
    m = pkg.IntNBitTableBatchedEmbeddingBagsCodegen([(50, D, pkg.SparseType(ty))], device=gpu, pooling_mode=2,
                                                    output_dtype=out)
    m.fill_random_weights(4)
    idx = torch.arange(-1, 65, dtype=torch.int32, device=gpu)  # -1 and 50 on: zero rows
    off = torch.tensor([0, idx.numel()], dtype=torch.int32, device=gpu)
    want = m(idx, off, None)
    stride = ((1 << 32) // (64 * want.element_size())) + 16
    far = torch.empty((idx.numel(), stride), dtype=want.dtype, device=gpu)
    far[:, :D] = 7
    print(f"[gpu] nobag far rows ty={ty} stride={stride}", flush=True)
    pkg.capi.forward_tensors(m.weights_dev, m.weights_offsets, m.weights_tys, m.D_offsets, idx, off, 2, None,
                             m.output_dtype, m.row_alignment, out=far)
    assert torch.equal(far[:, :D], want)
