"""The routes of large calls: a launch per table group on the group streams, and the
general path of block_bucketize.  Small calls take one launch and two launches instead,
so these run at sizes past those, or with TBE_FLAG_NO_STREAM, which excludes the
any-type kernel (a launch of the per-bag kernel per group)."""
import numpy as np
import pytest
import torch

import test_gpu_graphs
from _bucketize_cases import Case, gen_case
from test_gpu_coverage import _fp8_case, _fp8_params
from test_gpu_parity import (BF16, FP8, FP16, FP32, INT2, INT4, INT8, _check_module, _matrix_params, _random_case,
                             _say)
from test_gpu_sparse_ops import _check

pytestmark = pytest.mark.gpu

B_GROUPS = 20_000  # 120 k bags of the six-group module, ~20 rows each: past the one launch


def _kinds(pkg, m, B, rows, flags=0):
    offs = m.weights_offsets.cpu().numpy()
    _, _, s = pkg.capi.plan(offs, m.weights_tys.cpu().numpy(), m.D_offsets.cpu().numpy(), m.weights_dev.numel(),
                            fp8_exponent_bits=4, fp8_exponent_bias=7)
    return pkg.capi.pooled_kernels(s, len(offs), B, len(offs) * B * rows, flags=flags)


@pytest.mark.parametrize("pm,weighted,out_ty", [(0, False, FP16), (1, True, FP32)])
def test_groups_in_a_graph(pkg, gpu, pm, weighted, out_ty):
    # the forked group streams come along into the capture
    ks = _kinds(pkg, test_gpu_graphs._mixed_module(pkg, gpu, pm, out_ty), B_GROUPS, 20)
    assert len(ks) == 6 and pkg.capi.TBE_POOLED_ONE not in ks
    test_gpu_graphs.test_tbe_forward_graph_replays(pkg, gpu, pm, weighted, out_ty, B=B_GROUPS)


def test_groups_on_caller_streams_and_threads(pkg, gpu):
    test_gpu_graphs.test_concurrent_caller_streams_and_threads(pkg, gpu, B=B_GROUPS)


def test_group_streams_do_not_change_results(pkg, gpu):
    # 64 mixed tables: forked and serial groups, with and without the XCD order, and the default
    # call of the same size, bit for bit where the kernels are the same
    from fbgemm_ascend_amd.workloads import make_workload
    c = pkg.capi
    wl = make_workload(3, device=gpu, scale_rows=0.01, batch=256)
    m = wl.module
    _say("[gpu] group streams, 64 tables")

    def run(flags):
        out = c.forward_tensors(m.weights_dev, m.weights_offsets, m.weights_tys, m.D_offsets, wl.indices, wl.offsets,
                                int(m.pooling_mode), wl.per_sample_weights, m.output_dtype, flags=flags)
        torch.cuda.synchronize()
        return out

    want = run(c.TBE_FLAG_NO_STREAM)
    assert c.TBE_POOLED_ONE not in _kinds(pkg, m, 256, 32, c.TBE_FLAG_NO_STREAM)
    for extra in (c.TBE_FLAG_SERIAL_GROUPS, c.TBE_FLAG_NO_XCD_REMAP,
                  c.TBE_FLAG_SERIAL_GROUPS | c.TBE_FLAG_NO_XCD_REMAP):
        assert torch.equal(run(c.TBE_FLAG_NO_STREAM | extra), want), extra


@pytest.mark.parametrize("T", [5])
@pytest.mark.parametrize("ty,pm,weighted,idx_dtype,out_ty",
                         [p for p in _matrix_params([INT8, INT4, INT2, FP16, FP32, BF16, FP8]) if p[1] != 2])
def test_types_per_bag(pkg, oracle, gpu, T, ty, pm, weighted, idx_dtype, out_ty):
    m, idx, off, psw = _random_case(pkg, gpu, 77 + ty, T, ty, pm, weighted, idx_dtype, out_ty)
    _check_module(oracle, m, idx, off, psw, f"per-bag ty={ty} pm={pm} w={weighted} {idx_dtype} out={out_ty}",
                  flags=pkg.capi.TBE_FLAG_NO_STREAM)


@pytest.mark.parametrize("eb,bias,pm,weighted,idx_dtype,out_ty", [p for p in _fp8_params() if p[2] != 2])
def test_fp8_params_per_bag(pkg, oracle, gpu, eb, bias, pm, weighted, idx_dtype, out_ty):
    m, idx, off, psw = _fp8_case(pkg, gpu, eb * 16 + pm, 3, eb, bias, pm, weighted, idx_dtype, out_ty)
    _check_module(oracle, m, idx, off, psw, f"per-bag fp8 ({eb},{bias}) pm={pm} w={weighted} out={out_ty}",
                  flags=pkg.capi.TBE_FLAG_NO_STREAM)


# ----------------------------------------------------------------- block_bucketize, general path

@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("my_size", [16, 40])
@pytest.mark.parametrize("at", [5, 600, 1500])
def test_bucketize_rows_given_up(pkg, oracle, gpu, dtype, my_size, at):
    # rows of 400-1800 indices, 1.3 M in all: the fast scatter pass writes the chunks before
    # an index at or above the blocks, gives the row up, and the general pass rewrites it
    case = Case(f"given_up_at{at}_my{my_size}", 6, 200, 400, 1800, 8, 40, my_size, dtype)
    for seed, kw in ((61, dict(weights=True, sequence=True)), (62, dict(sequence=True, keep=True)),
                     (63, dict(weights=True, bucketize_pos=True))):
        lengths = gen_case(case, seed, kw.get("weights", False))[0]
        off = np.concatenate([[0], np.cumsum(lengths)])
        assert off[-1] > 1 << 20  # past the two launches

        def mutate(ix, lengths=lengths, off=off):
            ix = ix.copy()
            rows = np.flatnonzero(lengths > at)[::3]
            ix[off[rows] + at] = np.iinfo(ix.dtype).max - rows
            return ix

        _check(oracle, gpu, case, seed, mutate=mutate, **kw)


@pytest.mark.parametrize("my_size", [2, 16, 17, 64, 100])
@pytest.mark.parametrize("pos", [False, True])
def test_bucketize_many_rows(pkg, oracle, gpu, my_size, pos):
    case = Case(f"many_rows_my{my_size}", 5, 2700, 0, 12, 8, 40, my_size, np.int64)  # 13500 rows
    _check(oracle, gpu, case, 71, weights=True, sequence=True, pos=pos)
    _check(oracle, gpu, case, 72, bucketize_pos=True, bspf=True, pos=pos)


@pytest.mark.parametrize("sequence,weighted", [(False, False), (True, True)])
def test_bucketize_general_path_in_a_graph(pkg, gpu, sequence, weighted):
    # offsets scan, count, scan and the two scatter passes
    case = Case("graph_many_rows", 5, 2700, 0, 12, 8, 40, 8, np.int64)
    test_gpu_graphs.test_block_bucketize_graph_replays(pkg, gpu, sequence, weighted, case=case)
