"""Which kernel a pooled call takes (tbe_nbit_pooled_kernels): host arithmetic, no GPU."""
import numpy as np
import pytest

FP32, FP16, INT8, INT4, INT2, BF16, FP8 = 0, 1, 2, 3, 4, 5, 6
BITS = {FP32: 32, FP16: 16, INT8: 8, INT4: 4, INT2: 2, BF16: 16, FP8: 8}


def kinds(pkg, specs, B, rows, **kw):
    """Kernel per group of tables [(rows, D, type)] at B samples of `rows` rows a bag."""
    offs, total = [], 0
    for E, D, ty in specs:
        offs.append(total)
        total += E * ((D * BITS[ty] // 8 + (4 if ty in (INT8, INT4, INT2) else 0) + 15) // 16 * 16)
    _, _, s = pkg.capi.plan(offs, [ty for _, _, ty in specs], np.cumsum([0] + [D for _, D, _ in specs]), total,
                            fp8_exponent_bits=4, fp8_exponent_bias=7)
    return pkg.capi.pooled_kernels(s, len(specs), B, len(specs) * B * rows, **kw)


@pytest.mark.parametrize("ty,D,rows", [(FP8, 516, 1), (INT8, 516, 20), (FP32, 514, 1), (INT4, 264, 30)])
def test_launch_fits_the_grid(pkg, ty, D, rows):
    # a wave per bag: a launch of 2^32 or more threads is refused, so such a call takes a
    # kernel that needs no more waves than the GPU holds
    c = pkg.capi
    most = 4 * (0xFFFFFFFF // 256)  # items of the largest launch
    tiles = -(-(D * BITS[ty] // 32) // 64)
    for B in (most - 3, most + 1, 0x7FFFFFFF // tiles):
        for k in kinds(pkg, [(1000, D, ty)], B, rows):
            assert k in (c.TBE_POOLED_BAG, c.TBE_POOLED_STREAM) or (k == c.TBE_POOLED_ANY and B <= most), B


NARROW2 = [(1000, 64, INT8), (1000, 64, INT4)]
NARROW12 = [(1000, D, ty) for ty in (INT8, INT4, INT2, FP16) for D in (32, 64, 128)]


@pytest.mark.parametrize("specs,bags,rows,one", [
    # short bags: the waves of one launch against the launches it saves
    (NARROW2 * 8, 69_632, 2, True), (NARROW2 * 8, 69_648, 2, False), (NARROW2 * 8, 131_072, 23, False),
    (NARROW12 * 4, 131_040, 2, True),
    # long bags
    (NARROW2 * 8, 131_072, 24, True), (NARROW2 * 8, 131_088, 24, False), (NARROW12 * 4, 131_136, 60, False),
    # every table gets the column tiles of the widest: 16
    (NARROW2 * 7 + [(1000, 4096, FP32)], 16_384, 2, False), (NARROW2 * 7 + [(1000, 4096, FP32)], 4_096, 2, True),
    (NARROW2 * 7 + [(1000, 4096, FP32)], 8_175, 40, True), (NARROW2 * 7 + [(1000, 4096, FP32)], 16_384, 40, False),
])
def test_one_launch_of_several_groups(pkg, specs, bags, rows, one):
    c = pkg.capi
    got = kinds(pkg, specs, bags // len(specs), rows)
    assert all((k == c.TBE_POOLED_ONE) == one for k in got), got
    flagged = kinds(pkg, specs, bags // len(specs), rows, flags=c.TBE_FLAG_NO_STREAM)
    assert c.TBE_POOLED_ONE not in flagged and c.TBE_POOLED_ANY not in flagged
