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


@pytest.mark.parametrize("ty,D,bags,rows,want", [
    # row streams: short bags, not for rows of 512 columns of few bits
    (INT8, 64, 49_152, 1, "STREAM"), (INT8, 64, 49_151, 1, "BAG"), (INT4, 512, 262_144, 2, "BAG"),
    (INT4, 512, 262_144, 5, "STREAM"), (INT4, 1024, 262_144, 5, "BAG"), (INT2, 512, 524_288, 2, "BAG"),
    (INT2, 512, 524_288, 5, "STREAM"), (INT2, 1024, 262_144, 5, "BAG"), (FP32, 64, 8192, 8, "STREAM"),
    (FP32, 64, 8192, 9, "BAG"), (FP16, 256, 131_072, 12, "STREAM"), (FP16, 256, 131_072, 13, "BAG"),
    (INT8, 256, 32_768, 2, "STREAM"), (INT8, 256, 32_768, 3, "BAG"), (INT8, 256, 131_072, 6, "STREAM"),
    (INT8, 512, 131_072, 6, "BAG"), (FP8, 512, 131_072, 6, "STREAM"), (FP8, 512, 131_072, 7, "BAG"),
    # 33-128 words: waves that end with their bag, for about a round of the GPU's waves
    (FP16, 128, 4095, 24, "ANY"), (FP16, 128, 4096, 24, "BAG"), (FP16, 128, 2048, 23, "BAG"),
    (FP32, 128, 8191, 16, "ANY"), (FP32, 128, 4096, 17, "BAG"), (INT8, 512, 1023, 60, "BAG"),
    (INT8, 512, 1024, 60, "ANY"), (INT8, 512, 4096, 60, "BAG"), (FP8, 256, 32_767, 24, "ANY"),
    (FP8, 256, 32_768, 24, "BAG"), (FP8, 512, 131_071, 24, "ANY"), (FP8, 512, 131_072, 24, "BAG"),
    (INT4, 512, 2048, 48, "ANY"), (INT4, 512, 32_768, 48, "BAG"), (INT4, 512, 2048, 47, "BAG"),
    # past 128 words: not long bags that are few
    (FP32, 512, 8192, 30, "BAG"), (FP32, 512, 12_288, 30, "ANY"), (FP32, 512, 8192, 12, "ANY"),
    (FP32, 256, 2048, 16, "ANY"), (INT8, 1024, 8191, 30, "BAG"), (INT8, 1024, 8192, 30, "ANY"),
    (FP8, 1024, 1023, 9, "BAG"), (FP8, 1024, 1024, 100, "ANY"), (FP16, 512, 32_768, 8, "STREAM"),
])
def test_kernel_of_one_group(pkg, ty, D, bags, rows, want):
    c = pkg.capi
    assert kinds(pkg, [(1000, D, ty)], bags, rows) == [getattr(c, "TBE_POOLED_" + want)]
