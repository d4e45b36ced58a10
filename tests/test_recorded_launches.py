"""What a recorded program holds (tch_program_launches): which kernel a call is sent to, on the CPU.  Nothing runs: the
addresses are made up."""
import ctypes
import os
import subprocess
import sys

import pytest

from sirius_amd._lib import LaunchStat, check, lib

F32, BF16 = 0, 1
dtypes = pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])


def address(i):
    return ctypes.c_void_p(0x10000000 * (i + 1))


class Recorder:
    """A context and the programs recorded on it."""

    def __init__(self):
        self.ctx = ctypes.c_void_p()
        check(lib().tch_context_create(None, ctypes.byref(self.ctx)))
        self.progs = []

    def begin(self):
        prog = ctypes.c_void_p()
        check(lib().tch_program_create(ctypes.byref(prog)))
        check(lib().tch_program_begin_record(self.ctx, prog))
        self.progs.append(prog)

    def end(self):
        """End the recording; [(kernel name, workgroups, lane)] of the launches in it (joins of the lanes: '')."""
        check(lib().tch_program_end_record(self.ctx))
        prog = self.progs[-1]
        cap = int(lib().tch_program_size(prog))
        rows, n = (LaunchStat * max(cap, 1))(), ctypes.c_int64()
        check(lib().tch_program_launches(prog, rows, cap, ctypes.byref(n)))
        assert n.value == cap
        return [(r.name.decode(), int(r.workgroups), int(r.lane)) for r in rows[:cap]]

    def close(self):
        for p in self.progs:
            lib().tch_program_destroy(p)
        lib().tch_context_destroy(self.ctx)


@pytest.fixture
def rec():
    r = Recorder()
    yield r
    r.close()


K, C, ROWS = 256, 192, 4096
NAMES = {F32: "f32", BF16: "bf16"}


def wgrad(rec, dtype, tile_cfg, splits, trailing=False):
    args = [rec.ctx, dtype, address(0), address(1), address(2)]
    tail = [address(3), splits, 0, ROWS, 1, 1, C, K, 1, 1, 1, 0, tile_cfg, 0]
    if trailing:
        check(lib().tch_conv2d_wgrad_trailing(*args, None, *tail))
    else:
        check(lib().tch_conv2d_wgrad(*args, *tail))


@dtypes
@pytest.mark.parametrize("tile_cfg", range(25))
def test_every_tiling_number_of_a_weight_gradient_runs_its_kernel(rec, dtype, tile_cfg):
    """The tilings of the other directions stand for a shape; none of their kernels may get a weight gradient's operands."""
    side = {0: (128, 128), 1: (128, 64)}.get({9: 0, 10: 0, 11: 0, 12: 0, 23: 0, 24: 0, 5: 1, 6: 1, 13: 1, 22: 1}.get(tile_cfg, tile_cfg), (64, 64))
    tiles = (K // side[0]) * (-(-C // side[1]))
    for splits in (1, 4):
        rec.begin()
        wgrad(rec, dtype, tile_cfg, splits)
        got = rec.end()
        assert got[0][:2] == (f"wgrad_kernel<{NAMES[dtype]},{side[0]}x{side[1]}>", tiles * splits)
        assert [g[0] for g in got[1:]] == ["splitk_reduce_kernel"] * (splits > 1)


@dtypes
@pytest.mark.parametrize("tile_cfg", [2, 15, 20])
def test_a_pending_reduction_rides_whatever_tiling_is_asked_for(rec, dtype, tile_cfg):
    rec.begin()
    wgrad(rec, dtype, 2, 4, trailing=True)
    wgrad(rec, dtype, tile_cfg, 4, trailing=True)
    check(lib().tch_conv2d_wgrad_flush(rec.ctx))
    first, second, last = rec.end()
    assert last[0] == "splitk_reduce_kernel" and second[1] == first[1] + last[1]


@dtypes
def test_pending_sums_end_with_the_recording(rec, dtype):
    """A recording that ends before its flush (a plan whose building raised) leaves nothing for the next one to take along:
    the sums are the last launches of their own program, behind a join of the lanes."""
    rec.begin()
    wgrad(rec, dtype, 2, 4, trailing=True)
    check(lib().tch_conv2d_wgrad_flush(rec.ctx))
    clean = rec.end()

    rec.begin()
    check(lib().tch_layernorm_defer_sums(rec.ctx, 1))
    check(lib().tch_layernorm_bwd(rec.ctx, dtype, *[address(i) for i in range(3)], None, *[address(i) for i in range(3, 8)],
                                  0, ROWS, C, address(8)))
    check(lib().tch_layernorm_defer_sums(rec.ctx, 0))
    check(lib().tch_context_set_lane(rec.ctx, 1, 1))
    wgrad(rec, dtype, 2, 4)                     # not one that takes sums along: the column sums stay pending ...
    check(lib().tch_conv2d_wgrad_flush(rec.ctx))
    wgrad(rec, dtype, 2, 4, trailing=True)      # ... until the flush; this reduction pends when the recording ends
    cut = rec.end()
    names = [c[0] for c in cut]
    assert names[0].startswith("ln_bwd_kernel") and "col_sum_kernel" in names
    assert names[-2:] == ["", "splitk_reduce_kernel"] and cut[-1][2] == 0

    rec.begin()
    wgrad(rec, dtype, 2, 4, trailing=True)
    check(lib().tch_conv2d_wgrad_flush(rec.ctx))
    assert rec.end() == clean


def test_pending_column_sums_end_with_the_recording(rec):
    rec.begin()
    check(lib().tch_layernorm_defer_sums(rec.ctx, 1))
    check(lib().tch_layernorm_bwd(rec.ctx, BF16, *[address(i) for i in range(3)], None, *[address(i) for i in range(3, 8)],
                                  0, ROWS, C, address(8)))
    check(lib().tch_layernorm_defer_sums(rec.ctx, 0))
    assert [r[0] for r in rec.end()] == ["ln_bwd_kernel<bf16>", "", "col_sum_kernel"]
    rec.begin()
    check(lib().tch_conv2d_wgrad_flush(rec.ctx))
    assert rec.end() == []


def in_own_process(body, **env):
    """What `body` prints, with the settings of `env` (they are read once per process)."""
    head = "import sys\nsys.path[:0] = [%r, %r]\nimport test_recorded_launches as T\nrec, a = T.Recorder(), T.address\n" % (
        os.path.dirname(os.path.abspath(__file__)), os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    out = subprocess.run([sys.executable, "-c", head + body], env=dict(os.environ, **env), stdout=subprocess.PIPE, check=True)
    return out.stdout.decode().split("|")


def choice(**env):
    """Splits and kernel of a weight gradient, and the kernel of a shallow pointwise product."""
    sp, wgrad_name, fwd_name = in_own_process("""
sp = T.lib().tch_conv2d_wgrad_pick_splits(1, 8192, 1, 1, 1024, 1024, 1, 1, 1, 0)
rec.begin()
T.check(T.lib().tch_conv2d_wgrad(rec.ctx, 1, a(0), a(1), a(2), a(3), sp, 0, 8192, 1, 1, 1024, 1024, 1, 1, 1, 0, -1, 0))
T.check(T.lib().tch_conv2d_fwd(rec.ctx, 1, a(0), a(1), a(2), None, None, None, 0, 200704, 1, 1, 64, 256, 1, 1, 1, 0, -1, 0))
names = [r[0] for r in rec.end()]
print(sp, names[0], names[-1], sep="|", end="")
""", **env)
    return int(sp), wgrad_name, fwd_name


def test_settings_of_the_library_s_own_choice():
    """TCH_WGRAD_WGS, TCH_WGRAD_BIG_TILE_WGS and TCH_IGEMM_K32 override what the tables of costs say."""
    splits, wgrad_name, fwd_name = choice()
    assert wgrad_name == "wgrad_kernel<bf16,128x128>" and ",k32" in fwd_name
    assert choice(TCH_WGRAD_WGS="64")[0] == 1 and choice(TCH_WGRAD_WGS="1024")[0] == 16 and 1 < splits < 16
    assert choice(TCH_WGRAD_BIG_TILE_WGS="100000")[1] == "wgrad_kernel<bf16,64x64>"
    assert ",k32" not in choice(TCH_IGEMM_K32="0")[2]


@dtypes
@pytest.mark.parametrize("setting", ["", "0", "2", "3"])
def test_row_tiles_of_the_statistics_are_those_of_the_kernel(dtype, setting):
    """Callers size the BatchNorm sums by tch_conv2d_fwd_stat_rows / tch_conv2d_dgrad_stat_rows: the kernel that runs has that
    many row tiles, for every tiling and setting of TCH_IGEMM2.  0: igemm_kernel whatever tiling is asked for."""
    got = in_own_process("""
dtype, staged, L = %d, %r, T.lib()
for cfg in [-2, -1] + list(range(25)):
    for shape in ((2, 14, 14, 128, 256, 3, 3, 1, 1), (1, 56, 56, 64, 128, 1, 1, 2, 0), (3, 9, 7, 24, 40, 3, 3, 1, 1),
                  (64, 56, 56, 256, 64, 1, 1, 1, 0), (1, 7, 7, 32, 512, 1, 1, 1, 0)):
        rec.begin()
        T.check(L.tch_conv2d_fwd_bnstats(rec.ctx, dtype, a(0), a(1), a(2), *shape, cfg, 0, a(3)))
        T.check(L.tch_conv2d_dgrad_bnsums(rec.ctx, dtype, a(0), a(1), a(2), None, None, *shape, cfg, 0, a(3), a(4), a(5), a(6),
                                          a(7), 1))
        rows = (L.tch_conv2d_fwd_stat_rows(dtype, *shape, cfg), L.tch_conv2d_dgrad_stat_rows(dtype, *shape, cfg))
        n, h, w, c, k, r, s, stride, pad = shape
        out = (h + 2 * pad - r) // stride + 1, (w + 2 * pad - r) // stride + 1
        for (name, wgs, _), row_tiles, m, cols in zip(rec.end(), rows, (n * out[0] * out[1], n * h * w), (k, c)):
            bm, bn = map(int, name.split(",")[2].rstrip(">").split("x"))
            assert row_tiles == -(-m // bm) and wgs == row_tiles * -(-cols // bn), (cfg, name)
            assert not staged or name.startswith("igemm_kernel<"), (cfg, name)
print("ok", end="")
""" % (dtype, setting == "0"), **({"TCH_IGEMM2": setting} if setting else {}))
    assert got == ["ok"]


@dtypes
@pytest.mark.parametrize("tile_cfg", range(25))
def test_floor_table_files_every_convolution_kernel_under_its_direction(rec, dtype, tile_cfg):
    from sirius_amd.floor_table import family
    rec.begin()
    check(lib().tch_conv2d_fwd(rec.ctx, dtype, address(0), address(1), address(2), None, None, None, 0, 2, 14, 14, 128, 128, 3, 3, 1, 1,
                               tile_cfg, 0))
    check(lib().tch_conv2d_dgrad(rec.ctx, dtype, address(0), address(1), address(2), None, None, 2, 14, 14, 128, 128, 3, 3, 1, 1,
                                 tile_cfg, 0, 1))
    wgrad(rec, dtype, tile_cfg, 1)
    assert [family(r[0]) for r in rec.end()] == ["conv forward", "conv data gradient", "conv weight gradient"]


# rows, output columns, reduction, and what the library takes for them in fp32: both sides of every line of its choice
F32_CHOICE = [
    (196, 256, 1008, "32x32,4way"), (196, 256, 1024, "32x32,8way"), (196, 256, 128, "32x32,4way"),
    (256, 1024, 1024, "32x32,8way"), (257, 1024, 1024, "32x32,4way"), (257, 1024, 1520, "32x32,4way"), (257, 1024, 1536, "64x32,8way"),
    (512, 1024, 1024, "32x32,4way"), (513, 1024, 1024, "64x64,8way"), (513, 1024, 768, "64x64,8way"), (513, 1024, 752, "64x32,4way"),
    (1024, 1024, 1024, "64x64,8way"), (1025, 1024, 1024, "64x32,4way"), (513, 1024, 512, "64x32,4way"), (513, 1024, 496, "64x64,4way"),
    (2048, 1024, 512, "64x32,4way"), (2049, 1024, 512, "64x64,4way"), (2049, 1024, 256, "64x64,4way"), (2049, 1024, 240, "igemm_kernel<f32,fwd,64x64"),
    (6016, 1024, 256, "64x64,4way"), (6017, 1024, 256, "igemm_kernel<f32,fwd,128x128"), (6017, 1024, 128, "igemm_kernel<f32,fwd,64x64"),
]


def product(rec, dtype, rows, cols, depth, tile_cfg):
    rec.begin()
    check(lib().tch_conv2d_fwd(rec.ctx, dtype, address(0), address(1), address(2), None, None, None, 0, rows, 1, 1, depth, cols, 1, 1,
                               1, 0, tile_cfg, 0))
    (name, _, _), = rec.end()
    return name


@pytest.mark.parametrize("rows,cols,depth,want", F32_CHOICE)
def test_fp32_choice_on_both_sides_of_its_lines(rec, rows, cols, depth, want):
    assert want in product(rec, F32, rows, cols, depth, -1)
    assert product(rec, F32, rows, cols, depth, -2).startswith("igemm_kernel<f32,fwd,")


# rows, output columns, reduction, tiling and whether a forward product and a data gradient multiply in bf16 parts: both sides of
# every line of that choice
F32_PARTS = [
    (257, 1024, 512, "32x32,4way", False, False), (132, 1024, 1024, "32x32,8way", True, False), (128, 1024, 1024, "32x32,8way", False, False),
    (513, 1024, 768, "64x64,8way", True, True), (1025, 1024, 16368, "64x32,4way", True, False), (1025, 1024, 16384, "64x32,4way", False, False),
    (257, 1024, 1536, "64x32,8way", True, False), (1025, 1024, 256, "64x64,4way", True, True), (784, 1024, 256, "64x64,4way", False, False),
    (6017, 1024, 256, "128x128", True, True), (6017, 1024, 240, "128x128", False, False),
]


@pytest.mark.parametrize("rows,cols,depth,tiling,parts,dgrad_parts", F32_PARTS)
def test_fp32_products_in_parts(rec, rows, cols, depth, tiling, parts, dgrad_parts):
    name = product(rec, F32, rows, cols, depth, -1)
    assert tiling in name and name.endswith(",parts>") == parts, name
    assert "parts" not in product(rec, F32, rows, cols, depth, -2)
    rec.begin()
    check(lib().tch_conv2d_dgrad(rec.ctx, F32, address(0), address(1), address(2), None, None, rows, 1, 1, cols, depth, 1, 1, 1, 0, -1, 0, 1))
    check(lib().tch_conv2d_dgrad(rec.ctx, F32, address(0), address(1), address(2), None, None, rows, 1, 1, cols, depth, 1, 1, 1, 0, -2, 0, 1))
    check(lib().tch_conv2d_fwd_bnstats(rec.ctx, F32, address(0), address(1), address(2), rows, 1, 1, depth, cols, 1, 1, 1, 0, -1, 0, address(3)))
    names = [r[0] for r in rec.end()]
    assert [n.endswith(",parts>") for n in names] == [dgrad_parts, False, False], names


@pytest.mark.parametrize("pixels,cols,tiling,parts", [(65, 1040, 2, True), (64, 1040, 2, False), (65, 1024, 2, False), (65, 2112, 0, True)])
def test_fp32_weight_gradients_in_parts(rec, pixels, cols, tiling, parts):
    rows = 2048 if tiling == 0 else 1024
    rec.begin()
    check(lib().tch_conv2d_wgrad(rec.ctx, F32, address(0), address(1), address(2), None, 1, 0, pixels, 1, 1, cols, rows, 1, 1, 1, 0, tiling, 0))
    (name, _, _), = rec.end()
    assert name.endswith(",parts>") == parts, name


def test_bf16_choice_of_16x16_tiles(rec):
    """Up to a workgroup on every compute unit, and from a reduction step for each of the eight wavefronts on."""
    assert "16x16,8way" in product(rec, BF16, 98, 256, 256, -1) and "16x16" not in product(rec, BF16, 98, 256, 192, -1)
    assert "16x16,8way" in product(rec, BF16, 256, 256, 512, -1) and "16x16" not in product(rec, BF16, 272, 256, 512, -1)


def test_bf16_choice_for_large_products_and_in_order(rec):
    """From 384 tiles of 128 x 128 on a plain product takes no smaller one; with one order of additions asked for neither a
    split tiling nor the 3x3 patch kernel runs."""
    assert ",128x128," in product(rec, BF16, 8192, 768, 768, -1) and ",128x128," in product(rec, BF16, 100352, 128, 128, -1)
    assert ",128x128," not in product(rec, BF16, 8192 - 128, 768, 768, -1)
    assert product(rec, BF16, 196, 256, 1024, -1).startswith("igemm4_kernel")
    for rows in (1, 49, 196, 1000, 8192, 300000):
        for cols, depth in ((64, 256), (256, 1024), (768, 64), (512, 96)):
            assert not product(rec, BF16, rows, cols, depth, -2).startswith(("igemm3", "igemm4"))
    for cfg, patch in ((-1, True), (-2, False)):
        rec.begin()
        check(lib().tch_conv2d_fwd(rec.ctx, BF16, address(0), address(1), address(2), None, None, None, 0, 64, 14, 14, 256, 256, 3, 3, 1, 1,
                                   cfg, 0))
        assert rec.end()[0][0].startswith("igemm3_kernel") == patch
