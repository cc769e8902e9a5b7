"""Which kernel an fp32 product takes, without a GPU: the built object linked with a stand-in for the runtime (gemm_f32_dispatch.hip),
which prints what would be launched."""
import os
import subprocess
from collections import namedtuple

import pytest

from alpha2_amd import _ffi as ffi, build

HERE = os.path.dirname(os.path.abspath(__file__))
Launched = namedtuple("Launched", "code kernel slices blocks launches")


@pytest.fixture(scope="module")
def dispatch(tmp_path_factory):
    d = tmp_path_factory.mktemp("dispatch")
    subprocess.run([build._hipcc(), "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-O1", "-fPIC", "-c",
                    os.path.join(HERE, "gemm_f32_dispatch.hip"), "-o", str(d / "main.o")], check=True, capture_output=True)
    subprocess.run(["g++", str(d / "main.o"), build._compile("gemm_f32", False), "-o", str(d / "main")], check=True, capture_output=True)

    def ask(m, n, k, layout, epi=ffi.EPI_NONE, refuse=False, lda=0):
        line = "%d %d %d %d %d %d %d\n" % (m, n, k, layout, epi, refuse, lda)
        out = subprocess.run([str(d / "main")], input=line, capture_output=True, text=True, check=True).stdout
        code, kernel, slices, blocks, launches = out.rstrip("\n").split("|")
        return Launched(int(code), kernel, int(slices), int(blocks), launches.split())
    return ask


def test_a_product_whose_slices_get_no_memory_runs_without_them(dispatch):
    """64-wide and 128-wide tiles in slices, all layouts, and accumulating: the same product in one launch, nothing left allocated."""
    for m, n, k in ((384, 128, 1030), (700, 256, 4750), (640, 768, 4096)):
        for layout in (ffi.GEMM_NN, ffi.GEMM_NT, ffi.GEMM_TN):
            for epi in (ffi.EPI_NONE, ffi.EPI_ACCUM):
                sliced = dispatch(m, n, k, layout, epi)
                assert sliced.code == 0 and sliced.slices > 1 and sliced.launches[-1] == "join" and sliced.blocks == 0
                whole = dispatch(m, n, k, layout, epi, refuse=True)
                assert whole.code == 0 and whole.blocks == 0 and len(whole.launches) == 1 and whole.launches[0].endswith(",%d" % k)


def test_a_join_that_fails_to_launch_gives_the_slices_back(dispatch):
    """The residual's join is launched by the product itself."""
    for layout in (ffi.GEMM_NN, ffi.GEMM_NT, ffi.GEMM_TN):
        ok = dispatch(384, 128, 1030, layout, ffi.EPI_RESIDUAL)
        assert ok.code == 0 and ok.slices > 1 and ok.launches[-1] == "join" and ok.blocks == 0
        failed = dispatch(384, 128, 1030, layout, ffi.EPI_RESIDUAL, refuse=2)
        assert failed.code != 0 and len(failed.launches) == 2 and failed.blocks == 0


def test_slices_under_an_epilogue(dispatch):
    """A residual never changes the kernel.  gelu and its backward run in the plain product's slices where few rows meet a long contraction,
    and in one piece where those gain little (a second launch); refused memory, and zero for `nsplit` (nothing may be allocated),
    leave one piece."""
    gelu = {ffi.GEMM_NT: ffi.EPI_GELU, ffi.GEMM_NN: ffi.EPI_GELU_BWD, ffi.GEMM_TN: ffi.EPI_GELU}
    for m, n, k, as_plain in ((33, 5120, 5120, True), (64, 4096, 4096, True), (490, 8192, 2048, True), (256, 6144, 1536, True), (108, 3584, 896, True), (777, 768, 3072, True),
                              (16384, 1024, 256, True), (1, 4096, 1024, False), (65, 2688, 672, False), (88, 2048, 512, False), (912, 4096, 1024, False)):
        for layout in (ffi.GEMM_NN, ffi.GEMM_NT, ffi.GEMM_TN):
            plain = dispatch(m, n, k, layout)
            for epi in (gelu[layout], ffi.EPI_RESIDUAL):
                whole = dispatch(m, n, k, layout, epi, refuse=1)
                assert whole.code == 0 and whole.blocks == 0 and len(whole.launches) == 1
                assert dispatch(m, n, k, layout, epi, refuse=3) == whole
                got = dispatch(m, n, k, layout, epi)
                assert got in (plain, whole)
                if layout != ffi.GEMM_TN:
                    assert got == (plain if as_plain or epi == ffi.EPI_RESIDUAL else whole), (m, n, k, layout, epi)


def test_slices_are_reported_where_a_second_launch_joins_them(dispatch):
    """The waves of a 32-wide piece add up their sums inside the launch: one slice."""
    for m, n, k, layout in ((127, 260, 1000, ffi.GEMM_NN), (1, 64, 768, ffi.GEMM_NT), (500, 300, 512, ffi.GEMM_TN), (384, 128, 1030, ffi.GEMM_NN), (4000, 1200, 64, ffi.GEMM_NT)):
        got = dispatch(m, n, k, layout)
        assert (got.slices > 1) == (got.launches[-1] == "join"), got
        if "pieces" in got.kernel:
            assert got.slices == 1


def test_a_launch_stays_below_two_to_the_32_threads(dispatch):
    """Rows of more than 2^30 columns, also where the rows of A lie far apart, and 2^30 rows of one column."""
    for m, n, k, lda in ((1, 1100000000, 1, 0), (1, 2100000000, 1, 0), (1, 1100000000, 1, 1 << 22), (2, 600000000, 1, 1 << 22), (1 << 30, 1, 1, 0)):
        for layout in (ffi.GEMM_NN, ffi.GEMM_NT, ffi.GEMM_TN):
            got = dispatch(m, n, k, layout, lda=lda)
            assert got.code == 0 and all(int(x.split(",")[0]) < 1 << 32 for x in got.launches if x != "join"), (m, n, lda, layout, got)


def test_rows_that_lie_far_apart_keep_the_tiles_out(dispatch):
    """128 rows of A (or B) a tile spans: less than 4 GiB for its 32-bit offsets."""
    inside, outside = (1 << 30) // 127 - 16, (1 << 30) // 127 + 16
    assert "split" in dispatch(8200, 640, 33, ffi.GEMM_NN, lda=inside).kernel
    assert "pieces" in dispatch(8200, 640, 33, ffi.GEMM_NN, lda=outside).kernel
    assert "split" in dispatch(8200, 640, 33, ffi.GEMM_TN, lda=outside).kernel
