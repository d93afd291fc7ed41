"""The choice of an attention form (csrc/attention_form.hpp), host code compiled and called here."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aitemplate_amd", "csrc")
ROWS128, ROWS256, GROUPS, SMALL, ROWS64 = range(5)


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    build = tmp_path_factory.mktemp("form")
    (build / "form.cpp").write_text("""
        #include "attention_form.hpp"
        extern "C" int choose(int64_t B, int64_t M, int64_t N, int ks, int ot, int causal, int cus, int32_t* paired) {
          return aitamd::choose_form(B, M, N, ks, ot, causal != 0, cus, paired);
        }""")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, str(build / "form.cpp"), "-o", str(build / "form.so")], check=True)
    fn = ctypes.CDLL(str(build / "form.so")).choose
    fn.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] * 4 + [ctypes.POINTER(ctypes.c_int32)]

    def call(B, M, N, d, causal, cus):
        paired = ctypes.c_int32(0)
        return fn(B, M, N, (d + 15) // 16, (d + 31) // 32, causal, cus, ctypes.byref(paired)), paired.value
    return call


# (batch x heads, queries, keys, head dim, causal) on 256 CUs, around the measured lines
@pytest.mark.parametrize("case,form,paired", [
    ((12, 384, 384, 64, 0), SMALL, 0), ((66, 384, 384, 64, 0), SMALL, 0), ((67, 384, 384, 64, 0), ROWS128, 0),
    ((72, 316, 77, 128, 0), ROWS128, 0), ((992, 34, 34, 64, 0), ROWS64, 0), ((12, 2048, 2048, 64, 0), SMALL, 0),
    ((16, 2000, 2000, 128, 0), GROUPS, 0), ((16, 8192, 8192, 64, 0), ROWS256, 0), ((16, 4096, 4096, 40, 0), ROWS128, 0),
    ((64, 2048, 2048, 64, 1), ROWS128, 1), ((16, 4096, 4096, 40, 1), GROUPS, 1), ((32, 4096, 4096, 128, 1), ROWS128, 1),
    ((24, 900, 900, 64, 1), SMALL, 0)])
def test_lines_on_256_cus(choose, case, form, paired):
    assert choose(*case, 256) == (form, paired)


def test_lines_move_with_the_number_of_cus(choose):
    """An eighth of the CUs takes an eighth of the batch the same way."""
    rng = random.Random(0)
    for _ in range(3000):
        B, M, N, d, causal = rng.randint(1, 200), rng.randint(1, 5000), rng.randint(1, 5000), rng.choice([40, 64, 128]), rng.randint(0, 1)
        assert choose(B, M, N, d, causal, 32) == choose(8 * B, M, N, d, causal, 256), (B, M, N, d, causal)


@pytest.mark.parametrize("case,form,paired", [
    ((48, 28, 28, 160, 0), ROWS64, 0), ((48, 28, 28, 32, 0), ROWS64, 0), ((48, 40, 40, 32, 0), SMALL, 0),     # one tile of queries
    ((16, 285, 77, 160, 0), ROWS64, 0), ((48, 390, 77, 32, 0), ROWS128, 0), ((99, 400, 77, 64, 0), ROWS64, 0),  # few keys
    ((64, 219, 219, 160, 0), SMALL, 0), ((64, 219, 190, 160, 0), ROWS64, 0),
    ((60, 275, 275, 128, 0), ROWS128, 0), ((60, 275, 275, 80, 0), SMALL, 0),                                    # idle CUs
    ((32, 2237, 2237, 64, 1), SMALL, 0), ((276, 508, 508, 64, 1), ROWS64, 0), ((276, 520, 520, 64, 1), ROWS64, 1),
    ((248, 1781, 1781, 64, 1), ROWS128, 1), ((224, 400, 400, 40, 1), ROWS64, 0),                                # causal, narrow
    ((24, 1741, 1741, 80, 1), SMALL, 0), ((36, 3341, 3341, 80, 1), ROWS128, 1), ((96, 639, 639, 128, 1), ROWS128, 0),
    ((208, 397, 397, 80, 1), ROWS128, 1), ((164, 268, 268, 80, 1), ROWS64, 0), ((70000, 600, 600, 64, 1), ROWS64, 0),
    ((768, 256, 256, 64, 0), ROWS128, 0), ((768, 384, 384, 64, 0), ROWS128, 0), ((768, 384, 384, 32, 0), ROWS64, 0), ((64, 1268, 1268, 32, 0), SMALL, 0),
    ((64, 2209, 2209, 64, 0), ROWS128, 0), ((64, 2048, 2048, 64, 0), ROWS256, 0)])                              # full grids
def test_lines_within_a_grid_size(choose, case, form, paired):
    assert choose(*case, 256) == (form, paired)


# where the lines are drawn differently from before: us, and those of the form on the line's other side
@pytest.mark.parametrize("case,form,paired", [
    ((768, 256, 256, 64, 0), ROWS128, 0), ((768, 200, 200, 40, 0), ROWS128, 0),       # 27.0, 29.4 with 64 rows; 17.7, 20.7
    ((768, 135, 135, 64, 0), ROWS64, 0), ((192, 256, 256, 64, 0), ROWS64, 0),         # (half of 128 rows empty; few workgroups)
    ((244, 381, 381, 32, 0), ROWS128, 0),                                             # 12.7, 14.7 with 64 rows
    ((168, 748, 77, 64, 0), ROWS128, 0), ((256, 3234, 77, 40, 1), ROWS128, 0),        # 12.0, 14.2; 41.8, 47.7
    ((32, 3290, 328, 40, 1), ROWS128, 0),                                             # 17.1, 21.8 with two groups of 64 rows
    ((8, 6164, 6164, 128, 1), GROUPS, 1), ((24, 2161, 2161, 40, 1), GROUPS, 1),       # 107, 132 unpaired; 27, 36
    ((8, 2563, 2563, 160, 1), SMALL, 0), ((32, 703, 703, 160, 1), GROUPS, 0),         # 50, 58 in groups of 128 rows
    ((128, 474, 474, 40, 1), ROWS64, 0), ((96, 1154, 1154, 40, 1), ROWS128, 1),       # 12.9, 15.5 in two groups; 31.4, 33.2
    ((112, 629, 629, 32, 1), SMALL, 0), ((880, 135, 77, 64, 1), ROWS64, 0),           # 12.4, 15.9 with 64 rows; 14.7, 17.8 with 128
    ((180, 1274, 1274, 64, 1), ROWS128, 1), ((240, 993, 993, 64, 1), ROWS128, 1),     # 65.9, 73.8 with 64 rows; 58, 65
    ((156, 1143, 1143, 64, 1), ROWS64, 1), ((200, 702, 702, 64, 1), ROWS64, 1),       # 49, 57 with 128 rows; 31, 35
    ((64, 4811, 4811, 64, 0), ROWS256, 0), ((60, 3092, 3092, 64, 0), ROWS128, 0)])    # 429, 460 with 128 rows; 188, 215 with 256
def test_lines_between_forms_on_256_cus(choose, case, form, paired):
    assert choose(*case, 256) == (form, paired)


@pytest.mark.parametrize("d", [32, 40, 64, 80, 128, 160])
@pytest.mark.parametrize("M", [1, 16, 64])
def test_few_queries_over_many_keys_share_them(choose, d, M):
    """Two groups halve the chain over the keys as long as all workgroups fit the chip at once; no chain under a causal mask."""
    resident = 256 * (3 if d <= 32 else 2 if d <= 96 else 1)
    for N in (256, 1024, 4096):
        for B in (1, 8, 64, resident):
            assert choose(B, M, N, d, 0, 256) == (SMALL, 0), (B, N)
        assert choose(resident + 1, M, N, d, 0, 256) == (ROWS64, 0), N
    for N in (1, 32, 96 if d > 32 else 32, 192 if d > 96 else 32):
        assert choose(8, M, N, d, 0, 256) == (ROWS64, 0), N
    assert choose(8, M, 4096, d, 1, 256) == choose(8, M, 64, d, 1, 256) == choose(8, M, 64, d, 0, 256)


def test_pairs_are_of_causal_tiles_that_the_grid_can_hold(choose):
    rng = random.Random(1)
    for _ in range(20000):
        B, M, N = (int(2 ** rng.uniform(0, e)) for e in (17, 14, 14))
        d, causal = rng.choice([8, 32, 40, 64, 80, 96, 128, 160]), rng.randint(0, 1)
        form, paired = choose(B, M, N, d, causal, 256)
        assert form in range(5) and (not paired or (causal and B <= 65535 and form != ROWS256 and M > 128)), (B, M, N, d, causal)
