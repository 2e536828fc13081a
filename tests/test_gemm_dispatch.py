"""Which kernel the grouped GEMMs take, asked of the rules themselves (no GPU needed: they are host code)."""
import os
import shutil
import subprocess

import pytest

from memfabric_hybrid_amd import build

HIPCC = os.path.join(build.ROCM, "bin", "hipcc")

PROGRAM = r"""
#include <cstdio>
#include <hip/hip_runtime.h>
#include <type_traits>
#include "zbal_gemm_stream.h"
#include "zbal_gemm_tall.h"

template <int MODE, bool GMM1, int SPLIT> long workgroups(GemmParams p, int n_tiles, bool parts)
{
    static float sums;
    p.part_sums = parts ? &sums : nullptr;
    p.part_cus = 32;
    return stream_workgroups<MODE, GMM1, SPLIT == 2 ? 16 : 64, SPLIT>(p, n_tiles);
}
template <int MODE, bool GMM1, int SPLIT> long beyond(const GemmParams &p, int n_tiles)
{
    return workgroups<MODE, GMM1, SPLIT>(p, n_tiles, true) - workgroups<MODE, GMM1, SPLIT>(p, n_tiles, false);
}
template <int MODE> long beyond(int gmm1, int split, const GemmParams &p, int n_tiles)
{
    if (gmm1) return split == 1 ? beyond<MODE, true, 1>(p, n_tiles) : beyond<MODE, true, 2>(p, n_tiles);
    return split == 1 ? beyond<MODE, false, 1>(p, n_tiles) : beyond<MODE, false, 2>(p, n_tiles);
}
long beyond(int mode, int gmm1, int split, int experts, int rows, int n_tiles)
{
    GemmParams p = {};
    p.experts = experts;
    p.max_rows = rows;
    const long n = mode == MODE_W8A8 ? beyond<MODE_W8A8>(gmm1, split, p, n_tiles)
                 : mode == MODE_FP8 ? beyond<MODE_FP8>(gmm1, split, p, n_tiles) : beyond<MODE_W4A8>(gmm1, split, p, n_tiles);
    if (n != 0 && n != 256) exit(1);
    return n;
}

int main()
{
    int mode, slabs, experts, rows;
    while (scanf("%d %d %d %d", &mode, &slabs, &experts, &rows) == 4) {
        if (mode >= 10) {                      /* mode - 10: whether memory for shared tiles adds workgroups to a launch of the weight stream */
            int gmm1, split, n_tiles;
            if (scanf("%d %d %d", &gmm1, &split, &n_tiles) != 3) return 1;
            printf("%d\n", beyond(mode - 10, gmm1, split, experts, rows, n_tiles) == 256);
            continue;
        }
        if (mode == MODE_W4A8) {
            int n_tiles, cus;
            if (scanf("%d %d", &n_tiles, &cus) != 2) return 1;
            printf("%d\n", w4a8_taller_tile(rows, experts, n_tiles, cus));
            continue;
        }
        GemmParams p = {};
        p.K = slabs * 128;
        p.experts = experts;
        p.max_rows = rows;
        printf("%d\n", mode == MODE_FP8 ? tall_accepts<MODE_FP8>(p) : tall_accepts<MODE_W8A8>(p));
    }
}
"""


@pytest.fixture(scope="module")
def accepts(tmp_path_factory):
    if not (os.path.exists(HIPCC) or shutil.which("hipcc")):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("dispatch")
    (d / "accepts.hip").write_text(PROGRAM)
    cmd = [HIPCC] + build.HIP_FLAGS + build.INCLUDES + [str(d / "accepts.hip"), "-o", str(d / "accepts")]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout

    def ask(cases):
        out = subprocess.run([str(d / "accepts")], input="".join(" ".join(map(str, c)) + "\n" for c in cases), capture_output=True, text=True)
        assert out.returncode == 0, out.stderr
        return [v == "1" for v in out.stdout.split()]
    return ask


@pytest.mark.parametrize("mode", [1, 2])
def test_the_many_row_kernel_takes_every_k(accepts, mode):
    """Two to 256 steps of 128 (the entry points take no more), at any number of experts that its tables hold."""
    cases = [(mode, kb, e, 256 * e) for kb in range(2, 257) for e in (2, 32, 512)]
    got = accepts(cases)
    assert len(got) == len(cases) and all(got), [c for c, ok in zip(cases, got) if not ok][:5]


def test_the_many_row_kernel_refuses_what_it_has_no_room_for(accepts):
    # a single step; more experts than the tables hold; fp8 rows of two or three scales where one tile has all rows
    refused = [(1, 1, 8, 4096), (2, 1, 8, 4096), (1, 8, 513, 1 << 20), (2, 8, 513, 1 << 20), (2, 2, 1, 320), (2, 3, 1, 320)]
    taken = [(1, 2, 1, 320), (2, 2, 1, 321), (2, 3, 1, 321), (2, 4, 1, 320)]
    assert accepts(refused + taken) == [False] * len(refused) + [True] * len(taken)


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_the_taller_w4a8_tile_wants_a_full_chip(accepts, cus):
    """rows * channel tiles from 500 per CU on, from 256 with more than 640 rows per expert; none up to 112 rows. Unknown: as on a whole GPU."""
    case = lambda rows, experts, n_tiles, cus=cus: (3, 4, experts, rows, n_tiles, cus)
    low = [case(112 * 64, 64, 1000), case(500 * 8, 8, cus // 8 - 1), case(640 * 8, 8, (500 * cus - 1) // 5120), case(641 * 8, 8, 256 * cus // 5128),
           case(256 * cus - 1, 1, 1)]
    tall = [case(113 * 64, 64, 1000), case(500 * 8, 8, cus // 8), case(640 * 8, 8, (500 * cus - 1) // 5120 + 1), case(641 * 8, 8, 256 * cus // 5128 + 1),
            case(256 * cus, 1, 1)]
    assert accepts(low + tall) == [False] * len(low) + [True] * len(tall)
    if cus == 256:
        assert accepts([c[:5] + (0,) for c in low + tall]) == [False] * len(low) + [True] * len(tall)


@pytest.mark.parametrize("mode", [1, 2, 3])
def test_workgroups_for_shared_tiles_only_where_tiles_are_shared(accepts, mode):
    """Memory for shared tiles adds a workgroup per CU to W8A8's first GEMM with whole tiles, and none to any other launch: a token or two's
    (two workgroups per tile), the second GEMM's, the other modes'."""
    shapes = [(33, 8), (33, 264), (1, 1), (300, 5000)]
    for gmm1 in (1, 0):
        for split in (1, 2):
            got = accepts([(10 + mode, 56, e, r, gmm1, split, n) for e, r in shapes for n in (1, 8, 16)])
            assert got == [mode == 1 and gmm1 == 1 and split == 1] * len(got), (gmm1, split)
