"""The rules by which calls choose among kernels and builds that compute the same (csrc/routes.h), on the CPU: at the
sizes where each was measured to be the faster one, the rule takes it."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    """routes(expression, ...): the values of C++ expressions over routes.h, as ints."""
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host compiler")
    tmp = tmp_path_factory.mktemp("routes")

    def run(*exprs):
        src, exe = tmp / "r.cpp", tmp / "r"
        body = "".join(f'  printf("%ld\\n", (long)({e}));\n' for e in exprs)
        src.write_text('#include <stdio.h>\n#include "routes.h"\nusing namespace ffa;\nint main() {\n' + body + "}\n")
        subprocess.run([cxx, "-std=c++17", f"-I{ROOT / 'ffa-speedtest_amd' / 'csrc'}", str(src), "-o", str(exe)], check=True)
        return [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]

    return run


def test_four_bit_appends(routes):
    """Whole pages for few (sequence, head, page) blocks and for many tokens of each; the per-token kernel for a few
    tokens of many sequences."""
    nf4, nvfp4 = "true", "false"
    whole = [(f, B, Tn, H) for f in (nf4, nvfp4) for B, Tn, H in
             ((1, 1, 1), (64, 1, 8), (1, 4, 8), (1, 16384, 8), (4, 100, 4), (1024, 32, 1), (2048, 64, 16), (1, 2 ** 31 - 1, 8))]
    whole += [(nvfp4, 1024, 1, 1), (nvfp4, 64, 4, 8), (nvfp4, 256, 16, 8), (nvfp4, 65536, 32, 64)]
    tokens = [(f, B, Tn, H) for f in (nf4, nvfp4) for B, Tn, H in
              ((2048, 2, 4), (512, 2, 16), (1024, 1, 4), (1024, 8, 2), (2048, 16, 1), (65535, 1, 1024))]
    tokens += [(nf4, 256, 1, 8), (nf4, 512, 8, 8)]
    got = routes(*(f"k4_whole_pages({f}, {B}, {Tn}, {H})" for f, B, Tn, H in whole + tokens))
    assert got == [1] * len(whole) + [0] * len(tokens)


def test_two_bit_appends(routes):
    """Whole pages from about 4600 rows (tokens x heads) on, of 32 tokens a sequence or more."""
    whole = [(1, 16384, 8), (1, 1024, 8), (2, 3000, 4), (144, 32, 1), (1, 8192, 1), (1, 2 ** 31 - 1, 64)]
    tokens = [(1, 1024, 1), (40, 33, 1), (4, 64, 16), (1, 512, 8), (64, 1, 8), (4096, 31, 8), (65535, 1, 64)]
    got = routes(*(f"q2_whole_pages({B}, {Tn}, {H})" for B, Tn, H in whole + tokens))
    assert got == [1] * len(whole) + [0] * len(tokens)


def test_projection_tiles(routes):
    """Each tile, and the split kernel, where it was measured to be the fastest (256 CUs)."""
    want = {"kKprojSplit": [(64, 1024), (128, 1024), (4096, 32), (4100, 32), (100, 2048), (128, 2048), (1, 32), (16, 8192)],
            "kKproj32x64": [(32, 8192), (64, 4096), (256, 1024), (512, 1024), (4096, 64), (5200, 32), (2048, 128)],
            "kKproj64x64": [(1024, 1024), (1100, 1024)],
            "kKproj128x64": [(2048, 1024), (2100, 1024), (4100, 1024), (4224, 1024), (5200, 1024), (8200, 1024)],
            "kKproj128x128": [(4096, 1024), (4096 + 128 * 17, 1024), (8192, 1024), (12000, 384), (1 << 22, 1024)]}
    for tile, sizes in want.items():
        assert routes(*(f"kproj_route({M}, {N}, 256) == {tile}" for M, N in sizes)) == [1] * len(sizes), tile


def test_nvfp4_vectors(routes):
    """Vectors of 8 channels for pages of more than 256 values."""
    vectors, scalar = [(128, 128), (8, 33), (24, 16), (8, 2 ** 31 - 1)], [(8, 16), (16, 16), (128, 2), (12, 128), (1, 1000)]
    got = routes(*(f"nvfp4_by_vectors({D}, {page})" for D, page in vectors + scalar))
    assert got == [1] * len(vectors) + [0] * len(scalar)


def test_decode_of_several_quads(routes):
    """Quads of a KV head share its data with 8 or 16 heads or one, and in grids of more than 2.5 workgroups a CU."""
    share = [(2, 8, 128), (4, 16, 10000), (2, 1, 64), (4, 1, 2000), (2, 4, 784), (2, 3, 672), (2, 2, 641)]
    apart = [(1, 8, 100000), (1, 1, 10), (2, 4, 256), (2, 4, 576), (2, 2, 256), (2, 3, 384), (4, 6, 640)]
    got = routes(*(f"quads_share({nq}, {H}, {n}, 256)" for nq, H, n in share + apart))
    assert got == [1] * len(share) + [0] * len(apart)


def test_contiguous_decode_of_many_workgroups(routes):
    """Three workgroups a CU: several quads from more than two a CU on, one quad from more than five where the threshold
    lies near the maximum."""
    three = [(2, 513, 5.0), (4, 100000, 1000.0), (1, 1281, 5.0), (1, 8520, 0.0)]
    two = [(2, 512, 5.0), (1, 1280, 5.0), (1, 944, 5.0), (1, 8520, 8.0), (1, 8520, 1000.0)]
    got = routes(*(f"three_per_cu({nq}, {n}, 256, {d}f)" for nq, n, d in three + two))
    assert got == [1] * len(three) + [0] * len(two)
