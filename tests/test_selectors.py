"""CPU: how many row selectors the single launch gets (csrc/selectors.h, compiled with g++)."""

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "vllm-ascend-hust-diffspec_amd" / "csrc"
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "selectors.h"
int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3)
    std::printf("%d\n", ds355::row_selectors(std::atoi(argv[i]), std::atoll(argv[i + 1]), std::atoi(argv[i + 2])));
}
"""


@pytest.fixture(scope="module")
def selectors(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    build = tmp_path_factory.mktemp("selectors")
    (build / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), str(build / "main.cpp"), "-o", str(build / "main")], check=True)

    def run(*cases):
        flat = [str(x) for case in cases for x in case]
        out = subprocess.run([str(build / "main"), *flat], check=True, capture_output=True, text=True).stdout
        return [int(x) for x in out.split()]

    return run


def test_short_rows_get_more_selectors_and_long_rows_eight(selectors):
    keys = lambda rows, tokens, hkv, dim: rows * tokens * hkv * dim * 2  # noqa: E731
    assert selectors((36, keys(36, 1700, 2, 64), 256), (11, keys(11, 1600, 2, 64), 256),
                     (16, keys(16, 40960, 4, 128), 256), (64, keys(64, 40960, 4, 128), 256),
                     (200, 1, 256), (5, 1, 256), (9, 0, 256)) == [36, 11, 8, 8, 64, 5, 9]


def test_selectors_are_a_small_share_of_any_device(selectors):
    """Of the 3 resident workgroups per CU at least eleven twelfths score, whatever the rows (a
    device with fewer than 32 CUs keeps 8), and the count shrinks with the device."""
    rows, key_bytes = [1, 8, 9, 64, 256], [0, 1, 1 << 20, 1 << 24, 1 << 30, 1 << 40]
    last = None
    for cus in (304, 256, 128, 64, 38, 32, 16, 4):
        got = selectors(*[(r, b, cus) for r in rows for b in key_bytes])
        for r, n in zip([r for r in rows for _ in key_bytes], got):
            assert min(r, 8) <= n <= min(r, max(8, 3 * cus // 12))
        if last is not None:
            assert all(a <= b for a, b in zip(got, last))
        last = got
