"""Index arithmetic of the grouped kernels at the largest blocks the library
accepts (2^31 - 1 elements): the helpers the kernels use, compiled for the host
and compared with exact integers.  A rank-1 complex64 block of such a length
would need 16 GiB per operand to reach the same indexes on a device."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
TOP = 2 ** 31 - 1

SOURCE = r"""
#include <cstdio>
#include "qlt_internal.h"
int main() {
  long k, x;
  while (std::scanf("%ld %ld", &k, &x) == 2)
    std::printf("%lld %lld %d\n", static_cast<long long>(qlt::run_offset(static_cast<int32_t>(k), 1)),
                static_cast<long long>(qlt::run_offset(static_cast<int32_t>(k), 2)),
                qlt::chunks_from(static_cast<int32_t>(k), static_cast<int32_t>(x)));
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_offsets_and_chunk_counts_up_to_the_largest_block(tmp_path):
    src, exe = tmp_path / "index.cc", tmp_path / "index"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'tensortoolkit_amd' / 'csrc'}", str(src), "-o", str(exe)], check=True)
    pairs = [(k, x) for x in (1, 15, 16, 17, 31, 33, 1000, 2 ** 30 - 1, 2 ** 30 + 1, TOP - 16, TOP - 1, TOP)
             for k in (0, 1, 15, 16, 17, 2 ** 30 - 4, 2 ** 30, TOP - 17, TOP - 1) if k < x]
    out = subprocess.run([str(exe)], input="\n".join(f"{k} {x}" for k, x in pairs), text=True, capture_output=True,
                         check=True).stdout.split("\n")
    assert len(out) - 1 == len(pairs)
    for (k, x), line in zip(pairs, out):
        one, two, chunks = map(int, line.split())
        assert one == k
        assert two == 2 * k
        assert chunks == -(-(x - k) // 16)
