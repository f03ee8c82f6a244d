"""The byte offsets of masked rows, on the CPU: the arithmetic that the kernels share (row_offset.hpp) at every tile height over results just below 2 GiB, and
that the kernels ask it for the scalar offset of each row that a lane may be masked for."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "onenew_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "row_offset.hpp"
using namespace onhip;
int main() {
    for (int rows = 1; rows <= 600; ++rows)
        for (int from_limit = 1; from_limit <= 4; ++from_limit) {
            const unsigned row_bytes = (unsigned) (((1ull << 31) - 1) / rows / from_limit / 4 * 4);
            for (int row = 0; row < (rows + 255) / 256 * 256; ++row) {
                const unsigned at = row_offset(row, rows, row_bytes);
                if (row < rows && at != (unsigned) row * row_bytes) return printf("row %d of %d is at %u\n", row, rows, at), 1;
                // a masked lane of this row, and of any row whose column does not exist
                const unsigned long long sum = (unsigned long long) OOB + at;
                if (sum < RSRC_RANGE || sum >= 1ull << 32) return printf("row %d of %d, %u bytes each: %llu\n", row, rows, row_bytes, sum), 1;
            }
        }
    // images of three channels up to just below 2 GiB, rows far above and below
    for (int h : {1, 2, 10, 224, 4700, 13000})
        for (long long bytes : {4ll, 896ll, 120000ll, (long long) (((1ll << 31) - 1) / 3 / h / 4 * 4)}) {
            if (3 * h * bytes >= 1ll << 31) continue;
            for (int c = 0; c < 3; ++c)
                for (int ih = -300; ih < h + 30000; ++ih) {
                    const unsigned at = patch_row_offset(c, ih, h, (unsigned) bytes);
                    if (ih >= 0 && ih < h && at != (unsigned) ((c * h + ih) * bytes)) return printf("row %d of %d is at %u\n", ih, h, at), 1;
                    if ((unsigned long long) OOB + at >= 1ull << 32 || at >= 3ull * h * bytes) return printf("row %d of %d, %lld bytes each: %u\n", ih, h, bytes, at), 1;
                }
        }
    return 0;
}
"""


def test_masked_rows_stay_outside(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)])
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


def scalar_offsets(text):
    """(call, its scalar offset) of the buffer accesses in a source"""
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r"(raw_buffer_(?:store|load)_b\d+|buf_load_\w+)\s*\(", text):
        args, depth, start = [], 0, m.end()
        for i in range(m.end(), len(text)):
            if text[i] == "," and depth == 0 or text[i] == ")" and depth == 0:
                args.append(" ".join(text[start:i].split()))
                start = i + 1
                if text[i] == ")":
                    break
            depth += (text[i] in "([{") - (text[i] in ")]}")
        yield m.group(1), args[3 if "store" in m.group(1) else 2]


@pytest.mark.parametrize("name", ["stem.hip", "igemm_kernel.hpp", "igemm_f3_kernel.hpp"])
def test_kernels_bound_the_rows_they_mask(name):
    """no buffer access takes a product of a result's row and the bytes of one as its scalar offset"""
    offsets = list(scalar_offsets(open(os.path.join(CSRC, name)).read()))
    assert any("row_offset(" in at for _, at in offsets)
    assert name != "stem.hip" or any("patch_row_offset(" in at for _, at in offsets)
    bare = [(call, at) for call, at in offsets if re.search(r"\b(m(_uni)?|ih)\b", at) and "row_offset(" not in at and not at.endswith("* 4u")]
    assert not bare, bare
