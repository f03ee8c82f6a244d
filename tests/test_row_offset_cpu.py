"""The byte offsets of masked rows, on the CPU: the arithmetic that the kernels share (row_offset.hpp) at every tile height over results just below 2 GiB, when a
first-layer convolution needs its variant for large planes, and that the kernels ask about each row that a lane may be masked for."""
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
// what a masked lane asks for has to stay outside, whether the range check adds in 32 bits or in more
static bool outside(unsigned long long masked) { return masked >= RSRC_RANGE && masked < 1ull << 32; }
int main() {
    for (int rows = 1; rows <= 600; ++rows)
        for (int from_limit = 1; from_limit <= 4; ++from_limit) {
            const unsigned row_bytes = (unsigned) (((1ull << 31) - 1) / rows / from_limit / 4 * 4);
            for (int row = 0; row < (rows + 255) / 256 * 256; ++row) {
                const unsigned at = row_offset(row, rows, row_bytes);
                if (row < rows && at != (unsigned) row * row_bytes) return printf("row %d of %d is at %u\n", row, rows, at), 1;
                // a masked lane of this row, and of any row whose column does not exist
                if (!outside((unsigned long long) OOB + at)) return printf("row %d of %d, %u bytes each: %u\n", row, rows, row_bytes, at), 1;
                if (row_there<true>(row, rows) != (row < rows) || !row_there<false>(row, rows)) return printf("row %d of %d\n", row, rows), 1;
                if (row_there<true>(row, rows) && !outside((unsigned long long) OOB + (unsigned long long) row * row_bytes)) return 1;
            }
        }
    // images of three channels up to just below 2 GiB, rows far above and below
    for (int h : {1, 2, 10, 224, 4700, 13000})
        for (long long w : {1ll, 224ll, 30000ll, (long long) (((1ll << 31) - 1) / 3 / h / 4)}) {
            if (3 * h * w * 4 >= 1ll << 31) continue;
            for (int pad : {0, 1, 3, 300})
                for (int last : {h + 2, h + 300, h + 30000})
                    for (int rows : {32, 64})
                        for (long long plane : {1ll, 4700ll * 4700, (long long) ((1ll << 31) / 4 / rows) - 1, (long long) ((1ll << 31) / 4 / rows)}) {
                            const bool far = far_rows(h, w, pad, last, rows, plane);
                            for (int c = 0; c < 3; ++c)
                                for (int ih = -pad; ih <= last; ++ih) {
                                    const unsigned own = (unsigned) ((c * h + ih) * w) * 4u, near = patch_row_offset(c, ih, h, (unsigned) (w * 4));
                                    const bool in = ih >= 0 && ih < h;
                                    if (in && near != own) return printf("row %d of %d is at %u\n", ih, h, near), 1;
                                    if (!outside((unsigned long long) OOB + near) || near >= 3ull * h * w * 4) return printf("row %d of %d x %lld: %u\n", ih, h, w, near), 1;
                                    // without the bounds: as it wraps, and as it does not, beyond the image
                                    const long long place = ((long long) c * h + ih) * w * 4;
                                    if (!far && !in && (OOB + own < 3ull * h * w * 4 || (long long) OOB + place < 3 * h * w * 4 || (long long) OOB + place >= 1ll << 32))
                                        return printf("row %d of %d x %lld, padding %d: %lld\n", ih, h, w, pad, place), 1;
                                }
                            if (!far && !outside((unsigned long long) OOB + (rows - 1) * plane * 4)) return printf("%d rows of %lld\n", rows, plane), 1;
                        }
        }
    // layers as networks have them do not
    if (far_rows(224, 224, 3, 229, 64, 112 * 112) || far_rows(640, 640, 1, 641, 32, 320 * 320) || far_rows(2160, 3840, 3, 2165, 64, 1080 * 1920)) return printf("small planes\n"), 1;
    if (!far_rows(4700, 4700, 1, 4701, 32, 4700ll * 4700) || !far_rows(10, 30000, 1, 20010, 32, 100)) return printf("large planes\n"), 1;
    return 0;
}
"""


def test_masked_rows_stay_outside(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)])
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


def accesses(text):
    """(place in the text, call, its scalar offset) of the buffer accesses in a source"""
    for m in re.finditer(r"(raw_buffer_(?:store|load)_b\d+|buf_load_\w+)\s*\(", text):
        args, depth, start = [], 0, m.end()
        for i in range(m.end(), len(text)):
            if text[i] == "," and depth == 0 or text[i] == ")" and depth == 0:
                args.append(" ".join(text[start:i].split()))
                start = i + 1
                if text[i] == ")":
                    break
            depth += (text[i] in "([{") - (text[i] in ")]}")
        yield m.start(), m.group(1), args[3 if "store" in m.group(1) else 2]


@pytest.mark.parametrize("name", ["stem.hip", "igemm_kernel.hpp", "igemm_f3_kernel.hpp"])
def test_kernels_bound_the_rows_they_mask(name):
    """no buffer access takes a product of a row and the bytes of one as its scalar offset but where the row has been asked about, or the place is bounded"""
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())
    asked, bare = 0, []
    for at, call, offset in accesses(text):
        if offset == "soff":   # the row's place under another name: what it stands for
            named = re.findall(r"\bsoff = ([^,;]*)[,;]", text[:at])
            offset = named[-1] if named else offset
        if not re.search(r"\b(m(_uni)?|ih)\b", offset) or offset.endswith("* 4u") and "row" not in offset and "width" not in offset and "ih" not in offset:
            continue
        # since the row got its name
        since = max(text.rfind(decl, 0, at) for decl in ("const int m_uni =", "const int m =", "const int ih =", "int m_uni, auto edge"))
        if "row_offset(" in offset or "row_there<" in text[since:at]:
            asked += 1
        else:
            bare.append((call, offset))
    assert asked and not bare, bare
