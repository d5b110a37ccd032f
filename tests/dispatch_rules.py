"""The rules by which the library chooses a kernel, compiled from its own source (dscuda_amd/csrc/index_math.h), so that a
test can state which kernels it runs.  Decode forms: 0 is 128 rows per workgroup, 1 is 32, 2 is 64."""

import ctypes
import functools
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "dscuda_amd" / "csrc"
SOURCE = """#include "index_math.h"
using namespace dscuda::index_math;
extern "C" int call_rows(int batch, int heads, int splits, int page_size, int compute_units) {
    return decode_form_of_call(batch, heads, splits, page_size, compute_units, 512).row_blocks;
}
extern "C" int plan_rows(int batch, int heads, int splits, int compute_units) {
    return decode_form(batch, heads, splits, compute_units, 512).row_blocks;
}
extern "C" int backward_ranges(int batch, int tokens, int heads, int compute_units) {
    const KeyVisits visits = key_visits(tokens, heads);
    return (int)key_gradient_ranges(visits.per_batch() * batch, (long long)visits.key_blocks * batch, visits.row_tiles,
                                    (long long)tokens * heads * batch * 1024, compute_units);
}
extern "C" int walks_are_cut(int pairs, int tokens, int sharing) {
    return choose_walk_cut(pairs, (tokens + 127) / 128, (tokens + 63) / 64, sharing, 256).part_steps > 0;
}
extern "C" long long workspace_slots(int batch, int tokens, int heads) {   // of a call whose dS is kept, in bytes
    return kept_cut(tokens, heads, batch, slot_bytes_of_workspace(tokens, heads, batch), 256).slot_bytes;
}
extern "C" int forward_rows(int batch, int tokens, int heads, int compute_units) {   // of a workgroup, absorbed prefill forward
    const int blocks = forward_row_blocks(tokens, heads, batch, compute_units);
    return blocks == 0 ? 128 : 32 * blocks;
}
extern "C" int keeps_scores(int batch, int tokens, int heads) { return short_backward(batch, tokens, heads); }
"""


@functools.lru_cache(maxsize=None)
def rules():
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    directory = Path(tempfile.mkdtemp())
    (directory / "rules.cpp").write_text(SOURCE)
    subprocess.run([compiler, "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(directory / "rules.cpp"), "-o",
                    str(directory / "rules.so")], check=True, timeout=120)
    library = ctypes.CDLL(str(directory / "rules.so"))
    library.workspace_slots.restype = ctypes.c_longlong
    return library
