"""The verdict word of the plans' set-up checks: only a word that the checking kernel wrote, and
that no failing place marked, passes (a word read before it was written does not)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "feat3amd_check.hpp"
using namespace feat3amd_detail;
static_assert(check_passed(kCheckRan), "the check ran and nothing failed");
static_assert(!check_passed(0), "never written, or not yet read");
static_assert(!check_passed(kCheckBad), "a failing place, the mark lost");
static_assert(!check_passed(kCheckRan | kCheckBad), "a failing place");
static_assert(!check_passed(~uint32_t(0)), "other memory");
int main() { return 0; }
"""


def test_only_a_written_word_passes(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    src = tmp_path / "check.cpp"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", os.path.join(ROOT, "feat3.doxytest_amd", "csrc"), str(src)],
                   check=True)


def test_plans_read_verdicts_through_it():
    """No set-up check of the plans reads its verdict into a flag of its own that starts at 'passed'."""
    with open(os.path.join(ROOT, "feat3.doxytest_amd", "csrc", "feat3amd_kernels.hip")) as f:
        text = f.read()
    for kernel in ("k_sten_check", "k_band_check", "k_band_symmetric", "k_dict_fill_diag", "k_sell_fill_code"):
        body = text[text.index("__global__ void " + kernel):]
        body = body[:body.index("\n}\n")]
        assert "mark_checked(" in body and "kCheckBad" in body, kernel
    for flag in ("bad = 0", "unsorted = 0", "hmiss = 0", "asym = 1", "hb = 1"):
        assert flag not in text, flag
