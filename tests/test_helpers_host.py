"""Helper threads of the staged copies where memory or threads run out: those
that could be started work and are joined, and nothing is thrown."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcmurchie-davidson_amd", "csrc")

PROGRAM = r"""
#include <atomic>
#include <cstdlib>
#include <new>
#include <system_error>
#include "mmd_helpers.h"

static std::atomic<int> left{1 << 30};   // allocations until memory runs out
static bool threads_out = false;

void* operator new(std::size_t n)
{
    if (left.fetch_sub(1) <= 0) {
        left = 1 << 30;   // the exception's own
        if (threads_out) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
        throw std::bad_alloc();
    }
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main()
{
    for (int mode = 0; mode < 2; ++mode)
        for (int allowed = 0; allowed <= mmd::helper_count(); ++allowed) {
            std::atomic<int> ran{0};
            threads_out = mode == 1;
            left = allowed;   // a thread allocates its state
            mmd::Helpers h([&] { ++ran; });
            left = 1 << 30;
            const int n = h.n;
            h.join();
            if (n != allowed || ran != allowed) return 1;
        }
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_helpers_without_memory_or_threads(tmp_path):
    src, exe = tmp_path / "helpers.cpp", tmp_path / "helpers"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe), "-pthread"], check=True)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
