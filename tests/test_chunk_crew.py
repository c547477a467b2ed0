"""The host threads of a staged copy (chunk_crew.h), on the CPU: every byte of
every chunk is moved once through a ring of slots, and threads that wait for a
chunk that is long in coming do not burn their cores."""
import os
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include "chunk_crew.h"
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <ctime>
#include <vector>
using namespace mcmb;
static double cpu()
{
    timespec t;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
    return t.tv_sec + 1e-9 * t.tv_nsec;
}
int main(int argc, char** argv)
{
    const size_t bytes = atol(argv[1]), slot = atol(argv[2]), slots = atol(argv[3]);
    const int nth = atoi(argv[4]), late = atoi(argv[5]);   // ms that the first chunk comes late
    const size_t nk = (bytes + slot - 1) / slot;
    std::vector<unsigned char> src(bytes), dst(bytes, 0), ring(slot * slots);
    for (size_t i = 0; i < bytes; ++i) src[i] = (unsigned char)(i * 2654435761u >> 13);
    auto len = [&](size_t k) { return std::min(slot, bytes - k * slot); };
    double spent = 0.0;
    {
        ChunkCrew crew(nth, nk, [&](int t, size_t k) {
            const size_t a = len(k) * t / nth, b = len(k) * (t + 1) / nth;
            memcpy(dst.data() + k * slot + a, ring.data() + (k % slots) * slot + a, b - a);
        });
        for (size_t k = 0; k < nk; ++k) {
            if (k >= slots) crew.wait(k - slots);
            if (k == 0 && late) {
                const double c0 = cpu();
                std::this_thread::sleep_for(std::chrono::milliseconds(late));
                spent = cpu() - c0;
            }
            memcpy(ring.data() + (k % slots) * slot, src.data() + k * slot, len(k));
            crew.ready.store((long)k + 1, std::memory_order_release);
        }
        crew.wait(nk - 1);
    }
    if (memcmp(src.data(), dst.data(), bytes)) return printf("bytes differ\n"), 1;
    // eight threads yield for 2 ms and then wake once a ms, for less than 50 us
    // (0.2 s in 500 ms at most); spinning takes a core each (4 s)
    if (late && spent > nth * (2e-3 + 50e-6 * late)) return printf("%g s of CPU time in a wait of %d ms\n", spent, late), 1;
    {   // given up half-way: the threads end
        ChunkCrew crew(nth, nk, [](int, size_t) {});
        crew.ready.store((long)(nk / 2));
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def crew(tmp_path_factory):
    d = tmp_path_factory.mktemp("chunk_crew")
    (d / "crew.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I",
                    os.path.join(ROOT, "modal-cmb_amd", "csrc"), "-o", str(d / "crew"), str(d / "crew.cpp")],
                   check=True, timeout=120)
    return str(d / "crew")


# one byte, one chunk, fewer chunks than slots, as many, a short last chunk, one thread
@pytest.mark.parametrize("nbytes,slot,slots,nth", [(1, 4096, 4, 8), (4096, 4096, 4, 8), (3 * 4096, 4096, 8, 8),
                                                   (8 * 4096, 4096, 8, 8), (100 * 4096 + 7, 4096, 4, 8),
                                                   (100 * 4096 - 1, 4096, 8, 3), (50 * 4096 + 1, 4096, 4, 1)])
def test_every_chunk_is_moved(crew, nbytes, slot, slots, nth):
    r = subprocess.run([crew, str(nbytes), str(slot), str(slots), str(nth), "0"], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout


def test_waiting_threads_sleep(crew):
    r = subprocess.run([crew, str(9 * 4096), "4096", "4", "8", "500"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
