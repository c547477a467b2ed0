"""Status words of a chain of launches (step_status.h), on the CPU: whatever the
order in which the waves of a step run, all of them find the same status, and
the word that the host reads holds the code of the step that stopped."""
import os
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include "step_status.h"
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <random>
#include <vector>
using namespace mcmb;
int main(int argc, char** argv)
{
    const int amax = atoi(argv[1]), stop = atoi(argv[2]), code = atoi(argv[3]), waves = 48;
    std::mt19937 rng(amax + 97 * stop);
    std::vector<int> st(step_words(amax), STEP_RUNNING);
    for (int a = 0; a <= amax; ++a) {
        // wave 0 stores; the others may look before or after it
        std::vector<int> order(waves);
        std::iota(order.begin(), order.end(), 0);
        std::shuffle(order.begin(), order.end(), rng);
        std::vector<int> seen;
        for (int w : order) {
            const int s = step_status(st.data(), a);
            seen.push_back(s);
            if (w != 0) continue;
            if (s != STEP_RUNNING) step_stop(st.data(), a, s);
            else if (a == stop) step_stop(st.data(), a, code);
        }
        for (int s : seen)
            if (s != seen[0] || (s == STEP_RUNNING) != (a <= stop)) return printf("step %d: %d\n", a, s), 1;
    }
    for (int a = 0; a <= amax + 1; ++a)
        if (st[a] != (a <= stop ? STEP_RUNNING : code)) return printf("word %d: %d\n", a, st[a]), 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def chain(tmp_path_factory):
    d = tmp_path_factory.mktemp("step_status")
    (d / "chain.cpp").write_text("#include <algorithm>\n" + SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "modal-cmb_amd", "csrc"), "-o", str(d / "chain"), str(d / "chain.cpp")],
                   check=True, timeout=120)
    return str(d / "chain")


@pytest.mark.parametrize("amax,stop,code", [(0, 0, 0), (1, 1, -2), (14, 0, 0), (14, 13, 13), (14, 14, -2), (264, 63, 63),
                                            (264, 264, -2)])
def test_every_wave_of_a_step_agrees(chain, amax, stop, code):
    r = subprocess.run([chain, str(amax), str(stop), str(code)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
