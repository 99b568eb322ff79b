"""The round flag of the several-wave Jacobi kernels (csrc/round_flag.h, the code the kernels run, compiled
for the host): every interleaving of wave 0 and a late wave between barriers, for every pattern of rounds with and
without a rotation, gives both waves the flag of their own round."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MODEL = r"""
#include <cstdio>
#include <initializer_list>
#include "round_flag.h"
struct ByParity {  // a word per parity of the round within its sweep
    int r = 0, rounds = 0;
    void put(int* w, int v) const { w[r & 1] = v; }
    int take(const int* w) { const int v = w[r & 1]; r = (r + 1) % rounds; return v; }
};
template <class F> struct Wave {
    F flag;
    int sweep = 0, round = 0, step = 0;  // step: 0 put, 1 barrier, 2 take, 3 barrier of a rotation, 4 done
    bool swept = false;
};
struct Pattern { int sweeps, rounds; unsigned bits; bool at(int s, int r) const { return bits >> (s * rounds + r) & 1; } };
template <class F> void advance(Wave<F>& w, const Pattern& p) {
    w.step = 0;
    if (++w.round < p.rounds) return;
    w.round = 0;
    if (!w.swept || ++w.sweep == p.sweeps) w.step = 4;
    w.swept = false;
}
template <class F> bool wrong(Wave<F> w0, Wave<F> w1, int a, int b, const Pattern& p) {
    int words[2] = {a, b};
    auto at_barrier = [](const Wave<F>& w) { return w.step == 1 || w.step == 3; };
    if (w0.step == 4 && w1.step == 4) return false;
    if (at_barrier(w0) && at_barrier(w1)) {
        if (w0.step != w1.step) return true;
        for (Wave<F>* w : {&w0, &w1}) if (w->step == 1) w->step = 2; else advance(*w, p);
        return wrong(w0, w1, a, b, p);
    }
    if ((at_barrier(w0) || w0.step == 4) && (at_barrier(w1) || w1.step == 4)) return true;
    for (int i = 0; i < 2; ++i) {  // either wave goes on
        Wave<F> v[2] = {w0, w1};
        Wave<F>& w = v[i];
        if (at_barrier(w) || w.step == 4) continue;
        int m[2] = {words[0], words[1]};
        if (w.step == 0) {
            if (i == 0) w.flag.put(m, p.at(w.sweep, w.round));
            w.step = 1;
        } else {
            const bool any = w.flag.take(m) != 0;
            if (any != p.at(w.sweep, w.round)) return true;
            if (any) { w.swept = true; w.step = 3; } else advance(w, p);
        }
        if (wrong(v[0], v[1], m[0], m[1], p)) return true;
    }
    return false;
}
int main() {
    int bad = 0, bad_parity = 0;
    for (int rounds : {1, 3}) {
        const int sweeps = rounds == 1 ? 4 : 2;
        for (unsigned bits = 0; bits < 1u << (sweeps * rounds); ++bits) {
            const Pattern p{sweeps, rounds, bits};
            bad += wrong(Wave<RoundFlag>{}, Wave<RoundFlag>{}, 0, 0, p);
            Wave<ByParity> w;
            w.flag.rounds = rounds;
            bad_parity += wrong(w, w, 0, 0, p);
        }
    }
    std::printf("%d %d\n", bad, bad_parity);
}
"""


def test_round_flag(tmp_path):
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(MODEL)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "wannier-berri_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    bad, bad_parity = (int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    assert bad == 0
    assert bad_parity > 0   # the model sees a word used twice running


@pytest.mark.parametrize("kernel", ["k_eigh_jacobi_b", "k_eigh_jacobi_reg"])
def test_kernels_use_it(kernel):
    text = open(os.path.join(ROOT, "wannier-berri_amd", "csrc", "eigh.hip")).read()
    body = text[text.index(f" {kernel}("):]
    body = body[:body.index("\n}\n")]
    assert "flag.put(flags, w)" in body and "flag.take(flags)" in body and "flags[" not in body
