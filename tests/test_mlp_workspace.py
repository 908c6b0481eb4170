"""Allocation of the training workspace (csrc/hcg_mlp_work.h) with an allocator that fails, on the CPU."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "homotopycontinuation.jl_amd" / "csrc"

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <set>
#include "hcg_mlp_work.h"
static long calls = 0, fail_at = -1;
static std::set<void*> live;
static void* get(size_t bytes) {
    if (calls++ == fail_at) return nullptr;
    void* p = std::calloc(bytes, 1);
    live.insert(p);
    return p;
}
static void give(void* p) {
    if (!live.erase(p)) { std::printf("freed twice\n"); std::exit(1); }
    std::free(p);
}
static bool ensure(hcg::MlpWork* w, long n) { return hcg::mlp_work_ensure(w, n, 8, 2, 4866, 5000, get, give); }
static bool whole(const hcg::MlpWork& w, long n) {
    for (void* p : {(void*)w.params, (void*)w.grad, (void*)w.adam_m, (void*)w.adam_v, (void*)w.loss, (void*)w.part, (void*)w.x,
                    (void*)w.y, (void*)w.w, (void*)w.pred, (void*)w.perm})
        if (!p || !live.count(p)) return false;
    return w.cap >= n && live.size() == 11;
}
int main() {
    for (int k = 0; k < 11; k++)            // every allocation of a first call, then of a growing one
        for (int grow = 0; grow < 2; grow++) {
            if (grow && k >= 5) continue;
            hcg::MlpWork w;
            live.clear();
            fail_at = -1;
            if (grow && !(ensure(&w, 10) && whole(w, 10))) return 1;
            calls = 0, fail_at = k;
            if (ensure(&w, 100)) { std::printf("no failure at %d\n", k); return 1; }
            for (long n : {10L, 100L, 50L}) {
                if (!ensure(&w, n) || !whole(w, n)) { std::printf("not whole after a failure at %d, n = %ld\n", k, n); return 1; }
            }
            const long before = calls;
            if (!ensure(&w, 100) || calls != before) return 1;  // kept
        }
    std::printf("ok\n");
}
"""


def test_failed_allocation_leaves_a_usable_workspace(tmp_path):
    (tmp_path / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")],
                   check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.stdout == "ok\n" and r.returncode == 0, r.stdout + r.stderr
