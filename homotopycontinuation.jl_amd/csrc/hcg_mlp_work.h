// Workspace of the training kernels (no HIP types, so that its allocation can be run on the CPU).
#pragma once
#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace hcg {

// Device workspace reused across calls (grow-only).
struct MlpWork {
    float* params = nullptr;   // HCG_MLP_NPARAMS
    float* grad = nullptr;     // HCG_MLP_NPARAMS
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    float* x = nullptr;        // cap * 8
    float* y = nullptr;        // cap * 2
    float* w = nullptr;        // cap * 2
    float* pred = nullptr;     // cap * 2
    float* loss = nullptr;     // 1
    float* part = nullptr;     // partial gradients, a row per workgroup
    int32_t* perm = nullptr;   // cap
    long cap = 0;
};

// Makes the workspace hold `n` records of `in` inputs and `out` outputs, `np` parameters and `npart` floats of
// partial gradients.  alloc(bytes) returns null when it fails; the call then returns false, and a later
// one allocates what is missing (no buffer's presence stands for another's).
template <class Alloc, class Free>
bool mlp_work_ensure(MlpWork* w, long n, size_t in, size_t out, size_t np, size_t npart, Alloc alloc, Free release) {
    auto once = [&](float*& p, size_t count) { return p || (p = (float*)alloc(sizeof(float) * count)); };
    if (!once(w->params, np) || !once(w->grad, np) || !once(w->adam_m, np) || !once(w->adam_v, np) || !once(w->loss, 1) ||
        !once(w->part, npart))
        return false;
    if (n > w->cap) {
        w->cap = 0;  // until all five are there
        for (float** p : {&w->x, &w->y, &w->w, &w->pred}) {
            if (*p) release(*p);
            *p = nullptr;
        }
        if (w->perm) release(w->perm);
        w->perm = nullptr;
        if (!once(w->x, in * n) || !once(w->y, out * n) || !once(w->w, out * n) || !once(w->pred, out * n)) return false;
        if (!(w->perm = (int32_t*)alloc(sizeof(int32_t) * n))) return false;
        w->cap = n;
    }
    return true;
}

}  // namespace hcg
