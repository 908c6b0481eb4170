// Training kernels of the learned step-size proposer (8 -> 64 -> 64 GELU -> 2).
//
// Forward uses BF16-rounded copies of the FP32 master weights (round to nearest even)
// with FP32 accumulation; gradients flow to the master weights unchanged (straight-
// through).  Loss per record: w0 * (o0 - y0)^2 / 2 + w1 * BCEWithLogits(o1, y1),
// averaged over the batch.
//
// mlp_tile: one workgroup of four waves takes tiles of 32 records through forward and backward.  The
// products over the hidden layers run on the FP32 matrix cores (v_mfma_f32_16x16x4: FP32
// operands and sums, so no precision is given up for them), activations and weights staged in
// LDS with rows of 68 floats, which the operand reads along rows cross without bank conflicts (the transposed
// ones, of da2, h1 and w2 in the backward products, put up to four addresses on a bank).  GELU and
// its derivative are computed once per activation, the derivative kept in the registers of the
// lane that needs it.  Each workgroup writes its partial gradient; grad_step adds the partials in a
// fixed order and, in training, makes the Adam step in the same launch.  A batch of 4,096 is 128
// tiles: half the CUs, bound by the latency of a tile's chain of products.  Measured (200,003 records,
// one epoch of batches of 4,096, the whole call): 39.5 -> 1.8 ms; the vector kernel it replaces took
// 787 us a batch, mostly recomputing GELU for every product and adding gradients with atomics.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <numeric>
#include <random>
#include <vector>

#include "hcg_mlp.h"

namespace {

constexpr int IN = HCG_MLP_IN, H = HCG_MLP_HIDDEN, OUT = HCG_MLP_OUT;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + H * IN, OFF_W2 = OFF_B1 + H, OFF_B2 = OFF_W2 + H * H,
              OFF_W3 = OFF_B2 + H, OFF_B3 = OFF_W3 + OUT * H, NP = OFF_B3 + OUT;
static_assert(NP == HCG_MLP_NPARAMS, "parameter layout");
constexpr int R = 32;        // records per tile
constexpr int LS = H + 4;    // LDS row of an activation or of W2: 16 rows x 4 entries touch 64 banks
constexpr int XS = IN + 4;   // LDS row of a record or of W1, likewise
constexpr int PS = (NP + 4) / 4 * 4;  // a workgroup's partial: NP gradient entries, then its summed loss
static_assert(PS > NP, "room for the loss");
constexpr int kMaxBlocks = 512;       // larger batches loop over tiles: two workgroups per CU

typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__device__ __forceinline__ float bf16r(float x) {
    unsigned u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u) return x;  // inf / nan unchanged
    unsigned r = u + 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(r & 0xffff0000u);
}
__device__ __forceinline__ float gelu(float a) { return 0.5f * a * (1.0f + erff(a * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float a) {
    return 0.5f * (1.0f + erff(a * 0.70710678118654752f)) + a * 0.39894228040143268f * expf(-0.5f * a * a);
}

// Partial gradients d loss / d params of the records idx[0..cnt) (or 0..cnt when idx == nullptr),
// one row of `part` per workgroup; pred (optional) receives the outputs.
// Matrix operand layout (16x16x4): lane l holds A[l % 16][l / 16] and B[l / 16][l % 16], and rows
// 4 (l / 16) .. + 3 of column l % 16 of the result.
__global__ void __launch_bounds__(256) mlp_tile(const float* __restrict__ P, const float* __restrict__ X,
                                                const float* __restrict__ Y, const float* __restrict__ Wt,
                                                const int32_t* __restrict__ idx, int cnt, float inv_n,
                                                float* __restrict__ part, float* __restrict__ pred) {
    __shared__ float w1[H * XS], w2[H * LS], w3[OUT * H], bias[2 * H + OUT];
    __shared__ float xs[R * XS], h1[R * LS], h2[R * LS], da2[R * LS], os[R * OUT], dO[R * OUT];
    const int t = threadIdx.x, wave = t >> 6, l = t & 63, c16 = l & 15, q = l >> 4;
    for (int i = t; i < H * IN; i += 256) w1[(i / IN) * XS + i % IN] = bf16r(P[OFF_W1 + i]);
    for (int i = t; i < H * H; i += 256) w2[(i / H) * LS + i % H] = bf16r(P[OFF_W2 + i]);
    if (t < OUT * H) w3[t] = bf16r(P[OFF_W3 + t]);
    if (t < H) bias[t] = bf16r(P[OFF_B1 + t]);
    else if (t < 2 * H) bias[t] = bf16r(P[OFF_B2 + t - H]);
    else if (t < 2 * H + OUT) bias[t] = bf16r(P[OFF_B3 + t - 2 * H]);
    const int col = wave * 16 + c16;  // this lane's hidden unit in every tile of the hidden layers
    f32x4 g2[4];                      // W2 gradient rows 16 wave .. + 15, columns 16 k .. + 15
    for (int k = 0; k < 4; k++) g2[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float g3 = 0.0f, gb3 = 0.0f, gb2 = 0.0f, gb1 = 0.0f, g1a = 0.0f, g1b = 0.0f, lsum = 0.0f;
    const int ntiles = (cnt + R - 1) / R;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        {   // a record's 8 features: one per thread
            const int r = t >> 3, rr = tile * R + r;
            const bool valid = rr < cnt;
            const int rec = valid ? (idx ? idx[rr] : rr) : 0;
            xs[r * XS + (t & 7)] = valid ? X[(size_t)rec * IN + (t & 7)] : 0.0f;
        }
        __syncthreads();
        float d1[2][4], d2[2][4];
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {  // layer 1
            const float b = bias[col];
            f32x4 z = {b, b, b, b};
#pragma unroll
            for (int k = 0; k < IN; k += 4) z = mma(xs[(rt * 16 + c16) * XS + k + q], w1[col * XS + k + q], z);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                h1[(rt * 16 + q * 4 + i) * LS + col] = gelu(z[i]);
                d1[rt][i] = gelu_d(z[i]);
            }
        }
        __syncthreads();
        {   // layer 2
            const float b = bias[H + col];
            f32x4 z[2] = {{b, b, b, b}, {b, b, b, b}};
#pragma unroll
            for (int k = 0; k < H; k += 4) {
                const float w = w2[col * LS + k + q];
                z[0] = mma(h1[c16 * LS + k + q], w, z[0]);
                z[1] = mma(h1[(16 + c16) * LS + k + q], w, z[1]);
            }
#pragma unroll
            for (int rt = 0; rt < 2; rt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    h2[(rt * 16 + q * 4 + i) * LS + col] = gelu(z[rt][i]);
                    d2[rt][i] = gelu_d(z[rt][i]);
                }
        }
        __syncthreads();
        {   // outputs: four lanes per (record, output), 16 units each
            const int o = t >> 2, r = o >> 1, j = o & 1, k0 = (t & 3) * 16;
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < 16; k++) s = fmaf(w3[j * H + k0 + k], h2[r * LS + k0 + k], s);
            s += __shfl_xor(s, 1, 64);
            s += __shfl_xor(s, 2, 64);
            if ((t & 3) == 0) os[o] = s + bias[2 * H + j];
        }
        __syncthreads();
        if (t < R) {
            const int rr = tile * R + t;
            const bool valid = rr < cnt;
            float e0 = 0.0f, e1 = 0.0f;
            if (valid) {
                const size_t rec = idx ? idx[rr] : rr;
                const float o0 = os[t * OUT], o1 = os[t * OUT + 1];
                const float y0 = Y[rec * OUT], y1 = Y[rec * OUT + 1], c0 = Wt[rec * OUT], c1 = Wt[rec * OUT + 1];
                const float e = o0 - y0, sg = 1.0f / (1.0f + expf(-o1));
                // BCE with logits, stable form: max(o,0) - o*y + log(1 + exp(-|o|))
                const float bce = fmaxf(o1, 0.0f) - o1 * y1 + log1pf(expf(-fabsf(o1)));
                lsum += c0 * 0.5f * e * e + c1 * bce;
                e0 = c0 * e * inv_n;
                e1 = c1 * (sg - y1) * inv_n;
                if (pred) { pred[(size_t)rr * OUT] = o0; pred[(size_t)rr * OUT + 1] = o1; }
            }
            dO[t * OUT] = e0;
            dO[t * OUT + 1] = e1;
        }
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = rt * 16 + q * 4 + i;
                da2[r * LS + col] = (dO[r * OUT] * w3[col] + dO[r * OUT + 1] * w3[H + col]) * d2[rt][i];
            }
        if (t < OUT * H) {  // layer 3 gradients
#pragma unroll 8
            for (int r = 0; r < R; r++) g3 = fmaf(dO[r * OUT + (t >> 6)], h2[r * LS + (t & 63)], g3);
        } else if (t < OUT * H + OUT) {
            for (int r = 0; r < R; r++) gb3 += dO[r * OUT + t - OUT * H];
        }
        __syncthreads();
        // layer 2 gradients: W2 rows of this wave
#pragma unroll
        for (int r = 0; r < R; r += 4) {
            const float a = da2[(r + q) * LS + col];
#pragma unroll
            for (int k = 0; k < 4; k++) g2[k] = mma(a, h1[(r + q) * LS + k * 16 + c16], g2[k]);
        }
        if (t < H) {
#pragma unroll 8
            for (int r = 0; r < R; r++) gb2 += da2[r * LS + t];
        }
        {   // d loss / d z1, into h2 (no longer needed)
            f32x4 z[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
            for (int k = 0; k < H; k += 4) {
                const float w = w2[(k + q) * LS + col];
                z[0] = mma(da2[c16 * LS + k + q], w, z[0]);
                z[1] = mma(da2[(16 + c16) * LS + k + q], w, z[1]);
            }
#pragma unroll
            for (int rt = 0; rt < 2; rt++)
#pragma unroll
                for (int i = 0; i < 4; i++) h2[(rt * 16 + q * 4 + i) * LS + col] = z[rt][i] * d1[rt][i];
        }
        __syncthreads();
        {   // layer 1 gradients: thread t has unit t / 4, features 2 (t % 4) and the next
            const int j = t >> 2, i = (t & 3) * 2;
#pragma unroll 8
            for (int r = 0; r < R; r++) {
                const float d = h2[r * LS + j];
                g1a = fmaf(d, xs[r * XS + i], g1a);
                g1b = fmaf(d, xs[r * XS + i + 1], g1b);
            }
            if (t < H) {
#pragma unroll 8
                for (int r = 0; r < R; r++) gb1 += h2[r * LS + t];
            }
        }
        __syncthreads();
    }
    float* g = part + (size_t)blockIdx.x * PS;
    g[OFF_W1 + (t >> 2) * IN + (t & 3) * 2] = g1a;
    g[OFF_W1 + (t >> 2) * IN + (t & 3) * 2 + 1] = g1b;
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int i = 0; i < 4; i++) g[OFF_W2 + (wave * 16 + q * 4 + i) * H + k * 16 + c16] = g2[k][i];
    if (t < H) {
        g[OFF_B1 + t] = gb1;
        g[OFF_B2 + t] = gb2;
    }
    if (t < OUT * H) g[OFF_W3 + t] = g3;
    else if (t < OUT * H + OUT) g[OFF_B3 + t - OUT * H] = gb3;
    if (wave == 0) {  // the loss sums of threads 0 .. R - 1
        for (int off = R / 2; off > 0; off >>= 1) lsum += __shfl_down(lsum, off, 64);
        if (t == 0) g[NP] = lsum;
    }
}

// The gradient (sum of the nb partials, in a fixed order) and the batch's loss, added to *loss; with
// `adam`, the Adam step on the parameters, else the gradient is written to G.
__global__ void __launch_bounds__(256) grad_step(const float* __restrict__ part, int nb, float* __restrict__ loss, bool adam,
                                                 float* __restrict__ G, float* __restrict__ P, float* __restrict__ M,
                                                 float* __restrict__ V, float lr, float b1, float b2, float eps, float c1,
                                                 float c2) {
    __shared__ float sums[4][64];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, i = blockIdx.x * 64 + l;
    float s = 0.0f;
    if (i <= NP) {
#pragma unroll 8
        for (int b = w; b < nb; b += 4) s += part[(size_t)b * PS + i];
    }
    sums[w][l] = s;
    __syncthreads();
    if (w != 0 || i > NP) return;
    const float g = (sums[0][l] + sums[1][l]) + (sums[2][l] + sums[3][l]);
    if (i == NP) {
        *loss += g;
    } else if (!adam) {
        G[i] = g;
    } else {
        float m = b1 * M[i] + (1.0f - b1) * g;
        float v = b2 * V[i] + (1.0f - b2) * g * g;
        M[i] = m;
        V[i] = v;
        P[i] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
    }
}

__global__ void fill_zero(float* p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

#define CK(x)                                                            \
    do {                                                                 \
        hipError_t e_ = (x);                                             \
        if (e_ != hipSuccess) { *err = std::string(#x ": ") + hipGetErrorString(e_); return HCG_ERR_HIP; } \
    } while (0)

int ensure(hcg::MlpWork* w, long n, std::string* err) {
    auto alloc = [&](size_t bytes) -> void* {
        void* p = nullptr;
        const hipError_t e = hipMalloc(&p, bytes);
        if (e == hipSuccess) return p;
        (void)hipGetLastError();
        *err = std::string("hipMalloc of the training workspace: ") + hipGetErrorString(e);
        return nullptr;
    };
    const bool ok = hcg::mlp_work_ensure(w, n, IN, OUT, NP, (size_t)PS * kMaxBlocks, alloc, [](void* p) { (void)hipFree(p); });
    return ok ? HCG_OK : HCG_ERR_HIP;
}

int tile_blocks(int cnt) { return std::min((cnt + R - 1) / R, kMaxBlocks); }

}  // namespace

namespace hcg {

void mlp_work_free(MlpWork* w) {
    void* ps[] = {w->params, w->grad, w->adam_m, w->adam_v, w->x, w->y, w->w, w->pred, w->loss, w->perm, w->part};
    for (void* p : ps) if (p) hipFree(p);
    *w = MlpWork();
}

int mlp_forward_backward(MlpWork* w, hipStream_t st, const float* params, int32_t n, const float* x, const float* y,
                         const float* wt, float* out_pred, float* loss, float* grad, std::string* err) {
    int rc = ensure(w, std::max<int32_t>(n, 1), err);
    if (rc) return rc;
    CK(hipMemcpyAsync(w->params, params, sizeof(float) * NP, hipMemcpyHostToDevice, st));
    if (n > 0) {
        CK(hipMemcpyAsync(w->x, x, sizeof(float) * IN * n, hipMemcpyHostToDevice, st));
        CK(hipMemcpyAsync(w->y, y, sizeof(float) * OUT * n, hipMemcpyHostToDevice, st));
        CK(hipMemcpyAsync(w->w, wt, sizeof(float) * OUT * n, hipMemcpyHostToDevice, st));
    }
    fill_zero<<<1, 64, 0, st>>>(w->loss, 1);
    if (n > 0) mlp_tile<<<tile_blocks(n), 256, 0, st>>>(w->params, w->x, w->y, w->w, nullptr, n, 1.0f / n, w->part, w->pred);
    grad_step<<<NP / 64 + 1, 256, 0, st>>>(w->part, tile_blocks(n), w->loss, false, w->grad, nullptr, nullptr, nullptr, 0.0f,
                                           0.0f, 0.0f, 0.0f, 1.0f, 1.0f);
    CK(hipGetLastError());
    float l = 0.0f;
    CK(hipMemcpyAsync(&l, w->loss, sizeof(float), hipMemcpyDeviceToHost, st));
    if (grad) CK(hipMemcpyAsync(grad, w->grad, sizeof(float) * NP, hipMemcpyDeviceToHost, st));
    if (out_pred && n > 0) CK(hipMemcpyAsync(out_pred, w->pred, sizeof(float) * OUT * n, hipMemcpyDeviceToHost, st));
    CK(hipStreamSynchronize(st));
    if (loss) *loss = n > 0 ? l / n : 0.0f;
    return HCG_OK;
}

int mlp_train(MlpWork* w, hipStream_t st, float* params, int32_t n, const float* x, const float* y, const float* wt,
              int32_t epochs, int32_t batch, float lr, uint64_t seed, float* final_loss, std::string* err) {
    int rc = ensure(w, n, err);
    if (rc) return rc;
    CK(hipMemcpyAsync(w->params, params, sizeof(float) * NP, hipMemcpyHostToDevice, st));
    CK(hipMemcpyAsync(w->x, x, sizeof(float) * IN * n, hipMemcpyHostToDevice, st));
    CK(hipMemcpyAsync(w->y, y, sizeof(float) * OUT * n, hipMemcpyHostToDevice, st));
    CK(hipMemcpyAsync(w->w, wt, sizeof(float) * OUT * n, hipMemcpyHostToDevice, st));
    fill_zero<<<(NP + 255) / 256, 256, 0, st>>>(w->adam_m, NP);
    fill_zero<<<(NP + 255) / 256, 256, 0, st>>>(w->adam_v, NP);
    std::vector<int32_t> perm(n), next;
    std::iota(perm.begin(), perm.end(), 0);
    std::mt19937_64 rng(seed);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    long step = 0;
    float last = 0.0f;
    if (epochs > 0) std::shuffle(perm.begin(), perm.end(), rng);
    for (int ep = 0; ep < epochs; ep++) {
        CK(hipMemcpyAsync(w->perm, perm.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, st));
        fill_zero<<<1, 64, 0, st>>>(w->loss, 1);
        for (int off = 0; off < n; off += batch) {
            int cnt = std::min(batch, n - off), nb = tile_blocks(cnt);
            mlp_tile<<<nb, 256, 0, st>>>(w->params, w->x, w->y, w->w, w->perm + off, cnt, 1.0f / cnt, w->part, nullptr);
            step++;
            float c1 = 1.0f - std::pow(b1, (float)step), c2 = 1.0f - std::pow(b2, (float)step);
            grad_step<<<NP / 64 + 1, 256, 0, st>>>(w->part, nb, w->loss, true, nullptr, w->params, w->adam_m, w->adam_v, lr,
                                                   b1, b2, eps, c1, c2);
        }
        CK(hipGetLastError());
        CK(hipMemcpyAsync(&last, w->loss, sizeof(float), hipMemcpyDeviceToHost, st));
        if (ep + 1 < epochs) {  // the next epoch's order, while this one runs
            next = perm;
            std::shuffle(next.begin(), next.end(), rng);
        }
        CK(hipStreamSynchronize(st));
        perm.swap(next);
    }
    CK(hipMemcpyAsync(params, w->params, sizeof(float) * NP, hipMemcpyDeviceToHost, st));
    CK(hipStreamSynchronize(st));
    if (final_loss) *final_loss = last / n;
    return HCG_OK;
}

}  // namespace hcg
