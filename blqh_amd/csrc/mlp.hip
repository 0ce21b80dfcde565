// mlp.hip -- learned warm start for the Lanczos solver.
//
// No counterpart in the reference: it replaces the seeded random start vector
// of pass 1 (BLQH_without_spin/lanczos_hamiltonian.cpp:466-483, Vec::init_random
// matrix.cpp:54-75) by a network's guess of the ground state; the seeded start
// stays available and every solve still runs to the same stopping rule.
//
// Network (FP32): inputs x = (2 b_k - 1 for the occupation bits b_k of the
// basis word, k < nbits; d / 3; 10 Delta_SAS), two hidden layers of 64 tanh
// units, two outputs: o0 = log |psi_i| and o1 = logit of sign(psi_i) > 0.
// Parameters, flat: W1[nin][64], b1[64], W2[64][64], b2[64], W3[64][2], b3[2].
//
// Training data: ground states psi of (sector, d, Delta_SAS) sets computed by
// the engine, gauge-fixed to real (the phase of the largest component is
// removed).  A minibatch draws states with probability |psi_i|^2 within a set
// chosen uniformly, so the loss
//     L = mean_s [ (o0_s - log|psi_s|)^2 + softplus(o1_s) - sign01_s o1_s ]
// weighs configurations by their weight in the ground state.
// Step kernels: k_sample (draw the minibatch), k_fwd_bwd (a workgroup per tile
// of 16 states: forward, loss, back-propagation and gradient sums), k_grad_sum (per
// parameter, workgroups summed in order: deterministic), k_adam.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "engine.hpp"

namespace {

using namespace blqh;

constexpr int kH = 64;      // hidden width
constexpr int kMaxIn = 66;  // 64 occupation bits + 2 parameters
constexpr int kT = 256;

struct Dims {
    int nbits, nin;
    int oW1, ob1, oW2, ob2, oW3, ob3, n;  // offsets into the flat parameter vector
};

Dims make_dims(int nbits) {
    Dims d;
    d.nbits = nbits;
    d.nin = nbits + 2;
    d.oW1 = 0;
    d.ob1 = d.oW1 + d.nin * kH;
    d.oW2 = d.ob1 + kH;
    d.ob2 = d.oW2 + kH * kH;
    d.oW3 = d.ob2 + kH;
    d.ob3 = d.oW3 + kH * 2;
    d.n = d.ob3 + 2;
    return d;
}

// one minibatch in HBM, struct-of-arrays
struct Samples {
    uint64_t* word;
    float* pd;     // d
    float* ps;     // Delta_SAS
    float* ya;     // log |psi|
    float* ys;     // 1 if psi > 0 else 0
    float* loss;   // [B]
};

__device__ __forceinline__ float feature(const Dims& D, uint64_t w, float pd, float ps, int k) {
    if (k < D.nbits) return ((w >> k) & 1ull) ? 1.0f : -1.0f;
    return k == D.nbits ? pd * (1.0f / 3.0f) : ps * 10.0f;
}

// Inference: a workgroup of kT threads evaluates a tile of kTile states.  LDS holds the
// parameters (W2 with a padded row stride so that a wavefront reading one
// column touches 64 different banks), the tile's inputs and activations.
constexpr int kTile = 64;
constexpr int kLd = kH + 1;  // padded row stride of the 64-wide LDS matrices
struct Lds {
    float W1[kMaxIn * kH], b1[kH], W2[kH * kLd], b2[kH], W3[kH * 2], b3[2];
    float X[kTile * (kMaxIn + 1)];  // inputs, row stride nin + 1
    float H1[kTile * kLd], H2[kTile * kLd];
    float O[kTile * 2];
};

__device__ __forceinline__ void stage_params(const Dims& D, const float* __restrict__ P, Lds& L) {
    for (int i = threadIdx.x; i < D.nin * kH; i += kT) L.W1[i] = P[D.oW1 + i];
    for (int i = threadIdx.x; i < kH * kH; i += kT) L.W2[(i / kH) * kLd + i % kH] = P[D.oW2 + i];
    for (int i = threadIdx.x; i < kH; i += kT) {
        L.b1[i] = P[D.ob1 + i];
        L.b2[i] = P[D.ob2 + i];
    }
    for (int i = threadIdx.x; i < 2 * kH; i += kT) L.W3[i] = P[D.oW3 + i];
    if (threadIdx.x < 2) L.b3[threadIdx.x] = P[D.ob3 + threadIdx.x];
}

// Forward of a tile (nt <= kTile valid states, the rest zero inputs): L.H1,
// L.H2 (tanh activations), L.O (outputs).  Thread t computes unit t % 64 for
// states t / 64, t / 64 + 4, ...: a wavefront shares the state (broadcast
// reads of X / H) and spans the units (consecutive weight reads).
__device__ __forceinline__ void tile_forward(const Dims& D, Lds& L, const uint64_t* __restrict__ word,
                                             const float* __restrict__ pd, const float* __restrict__ ps, int nt) {
    const int ldx = D.nin + 1;
    for (int e = threadIdx.x; e < kTile * D.nin; e += kT) {
        const int s = e / D.nin, k = e % D.nin;
        L.X[s * ldx + k] = s < nt ? feature(D, word[s], pd[s], ps[s], k) : 0.0f;
    }
    __syncthreads();
    const int j = threadIdx.x % kH;
    for (int s = threadIdx.x / kH; s < kTile; s += kT / kH) {
        float z = L.b1[j];
        for (int k = 0; k < D.nin; ++k) z += L.X[s * ldx + k] * L.W1[k * kH + j];
        L.H1[s * kLd + j] = tanhf(z);
    }
    __syncthreads();
    for (int s = threadIdx.x / kH; s < kTile; s += kT / kH) {
        float z = L.b2[j];
#pragma unroll 8
        for (int i = 0; i < kH; ++i) z += L.H1[s * kLd + i] * L.W2[i * kLd + j];
        L.H2[s * kLd + j] = tanhf(z);
    }
    __syncthreads();
    if (threadIdx.x < 2 * kTile) {
        const int s = threadIdx.x / 2, c = threadIdx.x % 2;
        float z = L.b3[c];
#pragma unroll 8
        for (int i = 0; i < kH; ++i) z += L.H2[s * kLd + i] * L.W3[2 * i + c];
        L.O[2 * s + c] = z;
    }
    __syncthreads();
}

// Start vector: psi_i = exp(o0) * sign(o1) for every basis word
__global__ void __launch_bounds__(kT) k_infer(Dims D, const float* __restrict__ P, int64_t n,
                                              const uint64_t* __restrict__ words, float pd, float ps,
                                              double2* __restrict__ out) {
    __shared__ Lds L;
    __shared__ float spd[kTile], sps[kTile];
    stage_params(D, P, L);
    if (threadIdx.x < kTile) {
        spd[threadIdx.x] = pd;
        sps[threadIdx.x] = ps;
    }
    for (int64_t t0 = (int64_t)blockIdx.x * kTile; t0 < n; t0 += (int64_t)gridDim.x * kTile) {
        const int nt = (int)(n - t0 < kTile ? n - t0 : kTile);
        __syncthreads();  // parameters staged / previous tile read
        tile_forward(D, L, words + t0, spd, sps, nt);
        if (threadIdx.x < nt) {
            const double a = exp((double)L.O[2 * threadIdx.x]);
            out[t0 + threadIdx.x] = make_double2(L.O[2 * threadIdx.x + 1] > 0.0f ? a : -a, 0.0);
        }
    }
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Draw the minibatch: set uniform, state ~ |psi|^2 by binary search in the set's CDF.
__global__ void __launch_bounds__(kT) k_sample(int B, uint64_t key, int nsets, const int64_t* __restrict__ set0,
                                               const double* __restrict__ cdf, const uint64_t* __restrict__ words,
                                               const float* __restrict__ ya, const float* __restrict__ ys,
                                               const float* __restrict__ setd, const float* __restrict__ sets,
                                               Samples S) {
    const int s = blockIdx.x * kT + threadIdx.x;
    if (s >= B) return;
    const uint64_t r1 = mix64(key ^ (uint64_t)s * 0xD1B54A32D192ED03ull);
    const uint64_t r2 = mix64(r1);
    const int set = (int)(r1 % (uint64_t)nsets);
    const int64_t a = set0[set], b = set0[set + 1];
    const double u = (double)(r2 >> 11) * (1.0 / 9007199254740992.0);  // [0, 1)
    int64_t lo = a, hi = b - 1;  // first i with cdf[i] > u
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (cdf[mid] > u) hi = mid;
        else lo = mid + 1;
    }
    S.word[s] = words[lo];
    S.pd[s] = setd[set];
    S.ps[s] = sets[set];
    S.ya[s] = ya[lo];
    S.ys[s] = ys[lo];
}

// value of lane i of the wavefront, the same for all of it
__device__ __forceinline__ float lane_value(float v, int i) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i));
}

// a word that is the same on every lane, in scalar registers
__device__ __forceinline__ uint64_t scalar(uint64_t w) {
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(w >> 32)) << 32 |
           (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
}

// Forward, loss, back-propagation and the parameter-gradient sums of the workgroup's tiles
// of kSt states (part[workgroup][param], summed by k_grad_sum in order).
//
// A wavefront takes kSw states, lane = unit: activations and deltas stay in registers and
// reach the other units by lane reads, so a weight read serves kSw states and the LDS
// holds only W2 (padded: the backward pass reads it across) and what the gradient sums
// share.  Bound by latency: a minibatch of 4,096 states is 256 tiles, one for each CU;
// with tiles of 64 states, every product through LDS and a quarter of the CUs busy the
// forward and backward of that took 66 us, 50 now, and the sums 16, 4 now.
// Past kMaxWgs tiles a workgroup takes several and keeps their sums in registers.
constexpr int kSt = 16, kSw = kSt / (kT / 64), kMaxWgs = 512;
constexpr int kR1 = (kMaxIn + kT / 64 - 1) / (kT / 64);  // rows of W1 a wavefront sums

__global__ void __launch_bounds__(kT) k_fwd_bwd(Dims D, const float* __restrict__ P, int B, Samples S,
                                                float* __restrict__ part) {
    __shared__ float W2[kH * kLd], H1[kSt * kH], D2[kSt * kH], D1[kSt * kH];
    __shared__ uint64_t sw[kSt];
    __shared__ float sd[kSt], ss[kSt], sa[kSt], sy[kSt];
    __shared__ float red[kT / 64][4][kH + 1];  // the wavefronts' sums of W3's columns and the biases
    const int j = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int ntiles = (B + kSt - 1) / kSt;
    for (int i = threadIdx.x; i < kH * kH; i += kT) W2[(i / kH) * kLd + i % kH] = P[D.oW2 + i];
    const float b1 = P[D.ob1 + j], b2 = P[D.ob2 + j], w30 = P[D.oW3 + 2 * j], w31 = P[D.oW3 + 2 * j + 1];
    const float b30 = P[D.ob3], b31 = P[D.ob3 + 1];
    float g2[kH / 4], g1[kR1];  // sums of rows wv kH/4 + i of W2, wv + 4 i of W1
    float g30 = 0.0f, g31 = 0.0f, gb1 = 0.0f, gb2 = 0.0f, gb30 = 0.0f, gb31 = 0.0f;
#pragma unroll
    for (int i = 0; i < kH / 4; ++i) g2[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < kR1; ++i) g1[i] = 0.0f;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int t0 = tile * kSt;
        __syncthreads();  // W2 staged / the previous tile's sums done
        if (threadIdx.x < kSt) {
            const int s = threadIdx.x;
            const bool on = t0 + s < B;
            sw[s] = on ? S.word[t0 + s] : 0;
            sd[s] = on ? S.pd[t0 + s] * (1.0f / 3.0f) : 0.0f;
            ss[s] = on ? S.ps[t0 + s] * 10.0f : 0.0f;
            sa[s] = on ? S.ya[t0 + s] : 0.0f;
            sy[s] = on ? S.ys[t0 + s] : 0.0f;
        }
        __syncthreads();
        uint64_t w[kSw];
        float h1[kSw], h2[kSw], z[kSw];
#pragma unroll
        for (int q = 0; q < kSw; ++q) {
            w[q] = scalar(sw[wv * kSw + q]);
            z[q] = b1;
        }
#pragma unroll 8
        for (int k = 0; k < D.nbits; ++k) {
            const float wt = P[D.oW1 + k * kH + j];
#pragma unroll
            for (int q = 0; q < kSw; ++q) z[q] += (w[q] >> k & 1ull) ? wt : -wt;
        }
        {
            const float wd = P[D.oW1 + D.nbits * kH + j], ws = P[D.oW1 + (D.nbits + 1) * kH + j];
#pragma unroll
            for (int q = 0; q < kSw; ++q) {
                z[q] += sd[wv * kSw + q] * wd;
                z[q] += ss[wv * kSw + q] * ws;
                h1[q] = tanhf(z[q]);
                z[q] = b2;
            }
        }
#pragma unroll 16
        for (int i = 0; i < kH; ++i) {
            const float wt = W2[i * kLd + j];
#pragma unroll
            for (int q = 0; q < kSw; ++q) z[q] += lane_value(h1[q], i) * wt;
        }
        float d2[kSw], d1[kSw], o0 = 0.0f, o1 = 0.0f;
#pragma unroll
        for (int q = 0; q < kSw; ++q) {
            h2[q] = tanhf(z[q]);
            float a0 = h2[q] * w30, a1 = h2[q] * w31;
            for (int o = 32; o > 0; o >>= 1) {
                a0 += __shfl_xor(a0, o, 64);
                a1 += __shfl_xor(a1, o, 64);
            }
            if (j == q) {
                o0 = a0 + b30;
                o1 = a1 + b31;
            }
        }
        // loss and dL/do of the wavefront's states, one a lane (past B: none)
        float e0 = 0.0f, e1 = 0.0f;
        {
            const int s = wv * kSw + (j & (kSw - 1));
            const float ea = o0 - sa[s], y = sy[s], ex = expf(o1 > 0.0f ? -o1 : o1);
            const float sp = (o1 > 0.0f ? o1 : 0.0f) + log1pf(ex);  // softplus
            if (j < kSw && t0 + s < B) {
                S.loss[t0 + s] = ea * ea + sp - y * o1;
                e0 = 2.0f * ea;
                e1 = 1.0f / (1.0f + expf(-o1)) - y;
            }
        }
#pragma unroll
        for (int q = 0; q < kSw; ++q) {
            const float f0 = lane_value(e0, q), f1 = lane_value(e1, q);
            d2[q] = (1.0f - h2[q] * h2[q]) * (w30 * f0 + w31 * f1);
            g30 += h2[q] * f0;
            g31 += h2[q] * f1;
            gb30 += f0;
            gb31 += f1;
            gb2 += d2[q];
            d1[q] = 0.0f;
        }
#pragma unroll 16
        for (int i = 0; i < kH; ++i) {
            const float wt = W2[j * kLd + i];
#pragma unroll
            for (int q = 0; q < kSw; ++q) d1[q] += wt * lane_value(d2[q], i);
        }
#pragma unroll
        for (int q = 0; q < kSw; ++q) {
            const int s = wv * kSw + q;
            d1[q] *= 1.0f - h1[q] * h1[q];
            gb1 += d1[q];
            H1[s * kH + j] = h1[q];
            D2[s * kH + j] = d2[q];
            D1[s * kH + j] = d1[q];
        }
        __syncthreads();
        // W2: sum_s H1[s][i] D2[s][j];  W1: sum_s x[s][k] D1[s][j]
        for (int s = 0; s < kSt; ++s) {
            const float e2 = D2[s * kH + j], e1 = D1[s * kH + j];
            const uint64_t word = scalar(sw[s]);
#pragma unroll
            for (int i = 0; i < kH / 4; ++i) g2[i] += H1[s * kH + wv * (kH / 4) + i] * e2;
#pragma unroll
            for (int i = 0; i < kR1; ++i) {
                const int k = wv + 4 * i;
                if (k < D.nbits) g1[i] += (word >> k & 1ull) ? e1 : -e1;
                else if (k == D.nbits) g1[i] += sd[s] * e1;
                else if (k == D.nbits + 1) g1[i] += ss[s] * e1;
            }
        }
    }
    float* out = part + (int64_t)blockIdx.x * D.n;
#pragma unroll
    for (int i = 0; i < kH / 4; ++i) out[D.oW2 + (wv * (kH / 4) + i) * kH + j] = g2[i];
#pragma unroll
    for (int i = 0; i < kR1; ++i)
        if (wv + 4 * i < D.nin) out[D.oW1 + (wv + 4 * i) * kH + j] = g1[i];
    red[wv][0][j] = g30;
    red[wv][1][j] = g31;
    red[wv][2][j] = gb1;
    red[wv][3][j] = gb2;
    if (j == 0) {
        red[wv][0][kH] = gb30;
        red[wv][1][kH] = gb31;
    }
    __syncthreads();
    if (wv < 4) {  // a wavefront per kind, the wavefronts' shares in order
        float t = 0.0f;
        for (int q = 0; q < kT / 64; ++q) t += red[q][wv][j];
        out[wv < 2 ? D.oW3 + 2 * j + wv : (wv == 2 ? D.ob1 : D.ob2) + j] = t;
        if (j == 0 && wv < 2) {
            t = 0.0f;
            for (int q = 0; q < kT / 64; ++q) t += red[q][wv][kH];
            out[D.ob3 + wv] = t;
        }
    }
}

// grad = (sum over the workgroups of k_fwd_bwd) / B: 64 parameters a workgroup, its 16
// wavefronts sum a sixteenth of the partials each, added in order.  The last workgroup
// sums the losses (fixed order), if wanted.
constexpr int kGs = 1024;
__device__ void loss_total(int B, const float* __restrict__ loss, double* sh, int nt, double* out) {
    double a = 0.0;
    for (int s = threadIdx.x; s < B; s += nt) a += loss[s];
    sh[threadIdx.x] = a;
    __syncthreads();
    for (int o = nt / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0] / B;
}
__global__ void __launch_bounds__(kGs) k_grad_sum(int n, int nparts, int B, const float* __restrict__ part,
                                                  float* __restrict__ grad, const float* __restrict__ loss,
                                                  double* __restrict__ out) {
    __shared__ double sh[kGs];
    if ((int)blockIdx.x == (n + 63) / 64) {
        loss_total(B, loss, sh, kGs, out);
        return;
    }
    float* f = reinterpret_cast<float*>(sh);
    const int p = blockIdx.x * 64 + (threadIdx.x & 63), wv = threadIdx.x >> 6, per = (nparts + 15) / 16;
    const int t1 = (wv + 1) * per < nparts ? (wv + 1) * per : nparts;
    float acc = 0.0f;
    if (p < n) {
#pragma unroll 8
        for (int t = wv * per; t < t1; ++t) acc += part[(int64_t)t * n + p];
    }
    f[threadIdx.x] = acc;
    __syncthreads();
    if (wv == 0 && p < n) {
        float t = 0.0f;
        for (int q = 0; q < 16; ++q) t += f[q * 64 + threadIdx.x];
        grad[p] = t / (float)B;
    }
}

__global__ void __launch_bounds__(kT) k_adam(int n, float* __restrict__ P, const float* __restrict__ g,
                                             float* __restrict__ m, float* __restrict__ v, float lr, float b1t,
                                             float b2t) {
    const int i = blockIdx.x * kT + threadIdx.x;
    if (i >= n) return;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    P[i] -= lr * (mi / (1.0f - b1t)) / (sqrtf(vi / (1.0f - b2t)) + eps);
}

// mean of the minibatch losses alone
__global__ void __launch_bounds__(kGs) k_loss_sum(int B, const float* __restrict__ loss, double* __restrict__ out) {
    __shared__ double sh[kGs];
    loss_total(B, loss, sh, kGs, out);
}

int fb_grid(int B) { return (int)std::min<int64_t>(ceil_div(B, kSt), kMaxWgs); }

void launch_grad(const Dims& D, const float* P, int B, const Samples& S, float* part, float* grad, double* loss,
                 hipStream_t st) {
    hipLaunchKernelGGL(k_fwd_bwd, dim3(fb_grid(B)), dim3(kT), 0, st, D, P, B, S, part);
    hipLaunchKernelGGL(k_grad_sum, dim3((D.n + 63) / 64 + (loss ? 1 : 0)), dim3(kGs), 0, st, D.n, fb_grid(B), B, part,
                       grad, S.loss, loss);
}

// B samples in one block at p: words, then pd, ps, ya, ys
Samples packed(char* p, int B, float* loss) {
    float* f = (float*)(p + (size_t)B * 8);
    return Samples{(uint64_t*)p, f, f + B, f + 2 * (size_t)B, f + 3 * (size_t)B, loss};
}

struct Buffers {
    DevBuf<uint64_t> word;
    DevBuf<float> pd, ps, ya, ys, loss, part;
    int cap = 0;
    void ensure(int B, int nparams) {
        if (B <= cap) return;
        word.alloc(B);
        pd.alloc(B);
        ps.alloc(B);
        ya.alloc(B);
        ys.alloc(B);
        loss.alloc(B);
        part.alloc((size_t)fb_grid(B) * nparams);
        cap = B;
    }
    Samples view() { return Samples{word.get(), pd.get(), ps.get(), ya.get(), ys.get(), loss.get()}; }
};

// Pinned host memory of a network's explicit minibatches of up to kPinned states: samples,
// gradient, loss (grow-only, freed with the network).
constexpr int kPinned = 1 << 16;
struct Pinned {
    char* p = nullptr;
    int cap = 0;
    float* grad = nullptr;
    double* lsum = nullptr;
    ~Pinned() {
        if (p) (void)hipHostFree(p);
    }
    void ensure(int B, int nparams) {
        if (B <= cap) return;
        if (p) (void)hipHostFree(p);
        p = nullptr;
        cap = 0;
        const int c = std::min(kPinned, std::max(B, 4096));
        BLQH_HIP(hipHostMalloc((void**)&p, 64 + (size_t)c * 24 + (size_t)nparams * 4, hipHostMallocDefault));
        cap = c;
        lsum = (double*)p;
        grad = (float*)(p + 64 + (size_t)c * 24);
    }
};

}  // namespace

struct blqh_mlp {
    Dims D{};
    DevBuf<float> P, g, m, v;
    int64_t adam_t = 0;
    Buffers buf;
    DevBuf<double> lsum;
    Pinned pin;
};

blqh_mlp* blqh_mlp_create_impl(int nbits, uint32_t seed) {
    BLQH_REQUIRE(nbits >= 1 && nbits <= 64, BLQH_EINVAL, "nbits must be 1..64");
    auto* M = new blqh_mlp;
    try {
        M->D = make_dims(nbits);
        const int n = M->D.n;
        // Glorot-uniform weights from std::mt19937(seed), zero biases
        std::vector<float> h(n, 0.0f);
        std::mt19937 rng(seed);
        auto fill = [&](int off, int fan_in, int fan_out) {
            const float a = std::sqrt(6.0f / (float)(fan_in + fan_out));
            for (int i = 0; i < fan_in * fan_out; ++i) h[off + i] = (float)((rng() * (1.0 / 4294967296.0)) * 2.0 - 1.0) * a;
        };
        fill(M->D.oW1, M->D.nin, kH);
        fill(M->D.oW2, kH, kH);
        fill(M->D.oW3, kH, 2);
        M->P.alloc(n);
        M->g.alloc(n);
        M->m.alloc(n);
        M->v.alloc(n);
        M->lsum.alloc(1);
        copy_sync(M->P.get(), h.data(), n * 4, hipMemcpyHostToDevice);
        BLQH_HIP(hipMemsetAsync(M->m.get(), 0, n * 4, stream()));
        BLQH_HIP(hipMemsetAsync(M->v.get(), 0, n * 4, stream()));
        BLQH_HIP(hipStreamSynchronize(stream()));
    } catch (...) {
        delete M;
        throw;
    }
    return M;
}

void blqh_mlp_destroy_impl(blqh_mlp* M) { delete M; }
int blqh_mlp_nparams_impl(const blqh_mlp* M) { return M->D.n; }
int blqh_mlp_nbits_impl(const blqh_mlp* M) { return M->D.nbits; }

void blqh_mlp_get_params_impl(const blqh_mlp* M, float* out) {
    copy_sync(out, M->P.get(), M->D.n * 4, hipMemcpyDeviceToHost);
}

void blqh_mlp_set_params_impl(blqh_mlp* M, const float* in) {
    copy_sync(M->P.get(), in, M->D.n * 4, hipMemcpyHostToDevice);
    BLQH_HIP(hipMemsetAsync(M->m.get(), 0, M->D.n * 4, stream()));
    BLQH_HIP(hipMemsetAsync(M->v.get(), 0, M->D.n * 4, stream()));
    BLQH_HIP(hipStreamSynchronize(stream()));
    M->adam_t = 0;
}

// Mean loss and gradient over explicit samples (host arrays).
void blqh_mlp_loss_grad_impl(blqh_mlp* M, int64_t ns, const uint64_t* words, const float* pd, const float* ps,
                             const float* ya, const float* ys, double* loss, float* grad) {
    BLQH_REQUIRE(ns >= 1 && ns <= (1 << 24), BLQH_EINVAL, "sample count out of range");
    hipStream_t st = stream();
    const int B = (int)ns;
    M->buf.ensure(B, M->D.n);
    Samples S = M->buf.view();
    const int n = M->D.n;
    if (B <= kPinned) {
        // the kernels read the samples, each once, from pinned host memory and leave gradient
        // and loss there: seven copies of 8 us each otherwise (one copy of all: 6 us more)
        M->pin.ensure(B, n);
        const Samples H = packed(M->pin.p + 64, B, S.loss);
        std::memcpy(H.word, words, (size_t)B * 8);
        std::memcpy(H.pd, pd, (size_t)B * 4);
        std::memcpy(H.ps, ps, (size_t)B * 4);
        std::memcpy(H.ya, ya, (size_t)B * 4);
        std::memcpy(H.ys, ys, (size_t)B * 4);
        launch_grad(M->D, M->P.get(), B, H, M->buf.part.get(), M->pin.grad, M->pin.lsum, st);
        BLQH_HIP(hipGetLastError());
        BLQH_HIP(hipStreamSynchronize(st));
        if (grad) std::memcpy(grad, M->pin.grad, (size_t)n * 4);
        if (loss) *loss = *M->pin.lsum;
        return;
    }
    BLQH_HIP(hipMemcpyAsync(S.word, words, (size_t)B * 8, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(S.pd, pd, (size_t)B * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(S.ps, ps, (size_t)B * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(S.ya, ya, (size_t)B * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(S.ys, ys, (size_t)B * 4, hipMemcpyHostToDevice, st));
    launch_grad(M->D, M->P.get(), B, S, M->buf.part.get(), M->g.get(), M->lsum.get(), st);
    BLQH_HIP(hipGetLastError());
    if (grad) BLQH_HIP(hipMemcpyAsync(grad, M->g.get(), n * 4, hipMemcpyDeviceToHost, st));
    double l = 0;
    BLQH_HIP(hipMemcpyAsync(&l, M->lsum.get(), 8, hipMemcpyDeviceToHost, st));
    BLQH_HIP(hipStreamSynchronize(st));
    if (loss) *loss = l;
}

// Train on ground states: set k = (basis, d, Delta_SAS, psi).
void blqh_mlp_train_impl(blqh_mlp* M, int nsets, const blqh_basis* const* bases, const double* params,
                         const double* const* psi, const blqh_mlp_train_opts& o, blqh_mlp_train_result& r) {
    auto t0 = std::chrono::steady_clock::now();
    BLQH_REQUIRE(nsets >= 1 && bases && params && psi, BLQH_EINVAL, "bad training sets");
    BLQH_REQUIRE(o.steps >= 1 && o.batch >= 1 && o.batch <= (1 << 22) && o.lr > 0, BLQH_EINVAL,
                 "bad training options");
    hipStream_t st = stream();
    // labels: gauge-fixed real ground states, |psi|^2 CDFs
    std::vector<int64_t> set0(nsets + 1, 0);
    for (int k = 0; k < nsets; ++k) {
        BLQH_REQUIRE(bases[k] && psi[k], BLQH_EINVAL, "null training set");
        BLQH_REQUIRE(bases[k]->geo.S * bases[k]->geo.nphi <= M->D.nbits, BLQH_EINVAL, "basis words wider than the network input");
        set0[k + 1] = set0[k] + bases[k]->n;
    }
    const int64_t N = set0[nsets];
    std::vector<uint64_t> words(N);
    std::vector<float> ya(N), ys(N);
    std::vector<double> cdf(N);
    std::vector<float> sd(nsets), ss(nsets);
    for (int k = 0; k < nsets; ++k) {
        const int64_t n = bases[k]->n, a = set0[k];
        std::memcpy(words.data() + a, bases[k]->h_id.data(), n * 8);
        const double2* z = (const double2*)psi[k];
        int64_t imax = 0;
        double amax = -1;
        for (int64_t i = 0; i < n; ++i) {
            const double m2 = z[i].x * z[i].x + z[i].y * z[i].y;
            if (m2 > amax) { amax = m2; imax = i; }
        }
        BLQH_REQUIRE(amax > 0, BLQH_EINVAL, "zero training state");
        const double ph = std::atan2(z[imax].y, z[imax].x);
        const double c = std::cos(ph), s = std::sin(ph);
        double tot = 0;
        for (int64_t i = 0; i < n; ++i) {
            const double re = z[i].x * c + z[i].y * s;  // Re(psi e^{-i ph})
            const double m2 = z[i].x * z[i].x + z[i].y * z[i].y;
            ya[a + i] = (float)std::log(std::max(std::sqrt(m2), 1e-30));
            ys[a + i] = re > 0 ? 1.0f : 0.0f;
            tot += m2;
            cdf[a + i] = tot;
        }
        for (int64_t i = 0; i < n; ++i) cdf[a + i] /= tot;
        cdf[a + n - 1] = 1.0;
        sd[k] = (float)params[2 * k];
        ss[k] = (float)params[2 * k + 1];
    }
    DevBuf<int64_t> dset0(nsets + 1);
    DevBuf<uint64_t> dwords(N);
    DevBuf<float> dya(N), dys(N), dsd(nsets), dss(nsets);
    DevBuf<double> dcdf(N);
    BLQH_HIP(hipMemcpyAsync(dset0.get(), set0.data(), (nsets + 1) * 8, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(dwords.get(), words.data(), N * 8, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(dya.get(), ya.data(), N * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(dys.get(), ys.data(), N * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(dcdf.get(), cdf.data(), N * 8, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(dsd.get(), sd.data(), nsets * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(dss.get(), ss.data(), nsets * 4, hipMemcpyHostToDevice, st));
    const int B = o.batch;
    M->buf.ensure(B, M->D.n);
    Samples S = M->buf.view();
    const int gb = (int)ceil_div(B, kT), gp = (int)ceil_div(M->D.n, kT);
    const double b1 = 0.9, b2 = 0.999;
    std::vector<double> losses;
    auto record = [&]() {
        hipLaunchKernelGGL(k_loss_sum, dim3(1), dim3(kGs), 0, st, B, S.loss, M->lsum.get());
        double l = 0;
        BLQH_HIP(hipMemcpyAsync(&l, M->lsum.get(), 8, hipMemcpyDeviceToHost, st));
        BLQH_HIP(hipStreamSynchronize(st));
        losses.push_back(l);
    };
    const int tail = std::max(1, std::min(o.steps, 20));  // last steps averaged for the reported loss
    double last = 0;
    for (int step = 0; step < o.steps; ++step) {
        const uint64_t key = ((uint64_t)o.seed << 32) ^ (uint64_t)(M->adam_t + 1) * 0x9E3779B97F4A7C15ull;
        hipLaunchKernelGGL(k_sample, dim3(gb), dim3(kT), 0, st, B, key, nsets, dset0.get(), dcdf.get(),
                           dwords.get(), dya.get(), dys.get(), dsd.get(), dss.get(), S);
        launch_grad(M->D, M->P.get(), B, S, M->buf.part.get(), M->g.get(), nullptr, st);
        if (step == 0) record();
        if (step >= o.steps - tail) {
            record();
            last += losses.back();
        }
        ++M->adam_t;
        const float lr = o.lr * (o.lr_final > 0 ? (float)std::pow(o.lr_final / o.lr, (double)step / std::max(1, o.steps - 1)) : 1.0f);
        hipLaunchKernelGGL(k_adam, dim3(gp), dim3(kT), 0, st, M->D.n, M->P.get(), M->g.get(), M->m.get(),
                           M->v.get(), lr, (float)std::pow(b1, (double)M->adam_t), (float)std::pow(b2, (double)M->adam_t));
        BLQH_HIP(hipGetLastError());
    }
    BLQH_HIP(hipStreamSynchronize(st));
    r.loss_first = losses.front();
    r.loss_last = last / tail;
    r.steps = o.steps;
    r.samples = N;
    r.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

// Start vector (normalised, real) for a basis at (d, Delta_SAS).
void blqh_mlp_start_vector_impl(const blqh_mlp* M, const blqh_basis* B, double d, double dsas, double* out) {
    BLQH_REQUIRE(B->geo.S * B->geo.nphi <= M->D.nbits, BLQH_EINVAL, "basis words wider than the network input");
    hipStream_t st = stream();
    const int64_t n = B->n;
    DevBuf<double2> v(std::max<int64_t>(n, 1));
    const int g = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, kTile), 4096));
    hipLaunchKernelGGL(k_infer, dim3(g), dim3(kT), 0, st, M->D, M->P.get(), n, B->id.get(), (float)d, (float)dsas,
                       v.get());
    BLQH_HIP(hipGetLastError());
    BLQH_HIP(hipMemcpyAsync(out, v.get(), n * sizeof(double2), hipMemcpyDeviceToHost, st));
    BLQH_HIP(hipStreamSynchronize(st));
    double s = 0;
    for (int64_t i = 0; i < n; ++i) s += out[2 * i] * out[2 * i];
    BLQH_REQUIRE(s > 0 && std::isfinite(s), BLQH_EINTERNAL, "network start vector is zero or not finite");
    s = 1.0 / std::sqrt(s);
    for (int64_t i = 0; i < 2 * n; ++i) out[i] *= s;
}
