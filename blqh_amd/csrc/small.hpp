// small.hpp -- many Lanczos steps of a small matrix in one workgroup.
//
// A step of a small matrix as three kernels costs 12 us of launches and waits for 1 us of
// work.  Here one workgroup of 16 wavefronts keeps the value table, the vector and the
// row sums in LDS and runs the steps back to back; only the new vector goes to memory, for
// the states.  The sums are taken in the order of k_cod (teams of eight wavefronts on
// 64-row slices), k_lz2 and k_lz3, so the coefficients of a single solve have the same bits
// whichever runs.  A batch's kernels (k_b1x, k_b2, k_b3) sum in another order: the last bits
// of its members depend on whether all of them are small.
// Bound by the instructions of the step's chain (sums, two reductions, a root and a division)
// on one CU: 5.9 us a step at 79 rows (three launches: 15), 8.4 us at 172 rows (16).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "coded.hpp"

namespace blqh {

// Mailbox of a solve in pinned host memory: step j leaves alpha_j and beta_{j+1}
// in entry j mod kMail and then its tag (solve number, step), which the host polls.
// A copy and a stream synchronisation per convergence test cost 31 us of an idle GPU.
struct alignas(64) StepMail {
    double alpha, beta;
    uint64_t tag;
};
constexpr int kMail = 64;

// The stores go through to the host's memory by themselves (system scope), so the tag only
// has to wait for the two before it, not for the caches' write-back.
__device__ __forceinline__ void post_mail(StepMail* mail, int j, double alpha, double beta, uint64_t tag) {
    StepMail* e = mail + (j & (kMail - 1));
    __hip_atomic_store(&e->alpha, alpha, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&e->beta, beta, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(&e->tag, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr int kSmallT = 1024;      // threads
constexpr int kSmallTeam = 8;      // wavefronts of a slice, as k_cod's of a small matrix
constexpr int kSmallRows = 2048;   // rows at most: two a thread
constexpr int kSmallSlices = kSmallRows / 64;

// A matrix of n rows and nnz entries is stepped by one workgroup.  Its step takes 5 us and
// 0.4 us for every 1,000 entries, on its one CU; the kernels' takes 15 to 18 us for one
// matrix of up to 60,000 entries.  Batch of 1 / 8 / 36 members, this against the kernels: 9,400
// entries 8.6 / 20 / 17 us against 16 / 27 / 30; 23,800 entries 12 / 24 / 20 us against 17 / 29 /
// 28; 36,000 entries (1 / 4 / 32 members) 19 / 25 / 29 against 18 / 23 / 31.  Single solves of 60
// steps: 23,800 entries 0.80 ms against 0.91, 36,000 entries 1.17 against 0.94.
constexpr int64_t kSmallWords = (int64_t)3 << 13;
inline bool small_matrix(int64_t n, int64_t nnz) { return n <= kSmallRows && nnz <= kSmallWords; }

constexpr int kSmallLaunch = 64;   // steps of a launch at most (the mailbox's entries)

// LDS: value table, vector, row sums, the teams' shares, row lengths; resident: the matrix as well (words
// and rest)
inline size_t small_lds_bytes(bool real, int ntab, int64_t n, int64_t ncod = 0, int64_t nrest = 0) {
    const auto up = [](size_t b) { return (b + 15) & ~(size_t)15; };
    return cod_lds_bytes(real, ntab) + (size_t)(2 * n + kSmallT) * sizeof(double2) + (size_t)((n + 63) >> 6) * 256 +
           up((size_t)ncod * 4) + up((size_t)nrest * 4) + (size_t)nrest * (real ? 8 : 16);
}
constexpr size_t kSmallLdsMax = 152 * 1024;  // dynamic; a static part of 2 KiB an instantiation

// Sum over lanes 0 .. N - 1 (N = 8, 16, 32 or 64; the others hold zero, or are not read), the
// same on every lane, in the order of the butterfly of __shfl_xor from 32 down to 1: adding
// the lane 8, 4, 2 or 1 behind within a row of 16 is that order, since by then lanes that
// differ in a higher bit hold the same sum.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
template <int N>
__device__ __forceinline__ double wave_total(double v) {
    if (N > 32) v += __shfl_xor(v, 32, 64);
    if (N > 16) v += __shfl_xor(v, 16, 64);
    v += dpp_f64<0x128>(v);  // row_ror:8
    v += dpp_f64<0x124>(v);
    v += dpp_f64<0x122>(v);
    v += dpp_f64<0x121>(v);
    const int64_t b = __double_as_longlong(v);  // lane 0 holds the sum whatever N
    return __longlong_as_double((int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32 |
                                          (uint32_t)__builtin_amdgcn_readfirstlane((int)b)));
}

// Steps j0 .. j1 - 1 of one problem by the whole workgroup (kSmallT threads): W holds the
// vectors, W_j at j n, up to W_j0; alpha[j], beta[j + 1] and invb[j + 1] are written, and to
// mail, if any, with tags tag0 | j + 1.  ZERO: 1/0 is 0 (the batch's convention).  RES: the
// matrix fits in LDS beside the vectors and is staged there.  SH: a shared-scale template,
// flagged entries scaled by ts.
template <bool REAL, bool ZERO, bool RES, bool SH>
__device__ __forceinline__ void small_steps(const CodView& P, int64_t ncod, int64_t nrest, double2* W, double* alpha,
                                            double* beta, double* invb, int j0, int j1, StepMail* mail, uint64_t tag0,
                                            double* lds, double ts) {
    __shared__ double part[kSmallSlices], nrm[kSmallSlices];  // a slice's shares of the two sums
    __shared__ int32_t sbase[kSmallSlices], srbase[kSmallSlices];
    __shared__ double sal[kSmallLaunch], sbe[kSmallLaunch];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, team = wv / kSmallTeam, par = wv % kSmallTeam;
    constexpr int TM = kSmallT / 64 / kSmallTeam;
    const int n = (int)P.n, nsl = (int)P.nslices, gv = (n + 255) >> 8;
    const auto up = [](size_t b) { return (b + 15) & ~(size_t)15; };
    char* at = reinterpret_cast<char*>(lds) + cod_lds_bytes(REAL, P.ntab);
    double2* xs = reinterpret_cast<double2*>(at);
    double2* ys = xs + n;
    double2* red = ys + n;
    uint32_t* slen = reinterpret_cast<uint32_t*>(red + kSmallT);  // words and rest entries of a row: len | rest << 16
    cod_stage<REAL>(P.tab, P.ntab, lds, kSmallT);
    const uint32_t* ent = P.ent;
    const uint32_t* rcol = P.rcol;
    const double* rval = P.rval;
    if (RES) {
        uint32_t* le = slen + nsl * 64;
        uint32_t* lc = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(le) + up((size_t)ncod * 4));
        double* lv = reinterpret_cast<double*>(reinterpret_cast<char*>(lc) + up((size_t)nrest * 4));
        for (int i = tid; i < (int)ncod; i += kSmallT) le[i] = ent[i];
        for (int i = tid; i < (int)nrest; i += kSmallT) lc[i] = rcol[i];
        for (int i = tid; i < (int)nrest * (REAL ? 1 : 2); i += kSmallT) lv[i] = rval[i];
        ent = le;
        rcol = lc;
        rval = lv;
    }
    if (tid < kSmallSlices) nrm[tid] = 0.0;  // of the slices past the last
    if (tid < nsl) {
        sbase[tid] = (int32_t)P.base[tid];
        srbase[tid] = (int32_t)P.rbase[tid];
    }
    for (int r = tid; r < nsl * 64; r += kSmallT) slen[r] = (uint32_t)P.len[r] | (uint32_t)P.rlen[r] << 16;
    double2 w[2], wp[2], dg[2];  // the thread's rows tid and tid + kSmallT
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = tid + k * kSmallT;
        w[k] = wp[k] = dg[k] = make_double2(0.0, 0.0);
        if (r < n) {
            xs[r] = w[k] = W[(int64_t)j0 * n + r];
            if (j0 > 0) wp[k] = W[(int64_t)(j0 - 1) * n + r];
            dg[k] = cod_diag(P, REAL, r);
        }
    }
    double ib = invb[j0], bj = beta[j0], ibp = j0 > 0 ? invb[j0 - 1] : 0.0;
    wait_vmem();
    __syncthreads();
    for (int j = j0; j < j1; ++j) {
        for (int s0 = 0; s0 < nsl; s0 += TM) {
            const int sl = s0 + team;
            double2 y = make_double2(0.0, 0.0);
            if (sl < nsl) {  // uniform over the wavefront
                const uint32_t ln = slen[sl * 64 + lane];
                cod_run_sum<REAL, kSmallTeam, 8, true, SH>(ent + sbase[sl], lds, xs, ln & 0xffff, par, y.x, y.y, ts);
                const int q0 = srbase[sl];
                cod_rest_sum<REAL, kSmallTeam, SH>(rcol + q0, rval + q0 * (REAL ? 1 : 2), xs, ln >> 16, par, y.x, y.y,
                                                   ts);
            }
            red[tid] = y;
            __syncthreads();
            if (par == 0 && sl * 64 + lane < n) {
#pragma unroll
                for (int q = 1; q < kSmallTeam; ++q) {
                    const double2 o = red[tid + q * 64];
                    y.x += o.x;
                    y.y += o.y;
                }
                ys[sl * 64 + lane] = y;
            }
            __syncthreads();
        }
        double2 u[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int r = tid + k * kSmallT;
            double dacc = 0.0;
            u[k] = make_double2(0.0, 0.0);
            if (r < n) {
                u[k] = lz_row(ys[r], dg[k], w[k], ib, j > 0, bj * ibp, wp[k]);
                dacc = re_dot(w[k], u[k]);
            }
            if (wv + 16 * k < nsl) {
                dacc = wave_total<64>(dacc);
                if (lane == 0) part[wv + 16 * k] = dacc;
            }
        }
        __syncthreads();
        const double pl = lane < nsl ? part[lane & (kSmallSlices - 1)] : 0.0;
        const double al = (nsl > 16 ? wave_total<32>(pl) : wave_total<16>(pl)) * ib;
        const double a = al * ib;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int r = tid + k * kSmallT;
            double acc = 0.0;
            const double2 v = lz_next(u[k], a, w[k], acc);
            wp[k] = w[k];
            w[k] = v;
            if (r < n) {
                W[(int64_t)(j + 1) * n + r] = v;
                xs[r] = v;
            }
            if (wv + 16 * k < nsl) {
                acc = wave_total<64>(r < n ? acc : 0.0);
                if (lane == 0) nrm[wv + 16 * k] = acc;
            }
        }
        __syncthreads();
        double t = 0.0;  // k_lz2's partial of 256 rows
        if (lane < gv) {
            t += nrm[4 * lane];
            t += nrm[4 * lane + 1];
            t += nrm[4 * lane + 2];
            t += nrm[4 * lane + 3];
        }
        const double b = sqrt(wave_total<8>(t));
        ibp = ib;
        ib = ZERO ? (b > 0 ? 1.0 / b : 0.0) : 1.0 / b;
        bj = b;
        if (tid == 0) {
            alpha[j] = al;
            beta[j + 1] = b;
            invb[j + 1] = ib;
            sal[j - j0] = al;
            sbe[j - j0] = b;
        }
    }
    if (mail) {  // a store to the host per step would be waited for in every step
        __syncthreads();
        if (tid < j1 - j0) post_mail(mail, j0 + tid, sal[tid], sbe[tid], tag0 | (uint64_t)(uint32_t)(j0 + tid + 1));
    }
}

}  // namespace blqh
