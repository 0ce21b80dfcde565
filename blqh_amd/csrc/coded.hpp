// coded.hpp -- the coded Hamiltonian layout of the SpMV hot loops (built in
// coded.hip) and its per-row sums.
//
// A matrix element is a sum of a few Coulomb table entries times a translation
// phase, so a sector's entries take few distinct values: the 1,023 most
// frequent magnitudes of a real sector and the 4,095 most frequent (|re|, |im|)
// pairs of a complex one cover 99 % of the entries and more (N_phi = 12: 99.2 /
// 99.4 %, N_phi = 14: 99.6 / 99.5 %, N_phi = 16 at half filling: 99.7 %).  Those
// values sit in a table that every workgroup holds in LDS, and an entry is one
// 32-bit word: column within its panel in the low 16 bits, table index above,
// sign of the real (and imaginary) part on top.  The matrix stream is 4 bytes an
// entry instead of 10 (real) or 18 (complex), and the values are the CSR's bit for
// bit, but for one case: a matrix whose imaginary parts are all at most 1e-14 of
// its largest entry is a real one (as for the panels), and those parts, the
// rounding of its phases, are left out.  Entries whose value is not in the
// table form the rest: 32-bit column and value, one run per 64-row slice.  The
// diagonal, whose values are nearly all different, is an array of its own.
//
// Order: columns in panels of 65,536, 64-row slices; run (panel, slice) is
// step-major: step t holds entry t of every row with more than t entries in the
// panel, rows in order, columns ascending in a row.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "common.hpp"
#include "panel.hpp"

namespace blqh {

constexpr int kCodReal = 1023;   // table entries of a real matrix (8 KiB of LDS), at most
constexpr int kCodCplx = 4095;   // of a complex one (64 KiB)
constexpr uint32_t kCodTun = 0x8000u;  // tunnelling flag of a shared-scale template's columns

struct Coded {
    bool built = false;
    bool real = false;
    int npan = 0;
    int ntab = 0;
    int64_t ncod = 0, nrest = 0;
    double* tab = nullptr;      // [ntab] |v| (an even number of places), or [2 ntab] (|re|, |im|)
    int64_t* base = nullptr;    // [npan * nslices + 1] first word of run p * nslices + s
    uint16_t* len = nullptr;    // [npan][nslices * 64] words of the row in the run
    uint32_t* ent = nullptr;    // [ncod]
    int64_t* rbase = nullptr;   // [nslices + 1]
    uint16_t* rlen = nullptr;   // [nslices * 64], behind len
    uint32_t* rcol = nullptr;   // [nrest]
    double* rval = nullptr;     // [nrest] or [2 nrest]
    double* diag = nullptr;     // [n] or [2 n]
    // where they lie: what the rows' number sizes, and what the entries' split does.  Two blocks,
    // since a block costs the build of a small matrix some 10 us to take and give back.
    DevBuf<char> rows, words;
};

struct CodView {
    int64_t n, nslices;
    int npan, ntab;
    const double* tab;
    const int64_t* base;
    const uint16_t* len;
    const uint32_t* ent;
    const int64_t* rbase;
    const uint16_t* rlen;
    const uint32_t* rcol;
    const double* rval;
    const double* diag;
};

inline CodView cview(const Coded& C, int64_t n) {
    return CodView{n,     (n + 63) >> 6, C.npan, C.ntab, C.tab,  C.base, C.len,
                   C.ent, C.rbase,       C.rlen, C.rcol, C.rval, C.diag};
}

__host__ __device__ inline size_t cod_lds_bytes(bool real, int ntab) {
    const size_t n = ntab > 0 ? ntab : 1;
    return real ? (n + 1) / 2 * 16 : n * 16;
}

// 16 bytes a lane from global memory straight to LDS, lane l to dst + l; complete
// after wait_vmem.  dst: uniform over the wavefront.
__device__ __forceinline__ void load_lds16(const double2* src, double2* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
__device__ __forceinline__ void wait_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The value of word e: magnitudes from the LDS table, signs from the top bits.
__device__ __forceinline__ double cod_sign(double v, uint32_t top) {  // top: sign in bit 31
    return __hiloint2double(__double2hiint(v) ^ (int)(top & 0x80000000u), __double2loint(v));
}
__device__ __forceinline__ double cod_real(const double* tab, uint32_t e) {
    return cod_sign(tab[(e >> 16) & 0x7fffu], e);
}
__device__ __forceinline__ double2 cod_cplx(const double2* tab, uint32_t e) {
    const double2 v = tab[(e >> 16) & 0x3fffu];
    return make_double2(cod_sign(v.x, e), cod_sign(v.y, e << 1));
}

// (ar, ai) += v x in four multiply-adds, in this order wherever a sum has to have the same
// bits in two kernels
__device__ __forceinline__ void cmac(double2 v, double2 x, double& ar, double& ai) {
    ar = fma(v.x, x.x, ar);
    ai = fma(v.x, x.y, ai);
    ar = fma(-v.y, x.y, ar);
    ai = fma(v.y, x.x, ai);
}

// diagonal element of a row
__device__ __forceinline__ double2 cod_diag(const CodView& C, bool real, int64_t row) {
    return real ? make_double2(C.diag[row], 0.0) : reinterpret_cast<const double2*>(C.diag)[row];
}

// Table to LDS, every load of a wavefront in flight at once (the caller waits, wait_vmem, and
// synchronises the workgroup).
template <bool REAL>
__device__ __forceinline__ void cod_stage(const double* __restrict__ tab, int ntab, double* lds, int nthreads) {
    const double2* t = reinterpret_cast<const double2*>(tab);
    double2* l = reinterpret_cast<double2*>(lds);
    const int n = REAL ? (ntab + 1) >> 1 : ntab, lane = threadIdx.x & 63;
    for (int i = threadIdx.x; i < n; i += nthreads) load_lds16(t + i, l + (i - lane));
}

// Sum of v over the wavefront's lanes (all active), the same on every lane.  A step's place in
// a run is such a sum; counted ballot by ballot over the other wavefronts' steps, those
// were half of the kernels' instructions, and a launch on a small matrix is as long as its
// instructions take to arrive: k_cod at 1,855 rows 8.5 -> 7.0 us, k_small's step at 205
// rows 10.9 -> 7.6.
__device__ __forceinline__ uint32_t lane_total(uint32_t v) {
    int t = (int)v;
    t += __builtin_amdgcn_update_dpp(0, t, 0x128, 0xf, 0xf, false);  // row_ror:8, 4, 2, 1
    t += __builtin_amdgcn_update_dpp(0, t, 0x124, 0xf, 0xf, false);
    t += __builtin_amdgcn_update_dpp(0, t, 0x122, 0xf, 0xf, false);
    t += __builtin_amdgcn_update_dpp(0, t, 0x121, 0xf, 0xf, false);
    return (uint32_t)(__builtin_amdgcn_readlane(t, 0) + __builtin_amdgcn_readlane(t, 16) +
                      __builtin_amdgcn_readlane(t, 32) + __builtin_amdgcn_readlane(t, 48));
}

// Row sums of one run: lane l owns row l (`len` words); the step groups (U
// steps each) are dealt to NP wavefronts, this one taking those with g mod NP
// == par.  The words of the next group are loaded before the x gathers of the
// current one, so a wavefront always has loads in flight.
// KEEP: the words are read again soon (small.hpp), leave them in the caches.  SH: values of
// words with the tunnelling flag are scaled by ts (columns have 15 bits).  ANY: x may hold
// infinities and NaN (the public product's), which a lane past its row's end, reading the
// panel's first entry, is not to multiply with its zero; the solvers' vectors are finite.
template <bool REAL, int NP, int U, bool KEEP = false, bool SH = false, bool ANY = false>
__device__ __forceinline__ void cod_run_sum(const uint32_t* __restrict__ er, const double* tab,
                                            const double2* __restrict__ xp, uint32_t len, int par, double& ar,
                                            double& ai, double ts = 1.0) {
    uint32_t off = 0;
    auto issue = [&](uint32_t t, uint32_t* e, bool& any) {
        uint64_t m[U];
#pragma unroll
        for (int u = 0; u < U; ++u) m[u] = __ballot(t + u < len);
        any = m[0] != 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t q = off + lanes_below(m[u]);
            off += (uint32_t)__popcll(m[u]);
            e[u] = t + u < len ? (KEEP ? er[q] : __builtin_nontemporal_load(&er[q])) : 0u;
        }
    };
    uint32_t e0[U], e1[U];
    bool any0, any1;
    uint32_t t0 = (uint32_t)(U * par);
    if (NP > 1) off = lane_total(t0 < len ? t0 : len);  // words of the steps before: the other wavefronts' groups
    issue(t0, e0, any0);
    while (any0) {
        const uint32_t t = t0 + (uint32_t)(U * NP);
        if (NP > 1) off = lane_total(t < len ? t : len);
        issue(t, e1, any1);
        double2 xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            xv[u] = xp[e0[u] & (SH ? kCodTun - 1 : 0xffffu)];
            if (ANY && !(t0 + u < len)) xv[u] = make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool act = t0 + u < len;
            if (REAL) {
                double v = act ? cod_real(tab, e0[u]) : 0.0;
                if (SH && (e0[u] & kCodTun)) v *= ts;
                ar = fma(v, xv[u].x, ar);
                ai = fma(v, xv[u].y, ai);
            } else {
                double2 v = cod_cplx(reinterpret_cast<const double2*>(tab), e0[u]);
                if (!act) v = make_double2(0.0, 0.0);
                if (SH && (e0[u] & kCodTun)) v = make_double2(ts * v.x, ts * v.y);
                cmac(v, xv[u], ar, ai);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) e0[u] = e1[u];
        any0 = any1;
        t0 = t;
    }
}

// Epilogue of a Lanczos row: u = y / beta_j - c q from its product's row y (the diagonal added
// here) and the previous vector's q (c = beta_j / beta_{j-1}; prev false at j = 0).
__device__ __forceinline__ double2 lz_row(double2 y, double2 dg, double2 w, double ib, bool prev, double c, double2 q) {
    cmac(dg, w, y.x, y.y);
    double ur = ib * y.x, ui = ib * y.y;
    if (prev) {
        ur = fma(-c, q.x, ur);
        ui = fma(-c, q.y, ui);
    }
    return make_double2(ur, ui);
}
__device__ __forceinline__ double re_dot(double2 a, double2 b) { return fma(a.x, b.x, a.y * b.y); }
// u - a w, and its |.|^2 added to acc
__device__ __forceinline__ double2 lz_next(double2 u, double a, double2 w, double& acc) {
    const double2 r = make_double2(fma(-a, w.x, u.x), fma(-a, w.y, u.y));
    acc = fma(r.x, r.x, fma(r.y, r.y, acc));
    return r;
}

// The rest of a slice: one step at a time (about one entry a row), step t to
// the wavefront t mod NP.
template <bool REAL, int NP, bool SH = false>
__device__ __forceinline__ void cod_rest_sum(const uint32_t* __restrict__ rc, const double* __restrict__ rv,
                                             const double2* __restrict__ x, uint32_t len, int par, double& ar,
                                             double& ai, double ts = 1.0) {
    uint32_t off = 0;
    for (uint32_t t = 0;; ++t) {
        const uint64_t m = __ballot(t < len);
        if (m == 0) break;
        if ((NP == 1 || (int)(t % NP) == par) && t < len) {
            const uint32_t q = off + lanes_below(m);
            const uint32_t c = rc[q];
            const double2 xv = x[SH ? c & (kCodTun - 1) : c];
            const double s = SH && (c & kCodTun) ? ts : 1.0;
            if (REAL) {
                const double v = SH ? s * rv[q] : rv[q];
                ar = fma(v, xv.x, ar);
                ai = fma(v, xv.y, ai);
            } else {
                double2 v = reinterpret_cast<const double2*>(rv)[q];
                if (SH) v = make_double2(s * v.x, s * v.y);
                cmac(v, xv, ar, ai);
            }
        }
        off += (uint32_t)__popcll(m);
    }
}

}  // namespace blqh
