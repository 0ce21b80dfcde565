// batch.hip -- many Lanczos ground-state solves advanced together.
//
// Ancestor: the reference's serial sweeps over sectors and parameter points
// (BLQH_without_spin/main.cpp:76-165, BLQH_with_spin/main.cpp:158-302), each
// of which runs lhamil's three passes (lanczos_hamiltonian.cpp:453-656) on one
// Hamiltonian at a time.  Here every problem of a batch (one resident
// Hamiltonian + one start vector) takes Lanczos step j in the same two
// launches:
//   K1  u = (H W_j)/beta_j - (beta_j/beta_{j-1}) W_{j-1},  alpha partials
//   K2  alpha_j = sum of the problem's K1 partials (fixed order),
//       W_{j+1} = u - alpha_j W_j / beta_j,               |W_{j+1}|^2 partials
//   K3  beta_{j+1} = sqrt(sum of the K2 partials)          (one wave per problem)
// The rows of every problem are cut into work items of kItemRows rows; a
// persistent grid walks the item list, so problems of any size share one
// launch and each item's partial sum has a fixed owner (bit-reproducible).
// Kernels read the step from a device counter and skip problems whose active
// flag is clear, so `check_every` steps are captured once in a hipGraph and
// replayed; between replays the host reads alpha/beta of every problem,
// runs the convergence test of the single-problem solver and clears the flags
// of the converged ones (data-dependent termination without a host round trip
// per step).  The Krylov vectors of every problem stay in HBM, so the ground
// state is one weighted sum per problem afterwards (no replay pass); the same
// pass forms the excited mix (second and third Ritz vectors), and both stay
// on the device in the reference row order as the start of a continuation
// solve at the next parameter point (k_bcont).  A batch of small members only
// takes its steps in one workgroup per problem instead (k_bsmall, small.hpp).
#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>

#include "ritz.hpp"
#include "engine.hpp"
#include "mtstart.hpp"
#include "small.hpp"
#include "xcdplan.hpp"

namespace blqh {
void start_vector(int64_t n, uint32_t seed, std::vector<double2>& v);
double tridiag_lowest(int m, const double* a, const double* b, double* vec);
double tridiag_lowest_next(int m, const double* a, const double* b, double prev, double step);
}  // namespace blqh
void blqh_hamil_combine_impl(const blqh_hamil* base, const blqh_hamil* tun, double dsas, blqh_hamil* H, bool formats);

namespace {

using namespace blqh;

constexpr int kItemRows = 256;  // rows per work item
constexpr int kBT = 256;        // threads per workgroup
constexpr int kSplit = 2;       // k_b1j: wavefronts per 64-row slice (measured: 2 beats 1 and 4)
constexpr int kBTj = kSplit * 256;  // threads per workgroup of k_b1j (an item's four slices)

// A one-panel coded layout regrouped for k_b1x: by 64-row slice, then column tile of
// tw columns, then groups of four steps; a group holds four words of every lane
// (ent[group * 64 + lane]), rows shorter than the slice's longest in that tile
// padded with words of value zero.  Tile t of slice s is groups goff[s nt + t] ..
// goff[s nt + t + 1).
struct ColTiles {
    int tw, nt;
    const uint4* ent;
    const int64_t* goff;
};

// device descriptor of one problem
struct BProb {
    int64_t n;
    int32_t npan, real;
    CodView c;              // coded layout: k_b1x, k_b1j
    ColTiles t;            // its column tiles: k_b1x
    const int64_t* pbase;   // panels: k_b1
    const uint32_t* prow;
    const uint16_t* pcol;
    const double* pvr;
    const double2* pvc;
    int64_t item0;  // first work item
    int64_t voff;   // row offset in the pooled vectors
    double2* W;     // Krylov block: W_0 .. W_cap, n each
};

// per-step device state
struct BState {
    const BProb* probs;
    const int32_t* item_prob;  // work item -> problem
    int64_t nitems;
    const int32_t* xitems;     // work lists of k_b1j (items) and k_b1x (units) per XCD (real, complex, all members)
    const int32_t* xseg;       // [3][9] list offsets: kind (real, complex, all) x XCD
    const int32_t* active;     // [P]
    int32_t* jbase;            // step of the first kernel in a replay (advanced by k_bnext)
    int cap;                   // lambda
    double* alpha;             // [P][cap]
    double* beta;              // [P][cap + 1], beta[p][0] = 1
    double* invb;              // [P][cap + 1]
    double2* u;                // pooled rows
    double* part1;             // [nitems]
    double* part2;             // [nitems]
};

template <int NT = kBT>
__device__ __forceinline__ double block_sum(double v, double* sh) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
    for (int w = 0; w < NT / 64; ++w) t += sh[w];
    return t;
}

// sum of part[i0 .. i0+cnt) by one wavefront in a fixed order; every lane
// returns the same bits (the butterfly adds commutative pairs)
__device__ __forceinline__ double wave_sum(const double* part, int64_t i0, int64_t cnt, int lane) {
    double s = 0;
    for (int64_t i = lane; i < cnt; i += 64) s += part[i0 + i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}

// y_r = sum_k H_rk x_k for one row, LPR lanes (panel storage, any panel count)
template <int LPR>
__device__ __forceinline__ double2 prow_dot(const BProb& P, const double2* __restrict__ x, int64_t r, int lane) {
    double re = 0.0, im = 0.0;
    for (int pan = 0; pan < P.npan; ++pan) {
        const uint32_t* rp = P.prow + (int64_t)pan * (P.n + 1);
        const uint32_t s = rp[r], e = rp[r + 1];
        const int64_t base = P.pbase[pan];
        const double2* xp = x + (int64_t)pan * kPanelWidth;
        if (P.real) {
            for (uint32_t k = s + lane; k < e; k += LPR) {
                const int c = __builtin_nontemporal_load(&P.pcol[base + k]);
                const double v = __builtin_nontemporal_load(&P.pvr[base + k]);
                const double2 xv = xp[c];
                re += v * xv.x;
                im += v * xv.y;
            }
        } else {
            for (uint32_t k = s + lane; k < e; k += LPR) {
                const int c = __builtin_nontemporal_load(&P.pcol[base + k]);
                const double2 v = P.pvc[base + k];
                const double2 xv = xp[c];
                re += v.x * xv.x - v.y * xv.y;
                im += v.x * xv.y + v.y * xv.x;
            }
        }
    }
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) {
        re += __shfl_xor(re, o, LPR);
        im += __shfl_xor(im, o, LPR);
    }
    return make_double2(re, im);
}

// K1 (LZ) or a plain product y = H x with partial Re<x|y> (!LZ: x and y are
// the pooled vectors xs / ys).
template <int LPR, bool LZ>
__global__ void __launch_bounds__(kBT) k_b1(BState S, int jrel, const double2* __restrict__ xs,
                                            double2* __restrict__ ys, double* __restrict__ part) {
    __shared__ double sh[kBT / 64];
    const int j = LZ ? *S.jbase + jrel : 0;
    if (LZ && j >= S.cap) return;
    constexpr int RPP = kBT / LPR;
    const int sub = threadIdx.x / LPR, lane = threadIdx.x % LPR;
    for (int64_t it = blockIdx.x; it < S.nitems; it += gridDim.x) {
        const int p = S.item_prob[it];
        if (!S.active[p]) continue;  // uniform over the workgroup
        const BProb P = S.probs[p];
        const int64_t r0 = (it - P.item0) * kItemRows;
        const int64_t r1 = r0 + kItemRows < P.n ? r0 + kItemRows : P.n;
        const double2* x;
        double2* y;
        const double2* Wp = nullptr;
        double ib = 1.0, cp = 0.0;
        if (LZ) {
            const int64_t ld = S.cap + 1;
            ib = S.invb[p * ld + j];
            cp = j > 0 ? S.beta[p * ld + j] * S.invb[p * ld + j - 1] : 0.0;
            x = P.W + (int64_t)j * P.n;
            Wp = j > 0 ? x - P.n : x;
            y = S.u + P.voff;
        } else {
            x = xs + P.voff;
            y = ys + P.voff;
        }
        double acc = 0.0;
        for (int64_t r = r0 + sub; r < r1; r += RPP) {
            const double2 h = prow_dot<LPR>(P, x, r, lane);
            if (lane == 0) {
                double ur = h.x, ui = h.y;
                if (LZ) {
                    ur = ib * h.x;
                    ui = ib * h.y;
                    if (j > 0) {
                        const double2 q = Wp[r];
                        ur -= cp * q.x;
                        ui -= cp * q.y;
                    }
                }
                y[r] = make_double2(ur, ui);
                const double2 w = x[r];
                acc += w.x * ur + w.y * ui;
            }
        }
        const double t = block_sum(acc, sh);
        if (threadIdx.x == 0) part[it] = t;
    }
}

// Workgroup's share of its XCD's work list: workgroups reach the XCDs round
// robin (workgroup b on XCD b mod 8, grid a multiple of 8) and each takes a
// stretch of consecutive items, so that it stays with one member's value table
// and its XCD gathers from the x vectors of few members at a time.
__device__ __forceinline__ void list_share(const int32_t* seg, int32_t& k0, int32_t& k1) {
    const int32_t s0 = seg[0], cnt = seg[1] - s0, nb = (int32_t)(gridDim.x >> 3), b = (int32_t)(blockIdx.x >> 3);
    k0 = s0 + (int32_t)((int64_t)cnt * b / nb);
    k1 = s0 + (int32_t)((int64_t)cnt * (b + 1) / nb);
}

// Same contract as k_b1 over the coded layout: kSplit wavefronts
// per 64-row slice of the item (waves kSplit*s .. kSplit*s + kSplit-1 own
// slice s, one lane per row), each summing every kSplit-th step group
// (cod_run_sum); the partial sums of waves 1.. go through LDS to wave 0
// of the slice, which adds them in wave order and runs the K1 epilogue.  KIND 0 / 1 walk only the members with real / complex
// values, KIND 2 walks all members and branches per work item (one launch per
// step for a mixed batch, so that the members of both kinds run side by side).
template <bool LZ, int KIND>
__global__ void __launch_bounds__(kBTj) k_b1j(BState S, int jrel, const double2* __restrict__ xs,
                                              double2* __restrict__ ys, double* __restrict__ part) {
    __shared__ double sh[kBTj / 64];
    __shared__ double2 red[kItemRows / 64][kSplit - 1][64];  // partial row sums of waves 1.. of each slice
    extern __shared__ __align__(16) double ctab[];
    const int j = LZ ? *S.jbase + jrel : 0;
    if (LZ && j >= S.cap) return;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int sl = wv / kSplit, par = wv % kSplit;
    int32_t k0, k1;
    list_share(S.xseg + KIND * 9 + (blockIdx.x & 7), k0, k1);
    int pt = -1;  // member whose value table is in LDS
    for (int32_t k = k0; k < k1; ++k) {
        const int64_t it = S.xitems[k];
        const int p = S.item_prob[it];
        if (!S.active[p]) continue;  // uniform over the workgroup
        const BProb P = S.probs[p];
        const bool real = KIND == 2 ? P.real != 0 : KIND == 0;
        if (p != pt) {
            __syncthreads();  // the previous member's table is no longer read
            if (real) cod_stage<true>(P.c.tab, P.c.ntab, ctab, kBTj);
            else cod_stage<false>(P.c.tab, P.c.ntab, ctab, kBTj);
            wait_vmem();
            __syncthreads();
            pt = p;
        }
        const double2* x;
        double2* y;
        const double2* Wp = nullptr;
        double ib = 1.0, cp = 0.0;
        if (LZ) {
            const int64_t ld = S.cap + 1;
            ib = S.invb[p * ld + j];
            cp = j > 0 ? S.beta[p * ld + j] * S.invb[p * ld + j - 1] : 0.0;
            x = P.W + (int64_t)j * P.n;
            Wp = j > 0 ? x - P.n : x;
            y = S.u + P.voff;
        } else {
            x = xs + P.voff;
            y = ys + P.voff;
        }
        const int64_t n = P.n;
        const int64_t row0 = (it - P.item0) * kItemRows + sl * 64, myrow = row0 + lane;
        double ar = 0.0, ai = 0.0;
        if (row0 < n) {  // uniform over the wavefront
            const int64_t slc = row0 >> 6;
            for (int pan = 0; pan < P.npan; ++pan) {
                const int64_t run = (int64_t)pan * P.c.nslices + slc;
                const double2* xp = x + (int64_t)pan * kPanelWidth;
                const uint32_t len = P.c.len[run * 64 + lane];
                if (real) cod_run_sum<true, kSplit, 4>(P.c.ent + P.c.base[run], ctab, xp, len, par, ar, ai);
                else cod_run_sum<false, kSplit, 4>(P.c.ent + P.c.base[run], ctab, xp, len, par, ar, ai);
            }
            const int64_t q0 = P.c.rbase[slc];
            const uint32_t rl = P.c.rlen[myrow];
            if (real) cod_rest_sum<true, kSplit>(P.c.rcol + q0, P.c.rval + q0, x, rl, par, ar, ai);
            else cod_rest_sum<false, kSplit>(P.c.rcol + q0, P.c.rval + 2 * q0, x, rl, par, ar, ai);
        }
        if (par) red[sl][par - 1][lane] = make_double2(ar, ai);
        __syncthreads();
        double acc = 0.0;
        if (!par && myrow < n) {
#pragma unroll
            for (int q = 0; q < kSplit - 1; ++q) {
                const double2 o = red[sl][q][lane];
                ar += o.x;
                ai += o.y;
            }
            const double2 w = x[myrow], dg = cod_diag(P.c, real, myrow);
            ar += dg.x * w.x - dg.y * w.y;
            ai += dg.x * w.y + dg.y * w.x;
            double ur = ar, ui = ai;
            if (LZ) {
                ur = ib * ar;
                ui = ib * ai;
                if (j > 0) {
                    const double2 q = Wp[myrow];
                    ur -= cp * q.x;
                    ui -= cp * q.y;
                }
            }
            y[myrow] = make_double2(ur, ui);
            acc = w.x * ur + w.y * ui;
        }
        const double t = block_sum<kBTj>(acc, sh);
        if (threadIdx.x == 0) part[it] = t;
    }
}

// ---- K1 with x in LDS -------------------------------------------------------
// For members of one panel.  The x gathers bound k_b1j: the vector memory path
// serves about one 16-byte lane address per clock and CU (0.75 measured), LDS a
// wavefront's 64 in about 20 clocks.  So a workgroup of 16 wavefronts (one per CU:
// it takes the whole LDS) owns a unit of 16 slices (fewer in batches of few members,
// batch_team), stages x tile by tile beside the value table and sums its slices' words of
// that tile from LDS.  The tiles are as
// wide as the LDS allows (8,192 columns of one vector at most), so a unit of an
// 18.8k-row member stages 300 KB for 158k entries.  With x in LDS the address
// arithmetic counts: a word's fields are LDS byte offsets (one mask each), rows are
// padded to their slice's longest (no lane masks or prefix sums) and a lane loads
// four words at once.
//
// Shared-scale groups (SH): G problems of one sector whose Hamiltonians are
// H0 + s_g T (the Delta_SAS points of one d) share one coded layout of H0 + T: the
// entries of T (those between words of different upper-layer occupation) carry the
// tunnelling flag (a sector of at most 32,768 states), and problem
// g scales them by s_g.  One pass over the entries serves all G problems: an
// entry's word and value are read once and multiplied with G tiles.
//
// Bound by vector-ALU work per padded word (decode, sign, two to four 64-bit
// multiply-adds) and, in sweeps, by the staging of x and the barrier around it (about
// half at G = 3); bank conflicts cost nothing measurable (a conflict-free order of
// the words took the same time).  K1 with every member live, jagged panels gathering
// x -> this: 64 spinful N_phi = 8 sectors 446 -> 193 us, N_phi = 12 sweep, 144 sectors
// at three scales, 2,393 -> 1,203 us.
//
// Word: bit 31 / 30 sign of the real / imaginary part, bits 17..28 index of the
// value in the LDS table (0: the value zero), bits 4..16 column in the tile, bit 0
// the tunnelling flag.
constexpr int kBTx = kUnit * 64;
constexpr int kUnitItems = kUnit * 64 / kItemRows;
constexpr size_t kLdsMax = 160 * 1024 - 1024;  // dynamic LDS; the rest is k_b1x's static part
constexpr size_t kLdsHalf = 79 * 1024;
constexpr int kTileMax = 8192;         // columns of a tile (13 bits)

// An element of k_b1x's work list names an owner (a problem; SH: a group) and, counted
// in elements, the place in it: owner << kElemBits | element.  An element is `span`
// (S.xseg[27], 1 or 2; 1 with teams) consecutive units (xcdplan.hpp).
constexpr int kElemBits = 8;  // at most 256 units of a one-panel member
// sums of a slice's later wavefronts, which take the tile's place
constexpr size_t kTeamLds = kBTx / kTeamMax * (kTeamMax - 1) * sizeof(double2);
static_assert(kLdsHalf >= 4096 * sizeof(double2) + kTeamLds, "team sums fit beside the largest table");

// LDS bytes of the table: the value zero, then the layout's values
__host__ __device__ inline size_t tile_tab_bytes(bool real, int ntab) {
    return ((size_t)(ntab + 1) * (real ? 8 : 16) + 15) / 16 * 16;
}

__device__ __forceinline__ double with_sign(double mag, uint32_t top) {  // mag >= 0, sign in bit 31
    return __hiloint2double((int)((uint32_t)__double2hiint(mag) | (top & 0x80000000u)), __double2loint(mag));
}

// (ar, ai) += (wr, wi) xv in four multiply-adds
__device__ __forceinline__ void cfma(double wr, double wi, double2 xv, double& ar, double& ai) {
    ar = fma(wr, xv.x, ar);
    ai = fma(wr, xv.y, ai);
    ar = fma(-wi, xv.y, ar);
    ai = fma(wi, xv.x, ai);
}

// the rest of a slice, x in global memory; four steps of loads in flight
template <bool REAL, int G, bool SH>
__device__ __forceinline__ void tile_rest_sum(const uint32_t* __restrict__ rc, const double* __restrict__ rv,
                                              const double2* const* x, const double* ts, uint32_t len, double* ar,
                                              double* ai) {
    constexpr int U = 4;
    uint32_t off = 0;
    for (uint32_t t = 0; __ballot(t < len) != 0; t += U) {
        uint32_t c[U];
        double2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t m = __ballot(t + u < len);
            const uint32_t q = off + lanes_below(m);
            off += (uint32_t)__popcll(m);
            c[u] = 0;
            v[u] = make_double2(0.0, 0.0);
            if (t + u < len) {
                c[u] = rc[q];
                v[u] = REAL ? make_double2(rv[q], 0.0) : reinterpret_cast<const double2*>(rv)[q];
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            double2 xv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) xv[u] = x[g][SH ? c[u] & (kCodTun - 1) : c[u]];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (!(t + u < len)) continue;
                const double sc = SH && (c[u] & kCodTun) ? ts[g] : 1.0;
                if (REAL) {
                    ar[g] = fma(sc * v[u].x, xv[u].x, ar[g]);
                    ai[g] = fma(sc * v[u].x, xv[u].y, ai[g]);
                } else {
                    cfma(sc * v[u].x, sc * v[u].y, xv[u], ar[g], ai[g]);
                }
            }
        }
    }
}

// SC: some lane's word carries the tunnelling flag
template <bool REAL, int G, bool SC>
__device__ __forceinline__ void tile_fma(uint32_t e, const char* lds, uint32_t xbase, uint32_t xstep, const double* ts,
                                         double* ar, double* ai) {
    double vr, vi = 0.0;
    if (REAL) {
        vr = with_sign(*reinterpret_cast<const double*>(lds + ((e >> 14) & 0x7ff8u)), e);
    } else {
        const double2 v = *reinterpret_cast<const double2*>(lds + ((e >> 13) & 0xfff0u));
        vr = with_sign(v.x, e);
        vi = with_sign(v.y, e << 1);
    }
    const char* xp = lds + xbase + (e & 0x1fff0u);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const double2 xv = *reinterpret_cast<const double2*>(xp + (uint32_t)g * xstep);
        double wr = vr, wi = vi;
        if (SC) {
            const double sc = (e & 1u) ? ts[g] : 1.0;
            wr *= sc;
            wi *= sc;
        }
        if (REAL) {
            ar[g] = fma(wr, xv.x, ar[g]);
            ai[g] = fma(wr, xv.y, ai[g]);
        } else {
            cfma(wr, wi, xv, ar[g], ai[g]);
        }
    }
}

// A wavefront's words of one tile: K groups, NP apart, from ent, two groups loaded ahead (a0
// and a1 hold the first two).  A row's flagged words come first, so most groups have none.
template <bool REAL, int G, bool SH, int NP>
__device__ __forceinline__ void tile_sum(const uint4* __restrict__ ent, uint32_t K, uint4 a0, uint4 a1, const char* lds,
                                         uint32_t xbase, uint32_t xstep, const double* ts, double* ar, double* ai) {
    for (uint32_t k = 0; k < K; ++k) {
        const uint4 e = a0;
        a0 = a1;
        if (k + 2 < K) a1 = ent[(k + 2) * (64 * NP)];
        if (SH && __ballot(((e.x | e.y | e.z | e.w) & 1u) != 0)) {
            tile_fma<REAL, G, true>(e.x, lds, xbase, xstep, ts, ar, ai);
            tile_fma<REAL, G, true>(e.y, lds, xbase, xstep, ts, ar, ai);
            if (G > 1) __builtin_amdgcn_sched_barrier(0);  // two words' LDS reads in flight: no spills
            tile_fma<REAL, G, true>(e.z, lds, xbase, xstep, ts, ar, ai);
            tile_fma<REAL, G, true>(e.w, lds, xbase, xstep, ts, ar, ai);
        } else {
            tile_fma<REAL, G, false>(e.x, lds, xbase, xstep, ts, ar, ai);
            tile_fma<REAL, G, false>(e.y, lds, xbase, xstep, ts, ar, ai);
            if (G > 1) __builtin_amdgcn_sched_barrier(0);
            tile_fma<REAL, G, false>(e.z, lds, xbase, xstep, ts, ar, ai);
            tile_fma<REAL, G, false>(e.w, lds, xbase, xstep, ts, ar, ai);
        }
    }
}

// Values that are the same on every lane, into scalar registers (the kernel writes
// memory, so the compiler keeps what it loads per owner in vector ones).
__device__ __forceinline__ int sgpr(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t sgpr(int64_t v) {
    return (int64_t)((uint64_t)(uint32_t)sgpr((int)(v >> 32)) << 32 | (uint32_t)sgpr((int)v));
}
__device__ __forceinline__ double sgpr(double v) { return __longlong_as_double(sgpr((int64_t)__double_as_longlong(v))); }
template <class T>
__device__ __forceinline__ T* sgpr(T* p) {
    return reinterpret_cast<T*>(sgpr((int64_t)reinterpret_cast<uintptr_t>(p)));
}

// Problem p0 + g, g < G, of an owner (SH: p0 = owner G; else G = 1, p0 = owner);
// problem p's item li is item0 + li, as in k_b2 / k_b3.  A stopped problem of a
// live group is summed along and not written.  NP: wavefronts of a slice (batch_team); they
// take its groups of a tile in turn, and the first adds the others' sums in their order.
template <bool LZ, int G, bool SH, int NP>
__global__ void __launch_bounds__(kBTx) k_b1x(BState S, const double* __restrict__ tscale, int jrel,
                                              const double2* __restrict__ xs, double2* __restrict__ ys,
                                              double* __restrict__ part) {
    constexpr int NS = kUnit / NP;       // slices of a unit
    constexpr int NQ = NP == 1 ? 2 : 1;  // units of an element at most
    constexpr int NI = kUnitItems / NP;  // items of a unit
    extern __shared__ __align__(16) double ctab[];
    __shared__ double red[NQ][G][NS];
    const int j = LZ ? *S.jbase + jrel : 0;
    if (LZ && j >= S.cap) return;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, ws = wv / NP, par = wv % NP;
    const char* lds = reinterpret_cast<const char*>(ctab);
    // The XCD's workgroups walk its list side by side (unlike k_b1j's stretches):
    // they stage the x of the same one or two owners, out of the L2.
    const int32_t* seg = S.xseg + 2 * 9 + (blockIdx.x & 7);
    const int span = sgpr(S.xseg[27]);
    int ot = -1;  // owner whose value table is in LDS
    for (int32_t k = seg[0] + (int32_t)(blockIdx.x >> 3), k1 = seg[1]; k < k1; k += (int32_t)(gridDim.x >> 3)) {
        const int32_t id = sgpr(S.xitems[k]);
        const int o = id >> kElemBits, p0 = SH ? o * G : o;
        bool act[G], any = false;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            act[g] = sgpr(S.active[p0 + g]) != 0;
            any = any || act[g];
        }
        if (!any) continue;  // uniform over the workgroup
        const BProb& P = S.probs[p0];
        const int64_t n = sgpr(P.n), nsl = (n + 63) >> 6;
        const bool real = sgpr(P.real) != 0;
        const int ntab = sgpr(P.c.ntab), tw = sgpr(P.t.tw), nt = sgpr(P.t.nt);
        const uint4* tent = sgpr(P.t.ent);
        const int64_t* goff = sgpr(P.t.goff);
        const uint32_t xbase = (uint32_t)tile_tab_bytes(real, ntab), xstep = (uint32_t)tw * 16u;
        double2* xt = reinterpret_cast<double2*>(reinterpret_cast<char*>(ctab) + xbase);
        const double2* x[G];
        double ts[G], ar[NQ][G], ai[NQ][G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const BProb& Pg = S.probs[p0 + g];
            x[g] = sgpr(LZ ? Pg.W + (int64_t)j * n : xs + Pg.voff);
            ts[g] = SH ? sgpr(tscale[p0 + g]) : 1.0;
#pragma unroll
            for (int q = 0; q < NQ; ++q) ar[q][g] = ai[q][g] = 0.0;
        }
        const int32_t u0 = (id & ((1 << kElemBits) - 1)) * span;  // the element's first unit
        const int64_t sl0 = (int64_t)u0 * NS + ws;                // this wavefront's slices: sl0, sl0 + NS
        for (int t = 0; t < nt; ++t) {
            // the first words are on their way while the tile is staged
            uint32_t K[NQ];
            const uint4* ent[NQ];
            uint4 a0[NQ], a1[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int64_t sl = sl0 + q * NS;
                const bool mine = q < span && sl < nsl;  // uniform over the wavefront
                const int64_t g0 = mine ? goff[sl * nt + t] : 0;
                K[q] = mine ? (uint32_t)(goff[sl * nt + t + 1] - g0) : 0u;
                if (NP > 1) K[q] = K[q] > (uint32_t)par ? (K[q] - par + NP - 1) / NP : 0u;
                ent[q] = tent + (g0 + par) * 64 + lane;
                a0[q] = a1[q] = make_uint4(0, 0, 0, 0);
                if (K[q] > 0) a0[q] = ent[q][0];
                if (K[q] > 1) a1[q] = ent[q][64 * NP];
            }
            __syncthreads();  // the previous tile (and table) is no longer read
            if (o != ot) {
                if (real) {
                    for (int i = threadIdx.x; i <= ntab; i += kBTx) ctab[i] = i ? P.c.tab[i - 1] : 0.0;
                } else {
                    const double2* t2 = reinterpret_cast<const double2*>(P.c.tab);
                    double2* l2 = reinterpret_cast<double2*>(ctab);
                    for (int i = threadIdx.x; i <= ntab; i += kBTx) l2[i] = i ? t2[i - 1] : make_double2(0.0, 0.0);
                }
                ot = o;
            }
            const int64_t c0 = (int64_t)t * tw;
            const int w = (int)(n - c0 < tw ? n - c0 : tw);
#pragma unroll
            for (int g = 0; g < G; ++g)
                for (int i = threadIdx.x; i < w; i += kBTx)
                    load_lds16(&x[g][c0 + i], xt + g * tw + (i - lane));
            wait_vmem();
            __syncthreads();
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                if (real) tile_sum<true, G, SH, NP>(ent[q], K[q], a0[q], a1[q], lds, xbase, xstep, ts, ar[q], ai[q]);
                else tile_sum<false, G, SH, NP>(ent[q], K[q], a0[q], a1[q], lds, xbase, xstep, ts, ar[q], ai[q]);
            }
        }
        if (NP > 1) {  // the team's sums, over the tile (at most 12 KiB, kTeamLds)
#pragma unroll
            for (int g = 0; g < G; ++g) {
                double2* const sum = xt + (ws * (NP - 1) - 1) * 64 + lane;  // of wavefront par: sum[par * 64]
                __syncthreads();  // the tile, or the previous sums, are read
                if (par) sum[par * 64] = make_double2(ar[0][g], ai[0][g]);
                __syncthreads();
                if (!par) {
#pragma unroll
                    for (int w = 1; w < NP; ++w) {
                        ar[0][g] += sum[w * 64].x;
                        ai[0][g] += sum[w * 64].y;
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int64_t sl = sl0 + q * NS, row = sl * 64 + lane;
            const bool slice = q < span && sl < nsl && par == 0, mine = slice && row < n;
            if (slice) {
                const int64_t q0 = P.c.rbase[sl];
                const uint32_t rl = P.c.rlen[row];
                if (real) tile_rest_sum<true, G, SH>(P.c.rcol + q0, P.c.rval + q0, x, ts, rl, ar[q], ai[q]);
                else tile_rest_sum<false, G, SH>(P.c.rcol + q0, P.c.rval + 2 * q0, x, ts, rl, ar[q], ai[q]);
            }
            const double2 dg = mine ? cod_diag(P.c, real, row) : make_double2(0.0, 0.0);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                double acc = 0.0;
                if (act[g] && mine) {
                    double2* y = (LZ ? S.u : ys) + S.probs[p0 + g].voff;
                    double yr = ar[q][g], yi = ai[q][g];
                    const double2 w = x[g][row];
                    cfma(dg.x, dg.y, w, yr, yi);
                    if (LZ) {
                        const int64_t ld = S.cap + 1;
                        const int p = p0 + g;
                        const double ib = S.invb[p * ld + j];
                        yr *= ib;
                        yi *= ib;
                        if (j > 0) {
                            const double cp = S.beta[p * ld + j] * S.invb[p * ld + j - 1];
                            const double2 wp = x[g][row - n];  // W_{j-1}
                            yr -= cp * wp.x;
                            yi -= cp * wp.y;
                        }
                    }
                    y[row] = make_double2(yr, yi);
                    acc = w.x * yr + w.y * yi;
                }
                for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d, 64);
                if (lane == 0 && par == 0) red[q][g][ws] = acc;
            }
        }
        __syncthreads();
        if (threadIdx.x < NQ * G * NI) {  // item partials: its four slices in order
            const int q = threadIdx.x / (G * NI), g = threadIdx.x / NI % G, m = threadIdx.x % NI;
            const int64_t li = (int64_t)(u0 + q) * NI + m;
            if (q < span && S.active[p0 + g] && li * kItemRows < n) {
                double t = 0;
                for (int i = 0; i < kItemRows / 64; ++i) t += red[q][g][m * (kItemRows / 64) + i];
                part[S.probs[p0 + g].item0 + li] = t;
            }
        }
    }
}

// Coded words of one-panel members regrouped into ColTiles, one wavefront per slice,
// grid.y = member: first (FILL false) each tile's groups into cnt, then the words
// (goff: the scanned counts of all members).  LDS: words per tile and lane, and
// per step of the slice its first word and the lanes that hold one.
struct TileJob {
    CodView c;
    int tw, nt;
    int real;
    uint32_t cmask;  // column bits of a coded word
    int64_t goff0;   // this member's first (slice, tile)
};

template <bool FILL>
__global__ void __launch_bounds__(64) k_tiles(const TileJob* __restrict__ jobs, int maxrow, int maxnt,
                                              int32_t* __restrict__ cnt, const int64_t* __restrict__ goff,
                                              uint4* __restrict__ ent) {
    extern __shared__ uint64_t lds_tiles[];
    uint64_t* mk = lds_tiles;
    uint32_t* so = reinterpret_cast<uint32_t*>(mk + (FILL ? maxrow : 0));
    uint16_t* tc = reinterpret_cast<uint16_t*>(so + (FILL ? maxrow : 0));  // [maxnt][64]
    const TileJob J = jobs[blockIdx.y];
    const int lane = threadIdx.x;
    const uint64_t below = lane ? ~0ull >> (64 - lane) : 0;
    const int64_t nsl = J.c.nslices;
    for (int64_t sl = blockIdx.x; sl < nsl; sl += gridDim.x) {
        const uint32_t len = J.c.len[sl * 64 + lane];
        const uint32_t* src = J.c.ent + J.c.base[sl];
        __syncthreads();  // the previous slice's steps are read
        uint32_t off = 0, nw = 0, end = (uint32_t)J.tw;
        int cur = 0;
        for (uint32_t i = 0; i < (uint32_t)maxrow; ++i) {
            const uint64_t m = __ballot(i < len);
            if (m == 0) break;
            if (FILL && lane == 0) {
                mk[i] = m;
                so[i] = off;
            }
            if (i < len) {
                const uint32_t c = src[off + (uint32_t)__popcll(m & below)] & J.cmask;
                for (; c >= end && cur < J.nt - 1; ++cur) {
                    tc[cur * 64 + lane] = (uint16_t)nw;
                    nw = 0;
                    end += (uint32_t)J.tw;
                }
                ++nw;
            }
            off += (uint32_t)__popcll(m);
        }
        for (; cur < J.nt; ++cur) {
            tc[cur * 64 + lane] = (uint16_t)nw;
            nw = 0;
        }
        __syncthreads();
        uint32_t first = 0;
        for (int t = 0; t < J.nt; ++t) {
            const uint32_t ln = tc[t * 64 + lane];
            const int64_t at = J.goff0 + sl * J.nt + t;
            if (!FILL) {
                uint32_t mx = ln;
                for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, 64));
                if (lane == 0) cnt[at] = (int32_t)((mx + 3) / 4);
                continue;
            }
            const int64_t g0 = goff[at], K = goff[at + 1] - g0;
            const uint32_t sub = (uint32_t)t * (uint32_t)J.tw;
            uint32_t* out = reinterpret_cast<uint32_t*>(ent + g0 * 64 + lane);  // word k: out[(k / 4) * 256 + k % 4]
            auto word = [&](uint32_t i) { return src[so[i] + (uint32_t)__popcll(mk[i] & below)]; };
            uint32_t nt = 0, pt = 0;  // flagged words of the lane, and those placed
            for (uint32_t i = 0; i < ln; ++i) nt += (word(first + i) & ~J.cmask & kCodTun) != 0;
            for (uint32_t i = 0; i < ln; ++i) {
                const uint32_t w = word(first + i);
                const bool tun = (w & ~J.cmask & kCodTun) != 0;
                const uint32_t id = ((w >> 16) & (J.real ? 0x7fffu : 0x3fffu)) + 1;
                const uint32_t k = tun ? pt : nt + i - pt;
                pt += tun;
                out[(k >> 2) * 256 + (k & 3)] = (w & (J.real ? 0x80000000u : 0xc0000000u)) | id << 17 |
                                                ((w & J.cmask) - sub) << 4 | (uint32_t)tun;
            }
            for (uint32_t k = ln; k < (uint32_t)K * 4; ++k) out[(k >> 2) * 256 + (k & 3)] = 0;
            first += ln;
        }
    }
}

// ---- steps of small members ----------------------------------------------------
// Steps j0 .. j1 - 1 of every live problem, a workgroup each (small.hpp).
template <bool RES, bool SH>
__global__ void __launch_bounds__(kSmallT) k_bsmall(BState S, const double* __restrict__ tscale, int j0, int j1) {
    extern __shared__ __align__(16) double ctab[];
    const int p = blockIdx.x;
    if (!S.active[p]) return;
    const BProb& P = S.probs[p];
    double *alpha = S.alpha + (int64_t)p * S.cap, *beta = S.beta + (int64_t)p * (S.cap + 1),
           *invb = S.invb + (int64_t)p * (S.cap + 1);
    const int nsl = (int)((P.n + 63) >> 6);
    const int64_t ncod = P.c.base[nsl], nrest = P.c.rbase[nsl];
    const double ts = SH ? tscale[p] : 1.0;
    if (P.real)
        small_steps<true, true, RES, SH>(P.c, ncod, nrest, P.W, alpha, beta, invb, j0, j1, nullptr, 0, ctab, ts);
    else
        small_steps<false, true, RES, SH>(P.c, ncod, nrest, P.W, alpha, beta, invb, j0, j1, nullptr, 0, ctab, ts);
}

// K2: alpha_j, W_{j+1} = u - alpha_j W_j / beta_j, |W_{j+1}|^2 partials
__global__ void __launch_bounds__(kBT) k_b2(BState S, int jrel) {
    __shared__ double sh[kBT / 64];
    __shared__ double sa;
    const int j = *S.jbase + jrel;
    if (j >= S.cap) return;
    const int64_t ld = S.cap + 1;
    for (int64_t it = blockIdx.x; it < S.nitems; it += gridDim.x) {
        const int p = S.item_prob[it];
        if (!S.active[p]) continue;
        const BProb P = S.probs[p];
        const int64_t nit = (P.n + kItemRows - 1) / kItemRows;
        const double ib = S.invb[p * ld + j];
        if (threadIdx.x < 64) {
            const double s = wave_sum(S.part1, P.item0, nit, threadIdx.x);
            if (threadIdx.x == 0) {
                sa = s * ib;
                if (it == P.item0) S.alpha[p * S.cap + j] = s * ib;
            }
        }
        __syncthreads();
        const double a = sa * ib;
        const int64_t r = (it - P.item0) * kItemRows + threadIdx.x;
        double acc = 0.0;
        if (r < P.n) {
            const double2 w = P.W[(int64_t)j * P.n + r], x = S.u[P.voff + r];
            const double2 v = make_double2(x.x - a * w.x, x.y - a * w.y);
            P.W[(int64_t)(j + 1) * P.n + r] = v;
            acc = v.x * v.x + v.y * v.y;
        }
        const double t = block_sum(acc, sh);
        if (threadIdx.x == 0) S.part2[it] = t;
        __syncthreads();  // sa is reused by the next item
    }
}

// K3: beta_{j+1}, 1/beta_{j+1}; one wavefront per problem
__global__ void __launch_bounds__(64) k_b3(BState S, int jrel, int nprob) {
    const int j = *S.jbase + jrel;
    if (j >= S.cap) return;
    const int p = blockIdx.x;
    if (p >= nprob || !S.active[p]) return;
    const BProb P = S.probs[p];
    const int64_t nit = (P.n + kItemRows - 1) / kItemRows;
    const double s = wave_sum(S.part2, P.item0, nit, threadIdx.x);
    if (threadIdx.x == 0) {
        const int64_t ld = S.cap + 1;
        const double b = sqrt(s);
        S.beta[p * ld + j + 1] = b;
        S.invb[p * ld + j + 1] = b > 0 ? 1.0 / b : 0.0;
    }
}

// end of a replay: the next replay starts `count` steps later
__global__ void k_bnext(int32_t* jbase, int count) {
    if (threadIdx.x == 0) *jbase += count;
}

// psi_r = sum_l coef_l conj(W_l[r]) over the problem's m vectors; |psi|^2 partials
// Seeded start vectors of a batch on the device: one workgroup per problem
// draws its std::mt19937 entries (mt_start_block) into gen; k_bstart_scale
// then writes dst[r] = gen[iperm[r]] / s (the member's internal row order;
// identity without one), s = sqrt of the problem's entry sum taken on the
// host as start_vector does: the same values as the host's start vectors.
struct BStart {
    int64_t n;
    uint32_t seed;
    double2* gen;
    double2* dst;
    const int32_t* iperm;
};

__global__ void __launch_bounds__(1024) k_bmt_start(const BStart* __restrict__ jobs, double* __restrict__ nrm2) {
    const BStart J = jobs[blockIdx.x];
    mt_start_block(J.n, J.seed, J.gen, nrm2 + blockIdx.x);
}

__global__ void __launch_bounds__(kBT) k_bstart_scale(const BStart* __restrict__ jobs, const double* __restrict__ s) {
    const BStart J = jobs[blockIdx.y];
    const double sj = s[blockIdx.y];
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < J.n; r += (int64_t)gridDim.x * blockDim.x) {
        double2 z = J.gen[J.iperm ? J.iperm[r] : r];
        z.x /= sj;
        z.y /= sj;
        J.dst[r] = z;
    }
}

// Continuation starts: the previous solve's ground state, kept in the
// reference row order (prev), conjugated (psi = sum_l c_l conj(v_l) is the
// eigenvector of conj(H), so conj(psi) is that of H), plus mix times the
// seeded unit vector: dst[r] = conj(prev[ip(r)]) + mix / |gen| * gen[ip(r)]
// + xmix * conj(prevx[ip(r)]) (ip = the member's internal order, the
// identity without one; prevx the previous solve's excited mix).  One
// 1024-thread workgroup per problem; nrm2 gets |dst|^2, the same fixed-order
// sum on every call.
struct BCont {
    int64_t n;
    const double2* prev;
    const double2* gen;  // seeded entries, reference order (read when mix > 0)
    const double2* prevx;  // the previous solve's excited mix, reference order (read when xmix > 0)
    double2* dst;
    const int32_t* iperm;
    double mix;          // start_mix / |gen|
    double xmix;
};

__global__ void __launch_bounds__(1024) k_bcont(const BCont* __restrict__ jobs, double* __restrict__ nrm2) {
    __shared__ double sh[1024 / 64];
    const BCont J = jobs[blockIdx.x];
    double acc = 0.0;
    for (int64_t r = threadIdx.x; r < J.n; r += 1024) {
        const int64_t q = J.iperm ? J.iperm[r] : r;
        const double2 a = J.prev[q];
        double2 z = make_double2(a.x, -a.y);
        if (J.mix > 0) {
            const double2 g = J.gen[q];
            z.x += J.mix * g.x;
            z.y += J.mix * g.y;
        }
        if (J.xmix > 0) {
            const double2 g = J.prevx[q];
            z.x += J.xmix * g.x;
            z.y -= J.xmix * g.y;
        }
        J.dst[r] = z;
        acc += z.x * z.x + z.y * z.y;
    }
    const double t = block_sum<1024>(acc, sh);
    if (threadIdx.x == 0) nrm2[blockIdx.x] = t;
}

// Ground states back to the reference row order for the copy to the host:
// dst[iperm[r]] = src[r] (a member in its internal order), dst[r] = src[r]
// otherwise; one job per problem (blockIdx.y).
struct BPsi {
    int64_t n;
    const int32_t* iperm;
    const double2* src;
    double2* dst;
};

__global__ void __launch_bounds__(kBT) k_bpsi_ref(const BPsi* __restrict__ jobs) {
    const BPsi J = jobs[blockIdx.y];
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < J.n; r += (int64_t)gridDim.x * blockDim.x)
        J.dst[J.iperm ? J.iperm[r] : r] = J.src[r];
}

__global__ void __launch_bounds__(kBT) k_bcombine(BState S, const double* __restrict__ coef,
                                                  const double* __restrict__ coefx, const int32_t* __restrict__ mvec,
                                                  double2* __restrict__ psi, double2* __restrict__ xs) {
    __shared__ double sh[kBT / 64];
    for (int64_t it = blockIdx.x; it < S.nitems; it += gridDim.x) {
        const int p = S.item_prob[it];
        const BProb P = S.probs[p];
        const int m = mvec[p];
        const double* cf = coef + (int64_t)p * S.cap;
        const double* cx = coefx + (int64_t)p * S.cap;
        const int64_t r = (it - P.item0) * kItemRows + threadIdx.x;
        double acc = 0.0;
        if (r < P.n) {
            double re = 0.0, im = 0.0, xr = 0.0, xi = 0.0;
            for (int l = 0; l < m; ++l) {
                const double2 w = P.W[(int64_t)l * P.n + r];
                re += cf[l] * w.x;
                im -= cf[l] * w.y;
                xr += cx[l] * w.x;
                xi -= cx[l] * w.y;
            }
            psi[P.voff + r] = make_double2(re, im);
            xs[P.voff + r] = make_double2(xr, xi);
            acc = re * re + im * im;
        }
        const double t = block_sum(acc, sh);
        if (threadIdx.x == 0) S.part1[it] = t;
    }
}

__global__ void __launch_bounds__(kBT) k_bscale(BState S, const double* __restrict__ scale, double2* __restrict__ psi) {
    for (int64_t it = blockIdx.x; it < S.nitems; it += gridDim.x) {
        const int p = S.item_prob[it];
        const BProb P = S.probs[p];
        const int64_t r = (it - P.item0) * kItemRows + threadIdx.x;
        if (r < P.n) {
            double2 z = psi[P.voff + r];
            z.x *= scale[p];
            z.y *= scale[p];
            psi[P.voff + r] = z;
        }
    }
}

}  // namespace

namespace {
// Pooled per-problem scalars and vectors of a batched solve.
// Host worker threads for the per-replay convergence tests, kept for the
// batch's lifetime: starting 16 threads costs about 0.5 ms, as much as a
// replay of two Lanczos steps.  run(nt, f) calls f(t) for t < nt, the caller
// taking t = 0, and returns when every call has returned.
class HostPool {
public:
    explicit HostPool(int workers) {
        for (int w = 1; w <= workers; ++w) th_.emplace_back([this, w] { loop(w); });
    }
    ~HostPool() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto& t : th_) t.join();
    }
    int size() const { return (int)th_.size() + 1; }
    void run(int nt, const std::function<void(int)>& f) {
        nt = std::max(1, std::min(nt, size()));
        {
            std::lock_guard<std::mutex> lk(mu_);
            job_ = &f;
            nt_ = nt;
            left_ = nt - 1;
            ++gen_;
        }
        if (nt > 1) cv_.notify_all();
        f(0);
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [this] { return left_ == 0; });
        job_ = nullptr;
    }

private:
    void loop(int w) {
        int seen = 0;
        while (true) {
            const std::function<void(int)>* job;
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return stop_ || gen_ != seen; });
                if (stop_) return;
                seen = gen_;
                if (w >= nt_) continue;
                job = job_;
            }
            (*job)(w);
            std::lock_guard<std::mutex> lk(mu_);
            if (--left_ == 0) done_.notify_one();
        }
    }
    std::vector<std::thread> th_;
    std::mutex mu_;
    std::condition_variable cv_, done_;
    const std::function<void(int)>* job_ = nullptr;
    int nt_ = 0, left_ = 0, gen_ = 0;
    bool stop_ = false;
};

struct Pools {
    DevBuf<BProb> probs;
    DevBuf<int32_t> active, jbase, mvec;
    DevBuf<double> alpha, beta, invb, part1, part2, coef, coefx, scale;
    DevBuf<double2> u, psi, W;
    // the previous solve's excited mix (normalised sum of its second and
    // third lowest Ritz vectors): internal order, then reference order
    DevBuf<double2> xs, xref;
};
}  // namespace

struct blqh_batch {
    std::vector<blqh_hamil*> hs;
    std::vector<BProb> h_probs;
    std::vector<int64_t> item0;  // [P + 1]
    int64_t rows = 0, nitems = 0, nnz = 0;
    DevBuf<int32_t> item_prob;
    DevBuf<int32_t> xitems, xseg;    // per-XCD work lists of k_b1j (rebuilt by refresh_probs)
    std::vector<int32_t> h_xitems, h_xseg;
    int lpr = 0;                 // 64: k_b1j over the coded layout; else lanes per row of k_b1
    size_t tab_bytes = 0;        // LDS for the members' largest value table
    bool has_real = false, has_complex = false;  // value kinds among the members
    int grid = 0;
    // kept between solves of the same lambda: device pools, the captured
    // replay (for one check interval and lane count) and pinned staging
    Pools pl;
    int pool_cap = -1;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    int g_chk = -1, g_lpr = -1, g_cap = -1, g_kinds = -1;
    std::array<size_t, 3> g_tab{};  // launch shape of the captured K1 (k1_shape)
    char* pin = nullptr;
    double2* psi_pin = nullptr;  // pinned staging of the ground states (b->rows entries, on first use)
    // pl.u holds every problem's ground state of the last finished solve in
    // the reference row order (the start of a continuation solve)
    bool cont_ok = false;
    DevBuf<char> relayout;       // scratch for reordering members' panels
    // Shared-scale groups (blqh_batch_create_scaled); G = 0: every member
    // has its own matrix.  Problem p = s G + g is H0[s] + scale[g] T[s];
    // hs[p] is the sector's template tpl[s] (owned, flagged T entries).
    int G = 0;
    std::vector<blqh_hamil*> tpl;
    std::vector<double> tscale;   // [P]
    DevBuf<double> dtscale;
    // k_b1x (members of one panel, lanes 64): every owner's (problem's, or group of
    // G's) column tiles, made when the members change
    bool one_panel = false;
    bool tiles_ok = false;
    std::vector<ColTiles> tiles;
    DevBuf<uint4> tent;
    DevBuf<int64_t> tgoff;
    size_t x_bytes = 0;           // k_b1x's dynamic LDS
    int x_grid = 0;
    int x_team = 1;               // wavefronts of a slice (batch_team)
    std::unique_ptr<HostPool> hpool;  // convergence-test threads (batches of 32 or more problems)
    ~blqh_batch() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        if (pin) (void)hipHostFree(pin);
        if (psi_pin) (void)hipHostFree(psi_pin);
        for (blqh_hamil* H : tpl) delete H;
    }
};

namespace {

bool use_tiles(const blqh_batch* b) { return b->lpr == 64 && b->one_panel; }

// Batches whose members a workgroup each steps through (k_bsmall): lanes 64, small members
// only (small_matrix).  lds: its dynamic LDS (0: another batch),
// res: with every matrix in LDS.
constexpr int kSmallSteps = 8;  // steps a launch, at least
struct SmallShape {
    size_t lds = 0;
    bool res = false;
};
SmallShape small_shape(const blqh_batch* b) {
    if (b->lpr != 64) return {};
    size_t vec = 0, all = 0;
    for (const blqh_hamil* H : b->hs) {
        if (!small_matrix(H->n, H->nnz) || !H->cod.built) return {};
        const Coded& C = H->cod;
        vec = std::max(vec, small_lds_bytes(C.real, C.ntab, H->n));
        all = std::max(all, small_lds_bytes(C.real, C.ntab, H->n, C.ncod, C.nrest));
    }
    return all <= kSmallLdsMax ? SmallShape{all, true} : vec <= kSmallLdsMax ? SmallShape{vec, false} : SmallShape{};
}

// What the captured K1 launches depend on beside the lanes and the value kinds.
std::array<size_t, 3> k1_shape(const blqh_batch* b) {
    if (!use_tiles(b)) return {0, b->tab_bytes, 0};
    return {(size_t)b->x_grid, b->x_bytes, (size_t)b->x_team};
}

// Work lists (xcd_lists) over the members (all, or those with live[p] set); with
// shared-scale groups over the groups (live when one of their problems is).  k_b1x:
// elements of two units while that leaves every workgroup at least four (an element
// stages the owner's whole x), else of one; seg[27] = units per element.
void work_lists(const blqh_batch* b, const std::vector<char>* live, std::vector<int32_t>& items,
                std::vector<int32_t>& seg) {
    std::vector<XcdMember> mem;
    const int per = b->G ? b->G : 1, no = (int)b->hs.size() / per;
    const int64_t unit = (int64_t)kUnit * 64 / b->x_team;  // rows
    mem.reserve(no);
    std::vector<int> on;
    int64_t units = 0;
    for (int o = 0; o < no; ++o) {
        bool l = !live;
        for (int g = 0; g < per && !l; ++g) l = (*live)[o * per + g] != 0;
        if (!l) continue;
        on.push_back(o);
        units += ceil_div(b->h_probs[o * per].n, unit);
    }
    const bool tiled = use_tiles(b);
    const int span = tiled && b->x_team == 1 && units >= 8 * (int64_t)b->x_grid ? 2 : 1;
    for (int o : on) {
        const BProb& d = b->h_probs[o * per];
        if (tiled) {
            const int64_t e0 = (int64_t)o << kElemBits;
            mem.push_back({e0, e0 + ceil_div(d.n, unit * span), b->hs[o * per]->nnz * per, 1, d.real});
        } else {
            mem.push_back({b->item0[o], b->item0[o + 1], b->hs[o]->nnz, d.npan, d.real});
        }
    }
    xcd_lists(mem, items, seg);
    seg.push_back(span);
}

// Column tiles of every owner's coded layout, as wide as the LDS beside its value
// table allows.
void make_tiles(blqh_batch* b) {
    hipStream_t st = stream();
    const int per = b->G ? b->G : 1, no = (int)b->hs.size() / per;
    std::vector<TileJob> jobs(no);
    int64_t runs = 0, smax = 1;
    int rmax = 64, ntmax = 1;
    b->x_bytes = 0;
    for (int o = 0; o < no; ++o) {
        const blqh_hamil* H = b->hs[o * per];
        const size_t tabb = tile_tab_bytes(H->cod.real, H->cod.ntab);
        const int64_t most = std::min<int64_t>(kTileMax, (int64_t)((kLdsMax - tabb) / (sizeof(double2) * per)));
        const int nt = (int)ceil_div(H->n, most), tw = (int)ceil_div(H->n, (int64_t)nt);
        const int64_t nsl = ceil_div(H->n, (int64_t)64);
        jobs[o] = TileJob{cview(H->cod, H->n), tw, nt, H->cod.real ? 1 : 0, b->G ? kCodTun - 1 : 0xffffu, runs};
        runs += nsl * nt;
        smax = std::max(smax, nsl);
        ntmax = std::max(ntmax, nt);
        rmax = std::max(rmax, std::min(H->row_max > 0 ? H->row_max : 4096, 4096));
        b->x_bytes = std::max(b->x_bytes, tabb + sizeof(double2) * per * (size_t)tw);
    }
    DevBuf<TileJob> dj(no);
    DevBuf<int32_t> cnt(runs);
    if ((int64_t)b->tgoff.n < runs + 1) b->tgoff.alloc(runs + 1);
    BLQH_HIP(hipMemcpyAsync(dj.get(), jobs.data(), no * sizeof(TileJob), hipMemcpyHostToDevice, st));
    auto launch = [&](auto kern, bool fill) {
        for (int o = 0; o < no; o += 65535)
            hipLaunchKernelGGL(kern, dim3((unsigned)std::min<int64_t>(smax, 4096), (unsigned)std::min(65535, no - o)),
                               dim3(64), (fill ? (size_t)rmax * 12 : 0) + (size_t)ntmax * 128, st, dj.get() + o, rmax,
                               ntmax, cnt.get(), b->tgoff.get(), b->tent.get());
        BLQH_HIP(hipGetLastError());
    };
    launch(k_tiles<false>, false);
    exclusive_scan(cnt.get(), b->tgoff.get(), runs, st);
    int64_t groups = 0;
    copy_sync(&groups, b->tgoff.get() + runs, 8, hipMemcpyDeviceToHost);
    if ((int64_t)b->tent.n < groups * 64) b->tent.alloc(std::max<int64_t>(groups * 64, 1));
    launch(k_tiles<true>, true);
    BLQH_HIP(hipStreamSynchronize(st));
    b->tiles.resize(no);
    for (int o = 0; o < no; ++o)
        b->tiles[o] = ColTiles{jobs[o].tw, jobs[o].nt, b->tent.get(), b->tgoff.get() + jobs[o].goff0};
    const int wpc = b->x_bytes <= kLdsHalf ? 2 : 1;  // workgroups of 1024 threads that share a CU's LDS
    std::vector<int64_t> rows(no);
    for (int o = 0; o < no; ++o) rows[o] = jobs[o].c.n;
    b->x_team = batch_team(rows, runtime().num_cus);
    // an XCD's list holds up to a chunk (xcd_lists) more than its even share: room for all of it at once
    const int64_t units = batch_units(rows, b->x_team), share = ceil_div(units, kXcds) + ceil_div(units, 64);
    // one of two sizes, so that the next point's tables leave the captured launches as they are
    b->x_bytes = wpc == 2 ? kLdsHalf : kLdsMax;
    b->x_grid = (int)(kXcds * std::min(share, ceil_div((int64_t)runtime().num_cus * wpc, kXcds)));
    b->tiles_ok = true;
}

// Work lists of k_b1j (xcd_lists), uploaded when they change.
void build_xcd_lists(blqh_batch* b) {
    std::vector<int32_t> items, seg;
    work_lists(b, nullptr, items, seg);
    if (items == b->h_xitems && seg == b->h_xseg) return;
    b->h_xitems.swap(items);
    b->h_xseg.swap(seg);
    // ordered after every kernel queued so far; the host vectors are not
    // touched again before the copies have completed
    hipStream_t st = stream();
    BLQH_HIP(hipMemcpyAsync(b->xitems.get(), b->h_xitems.data(), b->h_xitems.size() * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(b->xseg.get(), b->h_xseg.data(), 28 * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipStreamSynchronize(st));
}

// The layout that the batch's kernels read and its current buffers, of every
// member: the coded one (lanes 64), else row-major panels.
void refresh_probs(blqh_batch* b) {
    b->has_real = b->has_complex = false;
    b->tab_bytes = 0;
    const bool coded = b->lpr == 64;
    if (!coded) {
        for (blqh_hamil* H : b->hs) ensure_panels(H);
        const size_t scratch = panel_layout_scratch_bytes(b->hs.data(), (int)b->hs.size());
        if (scratch > b->relayout.bytes()) b->relayout.alloc(scratch);
        set_panel_layouts(b->hs.data(), (int)b->hs.size(), false, b->relayout.get(), b->relayout.bytes(), false);
    }
    for (size_t p = 0; p < b->hs.size(); ++p) {
        blqh_hamil* H = b->hs[p];
        BProb& d = b->h_probs[p];
        if (coded) ensure_coded(H);
        const bool real = coded ? H->cod.real : H->pan.real;
        d.real = real ? 1 : 0;
        (real ? b->has_real : b->has_complex) = true;
        if (coded) {
            d.c = cview(H->cod, H->n);
            b->tab_bytes = std::max(b->tab_bytes, cod_lds_bytes(real, H->cod.ntab));
        } else {
            d.pbase = H->pan.pbase.get();
            d.prow = H->pan.prow.get();
            d.pcol = H->pan.pcol.get();
            d.pvr = H->pan.pvr.get();
            d.pvc = H->pan.pvc.get();
        }
    }
    if (use_tiles(b)) {
        if (!b->tiles_ok) make_tiles(b);
        for (size_t p = 0; p < b->hs.size(); ++p) b->h_probs[p].t = b->tiles[p / (b->G ? b->G : 1)];
    }
    // one of three sizes (as x_bytes)
    const size_t small = cod_lds_bytes(true, kCodReal), half = cod_lds_bytes(false, kCodCplx / 2);
    b->tab_bytes = b->tab_bytes <= small ? small : b->tab_bytes <= half ? half : cod_lds_bytes(false, kCodCplx);
    build_xcd_lists(b);
}

// Dynamic LDS above the default, allowed once per kernel.
template <class K>
void allow_lds(K kern, size_t bytes) {
    BLQH_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

template <bool LZ, int G, bool SH, int NP>
void launch_b1x_team(const blqh_batch* b, const BState& S, int jrel, const double2* xs, double2* ys, double* part,
                     hipStream_t st, bool go) {
    static const bool attr = (allow_lds(k_b1x<LZ, G, SH, NP>, kLdsMax), true);  // once per instantiation, thread-safe
    (void)attr;
    if (!go) return;
    hipLaunchKernelGGL((k_b1x<LZ, G, SH, NP>), dim3(b->x_grid), dim3(kBTx), b->x_bytes, st, S, b->dtscale.get(), jrel,
                       xs, ys, part);
}

template <bool LZ, int G, bool SH>
void launch_b1x(const blqh_batch* b, const BState& S, int jrel, const double2* xs, double2* ys, double* part,
                hipStream_t st, bool go) {
    if (b->x_team == 4) launch_b1x_team<LZ, G, SH, 4>(b, S, jrel, xs, ys, part, st, go);
    else if (b->x_team == 2) launch_b1x_team<LZ, G, SH, 2>(b, S, jrel, xs, ys, part, st, go);
    else launch_b1x_team<LZ, G, SH, 1>(b, S, jrel, xs, ys, part, st, go);
}

template <bool LZ, int KIND>
void launch_b1j(const blqh_batch* b, const BState& S, int jrel, const double2* xs, double2* ys, double* part,
                hipStream_t st, bool go) {
    static const bool attr = (allow_lds(k_b1j<LZ, KIND>, cod_lds_bytes(false, kCodCplx)), true);
    (void)attr;
    if (!go) return;
    hipLaunchKernelGGL((k_b1j<LZ, KIND>), dim3(b->grid), dim3(kBTj), b->tab_bytes, st, S, jrel, xs, ys, part);
}

// go false (lanes 64): only the kernel's attributes are set, which a capture is not to do.
template <bool LZ>
void launch_b1(const blqh_batch* b, const BState& S, int jrel, const double2* xs, double2* ys, double* part,
               hipStream_t st, bool go = true) {
    const dim3 g(b->grid), t(kBT);
    switch (b->G) {  // shared-scale groups: one pass over each sector's entries for all its problems
        case 0: break;
        case 1: launch_b1x<LZ, 1, true>(b, S, jrel, xs, ys, part, st, go); return;
        case 2: launch_b1x<LZ, 2, true>(b, S, jrel, xs, ys, part, st, go); return;
        case 3: launch_b1x<LZ, 3, true>(b, S, jrel, xs, ys, part, st, go); return;
        case 4: launch_b1x<LZ, 4, true>(b, S, jrel, xs, ys, part, st, go); return;
        default: throw Error(BLQH_EINTERNAL, "unsupported group size");
    }
    if (use_tiles(b)) {
        launch_b1x<LZ, 1, false>(b, S, jrel, xs, ys, part, st, go);
        return;
    }
    switch (b->lpr) {
        case 64:
            if (b->has_real && b->has_complex) {  // measured faster than one launch per kind
                launch_b1j<LZ, 2>(b, S, jrel, xs, ys, part, st, go);
                break;
            }
            if (b->has_real) launch_b1j<LZ, 0>(b, S, jrel, xs, ys, part, st, go);
            if (b->has_complex) launch_b1j<LZ, 1>(b, S, jrel, xs, ys, part, st, go);
            break;
        case 4: hipLaunchKernelGGL((k_b1<4, LZ>), g, t, 0, st, S, jrel, xs, ys, part); break;
        case 8: hipLaunchKernelGGL((k_b1<8, LZ>), g, t, 0, st, S, jrel, xs, ys, part); break;
        case 16: hipLaunchKernelGGL((k_b1<16, LZ>), g, t, 0, st, S, jrel, xs, ys, part); break;
        case 32: hipLaunchKernelGGL((k_b1<32, LZ>), g, t, 0, st, S, jrel, xs, ys, part); break;
        default: throw Error(BLQH_EINTERNAL, "unsupported batched SpMV lanes");
    }
}

BState make_state(const blqh_batch* b, Pools& pl, int cap) {
    BState S{};
    S.probs = pl.probs.get();
    S.item_prob = b->item_prob.get();
    S.nitems = b->nitems;
    S.xitems = b->xitems.get();
    S.xseg = b->xseg.get();
    S.active = pl.active.get();
    S.jbase = pl.jbase.get();
    S.cap = cap;
    S.alpha = pl.alpha.get();
    S.beta = pl.beta.get();
    S.invb = pl.invb.get();
    S.u = pl.u.get();
    S.part1 = pl.part1.get();
    S.part2 = pl.part2.get();
    return S;
}

}  // namespace

blqh_batch* blqh_batch_create_impl(blqh_hamil* const* hs, int count, int lanes) {
    BLQH_REQUIRE(lanes == 0 || lanes == 4 || lanes == 8 || lanes == 16 || lanes == 32 || lanes == 64, BLQH_EINVAL,
                 "unsupported lanes per row");
    BLQH_REQUIRE(count >= 1, BLQH_EINVAL, "empty batch");
    auto* b = new blqh_batch;
    try {
        b->hs.assign(hs, hs + count);
        b->item0.assign(count + 1, 0);
        std::vector<int32_t> ip;
        for (int p = 0; p < count; ++p) {
            blqh_hamil* H = hs[p];
            BLQH_REQUIRE(H != nullptr, BLQH_EINVAL, "null hamiltonian in batch");
            BLQH_REQUIRE(H->n > 0, BLQH_EINVAL, "batched solve needs non-empty Hamiltonians");
            BProb d{};
            d.n = H->n;
            d.npan = (int32_t)ceil_div(H->n, (int64_t)kPanelWidth);
            d.item0 = b->nitems;
            d.voff = b->rows;
            const int64_t nit = ceil_div(H->n, kItemRows);
            for (int64_t i = 0; i < nit; ++i) ip.push_back(p);
            b->nitems += nit;
            b->rows += H->n;
            b->nnz += H->nnz;
            b->item0[p + 1] = b->nitems;
            b->h_probs.push_back(d);
        }
        BLQH_REQUIRE(b->nitems < (int64_t)1 << 31, BLQH_ERANGE, "batch too large");
        b->item_prob.alloc(ip.size());
        copy_sync(b->item_prob.get(), ip.data(), ip.size() * 4, hipMemcpyHostToDevice);
        // a multiple of 8 (one share per XCD in k_b1j)
        b->grid = (int)(8 * ceil_div(std::min<int64_t>(b->nitems, (int64_t)runtime().num_cus * 8), 8));
        b->xitems.alloc(2 * b->nitems);
        b->xseg.alloc(28);
        b->one_panel = b->hs.size() < ((size_t)1 << (31 - kElemBits));
        for (const BProb& d : b->h_probs) b->one_panel = b->one_panel && d.npan == 1;
        b->lpr = lanes ? lanes : 64;
        refresh_probs(b);
    } catch (...) {
        delete b;
        throw;
    }
    return b;
}

// New members of the same shapes (a sweep's next parameter point): the work
// items, pools, captured replay and lane choice are kept.
void blqh_batch_rebind_impl(blqh_batch* b, blqh_hamil* const* hs, int count) {
    BLQH_REQUIRE(b->G == 0, BLQH_EINVAL, "a shared-scale batch is rebound with blqh_batch_rebind_scaled");
    BLQH_REQUIRE(count == (int)b->hs.size(), BLQH_EINVAL, "rebind needs as many Hamiltonians as the batch has");
    int64_t nnz = 0;
    for (int p = 0; p < count; ++p) {
        BLQH_REQUIRE(hs[p] != nullptr, BLQH_EINVAL, "null hamiltonian in batch");
        BLQH_REQUIRE(hs[p]->n == b->h_probs[p].n, BLQH_EINVAL,
                     "rebind needs Hamiltonians of the same sizes, in the same order");
        nnz += hs[p]->nnz;
    }
    b->nnz = nnz;
    b->hs.assign(hs, hs + count);
    b->tiles_ok = false;
    refresh_probs(b);
}

namespace {
// H0 + 1 T of one sector (blqh_hamil_combine) in the coded layout, the tunnelling
// flag set on the column of every T entry (those between words of different
// upper-layer occupation; nu per row in the internal order).  The tunnelling terms are the
// only ones that move an electron between the layers, so T's entries are
// exactly those between words of different upper-layer occupation; their
// count must equal T's.
blqh_hamil* make_template(const blqh_hamil* base, const blqh_hamil* tun) {
    BLQH_REQUIRE(base != nullptr && tun != nullptr, BLQH_EINVAL, "null hamiltonian in batch");
    BLQH_REQUIRE(base->basis->geo.S >= 2, BLQH_EINVAL, "a shared-scale batch needs bilayer sectors");
    BLQH_REQUIRE(base->n <= (int64_t)kCodTun, BLQH_EINVAL,
                 "a shared-scale batch takes sectors of at most 32768 states");
    auto* H = new blqh_hamil;
    try {
        blqh_hamil_combine_impl(base, tun, 1.0, H, false);
        build_order(H);
        const blqh_basis* B = H->basis;
        const int64_t n = H->n;
        const uint64_t upper = lowbits(B->geo.S * B->geo.nphi / 2);
        std::vector<uint8_t> nu(n);
        const int32_t* ip = H->ord.on ? host_iperm(H).data() : nullptr;
        for (int64_t r = 0; r < n; ++r) {
            const int64_t i = ip ? ip[r] : r;
            nu[r] = (uint8_t)popc(B->h_id[i] & upper);
        }
        DevBuf<uint8_t> dnu(n);
        BLQH_HIP(hipMemcpyAsync(dnu.get(), nu.data(), n, hipMemcpyHostToDevice, stream()));
        int64_t ntun = 0;
        build_coded(H, dnu.get(), &ntun);
        BLQH_REQUIRE(ntun == tun->nnz, BLQH_EINTERNAL, "the tunnelling entries are not the layer-changing entries");
    } catch (...) {
        delete H;
        throw;
    }
    return H;
}

// Templates of nsec sectors, built on up to 8 host threads: one sector's
// merge, panels and marking are small launches with host waits between
// them, so several sectors on their own streams keep the GPU busy.  On an
// error every built template is freed and the first error is raised.
std::vector<blqh_hamil*> make_templates(const blqh_hamil* const* base, const blqh_hamil* const* tun, int nsec) {
    std::vector<blqh_hamil*> out(nsec, nullptr);
    const int nt = std::max(1, std::min(nsec, 8));
    std::vector<std::exception_ptr> err(nt);
    auto work = [&](int t) {
        try {
            for (int q = t; q < nsec; q += nt) out[q] = make_template(base[q], tun[q]);
        } catch (...) {
            err[t] = std::current_exception();
        }
    };
    if (nt == 1) {
        work(0);
    } else {
        std::vector<std::thread> th;
        for (int t = 1; t < nt; ++t) th.emplace_back(work, t);
        work(0);
        for (auto& x : th) x.join();
    }
    for (auto& e : err)
        if (e) {
            for (blqh_hamil* H : out) delete H;
            std::rethrow_exception(e);
        }
    return out;
}

}  // namespace

blqh_batch* blqh_batch_create_scaled_impl(const blqh_hamil* const* base, const blqh_hamil* const* tun, int nsec,
                                          const double* scales, int nscale) {
    BLQH_REQUIRE(nsec >= 1, BLQH_EINVAL, "empty batch");
    BLQH_REQUIRE(nscale >= 1 && nscale <= 4, BLQH_EINVAL, "a shared-scale batch takes 1 to 4 scales");
    for (int g = 0; g < nscale; ++g)
        BLQH_REQUIRE(std::isfinite(scales[g]) && scales[g] >= 0.0, BLQH_EINVAL, "scales must be finite and >= 0");
    auto* b = new blqh_batch;
    try {
        const int G = nscale;
        b->G = G;
        b->tpl = make_templates(base, tun, nsec);
        const int P = nsec * G;
        b->hs.resize(P);
        b->item0.assign(P + 1, 0);
        b->tscale.resize(P);
        std::vector<int32_t> ip;
        for (int q = 0; q < nsec; ++q) {
            blqh_hamil* H = b->tpl[q];
            const int64_t nit = ceil_div(H->n, kItemRows);
            b->nnz += H->nnz;
            for (int g = 0; g < G; ++g) {
                const int p = q * G + g;
                b->hs[p] = H;
                b->tscale[p] = scales[g];
                BProb d{};
                d.n = H->n;
                d.npan = 1;
                d.item0 = b->nitems;
                d.voff = b->rows;
                for (int64_t i = 0; i < nit; ++i) ip.push_back(p);
                b->nitems += nit;
                b->rows += H->n;
                b->item0[p + 1] = b->nitems;
                b->h_probs.push_back(d);
            }
        }
        BLQH_REQUIRE(b->nitems < (int64_t)1 << 31, BLQH_ERANGE, "batch too large");
        b->item_prob.alloc(ip.size());
        copy_sync(b->item_prob.get(), ip.data(), ip.size() * 4, hipMemcpyHostToDevice);
        b->dtscale.alloc(P);
        copy_sync(b->dtscale.get(), b->tscale.data(), P * 8, hipMemcpyHostToDevice);
        b->grid = (int)(8 * ceil_div(std::min<int64_t>(b->nitems, (int64_t)runtime().num_cus * 8), 8));
        b->xitems.alloc(2 * b->nitems);
        b->xseg.alloc(28);
        b->lpr = 64;
        b->one_panel = b->hs.size() < ((size_t)1 << (31 - kElemBits));
        for (const BProb& d : b->h_probs) b->one_panel = b->one_panel && d.npan == 1;
        refresh_probs(b);
    } catch (...) {
        delete b;
        throw;
    }
    return b;
}

// The next parameter point of a shared-scale batch: new H0 and T of the same
// sectors (same sizes, same order); the scales stay.
void blqh_batch_rebind_scaled_impl(blqh_batch* b, const blqh_hamil* const* base, const blqh_hamil* const* tun,
                                   int nsec) {
    BLQH_REQUIRE(b->G > 0, BLQH_EINVAL, "not a shared-scale batch");
    BLQH_REQUIRE(nsec == (int)b->tpl.size(), BLQH_EINVAL, "rebind needs as many sectors as the batch has");
    for (int q = 0; q < nsec; ++q)
        BLQH_REQUIRE(base[q] != nullptr && base[q]->n == b->tpl[q]->n, BLQH_EINVAL,
                     "rebind needs sectors of the same sizes, in the same order");
    std::vector<blqh_hamil*> fresh = make_templates(base, tun, nsec);
    BLQH_HIP(hipStreamSynchronize(stream()));  // no queued work reads the old templates
    for (blqh_hamil* H : b->tpl) delete H;
    b->tpl.swap(fresh);
    b->nnz = 0;
    for (int q = 0; q < nsec; ++q) {
        b->nnz += b->tpl[q]->nnz;
        for (int g = 0; g < b->G; ++g) b->hs[q * b->G + g] = b->tpl[q];
    }
    b->tiles_ok = false;
    refresh_probs(b);
}

int blqh_batch_group_size_impl(const blqh_batch* b) { return b->G; }

void blqh_batch_destroy_impl(blqh_batch* b) { delete b; }

int blqh_batch_lanes_impl(const blqh_batch* b) { return b->lpr; }

void blqh_batch_set_lanes_impl(blqh_batch* b, int lanes) {
    BLQH_REQUIRE(lanes == 4 || lanes == 8 || lanes == 16 || lanes == 32 || lanes == 64, BLQH_EINVAL,
                 "unsupported lanes per row");
    BLQH_REQUIRE(b->G == 0 || lanes == 64, BLQH_EINVAL, "a shared-scale batch runs one lane per row");
    b->lpr = lanes;
}

void blqh_batch_lanczos_impl(blqh_batch* b, const blqh_lanczos_opts& o, const uint32_t* seeds,
                             const double* const* starts, blqh_lanczos_result* res, double* const* psi_out,
                             bool cont, double excited) {
    BLQH_REQUIRE(o.start_mix >= 0 && std::isfinite(o.start_mix), BLQH_EINVAL, "start_mix must be finite and >= 0");
    BLQH_REQUIRE(excited >= 0 && std::isfinite(excited), BLQH_EINVAL, "excited_mix must be finite and >= 0");
    if (cont)
        BLQH_REQUIRE(b->cont_ok && b->pool_cap == o.lambda && !starts, BLQH_EINVAL,
                     "a continuation solve needs a finished solve of the same lambda on this batch");
    b->cont_ok = false;  // the steps below overwrite pl.u
    auto t0 = std::chrono::steady_clock::now();
    // BLQH_BATCH_TIMING=1 prints the host-side phases of every solve to stderr
    const bool phase_log = std::getenv("BLQH_BATCH_TIMING") != nullptr;
    auto tp = t0;
    auto phase = [&](const char* what) {
        if (!phase_log) return;
        BLQH_HIP(hipStreamSynchronize(stream()));
        const auto now = std::chrono::steady_clock::now();
        std::fprintf(stderr, "blqh batch: %-12s %8.2f ms\n", what, std::chrono::duration<double>(now - tp).count() * 1e3);
        tp = now;
    };
    hipStream_t st = stream();
    DrainGuard drain{st};  // of the batch's own pools and pinned memory
    const int P = (int)b->hs.size();
    const int cap = o.lambda;
    BLQH_REQUIRE(cap >= 2 && cap <= 100000, BLQH_EINVAL, "lambda out of range");
    const int chk = std::max(1, o.check_every);
    const int64_t ld = cap + 1;

    // Layout pointers are re-read here: a single-problem solve or SpMV of a
    // member Hamiltonian may have reordered its panels since the batch was
    // created, and set_lanes changes the layout.
    refresh_probs(b);
    // Krylov blocks of all problems and the per-problem scalars (kept for the
    // next solve with the same lambda)
    Pools& pl = b->pl;
    if (b->pool_cap != cap) {
        if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
        if (b->graph) (void)hipGraphDestroy(b->graph);
        b->gexec = nullptr;
        b->graph = nullptr;
        b->pool_cap = -1;
        b->pl = Pools{};
        size_t vecs = 0;
        for (int p = 0; p < P; ++p) vecs += (size_t)ld * b->h_probs[p].n;
        pl.W.alloc(vecs);
        pl.probs.alloc(P);
        pl.active.alloc(P);
        pl.jbase.alloc(1);
        pl.mvec.alloc(P);
        pl.alpha.alloc((size_t)P * cap);
        pl.beta.alloc((size_t)P * ld);
        pl.invb.alloc((size_t)P * ld);
        pl.part1.alloc(b->nitems);
        pl.part2.alloc(b->nitems);
        pl.coef.alloc((size_t)P * cap);
        pl.coefx.alloc((size_t)P * cap);
        pl.xs.alloc(b->rows);
        pl.xref.alloc(b->rows);
        pl.scale.alloc(P);
        pl.u.alloc(b->rows);
        pl.psi.alloc(b->rows);
        if (b->pin) (void)hipHostFree(b->pin);
        b->pin = nullptr;
        // alpha, beta, two slots of active flags, two slots of live work lists
        const size_t pin_bytes = ((size_t)P * cap + (size_t)P * ld) * 8 + 2 * (size_t)P * 4 +
                                 2 * (2 * (size_t)b->nitems + 28) * 4;
        BLQH_HIP(hipHostMalloc((void**)&b->pin, pin_bytes, hipHostMallocDefault));
        b->pool_cap = cap;
    }
    std::vector<BProb> hp = b->h_probs;
    {
        size_t off = 0;
        for (int p = 0; p < P; ++p) {
            hp[p].W = pl.W.get() + off;
            off += (size_t)ld * hp[p].n;
        }
    }
    BLQH_HIP(hipMemcpyAsync(pl.probs.get(), hp.data(), P * sizeof(BProb), hipMemcpyHostToDevice, st));

    phase("setup");
    // start vectors, beta_0 = 1: the caller's on the host (normalised, mixed,
    // permuted), the seeded ones drawn on the device (k_bmt_start)
    if (cont) {
        // conj(previous ground state) + start_mix * seeded unit vector, drawn
        // into the second Krylov slot (free until the first step)
        std::vector<BStart> gj;
        std::vector<BCont> cj(P);
        for (int p = 0; p < P; ++p) {
            const blqh_hamil* Hp = b->hs[p];
            double2* gen = hp[p].W + hp[p].n;
            cj[p] = {hp[p].n, pl.u.get() + hp[p].voff, gen, pl.xref.get() + hp[p].voff, hp[p].W,
                     Hp->ord.on ? Hp->ord.iperm.get() : nullptr, 0.0, excited};
            if (o.start_mix > 0) gj.push_back({hp[p].n, seeds ? seeds[p] : o.seed, gen, gen, nullptr});
        }
        DevBuf<BStart> dgj;
        DevBuf<BCont> dcj(P);
        DevBuf<double> dnrm(2 * (size_t)P);
        std::vector<double> nrm(P);
        if (!gj.empty()) {
            dgj.alloc(P);
            BLQH_HIP(hipMemcpyAsync(dgj.get(), gj.data(), P * sizeof(BStart), hipMemcpyHostToDevice, st));
            hipLaunchKernelGGL(k_bmt_start, dim3(P), dim3(1024), 0, st, dgj.get(), dnrm.get());
            BLQH_HIP(hipGetLastError());
            BLQH_HIP(hipMemcpyAsync(nrm.data(), dnrm.get(), P * sizeof(double), hipMemcpyDeviceToHost, st));
            BLQH_HIP(hipStreamSynchronize(st));
            for (int p = 0; p < P; ++p) cj[p].mix = o.start_mix / std::sqrt(nrm[p]);
        }
        BLQH_HIP(hipMemcpyAsync(dcj.get(), cj.data(), P * sizeof(BCont), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_bcont, dim3(P), dim3(1024), 0, st, dcj.get(), dnrm.get());
        BLQH_HIP(hipGetLastError());
        BLQH_HIP(hipMemcpyAsync(nrm.data(), dnrm.get(), P * sizeof(double), hipMemcpyDeviceToHost, st));
        BLQH_HIP(hipStreamSynchronize(st));
        std::vector<BStart> sj(P);
        for (int p = 0; p < P; ++p) {
            BLQH_REQUIRE(nrm[p] > 0 && std::isfinite(nrm[p]), BLQH_EINVAL, "continuation start is zero or not finite");
            nrm[p] = std::sqrt(nrm[p]);
            sj[p] = {hp[p].n, 0u, hp[p].W, hp[p].W, nullptr};
        }
        BLQH_HIP(hipMemcpyAsync(dnrm.get() + P, nrm.data(), P * sizeof(double), hipMemcpyHostToDevice, st));
        DevBuf<BStart> dsj(P);
        BLQH_HIP(hipMemcpyAsync(dsj.get(), sj.data(), P * sizeof(BStart), hipMemcpyHostToDevice, st));
        int64_t nmax = 0;
        for (int p = 0; p < P; ++p) nmax = std::max(nmax, hp[p].n);
        const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(nmax, kBT), 256));
        for (int j0 = 0; j0 < P; j0 += 65535)
            hipLaunchKernelGGL(k_bstart_scale, dim3(gx, (unsigned)std::min(65535, P - j0)), dim3(kBT), 0, st,
                               dsj.get() + j0, dnrm.get() + P + j0);
        BLQH_HIP(hipGetLastError());
        std::vector<double> ones((size_t)P * ld, 1.0);
        BLQH_HIP(hipMemcpyAsync(pl.beta.get(), ones.data(), ones.size() * 8, hipMemcpyHostToDevice, st));
        BLQH_HIP(hipMemcpyAsync(pl.invb.get(), ones.data(), ones.size() * 8, hipMemcpyHostToDevice, st));
        BLQH_HIP(hipStreamSynchronize(st));  // job tables, norms and ones are freed at scope exit
    } else {
        std::vector<std::vector<double2>> v0(P);
        std::vector<char> seeded(P, 0);
        for (int p = 0; p < P; ++p) seeded[p] = !(starts && starts[p]);
        auto make = [&](int p0, int p1) {
            for (int p = p0; p < p1; ++p) {
                if (seeded[p]) continue;
                const int64_t n = hp[p].n;
                v0[p].assign((const double2*)starts[p], (const double2*)starts[p] + n);
                double s = 0;
                for (auto& z : v0[p]) s += z.x * z.x + z.y * z.y;
                if (!(s > 0) || !std::isfinite(s)) { v0[p].clear(); continue; }
                if (o.start_mix > 0) {  // start/|start| + start_mix * seeded unit vector
                    std::vector<double2> r;
                    start_vector(n, seeds ? seeds[p] : o.seed, r);
                    const double zs = 1.0 / std::sqrt(s);
                    s = 0;
                    for (int64_t i = 0; i < n; ++i) {
                        double2& z = v0[p][i];
                        z = make_double2(z.x * zs + o.start_mix * r[i].x, z.y * zs + o.start_mix * r[i].y);
                        s += z.x * z.x + z.y * z.y;
                    }
                }
                s = std::sqrt(s);
                for (auto& z : v0[p]) { z.x /= s; z.y /= s; }
                const blqh_hamil* Hp = b->hs[p];
                if (Hp->ord.on) {  // the member's SpMV formats are in its internal order
                    std::vector<double2> w(n);
                    for (int64_t r = 0; r < n; ++r) w[r] = v0[p][Hp->ord.h_iperm[r]];
                    v0[p].swap(w);
                }
            }
        };
        int ncaller = 0;
        for (int p = 0; p < P; ++p) {
            ncaller += seeded[p] ? 0 : 1;
            if (!seeded[p] && b->hs[p]->ord.on) (void)host_iperm(b->hs[p]);  // for the threads below
        }
        if (ncaller > 0) {
            const int nt = std::max(1, std::min<int>(ncaller, (int)std::min(16u, std::max(1u, std::thread::hardware_concurrency()))));
            std::vector<std::thread> th;
            for (int t = 0; t < nt; ++t)
                th.emplace_back(make, (int)((int64_t)P * t / nt), (int)((int64_t)P * (t + 1) / nt));
            for (auto& t : th) t.join();
        }
        for (int p = 0; p < P; ++p)
            BLQH_REQUIRE(seeded[p] || !v0[p].empty(), BLQH_EINVAL, "start vector is zero or not finite");
        for (int p = 0; p < P; ++p)
            if (!seeded[p])
                BLQH_HIP(hipMemcpyAsync(hp[p].W, v0[p].data(), hp[p].n * sizeof(double2), hipMemcpyHostToDevice, st));
        std::vector<BStart> jobs;
        int64_t nmax = 0;
        for (int p = 0; p < P; ++p)
            if (seeded[p]) {
                const blqh_hamil* Hp = b->hs[p];
                const bool perm = Hp->ord.on;
                jobs.push_back({hp[p].n, seeds ? seeds[p] : o.seed, perm ? pl.u.get() + hp[p].voff : hp[p].W, hp[p].W,
                                perm ? Hp->ord.iperm.get() : nullptr});
                nmax = std::max(nmax, hp[p].n);
            }
        DevBuf<BStart> djobs;
        DevBuf<double> dnrm;
        if (!jobs.empty()) {
            const int J = (int)jobs.size();
            djobs.alloc(J);
            dnrm.alloc(2 * (size_t)J);
            BLQH_HIP(hipMemcpyAsync(djobs.get(), jobs.data(), J * sizeof(BStart), hipMemcpyHostToDevice, st));
            hipLaunchKernelGGL(k_bmt_start, dim3(J), dim3(1024), 0, st, djobs.get(), dnrm.get());
            BLQH_HIP(hipGetLastError());
            std::vector<double> nrm(J);
            BLQH_HIP(hipMemcpyAsync(nrm.data(), dnrm.get(), J * sizeof(double), hipMemcpyDeviceToHost, st));
            BLQH_HIP(hipStreamSynchronize(st));
            for (double& x : nrm) x = std::sqrt(x);
            BLQH_HIP(hipMemcpyAsync(dnrm.get() + J, nrm.data(), J * sizeof(double), hipMemcpyHostToDevice, st));
            const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(nmax, kBT), 256));
            for (int j0 = 0; j0 < J; j0 += 65535)
                hipLaunchKernelGGL(k_bstart_scale, dim3(gx, (unsigned)std::min(65535, J - j0)), dim3(kBT), 0, st,
                                   djobs.get() + j0, dnrm.get() + J + j0);
            BLQH_HIP(hipGetLastError());
        }
        std::vector<double> ones((size_t)P * ld, 1.0);
        BLQH_HIP(hipMemcpyAsync(pl.beta.get(), ones.data(), ones.size() * 8, hipMemcpyHostToDevice, st));
        BLQH_HIP(hipMemcpyAsync(pl.invb.get(), ones.data(), ones.size() * 8, hipMemcpyHostToDevice, st));
        BLQH_HIP(hipStreamSynchronize(st));  // v0, ones, the job table and the norms are freed at scope exit
    }
    phase("start");
    std::vector<int32_t> act(P, 1);
    BLQH_HIP(hipMemcpyAsync(pl.active.get(), act.data(), P * 4, hipMemcpyHostToDevice, st));
    BState S = make_state(b, pl, cap);

    // `chk` steps as one graph; kernels read the first step from pl.jbase and
    // the graph's last kernel advances it
    Profile& prof = profile();
    const bool timed = prof.on;  // per-kernel events need plain launches
    std::vector<hipEvent_t> ev;
    int ntimed = 0;             // timed launches
    int64_t timed_steps = 0;    // and the steps in them
    auto event_before = [&] {
        while ((int)ev.size() < 2 * (ntimed + 1)) {
            hipEvent_t e;
            BLQH_HIP(hipEventCreate(&e));
            ev.push_back(e);
        }
        BLQH_HIP(hipEventRecord(ev[2 * ntimed], st));
    };
    auto event_after = [&](int steps) {
        BLQH_HIP(hipEventRecord(ev[2 * ntimed++ + 1], st));
        timed_steps += steps;
    };
    auto chunk = [&](bool record, int first) {
        for (int k = 0; k < chk; ++k) {
            const bool t = record && first + k < cap;
            if (t) event_before();
            launch_b1<true>(b, S, k, nullptr, nullptr, pl.part1.get(), st);
            if (t) event_after(1);
            hipLaunchKernelGGL(k_b2, dim3(b->grid), dim3(kBT), 0, st, S, k);
            hipLaunchKernelGGL(k_b3, dim3(P), dim3(64), 0, st, S, k, P);
        }
        hipLaunchKernelGGL(k_bnext, dim3(1), dim3(64), 0, st, pl.jbase.get(), chk);
    };
    struct EvList {
        std::vector<hipEvent_t>& ev;
        ~EvList() {
            for (auto x : ev) (void)hipEventDestroy(x);
        }
    } evguard{ev};
    const int kinds = (b->has_real ? 2 : 0) | (b->has_complex ? 1 : 0);  // which K1 launches a step has
    const SmallShape shape = small_shape(b);
    const bool small = shape.lds > 0;  // k_bsmall takes the steps
    void (*const bsmall)(BState, const double*, int, int) = b->G ? (shape.res ? k_bsmall<true, true> : k_bsmall<false, true>)
                                                                 : (shape.res ? k_bsmall<true, false> : k_bsmall<false, false>);
    if (small) {
        static const bool attr = (allow_lds(k_bsmall<true, true>, kSmallLdsMax), allow_lds(k_bsmall<false, true>, kSmallLdsMax),
                                  allow_lds(k_bsmall<true, false>, kSmallLdsMax),
                                  allow_lds(k_bsmall<false, false>, kSmallLdsMax), true);
        (void)attr;
    }
    if (!timed && !small && (b->g_chk != chk || b->g_lpr != b->lpr || b->g_cap != cap || b->g_kinds != kinds ||
                   b->g_tab != k1_shape(b) || !b->gexec)) {
        if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
        if (b->graph) (void)hipGraphDestroy(b->graph);
        b->gexec = nullptr;
        b->graph = nullptr;
        if (b->lpr == 64) launch_b1<true>(b, S, 0, nullptr, nullptr, pl.part1.get(), st, false);
        BLQH_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        chunk(false, 0);
        if (hipStreamEndCapture(st, &b->graph) == hipSuccess) {
            BLQH_HIP(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
        } else {  // another thread's call broke the capture: plain launches for this solve
            (void)hipGetLastError();
            b->graph = nullptr;
        }
        b->g_chk = chk;
        b->g_lpr = b->lpr;
        b->g_cap = cap;
        b->g_kinds = kinds;
        b->g_tab = k1_shape(b);
    }
    hipGraphExec_t gexec = b->gexec;
    const int stride = small ? std::max(chk, kSmallSteps) : chk;  // steps queued at a time
    const int zero = 0;
    copy_sync(pl.jbase.get(), &zero, 4, hipMemcpyHostToDevice);

    // pinned staging: alpha/beta read back per replay, active flags (two slots,
    // so a slot is rewritten only after its copy has run)
    char* pin = b->pin;
    double* ha = (double*)pin;
    double* hb = ha + (size_t)P * cap;
    int32_t* actpin = (int32_t*)(hb + (size_t)P * ld);
    // Work lists of the live members only, rebuilt whenever problems
    // converge: the lists deal whole members to XCDs, so without a rebuild
    // the last live members would sit on a few XCDs while the others idle.
    // Every item's sums keep their owner and order, so results do not depend
    // on the lists.  Two pinned slots, as for the active flags.
    int32_t* listpin = actpin + 2 * (size_t)P;
    const size_t list_slot = 2 * (size_t)b->nitems + 28;
    int lslot = 0;
    bool lists_live = false;
    hipEvent_t evc;
    BLQH_HIP(hipEventCreateWithFlags(&evc, hipEventDisableTiming));
    struct EvGuard {
        hipEvent_t e;
        ~EvGuard() { (void)hipEventDestroy(e); }
    } eguard{evc};

    std::vector<std::vector<double>> ritz(P);
    std::vector<int> m(P, 0), steps_run(P, 0);
    std::vector<char> conv(P, 0), live(P, 1);
    std::vector<double> dE(P, INFINITY), resid(P, INFINITY);
    // host threads for the convergence tests: worth it only for many problems
    const int nthr = P >= 32 ? (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency())) : 1;
    if (nthr > 1 && (!b->hpool || b->hpool->size() != nthr)) b->hpool.reset(new HostPool(nthr - 1));
    std::vector<std::vector<double>> svecs(nthr, std::vector<double>(cap));
    std::vector<int> live_ids;
    live_ids.reserve(P);
    // The next replays are queued before the host tests the last ones, so the
    // host test overlaps the GPU; a problem that converged in the tested
    // replays runs the queued ones too, whose steps are never used.  While
    // many problems are live one replay is queued ahead; with a quarter or
    // fewer a replay is short (a few tens of microseconds per step) and the
    // host test of each replay would leave the GPU idle, so two, then four
    // replays go ahead of each test.
    int queued = 0;  // steps queued so far
    auto enqueue = [&](int first) {
        if (small)
            for (int j = first; j < std::min(cap, first + stride); j += kSmallLaunch) {
                const int to = std::min({cap, first + stride, j + kSmallLaunch});
                if (timed) event_before();
                hipLaunchKernelGGL(bsmall, dim3(P), dim3(kSmallT), shape.lds, st, S, b->dtscale.get(), j, to);
                if (timed) event_after(to - j);
            }
        else if (timed || !gexec) chunk(timed, first);
        else BLQH_HIP(hipGraphLaunch(gexec, st));
        BLQH_HIP(hipGetLastError());
    };
    auto enqueue_n = [&](int r) {
        for (int i = 0; i < r && queued < cap; ++i) {
            enqueue(queued);
            queued += stride;
        }
    };
    auto readback = [&]() {
        BLQH_HIP(hipMemcpyAsync(ha, pl.alpha.get(), (size_t)P * cap * 8, hipMemcpyDeviceToHost, st));
        BLQH_HIP(hipMemcpyAsync(hb, pl.beta.get(), (size_t)P * ld * 8, hipMemcpyDeviceToHost, st));
        BLQH_HIP(hipEventRecord(evc, st));
    };
    int done = 0, nlive = P, slot = 0;
    enqueue_n(1);
    readback();
    while (true) {
        const int upto = std::min(cap, queued);  // steps the last readback covers
        const bool more = queued < cap;
        if (more) enqueue_n(4 * nlive > P ? 1 : 16 * nlive > P ? 2 : 4);  // speculative next replays
        BLQH_HIP(hipEventSynchronize(evc));
        // the single-problem solver's convergence test, per live problem
        // (problems split over host threads; each writes only its own entries)
        auto test = [&](int p, std::vector<double>& svec) {
            steps_run[p] = std::min(cap, queued);
            const double* a = ha + (size_t)p * cap;
            const double* bb = hb + (size_t)p * ld;
            for (int j = done; j < upto; ++j) {
                const std::vector<double>& rz = ritz[p];
                const double e = j == 0 ? tridiag_lowest(1, a, bb + 1, nullptr)
                                        : tridiag_lowest_next(j + 1, a, bb + 1, rz[j - 1],
                                                              j > 1 ? std::fabs(rz[j - 1] - rz[j - 2]) : INFINITY);
                ritz[p].push_back(e);
                m[p] = j + 1;
                if (j > 0) dE[p] = std::fabs(ritz[p][j] - ritz[p][j - 1]);
                const double scale = std::max(std::fabs(a[j]), 1.0);
                if (!(bb[j + 1] > 1e-13 * scale) || !std::isfinite(bb[j + 1])) {
                    resid[p] = 0;
                    conv[p] = 1;
                    break;
                }
                if (o.tol > 0 && j > 0 && dE[p] < o.tol) {
                    if (o.res_tol <= 0) { conv[p] = 1; break; }
                    resid[p] = INFINITY;
                    if (residual_exceeds(j + 1, a, bb + 1, ritz[p][j], bb[j + 1], o.res_tol)) continue;
                    (void)tridiag_lowest(j + 1, a, bb + 1, svec.data());
                    resid[p] = bb[j + 1] * std::fabs(svec[j]);
                    if (resid[p] < o.res_tol) { conv[p] = 1; break; }
                }
            }
        };
        {
            live_ids.clear();
            for (int p = 0; p < P; ++p)
                if (live[p]) live_ids.push_back(p);
            const int nl = (int)live_ids.size();
            // a test of m steps takes about 0.1 m us; waking a thread, some 20 us
            const int nt = std::min({nthr, nl, 1 + nl * (upto - done) * upto / 400});
            if (nt <= 1) {
                for (int p : live_ids) test(p, svecs[0]);
            } else {
                b->hpool->run(nt, [&](int t) {
                    for (int i = t; i < nl; i += nt) test(live_ids[i], svecs[t]);
                });
            }
        }
        bool changed = false;
        for (int p = 0; p < P; ++p)
            if (live[p] && conv[p]) {
                live[p] = 0;
                --nlive;
                changed = true;
            }
        done = upto;
        if (!more || nlive == 0) break;
        if (changed) {
            int32_t* dst = actpin + (size_t)slot * P;
            for (int p = 0; p < P; ++p) dst[p] = live[p];
            BLQH_HIP(hipMemcpyAsync(pl.active.get(), dst, P * 4, hipMemcpyHostToDevice, st));
            slot ^= 1;
            if (b->lpr == 64 && !small) {  // k_b1j and k_b1x walk the lists
                std::vector<int32_t> items, seg;
                work_lists(b, &live, items, seg);
                int32_t* lp = listpin + (size_t)lslot * list_slot;
                std::copy(items.begin(), items.end(), lp);
                std::copy(seg.begin(), seg.end(), lp + 2 * b->nitems);
                BLQH_HIP(hipMemcpyAsync(b->xitems.get(), lp, items.size() * 4, hipMemcpyHostToDevice, st));
                BLQH_HIP(hipMemcpyAsync(b->xseg.get(), lp + 2 * b->nitems, 28 * 4, hipMemcpyHostToDevice, st));
                lslot ^= 1;
                lists_live = true;
            }
        }
        readback();
    }
    BLQH_HIP(hipStreamSynchronize(st));  // a speculative replay may still run
    if (lists_live) {  // every member takes part in the final products again
        copy_sync(b->xitems.get(), b->h_xitems.data(), b->h_xitems.size() * 4, hipMemcpyHostToDevice);
        copy_sync(b->xseg.get(), b->h_xseg.data(), 28 * 4, hipMemcpyHostToDevice);
    }

    phase("iterate");
    // pass 2 per problem, then psi = sum_l c_l conj(v_l), normalised, and Re<psi|H psi>
    std::vector<double> hinvb((size_t)P * ld);
    BLQH_HIP(hipMemcpyAsync(hinvb.data(), pl.invb.get(), hinvb.size() * 8, hipMemcpyDeviceToHost, st));
    BLQH_HIP(hipStreamSynchronize(st));
    std::vector<double> w((size_t)P * cap, 0.0), wx((size_t)P * cap, 0.0), E0(P);
    std::vector<int32_t> hm(P);
    for (int p = 0; p < P; ++p)
        BLQH_REQUIRE(m[p] >= 1 && std::isfinite(ritz[p].back()), BLQH_EINTERNAL,
                     "Lanczos produced non-finite coefficients");
    auto pass2 = [&](int p, std::vector<double>& c) {
        c.resize(m[p]);
        E0[p] = tridiag_lowest(m[p], ha + (size_t)p * cap, hb + (size_t)p * ld + 1, c.data());
        for (int l = 0; l < m[p]; ++l) w[(size_t)p * cap + l] = c[l] * hinvb[(size_t)p * ld + l];
        excited_mix(m[p], ha + (size_t)p * cap, hb + (size_t)p * ld + 1, c.data(), wx.data() + (size_t)p * cap);
        for (int l = 0; l < m[p]; ++l) wx[(size_t)p * cap + l] *= hinvb[(size_t)p * ld + l];
        hm[p] = m[p];
        if (!std::isfinite(resid[p])) resid[p] = hb[(size_t)p * ld + m[p]] * std::fabs(c[m[p] - 1]);
    };
    {
        const int nt = std::min(nthr, (P + 3) / 4);  // per-problem results only: any split gives the same values
        if (nt <= 1) {
            for (int p = 0; p < P; ++p) pass2(p, svecs[0]);
        } else {
            b->hpool->run(nt, [&](int t) {
                for (int p = t; p < P; p += nt) pass2(p, svecs[t]);
            });
        }
    }
    BLQH_HIP(hipMemcpyAsync(pl.coef.get(), w.data(), w.size() * 8, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(pl.mvec.get(), hm.data(), P * 4, hipMemcpyHostToDevice, st));
    std::fill(act.begin(), act.end(), 1);
    BLQH_HIP(hipMemcpyAsync(pl.active.get(), act.data(), P * 4, hipMemcpyHostToDevice, st));
    BLQH_HIP(hipMemcpyAsync(pl.coefx.get(), wx.data(), wx.size() * 8, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_bcombine, dim3(b->grid), dim3(kBT), 0, st, S, pl.coef.get(), pl.coefx.get(), pl.mvec.get(),
                       pl.psi.get(), pl.xs.get());
    std::vector<double> hp1(b->nitems), hp2(b->nitems), sc(P);
    BLQH_HIP(hipMemcpyAsync(hp1.data(), pl.part1.get(), b->nitems * 8, hipMemcpyDeviceToHost, st));
    BLQH_HIP(hipStreamSynchronize(st));
    for (int p = 0; p < P; ++p) {
        double s = 0;
        for (int64_t i = b->item0[p]; i < b->item0[p + 1]; ++i) s += hp1[i];
        sc[p] = s > 0 ? 1.0 / std::sqrt(s) : 0.0;
    }
    BLQH_HIP(hipMemcpyAsync(pl.scale.get(), sc.data(), P * 8, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_bscale, dim3(b->grid), dim3(kBT), 0, st, S, pl.scale.get(), pl.psi.get());
    launch_b1<false>(b, S, 0, pl.psi.get(), pl.u.get(), pl.part2.get(), st);
    BLQH_HIP(hipGetLastError());
    BLQH_HIP(hipMemcpyAsync(hp2.data(), pl.part2.get(), b->nitems * 8, hipMemcpyDeviceToHost, st));
    // ground states: all of them in the reference order into u (free after
    // the last SpMV; the start of a continuation solve), then, when any is
    // wanted, one copy of u into pinned staging and host copies into the
    // caller's arrays on the pool threads
    std::vector<BPsi> pj;
    int64_t pmax = 0;
    bool want = false;
    for (int p = 0; p < P; ++p) {
        const blqh_hamil* Hp = b->hs[p];
        pj.push_back({hp[p].n, Hp->ord.on ? Hp->ord.iperm.get() : nullptr, pl.psi.get() + hp[p].voff,
                      pl.u.get() + hp[p].voff});
        pj.push_back({hp[p].n, Hp->ord.on ? Hp->ord.iperm.get() : nullptr, pl.xs.get() + hp[p].voff,
                      pl.xref.get() + hp[p].voff});
        pmax = std::max(pmax, hp[p].n);
        want = want || (psi_out && psi_out[p]);
    }
    DevBuf<BPsi> dpj(pj.size());
    BLQH_HIP(hipMemcpyAsync(dpj.get(), pj.data(), pj.size() * sizeof(BPsi), hipMemcpyHostToDevice, st));
    {
        const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(pmax, kBT), 256));
        for (size_t j0 = 0; j0 < pj.size(); j0 += 65535)
            hipLaunchKernelGGL(k_bpsi_ref, dim3(gx, (unsigned)std::min<size_t>(65535, pj.size() - j0)), dim3(kBT), 0,
                               st, dpj.get() + j0);
        BLQH_HIP(hipGetLastError());
    }
    if (want) {
        if (!b->psi_pin) BLQH_HIP(hipHostMalloc((void**)&b->psi_pin, (size_t)b->rows * sizeof(double2), hipHostMallocDefault));
        BLQH_HIP(hipMemcpyAsync(b->psi_pin, pl.u.get(), (size_t)b->rows * sizeof(double2), hipMemcpyDeviceToHost, st));
    }
    BLQH_HIP(hipStreamSynchronize(st));
    drain.finished = true;
    b->cont_ok = true;
    if (want) {
        auto put = [&](int p) {
            if (psi_out[p]) std::memcpy(psi_out[p], b->psi_pin + hp[p].voff, hp[p].n * sizeof(double2));
        };
        const int nt = std::min(nthr, (P + 3) / 4);
        if (nt <= 1) {
            for (int p = 0; p < P; ++p) put(p);
        } else {
            b->hpool->run(nt, [&](int t) {
                for (int p = t; p < P; p += nt) put(p);
            });
        }
    }
    if (timed) {
        for (int k = 0; k < ntimed; ++k) {
            float ms = 0;
            BLQH_HIP(hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]));
            prof.ms += ms;
        }
        prof.launches += timed_steps;
    }
    phase("finish");
    const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    for (int p = 0; p < P; ++p) {
        double erq = 0;
        for (int64_t i = b->item0[p]; i < b->item0[p + 1]; ++i) erq += hp2[i];
        // bytes of every K1 launch this problem took part in (speculative steps included)
        // (a shared-scale group reads its matrix once for its G problems)
        if (timed)
            prof.bytes += (double)steps_run[p] * (20.0 * b->hs[p]->nnz / (b->G ? b->G : 1) + 56.0 * hp[p].n + 8.0);
        blqh_lanczos_result& r = res[p];
        std::memset(&r, 0, sizeof(r));
        r.E0 = E0[p];
        r.E_rq = erq;
        r.dE = dE[p];
        r.iterations = m[p];
        r.converged = conv[p];
        r.passes = 2;
        r.seconds = secs;
        r.residual = resid[p];
    }
}
