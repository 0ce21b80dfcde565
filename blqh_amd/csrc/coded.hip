// coded.hip -- builds the coded layout (coded.hpp) of a Hamiltonian from its
// CSR and the internal row order.
//
// The reference's SpMV walks CSR rows (Mat::operator*,
// BLQH_without_spin/matrix.cpp:244-267); this copy is what the hot loops read.
// Stages, all on the device, two host waits and three blocks of memory:
//   k_dict_sample   counts the values of a strided sample in a hash table
//   k_dict_select   keeps the most frequent ones: the table and its lookup hash
//   k_cod_rows      a wavefront per row: columns to the internal order, sorted in
//                   LDS, values looked up; row lengths per panel
//   k_cod_fill / k_cod_rest   a wavefront per slice: step-major runs and the rest
// The kept set depends on the counts alone (every value at or above a count, the
// lowest count whose set fits), so two builds of one matrix give one layout.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "coded.hpp"
#include "engine.hpp"
#include "wavesort.hpp"

namespace {

using namespace blqh;

constexpr int kBlk = 256;
constexpr int kMaxRow = 4096;          // longest CSR row (the build's largest row hash)
constexpr uint64_t kNoKey = ~0ull;     // a NaN pattern: no matrix value
constexpr uint64_t kAbs = 0x7fffffffffffffffull;
constexpr int kHist = 1024;
constexpr double kCover = 0.98;  // share of the sample that makes half a table enough

// lookup hash of the kept values (twice as many slots as the table at most holds)
struct DictHash {
    uint64_t* kr;  // |re| bits
    uint64_t* ki;  // |im| bits (0 for real matrices)
    int32_t* id;   // table index, -1: free
    uint32_t mask_real, mask_cplx;  // slots - 1
};

// The matrix counts as real when every imaginary part is below 1e-14 of its
// largest entry (mx: bits of max |re|, max |im|).
__device__ __forceinline__ bool mx_real(const unsigned long long* mx) {
    const double r = __longlong_as_double((long long)mx[0]), i = __longlong_as_double((long long)mx[1]);
    return i <= 1e-14 * fmax(r, i);
}

__device__ __forceinline__ uint32_t dict_hash(uint64_t r, uint64_t i) {
    uint64_t z = r * 0x9E3779B97F4A7C15ull ^ (i + 0x7F4A7C15ull) * 0xC2B2AE3D27D4EB4Full;
    z ^= z >> 32;
    z *= 0xD6E8FEB86659FD93ull;
    return (uint32_t)(z >> 32);
}

// Fingerprint of a value (never 0): claims a slot of the sample's hash and
// decides equality there.  Two values of one fingerprint would merge their
// counts; the lookup compares the exact bits.
__device__ __forceinline__ uint64_t dict_tag(uint64_t r, uint64_t i) {
    uint64_t z = (r ^ (i << 1 | i >> 63)) * 0xBF58476D1CE4E5B9ull;
    z ^= z >> 29;
    z = (z ^ i * 0x94D049BB133111EBull) * 0x9E3779B97F4A7C15ull;
    z ^= z >> 32;
    return z | 1ull;
}

__global__ void k_dict_sample(int64_t nnz, int64_t samples, const double2* __restrict__ val,
                              const unsigned long long* __restrict__ mx, uint64_t* __restrict__ tag,
                              uint64_t* __restrict__ kr, uint64_t* __restrict__ ki, int32_t* __restrict__ cnt,
                              uint32_t mask) {
    const bool real = mx_real(mx);
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < samples;
         s += (int64_t)gridDim.x * blockDim.x) {
        // sample s sits at a place of its own inside stretch s of the entries
        const int64_t lo = s * nnz / samples, hi = (s + 1) * nnz / samples;
        const int64_t k = lo + (hi - lo > 1 ? (int64_t)((uint32_t)(s * 2654435761u) >> 4) % (hi - lo) : 0);
        const double2 v = val[k];
        const uint64_t r = (uint64_t)__double_as_longlong(v.x) & kAbs;
        const uint64_t i = real ? 0 : (uint64_t)__double_as_longlong(v.y) & kAbs;
        const uint64_t g = dict_tag(r, i);
        uint32_t h = dict_hash(r, i) & mask;
        for (uint32_t probe = 0; probe <= mask; ++probe) {
            uint64_t t = __atomic_load_n(&tag[h], __ATOMIC_RELAXED);
            if (t == 0) {
                t = atomicCAS((unsigned long long*)&tag[h], 0ull, (unsigned long long)g);
                if (t == 0) {
                    kr[h] = r;
                    ki[h] = i;
                    t = g;
                }
            }
            if (t == g) {
                atomicAdd(&cnt[h], 1);
                break;
            }
            h = (h + 1) & mask;
        }
    }
}

// How many values were counted k times, k = 2 .. kHist - 1 (more count as that),
// and their share of the sample (hist[kHist + k]).
__global__ void __launch_bounds__(kHist) k_dict_hist(const uint64_t* __restrict__ tag, const int32_t* __restrict__ cnt,
                                                     uint32_t slots, int32_t* __restrict__ hist) {
    __shared__ int h[2 * kHist];
    h[threadIdx.x] = h[kHist + threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t s = blockIdx.x * kHist + threadIdx.x; s < slots; s += gridDim.x * kHist)
        if (tag[s] && cnt[s] > 1) {
            const int k = min(cnt[s], kHist - 1);
            atomicAdd(&h[k], 1);
            atomicAdd(&h[kHist + k], cnt[s]);
        }
    __syncthreads();
    if (h[threadIdx.x]) {
        atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
        atomicAdd(&hist[kHist + threadIdx.x], h[kHist + threadIdx.x]);
    }
}

// Keeps the values whose count reaches the lowest threshold with at most cap of
// them (half the full table where that covers kCover of the sample): writes them to tab (in the order they are met, which only names the codes)
// and into the lookup hash.  info: kept values, real.
__global__ void __launch_bounds__(kHist) k_dict_select(const uint64_t* __restrict__ tag,
                                                       const uint64_t* __restrict__ kr,
                                                       const uint64_t* __restrict__ ki,
                                                       const int32_t* __restrict__ cnt, uint32_t slots,
                                                       const unsigned long long* __restrict__ mx,
                                                       int samples, const int32_t* __restrict__ hist,
                                                       double* __restrict__ tab, DictHash L,
                                                       int32_t* __restrict__ info) {
    __shared__ int suf[kHist], mass[kHist];
    __shared__ int sthr[2];
    const bool real = mx_real(mx);
    const int cap = real ? kCodReal : kCodCplx;
    const int t = threadIdx.x;
    suf[t] = hist[t];
    mass[t] = hist[kHist + t];
    if (t < 2) sthr[t] = kHist - 1;  // at most 64 values reach that count (kHist - 1 times 64 samples)
    __syncthreads();
    for (int o = 1; o < kHist; o <<= 1) {  // suffix sums
        const int y = t + o < kHist ? suf[t + o] : 0, z = t + o < kHist ? mass[t + o] : 0;
        __syncthreads();
        suf[t] += y;
        mass[t] += z;
        __syncthreads();
    }
    if (t >= 2 && suf[t] <= cap) atomicMin(&sthr[0], t);
    if (t >= 2 && suf[t] <= cap / 2) atomicMin(&sthr[1], t);
    __syncthreads();
    const int thr = mass[sthr[1]] >= kCover * samples ? sthr[1] : sthr[0];
    const uint32_t lmask = real ? L.mask_real : L.mask_cplx;
    for (uint32_t s = blockIdx.x * kHist + t; s < slots; s += gridDim.x * kHist) {
        if (!tag[s] || min(cnt[s], kHist - 1) < thr) continue;
        const int id = atomicAdd(&info[0], 1);
        const uint64_t r = kr[s], i = ki[s];
        if (real) {
            tab[id] = __longlong_as_double((long long)r);
        } else {
            tab[2 * id] = __longlong_as_double((long long)r);
            tab[2 * id + 1] = __longlong_as_double((long long)i);
        }
        uint32_t h = dict_hash(r, i) & lmask;
        for (uint32_t probe = 0; probe <= lmask; ++probe) {
            if (atomicCAS(&L.id[h], -1, id) == -1) {
                L.kr[h] = r;
                L.ki[h] = i;
                break;
            }
            h = (h + 1) & lmask;
        }
    }
    if (blockIdx.x == 0 && t == 0) info[1] = real ? 1 : 0;
}

// A wavefront per internal row r (reference row iperm[r]): key = rest flag and
// internal column in the high word, code, flag and source index in the low one; sorted,
// so the coded entries come first, columns ascending, then the rest, then (marked
// kNoKey) the diagonal, which goes to diag.  skey is
// indexed as the CSR (row iperm[r]'s place).  nu (a shared-scale template): upper-
// layer occupation per internal row; an entry between different ones carries the
// tunnelling flag and is counted.
__global__ void __launch_bounds__(64) k_cod_rows(int64_t n, int64_t npadrows, int npan, int maxrow,
                                                 const int32_t* __restrict__ iperm, const int32_t* __restrict__ perm,
                                                 const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                 const double2* __restrict__ val, DictHash L,
                                                 const int32_t* __restrict__ info, const uint8_t* __restrict__ nu,
                                                 uint64_t* __restrict__ skey, uint16_t* __restrict__ len,
                                                 uint16_t* __restrict__ rlen, double* __restrict__ diag,
                                                 int32_t* __restrict__ ctr) {
    extern __shared__ uint64_t key[];
    const int lane = threadIdx.x;
    const bool real = info[1] != 0;
    const uint32_t lmask = real ? L.mask_real : L.mask_cplx;
    int ntun = 0, dtot = 0;
    for (int64_t r = blockIdx.x; r < npadrows; r += gridDim.x) {
        if (r >= n) {  // padding rows of the last slice
            for (int p = lane; p < npan; p += 64) len[(int64_t)p * npadrows + r] = 0;
            if (lane == 0) rlen[r] = 0;
            continue;
        }
        const int64_t o = iperm ? iperm[r] : r;
        const int64_t s = rowptr[o];
        const int m = (int)(rowptr[o + 1] - s);
        if (m > maxrow) {  // uniform
            if (lane == 0) atomicAdd(&ctr[0], 1);
            continue;
        }
        int P = 64;
        while (P < m) P <<= 1;
        int nrest = 0, ndiag = 0;
        if (lane == 0) {
            diag[real ? r : 2 * r] = 0.0;
            if (!real) diag[2 * r + 1] = 0.0;
        }
        __syncthreads();
        for (int k = lane; k < P; k += 64) {
            uint64_t w = kNoKey;
            if (k < m) {
                const int32_t c0 = col[s + k];
                const uint32_t c = (uint32_t)(perm ? perm[c0] : c0);
                const double2 v = val[s + k];
                if (c0 == o) {
                    diag[real ? r : 2 * r] = v.x;
                    if (!real) diag[2 * r + 1] = v.y;
                    ++ndiag;
                    key[k] = kNoKey;
                    continue;
                }
                const uint64_t br = (uint64_t)__double_as_longlong(v.x), bi = (uint64_t)__double_as_longlong(v.y);
                const uint64_t kr = br & kAbs, ki = real ? 0 : bi & kAbs;
                uint32_t h = dict_hash(kr, ki) & lmask;
                int id = -1;
                for (uint32_t probe = 0; probe <= lmask; ++probe) {
                    const int a = L.id[h];
                    if (a < 0) break;
                    if (L.kr[h] == kr && (real || L.ki[h] == ki)) {
                        id = a;
                        break;
                    }
                    h = (h + 1) & lmask;
                }
                uint32_t code = 0;
                if (id >= 0)
                    code = (uint32_t)id | (uint32_t)((br >> 63) << 15) | (real ? 0u : (uint32_t)((bi >> 63) << 14));
                else
                    ++nrest;
                const bool tun = nu && nu[c] != nu[r];
                ntun += tun;
                w = (uint64_t)(id < 0) << 63 | (uint64_t)c << 32 | code << 16 | (tun ? kCodTun : 0u) | (uint32_t)k;
            }
            key[k] = w;
        }
        for (int q = 32; q > 0; q >>= 1) {
            nrest += __shfl_xor(nrest, q, 64);
            ndiag += __shfl_xor(ndiag, q, 64);
        }
        __syncthreads();
        if (P <= 64) {
            sort_lds<1>(key);
        } else if (P == 128) {
            sort_lds<2>(key);
        } else if (P == 256) {
            sort_lds<4>(key);
        } else if (P == 512) {
            sort_lds<8>(key);
        } else {
            for (int k = 2; k <= P; k <<= 1)
                for (int j = k >> 1; j > 0; j >>= 1) {
                    for (int i = lane; i < P / 2; i += 64) {
                        const int lo = 2 * i - (i & (j - 1)), hi = lo + j;
                        const uint64_t a = key[lo], b = key[hi];
                        if ((a > b) == ((lo & k) == 0)) {
                            key[lo] = b;
                            key[hi] = a;
                        }
                    }
                    __syncthreads();
                }
        }
        __syncthreads();
        for (int k = lane; k < m; k += 64) skey[s + k] = key[k];
        const int nc = m - nrest - ndiag;
        dtot += ndiag;
        for (int p = lane; p < npan; p += 64) {  // entries of panel p: between two lower bounds
            const uint64_t a = (uint64_t)p << 48, b = (uint64_t)(p + 1) << 48;
            int lo = 0, hi = nc;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (key[mid] < a) lo = mid + 1; else hi = mid;
            }
            int lo2 = lo;
            hi = nc;
            while (lo2 < hi) {
                const int mid = (lo2 + hi) >> 1;
                if (key[mid] < b) lo2 = mid + 1; else hi = mid;
            }
            len[(int64_t)p * npadrows + r] = (uint16_t)(lo2 - lo);
        }
        if (lane == 0) rlen[r] = (uint16_t)nrest;
    }
    if (lane == 0 && dtot) atomicAdd(&ctr[2], dtot);
    if (nu) {
        for (int q = 32; q > 0; q >>= 1) ntun += __shfl_xor(ntun, q, 64);
        if (lane == 0 && ntun) atomicAdd(&ctr[1], ntun);
    }
}

// run totals (a wavefront per run of 64 lengths)
__global__ void __launch_bounds__(kBlk) k_cod_runs(int64_t runs, const uint16_t* __restrict__ len,
                                                   int32_t* __restrict__ tot) {
    const int lane = threadIdx.x & 63;
    for (int64_t w = (int64_t)blockIdx.x * (kBlk / 64) + (threadIdx.x >> 6); w < runs;
         w += (int64_t)gridDim.x * (kBlk / 64)) {
        int t = len[w * 64 + lane];
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        if (lane == 0) tot[w] = t;
    }
}

// A wavefront per slice: its coded entries, panel by panel, in step-major order.
__global__ void __launch_bounds__(kBlk) k_cod_fill(int64_t n, int64_t nslices, int npan,
                                                   const int32_t* __restrict__ iperm,
                                                   const int64_t* __restrict__ rowptr,
                                                   const uint64_t* __restrict__ skey, const uint16_t* __restrict__ len,
                                                   const int64_t* __restrict__ base, uint32_t* __restrict__ ent) {
    const int lane = threadIdx.x & 63;
    for (int64_t sl = (int64_t)blockIdx.x * (kBlk / 64) + (threadIdx.x >> 6); sl < nslices;
         sl += (int64_t)gridDim.x * (kBlk / 64)) {
        const int64_t row = sl * 64 + lane;
        const uint64_t* src = skey + (row < n ? rowptr[iperm ? iperm[row] : row] : 0);
        for (int p = 0; p < npan; ++p) {
            const uint32_t ln = len[((int64_t)p * nslices + sl) * 64 + lane];
            uint32_t* out = ent + base[(int64_t)p * nslices + sl];
            uint32_t off = 0;
            for (uint32_t t = 0; __ballot(t < ln) != 0; t += 8) {
                uint64_t w[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) w[u] = t + u < ln ? src[t + u] : 0;
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint64_t m = __ballot(t + u < ln);
                    if (t + u < ln)
                        out[off + lanes_below(m)] = ((uint32_t)(w[u] >> 32) & 0xffffu) |
                                                    ((uint32_t)w[u] & (0xffff0000u | kCodTun));
                    off += (uint32_t)__popcll(m);
                }
            }
            src += ln;
        }
    }
}

// A wavefront per slice: its rest (32-bit column, value), step-major.
__global__ void __launch_bounds__(kBlk) k_cod_rest(int64_t n, int64_t nslices, int npan, int real,
                                                   const int32_t* __restrict__ iperm,
                                                   const int64_t* __restrict__ rowptr,
                                                   const double2* __restrict__ val, const uint64_t* __restrict__ skey,
                                                   const uint16_t* __restrict__ len,
                                                   const uint16_t* __restrict__ rlen,
                                                   const int64_t* __restrict__ rbase, uint32_t* __restrict__ rcol,
                                                   double* __restrict__ rval) {
    const int lane = threadIdx.x & 63;
    for (int64_t sl = (int64_t)blockIdx.x * (kBlk / 64) + (threadIdx.x >> 6); sl < nslices;
         sl += (int64_t)gridDim.x * (kBlk / 64)) {
        const int64_t row = sl * 64 + lane;
        const uint32_t ln = rlen[row];
        const int64_t o = row < n ? (iperm ? iperm[row] : row) : 0;
        const int64_t s = row < n ? rowptr[o] : 0;
        int64_t f = s;  // the row's first rest entry: behind its coded ones
        for (int p = 0; p < npan; ++p) f += len[((int64_t)p * nslices + sl) * 64 + lane];
        int64_t off = rbase[sl];
        for (uint32_t t = 0;; ++t) {
            const uint64_t m = __ballot(t < ln);
            if (m == 0) break;
            if (t < ln) {
                const uint64_t w = skey[f + t];
                const int64_t to = off + lanes_below(m);
                const double2 v = val[s + (int64_t)(w & (kMaxRow - 1))];
                rcol[to] = ((uint32_t)(w >> 32) & 0x7fffffffu) | ((uint32_t)w & kCodTun);
                if (real) {
                    rval[to] = v.x;
                } else {
                    rval[2 * to] = v.x;
                    rval[2 * to + 1] = v.y;
                }
            }
            off += __popcll(m);
        }
    }
}

__global__ void k_cod_totals(const int64_t* __restrict__ a, const int64_t* __restrict__ b, int64_t* __restrict__ out) {
    out[0] = *a;
    out[1] = *b;
}

// arrays of one device block, 256 bytes apart at least
struct Blocks {
    size_t bytes = 0;
    size_t add(size_t b) {
        const size_t at = bytes;
        bytes += (b + 255) / 256 * 256 + (b == 0 ? 256 : 0);
        return at;
    }
};

__global__ void k_fill64(uint64_t* __restrict__ p, int64_t n, uint64_t v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

int grid_waves(int64_t waves) {
    return (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(waves, kBlk / 64), 65536));
}

}  // namespace

namespace blqh {

void build_coded(blqh_hamil* H, const uint8_t* nu, int64_t* ntun) {
    build_order(H);
    hipStream_t st = stream();
    const int64_t n = H->n, nnz = H->nnz, nsl = ceil_div(std::max<int64_t>(n, 1), 64);
    Coded& C = H->cod;
    C.npan = (int)std::max<int64_t>(1, ceil_div(n, (int64_t)kPanelWidth));
    const int32_t* iperm = H->ord.on ? H->ord.iperm.get() : nullptr;
    const int32_t* perm = H->ord.on ? H->ord.perm.get() : nullptr;
    // value sample and table
    const int64_t samples = std::min<int64_t>(nnz, 1 << 16);
    uint32_t slots = 1024;
    while (slots < 2 * samples) slots <<= 1;
    constexpr uint32_t kLook = 2 * (kCodCplx + 1);
    // one block: maxima (2 words), info and counters (4 + 4 ints), totals (2 words), histogram,
    // the sample's hash, the lookup hash, the table in the making, sorted keys, run totals and
    // the scans' scratch
    constexpr size_t kHead = 8 + kHist;
    const int64_t runs = (int64_t)C.npan * nsl, rows = nsl * 64;
    const size_t hash = 3 * (size_t)slots + slots / 2, lookw = 2 * (size_t)kLook + kLook / 2, tabw = 2 * kCodCplx;
    DevBuf<uint64_t> work(kHead + hash + lookw + tabw + (size_t)std::max<int64_t>(nnz, 1) + (runs + nsl + 1) / 2 +
                          scan_scratch(std::max(runs, nsl)));
    unsigned long long* mx = (unsigned long long*)work.get();
    int32_t* info = (int32_t*)(work.get() + 2);
    int32_t* ctr = (int32_t*)(work.get() + 4);
    int64_t* totals = (int64_t*)(work.get() + 6);
    int32_t* hist = (int32_t*)(work.get() + 8);
    uint64_t* tag = work.get() + kHead;
    uint64_t* skr = tag + slots;
    uint64_t* ski = skr + slots;
    int32_t* cnt = (int32_t*)(ski + slots);
    uint64_t* look = ski + slots + slots / 2;
    const DictHash L{look, look + kLook, (int32_t*)(look + 2 * kLook), 2 * (kCodReal + 1) - 1, kLook - 1};
    double* tab = (double*)(look + lookw);
    uint64_t* skey = (uint64_t*)tab + tabw;
    int32_t* tot = (int32_t*)(skey + std::max<int64_t>(nnz, 1));
    int64_t* scan = (int64_t*)(skey + std::max<int64_t>(nnz, 1) + (runs + nsl + 1) / 2);
    auto fill = [&](void* p, int64_t words, uint64_t v) {
        hipLaunchKernelGGL(k_fill64, dim3((unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(words, kBlk), 2048))),
                           dim3(kBlk), 0, st, (uint64_t*)p, words, v);
    };
    fill(work.get(), (int64_t)(kHead + hash), 0);
    fill(L.id, kLook / 2, ~0ull);
    launch_absmax(nnz, H->val.get(), mx, st);
    const unsigned gs = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(samples, kBlk), 2048));
    hipLaunchKernelGGL(k_dict_sample, dim3(gs), dim3(kBlk), 0, st, nnz, samples, H->val.get(), mx, tag, skr, ski, cnt,
                       slots - 1);
    hipLaunchKernelGGL(k_dict_hist, dim3(slots / kHist), dim3(kHist), 0, st, tag, cnt, slots, hist);
    hipLaunchKernelGGL(k_dict_select, dim3(slots / kHist), dim3(kHist), 0, st, tag, skr, ski, cnt, slots, mx,
                       (int)samples, hist, tab, L, info);
    BLQH_HIP(hipGetLastError());
    // rows
    Blocks A;
    const size_t obase = A.add((runs + 1) * 8), orbase = A.add((nsl + 1) * 8),
                 odiag = A.add(2 * (size_t)std::max<int64_t>(n, 1) * 8), olen = A.add((size_t)(runs + nsl) * 64 * 2);
    C.rows.alloc(A.bytes);
    C.base = (int64_t*)(C.rows.get() + obase);
    C.rbase = (int64_t*)(C.rows.get() + orbase);
    C.diag = (double*)(C.rows.get() + odiag);
    C.len = (uint16_t*)(C.rows.get() + olen);
    C.rlen = C.len + (size_t)runs * 64;
    const int gr = (int)std::min<int64_t>(rows, (int64_t)runtime().num_cus * 40);
    int P = 64;  // LDS for the longest row the build can have kept
    const int rmax = std::min<int>(kMaxRow, H->row_max > 0 ? H->row_max : kMaxRow);
    while (P < rmax) P <<= 1;
    hipLaunchKernelGGL(k_cod_rows, dim3(gr), dim3(64), (size_t)P * 8, st, n, rows, C.npan, P, iperm, perm,
                       H->rowptr.get(), H->col.get(), H->val.get(), L, info, nu, skey, C.len, C.rlen, C.diag, ctr);
    hipLaunchKernelGGL(k_cod_runs, dim3(grid_waves(runs + nsl)), dim3(kBlk), 0, st, runs + nsl, C.len, tot);
    exclusive_scan(tot, C.base, runs, st, scan);
    exclusive_scan(tot + runs, C.rbase, nsl, st, scan);
    hipLaunchKernelGGL(k_cod_totals, dim3(1), dim3(1), 0, st, C.base + runs, C.rbase + nsl, totals);
    BLQH_HIP(hipGetLastError());
    int32_t hw[12];
    BLQH_HIP(hipMemcpyAsync(hw, work.get() + 2, 48, hipMemcpyDeviceToHost, st));
    BLQH_HIP(hipStreamSynchronize(st));
    std::memcpy(&C.ncod, hw + 8, 8);
    std::memcpy(&C.nrest, hw + 10, 8);
    C.ntab = hw[0];
    C.real = hw[1] != 0;
    BLQH_REQUIRE(hw[4] == 0, BLQH_EINTERNAL, "a CSR row is longer than the coded layout handles");
    BLQH_REQUIRE(C.ncod + C.nrest + hw[6] == nnz, BLQH_EINTERNAL, "coded layout lost entries");
    if (ntun) *ntun = hw[5];
    Blocks E;
    const size_t oent = E.add((size_t)C.ncod * 4), orval = E.add((size_t)C.nrest * (C.real ? 8 : 16)),
                 orcol = E.add((size_t)C.nrest * 4), otab = E.add(cod_lds_bytes(C.real, C.ntab));
    // a multiple of a 16th of its size, so that the next parameter point's layout, whose split
    // differs by a few entries, finds the block again
    size_t step = 256;
    while (step * 32 <= E.bytes) step *= 2;
    C.words.alloc((E.bytes + step - 1) / step * step);
    C.ent = (uint32_t*)(C.words.get() + oent);
    C.rval = (double*)(C.words.get() + orval);
    C.rcol = (uint32_t*)(C.words.get() + orcol);
    C.tab = (double*)(C.words.get() + otab);
    BLQH_HIP(hipMemcpyAsync(C.tab, tab, cod_lds_bytes(C.real, C.ntab), hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(k_cod_fill, dim3(grid_waves(nsl)), dim3(kBlk), 0, st, n, nsl, C.npan, iperm,
                       H->rowptr.get(), skey, C.len, C.base, C.ent);
    if (C.nrest > 0)
        hipLaunchKernelGGL(k_cod_rest, dim3(grid_waves(nsl)), dim3(kBlk), 0, st, n, nsl, C.npan, C.real ? 1 : 0, iperm,
                           H->rowptr.get(), H->val.get(), skey, C.len, C.rlen, C.rbase, C.rcol, C.rval);
    BLQH_HIP(hipGetLastError());
    BLQH_HIP(hipStreamSynchronize(st));  // complete for solves on other threads' streams
    C.built = true;
}

void ensure_coded(blqh_hamil* H) {
    if (!H->cod.built) build_coded(H, nullptr, nullptr);
}

}  // namespace blqh
