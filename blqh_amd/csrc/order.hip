// order.hip -- the SpMV formats' row order (internal_order, panel.hip) on the device.
//
// A basis state's key (lower layer's smallest rotation, necklace class of the upper layer,
// place in the necklace) takes S nphi + 5 bits; keys and rows go through a stable radix
// sort, eight bits a pass, which gives the order of the host's comparison sort (key, then
// row).  Bound by launches and the scans between them up to a few million rows: 2.05e5
// rows 17 ms on the host, 0.4 ms here.  Keys of more than 64 bits (S nphi > 59) are
// sorted on the host.
#include <algorithm>
#include <cstdlib>
#include <numeric>

#include "engine.hpp"

namespace {

using namespace blqh;

constexpr int kT = 256;               // threads of a workgroup
constexpr int kWaves = kT / 64;
constexpr int kRounds = 16;           // keys per thread
constexpr int kTile = kT * kRounds;   // keys per workgroup
constexpr int kBins = 256;

// Key of row i: for the rotation r that makes (lower word, upper word) smallest, the
// lower word, then the smallest rotation of the upper word and the number of rotations
// from there to the one at r.
__global__ void __launch_bounds__(kT) k_ord_keys(int64_t n, const uint64_t* __restrict__ id, int S, int nphi,
                                                 uint64_t* __restrict__ key, int32_t* __restrict__ idx) {
    const int half = S / 2, hb = half * nphi;
    const uint64_t m = lowbits(nphi);
    // rotate the `half` words of nphi bits in w left by r
    auto rot = [&](uint64_t w, int r) {
        uint64_t g = 0;
        for (int s = 0; s < half; ++s) {
            const uint64_t x = (w >> (s * nphi)) & m;
            g |= (r ? ((x << r) | (x >> (nphi - r))) & m : x) << (s * nphi);
        }
        return g;
    };
    for (int64_t i = blockIdx.x * (int64_t)kT + threadIdx.x; i < n; i += (int64_t)gridDim.x * kT) {
        const uint64_t w = id[i], up = w & lowbits(hb), lo = (w >> hb) & lowbits(hb);
        uint64_t bx = 0, by = 0, cls = 0;
        int rb = 0, r0 = 0;
        for (int r = 0; r < nphi; ++r) {
            const uint64_t x = rot(lo, r), y = rot(up, r);
            if (r == 0 || x < bx || (x == bx && y < by)) {
                bx = x;
                by = y;
                rb = r;
            }
            if (r == 0 || y < cls) {
                cls = y;
                r0 = r;
            }
        }
        // the first rotation past r0 that gives by (by's necklace may have a shorter period)
        int ridx = (rb - r0 + nphi) % nphi;
        for (int k = 0; k < ridx; ++k)
            if (rot(up, (r0 + k) % nphi) == by) ridx = k;
        key[i] = (bx << hb | cls) << 5 | (uint64_t)ridx;
        idx[i] = (int32_t)i;
    }
}

// keys of the tile per digit: cnt[digit * gridDim.x + tile]
__global__ void __launch_bounds__(kT) k_rs_count(int64_t n, const uint64_t* __restrict__ key, int shift,
                                                 int32_t* __restrict__ cnt) {
    __shared__ int h[kBins];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kTile;
    for (int k = threadIdx.x; k < kTile; k += kT)
        if (base + k < n) atomicAdd(&h[(key[base + k] >> shift) & (kBins - 1)], 1);
    __syncthreads();
    cnt[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter of the tile: a wavefront takes kRounds groups of 64 consecutive keys in
// order; within a group the lanes below with the same digit (eight ballots) give the rank.
__global__ void __launch_bounds__(kT) k_rs_scatter(int64_t n, const uint64_t* __restrict__ key,
                                                   const int32_t* __restrict__ idx, int shift,
                                                   const int64_t* __restrict__ off, uint64_t* __restrict__ okey,
                                                   int32_t* __restrict__ oidx) {
    __shared__ int at[kWaves][kBins];  // next place of the wavefront's keys of a digit
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t base = (int64_t)blockIdx.x * kTile + (int64_t)wv * 64 * kRounds + lane;
    for (int w = 0; w < kWaves; ++w) at[w][threadIdx.x] = 0;
    __syncthreads();
    for (int r = 0; r < kRounds; ++r)
        if (base + r * 64 < n) atomicAdd(&at[wv][(key[base + r * 64] >> shift) & (kBins - 1)], 1);
    __syncthreads();
    int p = (int)off[(int64_t)threadIdx.x * gridDim.x + blockIdx.x];
    for (int w = 0; w < kWaves; ++w) {
        const int c = at[w][threadIdx.x];
        at[w][threadIdx.x] = p;
        p += c;
    }
    __syncthreads();
    for (int r = 0; r < kRounds; ++r) {
        const bool on = base + r * 64 < n;
        const uint64_t k = on ? key[base + r * 64] : 0;
        const int d = (int)(k >> shift) & (kBins - 1);
        uint64_t same = __ballot(on);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t m = __ballot(d >> b & 1);
            same &= d >> b & 1 ? m : ~m;
        }
        const int pos = on ? at[wv][d] + lanes_below(same) : 0;
        __syncthreads();  // places read before they advance
        if (on) {
            if ((same >> lane) == 1) at[wv][d] = pos + 1;  // the digit's last lane
            okey[pos] = k;
            oidx[pos] = idx[base + r * 64];
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kT) k_ord_invert(int64_t n, const int32_t* __restrict__ iperm,
                                                   int32_t* __restrict__ perm) {
    for (int64_t r = blockIdx.x * (int64_t)kT + threadIdx.x; r < n; r += (int64_t)gridDim.x * kT)
        perm[iperm[r]] = (int32_t)r;
}

int grid(int64_t n) { return (int)std::min<int64_t>(std::max<int64_t>(ceil_div(n, kT), 1), 65536); }

}  // namespace

namespace blqh {

// internal_order into B->d_perm and B->d_iperm (complete when it returns), once per
// basis; false for the identity order.
bool device_order(const blqh_basis* B) {
    std::lock_guard<std::mutex> lk(B->dord_mu);
    if (B->dord_done) return B->d_perm.get() != nullptr;
    const char* env = std::getenv("BLQH_ORDER");
    const int S = B->geo.S, nphi = B->geo.nphi, bits = S * nphi + 5;
    const int64_t n = B->n;
    hipStream_t st = stream();
    if ((env && env[0] == '0') || B->sec.K < 0 || n < 2 || S < 2) {
        B->dord_done = true;
        return false;
    }
    DevBuf<int32_t> perm(n), iperm(n);
    if (bits > 64) {
        const std::vector<int32_t>& p = internal_order(B);
        BLQH_REQUIRE((int64_t)p.size() == n, BLQH_EINTERNAL, "internal order and basis sizes differ");
        std::vector<int32_t> ip(n);
        for (int64_t i = 0; i < n; ++i) ip[p[i]] = (int32_t)i;
        BLQH_HIP(hipMemcpyAsync(perm.get(), p.data(), n * 4, hipMemcpyHostToDevice, st));
        BLQH_HIP(hipMemcpyAsync(iperm.get(), ip.data(), n * 4, hipMemcpyHostToDevice, st));
        BLQH_HIP(hipStreamSynchronize(st));
    } else {
        const int tiles = (int)ceil_div(n, kTile);
        const int64_t nc = (int64_t)kBins * tiles;
        DevBuf<uint64_t> ka(n), kb(n);
        DevBuf<int32_t> tmp(n), cnt(nc);
        DevBuf<int64_t> off(nc + 1), sums(scan_scratch(nc));
        uint64_t *k0 = ka.get(), *k1 = kb.get();
        const int passes = (bits + 7) / 8;
        int32_t *i0 = passes & 1 ? tmp.get() : iperm.get(), *i1 = passes & 1 ? iperm.get() : tmp.get();
        hipLaunchKernelGGL(k_ord_keys, dim3(grid(n)), dim3(kT), 0, st, n, B->id.get(), S, nphi, k0, i0);
        for (int p = 0; p < passes; ++p) {
            hipLaunchKernelGGL(k_rs_count, dim3(tiles), dim3(kT), 0, st, n, k0, 8 * p, cnt.get());
            exclusive_scan(cnt.get(), off.get(), nc, st, sums.get());
            hipLaunchKernelGGL(k_rs_scatter, dim3(tiles), dim3(kT), 0, st, n, k0, i0, 8 * p, off.get(), k1, i1);
            std::swap(k0, k1);
            std::swap(i0, i1);
        }
        hipLaunchKernelGGL(k_ord_invert, dim3(grid(n)), dim3(kT), 0, st, n, iperm.get(), perm.get());
        BLQH_HIP(hipGetLastError());
        BLQH_HIP(hipStreamSynchronize(st));
    }
    B->d_perm = std::move(perm);
    B->d_iperm = std::move(iperm);
    B->dord_done = true;
    return true;
}

// Row order of H's SpMV formats from the basis order (no-op for the identity order).
void build_order(blqh_hamil* H) {
    blqh_hamil::Order& O = H->ord;
    if (O.on || !device_order(H->basis)) return;
    const int64_t n = H->n;
    BLQH_REQUIRE((int64_t)H->basis->d_perm.n == n, BLQH_EINTERNAL, "internal order and Hamiltonian sizes differ");
    hipStream_t st = stream();
    O.perm.alloc(n);
    O.iperm.alloc(n);
    BLQH_HIP(hipMemcpyAsync(O.perm.get(), H->basis->d_perm.get(), n * 4, hipMemcpyDeviceToDevice, st));
    BLQH_HIP(hipMemcpyAsync(O.iperm.get(), H->basis->d_iperm.get(), n * 4, hipMemcpyDeviceToDevice, st));
    O.on = true;
}

// iperm on the host, fetched on first use (not for several threads at once).
const std::vector<int32_t>& host_iperm(const blqh_hamil* H) {
    if ((int64_t)H->ord.h_iperm.size() != H->n) {
        H->ord.h_iperm.resize(H->n);
        copy_sync(H->ord.h_iperm.data(), H->ord.iperm.get(), H->n * 4, hipMemcpyDeviceToHost);
    }
    return H->ord.h_iperm;
}

}  // namespace blqh
