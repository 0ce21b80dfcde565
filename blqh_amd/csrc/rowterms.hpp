// rowterms.hpp -- per-element logic of the basis and Hamiltonian kernels,
// written once for host and device (the CPU test mirror runs the same code).
#pragma once
#include "bits.hpp"

namespace blqh {

// One-body (tunnelling) hop between orbitals n and nt; lo < hi is the range
// whose empty orbitals give the sign (BLQH_without_spin/basis.cpp:187-196).
struct HopTerm {
    int n, nt;
    int lo, hi;
    double coef;  // prefactor including Delta_SAS
    double qre, qim;
    int hasq;
};

struct RowCtx {
    Geo g;
    RankSpec spec;
    int64_t M;      // sector words (lookup-table length)
    int K;          // < 0: no translation reduction (D_l = D_r = 1)
    int spinless;   // operand order of the reference's spinless / spinful expressions
    int twist_sel;  // 1: spinless interlayer pairs, 2: spinful (0,3)/(1,2) pairs
    int mono_odd;   // monolayer with odd nphi: the pair sign counts occupied orbitals (below)
    int uniform;    // no twist and no theta_B phases: H commutes with the translations
    const int16_t* period;
    const int32_t* lut;
    const uint32_t* cnt;
    const uint32_t* rsplit;  // rank shares of a word's halves, null: rank_word (sector_rank)
    int rbits;
    const double* C;     // [2][nphi][nphi] Coulomb table V[alpha][|dm|][|t|]
    const double2* FT;   // [2 nphi - 1]: FT[ql - qr + nphi - 1] = exp(2 pi i (ql - qr) K / order)
    const double2* tw;   // [2 nphi - 1] twist phase per t
};

// True if the translated images of a term between full orbits are equal (a pair hop's up
// to image_count's signs): a translation
// carries the term of ql on to that of ql + 1 with the same element (the Coulomb table is
// symmetric under dm -> nphi - dm, and the signs and phases of a full turn cancel, each
// electron crossing its block's end once).  Rows or targets of shorter period, whose
// phases need not cancel, are summed image by image.
BLQH_HD bool images_equal(const RowCtx& c, int Dl, int Dr) {
    return c.uniform && c.K >= 0 && Dl == c.g.order() && Dr == Dl;
}

BLQH_HD double2 cmul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }

// s mod d from an FP32 reciprocal r of d: the truncated quotient s * r is off
// by at most one for 0 <= s < 2^16, 1 <= d <= 64 and r within 2 ulp of 1/d,
// and one correction step either way makes the remainder exact.
BLQH_HD int mod_by_rcp(int s, int d, float r) {
    const int q = (int)((float)s * r);
    int rem = s - q * d;
    if (rem < 0)
        rem += d;
    else if (rem >= d)
        rem -= d;
    return rem;
}

// s mod d for 0 <= s < 2^16, 1 <= d <= 64.  On the device the quotient comes
// from the hardware's FP32 reciprocal (mod_by_rcp) instead of an integer
// division sequence.
BLQH_HD int mod_small(int s, int d) {
#if defined(__HIP_DEVICE_COMPILE__)
    return mod_by_rcp(s, d, __builtin_amdgcn_rcpf((float)d));
#else
    return s % d;
#endif
}

// Survivor test of the reference's orbit reduction (basis.cpp:82-99): word c
// at position pos(c) of the map's iteration order survives when no other
// orbit member in the sector comes later.
template <class T>
BLQH_HD bool is_survivor(const Geo& g, const RankSpec& s, const T* cnt, const int32_t* posOf, uint64_t c, int32_t p) {
    for (int n = 1; n < g.order(); ++n) {
        int sg;
        const uint64_t c2 = inv_translate(g, c, n, sg);
        if (c2 != c && in_sector(s, c2) && posOf[rank_word(s, cnt, c2)] > p) return false;
    }
    return true;
}

// Lookup-table entry for a sector word y = translate(id[j], q): row j and the
// shift q with inv_translate(y, q) == id[j] as a word.
BLQH_HD int32_t lut_pack(int64_t j, int q) { return (int32_t)((j << 5) | q); }

// rank_word of a sector word.  What the walk over the set bits adds for the upper half
// depends on that half alone, and the state it leaves for the lower one is fixed by the
// lower half itself (its electrons, residual and counts, since the whole is in the sector):
// rank = shares of the two halves, one table entry each (rsplit: the lower half's 2^rbits
// entries, then the upper's), in place of nel dependent steps of some 35 instructions.
BLQH_HD int64_t sector_rank(const RowCtx& c, uint64_t w) {
    if (!c.rsplit) return rank_word(c.spec, c.cnt, w);
    const uint32_t lo = (uint32_t)(w & lowbits(c.rbits)), hi = (uint32_t)(w >> c.rbits) + (1u << c.rbits);
    return (int64_t)c.rsplit[lo] + (int64_t)c.rsplit[hi];
}

// Entry x of rsplit.
BLQH_HD uint32_t rank_share(const RankSpec& s, const uint32_t* cnt, int rbits, uint32_t x) {
    const bool upper = x >> rbits;
    uint64_t w = upper ? (uint64_t)(x - (1u << rbits)) << rbits : (uint64_t)x;
    int k = s.nel, r = s.Jt, a = s.nA, b = s.nB;
    if (!upper) {  // the state that a sector word's upper half leaves
        k = popc(w);
        a = s.maskA ? popc(w & s.maskA) : s.nA;
        b = s.maskB ? popc(w & s.maskB) : s.nB;
        r = 0;
        for (int p = 0; p < rbits; ++p)
            if (w >> p & 1) r += p % s.nphi;
        r %= s.R;
        if (k > s.nel || a > s.nA || b > s.nB) return 0;  // in no sector word
    }
    uint32_t rk = 0;
    for (; w; --k) {
        if (k <= 0 || a < 0 || b < 0) return 0;  // in no sector word
        const int p = top_bit(w);
        w ^= 1ULL << p;
        rk += cnt[rs_index(s, p, k, r, a, b)];
        r -= p % s.nphi;
        if (r < 0) r += s.R;
        if (s.R == 1) r = 0;
        a -= (int)((s.maskA >> p) & 1ULL);
        b -= (int)((s.maskB >> p) & 1ULL);
    }
    return rk;
}

// Row j of the orbit of sector word Rs, the table's shift q1
// (inv_translate(Rs, q1) == id[j]) and j's period Dr.
BLQH_HD bool locate_word(const RowCtx& c, uint64_t Rs, int& j, int& q1, int& Dr) {
    const int64_t rk = sector_rank(c, Rs);
    if (rk < 0 || rk >= c.M) return false;  // defensive: unreachable for sector words
    const int32_t e = c.lut[rk];
    if (e < 0) return false;
    j = e >> 5;
    q1 = e & 31;
    Dr = c.K < 0 ? 1 : c.period[j];
    return true;
}

// Representative of a hop target.  L = translate(id[i], ql) carries momentum
// J + ql*nel, so R0 (same momentum) is first rotated back by ql into the
// sector; the table then gives (j, q1) and the reference's shift is
// qr = (ql + q1) mod D_r, the unique qr < D_r with inv_translate(R0, qr) ==
// id[j] (lanczos_hamiltonian.cpp:147-165).  Its sign is recomputed for qr:
// rotating by the period itself may carry a fermion sign.
BLQH_HD bool locate(const RowCtx& c, uint64_t R0, int ql, int& j, int& qr, int& Dr, int& sr) {
    int s0, q1;
    const uint64_t Rs = ql ? inv_translate(c.g, R0, ql, s0) : R0;
    if (!locate_word(c, Rs, j, q1, Dr)) return false;
    if (c.K < 0) {
        qr = 0;
        sr = 1;
        return true;
    }
    qr = mod_small(ql + q1, Dr);
    (void)inv_translate(c.g, R0, qr, sr);
    return true;
}

// Pair hop n -> n + t, m -> m - t, each orbital shifted within its block
// (layer / species; |t| < nphi) with wrap-around.
struct PairHop {
    int a, b;      // blocks of n and m
    int n0, xm;    // n's orbital and m's target orbital within their blocks
    bool wn, wm;   // the electron wraps around its block
    int nt, mt;    // target orbitals
    uint64_t word; // L with n, m moved to nt, mt
};

// Targets of the pair hop of n and m (both occupied in L) by t; false when
// the hop is blocked (the targets coincide, or another electron of L holds
// one of them).  The compares replace integer divisions.
BLQH_HD bool pair_hop(int nphi, uint64_t L, int n, int m, int t, PairHop& h) {
    h.a = n >= nphi ? (n >= 2 * nphi ? (n >= 3 * nphi ? 3 : 2) : 1) : 0;
    h.b = m >= nphi ? (m >= 2 * nphi ? (m >= 3 * nphi ? 3 : 2) : 1) : 0;
    h.n0 = n - h.a * nphi;
    const int m0 = m - h.b * nphi;
    int xn = h.n0 + t, xm = m0 - t;
    h.wn = xn < 0 || xn >= nphi;
    h.wm = xm < 0 || xm >= nphi;
    xn += xn < 0 ? nphi : (xn >= nphi ? -nphi : 0);
    xm += xm < 0 ? nphi : (xm >= nphi ? -nphi : 0);
    h.xm = xm;
    h.nt = h.a * nphi + xn;
    h.mt = h.b * nphi + xm;
    const uint64_t rest = L ^ ((1ULL << n) | (1ULL << m));
    const uint64_t tgt = (1ULL << h.nt) | (1ULL << h.mt);
    h.word = rest | tgt;
    return h.nt != h.mt && !(rest & tgt);
}

// Two-body element of the open pair hop h of L (pair n < m, shift t) whose
// target lies in the orbit of row j (sector-table shift q1, period Dr).
// BLQH_without_spin/lanczos_hamiltonian.cpp:109-292, BLQH_with_spin/lanczos_hamiltonian.cpp:109-712.
BLQH_HD void pair_value(const RowCtx& c, uint64_t L, int signl, int Dl, int ql, int n, int m, int t, const PairHop& h,
                        int q1, int Dr, double& re, double& im) {
    const int nphi = c.g.nphi;
    const int a = h.a, b = h.b, n0 = h.n0, xm = h.xm, nt = h.nt, mt = h.mt;
    int qr = 0, sr = 1;
    if (c.K >= 0) {
        qr = mod_small(ql + q1, Dr);
        (void)inv_translate(c.g, h.word, qr, sr);
    }
    // The monolayer counts occupied orbitals between n and nt (and m and mt)
    // where sign2 counts empty ones (Monolayer/basis.cpp:169-195).  The counts
    // add up to |nt - n| - 1 and |mt - m| - 1, whose sum is even unless
    // exactly one of the two electrons wraps, and then has the parity of nphi.
    const int sign = sign2(L, n, m, nt, mt) * signl * sr * (c.mono_odd && h.wn != h.wm ? -1 : 1);
    const int sh = c.g.S == 4 ? 1 : 0;  // layer of block a: a / (S / 2)
    const int alpha = (a >> sh) != (b >> sh) ? 1 : 0;
    int dm = xm - n0;
    dm = dm < 0 ? -dm : dm;
    const int at = t < 0 ? -t : t;
    const double Cv = c.C[alpha * nphi * nphi + dm * nphi + at];
    double2 ft = c.FT[ql - qr + nphi - 1];
    const bool twisted = c.twist_sel == 1 ? (a != b) : (c.twist_sel == 2 && ((a == 0 && b == 3) || (a == 1 && b == 2)));
    if (twisted) ft = cmul(ft, c.tw[t + nphi - 1]);
    const double sq = sqrt((double)(Dl * Dr));
    if (c.spinless) {
        const double den = sq * sign;
        re = (ft.x * Cv) / den;
        im = (ft.y * Cv) / den;
    } else {
        const double cs = Cv * sign;
        re = (cs * ft.x) / sq;
        im = (cs * ft.y) / sq;
    }
}

// Two-body term: pair (n < m) occupied in L = translate(id[i], ql), shift t.
// Returns false when the hop is blocked or its target has no representative.
BLQH_HD bool pair_term(const RowCtx& c, uint64_t L, int signl, int Dl, int ql, int n, int m, int t, int& j, double& re,
                       double& im) {
    PairHop h;
    if (!pair_hop(c.g.nphi, L, n, m, t, h)) return false;
    int s0, q1, Dr;
    const uint64_t Rs = ql ? inv_translate(c.g, h.word, ql, s0) : h.word;
    if (!locate_word(c, Rs, j, q1, Dr)) return false;
    pair_value(c, L, signl, Dl, ql, n, m, t, h, q1, Dr, re, im);
    return true;
}

// Orbital x moved by k (0 <= k < nphi) within its block, with wrap-around
// (the translation's action on one orbital).
BLQH_HD int rot_in_block(int nphi, int x, int k) {
    const int a = x >= nphi ? (x >= 2 * nphi ? (x >= 3 * nphi ? 3 : 2) : 1) : 0;
    int y = x - a * nphi + k;
    y -= y >= nphi ? nphi : 0;
    return a * nphi + y;
}

// Sum of the signs of the Dl = nphi / step equal images of an open pair hop, the first one's
// taken as +1.  In the bilayers the reference's pair sign counts empty orbitals (sign2), which
// for odd nphi turns with each image in which exactly one of the two electrons wraps around
// its block: n in the t rotations that bring it to the block's last t orbitals, m
// in those that bring it to the first t.  (t - nphi: both complements, the same images.)
BLQH_HD int image_count(const RowCtx& c, int Dl, int n, int m, int t, const PairHop& h) {
    const int nphi = c.g.nphi;
    if (c.g.S == 1 || !(nphi & 1)) return Dl;
    const int tt = t < 0 ? t + nphi : t;
    const uint32_t full = (uint32_t)lowbits(nphi), first = (uint32_t)lowbits(tt), last = first << (nphi - tt);
    const int m0 = m - h.b * nphi;
    // bit k: rotation by k (the orbital x moves to (x + k) mod nphi)
    const uint32_t wn = ((last >> h.n0) | (last << (nphi - h.n0))) & full;
    const uint32_t wm = ((first >> m0) | (first << (nphi - m0))) & full;
    const int one = popc((uint64_t)(wn ^ wm));
    return h.wn != h.wm ? 2 * one - Dl : Dl - 2 * one;
}

// The pair hop h (n0 < m0 of the row word L0 = Ls[0], shift t) and its images
// in the translated words Ls[ql] = translate(L0, ql) (signs sgl[ql]), ql < Dl.
// A translation maps the open hops of L0 one to one onto those of Ls[ql] (the
// image moves the rotated orbitals; when the rotation swaps their order the
// image is the pair (m, n) with shift -t), and maps every hop target onto the
// same orbit, so the target (q1, Dr as locate_word gives them) is located once.  Returns
// the sum of the Dl elements, ql ascending, each computed as pair_term computes the
// image's term in Ls[ql]; where the images are equal (images_equal), one element with
// FT / sqrt(Dl Dr) taken Dl times, that is FT.  fold (0 <= t): with the hop of shift
// t - nphi, which has the same target.
BLQH_HD void pair_orbit_value(const RowCtx& c, const uint64_t* Ls, const int* sgl, int Dl, int n0, int m0, int t,
                              PairHop h, int q1, int Dr, bool fold, double& re, double& im) {
    const int nphi = c.g.nphi;
    if (images_equal(c, Dl, Dr)) {
        int sr;
        (void)inv_translate(c.g, h.word, q1, sr);
        const int sign = sign2(Ls[0], n0, m0, h.nt, h.mt) * sr * (c.mono_odd && h.wn != h.wm ? -1 : 1);
        const int sh = c.g.S == 4 ? 1 : 0;
        const int dm = h.xm < h.n0 ? h.n0 - h.xm : h.xm - h.n0, at = t < 0 ? -t : t;
        const double* Cm = c.C + (((h.a >> sh) != (h.b >> sh) ? nphi : 0) + dm) * nphi;
        const double Cv = fold && t ? Cm[at] + Cm[nphi - at] : Cm[at];
        const int cnt = image_count(c, Dl, n0, m0, t, h);
        const double f = cnt == Dl ? (double)sign : sign * ((double)cnt / Dl);
        const double2 ft = c.FT[nphi - 1 - q1];
        re = ft.x * Cv * f;
        im = ft.y * Cv * f;
        return;
    }
    re = 0.0;
    im = 0.0;
    for (int f = 0; f < (fold && t ? 2 : 1); ++f)
        for (int ql = 0; ql < Dl; ++ql) {
            const int k = ql * c.g.step;
            int n = rot_in_block(nphi, n0, k), m = rot_in_block(nphi, m0, k), tq = t - f * nphi;
            if (n > m) {
                const int x = n;
                n = m;
                m = x;
                tq = -tq;
            }
            (void)pair_hop(nphi, Ls[ql], n, m, tq, h);  // open: the image of an open hop
            double r, i;
            pair_value(c, Ls[ql], sgl[ql], Dl, ql, n, m, tq, h, q1, Dr, r, i);
            re += r;
            im += i;
        }
}

// pair_orbit_value of the hop of n0 < m0 by t; the row j of its target.  False when the
// hop is blocked or its target has no representative.
BLQH_HD bool pair_orbit_sum(const RowCtx& c, const uint64_t* Ls, const int* sgl, int Dl, int n0, int m0, int t, int& j,
                            double& re, double& im, bool fold = false) {
    PairHop h;
    if (!pair_hop(c.g.nphi, Ls[0], n0, m0, t, h)) return false;
    int q1, Dr;
    if (!locate_word(c, h.word, j, q1, Dr)) return false;
    pair_orbit_value(c, Ls, sgl, Dl, n0, m0, t, h, q1, Dr, fold, re, im);
    return true;
}

// One-body tunnelling term.  BLQH_without_spin/lanczos_hamiltonian.cpp:295-322,
// BLQH_with_spin/lanczos_hamiltonian.cpp:718-898.
BLQH_HD bool hop_term(const RowCtx& c, uint64_t L, int signl, int Dl, int ql, const HopTerm& h, int& j, int& Dr,
                      double& re, double& im) {
    const uint64_t mask = (1ULL << h.n) | (1ULL << h.nt);
    const uint64_t kn = L & mask;
    if (kn == 0 || kn == mask) return false;
    const uint64_t R0 = L ^ mask;
    if (c.spec.maskA && popc(R0 & c.spec.maskA) != c.spec.nA) return false;
    if (c.spec.maskB && popc(R0 & c.spec.maskB) != c.spec.nB) return false;
    int qr, sr;
    if (!locate(c, R0, ql, j, qr, Dr, sr)) return false;
    const int sign = sign1(L, h.lo, h.hi) * signl * sr;
    const int nphi = c.g.nphi;
    const double cs = h.coef * sign;
    const double2 f = c.FT[ql - qr + nphi - 1];
    double2 v = make_double2(cs * f.x, cs * f.y);
    if (h.hasq) v = cmul(v, make_double2(h.qre, h.qim));
    const double sq = sqrt((double)(Dl * Dr));
    re = v.x / sq;
    im = v.y / sq;
    return true;
}

// The same where the target's period is not asked for.
BLQH_HD bool hop_term(const RowCtx& c, uint64_t L, int signl, int Dl, int ql, const HopTerm& h, int& j, double& re,
                      double& im) {
    int Dr;
    return hop_term(c, L, signl, Dl, ql, h, j, Dr, re, im);
}

// The hop h of the row word L0 and its images in translate(L0, ql), ql < Dl (the hops of the
// rotated orbitals), summed; their targets lie in one orbit, row j.  For hop lists that
// the translations map onto themselves (c.uniform): summed over the list it is the sum of
// hop_term over list and ql.
BLQH_HD bool hop_orbit_sum(const RowCtx& c, uint64_t L0, int Dl, const HopTerm& h, int& j, double& re, double& im) {
    int Dr;
    if (!hop_term(c, L0, 1, Dl, 0, h, j, Dr, re, im)) return false;
    if (images_equal(c, Dl, Dr)) {
        re *= Dl;
        im *= Dl;
        return true;
    }
    for (int ql = 1; ql < Dl; ++ql) {
        const int k = ql * c.g.step;
        HopTerm x = h;
        x.n = rot_in_block(c.g.nphi, h.n, k);
        x.nt = rot_in_block(c.g.nphi, h.nt, k);
        x.lo = x.n < x.nt ? x.n : x.nt;
        x.hi = x.n < x.nt ? x.nt : x.n;
        int s, jq;
        const uint64_t L = translate(c.g, L0, ql, s);
        double r, i;
        if (!hop_term(c, L, s, Dl, ql, x, jq, Dr, r, i)) continue;  // unreachable: the image of an open hop
        re += r;
        im += i;
    }
    return true;
}

// Diagonal: background Ec*nel, charging -d n_U n_L / nphi, bias, Zeeman.
// BLQH_without_spin/lanczos_hamiltonian.cpp:324-339, BLQH_with_spin/lanczos_hamiltonian.cpp:901-908.
BLQH_HD double diag_term(const Geo& g, bool spinless, uint64_t c, double Ecn, double d, double dv, double dz) {
    const int nphi = g.nphi;
    const uint64_t m = lowbits(nphi);
    if (spinless) {
        const int nu = popc(c & m), nl = popc((c >> nphi) & m);
        return (dv > 0 ? 0.5 * dv * (nu - nl) : 0.0) + Ecn + (-d * nu * (g.nel - nu)) / nphi;
    }
    const int n0 = popc(c & m), n1 = popc((c >> nphi) & m), n2 = popc((c >> 2 * nphi) & m),
              n3 = popc((c >> 3 * nphi) & m);
    return Ecn + (-d * (n0 + n1) * (n2 + n3)) / nphi + (-0.5 * dv) * (n0 + n1 - n2 - n3) +
           (-0.5 * dz) * (n0 + n2 - n1 - n3);
}

// Pair index x (row-major over ia < ib) -> (ia, ib) packed as ia | ib << 8.
BLQH_HD unsigned short pair_decode(int nel, int x) {
    int ia = 0, rem = x;
    while (rem >= nel - 1 - ia) {
        rem -= nel - 1 - ia;
        ++ia;
    }
    return (unsigned short)(ia | ((ia + 1 + rem) << 8));
}

}  // namespace blqh
