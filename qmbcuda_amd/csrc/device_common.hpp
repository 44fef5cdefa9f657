// Device helpers shared by the basis and ELL kernels: group action, colex
// rank/unrank, next combination, orbit minimum and row lookup.
//
// S is the state word: uint32_t when the lattice has at most 32 sites (half the
// VALU work of 64-bit words), uint64_t otherwise. The group loops are uniform
// across a wavefront, so the per-element tables are read straight from global
// memory (scalar loads); only lane-divergent tables (binomials, generic
// permutations) are staged in LDS.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "internal.hpp"

namespace qmb {

// Binomial table C(p, j), p < 64, j <= 32, staged in LDS.
constexpr int kBinJ = 33;

__device__ inline int ctz_s(uint32_t x) { return __builtin_ctz(x); }
__device__ inline int ctz_s(uint64_t x) { return __builtin_ctzll(x); }
__device__ inline int clz_s(uint32_t x) { return __builtin_clz(x); }
__device__ inline int clz_s(uint64_t x) { return __builtin_clzll(x); }
__device__ inline int popc_s(uint32_t x) { return __popc(x); }
__device__ inline int popc_s(uint64_t x) { return __popcll(x); }

__device__ inline void stage_perm(uint8_t *perm_lds, const GroupView &g) {
    if (!g.torus)
        for (int i = threadIdx.x; i < g.G * g.n_sites; i += blockDim.x) perm_lds[i] = g.perm[i];
}

// Element tables of the lane-divergent image kernels. A group of cosets (lut 3
// and 4) only takes the images of its coset representatives c_1, c_2, ...: per
// representative one word per nibble value (entry (i - 1) * n_nib * 16 + k * 16 +
// v = the sites that the set bits of v, at sites 4k .. 4k+3, move to), so an
// image is ceil(N / 4) LDS reads instead of one per up spin (at most 128 / N
// cosets: 4 KB). Other groups without a cyclic form stage their permutations.
template <class S>
__device__ inline void stage_images(uint8_t *lds, const GroupView &g) {
    if (g.lut >= 3) {
        S *tab = reinterpret_cast<S *>(lds);
        const int N = g.n_sites, nn = (N + 3) / 4;
        for (int i = threadIdx.x; i < (g.n_cos - 1) * nn * 16; i += blockDim.x) {
            const uint8_t *p = g.perm + (size_t)g.cos_tab[(1 + i / (nn * 16)) * 128] * N;
            const int k = i / 16 % nn, v = i & 15;
            S w = 0;
            for (int b = 0; b < 4; ++b)
                if (((v >> b) & 1) && 4 * k + b < N) w |= (S)1 << p[4 * k + b];
            tab[i] = w;
        }
        return;
    }
    stage_perm(lds, g);
}

__device__ inline void stage_binom(uint64_t *bin_lds, const uint64_t *bin) {
    for (int i = threadIdx.x; i < 64 * kBinJ; i += blockDim.x) bin_lds[i] = bin[i];
}

template <class S>
__device__ inline S full_mask(const GroupView &gv) {
    return (S)gv.full;
}

// Image of state x under element g: the reference's bit move s -> group_el[g][s]
// (Q/exact_diagonalization/utils.cu:52-59), plus the spin flip of this build.
template <class S>
__device__ __forceinline__ S apply_elem(S x, int g, const GroupView &gv, const uint8_t *perm_lds) {
    const S full = (S)gv.full;
    S y;
    if (gv.torus) {
        y = x;
        const unsigned s = gv.small[g];
        if (s) {
            const S k = (S)gv.keep[g];
            y = (S)(((y & k) << s) | ((y & (S)~k & full) >> (gv.block - s)));
        }
        const unsigned b = gv.big[g];
        if (b) y = (S)(((y << b) | (y >> (gv.n_sites - b))) & full);
    } else {
        y = 0;
        const uint8_t *p = perm_lds + g * gv.n_sites;
        S t = x;
        while (t) {
            const int bit = ctz_s(t);
            y |= (S)1 << p[bit];
            t &= t - 1;
        }
    }
    if (gv.flip[g]) y ^= full;
    return y;
}

// LDS copy of the per-element tables for lane-divergent element indices, and
// (when the group has them) the torus orbit-minimum tables.
struct GroupLds {
    uint64_t keep[kMaxGroup];
    uint8_t small[kMaxGroup];
    uint8_t big[kMaxGroup];
    uint8_t flip[kMaxGroup];
    uint8_t lut[kLutBytes];
    uint8_t cos[kCosBytes];
};

__device__ inline void stage_group(GroupLds &t, const GroupView &g) {
    for (int i = threadIdx.x; i < g.G; i += blockDim.x) {
        t.keep[i] = g.keep[i];
        t.small[i] = g.small[i];
        t.big[i] = g.big[i];
        t.flip[i] = g.flip[i];
    }
    if (g.lut == 1 || g.lut == 2 || g.lut == 4)
        for (int i = threadIdx.x; i < kLutBytes; i += blockDim.x) t.lut[i] = g.lut_tab[i];
    if (g.lut >= 3)
        for (int i = threadIdx.x; i < kCosBytes; i += blockDim.x) t.cos[i] = g.cos_tab[i];
}

// LDS tables of the orbit minimum (orbit_min_any). blk (torus products): for a
// block value v the smallest in-block rotation of v and, under flip, of its
// complement (bits 0-7), and the shifts that reach it, plain (bits 8-15) and
// complemented (bits 16-23). einv: inverse element of (flip, shift) o c_i at the
// index of GroupView's element tables, 128 per coset.
struct OrbitLds {
    uint32_t blk[256];
    uint8_t einv[kCosBytes];
};

__device__ inline void stage_orbit(OrbitLds &t, const GroupView &g) {
    if (g.lut == 1 || g.lut == 4) {
        const unsigned mB = (1u << g.block) - 1u;
        for (unsigned v = threadIdx.x; v <= mB; v += blockDim.x) {
            const unsigned a = g.lut_tab[v], b = g.lut_flip ? g.lut_tab[v ^ mB] : 0xFFu, m = a < b ? a : b;
            t.blk[v] = m | (a == m ? (unsigned)g.lut_tab[256 + v] << 8 : 0u) |
                       (b == m && g.lut_flip ? (unsigned)g.lut_tab[256 + (v ^ mB)] << 16 : 0u);
        }
    }
    if (g.lut == 1 || g.lut == 2)
        for (int i = threadIdx.x; i < 128; i += blockDim.x) t.einv[i] = g.inv[g.lut_tab[512 + i]];
    if (g.lut >= 3)
        for (int i = threadIdx.x; i < g.n_cos * 128; i += blockDim.x) t.einv[i] = g.inv[g.cos_tab[i]];
}

// The smallest image found so far. Elements are named by their index in einv:
// the inverse is looked up once at the end, and at ties (which only states with a
// stabiliser have) for the smallest.
template <class S>
struct OrbitBest {
    S best = 0;
    int at = -1;    // index of the only element so far, or -1
    int elem = -1;  // smallest inverse element of several
    int mult = 0;
    __device__ __forceinline__ void take(S y, int i, const OrbitLds &t) {
        if (mult == 0 || y < best) {
            best = y;
            at = i;
            mult = 1;
        } else if (y == best) {
            ++mult;
            const int a = at >= 0 ? (int)t.einv[at] : elem, b = t.einv[i];
            elem = a < b ? a : b;
            at = -1;
        }
    }
    __device__ __forceinline__ int element(const OrbitLds &t) const { return at >= 0 ? (int)t.einv[at] : elem; }
};

// apply_elem with the element index varying across lanes (tables from LDS).
template <class S>
__device__ inline S apply_elem_div(S x, int g, const GroupView &gv, const GroupLds &t, const uint8_t *perm_lds) {
    const S full = (S)gv.full;
    S y;
    if (gv.torus) {
        y = x;
        const unsigned s = t.small[g];
        if (s) {
            const S k = (S)t.keep[g];
            y = (S)(((y & k) << s) | ((y & (S)~k & full) >> (gv.block - s)));
        }
        const unsigned b = t.big[g];
        if (b) y = (S)(((y << b) | (y >> (gv.n_sites - b))) & full);
    } else {
        y = 0;
        const uint8_t *p = perm_lds + g * gv.n_sites;
        S u = x;
        while (u) {
            const int bit = ctz_s(u);
            y |= (S)1 << p[bit];
            u &= u - 1;
        }
    }
    if (t.flip[g]) y ^= full;
    return y;
}

// Colex rank: sum over set bits p_0 < p_1 < ... of C(p_j, j+1); equals the
// reference's GetIndexInHilbertSubspace (utils.cu:9-36).
// (the table's entries: uint64, or the narrow RankOf<S> of stage_binom_rows)
template <class S, class T>
__device__ inline int64_t colex_rank(S x, const T *bin_lds) {
    int64_t r = 0;
    int j = 1;
    while (x) {
        const int p = ctz_s(x);
        r += (int64_t)bin_lds[p * kBinJ + j];
        ++j;
        x &= x - 1;
    }
    return r;
}

// Ranks of narrow states (at most 32 sites) fit 32 bits, table entries too.
template <class S>
struct RankOf {
    using T = uint64_t;
};
template <>
struct RankOf<uint32_t> {
    using T = uint32_t;
};

// The rows of the binomial table that unranking reads, as ranks of S.
template <class S>
__device__ inline void stage_binom_rows(typename RankOf<S>::T *lds, const uint64_t *bin, int n_sites) {
    for (int i = threadIdx.x; i < n_sites * kBinJ; i += blockDim.x) lds[i] = (typename RankOf<S>::T)bin[i];
}

// Inverse of colex_rank for popcount k (k <= 32): from the top site down, site p
// is up when at least C(p, j) states with the j remaining up spins lie below.
// Branch-free (lanes of a wave differ in where their up spins are); C(p, j) = 0
// for p < j places the last ones, and with j = 0 the rank left is 0 < C(p, 0).
template <class S>
__device__ __forceinline__ S colex_unrank(typename RankOf<S>::T r, int k, int n_sites,
                                 const typename RankOf<S>::T *bin_lds) {
    S x = 0;
    int at = (n_sites - 1) * kBinJ + k;
#pragma unroll 4
    for (int p = n_sites - 1; p >= 0; --p) {
        const typename RankOf<S>::T c = bin_lds[at];
        const bool up = r >= c;
        x = (S)((x << 1) | (up ? 1 : 0));
        r -= up ? c : 0;
        at -= kBinJ + (up ? 1 : 0);
    }
    return x;
}

// Next larger integer with the same popcount (ascending = colex order).
template <class S>
__device__ inline S next_comb(S x) {
    const S c = x & (S)(~x + (S)1);
    const S r = x + c;
    return (S)((((r ^ x) >> 2) >> ctz_s(x)) | r);
}

// Position of the k-th set bit of w (k below its number of set bits).
__device__ inline int select_bit(uint64_t w, int k) {
    int pos = 0;
#pragma unroll
    for (int width = 32; width >= 1; width >>= 1) {
        const int c = __popcll(w & ((1ULL << width) - 1ULL));
        const bool up = k >= c;
        k -= up ? c : 0;
        w >>= up ? width : 0;
        pos += up ? width : 0;
    }
    return pos;
}

// Image of x under coset representative c_i (i >= 1) of a lut-3 or lut-4 group:
// one bit reversal when c_i is the site reversal, else the nibble table of
// stage_images.
template <class S>
__device__ inline S reverse_sites(S x, int n);
template <>
__device__ inline uint32_t reverse_sites<uint32_t>(uint32_t x, int n) {
    return __builtin_bitreverse32(x) >> (32 - n);
}
template <>
__device__ inline uint64_t reverse_sites<uint64_t>(uint64_t x, int n) {
    return __builtin_bitreverse64(x) >> (64 - n);
}
template <class S>
__device__ __forceinline__ S coset_image(S x, int ci, const GroupView &gv, const uint8_t *perm_lds) {
    if ((gv.cos_rev >> ci) & 1) return reverse_sites<S>(x, gv.n_sites);
    const int nn = (gv.n_sites + 3) / 4;
    const S *tab = reinterpret_cast<const S *>(perm_lds) + (ci - 1) * nn * 16;
    S y = 0;
    for (int k = 0; k < nn; ++k) y |= tab[k * 16 + (int)((x >> (4 * k)) & 15)];
    return gv.flip[gv.cos_tab[ci * 128]] ? (S)(y ^ (S)gv.full) : y;
}

// Left rotation of an n-site ring state by s (0 <= s < n).
template <class S>
__device__ inline S rotl_ring(S y, int s, int n, S full) {
    return s ? (S)(((y << s) | (y >> (n - s))) & full) : y;
}

// Stabiliser of x for a group of ring rotations times cosets (gv.lut == 3):
// the images of (rotation s, flip f) o c_i are the rotations of c_i x.
template <class S>
__device__ inline void stabiliser_coset(S x, const GroupView &gv, const GroupLds &t, const uint8_t *perm_lds,
                                        uint64_t &stab_lo, uint64_t &stab_hi) {
    const int N = gv.n_sites;
    const S full = (S)gv.full;
    stab_lo = 0;
    stab_hi = 0;
    for (int ci = 0; ci < gv.n_cos; ++ci) {
        const uint8_t *ct = t.cos + ci * 128;
        S y = ci ? coset_image<S>(x, ci, gv, perm_lds) : x;
        for (int s = 0; s < N; ++s) {
            if (s) y = rotl_ring<S>(y, 1, N, full);
            for (int f = 0; f < (gv.lut_flip ? 2 : 1); ++f) {
                if ((f ? (S)(y ^ full) : y) != x) continue;
                const int g = ct[f * 64 + s];
                if (g < 64)
                    stab_lo |= 1ULL << g;
                else
                    stab_hi |= 1ULL << (g - 64);
            }
        }
    }
}

// Stabiliser (elements with image x) of an orbit minimum x; ring groups read the
// element table only for images equal to x.
template <class S>
__device__ inline void stabiliser(S x, const GroupView &gv, const GroupLds &t, const uint8_t *perm_lds,
                                  uint64_t &stab_lo, uint64_t &stab_hi) {
    if (gv.lut == 3) {
        stabiliser_coset<S>(x, gv, t, perm_lds, stab_lo, stab_hi);
        return;
    }
    stab_lo = 0;
    stab_hi = 0;
    if (gv.lut == 2) {
        const int N = gv.n_sites;
        const S full = (S)gv.full;
        S y = x;
        for (int st = 0; st < N; ++st) {
            if (st) y = rotl_ring<S>(y, 1, N, full);
            for (int f = 0; f < (gv.lut_flip ? 2 : 1); ++f) {
                if ((f ? (S)(y ^ full) : y) != x) continue;
                const int g = t.lut[512 + f * 64 + st];
                if (g < 64)
                    stab_lo |= 1ULL << g;
                else
                    stab_hi |= 1ULL << (g - 64);
            }
        }
        return;
    }
    for (int g = 0; g < gv.G; ++g) {
        if (apply_elem<S>(x, g, gv, perm_lds) != x) continue;
        if (g < 64)
            stab_lo |= 1ULL << g;
        else
            stab_hi |= 1ULL << (g - 64);
    }
}

// Orbit minimum of a state and the canonical element gm = the smallest g with
// image_g(min) == x (the reference's orbit_indices entry, utils.cu:66-80, made
// deterministic). mult = the number of elements mapping x to the minimum, i.e.
// the stabiliser size of the minimum (those elements form a coset of x's
// stabiliser, which has the same size as the minimum's).
template <class S>
__device__ __forceinline__ S orbit_min(S x, const GroupView &gv, const uint8_t *perm_lds, int &gm, int &mult) {
    S best = x;
    int bi = gv.inv[0];
    mult = 1;
    for (int g = 1; g < gv.G; ++g) {
        const S y = apply_elem<S>(x, g, gv, perm_lds);
        const int ig = gv.inv[g];
        if (y < best) {
            best = y;
            bi = ig;
            mult = 1;
        } else if (y == best) {
            ++mult;
            if (ig < bi) bi = ig;
        }
    }
    gm = bi;
    return best;
}

// Image of x under the torus element (in-block shift sh, block shift by big
// bits, flip f), formed directly (as apply_elem).
template <class S>
__device__ __forceinline__ S torus_image(S x, int sh, int big, int f, int B, int N, S rep_unit, S full) {
    S y = x;
    if (sh) {
        const S k = (S)(rep_unit * (S)((1u << (B - sh)) - 1u));
        y = (S)(((y & k) << sh) | ((y & (S)~k & full) >> (B - sh)));
    }
    if (big) y = (S)(((y << big) | (y >> (N - big))) & full);
    return f ? (S)(y ^ full) : y;
}

// orbit_min for a group that is the whole torus product (gv.lut == 1), or one
// times cosets (gv.lut == 4: the orbit is the union of the torus orbits of the
// images c_i x). An image's top block is source block j rotated by the in-block
// shift s (complemented under flip), placed on top by the block shift nb-1-j.
// Integer order is decided by the top block first, so the minimum image has the
// smallest top block over all (j, s, f), and only the elements reaching it need
// full images: one table read per block gives its smallest rotation and the
// shifts, and the candidates of all blocks form one list (bit 8 j + s), so a
// wavefront goes round as often as its longest list, not once per block and
// flip. Same result and same gm as orbit_min.
template <class S>
__device__ __forceinline__ S orbit_min_torus(S x, const GroupView &gv, const OrbitLds &t, const uint8_t *perm_lds, bool cosets,
                                    int &gm, int &mult) {
    const int B = gv.block, N = gv.n_sites, nb = N / B;
    const unsigned mB = (1u << B) - 1u;
    const S full = (S)gv.full;
    OrbitBest<S> o;
    unsigned tbest = 0xFFu;
    for (int ci = 0; ci < (cosets ? gv.n_cos : 1); ++ci) {
        const S z = ci ? coset_image<S>(x, ci, gv, perm_lds) : x;
        uint64_t c0 = 0, c1 = 0;
        S v = z;
        for (int j = 0; j < nb; ++j) {
            const unsigned e = t.blk[(unsigned)v & mB];
            v = (S)(v >> B);
            const unsigned m = e & 0xFFu;
            if (m > tbest) continue;
            const uint64_t k0 = (uint64_t)((e >> 8) & 0xFFu) << (8 * j), k1 = (uint64_t)(e >> 16) << (8 * j);
            c0 = m < tbest ? k0 : c0 | k0;
            c1 = m < tbest ? k1 : c1 | k1;
            if (m < tbest) o.mult = 0;  // images of earlier cosets have a larger top block
            tbest = m;
        }
        while (c0 | c1) {
            const bool f = c0 == 0;
            const uint64_t c = f ? c1 : c0;
            const int p = __builtin_ctzll(c);
            if (f)
                c1 = c & (c - 1);
            else
                c0 = c & (c - 1);
            const int sh = p & 7, a = nb - 1 - (p >> 3);
            o.take(torus_image<S>(z, sh, a * B, f, B, N, (S)gv.rep_unit, full), ci * 128 + (f ? 64 : 0) + a * 8 + sh,
                   t);
        }
    }
    gm = o.element(t);
    mult = o.mult;
    return o.best;
}

// Representative test for a full torus product (gv.lut == 1), or one times cosets
// (gv.lut == 4: the orbit is the union of the torus orbits of the images c_i x).
// x is the orbit minimum iff no image is smaller. Only the images whose top
// block reaches x's own, tmin, can be <= x (the others have a larger top block),
// so those candidates decide it, and the ones equal to x are the stabiliser.
// The caller has checked that no rotated block of x itself is below tmin.
template <class S>
__device__ inline bool rep_stab_lut(S x, const GroupView &gv, const GroupLds &t, const uint8_t *perm_lds,
                                    uint64_t &stab_lo, uint64_t &stab_hi) {
    const int B = gv.block, N = gv.n_sites, nb = N / B;
    const unsigned mB = (1u << B) - 1u;
    const unsigned tmin = (unsigned)(x >> ((nb - 1) * B)) & mB;
    const S full = (S)gv.full;
    const int n_cos = gv.lut == 4 ? gv.n_cos : 1;
    stab_lo = 0;
    stab_hi = 0;
    for (int ci = 0; ci < n_cos; ++ci) {
        const uint8_t *ct = gv.lut == 4 ? t.cos + ci * 128 : t.lut + 512;
        const S z = ci ? coset_image<S>(x, ci, gv, perm_lds) : x;
        for (int j = 0; j < nb; ++j) {
            const unsigned v0 = (unsigned)(z >> (j * B)) & mB;
            const int a = nb - 1 - j;
            for (int f = 0; f < (gv.lut_flip ? 2 : 1); ++f) {
                const unsigned v = f ? (v0 ^ mB) : v0;
                if (t.lut[v] > tmin) continue;
                if (t.lut[v] < tmin) return false;
                unsigned sm = t.lut[256 + v];
                while (sm) {
                    const int sh = __builtin_ctz(sm);
                    sm &= sm - 1;
                    const S y = torus_image<S>(z, sh, a * B, f, B, N, (S)gv.rep_unit, full);
                    if (y < x) return false;
                    if (y == x) {
                        const int g = ct[(f * 8 + a) * 8 + sh];
                        if (g < 64)
                            stab_lo |= 1ULL << g;
                        else
                            stab_hi |= 1ULL << (g - 64);
                    }
                }
            }
        }
    }
    return true;
}

// Window scan of the ring orbit minimum: the smallest top byte over the
// rotations of y (and their complements when hf) and the window positions p
// that reach it (c0: plain, c1: complemented). The top 8 bits of rotation s
// are the circular window of y starting at site p = (N - 8 - s) mod N, whose
// bit i is bit p + i of the doubled word. All windows are compared at once,
// bit-sliced from the top bit down: at bit i the candidates whose window bit
// is 0 (complemented: 1) survive if there are any, else bit i of the minimum
// is 1 and every candidate stays.
// Narrow states rotate within N <= 32 bits instead, in 32-bit words.
template <class S>
__host__ __device__ __forceinline__ unsigned ring_candidates(S y, int N, bool hf, S &c0, S &c1) {
    constexpr bool narrow = sizeof(S) == 4;
    const uint64_t yy = narrow ? 0 : (uint64_t)y | ((uint64_t)y << N);  // 8 <= N <= 56: bits p + i < 64
    const S all = (S)((N == 32 && narrow) ? ~(S)0 : (((S)1 << N) - 1));
    S a = all, b = hf ? all : (S)0;
    unsigned tmin = 0;
#pragma unroll
    for (int i = 7; i >= 0; --i) {
        // bit p: site p + i (mod N)
        const S bi = narrow ? (i ? (S)((y >> i) | (y << (N - i))) : y) : (S)(yy >> i);
        const S z0 = a & ~bi, z1 = b & bi;
        const bool any = (z0 | z1) != 0;
        a = any ? z0 : a;
        b = any ? z1 : b;
        tmin |= any ? 0u : (1u << i);
    }
    c0 = a;
    c1 = b;
    return tmin;
}

// ring_candidates with 64-bit masks for both widths: the form of the host check.
template <class S>
__host__ __device__ inline unsigned ring_windows(S y, int N, bool hf, uint64_t &c0, uint64_t &c1) {
    S a, b;
    const unsigned t = ring_candidates<S>(y, N, hf, a, b);
    c0 = a;
    c1 = b;
    return t;
}

// orbit_min for a ring group (gv.lut == 2), or ring rotations times cosets (gv.lut
// == 3: the orbit is the union of the ring orbits of the images c_i x):
// ring_candidates finds the smallest top byte over the rotations (and
// complements) and its positions; only cosets reaching the smallest so far take
// full images of their candidates. Same result and same gm as orbit_min.
template <class S>
__device__ __forceinline__ S orbit_min_ring(S x, const GroupView &gv, const OrbitLds &t, const uint8_t *perm_lds, bool cosets,
                                   int &gm, int &mult) {
    const int N = gv.n_sites;
    const S full = (S)gv.full;
    const bool hf = gv.lut_flip != 0;
    OrbitBest<S> o;
    unsigned tbest = 0x1FFu;
    for (int ci = 0; ci < (cosets ? gv.n_cos : 1); ++ci) {
        const S z = ci ? coset_image<S>(x, ci, gv, perm_lds) : x;
        S c0, c1;
        const unsigned tmin = ring_candidates<S>(z, N, hf, c0, c1);
        if (tmin > tbest) continue;
        tbest = tmin;
        while (c0 | c1) {
            const bool f = c0 == 0;
            const S c = f ? c1 : c0;
            const int p = ctz_s(c);
            if (f)
                c1 = c & (c - 1);
            else
                c0 = c & (c - 1);
            int s = N - 8 - p;
            s += s < 0 ? N : 0;
            const S y = rotl_ring<S>(z, s, N, full);
            o.take(f ? (S)(y ^ full) : y, ci * 128 + (f ? 64 : 0) + s, t);
        }
    }
    gm = o.element(t);
    mult = o.mult;
    return o.best;
}

// The orbit minimum by the group's form: LUT = GroupView::lut where the kernel
// is built for it (its registers and LDS then serve that form alone), -1 for
// the form that the view names.
template <class S, int LUT = -1>
__device__ __forceinline__ S orbit_min_any(S x, const GroupView &gv, const OrbitLds &t, const uint8_t *perm_lds, int &gm,
                                  int &mult) {
    const int lut = LUT < 0 ? gv.lut : LUT;
    if (lut == 1 || lut == 4) return orbit_min_torus<S>(x, gv, t, perm_lds, lut == 4, gm, mult);
    if (lut == 2 || lut == 3) return orbit_min_ring<S>(x, gv, t, perm_lds, lut == 3, gm, mult);
    return orbit_min<S>(x, gv, perm_lds, gm, mult);
}

// Colex rank by nibbles: T[(k * n_c + c) * 16 + v] is the rank contribution of
// nibble k (sites 4k..4k+3) holding v when c set bits lie below it, i.e. the sum
// over v's set bits i (ascending, j of v's bits below i) of C(4k + i, c + j + 1).
// ceil(n_sites / 4) table reads instead of one per set bit; same value as
// colex_rank for every state with at most n_c - 1 set bits.
template <class S, class T>
__host__ __device__ __forceinline__ int64_t colex_rank_nib(S x, const T *tab, int n_nib, int n_c) {
    int64_t r = 0;
    int c = 0;
    for (int k = 0; k < n_nib; ++k) {
        const unsigned v = (unsigned)(x >> (4 * k)) & 15u;
        r += (int64_t)tab[(k * n_c + c) * 16 + (int)v];
        c += __builtin_popcount(v);
    }
    return r;
}

// The nibble rank table in LDS, formed by the block from the staged binomial rows (no
// entry for sites past n_sites is read).
template <class S>
__device__ inline void stage_rank_nib(typename RankOf<S>::T *tab, const typename RankOf<S>::T *bin, int n_sites,
                                      int n_nib, int n_c) {
    for (int i = threadIdx.x; i < n_nib * n_c * 16; i += blockDim.x) {
        const int v = i & 15, c = (i >> 4) % n_c, k = (i >> 4) / n_c;
        typename RankOf<S>::T r = 0;
        int j = c;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (v >> q & 1) {
                ++j;
                if (4 * k + q < n_sites && j < kBinJ) r += bin[(4 * k + q) * kBinJ + j];
            }
        tab[i] = r;
    }
}

// Host: the nibble rank table for n_sites sites and states of n_up set bits
// (n_nib = ceil(n_sites / 4), n_c = n_up + 1); entries that no such state reads
// (more than n_up bits up to that nibble) hold the same formula.
inline std::vector<uint64_t> rank_nibble_table(int n_sites, int n_up, int &n_nib, int &n_c) {
    n_nib = (n_sites + 3) / 4;
    n_c = n_up + 1;
    const int P = 4 * n_nib + 1;
    std::vector<std::vector<uint64_t>> C(P, std::vector<uint64_t>(P + 8, 0));
    for (int n = 0; n < P; ++n) {
        C[n][0] = 1;
        for (int k = 1; k <= n; ++k) C[n][k] = C[n - 1][k - 1] + (k <= n - 1 ? C[n - 1][k] : 0);
    }
    auto binom = [&](int n, int k) -> uint64_t { return (k < 0 || k > n) ? 0 : C[n][k]; };
    std::vector<uint64_t> t((size_t)n_nib * n_c * 16, 0);
    for (int k = 0; k < n_nib; ++k)
        for (int c = 0; c < n_c; ++c)
            for (int v = 0; v < 16; ++v) {
                uint64_t r = 0;
                int j = 0;
                for (int i = 0; i < 4; ++i)
                    if ((v >> i) & 1) {
                        r += binom(4 * k + i, c + j + 1);
                        ++j;
                    }
                t[((size_t)k * n_c + c) * 16 + v] = r;
            }
    return t;
}

// Row of a representative through the rank dictionary (rank -> record -> rows
// before the word + popcount of the lower bits). Returns -1 when the
// representative is not a row.
__device__ __forceinline__ int64_t row_of_rank(int64_t rk, const uint64_t *dict) {
    const ulonglong2 rec = reinterpret_cast<const ulonglong2 *>(dict)[rk >> 6];
    const uint64_t w = rec.x;
    const int b = (int)(rk & 63);
    if (!((w >> b) & 1ULL)) return -1;
    const uint64_t below = b ? (w & ((1ULL << b) - 1ULL)) : 0ULL;
    return (int64_t)rec.y + __popcll(below);
}

template <class S, class T>
__device__ inline int64_t row_of_rep(S rep, const T *bin_lds, const uint64_t *dict) {
    return row_of_rank(colex_rank<S>(rep, bin_lds), dict);
}

}  // namespace qmb
