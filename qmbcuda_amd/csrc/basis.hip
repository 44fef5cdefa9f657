// Symmetry-reduced basis on device.
//
// Replaces the reference's host Sz enumeration plus its five full-sector
// kernels (BuildBasisStates, SetUpSRS, SolveSRS_min, sort/unique,
// SetUpSRS_from_indices, ComputeSRSNorms, ComputeOrbitIndices:
// Q/exact_diagonalization/HeisenbergGenericXXZ_AbelianSymms_CUDA.cu:277-400,
// Q/exact_diagonalization/utils.cu:39-80,716-805). Nothing of size
// C(N,k)*G is materialised:
//   mark    : a state is kept when it is the minimum of its orbit (and, in the
//             compact layout, when the irrep's character is 1 on its stabiliser)
//             -> one bit per state in ascending (colex) order. Cyclic groups
//             first drop groups of 256 states by the bits all of them share,
//             then test the rest one state per lane; other groups and small
//             sectors test runs of consecutive states (next-combination trick);
//   scan    : exclusive popcount scan of the words -> row offsets, stored
//             beside each word (16-byte records);
//   compact : rewrite the kept states in ascending order with their
//             stabiliser size and null flag.
// The records also serve as the rank -> row dictionary of the ELL build
// (replacing the C(N,k)*2 orbit_indices table): one random 16-byte read per
// lookup.
#include <cmath>
#include <cstring>
#include <memory>

#include "device_common.hpp"

qmb::GroupView qmb_basis::view() const {
    qmb::GroupView v;
    v.n_sites = group->n_sites;
    v.G = group->G;
    v.torus = group->torus;
    v.block = group->block;
    v.full = group->n_sites == 64 ? ~0ULL : ((1ULL << group->n_sites) - 1ULL);
    v.rep_unit = 0;
    if (group->torus || group->lut == 4)
        for (int b0 = 0; b0 < group->n_sites; b0 += group->block) v.rep_unit |= 1ULL << b0;
    const uint8_t *t = g_tab.as<uint8_t>();
    v.keep = reinterpret_cast<const uint64_t *>(t);
    v.small = t + o_small;
    v.big = t + o_big;
    v.flip = t + o_flip;
    v.perm = t + o_perm;
    v.inv = t + o_inv;
    v.lut = group->lut;
    v.lut_flip = group->lut_flip;
    v.lut_tab = (group->lut && group->lut != 3) ? t + o_lut : nullptr;
    v.n_cos = group->lut >= 3 ? group->n_cos : 0;
    v.cos_rev = group->lut >= 3 ? group->cos_rev : 0;
    v.cos_tab = group->lut >= 3 ? t + o_cos : nullptr;
    return v;
}

namespace qmb {

// 8 waves per block share the staged binomial and group tables (about 28 KB of
// LDS), so more waves fit a CU than with 4-wave blocks (6x6 sector basis: 43.5
// -> 35 ms)
constexpr int kBasisThreads = 512;

// basis_mark's run length: the longest that still gives this many runs (5x5
// translations without a run test, 5.2 million states: 115 us a basis with 2^20
// runs, 362 us with 2^17).
constexpr int64_t kMinRuns = (int64_t)1 << 20;
// Sectors of this many states and more are marked in two kernels (basis of a
// 28-site ring with flip: 156 us, 421 us with one word per lane in one kernel;
// 22 sites, 705,432 states: equal to basis_mark, 84-90 us; smaller ones lose the
// extra launch and clear: 20 sites, 71 us against 105 us).
constexpr int64_t kRejectDim = (int64_t)1 << 18;
constexpr int64_t kMaxMarkBlocks = 4096;
// basis_compact's words per wavefront: up to 8 with this many wavefronts, more
// with eight times as many (the words at low ranks hold most rows: 28-site ring,
// 627K words, 39 us at 8 a wavefront, 111 us at 64; 25 sites, 81K words, 17 us
// at 8, 29 us at 1, where most wavefronts find no row). Rows whose stabiliser costs
// more want shorter tiles, since the tiles full of rows end last: twice the wavefronts
// for a torus product (4x6 lattice, 42K words, 15.6 us at 2 a wavefront, 23 at 4; 5x6
// 149 at 16, 194 at 32), four times for one with cosets (5x5 with quarter turns, 81K
// words, 34 us at 2, 92 at 8).
constexpr int64_t kMinCompactWaves = 8192;

__device__ inline bool compatible(uint64_t slo, uint64_t shi, uint64_t tlo, uint64_t thi) {
    return ((slo & ~tlo) | (shi & ~thi)) == 0;
}

// True when no state of a run of consecutive sector states can be the minimum of
// its orbit, from the bits that all of them share: those above the highest bit
// in which the run's first and last state differ (the states lie between the
// two as integers). Ring (lut 2, and the ring subgroup of lut 3): the rotation
// that brings shared bit p to the top starts with the shared bits p .. d; when
// these are below the state's own top p - d + 1 bits, the image is smaller.
// Under the flip the complement of the rotation (the unrotated one included)
// likewise. Torus product (lut 1, and the torus subgroup of lut 4): every block inside the shared bits must have
// its smallest in-block rotation at or above the top block.
template <class S>
__device__ inline bool run_rejected(S first, S last, const GroupView &gv, const GroupLds &gt) {
    const int N = gv.n_sites;
    const S diff = first ^ last;
    const int d = diff ? (int)(sizeof(S) * 8) - clz_s(diff) : 0;  // bits d .. N-1 are shared
    const bool hf = gv.lut_flip != 0;
    if (gv.lut == 1 || gv.lut == 4) {
        const int B = gv.block, nb = N / B;
        const unsigned mB = (1u << B) - 1u;
        if (d > (nb - 1) * B) return false;
        const unsigned t = (unsigned)(first >> ((nb - 1) * B)) & mB;
        for (int j = nb - 1; j >= 0 && j * B >= d; --j) {
            const unsigned v = (unsigned)(first >> (j * B)) & mB;
            if (gt.lut[v] < t || (hf && gt.lut[v ^ mB] < t)) return true;
        }
        return false;
    }
    const int m = N - d;
    if (m < 2) return false;
    const S z = first >> d;  // the m shared bits
    if (hf && ((z >> (m - 1)) & 1)) return true;
    for (int len = m - 1; len >= 1; --len) {
        const S top = z >> (m - len), mask = (S)(((S)1 << len) - 1);
        if ((z & mask) < top || (hf && (S)(~z & mask) < top)) return true;
    }
    return false;
}

// Bit i of the result: state i of the run of cnt states from x is a row.
template <class S>
__device__ inline uint64_t mark_run(S x, int cnt, const GroupView &gv, const GroupLds &gt, const uint8_t *perm_lds,
                                    int compact, uint64_t triv_lo, uint64_t triv_hi) {
    uint64_t bits = 0;
    if (gv.lut == 1 || gv.lut == 4) {
        // Full torus product (times cosets for lut 4), two passes. Pass 1 keeps the states whose top block
        // equals the smallest in-block rotation of any block (complemented too
        // under flip): a necessary condition. The top block t is at most its own
        // rotation minimum only when it is one (lut[t] <= t), so the condition
        // is t == lut[t], t <= lut[t ^ mB] under flip, and t <= lut[v], lut[v ^ mB]
        // for the other blocks; the first part rejects most states with two
        // lookups, and since the top block changes rarely in colex order, whole
        // waves take that exit together. Pass 2 takes each lane's survivors in
        // turn (stepping its state forward) and decides them from the candidate
        // images alone.
        const int B = gv.block, nb = gv.n_sites / B;
        const unsigned mB = (1u << B) - 1u;
        const int topsh = (nb - 1) * B;
        const bool hf = gv.lut_flip != 0;
        uint64_t surv = 0;
        S y = x;
        for (int i = 0; i < cnt; ++i) {
            const unsigned t = (unsigned)(y >> topsh) & mB;
            bool ok = gt.lut[t] == t && (!hf || gt.lut[t ^ mB] >= t);
            if (ok) {
                for (int j = 0; j < nb - 1; ++j) {
                    const unsigned v = (unsigned)(y >> (j * B)) & mB;
                    ok = ok && gt.lut[v] >= t && (!hf || gt.lut[v ^ mB] >= t);
                }
            }
            if (ok) surv |= 1ULL << i;
            if (i + 1 < cnt) y = next_comb<S>(y);
        }
        y = x;
        int at = 0;
        while (surv) {
            const int i = __builtin_ctzll(surv);
            surv &= surv - 1;
            for (; at < i; ++at) y = next_comb<S>(y);
            uint64_t slo, shi;
            if (rep_stab_lut<S>(y, gv, gt, perm_lds, slo, shi) && (!compact || compatible(slo, shi, triv_lo, triv_hi)))
                bits |= 1ULL << i;
        }
        return bits;
    }
    if (gv.lut == 2 || gv.lut == 3) {
        // Ring rotations (times cosets for lut 3), two passes. Pass 1 keeps the
        // states that are not above their rotations by 1, 2 and 3 sites (nor,
        // with the spin flip, above their complements or theirs): a necessary
        // condition, branch-free. Pass 2 takes each lane's survivors in turn:
        // per coset c_i one image z = c_i y (the state itself for a plain ring) and
        // the scan of its top bytes (ring_candidates): a smaller byte rules the state
        // out, and only the rotations that reach its own are formed; element
        // indices are looked up only for images equal to the state (stabiliser).
        const int N = gv.n_sites;
        const S full = (S)gv.full;
        const bool hf = gv.lut_flip != 0;
        auto rotl = [&](S v, int k) { return (S)(((v << k) | (v >> (N - k))) & full); };
        uint64_t surv = 0;
        S y = x;
        for (int i = 0; i < cnt; ++i) {
            const S a1 = rotl(y, 1), a2 = rotl(y, 2), a3 = rotl(y, 3);
            bool ok = a1 >= y && a2 >= y && a3 >= y;
            if (hf) ok = ok && (S)(y ^ full) >= y && (S)(a1 ^ full) >= y && (S)(a2 ^ full) >= y && (S)(a3 ^ full) >= y;
            if (ok) surv |= 1ULL << i;
            if (i + 1 < cnt) y = next_comb<S>(y);
        }
        y = x;
        int at = 0;
        while (surv) {
            const int i = __builtin_ctzll(surv);
            surv &= surv - 1;
            for (; at < i; ++at) y = next_comb<S>(y);
            uint64_t slo = 0, shi = 0;
            auto mark = [&](int g) {
                if (g < 64)
                    slo |= 1ULL << g;
                else
                    shi |= 1ULL << (g - 64);
            };
            bool rep = true;
            const unsigned top = (unsigned)(y >> (N - 8));
            const int n_cos = gv.lut == 3 ? gv.n_cos : 1;
            for (int ci = 0; ci < n_cos && rep; ++ci) {
                const uint8_t *ct = gv.lut == 3 ? gt.cos + ci * 128 : gt.lut + 512;
                const S z = ci ? coset_image<S>(y, ci, gv, perm_lds) : y;
                S c0, c1;
                const unsigned tmin = ring_candidates<S>(z, N, hf, c0, c1);
                if (tmin > top) continue;
                rep = tmin == top;
                for (int f = 0; f < (hf ? 2 : 1); ++f) {
                    S c = f ? c1 : c0;
                    while (c && rep) {
                        const int p = ctz_s(c);
                        c &= c - 1;
                        int st = N - 8 - p;
                        if (st < 0) st += N;
                        S v = rotl_ring<S>(z, st, N, full);
                        if (f) v ^= full;
                        if (v < y)
                            rep = false;
                        else if (v == y)
                            mark(ct[f * 64 + st]);
                    }
                }
            }
            if (rep && (!compact || compatible(slo, shi, triv_lo, triv_hi))) bits |= 1ULL << i;
        }
        return bits;
    }
    // One flat loop over (state, element) steps per lane: a lane moves to its
    // next state as soon as an image is smaller (most states exit after a few
    // images), so lanes never wait for a neighbour's full orbit scan.
    int i = 0, g = 1;
    uint64_t slo = 1, shi = 0;  // element 0 (identity) always fixes x
    while (i < cnt) {
        bool done = false, rep = false;
        if (g >= gv.G) {
            done = true;
            rep = true;
        } else {
            const S y = apply_elem_div<S>(x, g, gv, gt, perm_lds);
            if (y < x) {
                done = true;
            } else {
                if (y == x) {
                    if (g < 64)
                        slo |= 1ULL << g;
                    else
                        shi |= 1ULL << (g - 64);
                }
                ++g;
            }
        }
        if (done) {
            if (rep && (!compact || compatible(slo, shi, triv_lo, triv_hi))) bits |= 1ULL << i;
            ++i;
            if (i < cnt) x = next_comb<S>(x);
            g = 1;
            slo = 1;
            shi = 0;
        }
    }
    return bits;
}

// Every state of the sector, for groups without a run test (lut 0) and small
// sectors. A lane takes the 2^ks consecutive states of one run; the 64 >> ks
// lanes of a word join their bits by shuffles. A word per lane (ks = 6) unranks
// once per 64 states but leaves a sector to few wavefronts, the ones at low
// ranks (where most representatives are) running longest.
template <class S>
__global__ __launch_bounds__(kBasisThreads) void basis_mark(GroupView gv, const uint64_t *binom, int n_up,
                                                            int64_t dim, int64_t n_words, int ks, int compact,
                                                            uint64_t triv_lo, uint64_t triv_hi,
                                                            uint64_t *dict) {
    __shared__ alignas(8) uint8_t perm_lds[kMaxGroup * 64];
    __shared__ typename RankOf<S>::T bin[sizeof(S) * 8 * kBinJ];
    __shared__ GroupLds gt;
    stage_images<S>(perm_lds, gv);
    stage_binom_rows<S>(bin, binom, gv.n_sites);
    stage_group(gt, gv);
    __syncthreads();
    const int per_word = 64 >> ks;
    const int64_t runs = n_words << (6 - ks);
    // whole wavefronts step together: the shuffles need every lane
    for (int64_t t0 = (int64_t)blockIdx.x * blockDim.x; t0 < runs; t0 += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = t0 + threadIdx.x;
        const int64_t r0 = t << ks;
        const int64_t left = dim - r0;
        const int cnt = (int)(left < 0 ? 0 : left < (1 << ks) ? left : (1 << ks));
        uint64_t bits = 0;
        if (cnt > 0)
            bits = mark_run<S>(colex_unrank<S>((typename RankOf<S>::T)r0, n_up, gv.n_sites, bin), cnt, gv, gt, perm_lds, compact, triv_lo,
                               triv_hi);
        const int at = (int)(t & (per_word - 1));
        bits <<= at << ks;
        for (int off = 1; off < per_word; off <<= 1) bits |= __shfl_xor(bits, off, 64);
        if (at == 0 && cnt > 0) dict[2 * (t >> (6 - ks))] = bits;
    }
}

// Large sectors, first of two kernels: one group of kRunWords words per lane. A
// group whose states are all ruled out by the bits they share gets its zeros
// here; the others are listed (group indexes, any order) in the second halves
// of the dict records, which the scan fills only later. *count = groups listed.
// On a 26-site ring 6 % (with the flip; 13 % without) of the 64-state words are
// not ruled out, and 1 % more in groups of four, at a quarter of the unranking.
constexpr int kRunWords = 4;

template <class S>
__global__ __launch_bounds__(kBasisThreads) void basis_reject(GroupView gv, const uint64_t *binom, int n_up,
                                                              int64_t dim, int64_t n_words, uint64_t *dict,
                                                              unsigned long long *count) {
    using R = typename RankOf<S>::T;
    __shared__ R bin[sizeof(S) * 8 * kBinJ];
    __shared__ GroupLds gt;
    stage_binom_rows<S>(bin, binom, gv.n_sites);
    stage_group(gt, gv);
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t n_runs = (n_words + kRunWords - 1) / kRunWords;
    for (int64_t t0 = (int64_t)blockIdx.x * blockDim.x; t0 < n_runs; t0 += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = t0 + threadIdx.x;
        bool keep = false;
        if (e < n_runs) {
            const int64_t r0 = e * kRunWords * 64, r1 = min(r0 + kRunWords * 64, dim) - 1;
            keep = !run_rejected<S>(colex_unrank<S>((R)r0, n_up, gv.n_sites, bin),
                                    colex_unrank<S>((R)r1, n_up, gv.n_sites, bin), gv, gt);
            if (!keep)
                for (int64_t w = e * kRunWords; w < min((e + 1) * kRunWords, n_words); ++w) dict[2 * w] = 0;
        }
        const uint64_t m = __ballot(keep);
        if (!m) continue;
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd(count, (unsigned long long)__popcll(m));
        base = __shfl(base, 0, 64);
        if (keep) dict[2 * (base + __popcll(m & ((1ULL << lane) - 1ULL))) + 1] = (uint64_t)e;
    }
}

// Second kernel: one wavefront per word of the listed groups, one state per lane.
template <class S>
__global__ __launch_bounds__(kBasisThreads) void basis_mark_words(GroupView gv, const uint64_t *binom, int n_up,
                                                                  int64_t dim, int64_t n_words, int compact,
                                                                  uint64_t triv_lo, uint64_t triv_hi,
                                                                  uint64_t *dict,
                                                                  const unsigned long long *count) {
    __shared__ alignas(8) uint8_t perm_lds[kMaxGroup * 64];
    __shared__ typename RankOf<S>::T bin[sizeof(S) * 8 * kBinJ];
    __shared__ GroupLds gt;
    stage_images<S>(perm_lds, gv);
    stage_binom_rows<S>(bin, binom, gv.n_sites);
    stage_group(gt, gv);
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t n = (int64_t)*count * kRunWords;
    const int waves = kBasisThreads / 64;
    for (int64_t i = (int64_t)blockIdx.x * waves + (threadIdx.x >> 6); i < n; i += (int64_t)gridDim.x * waves) {
        const int64_t w = (int64_t)dict[2 * (i / kRunWords) + 1] * kRunWords + i % kRunWords;
        if (w >= n_words) continue;
        const int64_t r = w * 64 + lane;
        uint64_t row = 0;
        if (r < dim)
            row = mark_run<S>(colex_unrank<S>((typename RankOf<S>::T)r, n_up, gv.n_sites, bin), 1, gv, gt, perm_lds, compact, triv_lo,
                              triv_hi);
        const uint64_t bits = __ballot(row != 0);
        if (lane == 0) dict[2 * w] = bits;
    }
}

// The rows in ascending order. A wavefront takes tile_words (a power of two, at
// most 64) consecutive words: their records are one coalesced load, and 64 rows
// at a time each lane finds its row's word among the tile's row offsets (a
// search over the lanes by shuffles), its bit and its state. Lanes of a wave
// hold consecutive rows, so the writes are coalesced; a word search in memory
// per row took a chain of ~20 dependent reads. Ring: a state has a stabiliser
// beyond the identity only if a rotation by N / q (q prime; bit N / q of
// periods) fixes it or, with the flip, its complement equals it rotated by N / 2
// (the anti-period's double is a period, and N is the only one left).
template <class S>
__global__ __launch_bounds__(kBasisThreads) void basis_compact(GroupView gv, const uint64_t *binom, int n_up,
                                                               int64_t n_words, int tile_words, uint64_t periods,
                                                               uint64_t triv_lo, uint64_t triv_hi,
                                                               const uint64_t *dict,
                                                               uint64_t *reps, uint8_t *stab, uint8_t *nullf) {
    using R = typename RankOf<S>::T;
    __shared__ alignas(8) uint8_t perm_lds[kMaxGroup * 64];
    __shared__ R bin[sizeof(S) * 8 * kBinJ];
    __shared__ GroupLds gt;
    stage_images<S>(perm_lds, gv);
    stage_binom_rows<S>(bin, binom, gv.n_sites);
    stage_group(gt, gv);
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int waves = kBasisThreads / 64;
    const int64_t n_tiles = (n_words + tile_words - 1) / tile_words;
    const bool narrow_group = gv.lut == 2;
    for (int64_t t = (int64_t)blockIdx.x * waves + (threadIdx.x >> 6); t < n_tiles; t += (int64_t)gridDim.x * waves) {
        const int64_t w = t * tile_words + lane;
        ulonglong2 rec = make_ulonglong2(0, 0);
        if (lane < tile_words && w < n_words) rec = reinterpret_cast<const ulonglong2 *>(dict)[w];
        const int mine = __popcll(rec.x);
        const int64_t row0 = (int64_t)__shfl(rec.y, 0, 64);  // the tile's first word exists
        // rows of the tile before this lane's word; lanes past the tile hold its total
        int before = mine;
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(before, off, 64);
            before += lane >= off ? o : 0;
        }
        const int total = __shfl(before, 63, 64);
        before -= mine;
        for (int q0 = 0; q0 < total; q0 += 64) {
            const int q = min(q0 + lane, total - 1);
            int at = 0;  // last word with at most q rows before it that holds row q
            for (int step = 32; step >= 1; step >>= 1) {
                const int o = __shfl(before, at + step, 64);
                at += o <= q ? step : 0;
            }
            const uint64_t bits = __shfl(rec.x, at, 64);
            const int i = select_bit(bits, q - __shfl(before, at, 64));
            if (q0 + lane >= total) continue;
            const S x = colex_unrank<S>((R)((t * tile_words + at) * 64 + i), n_up, gv.n_sites, bin);
            uint64_t slo = 1, shi = 0;
            if (gv.lut == 1 || gv.lut == 4) {
                rep_stab_lut<S>(x, gv, gt, perm_lds, slo, shi);  // x is a representative: the candidates hold its stabiliser
            } else {
                bool trivial = narrow_group;
                if (narrow_group) {
                    const S full = (S)gv.full;
                    for (uint64_t m = periods; m; m &= m - 1)
                        if (rotl_ring<S>(x, __builtin_ctzll(m), gv.n_sites, full) == x) trivial = false;
                    if (gv.lut_flip && !(gv.n_sites & 1) &&
                        (S)(rotl_ring<S>(x, gv.n_sites / 2, gv.n_sites, full) ^ full) == x)
                        trivial = false;
                }
                if (!trivial) stabiliser<S>(x, gv, gt, perm_lds, slo, shi);
            }
            const int64_t r = row0 + q;
            reps[r] = (uint64_t)x;
            stab[r] = (uint8_t)(__popcll(slo) + __popcll(shi));
            nullf[r] = compatible(slo, shi, triv_lo, triv_hi) ? 0 : 1;
        }
    }
}

template <class S>
__global__ __launch_bounds__(kBasisThreads) void basis_lookup(GroupView gv, const uint64_t *binom, int64_t n,
                                                              const uint64_t *states, const uint64_t *dict,
                                                              int64_t *rows,
                                                              int32_t *elems) {
    __shared__ uint8_t perm_lds[kMaxGroup * 64];
    __shared__ uint64_t bin[64 * kBinJ];
    stage_perm(perm_lds, gv);
    stage_binom(bin, binom);
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int gm, mult;
    const S rep = orbit_min<S>((S)states[i], gv, perm_lds, gm, mult);
    rows[i] = row_of_rep<S>(rep, bin, dict);
    elems[i] = gm;
}

static void upload_group(qmb_basis *b, const qmb_group *g) {
    const size_t G = (size_t)g->G, n = (size_t)g->n_sites;
    auto up16 = [](size_t x) { return (x + 15) & ~(size_t)15; };
    b->o_small = up16(G * 8);
    b->o_big = b->o_small + G;
    b->o_flip = b->o_big + G;
    b->o_inv = b->o_flip + G;
    b->o_perm = up16(b->o_inv + G);
    b->o_lut = up16(b->o_perm + G * n);
    b->o_cos = b->o_lut + kLutBytes;
    const size_t total = up16(b->o_cos + kCosBytes);
    std::vector<uint8_t> h(total, 0);
    std::memcpy(h.data(), g->keep.data(), G * 8);
    for (size_t e = 0; e < G; ++e) {
        h[b->o_small + e] = g->small[e];
        h[b->o_big + e] = g->big[e];
        h[b->o_flip + e] = g->flip[e];
        h[b->o_inv + e] = (uint8_t)g->inv[e];
    }
    for (size_t i = 0; i < G * n; ++i) h[b->o_perm + i] = (uint8_t)g->perm[i];
    if (g->lut && g->lut != 3) std::memcpy(h.data() + b->o_lut, g->lut_tab.data(), kLutBytes);
    if (g->lut >= 3) std::memcpy(h.data() + b->o_cos, g->cos_tab.data(), kCosBytes);
    b->g_tab.alloc(total);
    upload(b->ctx, b->g_tab.p, h.data(), total);
}

static uint64_t binom_host(int n, int k) {
    if (k < 0 || k > n) return 0;
    uint64_t acc = 1;
    for (int i = 1; i <= k; ++i) {
        // exact: acc * (n-k+i) / i stays integral at every step
        unsigned __int128 t = (unsigned __int128)acc * (uint64_t)(n - k + i);
        acc = (uint64_t)(t / (uint64_t)i);
    }
    return acc;
}

}  // namespace qmb

using namespace qmb;

extern "C" {

qmb_status qmb_basis_build(qmb_ctx *ctx, const qmb_group *g, int n_up, int irrep, int layout, qmb_basis **out) {
    return guarded([&] {
        PoolScope pool_scope(ctx ? &ctx->pool : nullptr);
        QMB_REQUIRE(out, "qmb_basis_build: out is NULL");
        *out = nullptr;
        QMB_REQUIRE(ctx && g, "qmb_basis_build: NULL context or group");
        QMB_REQUIRE(n_up >= 0 && n_up <= g->n_sites, "qmb_basis_build: n_up out of range");
        QMB_REQUIRE(n_up <= 32, "qmb_basis_build: at most 32 up spins (use the flipped sector)");
        QMB_REQUIRE(irrep >= 0 && irrep < g->n_irreps, "qmb_basis_build: irrep out of range");
        QMB_REQUIRE(g->irrep_ok[irrep], "qmb_basis_build: character row " + std::to_string(irrep) +
                                            " is not a one-dimensional representation of the group");
        QMB_REQUIRE(layout == QMB_LAYOUT_REFERENCE || layout == QMB_LAYOUT_COMPACT, "qmb_basis_build: bad layout");
        for (int e = 0; e < g->G; ++e)
            QMB_REQUIRE(!g->flip[e] || 2 * n_up == g->n_sites,
                        "qmb_basis_build: spin flip needs n_up == n_sites/2");
        const uint64_t dim = binom_host(g->n_sites, n_up);
        QMB_REQUIRE(dim > 0 && dim <= (1ULL << 38), "qmb_basis_build: sector too large for the rank dictionary");
        QMB_HIP(hipSetDevice(ctx->device));
        auto b = std::make_unique<qmb_basis>();
        b->ctx = ctx;
        b->group = g;
        b->n_sites = g->n_sites;
        b->n_up = n_up;
        b->irrep = irrep;
        b->layout = layout;
        b->sector_dim = (int64_t)dim;
        b->n_words = (int64_t)((dim + 63) / 64);
        const double *ch = &g->chars[(size_t)irrep * g->G * 2];
        b->all_rows = true;
        for (int e = 0; e < g->G; ++e) {
            const bool one = std::fabs(ch[2 * e] - 1.0) < 1e-9 && std::fabs(ch[2 * e + 1]) < 1e-9;
            b->all_rows = b->all_rows && one;
            if (one) {
                if (e < 64)
                    b->triv_lo |= 1ULL << e;
                else
                    b->triv_hi |= 1ULL << (e - 64);
            }
        }
        upload_group(b.get(), g);
        const GroupView gv = b->view();
        b->dict.alloc((size_t)b->n_words * 2 * sizeof(uint64_t));
        const bool narrow = g->n_sites <= 32;
        const int compact = layout == QMB_LAYOUT_COMPACT ? 1 : 0;
        auto blocks_for = [](int64_t threads) {
            return (unsigned)std::min<int64_t>((threads + kBasisThreads - 1) / kBasisThreads, kMaxMarkBlocks);
        };
        if (g->lut && b->sector_dim >= kRejectDim) {
            DevBuf count(sizeof(unsigned long long));
            QMB_HIP(hipMemsetAsync(count.p, 0, sizeof(unsigned long long), ctx->stream));
            hipLaunchKernelGGL(narrow ? basis_reject<uint32_t> : basis_reject<uint64_t>, dim3(blocks_for((b->n_words + kRunWords - 1) / kRunWords)),
                               dim3(kBasisThreads), 0, ctx->stream, gv, ctx->binom.as<uint64_t>(), n_up,
                               b->sector_dim, b->n_words, b->dict.as<uint64_t>(), count.as<unsigned long long>());
            QMB_HIP(hipGetLastError());
            hipLaunchKernelGGL(narrow ? basis_mark_words<uint32_t> : basis_mark_words<uint64_t>,
                               dim3(blocks_for(b->n_words * 64)), dim3(kBasisThreads), 0, ctx->stream, gv,
                               ctx->binom.as<uint64_t>(), n_up, b->sector_dim, b->n_words, compact, b->triv_lo,
                               b->triv_hi, b->dict.as<uint64_t>(), count.as<unsigned long long>());
        } else {
            int ks = 6;
            while (ks > 0 && (b->sector_dim >> ks) < kMinRuns) --ks;
            hipLaunchKernelGGL(narrow ? basis_mark<uint32_t> : basis_mark<uint64_t>,
                               dim3(blocks_for(b->n_words << (6 - ks))), dim3(kBasisThreads), 0, ctx->stream, gv,
                               ctx->binom.as<uint64_t>(), n_up, b->sector_dim, b->n_words, ks, compact, b->triv_lo,
                               b->triv_hi, b->dict.as<uint64_t>());
        }
        QMB_HIP(hipGetLastError());
        const int64_t rows = scan_popcount_dict(ctx, b->dict.as<uint64_t>(), b->n_words);
        QMB_REQUIRE(rows < (int64_t)INT32_MAX, "qmb_basis_build: more than 2^31 rows (int32 columns)");
        b->n_rows = rows;
        b->reps.alloc((size_t)std::max<int64_t>(rows, 1) * sizeof(uint64_t));
        b->stab.alloc((size_t)std::max<int64_t>(rows, 1));
        b->nullf.alloc((size_t)std::max<int64_t>(rows, 1));
        if (rows > 0) {
            int tile_words = 64;
            const int64_t waves = kMinCompactWaves * (g->lut == 4 ? 4 : g->lut == 1 ? 2 : 1);
            while (tile_words > 1 && b->n_words / tile_words < (tile_words > 8 ? 8 : 1) * waves) tile_words /= 2;
            uint64_t periods = 0;
            for (int q = 2, m = g->n_sites; m > 1; ++q)
                for (; m % q == 0; m /= q) periods |= 1ULL << (g->n_sites / q);
            hipLaunchKernelGGL(narrow ? basis_compact<uint32_t> : basis_compact<uint64_t>,
                               dim3(blocks_for((b->n_words + tile_words - 1) / tile_words * 64)),
                               dim3(kBasisThreads), 0, ctx->stream, gv, ctx->binom.as<uint64_t>(), n_up, b->n_words,
                               tile_words, periods, b->triv_lo, b->triv_hi,
                               b->dict.as<uint64_t>(), b->reps.as<uint64_t>(),
                               b->stab.as<uint8_t>(), b->nullf.as<uint8_t>());
            QMB_HIP(hipGetLastError());
        }
        // the compact layout returns with the compaction still queued (the ELL
        // build and every reader order after it on the stream)
        if (layout == QMB_LAYOUT_REFERENCE && rows > 0) {
            QMB_HIP(hipStreamSynchronize(ctx->stream));
            std::vector<uint8_t> nf(rows);
            QMB_HIP(hipMemcpy(nf.data(), b->nullf.p, rows, hipMemcpyDeviceToHost));
            int64_t nn = 0;
            for (auto v : nf) nn += v;
            b->n_null = nn;
        }
        *out = b.release();
    });
}

qmb_status qmb_basis_destroy(qmb_basis *b) {
    if (b && b->ctx) (void)hipStreamSynchronize(b->ctx->stream);
    qmb::release(b);
    return QMB_OK;
}

qmb_status qmb_basis_get_info(const qmb_basis *b, qmb_basis_info *info) {
    return guarded([&] {
        QMB_REQUIRE(b && info, "qmb_basis_get_info: NULL argument");
        info->sector_dim = b->sector_dim;
        info->n_rows = b->n_rows;
        info->n_null = b->n_null;
        info->n_sites = b->n_sites;
        info->n_up = b->n_up;
        info->irrep = b->irrep;
        info->layout = b->layout;
        info->device_bytes = (int64_t)(b->dict.bytes + b->reps.bytes + b->stab.bytes +
                                       b->nullf.bytes);
    });
}

qmb_status qmb_basis_export(const qmb_basis *b, uint64_t *reps, uint16_t *stab, uint8_t *is_null) {
    return guarded([&] {
        QMB_REQUIRE(b, "qmb_basis_export: NULL basis");
        QMB_HIP(hipSetDevice(b->ctx->device));
        QMB_HIP(hipStreamSynchronize(b->ctx->stream));
        const int64_t n = b->n_rows;
        if (n == 0) return;
        if (reps) QMB_HIP(hipMemcpy(reps, b->reps.p, n * sizeof(uint64_t), hipMemcpyDeviceToHost));
        if (stab) {
            std::vector<uint8_t> s(n);
            QMB_HIP(hipMemcpy(s.data(), b->stab.p, n, hipMemcpyDeviceToHost));
            for (int64_t i = 0; i < n; ++i) stab[i] = s[i];
        }
        if (is_null) QMB_HIP(hipMemcpy(is_null, b->nullf.p, n, hipMemcpyDeviceToHost));
    });
}

qmb_status qmb_basis_lookup(const qmb_basis *b, int64_t n, const uint64_t *states, int64_t *row, int32_t *elem) {
    return guarded([&] {
        PoolScope pool_scope(b && b->ctx ? &b->ctx->pool : nullptr);
        QMB_REQUIRE(b && states && row && elem, "qmb_basis_lookup: NULL argument");
        QMB_REQUIRE(n >= 0, "qmb_basis_lookup: negative count");
        if (n == 0) return;
        const uint64_t full = b->n_sites == 64 ? ~0ULL : ((1ULL << b->n_sites) - 1ULL);
        for (int64_t i = 0; i < n; ++i)
            QMB_REQUIRE((states[i] & ~full) == 0 && __builtin_popcountll(states[i]) == b->n_up,
                        "qmb_basis_lookup: state outside the sector");
        qmb_ctx *ctx = b->ctx;
        QMB_HIP(hipSetDevice(ctx->device));
        DevBuf ds(n * sizeof(uint64_t)), dr(n * sizeof(int64_t)), de(n * sizeof(int32_t));
        QMB_HIP(hipMemcpyAsync(ds.p, states, n * sizeof(uint64_t), hipMemcpyHostToDevice, ctx->stream));
        const unsigned blocks = (unsigned)((n + kBasisThreads - 1) / kBasisThreads);
        hipLaunchKernelGGL(b->n_sites <= 32 ? basis_lookup<uint32_t> : basis_lookup<uint64_t>, dim3(blocks), dim3(kBasisThreads), 0, ctx->stream, b->view(),
                           ctx->binom.as<uint64_t>(), n, ds.as<uint64_t>(), b->dict.as<uint64_t>(),
                           dr.as<int64_t>(), de.as<int32_t>());
        QMB_HIP(hipGetLastError());
        QMB_HIP(hipMemcpyAsync(row, dr.p, n * sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream));
        QMB_HIP(hipMemcpyAsync(elem, de.p, n * sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
        QMB_HIP(hipStreamSynchronize(ctx->stream));
    });
}

}  // extern "C"
