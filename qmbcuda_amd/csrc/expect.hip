// Expectation values of Sz-conserving operators in a symmetry-reduced sector.
//
// Replaces the device part of ComputeStaticExpValZeroT
// (Q/exact_diagonalization/HeisenbergGenericXXZ_AbelianSymms_CUDA.cu:421-601):
// the kernel ExpecValArbOperatorAbelianIrrepProjHeisenbergZeroT
// (Q/exact_diagonalization/utils.cu:451-548) and its thrust::reduce.
//
// Rows of the sector matrix represent the states v_r = sum_g conj(chi(g)) g|rep_r>
// (normalised); an eigenvector x of the sector matrix is the many-body state
// Psi = sum_r conj(x_r) v_r. For any operator A with a conjugated term table,
// <Psi|A|Psi> = conj(sum_r conj(x_r) (M x)_r), where M is the sector matrix of the
// group average (1/G) sum_g g A g^-1 (it has the same expectation value as A in
// every state of the sector). Row r of M x, for the element images u = j.rep_r:
//   sum_j sum_terms c(u -> u') conj(chi(j)) chi(gm(u')) (n_t / n_r) x_t / G,
// t = row of the orbit of u', gm(u') = the element taking its representative onto
// u' (the ELL kernel's formula, applied to every image of the source). When A
// commutes with the group the average is A itself and only j = identity is taken.
//
// Two deliberate differences from the reference kernel: it stops the loop over
// the images of a term at the first image the term annihilates (utils.cu:523,
// `if (interr_bool) break;`), dropping the remaining images of S+/S- terms, and it
// accumulates conj(phi_r) conj(V) phi_t, which equals <Psi|A|Psi> only when the
// vector is real up to a phase. Both agree with this kernel for Sz-diagonal
// operators and real vectors.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>

#include "device_common.hpp"
#include "reduce.hpp"
#include "terms.hpp"

namespace qmb {

constexpr int kExpThreads = 256;
constexpr int kExpMaxBlocks = 4096;  // 2048: 87 us for 82 (28 sites)
constexpr size_t kExpRankBytes = 16 * 1024;  // the nibble rank table's LDS
constexpr int kExpLdsTerms = 256;

// A product of Sz alone: 32 B and not a whole TermC (80), so that the few hundred of a
// structure factor stay in the scalar cache (378 terms, 717K rows: 188 / 94 us).
struct SzTerm {
    uint64_t sz;
    double2 coef;
};

// An operator's distinct terms on the device: t[0, n_off) change the state, t[n_off,
// n_terms) are diagonal with a condition, z[0, n_sz) are products of Sz alone.
struct ExpectTerms {
    int n_off, n_terms, n_sz;
    int imag;  // some coefficient has an imaginary part
    int half;  // Hermitian, t[0, n_off) holds only the terms that raise the state
    const TermC *t;
    const SzTerm *z;
};

// An off-diagonal term as the lookups read it, from LDS.
template <class S>
struct ExpectOff {
    double2 coef;
    S set, set_val, sz, pad;
};

// c with the sign of the Sz factors on down spins (down = ~state)
template <class S>
__device__ __forceinline__ double signed_coef(double c, S down, S sz) {
    return __hiloint2double(__double2hiint(c) ^ (int)((unsigned)popc_s((S)(down & sz)) << 31), __double2loint(c));
}

// Partial sums of x_r conj((M x)_r) over the rows, one row a lane. Bound by the
// orbit lookups of the terms that change the state (VALU and LDS): as in the ELL
// passes 64 terms are tested at a time (uniform loads) and each lane then looks its
// own candidates up, so that almost all lanes are busy, with the terms and the rank
// table in LDS and the orbit search of the group's form (LUT). 28 sites, 717K rows,
// seven lookups a row (half): 82 us; with all 14, 147. AVG: every image of the
// representative under the group; taken only when the operator's average has too many
// terms to be formed on the host (ExpectTable).
template <class S, bool CPLX, bool AVG, int LUT>
__global__ __launch_bounds__(kExpThreads, AVG ? 1 : 8) void expect_rows(
    GroupView gv, const uint64_t *binom, int n_nib, int n_c, int layout, int64_t n_rows, const uint64_t *reps,
    const uint8_t *stab, const uint8_t *nullf, const uint64_t *dict, ExpectTerms tv, const double2 *chi,
    const double *nrm, const double *x, double *partials) {
    using R = typename RankOf<S>::T;
    constexpr bool kPerm = LUT != 1 && LUT != 2;
    extern __shared__ __align__(16) unsigned char exp_dyn[];
    __shared__ alignas(8) uint8_t perm_lds[kPerm ? kMaxGroup * 64 : 8];
    __shared__ alignas(8) uint8_t img_lds[AVG ? 4096 : 8];  // coset representatives' images (stage_images)
    __shared__ double2 s_chi[kMaxGroup];
    __shared__ double s_nrm[kMaxGroup + 1];
    __shared__ OrbitLds gt;
    __shared__ double red[kWaves];
    const int n_lds = min(tv.n_off, kExpLdsTerms);
    ExpectOff<S> *off = reinterpret_cast<ExpectOff<S> *>(exp_dyn);
    R *rank = reinterpret_cast<R *>(off + n_lds);
    if (AVG) {
        stage_perm(perm_lds, gv);
        if (gv.lut >= 3) stage_images<S>(img_lds, gv);
    } else if (kPerm) {
        stage_images<S>(perm_lds, gv);
    }
    stage_orbit(gt, gv);
    R *bin = n_nib ? rank + n_nib * n_c * 16 : rank;
    stage_binom_rows<S>(bin, binom, gv.n_sites);
    for (int i = threadIdx.x; i < n_lds; i += blockDim.x) {
        const TermC &tm = tv.t[i];
        off[i] = ExpectOff<S>{tm.coef, (S)tm.set, (S)tm.set_val, (S)tm.sz, 0};
    }
    for (int i = threadIdx.x; i < gv.G; i += blockDim.x) s_chi[i] = chi[i];
    for (int i = threadIdx.x; i <= gv.G; i += blockDim.x) s_nrm[i] = nrm[i];
    __syncthreads();
    if (n_nib) {
        stage_rank_nib<S>(rank, bin, gv.n_sites, n_nib, n_c);
        __syncthreads();
    }
    const uint8_t *images = AVG && gv.lut >= 3 ? img_lds : perm_lds;
    double out_r = 0.0, out_i = 0.0;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n_rows;
         r += (int64_t)gridDim.x * blockDim.x) {
        if (layout == QMB_LAYOUT_REFERENCE && nullf[r]) continue;
        const S rep = (S)reps[r];
        const int m_src = (int)stab[r];
        double dr = 0.0, di = 0.0;  // the diagonal
        double ar = 0.0, ai = 0.0;  // the rest of (M x)_r
        const int n_img = AVG ? gv.G : 1;
        for (int j = 0; j < n_img; ++j) {
            const S u = AVG ? apply_elem<S>(rep, j, gv, perm_lds) : rep;
            const S down = (S)~u;
            // a diagonal term keeps the element: conj(chi(j)) chi(gm) = 1, n_t = n_r
#pragma unroll 8
            for (int h = 0; h < tv.n_sz; ++h) dr += signed_coef<S>(tv.z[h].coef.x, down, (S)tv.z[h].sz);
            if (tv.imag)
                for (int h = 0; h < tv.n_sz; ++h) di += signed_coef<S>(tv.z[h].coef.y, down, (S)tv.z[h].sz);
            for (int h = tv.n_off; h < tv.n_terms; ++h) {
                const TermC &tm = tv.t[h];
                const bool on = (u & (S)tm.req) == (S)tm.req_val;
                dr += on ? signed_coef<S>(tm.coef.x, down, (S)tm.sz) : 0.0;
                if (tv.imag) di += on ? signed_coef<S>(tm.coef.y, down, (S)tm.sz) : 0.0;
            }
            for (int h0 = 0; h0 < tv.n_off; h0 += 64) {
                const int nh = min(64, tv.n_off - h0);
                const TermC *tm0 = tv.t + h0;
                uint32_t lo = 0, hi = 0;
#pragma unroll 8
                for (int h = 0; h < min(32, nh); ++h)
                    lo |= (u & (S)tm0[h].req) == (S)tm0[h].req_val ? 1u << h : 0u;
#pragma unroll 8
                for (int h = 32; h < nh; ++h)
                    hi |= (u & (S)tm0[h].req) == (S)tm0[h].req_val ? 1u << (h - 32) : 0u;
                uint64_t cand = (uint64_t)hi << 32 | lo;
                while (cand) {
                    const int h = h0 + __builtin_ctzll(cand);
                    cand &= cand - 1;
                    ExpectOff<S> o;
                    if (h < n_lds) {
                        o = off[h];
                    } else {
                        const TermC &tm = tv.t[h];
                        o = ExpectOff<S>{tm.coef, (S)tm.set, (S)tm.set_val, (S)tm.sz, 0};
                    }
                    const S tgt = (S)((u & (S)~o.set) | o.set_val);
                    int gm, mult;
                    const S rep2 = orbit_min_any<S, LUT>(tgt, gv, gt, images, gm, mult);
                    const int64_t r2 = row_of_rank(
                        n_nib ? colex_rank_nib<S>(rep2, rank, n_nib, n_c) : colex_rank<S>(rep2, rank), dict);
                    if (r2 < 0) continue;
                    if (layout == QMB_LAYOUT_REFERENCE && nullf[r2]) continue;
                    if (tv.half && r2 < r) continue;
                    const double cr = signed_coef<S>(o.coef.x, down, o.sz), ci = signed_coef<S>(o.coef.y, down, o.sz);
                    // f = c * conj(chi(j)) * chi(gm) * n_t / n_r; mult = the target row's stabiliser size
                    double2 q = s_chi[gm];
                    if (AVG) {
                        const double2 cj = s_chi[j];
                        q = make_double2(cj.x * q.x + cj.y * q.y, cj.x * q.y - cj.y * q.x);
                    }
                    double ratio = mult == m_src ? 1.0 : s_nrm[mult] / s_nrm[m_src];
                    if (tv.half && r2 > r) ratio *= 2.0;
                    const double fr = (cr * q.x - ci * q.y) * ratio, fi = (cr * q.y + ci * q.x) * ratio;
                    if (CPLX) {
                        const double xr = x[2 * r2], xi = x[2 * r2 + 1];
                        ar += fr * xr - fi * xi;
                        ai += fr * xi + fi * xr;
                    } else {
                        const double xt = x[r2];
                        ar += fr * xt;
                        ai += fi * xt;
                    }
                }
            }
        }
        // x_r conj((M x)_r)
        const double xr = CPLX ? x[2 * r] : x[r], xi = CPLX ? x[2 * r + 1] : 0.0;
        ar += dr * xr - di * xi;
        ai += dr * xi + di * xr;
        out_r += xr * ar + xi * ai;
        out_i += xi * ar - xr * ai;
    }
    const double scale = AVG ? 1.0 / (double)gv.G : 1.0;
    const double sr = block_sum(out_r * scale, red);
    const double si = block_sum(out_i * scale, red);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = sr;
        partials[2 * blockIdx.x + 1] = tv.half ? 0.0 : si;
    }
}

// The partial sums in a fixed order (one block).
__global__ __launch_bounds__(kThreads) void expect_finish(const double *__restrict__ partials, int blocks,
                                                          double *__restrict__ out) {
    __shared__ double red[kWaves];
    double sr = 0.0, si = 0.0;
    for (int i = threadIdx.x; i < blocks; i += blockDim.x) {
        sr += partials[2 * i];
        si += partials[2 * i + 1];
    }
    sr = block_sum(sr, red);
    si = block_sum(si, red);
    if (threadIdx.x == 0) {
        out[0] = sr;
        out[1] = si;
    }
}

// Distinct terms with their coefficients summed, in order of first occurrence. Two
// terms are the same when they act on the same states with the same image and
// sign; that is decided on their masks, in one form: an Sz on a site whose value
// the condition fixes goes into the coefficient, a diagonal term sets nothing.
class TermSum {
public:
    std::vector<TermC> terms;

    TermSum() : slot_(64, -1) {}
    void add(TermC c) {
        const uint64_t fixed = c.sz & c.req;
        if (__builtin_popcountll(fixed & ~c.req_val) & 1) c.coef = make_double2(-c.coef.x, -c.coef.y);
        c.sz &= ~fixed;
        if (is_diagonal(c)) c.set = c.set_val = 0;
        c.vclass = 0;
        int64_t at = find(c);
        if (slot_[at] >= 0) {
            terms[slot_[at]].coef.x += c.coef.x;
            terms[slot_[at]].coef.y += c.coef.y;
            return;
        }
        slot_[at] = (int)terms.size();
        terms.push_back(c);
        if (2 * terms.size() > slot_.size()) {
            slot_.assign(2 * slot_.size(), -1);
            for (size_t i = 0; i < terms.size(); ++i) slot_[find(terms[i])] = (int)i;
        }
    }

private:
    std::vector<int> slot_;
    int64_t find(const TermC &c) const {  // the term's slot, or the free one where it belongs
        uint64_t h = 0;
        for (const uint64_t v : {c.req, c.req_val, c.set, c.set_val, c.sz}) h = (h ^ v) * 0x9E3779B97F4A7C15ull;
        h ^= h >> 29;
        for (size_t i = h & (slot_.size() - 1);; i = (i + 1) & (slot_.size() - 1)) {
            if (slot_[i] < 0) return (int64_t)i;
            const TermC &d = terms[slot_[i]];
            if (d.req == c.req && d.req_val == c.req_val && d.set == c.set && d.set_val == c.set_val && d.sz == c.sz)
                return (int64_t)i;
        }
    }
};

// T^dagger on the masks: the condition and the values set change places (a term sets
// every site of its condition but those of projectors, which it sets to what they are).
static TermC term_adjoint(const TermC &c) {
    TermC d = c;
    d.req_val = (c.req_val & ~c.set) | (c.set_val & c.set);
    d.set_val = c.req_val & c.set;
    d.coef = make_double2(c.coef.x, -c.coef.y);
    return d;
}

// Whether distinct terms come with their adjoints' conjugate coefficients, exactly.
static bool hermitian(const std::vector<TermC> &terms) {
    TermSum sum;
    for (const TermC &c : terms) sum.add(c);
    const size_t n = sum.terms.size();
    for (const TermC &c : terms) {
        TermC d = term_adjoint(c);
        d.coef = make_double2(-d.coef.x, -d.coef.y);
        sum.add(d);
        if (sum.terms.size() != n) return false;
    }
    for (const TermC &c : sum.terms)
        if (c.coef.x != 0.0 || c.coef.y != 0.0) return false;
    return true;
}

// g T g^-1 on the masks: the sites move; a spin flip turns the values round, and
// the Sz factors then count the up spins: (-1)^(number of factors) over.
static TermC term_image(const TermC &c, const qmb_group &g, int e) {
    const uint32_t *perm = &g.perm[(size_t)e * g.n_sites];
    TermC d{};
    for (uint64_t m = c.req | c.set | c.sz; m; m &= m - 1) {
        const int s = __builtin_ctzll(m);
        const int p = (int)perm[s];
        d.req |= (c.req >> s & 1) << p;
        d.req_val |= (c.req_val >> s & 1) << p;
        d.set |= (c.set >> s & 1) << p;
        d.set_val |= (c.set_val >> s & 1) << p;
        d.sz |= (c.sz >> s & 1) << p;
    }
    d.coef = c.coef;
    if (g.flip[e]) {
        d.req_val ^= d.req;
        d.set_val ^= d.set;
        if (__builtin_popcountll(d.sz) & 1) d.coef = make_double2(-d.coef.x, -d.coef.y);
    }
    return d;
}

// True when the operator commutes with every element: the images g A g^-1 (sites
// moved by the element, S+ <-> S- and Sz -> -Sz under a spin flip) have the same
// terms with the same summed scalars. Operators on one site keep their order.
// A term's key: its operators after a stable sort by site, one byte each (type, then
// site; no operator is 0), eight a word. An element maps the operator's distinct keys
// one to one, so each image is looked up among them: 784 terms of a structure factor
// under 56 elements 0.5 ms, 3.9 when each image was sorted and merged as strings.
static bool commutes_with_group(const qmb_terms &t, const qmb_group &g) {
    const int n = t.n_sites, words = std::max(1, (t.max_ops + 7) / 8);
    std::vector<uint8_t> ops(8 * words), image(8 * words);
    std::vector<uint64_t> keys;  // [distinct][words]
    std::vector<std::complex<double>> coef;
    size_t slots = 64;
    while (slots < 2 * (size_t)t.n_terms + 2) slots *= 2;
    std::vector<int> slot(slots, -1);
    // the operators v[0, k) sorted by site; their key's slot
    auto find = [&](std::vector<uint8_t> &v, int k) {
        for (int i = 1; i < k; ++i)
            for (int j = i; j > 0 && (v[j - 1] & 63) > (v[j] & 63); --j) std::swap(v[j - 1], v[j]);
        std::fill(v.begin() + k, v.end(), 0);
        const uint64_t *w = reinterpret_cast<const uint64_t *>(v.data());
        uint64_t h = 0;
        for (int i = 0; i < words; ++i) {
            h = (h ^ w[i]) * 0x9E3779B97F4A7C15ull;
            h ^= h >> 29;
        }
        size_t i = h & (slots - 1);
        while (slot[i] >= 0 && std::memcmp(&keys[(size_t)slot[i] * words], w, (size_t)words * 8) != 0)
            i = (i + 1) & (slots - 1);
        return i;
    };
    auto code = [](int type) { return type == QMB_OP_SP ? 64 : type == QMB_OP_SM ? 128 : 192; };
    for (int h = 0; h < t.n_terms; ++h) {
        const int k = t.n_ops[h];
        for (int q = 0; q < k; ++q)
            ops[q] = (uint8_t)(code(t.op_type[(size_t)h * t.max_ops + q]) + t.site[(size_t)h * t.max_ops + q]);
        const std::complex<double> c(t.scalar[2 * h], t.scalar[2 * h + 1]);
        const size_t i = find(ops, k);
        if (slot[i] >= 0) {
            coef[slot[i]] += c;
            continue;
        }
        slot[i] = (int)coef.size();
        coef.push_back(c);
        const uint64_t *w = reinterpret_cast<const uint64_t *>(ops.data());
        keys.insert(keys.end(), w, w + words);
    }
    const int distinct = (int)coef.size();
    double scale = 0.0;
    for (const auto &c : coef) scale = std::max(scale, std::abs(c));
    const double tol = 1e-12 * std::max(scale, 1e-300);
    std::vector<uint8_t> hit(distinct);
    for (int e = 0; e < g.G; ++e) {
        std::fill(hit.begin(), hit.end(), 0);
        for (int d = 0; d < distinct; ++d) {
            const uint8_t *v = reinterpret_cast<const uint8_t *>(&keys[(size_t)d * words]);
            std::complex<double> c = coef[d];
            int k = 0;
            for (; k < 8 * words && v[k]; ++k) {
                int type = v[k] & 192;
                if (g.flip[e]) {
                    if (type == 192)
                        c = -c;
                    else
                        type ^= 192;
                }
                image[k] = (uint8_t)(type + g.perm[(size_t)e * n + (v[k] & 63)]);
            }
            const int at = slot[find(image, k)];
            if (at >= 0) hit[at] = 1;
            if (std::abs(at >= 0 ? c - coef[at] : c) > tol) return false;
        }
        for (int d = 0; d < distinct; ++d)
            if (!hit[d] && std::abs(coef[d]) > tol) return false;
    }
    return true;
}

// ---- the entry point that allocates nothing ----------------------------------
// Scratch of qmb_expectation_noalloc: one file-scope device array per GPU, held
// until the process ends. Layout: [0, 256) the result (re, im); 64 KiB for the
// per-block partial sums; then the compiled terms, the character row
// (G double2) and the orbit-norm table (G + 1 doubles), each 256-byte aligned.
// Host code never uses the array's name as an address: the device address comes
// from hipGetSymbolAddress, once per device.
constexpr size_t kScratchBytes = (size_t)1 << 20;
constexpr size_t kScratchPart = 256;
constexpr size_t kScratchTerms = kScratchPart + ((size_t)64 << 10);
static_assert((size_t)kExpMaxBlocks * 2 * sizeof(double) <= kScratchTerms - kScratchPart);
constexpr size_t kScratchTabBytes = 4096;  // chi (<= 128 x 16 B) + norms (<= 129 x 8 B), aligned
constexpr int kNoAllocMaxTerms = (int)((kScratchBytes - kScratchTerms - kScratchTabBytes) / sizeof(TermC));
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;

// Device address of `scratch` on `device` (the current device), looked up once per device.
static unsigned char *scratch_ptr(int device) {
    static std::mutex mu;
    static unsigned char *ptrs[kMaxDevices] = {};
    QMB_REQUIRE(device >= 0 && device < kMaxDevices, "qmb_expectation_noalloc: device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!ptrs[device]) {
        void *p = nullptr;
        QMB_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        QMB_REQUIRE(p != nullptr, "qmb_expectation_noalloc: no device address for the scratch array");
        ptrs[device] = static_cast<unsigned char *>(p);
    }
    return ptrs[device];
}

// The terms of one expectation value: the operator's distinct ones, and where the
// group average is taken, those of (1/G) sum_g g A g^-1. That operator commutes with
// the group, so a row takes the image of its representative alone and not of all G
// elements: equal terms of the average are looked up once (28 sites with the spin
// flip: S+S- of two sites, half the lookups and no images to form; 717K rows, one
// correlation 551 us, 147 by the average, 82 with half as below). Formed on the host
// at about 20 ns an image, against 5 ps an image and row on the GPU: for few images or
// at least 4096 rows, and as long as the terms fit the scratch of
// qmb_expectation_noalloc, whose results are the same.
//
// half: the value of a Hermitian operator that commutes with the group is
// sum_r M_rr |x_r|^2 + 2 Re sum_{t > r} x_r conj(M_rt x_t). A representative is the least
// state of its orbit, so a term that lowers it ends in an orbit of a lower
// representative, a lower row: entries M_rt with t >= r come from the terms that raise
// the state alone, and only those are looked up.
//
// Both need every element listed equally often: of an uneven list the orbit weights of
// M_rt and M_tr differ, and an image's weights are not those of its representative.
struct ExpectTable {
    std::vector<unsigned char> bytes;  // t[n_terms], z[n_sz]
    ExpectTerms view{};
    bool images = false;  // expect_rows<AVG>
    ExpectTable(const qmb_terms &t, const qmb_group &g, bool average, int64_t n_rows) {
        TermSum own;
        const TermC *tc = reinterpret_cast<const TermC *>(t.compiled.data());
        for (int h = 0; h < t.n_terms; ++h)
            if (!never_acts(tc[h])) own.add(tc[h]);
        std::vector<TermC> terms = std::move(own.terms);
        images = average;
        const size_t all = terms.size() * (size_t)g.G;
        if (average && !g.uneven && (all <= 4096 || n_rows >= 4096)) {
            TermSum sum;
            for (const TermC &c : terms) {
                for (int e = 0; e < g.G; ++e) sum.add(term_image(c, g, e));
                if (sum.terms.size() > (size_t)kNoAllocMaxTerms) break;
            }
            if (sum.terms.size() <= (size_t)kNoAllocMaxTerms) {
                images = false;
                terms = std::move(sum.terms);
                for (TermC &c : terms) c.coef = make_double2(c.coef.x / g.G, c.coef.y / g.G);
            }
        }
        view.half = !images && !g.uneven && hermitian(terms);
        if (view.half)
            terms.erase(std::remove_if(terms.begin(), terms.end(),
                                       [](const TermC &c) { return c.set_val < (c.req_val & c.set); }),
                        terms.end());
        const auto mid = std::stable_partition(terms.begin(), terms.end(),
                                               [](const TermC &c) { return !is_diagonal(c); });
        const auto end = std::stable_partition(mid, terms.end(), [](const TermC &c) { return c.req != 0; });
        view.n_off = (int)(mid - terms.begin());
        view.n_terms = (int)(end - terms.begin());
        view.n_sz = (int)(terms.end() - end);
        for (const TermC &c : terms) view.imag |= c.coef.y != 0.0;
        bytes.resize(view.n_terms * sizeof(TermC) + view.n_sz * sizeof(SzTerm));
        std::memcpy(bytes.data(), terms.data(), view.n_terms * sizeof(TermC));
        for (int h = 0; h < view.n_sz; ++h) {
            const SzTerm z{end[h].sz, end[h].coef};
            std::memcpy(bytes.data() + view.n_terms * sizeof(TermC) + h * sizeof(SzTerm), &z, sizeof(z));
        }
    }
};

// <Psi|A|Psi> into res[0..1] (device); d_terms, chi, nrm, part: on the device.
static void launch_expectation(qmb_ctx *ctx, const qmb_basis *b, ExpectTable &tab, const void *d_terms,
                               const double2 *chi, const double *nrm, bool cplx, const double *x, double *part,
                               double *res) {
    const bool narrow = b->n_sites <= 32;
    const int64_t n = b->n_rows, total = (n + kExpThreads - 1) / kExpThreads;
    const int64_t passes = (total + kExpMaxBlocks - 1) / kExpMaxBlocks;
    const int blocks = (int)((total + passes - 1) / passes);
    const GroupView gv = b->view();
    ExpectTerms tv = tab.view;
    tv.t = static_cast<const TermC *>(d_terms);
    tv.z = reinterpret_cast<const SzTerm *>(tv.t + tv.n_terms);
    const size_t rank_size = narrow ? 4 : 8;
    int n_nib = (b->n_sites + 3) / 4;
    const int n_c = b->n_up + 1;
    const size_t nib_bytes = (size_t)n_nib * n_c * 16 * rank_size;
    size_t lds = (size_t)b->n_sites * kBinJ * rank_size;
    if (nib_bytes <= kExpRankBytes)
        lds += nib_bytes;
    else
        n_nib = 0;
    lds += (size_t)std::min(tv.n_off, kExpLdsTerms) *
           (narrow ? sizeof(ExpectOff<uint32_t>) : sizeof(ExpectOff<uint64_t>));
    using K = decltype(&expect_rows<uint32_t, false, false, -1>);
    static const K any[2][2][2] = {  // [narrow][complex][images]
        {{expect_rows<uint64_t, false, false, -1>, expect_rows<uint64_t, false, true, -1>},
         {expect_rows<uint64_t, true, false, -1>, expect_rows<uint64_t, true, true, -1>}},
        {{expect_rows<uint32_t, false, false, -1>, expect_rows<uint32_t, false, true, -1>},
         {expect_rows<uint32_t, true, false, -1>, expect_rows<uint32_t, true, true, -1>}}};
    static const K form[2][2] = {  // [complex][torus product, ring], narrow
        {expect_rows<uint32_t, false, false, 1>, expect_rows<uint32_t, false, false, 2>},
        {expect_rows<uint32_t, true, false, 1>, expect_rows<uint32_t, true, false, 2>}};
    const K k = narrow && !tab.images && (gv.lut == 1 || gv.lut == 2) ? form[cplx][gv.lut - 1]
                                                                     : any[narrow][cplx][tab.images];
    hipLaunchKernelGGL(k, dim3(blocks), dim3(kExpThreads), lds, ctx->stream, gv, ctx->binom.as<uint64_t>(), n_nib, n_c,
                       b->layout, n, b->reps.as<uint64_t>(), b->stab.as<uint8_t>(), b->nullf.as<uint8_t>(),
                       b->dict.as<uint64_t>(), tv, chi, nrm, x, part);
    QMB_HIP(hipGetLastError());
    hipLaunchKernelGGL(expect_finish, dim3(1), dim3(kThreads), 0, ctx->stream, part, blocks, res);
    QMB_HIP(hipGetLastError());
}

}  // namespace qmb

using namespace qmb;

extern "C" {

qmb_status qmb_expectation_noalloc(qmb_ctx *ctx, const qmb_basis *b, const qmb_terms *a, int is_complex,
                                   const double *x_dev, int flags, double *out, int *averaged) {
    return guarded([&] {
        QMB_REQUIRE(ctx && b && a && x_dev && out, "qmb_expectation_noalloc: NULL argument");
        QMB_REQUIRE(b->ctx == ctx, "qmb_expectation_noalloc: basis belongs to another context");
        QMB_REQUIRE(a->n_sites == b->n_sites, "qmb_expectation_noalloc: term table and basis disagree on n_sites");
        QMB_REQUIRE(is_complex == 0 || is_complex == 1, "qmb_expectation_noalloc: is_complex must be 0 or 1");
        QMB_REQUIRE(flags == 0 || flags == QMB_EXPECT_GROUP_AVERAGE, "qmb_expectation_noalloc: unknown flags");
        QMB_REQUIRE(a->n_terms <= kNoAllocMaxTerms,
                    "qmb_expectation_noalloc: " + std::to_string(a->n_terms) + " terms exceed the scratch limit of " +
                        std::to_string(kNoAllocMaxTerms) + " (use qmb_expectation)");
        const qmb_group *g = b->group;
        QMB_REQUIRE((size_t)g->G * 16 + 256 + (size_t)(g->G + 1) * 8 <= kScratchTabBytes,
                    "qmb_expectation_noalloc: group too large for the scratch tables");
        const double *ch = &g->chars[(size_t)b->irrep * g->G * 2];
        if (!is_complex)
            for (int e = 0; e < g->G; ++e)
                QMB_REQUIRE(ch[2 * e + 1] == 0.0, "qmb_expectation_noalloc: a real vector needs a real character row");
        const bool avg = (flags & QMB_EXPECT_GROUP_AVERAGE) || !commutes_with_group(*a, *g);
        if (averaged) *averaged = avg ? 1 : 0;
        out[0] = 0.0;
        out[1] = 0.0;
        const int64_t n = b->n_rows;
        if (n == 0 || a->n_terms == 0) return;
        QMB_HIP(hipSetDevice(ctx->device));
        QMB_REQUIRE(ctx->binom.p != nullptr, "qmb_expectation_noalloc: context has no binomial table");
        require_device_range(ctx, x_dev, (size_t)n * (is_complex ? 16 : 8), "qmb_expectation_noalloc: x_dev");
        unsigned char *sp = scratch_ptr(ctx->device);
        // tables into the scratch
        ExpectTable tab(*a, *g, avg, n);
        auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
        const size_t o_chi = kScratchTerms + up256(tab.bytes.size());
        const size_t o_nrm = o_chi + up256((size_t)g->G * 16);
        QMB_HIP(hipMemcpyAsync(sp + kScratchTerms, tab.bytes.data(), tab.bytes.size(),
                               hipMemcpyHostToDevice, ctx->stream));
        QMB_HIP(hipMemcpyAsync(sp + o_chi, ch, (size_t)g->G * 16, hipMemcpyHostToDevice, ctx->stream));
        QMB_HIP(hipMemcpyAsync(sp + o_nrm, g->orbit_norms.data(), (size_t)(g->G + 1) * sizeof(double),
                               hipMemcpyHostToDevice, ctx->stream));
        double *res = reinterpret_cast<double *>(sp);
        launch_expectation(ctx, b, tab, sp + kScratchTerms,
                           reinterpret_cast<const double2 *>(sp + o_chi), reinterpret_cast<const double *>(sp + o_nrm),
                           is_complex != 0, x_dev, reinterpret_cast<double *>(sp + kScratchPart), res);
        QMB_HIP(hipMemcpyAsync(out, res, 2 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        QMB_HIP(hipStreamSynchronize(ctx->stream));
    });
}

qmb_status qmb_expectation(qmb_ctx *ctx, const qmb_basis *b, const qmb_terms *a, int is_complex, const double *x,
                           int x_on_device, int flags, double *out, int *averaged) {
    return guarded([&] {
        PoolScope pool_scope(ctx ? &ctx->pool : nullptr);
        QMB_REQUIRE(ctx && b && a && x && out, "qmb_expectation: NULL argument");
        QMB_REQUIRE(b->ctx == ctx, "qmb_expectation: basis belongs to another context");
        QMB_REQUIRE(a->n_sites == b->n_sites, "qmb_expectation: term table and basis disagree on n_sites");
        QMB_REQUIRE(is_complex == 0 || is_complex == 1, "qmb_expectation: is_complex must be 0 or 1");
        QMB_REQUIRE(flags == 0 || flags == QMB_EXPECT_GROUP_AVERAGE, "qmb_expectation: unknown flags");
        const qmb_group *g = b->group;
        const double *ch = &g->chars[(size_t)b->irrep * g->G * 2];
        if (!is_complex)
            for (int e = 0; e < g->G; ++e)
                QMB_REQUIRE(ch[2 * e + 1] == 0.0, "qmb_expectation: a real vector needs a real character row");
        const bool avg = (flags & QMB_EXPECT_GROUP_AVERAGE) || !commutes_with_group(*a, *g);
        if (averaged) *averaged = avg ? 1 : 0;
        out[0] = 0.0;
        out[1] = 0.0;
        const int64_t n = b->n_rows;
        if (n == 0 || a->n_terms == 0) return;
        QMB_HIP(hipSetDevice(ctx->device));
        const size_t xbytes = (size_t)n * (is_complex ? 16 : 8);
        DevBuf d_x;
        const double *xd = x;
        if (!x_on_device) {
            d_x.alloc(xbytes);
            QMB_HIP(hipMemcpyAsync(d_x.p, x, xbytes, hipMemcpyHostToDevice, ctx->stream));
            xd = d_x.as<double>();
        } else {
            require_device_range(ctx, x, xbytes, "qmb_expectation: x");
        }
        ExpectTable tab(*a, *g, avg, n);
        // result, partial sums, terms, characters and norms in one block; one copy
        auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
        const size_t o_part = 256, o_terms = o_part + (size_t)kExpMaxBlocks * 2 * sizeof(double);
        const size_t o_chi = o_terms + up256(tab.bytes.size()), o_nrm = o_chi + up256((size_t)g->G * 16);
        std::vector<unsigned char> h(o_nrm - o_terms + (size_t)(g->G + 1) * sizeof(double));
        std::memcpy(h.data(), tab.bytes.data(), tab.bytes.size());
        std::memcpy(h.data() + (o_chi - o_terms), ch, (size_t)g->G * 16);
        std::memcpy(h.data() + (o_nrm - o_terms), g->orbit_norms.data(), (size_t)(g->G + 1) * sizeof(double));
        DevBuf blob(o_terms + h.size());
        char *d = static_cast<char *>(blob.p);
        QMB_HIP(hipMemcpyAsync(d + o_terms, h.data(), h.size(), hipMemcpyHostToDevice, ctx->stream));
        launch_expectation(ctx, b, tab, d + o_terms,
                           reinterpret_cast<const double2 *>(d + o_chi), reinterpret_cast<const double *>(d + o_nrm),
                           is_complex != 0, xd, reinterpret_cast<double *>(d + o_part), reinterpret_cast<double *>(d));
        QMB_HIP(hipMemcpyAsync(out, d, 2 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        QMB_HIP(hipStreamSynchronize(ctx->stream));
    });
}

}  // extern "C"
