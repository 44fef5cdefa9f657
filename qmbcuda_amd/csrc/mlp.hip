// Learned Lanczos start vector (no reference counterpart).
//
// Network: input = 8 spins of a window (+-1) + Delta + J2/J1 (10 values);
// tanh(128) -> tanh(128) -> (log-amplitude a, phase phi). For an N-site ring
// state s: log psi(s) = sum_t a(w_t) + i phi(w_t), w_t = spins t..t+7 (mod N),
// translation invariant by construction. The k=0 coefficient of representative
// r is c_r = psi(r) sqrt(G/m_r).
//
// Because a window takes only 256 values, the network is evaluated once per
// (pattern, coupling) row; states then cost N table lookups. Training
// back-propagates per-pattern gradient histograms. The 128x128 layer - the
// bulk of the arithmetic - runs on gfx950 MFMA (v_mfma_f32_32x32x16_bf16:
// bf16 weights and activations, FP32 accumulation) in the forward pass, the
// activation backward pass (dH1 = dA2 W2) and the weight gradient
// (dW2 = dA2^T H1); the 10-wide input layer and the 2-wide head use FP32 VALU.
// Weight-gradient partial sums, the pattern histograms (fixed-point int64) and
// every reduction are deterministic.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <memory>

#include "internal.hpp"
#include "reduce.hpp"

namespace qmb {

constexpr int kIn = 10, kH = 128, kOut = 2, kWin = 8;
constexpr int oW1 = 0, ob1 = oW1 + kH * kIn, oW2 = ob1 + kH, ob2 = oW2 + kH * kH, oW3 = ob2 + kH,
              ob3 = oW3 + kOut * kH, kParams = ob3 + kOut;
constexpr double kFix = 68719476736.0;  // 2^36 fixed-point scale of the pattern histograms
constexpr double kMarshallPi = 3.14159265358979323846;
constexpr double kStartNoise = 0.1;  // weight of the unit seeded noise in the Lanczos start

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ inline uint16_t to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even (finite inputs)
    return (uint16_t)(u >> 16);
}
__device__ inline float from_bf16_bits(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ inline bf16x8 load8(const uint16_t *p) {
    bf16x8 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// C/D layout of the 32x32 MFMA tile held by lane l: element v sits at
// row 8*(v/4) + 4*(l/32) + (v%4), column l%32. A fragment: row l%32, k = 8*(l/32)..+7;
// B fragment: column l%32, k = 8*(l/32)..+7 (16 k per instruction).
__device__ inline int mfma_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }

// ---- forward: four wavefronts per 32 rows --------------------------------------
// Row r = c*256 + p: pattern p, coupling c (whole couplings). Writes
// out[r][2]; with store, also H1 (FP32 and bf16) and H2 (FP32) for the backward
// pass. The tile's work is a chain of short phases, so its four wavefronts share
// the long ones: layer 1 by hidden unit and row half, layer 2 one 32-column MFMA
// tile each (one wavefront per tile: 41 us for 192 couplings, 28 us for one; now
// 26 and 11 us).
constexpr int kTileLd = kH + 8;  // bf16 row stride of the LDS activation tile
constexpr int kFwdThreads = 256;

__global__ __launch_bounds__(kFwdThreads) void mlp_forward(const float *__restrict__ theta,
                                                           const uint16_t *__restrict__ w2bf,
                                                           const double *__restrict__ coup, float *__restrict__ out, float *__restrict__ H1,
                                                           uint16_t *__restrict__ H1q, float *__restrict__ H2,
                                                           int store) {
    __shared__ float x[32][kIn];
    __shared__ alignas(16) uint16_t a_tile[32 * kTileLd];
    __shared__ float h2[32][kH + 1];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int r0 = blockIdx.x * 32;
    if (t < 32) {
        const int p = (r0 + t) & 255;
        const int c = (r0 + t) >> 8;
        for (int i = 0; i < kWin; ++i) x[t][i] = ((p >> i) & 1) ? 1.f : -1.f;
        x[t][8] = (float)coup[2 * c];
        x[t][9] = (float)coup[2 * c + 1];
    }
    bf16x8 bw[kH / 16];
#pragma unroll
    for (int kb = 0; kb < kH / 16; ++kb)
        bw[kb] = load8(w2bf + (size_t)(wv * 32 + (lane & 31)) * kH + kb * 16 + 8 * (lane >> 5));
    const int k = t & (kH - 1), half = t >> 7;
    float w[kIn];
    for (int i = 0; i < kIn; ++i) w[i] = theta[oW1 + k * kIn + i];
    const float b1 = theta[ob1 + k];
    __syncthreads();
    // layer 1 (VALU): hidden unit k, 16 rows
    for (int row = half * 16; row < half * 16 + 16; ++row) {
        float s = b1;
        for (int i = 0; i < kIn; ++i) s += w[i] * x[row][i];
        const float h = tanhf(s);
        const uint16_t q = to_bf16_bits(h);
        a_tile[row * kTileLd + k] = q;
        if (store) {
            H1[(size_t)(r0 + row) * kH + k] = h;
            H1q[(size_t)(r0 + row) * kH + k] = q;
        }
    }
    __syncthreads();
    // layer 2 (MFMA): H2 = tanh(H1q W2^T + b2)
    {
        f32x16 acc = {};
#pragma unroll
        for (int kb = 0; kb < kH / 16; ++kb) {
            const bf16x8 a = load8(a_tile + (lane & 31) * kTileLd + kb * 16 + 8 * (lane >> 5));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bw[kb], acc, 0, 0, 0);
        }
        const int col = wv * 32 + (lane & 31);
        const float b2 = theta[ob2 + col];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float h = tanhf(acc[v] + b2);
            h2[mfma_row(v, lane)][col] = h;
            if (store) H2[(size_t)(r0 + mfma_row(v, lane)) * kH + col] = h;
        }
    }
    __syncthreads();
    // head (VALU), in index order: lane -> (row = lane % 32, output = lane / 32)
    if (wv == 0) {
        const int row = lane & 31, o = lane >> 5;
        float s = theta[ob3 + o];
#pragma unroll 8
        for (int j = 0; j < kH; ++j) s += theta[oW3 + o * kH + j] * h2[row][j];
        out[(size_t)(r0 + row) * 2 + o] = s;
    }
}

// ---- backward: one block per coupling (256 rows), every weight gradient ------
// Tiles of 32 rows: dA2 = (dout W3) (1 - H2^2) goes to LDS in bf16, by rows and
// transposed, with H1q transposed; dA1 = (dA2 W2) (1 - H1^2) on MFMA (wavefront w
// owns columns 32 w .. 32 w + 31, its W2 fragments stay in registers), and
// dW2 += dA2^T H1q on MFMA (wavefront w owns rows 32 w .. of dW2). dA2 and dA1
// are used up where they are formed (the sums of b2, W3, b1, W1 too), so only
// H1, H1q and H2 are read; the tiles are double buffered, one barrier each.
// 192 couplings: 28 us, 38 us with the reduction; as four kernels that passed dA2 and dA1 through memory
// (and split the rows of dW2 over 48 blocks only) 626 us.
// dout comes from the pattern histograms: pattern p of the coupling has
// hist[2 p], hist[2 p + 1] in units of 1 / kFix.
constexpr int kBackThreads = 256;
constexpr int kTr = 40;  // bf16 row stride of the transposed tiles (32 rows, 16-byte aligned)

__global__ __launch_bounds__(kBackThreads) void mlp_backward(const float *__restrict__ theta,
                                                             const uint16_t *__restrict__ w2t,
                                                             const double *__restrict__ coup,
                                                             const unsigned long long *__restrict__ hist, float scale,
                                                             const float *__restrict__ H1,
                                                             const uint16_t *__restrict__ H1q,
                                                             const float *__restrict__ H2,
                                                             float *__restrict__ part) {
    __shared__ float dout[256][2];
    __shared__ alignas(16) uint16_t a_tile[2][32 * kTileLd];  // dA2: [row][k]
    __shared__ alignas(16) uint16_t at[2][kH * kTr];          // dA2^T: [k][row]
    __shared__ alignas(16) uint16_t bt[2][kH * kTr];          // H1q^T: [k][row]
    __shared__ float red[kH][3];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int g = blockIdx.x;
    const size_t r0 = (size_t)g * 256;
    for (int i = t; i < 512; i += kBackThreads)
        dout[i >> 1][i & 1] = (float)((double)(long long)hist[r0 * 2 + i] / kFix * scale);
    bf16x8 bw[kH / 16];
#pragma unroll
    for (int kb = 0; kb < kH / 16; ++kb)
        bw[kb] = load8(w2t + (size_t)(wv * 32 + (lane & 31)) * kH + kb * 16 + 8 * (lane >> 5));
    // element-wise part: hidden unit k, rows 16 half .. of each tile
    const int k = t & (kH - 1), half = t >> 7;
    const float w3a = theta[oW3 + k], w3b = theta[oW3 + kH + k];
    float gb2 = 0.f, gw3a = 0.f, gw3b = 0.f;
    // dA1 part: column col of this lane
    const int col = wv * 32 + (lane & 31), hi = lane >> 5;
    float gw1[kWin] = {}, gb1 = 0.f;
    f32x16 acc2[4] = {};
    __syncthreads();
    for (int tl = 0; tl < 8; ++tl) {
        const int bu = tl & 1;
        uint16_t *ta = a_tile[bu], *tt = at[bu], *tb = bt[bu];
        {
            float h[16];
            uint16_t q[16];
            const size_t base = (r0 + tl * 32 + half * 16) * kH + k;
#pragma unroll
            for (int i = 0; i < 16; ++i) h[i] = H2[base + (size_t)i * kH];
#pragma unroll
            for (int i = 0; i < 16; ++i) q[i] = H1q[base + (size_t)i * kH];
            __builtin_memcpy(__builtin_assume_aligned(tb + k * kTr + half * 16, 16), q, 32);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int row = half * 16 + i;
                const float da = dout[tl * 32 + row][0], db = dout[tl * 32 + row][1];
                const float v = (da * w3a + db * w3b) * (1.f - h[i] * h[i]);
                gb2 += v;
                gw3a += da * h[i];
                gw3b += db * h[i];
                q[i] = to_bf16_bits(v);
                ta[row * kTileLd + k] = q[i];
            }
            __builtin_memcpy(__builtin_assume_aligned(tt + k * kTr + half * 16, 16), q, 32);
        }
        __syncthreads();
        {
            f32x16 acc = {};
#pragma unroll
            for (int kb = 0; kb < kH / 16; ++kb) {
                const bf16x8 x = load8(ta + (lane & 31) * kTileLd + kb * 16 + 8 * hi);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, bw[kb], acc, 0, 0, 0);
            }
            // row 8 (v / 4) + 4 hi + v % 4 of the tile: pattern bits 0, 1 = v % 4, bit 2 = hi,
            // bits 3, 4 = v / 4, bits 5 .. 7 = the tile
            float sum = 0.f, s0 = 0.f, s1 = 0.f, s3 = 0.f, s4 = 0.f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float h = H1[(r0 + tl * 32 + mfma_row(v, lane)) * kH + col];
                const float d = acc[v] * (1.f - h * h);
                sum += d;
                s0 += (v & 1) ? d : -d;
                s1 += (v & 2) ? d : -d;
                s3 += (v & 4) ? d : -d;
                s4 += (v & 8) ? d : -d;
            }
            gb1 += sum;
            gw1[0] += s0;
            gw1[1] += s1;
            gw1[2] += hi ? sum : -sum;
            gw1[3] += s3;
            gw1[4] += s4;
            gw1[5] += (tl & 1) ? sum : -sum;
            gw1[6] += (tl & 2) ? sum : -sum;
            gw1[7] += (tl & 4) ? sum : -sum;
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const bf16x8 x = load8(tt + (wv * 32 + (lane & 31)) * kTr + kb * 16 + 8 * hi);
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const bf16x8 y = load8(tb + (nt * 32 + (lane & 31)) * kTr + kb * 16 + 8 * hi);
                acc2[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, acc2[nt], 0, 0, 0);
            }
        }
    }
    float *dst = part + (size_t)g * kParams;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int v = 0; v < 16; ++v)
            dst[oW2 + (wv * 32 + mfma_row(v, lane)) * kH + nt * 32 + (lane & 31)] = acc2[nt][v];
    // lanes l and l + 32 hold the two row halves of one column
    gb1 += __shfl_xor(gb1, 32, 64);
#pragma unroll
    for (int i = 0; i < kWin; ++i) gw1[i] += __shfl_xor(gw1[i], 32, 64);
    if (hi == 0) {
        for (int i = 0; i < kWin; ++i) dst[oW1 + col * kIn + i] = gw1[i];
        dst[oW1 + col * kIn + 8] = gb1 * (float)coup[2 * g];
        dst[oW1 + col * kIn + 9] = gb1 * (float)coup[2 * g + 1];
        dst[ob1 + col] = gb1;
    }
    if (half) {
        red[k][0] = gb2;
        red[k][1] = gw3a;
        red[k][2] = gw3b;
    }
    __syncthreads();
    if (!half) {
        dst[ob2 + k] = gb2 + red[k][0];
        dst[oW3 + k] = gw3a + red[k][1];
        dst[oW3 + kH + k] = gw3b + red[k][2];
    }
    if (wv == 3 && lane < 2) {
        float s = 0.f;
        for (int r = 0; r < 256; ++r) s += dout[r][lane];
        dst[ob3 + lane] = s;
    }
}

// grad = sum over the couplings' partials: 64 parameters a block, four slices of
// the couplings each, added in slice order. The last block: the mean loss.
constexpr int kReduceParams = 64;

__device__ inline void mean_loss(const double *__restrict__ stats, int ns, double *__restrict__ loss) {
    // the samples' losses in sample order, 256 loaded at a time
    __shared__ double v[256];
    double mean = 0.0;
    for (int k0 = 0; k0 < ns; k0 += 256) {
        __syncthreads();
        for (int k = threadIdx.x; k < 256 && k0 + k < ns; k += blockDim.x) v[k] = stats[(size_t)(k0 + k) * 8 + 4];
        __syncthreads();
        if (threadIdx.x == 0)
            for (int k = 0; k < 256 && k0 + k < ns; ++k) mean += v[k];
    }
    if (threadIdx.x == 0) *loss = mean / ns;
}

__global__ __launch_bounds__(256) void mlp_reduce_grad(int n_groups, const float *__restrict__ part,
                                                       float *__restrict__ grad, const double *__restrict__ stats,
                                                       int ns, double *__restrict__ loss) {
    if (blockIdx.x == gridDim.x - 1) {
        mean_loss(stats, ns, loss);
        return;
    }
    __shared__ float red[3][kReduceParams];
    const int sl = threadIdx.x / kReduceParams, at = threadIdx.x % kReduceParams;
    const int i = blockIdx.x * kReduceParams + at;
    float s = 0.f;
    if (i < kParams) {
        const float *p = part + i;
        int g = sl;
        for (; g + 28 < n_groups; g += 32) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = p[(size_t)(g + 4 * u) * kParams];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
        for (; g < n_groups; g += 4) s += p[(size_t)g * kParams];
    }
    if (sl) red[sl - 1][at] = s;
    __syncthreads();
    if (!sl && i < kParams) grad[i] = s + red[0][at] + red[1][at] + red[2][at];
}

// Adam (Kingma & Ba 2015) on the FP32 master weights; refresh the bf16 W2 and its transpose.
__global__ __launch_bounds__(256) void mlp_adam(float *__restrict__ theta, const float *__restrict__ grad,
                                                float *__restrict__ m1, float *__restrict__ m2, float lr, float b1,
                                                float b2, float bc1, float bc2, uint16_t *__restrict__ w2bf,
                                                uint16_t *__restrict__ w2t) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kParams) return;
    const float g = grad[i];
    const float a = b1 * m1[i] + (1.f - b1) * g;
    const float v = b2 * m2[i] + (1.f - b2) * g * g;
    m1[i] = a;
    m2[i] = v;
    const float t = theta[i] - lr * (a / bc1) / (sqrtf(v / bc2) + 1e-8f);
    theta[i] = t;
    if (i >= oW2 && i < ob2) {
        const int n = (i - oW2) / kH, k = (i - oW2) % kH;
        const uint16_t q = to_bf16_bits(t);
        w2bf[n * kH + k] = q;
        w2t[k * kH + n] = q;
    }
}

__global__ __launch_bounds__(256) void mlp_refresh_w2(const float *__restrict__ theta, uint16_t *__restrict__ w2bf,
                                                      uint16_t *__restrict__ w2t) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kH * kH) return;
    const int n = i / kH, k = i % kH;
    const uint16_t q = to_bf16_bits(theta[oW2 + i]);
    w2bf[n * kH + k] = q;
    w2t[k * kH + n] = q;
}

// ---- per-state kernels (one sample = one ground state) ---------------------
// A window is 8 site indices; its pattern has bit k = spin at site k of the
// window. Rings use windows q..q+7 (mod N); 2-D lattices register their own.
constexpr int kMaxWin = 128;

__device__ inline int window_pattern(uint64_t s, const uint8_t *w) {
    int p = 0;
#pragma unroll
    for (int k = 0; k < kWin; ++k) p |= (int)((s >> w[k]) & 1ull) << k;
    return p;
}

__device__ inline void stage_windows(uint8_t *lds, const uint8_t *win, int n_win) {
    for (int i = threadIdx.x; i < n_win * kWin; i += blockDim.x) lds[i] = win[i];
}

// Ring windows (sites q .. q + 7 mod N for every q, N >= 11) are taken four at a
// time: windows q .. q + 3 together are 11 consecutive sites, so one read of a
// table of 2048 sums replaces four reads of the 256 patterns' values, and one
// addition into a histogram of 2048 bins four into the patterns' (the bins are
// folded into the patterns once per block). The N % 4 windows left are taken one
// at a time. The sums of four 32-bit values are held in 64 bits.
constexpr int kGroupWin = 4, kGroupPat = 1 << (kWin + kGroupWin - 1);

// sites q, q + 1, ... of an n-site ring from bit 0 up (at least 11 of them right)
__device__ inline uint64_t ring_from(uint64_t s, int q, int n) { return q ? (s >> q) | (s << (n - q)) : s; }

// t4[p] = sum of t over the four windows inside p
__device__ inline void group_table(const float2 *t, double2 *t4) {
    for (int p = threadIdx.x; p < kGroupPat; p += blockDim.x) {
        double2 v = make_double2(0.0, 0.0);
#pragma unroll
        for (int i = 0; i < kGroupWin; ++i) {
            const float2 w = t[(p >> i) & 255];
            v.x += (double)w.x;
            v.y += (double)w.y;
        }
        t4[p] = v;
    }
}

// log-amplitude and phase sums over the windows of R states per thread
template <int R>
__device__ inline void window_sums(const uint64_t (&st)[R], int ring, int n_win, const float2 *t, const double2 *t4,
                                   const uint8_t *wl, double (&a)[R], double (&b)[R]) {
#pragma unroll
    for (int i = 0; i < R; ++i) a[i] = b[i] = 0.0;
    int q = 0;
    if (ring) {
        for (; q + kGroupWin <= n_win; q += kGroupWin) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const double2 v = t4[ring_from(st[i], q, n_win) & (kGroupPat - 1)];
                a[i] += v.x;
                b[i] += v.y;
            }
        }
    }
    for (; q < n_win; ++q) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const float2 v = t[ring ? (int)(ring_from(st[i], q, n_win) & 255) : window_pattern(st[i], wl + q * kWin)];
            a[i] += (double)v.x;
            b[i] += (double)v.y;
        }
    }
}

// The largest alpha of some rows, the first of them that has it and its beta.
struct Largest {
    double a;
    long long r;
    double b;
    __device__ void take(double a2, long long r2, double b2) {
        if (a2 > a || (a2 == a && r2 < r)) {
            a = a2;
            r = r2;
            b = b2;
        }
    }
};

__device__ inline Largest no_row() { return Largest{-1e300, LLONG_MAX, 0.0}; }

// That of the block (256 threads), to every thread.
__device__ inline Largest block_largest(Largest v, Largest *lds) {
    for (int off = 32; off > 0; off >>= 1) {
        const double a = __shfl_down(v.a, off, 64), b = __shfl_down(v.b, off, 64);
        const long long r = __shfl_down(v.r, off, 64);
        v.take(a, r, b);
    }
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    for (int i = 0; i < kWaves; ++i) v.take(lds[i].a, lds[i].r, lds[i].b);
    // thread 0 has the block's; the others take it from there
    __syncthreads();
    if (threadIdx.x == 0) lds[0] = v;
    __syncthreads();
    return lds[0];
}

// alpha_r, beta_r from the pattern table of this coupling; the block's largest alpha
// into part[block] (part[n_blocks + block] = its row, -1 for none, part[2 n_blocks +
// block] = its beta).
// beta_r also carries the Marshall sign prior pi * (up spins on sublattice A):
// the network learns the phase relative to the bipartite sign rule, whose
// state (and not the uniform one, which is the fully polarised multiplet and
// orthogonal to a singlet) is the natural starting point of training.
__global__ __launch_bounds__(256) void mlp_state_logpsi(int64_t n, int n_win, const uint8_t *__restrict__ win, int ring,
                                                        uint64_t sub_a, const uint64_t *__restrict__ reps,
                                                        const float *__restrict__ tab, double *__restrict__ alpha,
                                                        double *__restrict__ beta, double *__restrict__ part) {
    __shared__ float2 t[256];
    __shared__ double2 t4[kGroupPat];
    __shared__ Largest lds[kWaves];
    __shared__ uint8_t wl[kMaxWin * kWin];
    constexpr int R = 4;
    for (int i = threadIdx.x; i < 256; i += blockDim.x) t[i] = reinterpret_cast<const float2 *>(tab)[i];
    stage_windows(wl, win, n_win);
    __syncthreads();
    if (ring) group_table(t, t4);
    __syncthreads();
    Largest best = no_row();
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += R * step) {
        uint64_t st[R];
        double a[R], b[R];
#pragma unroll
        for (int i = 0; i < R; ++i) st[i] = r + i * step < n ? reps[r + i * step] : 0;
        window_sums<R>(st, ring, n_win, t, t4, wl, a, b);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if (r + i * step >= n) continue;
            const double beta_r = b[i] + kMarshallPi * (double)__popcll(st[i] & sub_a);
            alpha[r + i * step] = a[i];
            beta[r + i * step] = beta_r;
            best.take(a[i], r + i * step, beta_r);
        }
    }
    best = block_largest(best, lds);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = best.a;
        part[gridDim.x + blockIdx.x] = best.r == LLONG_MAX ? -1.0 : (double)best.r;
        part[2 * gridDim.x + blockIdx.x] = best.b;
    }
}

// Real start vector x_r = |c_r| cos(beta_r - beta_ref) with beta_ref the phase
// of the first representative of largest amplitude, found by every block among the
// n_best blocks' of mlp_state_logpsi (best; three launches fewer than by kernels of
// their own: a start vector of 12 to 22 sites 98-105 us, 66-76 so). Block
// partials: part[block] = sum of x_r^2, part[gridDim.x + block] = sum of xi_r^2
// for the seeded noise xi_r = 2 u_r - 1 (u_r = element r of the SplitMix64
// stream of `seed`) that the Lanczos start mixes in.
__global__ __launch_bounds__(256) void mlp_state_start(int64_t n, int G, const uint8_t *__restrict__ stab,
                                                       const double *__restrict__ alpha,
                                                       const double *__restrict__ beta,
                                                       const double *__restrict__ best, int n_best, uint64_t seed,
                                                       double *__restrict__ x, double *__restrict__ part) {
    __shared__ double lds[kWaves];
    __shared__ Largest s_best[kWaves];
    Largest top = no_row();
    for (int i = threadIdx.x; i < n_best; i += blockDim.x)
        if (best[n_best + i] >= 0.0) top.take(best[i], (long long)best[n_best + i], best[2 * n_best + i]);
    top = block_largest(top, s_best);
    const double am = top.a, br = top.b;
    double acc = 0.0, accn = 0.0;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
        const double mag = exp(alpha[r] - am) * sqrt((double)G / (double)stab[r]);
        const double v = mag * cos(beta[r] - br);
        x[r] = v;
        acc += v * v;
        const double xi = 2.0 * splitmix_uniform(seed, (uint64_t)r) - 1.0;
        accn += xi * xi;
    }
    const double t = block_sum(acc, lds);
    const double tn = block_sum(accn, lds);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = t;
        part[gridDim.x + blockIdx.x] = tn;
    }
}

// x_r <- x_r / ||x|| + eta * xi_r / ||xi|| (norms squared in sums[0], sums[1]).
__global__ __launch_bounds__(256) void mlp_mix_noise(int64_t n, uint64_t seed, double eta,
                                                     const double *__restrict__ sums, double *__restrict__ x) {
    const double ix = 1.0 / sqrt(sums[0]), in = eta / sqrt(sums[1]);
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
        const double xi = 2.0 * splitmix_uniform(seed, (uint64_t)r) - 1.0;
        x[r] = x[r] * ix + xi * in;
    }
}

// out[0], out[1] = fixed-order sums of part[0..n) and part[n..2n).
__global__ __launch_bounds__(256) void mlp_finish_sum2(const double *__restrict__ part, int n,
                                                       double *__restrict__ out) {
    __shared__ double lds[kWaves];
    const double t0 = sum_partials(part, n, lds);
    const double t1 = sum_partials(part + n, n, lds);
    if (threadIdx.x == 0) {
        out[0] = t0;
        out[1] = t1;
    }
}

// ---- the per-sample kernels batched over every sample of a training step ----
// One launch per phase covers all samples: block b works on sample task[b]. A
// wavefront task takes 64 * kBatchRows rows: kBatchRun * kBatchRows consecutive
// ones from each of 64 / kBatchRun equal parts of the sample. Consecutive
// representatives share their high sites, so with 64 consecutive rows a window
// there has one pattern for all lanes and their histogram additions queue at one
// bin; rows of one lane that share a pattern are summed before they are added.
constexpr int kBatchThreads = 512, kBatchRows = 8, kBatchWaves = kBatchThreads / 64;
constexpr int kBatchRun = 4;  // 192 samples, histogram / amplitude kernel: run 1 175 / 182 us, 2 131 / 120, 4 137 / 110, 8 151 / 112

struct BSample {
    int64_t n, off;  // rows; offset of the sample's rows in the concatenated amplitudes
    const uint64_t *reps;
    const uint8_t *stab;
    const double *u;
    const uint8_t *win;
    uint64_t sub_a;
    int n_win, ring, G, blk0, nblk;  // blocks [blk0, blk0 + nblk) of every batched launch
};

// wavefront tasks of a sample of n rows, and row i of a lane in task w (n or more: none)
__host__ __device__ inline int64_t batch_tasks(int64_t n) {
    return (n + 64 * kBatchRows - 1) / (64 * kBatchRows);
}
__device__ inline int64_t batch_row(int64_t n, int64_t w, int i, int lane) {
    constexpr int span = kBatchRun * kBatchRows;
    return w < batch_tasks(n) ? (lane / kBatchRun * batch_tasks(n) + w) * span + i * kBatchRun + lane % kBatchRun : n;
}

// Amplitudes c_r = exp(alpha_r - m) sqrt(G / m_r) (cos, sin)(beta_r), m = the
// block's largest alpha, into c, and the block's m and sums of u c, |c|^2, u^2:
// part[q * total + block], q = 0 .. 4. The sums of different blocks are brought
// to one m when they are added, so the amplitudes need no second pass over the
// windows. Bound by LDS reads and the 64-bit exp and sincos (192 samples, 9.9
// million rows: 110 us; as two kernels, one window at a time, 380 us).
__global__ __launch_bounds__(kBatchThreads) void mlp_batch_overlap(const BSample *__restrict__ S,
                                                                   const int *__restrict__ task,
                                                                   const float *__restrict__ tabs,
                                                                   double2 *__restrict__ c, double *__restrict__ part,
                                                                   int total) {
    __shared__ float2 t[256];
    __shared__ double2 t4[kGroupPat];
    __shared__ double lds[4][kBatchWaves];
    __shared__ uint8_t wl[kMaxWin * kWin];
    const int si = task[blockIdx.x];
    const BSample s = S[si];
    for (int i = threadIdx.x; i < 256; i += blockDim.x)
        t[i] = reinterpret_cast<const float2 *>(tabs)[(size_t)si * 256 + i];
    if (!s.ring) stage_windows(wl, s.win, s.n_win);
    __syncthreads();
    if (s.ring) group_table(t, t4);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t task_w = (int64_t)(blockIdx.x - s.blk0) * kBatchWaves + wv;
    uint64_t st[kBatchRows];
    double a[kBatchRows], b[kBatchRows];
    bool act[kBatchRows];
#pragma unroll
    for (int i = 0; i < kBatchRows; ++i) {
        const int64_t r = batch_row(s.n, task_w, i, lane);
        act[i] = r < s.n;
        st[i] = act[i] ? s.reps[r] : 0;
    }
    __syncthreads();
    window_sums<kBatchRows>(st, s.ring, s.n_win, t, t4, wl, a, b);
    double mx = -1e300;
#pragma unroll
    for (int i = 0; i < kBatchRows; ++i)
        if (act[i]) mx = fmax(mx, a[i]);
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    if (lane == 0) lds[0][wv] = mx;
    __syncthreads();
    for (int w = 0; w < kBatchWaves; ++w) mx = fmax(mx, lds[0][w]);
    __syncthreads();
    double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < kBatchRows; ++i) {
        if (!act[i]) continue;
        const int64_t r = batch_row(s.n, task_w, i, lane);
        const double mag = exp(a[i] - mx) * sqrt((double)s.G / (double)s.stab[r]);
        double sn, cs;
        sincos(b[i] + kMarshallPi * (double)__popcll(st[i] & s.sub_a), &sn, &cs);
        const double cr = mag * cs, ci = mag * sn;
        const double ur = s.u[r];
        c[s.off + r] = make_double2(cr, ci);
        v[0] += ur * cr;
        v[1] += ur * ci;
        v[2] += mag * mag;
        v[3] += ur * ur;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v[q] = wave_sum(v[q]);
        if (lane == 0) lds[q][wv] = v[q];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double tot = 0.0;
        for (int w = 0; w < kBatchWaves; ++w) tot += lds[threadIdx.x][w];
        part[(size_t)threadIdx.x * total + blockIdx.x] = tot;
    }
    if (threadIdx.x == 0) part[(size_t)4 * total + blockIdx.x] = mx;
}

// One block per sample: stats[8 si + 0..3] = Re O, Im O, Nc, Nu relative to the
// sample's largest alpha, stats[8 si + 4] = loss, stats[8 si + 5] = that alpha;
// hist (when set): the sample's bins are cleared.
__global__ __launch_bounds__(256) void mlp_batch_finish_overlap(const BSample *__restrict__ S,
                                                                const double *__restrict__ part, int total,
                                                                double *__restrict__ stats,
                                                                unsigned long long *__restrict__ hist) {
    __shared__ double lds[kWaves];
    __shared__ double s_mx;
    const BSample s = S[blockIdx.x];
    if (hist)
        for (int i = threadIdx.x; i < 512; i += blockDim.x) hist[(size_t)blockIdx.x * 512 + i] = 0ull;
    const double *pm = part + (size_t)4 * total + s.blk0;
    double mx = -1e300;
    for (int i = threadIdx.x; i < s.nblk; i += blockDim.x) mx = fmax(mx, pm[i]);
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_down(mx, off, 64));
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = lds[0];
        for (int i = 1; i < kWaves; ++i) m = fmax(m, lds[i]);
        s_mx = m;
    }
    __syncthreads();
    mx = s_mx;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < s.nblk; i += blockDim.x) {
        const double f = exp(pm[i] - mx);
        const double *pi = part + s.blk0 + i;
        v[0] += f * pi[0];
        v[1] += f * pi[(size_t)total];
        v[2] += f * f * pi[(size_t)2 * total];
        v[3] += pi[(size_t)3 * total];
    }
    for (int q = 0; q < 4; ++q) v[q] = block_sum(v[q], lds);
    if (threadIdx.x == 0) {
        double *st = stats + (size_t)blockIdx.x * 8;
        for (int q = 0; q < 4; ++q) st[q] = v[q];
        const double o2 = v[0] * v[0] + v[1] * v[1];
        st[4] = 1.0 - o2 / (v[2] * v[3]);
        st[5] = mx;
    }
}

// Per-pattern gradient histograms (fixed point) of every sample: each block adds
// its LDS histogram into its sample's hist[512] (integer sums, any order). Bound
// by the LDS additions and the reads of c (192 samples, 9.9 million rows: 137 us;
// 859 us with an addition per window, consecutive rows in a wavefront and the
// amplitudes formed again).
__global__ __launch_bounds__(kBatchThreads) void mlp_batch_grad(const BSample *__restrict__ S,
                                                                const int *__restrict__ task,
                                                                const double2 *__restrict__ c,
                                                                const double *__restrict__ part, int total,
                                                                const double *__restrict__ stats,
                                                                unsigned long long *__restrict__ hist) {
    __shared__ unsigned long long ha[256], hb[256], ha4[kGroupPat], hb4[kGroupPat];
    __shared__ uint8_t wl[kMaxWin * kWin];
    const int si = task[blockIdx.x];
    const BSample s = S[si];
    for (int i = threadIdx.x; i < 256; i += blockDim.x) ha[i] = hb[i] = 0ull;
    if (s.ring)
        for (int i = threadIdx.x; i < kGroupPat; i += blockDim.x) ha4[i] = hb4[i] = 0ull;
    else
        stage_windows(wl, s.win, s.n_win);
    const double *sv = stats + (size_t)si * 8;
    const double f = exp(part[(size_t)4 * total + blockIdx.x] - sv[5]);
    const double ore = sv[0], oim = sv[1], nc = sv[2], nu = sv[3];
    const double o2 = ore * ore + oim * oim;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t task_w = (int64_t)(blockIdx.x - s.blk0) * kBatchWaves + wv;
    uint64_t st[kBatchRows];
    unsigned long long qa[kBatchRows], qb[kBatchRows];
    bool act[kBatchRows];
#pragma unroll
    for (int i = 0; i < kBatchRows; ++i) {
        const int64_t r = batch_row(s.n, task_w, i, lane);
        act[i] = r < s.n;
        st[i] = 0;
        qa[i] = qb[i] = 0;
        if (act[i]) {
            double2 cv = c[s.off + r];
            cv.x *= f;
            cv.y *= f;
            const double ur = s.u[r];
            const double wr = ur * (ore * cv.x + oim * cv.y);
            const double wi = ur * (ore * cv.y - oim * cv.x);
            const double ga = -(2.0 * wr * nc - o2 * 2.0 * (cv.x * cv.x + cv.y * cv.y)) / (nc * nc * nu);
            const double gb = -(-2.0 * wi) / (nc * nu);
            qa[i] = (unsigned long long)(long long)llrint(ga * kFix);
            qb[i] = (unsigned long long)(long long)llrint(gb * kFix);
            st[i] = s.reps[r];
        }
    }
    __syncthreads();
    // one window (group) of the lane's rows: sums over equal patterns, then adds
    auto add = [&](unsigned long long *da, unsigned long long *db, auto pattern) {
        int cur = pattern(0);
        unsigned long long va = qa[0], vb = qb[0];
#pragma unroll
        for (int i = 1; i < kBatchRows; ++i) {
            const int p = pattern(i);
            if (p != cur) {
                atomicAdd(&da[cur], va);
                atomicAdd(&db[cur], vb);
                cur = p;
                va = vb = 0;
            }
            va += qa[i];
            vb += qb[i];
        }
        atomicAdd(&da[cur], va);
        atomicAdd(&db[cur], vb);
    };
    int q = 0;
    if (s.ring)
        for (; q + kGroupWin <= s.n_win; q += kGroupWin)
            add(ha4, hb4, [&](int i) { return (int)(ring_from(st[i], q, s.n_win) & (kGroupPat - 1)); });
    for (; q < s.n_win; ++q)
        add(ha, hb, [&](int i) {
            return s.ring ? (int)(ring_from(st[i], q, s.n_win) & 255) : window_pattern(st[i], wl + q * kWin);
        });
    __syncthreads();
    if (s.ring) {
        for (int p = threadIdx.x; p < kGroupPat; p += blockDim.x) {
            const unsigned long long va = ha4[p], vb = hb4[p];
            if (!va && !vb) continue;
#pragma unroll
            for (int i = 0; i < kGroupWin; ++i) {
                atomicAdd(&ha[(p >> i) & 255], va);
                atomicAdd(&hb[(p >> i) & 255], vb);
            }
        }
        __syncthreads();
    }
    unsigned long long *hs = hist + (size_t)si * 512;
    for (int i = threadIdx.x; i < 256; i += blockDim.x) {
        if (ha[i]) atomicAdd(&hs[2 * i], ha[i]);
        if (hb[i]) atomicAdd(&hs[2 * i + 1], hb[i]);
    }
}

// Loss only: the mean of the samples' losses.
__global__ __launch_bounds__(256) void mlp_batch_loss(const double *__restrict__ stats, int ns,
                                                      double *__restrict__ loss) {
    mean_loss(stats, ns, loss);
}

}  // namespace qmb

using namespace qmb;

// Window geometry of one basis: n_win windows of 8 sites and the sublattice A
// mask of the Marshall prior.
struct MlpGeom {
    Ref<const qmb_basis> basis;
    int n_win = 0;
    int ring = 0;  // the windows q .. q + 7 (mod n_win) of an n_win-site ring, n_win >= kGroupWin + 7
    DevBuf win;    // uint8 [n_win * 8]
    uint64_t sub_a = 0;
};

// Whether the windows are a whole ring's in order (MlpGeom::ring).
static int is_ring(const uint8_t *sites, int n_win, int n_sites) {
    if (n_win != n_sites || n_win < kWin + kGroupWin - 1) return 0;
    for (int q = 0; q < n_win; ++q)
        for (int k = 0; k < kWin; ++k)
            if (sites[q * kWin + k] != (q + k) % n_win) return 0;
    return 1;
}

struct MlpSample {
    Ref<const qmb_basis> basis;
    int geom = 0;  // index into qmb_mlp::geoms
    DevBuf u;      // target ground state
    double delta, j2;
};

// Device tables and work arrays of the batched per-sample kernels, rebuilt when
// the sample list changes.
struct MlpBatch {
    bool valid = false;
    int ns = 0, total_blocks = 0;
    int64_t total_rows = 0;
    DevBuf samples, task, amp, part, stats, hist, loss;
};

struct qmb_mlp : Counted {
    Ref<qmb_ctx> ctx;
    DevBuf theta, m1, m2, grad, w2bf, w2t;
    int64_t step = 0;
    std::vector<MlpGeom> geoms;
    std::vector<MlpSample> samples;
    MlpBatch batch;
    // row buffers (sized for the current row count)
    int rows_cap = 0;
    DevBuf coup, out, H1, H1q, H2, part;
    void ensure_rows(int rows);
};

void qmb_mlp::ensure_rows(int rows) {
    if (rows <= rows_cap) return;
    const int cap = ((rows + 255) / 256) * 256;
    coup.alloc((size_t)(cap / 256) * 2 * sizeof(double));
    out.alloc((size_t)cap * 2 * sizeof(float));
    H1.alloc((size_t)cap * kH * sizeof(float));
    H1q.alloc((size_t)cap * kH * sizeof(uint16_t));
    H2.alloc((size_t)cap * kH * sizeof(float));
    part.alloc((size_t)(cap / 256) * kParams * sizeof(float));
    rows_cap = cap;
}

namespace {

// The network's bases: compact layout, every character 1 (k = 0, and
// flip-even when the group has the spin flip).
void check_mlp_basis(const qmb_basis *b) {
    QMB_REQUIRE(b->layout == QMB_LAYOUT_COMPACT, "mlp: the basis must use the compact layout");
    QMB_REQUIRE(b->all_rows, "mlp: the basis must be the fully symmetric sector (k = 0, flip-even)");
    QMB_REQUIRE(b->n_sites >= kWin && b->n_sites <= 64, "mlp: lattice size must be in [8, 64]");
}

// Index of the geometry of basis b: registered windows, or for a plain ring
// (translation group G = N) the N windows q..q+7 (mod N) with sublattice A =
// the even sites.
int geom_for(qmb_mlp *m, const qmb_basis *b) {
    for (size_t i = 0; i < m->geoms.size(); ++i)
        if (m->geoms[i].basis == b) return (int)i;
    check_mlp_basis(b);
    const qmb_group *g = b->group;
    QMB_REQUIRE(g->torus && g->block == g->n_sites && g->G == g->n_sites && b->n_sites <= kMaxWin,
                "mlp: no windows registered for this basis and it is not a plain ring (G = N)");
    const int N = b->n_sites;
    std::vector<uint8_t> w((size_t)N * kWin);
    for (int q = 0; q < N; ++q)
        for (int k = 0; k < kWin; ++k) w[(size_t)q * kWin + k] = (uint8_t)((q + k) % N);
    MlpGeom gm;
    gm.basis = b;
    gm.n_win = N;
    gm.ring = is_ring(w.data(), N, N);
    gm.win.alloc(w.size());
    QMB_HIP(hipMemcpy(gm.win.p, w.data(), w.size(), hipMemcpyHostToDevice));
    for (int q = 0; q < N; q += 2) gm.sub_a |= 1ULL << q;
    m->geoms.push_back(std::move(gm));
    return (int)m->geoms.size() - 1;
}

// Forward pass over the given couplings (rows = 256 per coupling).
void forward_rows(qmb_mlp *m, const std::vector<double> &coup, bool store) {
    qmb_ctx *ctx = m->ctx;
    const int rows = (int)(coup.size() / 2) * 256;
    m->ensure_rows(rows);
    upload(ctx, m->coup.p, coup.data(), coup.size() * sizeof(double));
    hipLaunchKernelGGL(mlp_forward, dim3(rows / 32), dim3(kFwdThreads), 0, ctx->stream, m->theta.as<float>(),
                       m->w2bf.as<uint16_t>(), m->coup.as<double>(), m->out.as<float>(), m->H1.as<float>(),
                       m->H1q.as<uint16_t>(), m->H2.as<float>(), store ? 1 : 0);
    QMB_HIP(hipGetLastError());
}

// alpha/beta of one state set for the coupling whose table starts at tab.
constexpr int64_t kStartWith = 16384;  // rows of a start vector read back with its norms

struct StateWork {
    DevBuf alpha, beta, part, stats;  // part: mlp_state_logpsi's three, mlp_state_start's two a block
    int64_t cap = 0;
    int nb = 0;
    void ensure(int64_t n) {
        if (n <= cap) return;
        alpha.alloc(n * sizeof(double));
        beta.alloc(n * sizeof(double));
        nb = (int)std::min<int64_t>(1024, (n + 255) / 256);
        part.alloc((size_t)nb * 5 * sizeof(double));
        stats.alloc(8 * sizeof(double));
        cap = n;
    }
};

void state_logpsi(qmb_ctx *ctx, const qmb_basis *b, const MlpGeom &gm, const float *tab, StateWork &w) {
    w.ensure(b->n_rows);
    hipLaunchKernelGGL(mlp_state_logpsi, dim3(w.nb), dim3(256), 0, ctx->stream, b->n_rows, gm.n_win,
                       gm.win.as<uint8_t>(), gm.ring, gm.sub_a, b->reps.as<uint64_t>(), tab, w.alpha.as<double>(),
                       w.beta.as<double>(), w.part.as<double>());
    QMB_HIP(hipGetLastError());
}

// Sample table and work arrays of the batched kernels.
void ensure_batch(qmb_mlp *m) {
    MlpBatch &B = m->batch;
    if (B.valid) return;
    const int ns = (int)m->samples.size();
    std::vector<BSample> hs(ns);
    std::vector<int> task;
    int64_t off = 0;
    for (int i = 0; i < ns; ++i) {
        const MlpSample &sm = m->samples[i];
        const MlpGeom &gm = m->geoms[sm.geom];
        const qmb_basis *b = sm.basis;
        BSample &d = hs[i];
        d.n = b->n_rows;
        d.off = off;
        d.reps = b->reps.as<uint64_t>();
        d.stab = b->stab.as<uint8_t>();
        d.u = sm.u.as<double>();
        d.win = gm.win.as<uint8_t>();
        d.sub_a = gm.sub_a;
        d.n_win = gm.n_win;
        d.ring = gm.ring;
        d.G = b->group->G;
        d.blk0 = (int)task.size();
        d.nblk = (int)((batch_tasks(b->n_rows) + kBatchWaves - 1) / kBatchWaves);
        for (int k = 0; k < d.nblk; ++k) task.push_back(i);
        off += b->n_rows;
    }
    B.ns = ns;
    B.total_blocks = (int)task.size();
    B.total_rows = off;
    B.samples.alloc((size_t)ns * sizeof(BSample));
    B.task.alloc(task.size() * sizeof(int));
    B.amp.alloc((size_t)off * sizeof(double2));
    B.part.alloc((size_t)B.total_blocks * 5 * sizeof(double));
    B.stats.alloc((size_t)ns * 8 * sizeof(double));
    B.hist.alloc((size_t)ns * 512 * sizeof(unsigned long long));
    B.loss.alloc(sizeof(double));
    QMB_HIP(hipMemcpy(B.samples.p, hs.data(), hs.size() * sizeof(BSample), hipMemcpyHostToDevice));
    QMB_HIP(hipMemcpy(B.task.p, task.data(), task.size() * sizeof(int), hipMemcpyHostToDevice));
    B.valid = true;
}

// Loss statistics (and the pattern histograms when want_grad) of all samples,
// one launch per phase.
void batch_loss(qmb_mlp *m, bool want_grad) {
    qmb_ctx *ctx = m->ctx;
    ensure_batch(m);
    MlpBatch &B = m->batch;
    const BSample *S = B.samples.as<BSample>();
    const int *task = B.task.as<int>();
    const unsigned nb = (unsigned)B.total_blocks, ns = (unsigned)B.ns;
    hipLaunchKernelGGL(mlp_batch_overlap, dim3(nb), dim3(kBatchThreads), 0, ctx->stream, S, task, m->out.as<float>(),
                       B.amp.as<double2>(), B.part.as<double>(), B.total_blocks);
    QMB_HIP(hipGetLastError());
    hipLaunchKernelGGL(mlp_batch_finish_overlap, dim3(ns), dim3(256), 0, ctx->stream, S, B.part.as<double>(),
                       B.total_blocks, B.stats.as<double>(),
                       want_grad ? B.hist.as<unsigned long long>() : nullptr);
    QMB_HIP(hipGetLastError());
    if (!want_grad) {
        hipLaunchKernelGGL(mlp_batch_loss, dim3(1), dim3(256), 0, ctx->stream, B.stats.as<double>(), B.ns,
                           B.loss.as<double>());
        QMB_HIP(hipGetLastError());
        return;
    }
    hipLaunchKernelGGL(mlp_batch_grad, dim3(nb), dim3(kBatchThreads), 0, ctx->stream, S, task, B.amp.as<double2>(),
                       B.part.as<double>(), B.total_blocks, B.stats.as<double>(), B.hist.as<unsigned long long>());
    QMB_HIP(hipGetLastError());
}

// Learned start vector of a k=0 ring basis into dx (device, n_rows values),
// entirely on the device: network rows for (delta, j2), log-amplitude and
// phase per representative, reference phase of the first largest amplitude,
// x_r = |c_r| cos(beta_r - beta_ref); w.stats[0] = ||x||^2 and w.stats[1] =
// ||xi||^2 of the seeded noise. Returns false when ||x||^2 is zero or not
// finite (the caller then starts from the seeded random vector); those two numbers
// travel to the host, and the vector into x when that is given.
bool build_start(qmb_mlp *m, const qmb_basis *b, double delta, double j2, uint64_t seed, double *dx,
                 StateWork &w, double *x = nullptr) {
    const int gi = geom_for(m, b);
    qmb_ctx *ctx = m->ctx;
    std::vector<double> coup = {delta, j2};
    forward_rows(m, coup, false);
    state_logpsi(ctx, b, m->geoms[gi], m->out.as<float>(), w);
    hipLaunchKernelGGL(mlp_state_start, dim3(w.nb), dim3(256), 0, ctx->stream, b->n_rows, b->group->G,
                       b->stab.as<uint8_t>(), w.alpha.as<double>(), w.beta.as<double>(), w.part.as<double>(), w.nb,
                       seed, dx, w.part.as<double>() + 3 * w.nb);
    QMB_HIP(hipGetLastError());
    hipLaunchKernelGGL(mlp_finish_sum2, dim3(1), dim3(256), 0, ctx->stream, w.part.as<double>() + 3 * w.nb, w.nb,
                       w.stats.as<double>());
    QMB_HIP(hipGetLastError());
    // the norms, and a short vector with them, come back in one wait
    const bool with = x && b->n_rows <= kStartWith;
    double *sums = ctx->host_stage<double>((size_t)(2 + (with ? b->n_rows : 0)) * sizeof(double));
    QMB_HIP(hipMemcpyAsync(sums, w.stats.p, 2 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (with)
        QMB_HIP(hipMemcpyAsync(sums + 2, dx, b->n_rows * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    QMB_HIP(hipStreamSynchronize(ctx->stream));
    if (with)
        std::copy(sums + 2, sums + 2 + b->n_rows, x);
    else if (x)
        download(ctx, x, dx, b->n_rows * sizeof(double));
    return std::isfinite(sums[0]) && sums[0] > 0.0 && sums[1] > 0.0;
}

// Mean loss over the samples and, optionally, the gradient (device grad buffer).
double loss_and_grad(qmb_mlp *m, bool want_grad) {
    qmb_ctx *ctx = m->ctx;
    const int ns = (int)m->samples.size();
    std::vector<double> coup(2 * ns);
    for (int i = 0; i < ns; ++i) {
        coup[2 * i] = m->samples[i].delta;
        coup[2 * i + 1] = m->samples[i].j2;
    }
    forward_rows(m, coup, want_grad);
    batch_loss(m, want_grad);
    if (want_grad) {
        hipLaunchKernelGGL(mlp_backward, dim3(ns), dim3(kBackThreads), 0, ctx->stream, m->theta.as<float>(),
                           m->w2t.as<uint16_t>(), m->coup.as<double>(), m->batch.hist.as<unsigned long long>(),
                           1.0f / ns, m->H1.as<float>(), m->H1q.as<uint16_t>(), m->H2.as<float>(),
                           m->part.as<float>());
        QMB_HIP(hipGetLastError());
        hipLaunchKernelGGL(mlp_reduce_grad, dim3((kParams + kReduceParams - 1) / kReduceParams + 1), dim3(256), 0,
                           ctx->stream, ns, m->part.as<float>(), m->grad.as<float>(), m->batch.stats.as<double>(), ns,
                           m->batch.loss.as<double>());
        QMB_HIP(hipGetLastError());
    }
    double *hl = ctx->host_stage<double>(sizeof(double));
    QMB_HIP(hipMemcpyAsync(hl, m->batch.loss.p, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    QMB_HIP(hipStreamSynchronize(ctx->stream));
    return *hl;
}

std::vector<float> init_params(uint64_t seed) {
    std::vector<float> th(kParams);
    const int fan_for[] = {kIn, kIn, kH, kH, kH, kH};
    const int ends[] = {ob1, oW2, ob2, oW3, ob3, kParams};
    int seg = 0;
    for (int i = 0; i < kParams; ++i) {
        while (i >= ends[seg]) ++seg;
        uint64_t z = seed + ((uint64_t)i + 1ULL) * 0x9E3779B97F4A7C15ULL;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
        z ^= z >> 31;
        const double u = (double)((z >> 11) + 1ULL) * (1.0 / 9007199254740992.0);
        th[i] = (float)((2.0 * u - 1.0) / std::sqrt((double)fan_for[seg]));
    }
    return th;
}

}  // namespace

extern "C" {

int qmb_mlp_num_params(void) { return kParams; }

qmb_status qmb_mlp_create(qmb_ctx *ctx, uint64_t seed, qmb_mlp **out) {
    return guarded([&] {
        PoolScope pool_scope(ctx ? &ctx->pool : nullptr);
        QMB_REQUIRE(ctx && out, "qmb_mlp_create: NULL argument");
        *out = nullptr;
        QMB_HIP(hipSetDevice(ctx->device));
        auto m = std::make_unique<qmb_mlp>();
        m->ctx = ctx;
        m->theta.alloc(kParams * sizeof(float));
        m->m1.alloc(kParams * sizeof(float));
        m->m2.alloc(kParams * sizeof(float));
        m->grad.alloc(kParams * sizeof(float));
        m->w2bf.alloc(kH * kH * sizeof(uint16_t));
        m->w2t.alloc(kH * kH * sizeof(uint16_t));
        const std::vector<float> th = init_params(seed);
        QMB_HIP(hipMemcpy(m->theta.p, th.data(), kParams * sizeof(float), hipMemcpyHostToDevice));
        QMB_HIP(hipMemset(m->m1.p, 0, kParams * sizeof(float)));
        QMB_HIP(hipMemset(m->m2.p, 0, kParams * sizeof(float)));
        hipLaunchKernelGGL(mlp_refresh_w2, dim3(kH * kH / 256), dim3(256), 0, ctx->stream, m->theta.as<float>(),
                           m->w2bf.as<uint16_t>(), m->w2t.as<uint16_t>());
        QMB_HIP(hipGetLastError());
        QMB_HIP(hipStreamSynchronize(ctx->stream));
        *out = m.release();
    });
}

qmb_status qmb_mlp_destroy(qmb_mlp *m) {
    if (m && m->ctx) (void)hipStreamSynchronize(m->ctx->stream);
    release(m);
    return QMB_OK;
}

qmb_status qmb_mlp_get_params(const qmb_mlp *m, float *theta) {
    return guarded([&] {
        QMB_REQUIRE(m && theta, "qmb_mlp_get_params: NULL argument");
        QMB_HIP(hipStreamSynchronize(m->ctx->stream));
        QMB_HIP(hipMemcpy(theta, m->theta.p, kParams * sizeof(float), hipMemcpyDeviceToHost));
    });
}

qmb_status qmb_mlp_set_params(qmb_mlp *m, const float *theta) {
    return guarded([&] {
        QMB_REQUIRE(m && theta, "qmb_mlp_set_params: NULL argument");
        QMB_HIP(hipMemcpy(m->theta.p, theta, kParams * sizeof(float), hipMemcpyHostToDevice));
        hipLaunchKernelGGL(mlp_refresh_w2, dim3(kH * kH / 256), dim3(256), 0, m->ctx->stream, m->theta.as<float>(),
                           m->w2bf.as<uint16_t>(), m->w2t.as<uint16_t>());
        QMB_HIP(hipGetLastError());
        QMB_HIP(hipStreamSynchronize(m->ctx->stream));
    });
}

qmb_status qmb_mlp_forward(qmb_mlp *m, int n, const double *delta, const double *j2, float *out) {
    return guarded([&] {
        PoolScope pool_scope(m ? &m->ctx->pool : nullptr);
        QMB_REQUIRE(m && delta && j2 && out && n >= 1, "qmb_mlp_forward: bad argument");
        std::vector<double> coup(2 * (size_t)n);
        for (int i = 0; i < n; ++i) {
            coup[2 * i] = delta[i];
            coup[2 * i + 1] = j2[i];
        }
        forward_rows(m, coup, false);
        QMB_HIP(hipMemcpyAsync(out, m->out.p, (size_t)n * 512 * sizeof(float), hipMemcpyDeviceToHost, m->ctx->stream));
        QMB_HIP(hipStreamSynchronize(m->ctx->stream));
    });
}

qmb_status qmb_mlp_add_sample(qmb_mlp *m, const qmb_basis *b, const double *ground_state, double delta, double j2) {
    return guarded([&] {
        PoolScope pool_scope(m ? &m->ctx->pool : nullptr);
        QMB_REQUIRE(m && b && ground_state, "qmb_mlp_add_sample: NULL argument");
        QMB_REQUIRE(b->ctx == m->ctx, "qmb_mlp_add_sample: basis from another context");
        MlpSample s;
        s.geom = geom_for(m, b);
        s.basis = b;
        s.delta = delta;
        s.j2 = j2;
        s.u.alloc((size_t)b->n_rows * sizeof(double));
        QMB_HIP(hipMemcpy(s.u.p, ground_state, (size_t)b->n_rows * sizeof(double), hipMemcpyHostToDevice));
        m->samples.push_back(std::move(s));
        m->batch.valid = false;
    });
}

qmb_status qmb_mlp_set_windows(qmb_mlp *m, const qmb_basis *b, int n_win, const uint8_t *sites,
                               uint64_t sublattice_a) {
    return guarded([&] {
        QMB_REQUIRE(m && b && sites, "qmb_mlp_set_windows: NULL argument");
        QMB_REQUIRE(b->ctx == m->ctx, "qmb_mlp_set_windows: basis from another context");
        check_mlp_basis(b);
        QMB_REQUIRE(n_win >= 1 && n_win <= kMaxWin, "qmb_mlp_set_windows: n_win must be in [1, 128]");
        for (int i = 0; i < n_win * kWin; ++i)
            QMB_REQUIRE(sites[i] < b->n_sites, "qmb_mlp_set_windows: site index out of range");
        const uint64_t full = b->n_sites == 64 ? ~0ULL : ((1ULL << b->n_sites) - 1ULL);
        QMB_REQUIRE((sublattice_a & ~full) == 0, "qmb_mlp_set_windows: sublattice mask beyond the lattice");
        for (const auto &s : m->samples)
            QMB_REQUIRE(s.basis != b, "qmb_mlp_set_windows: the basis already has samples");
        MlpGeom gm;
        gm.basis = b;
        gm.n_win = n_win;
        gm.ring = is_ring(sites, n_win, b->n_sites);
        gm.win.alloc((size_t)n_win * kWin);
        QMB_HIP(hipMemcpy(gm.win.p, sites, (size_t)n_win * kWin, hipMemcpyHostToDevice));
        gm.sub_a = sublattice_a;
        for (auto &g : m->geoms)
            if (g.basis == b) {
                g = std::move(gm);
                return;
            }
        m->geoms.push_back(std::move(gm));
    });
}

qmb_status qmb_mlp_clear_samples(qmb_mlp *m) {
    return guarded([&] {
        QMB_REQUIRE(m, "qmb_mlp_clear_samples: NULL argument");
        QMB_HIP(hipStreamSynchronize(m->ctx->stream));
        m->samples.clear();
        m->batch = MlpBatch{};
    });
}

qmb_status qmb_mlp_loss_grad(qmb_mlp *m, double *loss, float *grad) {
    return guarded([&] {
        PoolScope pool_scope(m ? &m->ctx->pool : nullptr);
        QMB_REQUIRE(m && loss, "qmb_mlp_loss_grad: NULL argument");
        QMB_REQUIRE(!m->samples.empty(), "qmb_mlp_loss_grad: no samples");
        *loss = loss_and_grad(m, grad != nullptr);
        if (grad) QMB_HIP(hipMemcpy(grad, m->grad.p, kParams * sizeof(float), hipMemcpyDeviceToHost));
    });
}

qmb_status qmb_mlp_train(qmb_mlp *m, int steps, double lr, double *loss_history) {
    return guarded([&] {
        PoolScope pool_scope(m ? &m->ctx->pool : nullptr);
        QMB_REQUIRE(m && steps >= 1 && lr > 0, "qmb_mlp_train: bad argument");
        QMB_REQUIRE(!m->samples.empty(), "qmb_mlp_train: no samples");
        const float b1 = 0.9f, b2 = 0.999f;
        for (int s = 0; s < steps; ++s) {
            const double L = loss_and_grad(m, true);
            if (loss_history) loss_history[s] = L;
            ++m->step;
            const float bc1 = 1.f - std::pow(b1, (float)m->step), bc2 = 1.f - std::pow(b2, (float)m->step);
            hipLaunchKernelGGL(mlp_adam, dim3((kParams + 255) / 256), dim3(256), 0, m->ctx->stream,
                               m->theta.as<float>(), m->grad.as<float>(), m->m1.as<float>(), m->m2.as<float>(),
                               (float)lr, b1, b2, bc1, bc2, m->w2bf.as<uint16_t>(), m->w2t.as<uint16_t>());
            QMB_HIP(hipGetLastError());
        }
        QMB_HIP(hipStreamSynchronize(m->ctx->stream));
    });
}

qmb_status qmb_mlp_start_vector(qmb_mlp *m, const qmb_basis *b, double delta, double j2, double *x, int *fallback) {
    return guarded([&] {
        PoolScope pool_scope(m ? &m->ctx->pool : nullptr);
        QMB_REQUIRE(m && b && x, "qmb_mlp_start_vector: NULL argument");
        DevBuf dx((size_t)b->n_rows * sizeof(double));
        StateWork w;
        const bool ok = build_start(m, b, delta, j2, 0, dx.as<double>(), w, x);
        if (fallback) *fallback = ok ? 0 : 1;
    });
}

qmb_status qmb_lanczos_learned(qmb_mlp *m, const qmb_basis *b, const qmb_ell *e, double delta, double j2,
                               const qmb_lanczos_opts *opts, double *evals, double *eigvec, qmb_lanczos_report *report,
                               int *fallback) {
    qmb_status st = guarded([&] {
        PoolScope pool_scope(m ? &m->ctx->pool : nullptr);
        QMB_REQUIRE(m && b && e && evals, "qmb_lanczos_learned: NULL argument");
        QMB_REQUIRE(e->basis == b, "qmb_lanczos_learned: the ELL was not built on this basis");
        QMB_REQUIRE(e->ctx == m->ctx, "qmb_lanczos_learned: network and ELL live on different contexts");
        QMB_REQUIRE(e->value_type == QMB_REAL, "qmb_lanczos_learned: the learned start vector is real; "
                                               "build the ELL with QMB_REAL");
    });
    if (st != QMB_OK) return st;
    qmb_lanczos_opts o;
    if (opts)
        o = *opts;
    else
        qmb_lanczos_default_opts(&o);
    DevBuf dx;
    StateWork w;
    bool ok = false;
    st = guarded([&] {
        dx.alloc((size_t)b->n_rows * sizeof(double));
        ok = build_start(m, b, delta, j2, o.seed, dx.as<double>(), w);
        if (ok) {
            // unit learned vector + kStartNoise x unit seeded noise: the noise keeps
            // every eigenvector in the Krylov space even where the network's
            // vector misses the ground state
            hipLaunchKernelGGL(mlp_mix_noise, dim3(w.nb), dim3(256), 0, m->ctx->stream, b->n_rows, o.seed,
                               kStartNoise, w.stats.as<double>(), dx.as<double>());
            QMB_HIP(hipGetLastError());
        }
    });
    if (st != QMB_OK) return st;
    if (fallback) *fallback = ok ? 0 : 1;
    if (ok) {
        o.start = QMB_START_DEVICE;
        o.start_vec = dx.as<double>();
    } else {
        o.start = QMB_START_RANDOM;
        o.start_vec = nullptr;
    }
    st = qmb_lanczos(m->ctx, e, &o, evals, nullptr, eigvec, report);
    if (ok && st == QMB_ERR_NOT_CONVERGED) {
        // the Ritz residual of the learned run missed the tolerance within max_iter:
        // the seeded random start is the fallback and its run is the result
        if (fallback) *fallback = 2;
        o.start = QMB_START_RANDOM;
        o.start_vec = nullptr;
        st = qmb_lanczos(m->ctx, e, &o, evals, nullptr, eigvec, report);
    }
    return st;
}

}  // extern "C"
