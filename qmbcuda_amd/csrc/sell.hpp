// SELL-64 row products shared by the single and the batched SpMV kernels.
//
// One lane owns one row of a 64-row chunk; the chunk is stored slot-major, so
// slot k of the 64 rows is one coalesced 256 B (col) + 512 B / 1 KB (val)
// read. Slots are taken in groups of U: the next group's words are loaded, then
// this group's x values gathered, then its products added in slot order, so the
// sum has the same rounding sequence as a plain slot-by-slot loop (and as the
// FP64 oracle's row sum). The last group is a group like the others, with the
// slots past the row masked: taken one by one, its up to U - 1 slots were as many
// dependent word-gather chains (4x8 lattice, 9.4 million rows: 1366 us a product,
// 1468 with the one-by-one tail).
//
// L: the slots to go through, at least the chunk's longest row; it is the same for
// every wavefront of a block when `step` (called after each group) is a barrier.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qmb {

// Matrix-stream load: nontemporal (streamed past the caches) when NT, else
// plain (the lines may stay in L2 and the MALL for the next SpMV).
template <bool NT, class T>
__device__ inline T stream_load(const T *p) {
    if constexpr (NT)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

struct NoStep {
    __device__ inline void operator()() const {}
};

// sum over slots k < len of val[p0 + 64k] * x[col[p0 + 64k]]
template <bool NT, int U = 4, class Step = NoStep>
__device__ inline double sell_row_real(const int32_t *__restrict__ col, const double *__restrict__ val,
                                       const double *__restrict__ x, int64_t p0, int L, int len, Step step = Step()) {
    double acc = 0.0;
    int32_t jn[U];
    double vn[U];
    auto load = [&](int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k0 + u < len) {
                const int64_t p = p0 + (int64_t)(k0 + u) * 64;
                jn[u] = stream_load<NT>(col + p);
                vn[u] = stream_load<NT>(val + p);
            }
        }
    };
    load(0);
    for (int k = 0; k < L; k += U) {
        int32_t j[U];
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            j[u] = jn[u];
            v[u] = vn[u];
        }
        load(k + U);
        double g[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < len) g[u] = x[j[u]];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < len) acc += v[u] * g[u];
        step();
    }
    return acc;
}

// Packed real rows: slot 0 is the diagonal d (column = the row r itself); slot
// k >= 1 holds w = col | (index << cb) with the value vt[index]. Same products in
// the same order as sell_row_real on the unpacked matrix. Groups of 8 when the
// matrix is streamed from HBM (more loads in flight), 4 when it is cached.
template <bool NT, int U = (NT ? 8 : 4), class Step = NoStep>
__device__ inline double sell_row_packed(const uint32_t *__restrict__ w, const double *vt,
                                         const double *__restrict__ x, int64_t p0, int L, int len, int cb,
                                         double d, double xr, Step step = Step()) {
    const uint32_t mask = (1u << cb) - 1u;
    double acc = 0.0;
    if (len > 0) acc += d * xr;
    uint32_t jn[U];
    auto load = [&](int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k0 + u < len) jn[u] = stream_load<NT>(w + p0 + (int64_t)(k0 + u) * 64);
    };
    load(1);
    for (int k = 1; k < L; k += U) {
        uint32_t j[U];
#pragma unroll
        for (int u = 0; u < U; ++u) j[u] = jn[u];
        load(k + U);
        double g[U], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u < len) {
                g[u] = x[j[u] & mask];
                v[u] = vt[j[u] >> cb];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < len) acc += v[u] * g[u];
        step();
    }
    return acc;
}

// complex rows: val and x are interleaved (re, im) pairs
template <bool NT, int U = 4, class Step = NoStep>
__device__ inline double2 sell_row_cplx(const int32_t *__restrict__ col, const double *__restrict__ val,
                                        const double *__restrict__ x, int64_t p0, int L, int len,
                                        Step step = Step()) {
    const double2 *val2 = reinterpret_cast<const double2 *>(val);
    const double2 *x2 = reinterpret_cast<const double2 *>(x);
    double ar = 0.0, ai = 0.0;
    for (int k = 0; k < L; k += U) {
        int32_t j[U];
        double2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u < len) {
                const int64_t p = p0 + (int64_t)(k + u) * 64;
                j[u] = stream_load<NT>(col + p);
                v[u] = val2[p];
            }
        }
        double2 g[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < len) g[u] = x2[j[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u < len) {
                ar += v[u].x * g[u].x - v[u].y * g[u].y;
                ai += v[u].x * g[u].y + v[u].y * g[u].x;
            }
        }
        step();
    }
    return make_double2(ar, ai);
}

// Packed complex rows: slot 0 is the diagonal d; slot k >= 1 holds
// w = col | (re index << cb) | (im index << (cb + rb)) with the value
// (vre[re index], vim[im index]). Same products in the same order as
// sell_row_cplx on the unpacked matrix.
template <bool NT, int U = 4, class Step = NoStep>
__device__ inline double2 sell_row_cplx_packed(const uint32_t *__restrict__ w, const double *vre, const double *vim,
                                               const double *__restrict__ x, int64_t p0, int L, int len, int cb,
                                               int rb, double2 d, double2 xr, Step step = Step()) {
    const double2 *x2 = reinterpret_cast<const double2 *>(x);
    const uint32_t mask = (1u << cb) - 1u, rmask = (1u << rb) - 1u;
    const int sh2 = cb + rb;
    double ar = 0.0, ai = 0.0;
    if (len > 0) {
        ar += d.x * xr.x - d.y * xr.y;
        ai += d.x * xr.y + d.y * xr.x;
    }
    uint32_t jn[U];
    auto load = [&](int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k0 + u < len) jn[u] = stream_load<NT>(w + p0 + (int64_t)(k0 + u) * 64);
    };
    load(1);
    for (int k = 1; k < L; k += U) {
        uint32_t j[U];
#pragma unroll
        for (int u = 0; u < U; ++u) j[u] = jn[u];
        load(k + U);
        double2 g[U], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u < len) {
                g[u] = x2[j[u] & mask];
                v[u].x = vre[(j[u] >> cb) & rmask];
                v[u].y = vim[(uint32_t)((uint64_t)j[u] >> sh2)];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u < len) {
                ar += v[u].x * g[u].x - v[u].y * g[u].y;
                ai += v[u].x * g[u].y + v[u].y * g[u].x;
            }
        }
        step();
    }
    return make_double2(ar, ai);
}

}  // namespace qmb
