// sig_join by an appended segment and its adjoint for long rows: the words of a level are taken by their prefix u, so that
// the top level, nearly the whole row, is read and written once in memory order.
//
//   out_t[u x] = A_t[u x] + V_t(u) z[x]                                        |u| = t - 1
//   V_t(u) = V_{t,t-1}(u),   V_{t,0} = 1,   V_{t,l}(p_1 .. p_l) = V_{t,l-1}(p_1 .. p_{l-1}) z[p_l] / (t - l + 1) + A_l[p_1 .. p_l]
// (the Horner form of siglib/cpsig/cp_sig_join.h:107-160).  In memory the children u x of consecutive words u are consecutive, over the
// borders of the levels too: with y = 0 for the empty word and 1 + the position of u in the row otherwise, they
// are the d entries from y * d on.
//
// Adjoint: with a_{t,l}[u] the gradient with respect to V_{t,l}(u), and v_0 = the gradient of out_{l+1}, v_j = a_{l+1+j,l+1}, all over
// the words u x of length l + 1:
//   dA_{l+1}[u x] = sum_j v_j[u x],     a_{l+1+j,l}[u] = sum_x v_j[u x] z[x] / (j + 1),
//   dz[x] += sum_j sum_u v_j[u x] V_{l+1+j,l}(u) / (j + 1).
// In single precision the a_{t,l} are summed in double precision: with sums in single their nesting rounds more often than the general
// form's single sums (33 to 256 letters, degree 2: dA 1.46e-8 -> 1.73e-8 from 64 bits, now 0.8e-8; the calls take 1.007 of the time).
// One launch per l, from the top level down; each is a d-th of the one before.  The gradient row is read once, where the
// adjoint of the general Chen product with exp(z) as its right factor reads it twice.  Bound: HBM.  1024 rows of 10 letters,
// degree 5, double precision (0.91 GB an array): forward 491 -> 325 us (5.6 TB/s of what has to move), adjoint 840 -> 500 us (3.7).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "sig_kernels.h"

namespace sigamd {

constexpr int kJoinMaxDegree = 16;
constexpr uint32_t kJoinMaxDim = 256;

struct JoinPlan {
    int degree;
    uint32_t d;
    uint32_t lo[kJoinMaxDegree + 2];        // start of level t in a row, t = 1 .. degree + 1
    DivBy<uint32_t> dv{1};
};

// V_{t,l}(u), u the word of index `u` on level l: the factors A_i of its prefixes from the longest to the empty one
template <typename T>
__device__ __forceinline__ T join_horner(const T* __restrict__ a, const T* z, const JoinPlan& pl, int t, int l, uint32_t u)
{
    T v = T(0), prod = T(1);
    for (int i = l; i >= 1; --i) {
        v = fmadd(a[pl.lo[i] + u], prod, v);
        const uint32_t q = pl.dv.quot(u);
        prod *= z[u - q * pl.d] * (T(1) / T(t - i + 1));
        u = q;
    }
    return v + prod;
}

// out = A (x) exp(z).  Block (chunk of `words` consecutive y, row); VEC entries of 16 bytes at a time where the host found them
// aligned (VEC divides d).
template <typename T, int VEC>
__global__ __launch_bounds__(kBlock) void join_words_kernel(
    const T* __restrict__ A, const T* __restrict__ disp, T* __restrict__ out, int64_t batch, JoinPlan pl, uint32_t words, uint32_t total,
    int64_t stride, int off, T* __restrict__ scalar_out)
{
    using Vec = VecOf<T, VEC>;
    __shared__ T zl[kJoinMaxDim];
    __shared__ T vl[kBlock];
    const uint32_t d = pl.d, tid = threadIdx.x;
    const Block2 at = xcd_block_2d();
    for (int64_t b = at.y; b < batch; b += gridDim.y) {
        const T* a = A + b * stride + off;
        T* o = out + b * stride + off;
        __syncthreads();                    // the row before is done with z and V
        if (tid < d) zl[tid] = disp[b * int64_t(d) + tid];
        __syncthreads();
        const uint32_t y0 = at.x * words, n = min(words, total - y0);
        if (tid < n) {
            const uint32_t y = y0 + tid;
            int l = 0;
            T v = T(1);
            if (y) {
                l = 1;
                while (y - 1 >= pl.lo[l + 1]) ++l;
                v = join_horner(a, zl, pl, l + 1, l, y - 1 - pl.lo[l]);
            }
            vl[tid] = v;
        }
        __syncthreads();
        const uint32_t entries = n * d;
        const T* src = a + size_t(y0) * d;
        T* dst = o + size_t(y0) * d;
        constexpr int IN_FLIGHT = 4;
        for (uint32_t e0 = tid * VEC; e0 < entries; e0 += IN_FLIGHT * kBlock * VEC) {
            Vec g[IN_FLIGHT];
#pragma unroll
            for (int i = 0; i < IN_FLIGHT; ++i) {
                const uint32_t e = e0 + uint32_t(i) * kBlock * VEC;
                if (e < entries) g[i] = *reinterpret_cast<const Vec*>(src + e);
            }
#pragma unroll
            for (int i = 0; i < IN_FLIGHT; ++i) {
                const uint32_t e = e0 + uint32_t(i) * kBlock * VEC;
                if (e >= entries) break;
                const uint32_t u = pl.dv.quot(e), x = e - u * d;
                const T v = vl[u];
#pragma unroll
                for (int k = 0; k < VEC; ++k) g[i].v[k] = fmadd(v, zl[x + k], g[i].v[k]);
                *reinterpret_cast<Vec*>(dst + e) = g[i];
            }
        }
        if (scalar_out && at.x == 0 && tid == 0) scalar_out[b * stride] = T(1);
    }
}

// One level of the adjoint: words u of length l, `count` = d^l of them, `words` (a power of two, at least 4) to a block; 256 / words
// lanes, of one wave, to a word.  v_in: the n_in = degree - l - 1 arrays v_1 .. [n_in][batch][d^(l+1)];  a_out: [n_in + 1][batch][d^l].
// LDS: the chunk's entries of one v_j and, with n_in > 0, the sum over j, rows of `pitch` (odd) entries.
template <typename T, int VEC>
__global__ __launch_bounds__(kBlock) void join_words_bwd_kernel(
    const T* __restrict__ dout, const T* __restrict__ A, const T* __restrict__ disp, T* __restrict__ dA, T* __restrict__ dz,
    const T* __restrict__ v_in, T* __restrict__ a_out, int64_t batch, JoinPlan pl, int l, int n_in, uint32_t count, uint32_t words,
    uint32_t pitch, int64_t stride, int off)
{
    using Vec = VecOf<T, VEC>;
    extern __shared__ double join_tile_raw[];
    __shared__ T zl[kJoinMaxDim];
    __shared__ T vl[kBlock];
    const uint32_t d = pl.d, tid = threadIdx.x;
    T* tile = reinterpret_cast<T*>(join_tile_raw);
    T* sum = tile + words * pitch;
    const uint32_t lanes = kBlock / words, word = tid / lanes, part = tid % lanes;
    const uint32_t parts = kBlock / d, column = tid % d, row0 = tid / d;
    const Block2 at = xcd_block_2d();
    for (int64_t b = at.y; b < batch; b += gridDim.y) {
        const T* a = A + b * stride + off;
        __syncthreads();                    // the row before is done with the LDS
        if (tid < d) zl[tid] = disp[b * int64_t(d) + tid];
        const uint32_t u0 = at.x * words, n = min(words, count - u0), entries = n * d;
        T acc = T(0);
        for (int j = 0; j <= n_in; ++j) {
            const T scale = T(1) / T(j + 1);
            const T* src = (j == 0 ? dout + b * stride + off + pl.lo[l + 1] : v_in + (int64_t(j - 1) * batch + b) * (int64_t(count) * d)) + size_t(u0) * d;
            T* dst = n_in == 0 ? dA + b * stride + off + pl.lo[l + 1] + size_t(u0) * d : nullptr;
            if (j) __syncthreads();         // the tile and V of the array before have been read
            constexpr int IN_FLIGHT = 5;
            for (uint32_t e0 = tid * VEC; e0 < entries; e0 += IN_FLIGHT * kBlock * VEC) {
                Vec g[IN_FLIGHT];
#pragma unroll
                for (int i = 0; i < IN_FLIGHT; ++i) {
                    const uint32_t e = e0 + uint32_t(i) * kBlock * VEC;
                    if (e < entries) g[i] = *reinterpret_cast<const Vec*>(src + e);
                }
#pragma unroll
                for (int i = 0; i < IN_FLIGHT; ++i) {
                    const uint32_t e = e0 + uint32_t(i) * kBlock * VEC;
                    if (e >= entries) break;
                    const uint32_t u = pl.dv.quot(e), x = e - u * d;
                    if (dst) *reinterpret_cast<Vec*>(dst + e) = g[i];
#pragma unroll
                    for (int k = 0; k < VEC; ++k) {
                        T* s = sum + u * pitch + x + k;
                        tile[u * pitch + x + k] = g[i].v[k];
                        if (n_in) *s = j ? *s + g[i].v[k] : g[i].v[k];
                    }
                }
            }
            if (j == 0) __syncthreads();    // z
            if (tid < n) vl[tid] = l ? join_horner(a, zl, pl, l + 1 + j, l, u0 + tid) : T(1);
            __syncthreads();
            if (l) {
                double s = 0.0;             // in double precision: the array is rounded once at each of its levels
                if (word < n)
                    for (uint32_t x = part; x < d; x += lanes) s = fmadd(double(tile[word * pitch + x]), double(zl[x]), s);
                for (uint32_t h = lanes >> 1; h; h >>= 1) s += __shfl_xor(s, int(h));
                if (part == 0 && word < n) a_out[(int64_t(j) * batch + b) * count + u0 + word] = T(s * (1.0 / double(j + 1)));
            }
            if (row0 < parts) {
                T s = T(0);
                for (uint32_t u = row0; u < n; u += parts) s = fmadd(tile[u * pitch + column], vl[u], s);
                acc = fmadd(s, scale, acc);
            }
        }
        if (n_in) {
            T* dst = dA + b * stride + off + pl.lo[l + 1] + size_t(u0) * d;
            for (uint32_t e = tid; e < entries; e += kBlock) {
                const uint32_t u = pl.dv.quot(e);
                dst[e] = sum[u * pitch + (e - u * d)];
            }
        }
        __syncthreads();                    // V
        vl[tid] = acc;
        __syncthreads();
        if (tid < d) {
            T s = T(0);
            for (uint32_t i = 0; i < parts; ++i) s += vl[i * d + tid];
            dev_add(&dz[b * int64_t(d) + tid], s);
        }
        if (off && l == 0 && tid == 0) dA[b * stride] = T(0);
    }
}

}  // namespace sigamd
