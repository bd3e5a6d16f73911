// Tensor logarithm and its adjoint with a block per row, for rows that one compute unit can hold (sig_log.hip chooses).
//
//   log(1 + x) = P_1,   P_k = x / k - x (x) P_{k+1},   P_{N+1} = 0            (siglib/cpsig/cp_tensor_log.h:40-113)
//
// P_2 .. P_N and everything that the adjoint adds up for them lies on levels below N.  A block keeps those levels of its row
// in LDS (the adjoint of a few rows that need more: in a workspace that stays in the L2) and runs the whole recursion between
// barriers; the top level, most of the row, stays where it is.  The form that launches a kernel per step instead is bound by
// the number of its launches: six forward and some thirty backward, 5 us each for a few us of work.  257 rows of 7 letters,
// degree 5, single precision, Lyndon words, whole calls: forward 54 -> 34 us, backward 211 -> 77; one row 36 -> 27, 147 -> 60;
// 2048 rows 144 -> 63, 784 -> 290.  What bounds them now: the reads of the top level, 2 (N - 1) times from the L2, by a block
// that has its compute unit to itself.  With the whole row in LDS the adjoint of one row takes 67 instead of 74 us, that of
// 257 rows 99 instead of 84 (one block a unit instead of two): left out.
//
// The adjoint of a product x (x) P read from a gradient row g: with c(t) = d + .. + d^t, the entries g[u v] of all words u of
// length 1 .. top - m and all words v of length m form ONE matrix, g[c(m) + y * d^m + v], y = the position of u in the row.
// So   d/dx[y] = sum_m sum_v M_m[y][v] P_m[v]   and   d/dP_m[v] = sum_y M_m[y][v] x[y]   are plain matrix-vector products,
// one pair for each m.  Every sum has one owner and a fixed order: no atomics.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "sig_kernels.h"

namespace sigamd {

constexpr int kLogRowMaxDegree = 20;
constexpr int kLogRowBlock = 1024;

struct LogRowPlan {
    int degree;
    uint32_t d;
    uint32_t n, low;                            // coefficients of the row; of its levels below the top one
    uint32_t lo[kLogRowMaxDegree + 2];          // start of level t in the row, t = 1 .. degree + 1
    uint32_t pw[kLogRowMaxDegree + 1];          // d^t
    uint32_t poff[kLogRowMaxDegree + 2];        // adjoint: start of P_k among the stored ones, k = degree .. 2
    uint32_t p_total;
    DivBy<uint32_t> dv{1};
};

// the lanes of a block that see a row's levels: positions to levels and digits without touching the argument segment with
// an index that differs between lanes
struct LogRowLevels {
    uint32_t lo[kLogRowMaxDegree + 2], pw[kLogRowMaxDegree + 1];
};

// x_l (x) P summed over the splits of the word at position r (level t): prefix of x, suffix of P
template <typename T>
__device__ __forceinline__ T log_row_splits(const T* x, const T* p, uint32_t r, const LogRowLevels& lv, const DivBy<uint32_t>& dv)
{
    int t = 1;
    while (r >= lv.lo[t + 1]) ++t;
    const uint32_t w = r - lv.lo[t];
    uint32_t pre = w;
    T sum = T(0);
    for (int j = 1; j < t; ++j) {               // j letters of the suffix
        pre = dv.quot(pre);
        sum = fmadd(x[lv.lo[t - j] + pre], p[lv.lo[j] + (w - pre * lv.pw[j])], sum);
    }
    return sum;
}

__device__ __forceinline__ void log_row_levels(const LogRowPlan& pl, LogRowLevels& lv)
{
    for (int i = int(threadIdx.x); i <= pl.degree + 1; i += int(blockDim.x)) {
        lv.lo[i] = pl.lo[i];
        if (i <= pl.degree) lv.pw[i] = pl.pw[i];
    }
}

// Forward.  Block (part, row): every part of a row runs the recursion of the lower levels for itself, on copies of x and P in LDS (the
// host takes this form only where they fit), and evaluates its share of P_1: `index`: at the listed positions, the Lyndon words, one
// after the other; null: everywhere.  Coordinates in the Lyndon basis are combined by a launch of their own.
template <typename T>
__global__ __launch_bounds__(kLogRowBlock) void tensor_log_row_kernel(
    const T* __restrict__ X, T* __restrict__ out, int64_t batch, LogRowPlan pl, const uint64_t* __restrict__ index, uint32_t count,
    int64_t stride, int off, int64_t out_stride, int out_off)
{
    extern __shared__ double log_row_raw[];
    __shared__ LogRowLevels lv;
    constexpr int R = 4;
    const uint32_t nt = blockDim.x, tid = threadIdx.x;
    const int N = pl.degree;
    log_row_levels(pl, lv);
    for (int64_t b = blockIdx.y; b < batch; b += gridDim.y) {
        const T* src = X + b * stride + off;
        T* x = reinterpret_cast<T*>(log_row_raw);
        T* p = x + pl.low;
        __syncthreads();                        // the levels; the row before this one has been read
        for (uint32_t r = tid; r < pl.low; r += nt) x[r] = src[r];
        const T last = T(1) / T(N);
        for (uint32_t r = tid; r < pl.d; r += nt) p[r] = src[r] * last;
        __syncthreads();
        // P_k over P_{k+1} in place: a coefficient reads only levels below its own, so positions are done from the top down
        for (int k = N - 1; k >= 2; --k) {
            const T inv = T(1) / T(k);
            uint32_t end = pl.lo[N - k + 2];                    // levels <= N - k + 1
            while (end) {
                const uint32_t begin = end > nt * R ? end - nt * R : 0;
                T v[R];
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    const uint32_t r = begin + tid + uint32_t(i) * nt;
                    v[i] = r < end ? x[r] * inv - log_row_splits(x, p, r, lv, pl.dv) : T(0);
                }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    const uint32_t r = begin + tid + uint32_t(i) * nt;
                    if (r < end) p[r] = v[i];
                }
                __syncthreads();
                end = begin;
            }
        }
        T* o = out + b * out_stride + out_off;
        const uint32_t items = index ? count : pl.n;
        for (uint32_t i = blockIdx.x * nt + tid; i < items; i += gridDim.x * nt) {
            const uint32_t r = index ? uint32_t(index[i]) : i;
            o[i] = src[r] - log_row_splits(x, p, r, lv, pl.dv);
        }
        if (!index && out_off && blockIdx.x == 0 && tid == 0) o[-out_off] = T(0);
    }
}

// sum of x[xo + i * xs] * g[go + i * gs] over i < n: four entries' loads are in flight together.  In the last round entries
// past the end repeat the last one and are left out by selection.
template <typename T>
__device__ __forceinline__ T log_row_sum(const T* x, uint32_t xo, uint32_t xs, const T* g, uint32_t go, uint32_t gs, uint32_t n)
{
    T s0 = T(0), s1 = T(0), s2 = T(0), s3 = T(0);
    for (; n >= 4; n -= 4) {
        const T g0 = g[go], g1 = g[go + gs], g2 = g[go + 2 * gs], g3 = g[go + 3 * gs];
        const T x0 = x[xo], x1 = x[xo + xs], x2 = x[xo + 2 * xs], x3 = x[xo + 3 * xs];
        s0 = fmadd(x0, g0, s0);
        s1 = fmadd(x1, g1, s1);
        s2 = fmadd(x2, g2, s2);
        s3 = fmadd(x3, g3, s3);
        go += 4 * gs;
        xo += 4 * xs;
    }
    if (n) {
        const uint32_t i1 = n > 1 ? 1 : 0, i2 = n > 2 ? 2 : 0;
        const T g0 = g[go], g1 = g[go + i1 * gs], g2 = g[go + i2 * gs];
        const T x0 = x[xo], x1 = x[xo + i1 * xs], x2 = x[xo + i2 * xs];
        const T t1 = fmadd(x1, g1, s1), t2 = fmadd(x2, g2, s2);
        s0 = fmadd(x0, g0, s0);
        s1 = n > 1 ? t1 : s1;
        s2 = n > 2 ? t2 : s2;
    }
    return (s0 + s1) + (s2 + s3);
}

// entries of a level that a wave's lanes cover several times over: the waves' partial sums meet in `red`
constexpr uint32_t kLogRowRed = 16 * 128;       // waves times the entries of all levels below 64

// Adjoint.  out holds the gradient with respect to the signature; its top level is the expanded gradient of P_1, which the
// block writes there first and then reads from there.
template <typename T, bool SHARED>
__global__ __launch_bounds__(kLogRowBlock) void tensor_log_row_bwd_kernel(
    const T* __restrict__ X, T* out, const T* __restrict__ derivs, int64_t batch, LogRowPlan pl,
    const uint64_t* __restrict__ index, uint32_t count, const uint64_t* __restrict__ t_row_ptr, const uint32_t* __restrict__ t_col,
    const int32_t* __restrict__ t_val, int64_t stride, int off, T* ws, int64_t ws_stride)
{
    extern __shared__ double log_row_raw[];
    __shared__ LogRowLevels lv;
    __shared__ T red[kLogRowRed];
    const uint32_t nt = blockDim.x, tid = threadIdx.x, lane = tid % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), waves = nt / kWave;
    const int N = pl.degree;
    log_row_levels(pl, lv);
    for (int64_t b = blockIdx.x; b < batch; b += gridDim.x) {
        const T* src = X + b * stride + off;
        T* o = out + b * stride + off;
        T* mine = SHARED ? reinterpret_cast<T*>(log_row_raw) : ws + b * ws_stride;
        T* x = mine;
        T* dx = x + pl.low;
        T* ga = dx + pl.low;
        T* gb = ga + pl.low;
        T* ps = gb + pl.low;
        __syncthreads();                        // the levels; the row before this one has been read
        for (uint32_t r = tid; r < pl.low; r += nt) x[r] = src[r];
        // the gradient of the expanded logarithm: lower levels in ga, the top level in place
        if (index) {
            const T* gs = derivs + b * int64_t(count);
            for (uint32_t r = tid; r < pl.low; r += nt) ga[r] = T(0);
            for (uint32_t r = pl.low + tid; r < pl.n; r += nt) o[r] = T(0);
            __syncthreads();
            for (uint32_t j = tid; j < count; j += nt) {
                T acc = gs[j];
                if (t_row_ptr)
                    for (uint64_t e = t_row_ptr[j]; e < t_row_ptr[j + 1]; ++e) acc = fmadd(T(t_val[e]), gs[t_col[e]], acc);
                const uint32_t r = uint32_t(index[j]);
                if (r < pl.low) ga[r] = acc;
                else o[r] = acc;
            }
        } else {
            const T* gs = derivs + b * stride + off;
            for (uint32_t r = tid; r < pl.low; r += nt) ga[r] = gs[r];
            for (uint32_t r = pl.low + tid; r < pl.n; r += nt) o[r] = gs[r];
        }
        if (off && tid == 0) o[-off] = T(0);
        // P_N .. P_2
        for (uint32_t r = tid; r < pl.d; r += nt) ps[pl.poff[N] + r] = src[r] * (T(1) / T(N));
        __syncthreads();
        for (uint32_t r = tid; r < pl.low; r += nt) dx[r] = ga[r];
        for (int k = N - 1; k >= 2; --k) {
            const T inv = T(1) / T(k);
            const T* pin = ps + pl.poff[k + 1];
            T* po = ps + pl.poff[k];
            for (uint32_t r = tid; r < pl.lo[N - k + 2]; r += nt) po[r] = x[r] * inv - log_row_splits(x, pin, r, lv, pl.dv);
            __syncthreads();
        }
        if (N == 2) __syncthreads();            // dx, where no such step came in between
        T* g = ga;
        T* gn = gb;
        for (int k = 1; k < N; ++k) {
            const int top = N - k + 1;          // levels of the gradient of P_k
            const T* p = ps + pl.poff[k + 1];
            const bool split = k == 1;          // the top level is not among the levels in g
            // x: word u of level l against all words v that follow it; 1 to 64 lanes a word
            for (int l = top - 1; l >= 1; --l) {
                uint32_t lanes = 1;
                while (lanes < kWave && lanes * 16 <= pl.lo[top - l + 1]) lanes *= 2;
                const uint32_t own = lane & (lanes - 1), per_wave = kWave / lanes;
                for (uint32_t u = wave * per_wave + lane / lanes; u < pl.pw[l]; u += waves * per_wave) {
                    const uint32_t y = pl.lo[l] + u;
                    T s = T(0);
                    for (int m = 1; m <= top - l; ++m) {
                        const uint32_t w = pl.pw[m], at = pl.lo[m + 1] + y * w + own;
                        const uint32_t n = own < w ? (w - own + lanes - 1) / lanes : 0;
                        if (split && l + m == N) s += log_row_sum(p, pl.lo[m] + own, lanes, (const T*)o, at, lanes, n);
                        else s += log_row_sum(p, pl.lo[m] + own, lanes, (const T*)g, at, lanes, n);
                    }
                    for (uint32_t h = lanes >> 1; h; h >>= 1) s += __shfl_xor(s, int(h));
                    if (own == 0) dx[y] -= s;
                }
            }
            // P_{k+1}: word v against all words u in front of it.  Levels of fewer than 64 words: a wave takes 64 / w rows at a time
            uint32_t at_red = 0;
            for (int m = 1; m < top; ++m) {
                const uint32_t w = pl.pw[m], base = pl.lo[m + 1], rows = pl.lo[top - m + 1];
                const uint32_t inner = split ? pl.lo[top - m] : rows;       // rows below the top level
                if (w >= kWave) {
                    for (uint32_t v = tid; v < w; v += nt) {
                        T s = log_row_sum(x, 0, 1, (const T*)g, base + v, w, inner);
                        if (split) s += log_row_sum(x, inner, 1, (const T*)o, base + inner * w + v, w, rows - inner);
                        gn[pl.lo[m] + v] = -s;
                    }
                } else {
                    uint32_t q = lane;
                    for (int i = 0; i < m; ++i) q = pl.dv.quot(q);
                    const uint32_t v = lane - q * w, together = kWave / w, first = wave * together + q, step = waves * together;
                    T s = T(0);
                    if (q < together) {
                        if (first < inner) s = log_row_sum(x, first, step, (const T*)g, base + first * w + v, step * w, (inner - first + step - 1) / step);
                        if (split && inner + first < rows)
                            s += log_row_sum(x, inner + first, step, (const T*)o, base + (inner + first) * w + v, step * w,
                                             (rows - inner - first + step - 1) / step);
                    }
                    T sum = s;
                    for (uint32_t i = 1; i < together; ++i) sum += __shfl(s, int(v + i * w));
                    if (lane < w) red[at_red + wave * w + lane] = sum;
                    at_red += waves * w;
                }
            }
            __syncthreads();
            const T inv = T(1) / T(k + 1);
            at_red = 0;
            for (int m = 1; m < top; ++m) {
                const uint32_t w = pl.pw[m];
                for (uint32_t v = tid; v < w; v += nt) {
                    const uint32_t r = pl.lo[m] + v;
                    if (w < kWave) {
                        T s = T(0);
                        for (uint32_t i = 0; i < waves; ++i) s += red[at_red + i * w + v];
                        gn[r] = -s;
                    }
                    dx[r] = fmadd(gn[r], inv, dx[r]);
                }
                if (w < kWave) at_red += waves * w;
            }
            __syncthreads();
            T* h = g;
            g = gn;
            gn = h;
        }
        for (uint32_t r = tid; r < pl.low; r += nt) o[r] = dx[r];
    }
}

}  // namespace sigamd
