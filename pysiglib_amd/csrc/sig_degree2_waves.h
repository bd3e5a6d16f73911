// Degree 2 of plain paths (no augmentation) on the matrix cores, operands straight from memory: a wave computes all products
// of a 64 x 64 (16 TN x 16 TN) block of channels by itself, so that every point is read once and turned into an operand once.
// The staged kernels of sig_degree2.h share a block of channels out between four waves, each of which reads all points back from
// LDS and forms all increments anew: 1858 vector instructions beside 264 matrix ones a wave, and barriers around every
// chunk (matrix units busy 39 % of the time at 2048 paths of 256 points, 64 channels).  Whole calls, us, single / double
// precision, before -> now: forward 2048 x 256 x 64: 90 -> 71, 190 -> 122; 1000 x 200 x 48: 99 -> 37, 112 -> 55; 1000 x 200 x 32: 64 ->
// 28, 70 -> 36; 500 x 300 x 96: 100 -> 62, 214 -> 116.  Bound at 64 channels: the rounds of blocks (a wave holds 64 x 64 sums, so
// four blocks a CU in single and two in double precision), 40 % of the matrix units' rate.
//
// Forward: S2 = sum_t U_t (x) z_t.  The product's index i / j within tile q stands for the channel TN * i + q: the TN tiles of
// a lane are TN consecutive channels, one load a point, and results are stored as TN consecutive coefficients.  The four
// waves of a block take a quarter of the steps each (lane group lk a quarter of those, in order, so that a point serves the step before
// it and the one after) and add their sums through LDS.
#pragma once
#include <hip/hip_runtime.h>

#include "sig_degree2.h"

namespace sigamd {

// N consecutive elements, aligned like one of them
template <typename T, int N>
struct alignas(sizeof(T)) Piece {
    T v[N];
};

// WHOLE: TN divides d, a lane's channels are one piece.  Lanes past the last channel read channels that exist (nothing of theirs is
// stored).  The host keeps the points of a wave below 2^31 elements.
template <typename T, int TN, bool SAME, bool WHOLE>
__global__ __launch_bounds__(kBlock, TN < 4 ? 1 : sizeof(T) == 8 ? 2 : SAME ? 4 : 3) void degree2_fwd_waves_kernel(
    const T* __restrict__ path, T* __restrict__ out, int64_t len_raw, int d, int64_t out_stride, int scalar, int groups, int slices,
    int64_t slice_len, int* __restrict__ nonfinite)
{
    using M = Mfma16<T>;
    using P = Piece<T, TN>;
    constexpr int W = 16 * TN, AHEAD = TN < 4 ? (sizeof(T) == 8 ? 2 : 4) : (sizeof(T) == 8 ? 1 : 2);
    constexpr int OWNERS = sizeof(T) == 8 ? 1 : 2;                 // row tiles that are added up per round of the exchange
    __shared__ T part[OWNERS * 3 * TN * 4 * kWave];
    // SAME: row and column channels of the block are the same group (one group in all)
    const int64_t per_path = int64_t(SAME ? 1 : groups * groups) * slices;
    const int64_t b = int64_t(blockIdx.x) / per_path;
    int64_t rest = int64_t(blockIdx.x) - b * per_path;
    const int slice = int(rest % slices);
    rest /= slices;
    const int cg = SAME ? 0 : int(rest % groups), rg = SAME ? 0 : int(rest / groups);
    const int lane = threadIdx.x & (kWave - 1), li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const int64_t L = len_raw - 1;
    const T* x = path + b * len_raw * d;
    T* o = out + b * out_stride + scalar;

    const int64_t t_begin = int64_t(slice) * slice_len, t_end = t_begin + slice_len < L ? t_begin + slice_len : L;
    const int64_t quarter = (t_end - t_begin + 3) / 4;
    const int64_t w_begin = t_begin + wave * quarter < t_end ? t_begin + wave * quarter : t_end;
    const int64_t w_end = w_begin + quarter < t_end ? w_begin + quarter : t_end;
    const uint32_t mine = uint32_t(w_end - w_begin), steps = (mine + 3) / 4;   // of the wave, of a lane group; past the wave's last
    const uint32_t first = uint32_t(lk) * steps;                               // step points repeat and operands are zero (also
    const uint32_t past = first + steps < mine ? first + steps : mine;         // where the repeated point is infinite)
    const T* xw = x + w_begin * d;

    const int ra = rg * W + TN * li, ca = cg * W + TN * li;
    uint32_t ro[WHOLE ? 1 : TN], co[WHOLE ? 1 : TN];
#pragma unroll
    for (int q = 0; q < (WHOLE ? 1 : TN); ++q) {
        const int last = WHOLE ? d - TN : d - 1;
        ro[q] = uint32_t(ra + q < last ? ra + q : last);
        co[q] = uint32_t(ca + q < last ? ca + q : last);
    }
    auto load = [&](const T* base, uint32_t point, const uint32_t (&o)[WHOLE ? 1 : TN]) {
        P p;
        if constexpr (WHOLE) {
            p = *reinterpret_cast<const P*>(base + (point * uint32_t(d) + o[0]));
        } else {
#pragma unroll
            for (int q = 0; q < TN; ++q) p.v[q] = base[point * uint32_t(d) + o[q]];
        }
        return p;
    };
    const P x0 = load(x, 0, ro);
    typename M::Acc acc[TN][TN];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = typename M::Acc{T(0), T(0), T(0), T(0)};

    // U_t is formed from the differences to the first point, (Y_t + Y_{t+1}) / 2 with Y = X - X_0: a sum of the points themselves
    // would round at the size of the path's offset, which the signature does not depend on (256 points, 64 channels, steps of 1/16,
    // an offset of 1000, single precision: 2.7e-5 of the result instead of 2.2e-7)
    auto point = [&](uint32_t t) { return t < mine ? t : mine; };
    const P r0 = load(xw, point(first), ro);
    P c0 = SAME ? r0 : load(xw, point(first), co);
    T y0[TN];
#pragma unroll
    for (int q = 0; q < TN; ++q) y0[q] = r0.v[q] - x0.v[q];
    P rn[AHEAD], cn[SAME ? 1 : AHEAD];
    auto fetch = [&](uint32_t s) {
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            // a lane group ends with the first point of the next one; rounds past its last step repeat that point
            const uint32_t e = point(first + (s + k + 1 < steps ? s + k + 1 : steps));
            rn[k] = load(xw, e, ro);
            if constexpr (!SAME) cn[k] = load(xw, e, co);
        }
    };
    fetch(0);
    for (uint32_t s = 0; s < steps; s += AHEAD) {
        P r1[AHEAD], c1[SAME ? 1 : AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            r1[k] = rn[k];
            if constexpr (!SAME) c1[k] = cn[k];
        }
        if (s + AHEAD < steps) fetch(s + AHEAD);
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            const P& cp = SAME ? r1[k] : c1[SAME ? 0 : k];
            const bool live = first + s + k < past;
            T u[TN], z[TN];
#pragma unroll
            for (int q = 0; q < TN; ++q) {
                const T y1 = r1[k].v[q] - x0.v[q];
                u[q] = live ? T(0.5) * (y0[q] + y1) : T(0);
                z[q] = live ? cp.v[q] - c0.v[q] : T(0);
                y0[q] = y1;
            }
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = M::mma(u[i], z[j], acc[i][j]);
            c0 = cp;
        }
    }

    // wave i adds up and stores row tile i
    T chk = T(0);
#pragma unroll
    for (int i0 = 0; i0 < TN; i0 += OWNERS) {
        if (i0) __syncthreads();
#pragma unroll
        for (int i = i0; i < TN && i < i0 + OWNERS; ++i)
            if (wave != i) {
                T* dst = part + ((i - i0) * 3 + (wave < i ? wave : wave - 1)) * (TN * 4 * kWave) + lane;
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) dst[(j * 4 + r) * kWave] = acc[i][j][r];
            }
        __syncthreads();
#pragma unroll
        for (int i = i0; i < TN && i < i0 + OWNERS; ++i) {
            if (wave != i) continue;
            const T* src = part + (i - i0) * 3 * (TN * 4 * kWave) + lane;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = rg * W + TN * M::row(lk, r) + i;
                P p;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    T v = acc[i][j][r];
#pragma unroll
                    for (int w = 0; w < 3; ++w) v += src[(w * TN * 4 + j * 4 + r) * kWave];
                    p.v[j] = v;
                    if (row < d && ca + j < d) chk = fmadd(v, T(0), chk);
                }
                if (row < d) {
                    T* dst = o + d + int64_t(row) * d + ca;
                    if (slices > 1) {
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            if (ca + j < d) dev_add(dst + j, p.v[j]);
                    } else if (ca + TN <= d) {
                        *reinterpret_cast<P*>(dst) = p;
                    } else {
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            if (ca + j < d) dst[j] = p.v[j];
                    }
                }
            }
        }
    }
    if (cg == 0 && slice == 0 && threadIdx.x < W) {
        const int a = rg * W + int(threadIdx.x);
        if (a < d) {
            const T s1 = x[L * d + a] - x[a];
            o[a] = s1;
            chk = fmadd(s1, T(0), chk);
            if (scalar && a == 0) o[-1] = T(1);
        }
    }
    if (nonfinite && !(chk == T(0))) *nonfinite = 1;
}

// Backward for at most 16 TN = 48 channels: the path gradient itself, out_t = u_t A with A = (G2 - G2^T) / 2 and
//   u_t = X_{t-1} - X_{t+1} inside, u_0 = X_0 - X_1, u_L = X_{L-1} + X_L - 2 X_0;   out_0 takes -h, out_L takes h = G1 + G2 S1.
// The product is formed transposed, A^T in registers (built once per block through LDS) times sixteen rows of u at a time, so that
// a lane loads its operands as TN pieces of four consecutive channels of one row (k step 4 q + e of lane group lk stands for
// the channel 16 q + 4 lk + e) and holds four consecutive channels of one row of every result tile.  Nothing but A and h goes
// through LDS and the four waves of a block run on their own.  Whole calls, us, single / double precision, before -> now: 1000 x 200 x
// 48: 64 -> 48, 89 -> 65; 1000 x 200 x 32: 113 -> 37, 122 -> 48; 4000 x 100 x 16: 97 -> 33, 115 -> 44.  WHOLE: 4 divides d, pieces are all there or past the last
// channel (there they repeat the last piece and are set to zero).
template <typename T, int TN, bool WHOLE>
__global__ __launch_bounds__(kBlock, 2) void degree2_bwd_waves_kernel(
    const T* __restrict__ path, const T* __restrict__ gsig, T* __restrict__ out, int64_t len_raw, int d, int64_t sig_stride, int scalar,
    int parts, int64_t part_rows)
{
    using M = Mfma16<T>;
    using P = Piece<T, 4>;
    constexpr int W = 16 * TN, PITCH = W + 1;
    __shared__ T gl[W * PITCH], s1[W], hb[W];
    const int64_t b = int64_t(blockIdx.x) / parts;
    const int64_t L = len_raw - 1;
    const uint32_t begin = uint32_t((int64_t(blockIdx.x) - b * parts) * part_rows);
    const uint32_t end = uint32_t(begin + part_rows < len_raw ? begin + part_rows : len_raw);
    const T* x = path + b * len_raw * d;
    const T* g1 = gsig + b * sig_stride + scalar;
    const T* g2 = g1 + d;
    T* o = out + b * len_raw * d;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    uint32_t at[TN][WHOLE ? 1 : 4];
#pragma unroll
    for (int q = 0; q < TN; ++q)
#pragma unroll
        for (int e = 0; e < (WHOLE ? 1 : 4); ++e) {
            const int c = 16 * q + 4 * lk + e, last = WHOLE ? d - 4 : d - 1;
            at[q][e] = uint32_t(c < last ? c : last);
        }
    auto load = [&](uint32_t row, P (&p)[TN]) {
        const uint32_t base = row * uint32_t(d);
#pragma unroll
        for (int q = 0; q < TN; ++q) {
            if constexpr (WHOLE) {
                p[q] = *reinterpret_cast<const P*>(x + (base + at[q][0]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) p[q].v[e] = x[base + at[q][e]];
            }
        }
    };
    const uint32_t last_row = uint32_t(L);
    auto fetch = [&](uint32_t row0, P (&lo)[TN], P (&hi)[TN]) {
        const uint32_t t = row0 + li < last_row ? row0 + li : last_row;
        load(t ? t - 1 : 0, lo);
        load(t < last_row ? t + 1 : last_row, hi);
    };
    P lo[TN], hi[TN];
    uint32_t row0 = begin + 16 * wave;
    if (row0 < end) fetch(row0, lo, hi);

    // G2 and S1 to LDS, zeros past the last channel
    for (int e = tid; e < W * W; e += kBlock) {
        const int a = e / W, c = e % W;
        gl[a * PITCH + c] = (a < d && c < d) ? g2[int64_t(a) * d + c] : T(0);
    }
    if (tid < W) s1[tid] = tid < d ? x[L * d + tid] - x[tid] : T(0);
    __syncthreads();
    T af[4 * TN][TN];
#pragma unroll
    for (int kk = 0; kk < 4 * TN; ++kk)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            // result row i of a tile is the channel whose four neighbours a lane receives
            const int i = sizeof(T) == 8 ? 4 * (li & 3) + (li >> 2) : li;
            const int a = 16 * (kk >> 2) + 4 * lk + (kk & 3), c = 16 * j + i;
            af[kk][j] = T(0.5) * (gl[a * PITCH + c] - gl[c * PITCH + a]);
        }
    if (tid < W) {
        T sum[4] = {tid < d ? g1[tid] : T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int e = 0; e < W; e += 4) {
#pragma unroll
            for (int q = 0; q < 4; ++q) sum[q] = fmadd(gl[tid * PITCH + e + q], s1[e + q], sum[q]);
        }
        hb[tid] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    }
    __syncthreads();

    for (; row0 < end; row0 += 64) {
        const uint32_t t = row0 + li;
        T u[4 * TN];
#pragma unroll
        for (int q = 0; q < TN; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) u[4 * q + e] = lo[q].v[e] - hi[q].v[e];
        if (row0 + 15 >= last_row) {            // the path's last row is among the sixteen
            P x0[TN];
            load(0, x0);
#pragma unroll
            for (int q = 0; q < TN; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const T v = (lo[q].v[e] - x0[q].v[e]) + (hi[q].v[e] - x0[q].v[e]);
                    u[4 * q + e] = t == last_row ? v : u[4 * q + e];
                }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)             // channels past the last, all in the last tile
            u[4 * (TN - 1) + e] = 16 * (TN - 1) + 4 * lk + e < d ? u[4 * (TN - 1) + e] : T(0);
        if (row0 + 64 < end) fetch(row0 + 64, lo, hi);
        typename M::Acc acc[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[j] = typename M::Acc{T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int kk = 0; kk < 4 * TN; ++kk)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[j] = M::mma(af[kk][j], u[kk], acc[j]);
        if (t < end) {
            T* dst = o + (t * uint32_t(d) + 4 * lk);
            const T sign = t == last_row ? T(1) : T(-1);
            const bool edge = t == 0 || t == last_row;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int c = 16 * j + 4 * lk;
                P p;
#pragma unroll
                for (int r = 0; r < 4; ++r) p.v[r] = acc[j][r];
                if (edge) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) p.v[r] = fmadd(sign, hb[c + r], p.v[r]);
                }
                if (c + 4 <= d) {
                    *reinterpret_cast<P*>(dst + 16 * j) = p;
                } else if (!WHOLE) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (c + r < d) dst[16 * j + r] = p.v[r];
                }
            }
        }
    }
}

}  // namespace sigamd
