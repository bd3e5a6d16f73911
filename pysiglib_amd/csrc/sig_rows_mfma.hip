// Single-precision sweeps for paths of many channels (33 and more) on the matrix units, forward at degrees 3 .. 7, backward
// at degrees 3 .. 6.
//
// Arithmetic: siglib/cpsig/cp_signature.h:464-499 (forward) and :1137-1187 (reverse).  The lower levels run as in
// sig_rows.hip (a lane owns a word prefix of N - 1 letters and its chain); what bounds these sweeps is the top level, one
// (forward) or two (reverse) multiply-adds per coefficient and step, and over several steps these are matrix products:
//   forward   S_N[p, a]  += sum_t U_t[p] z_t[a]        K = steps
//   reverse   red_t[p]    = sum_a G[p, a] z_t[a]       K = letters,  G: the top-level adjoint, constant in the sweep
//             dz_t[a]    += sum_p G[p, a] U_t[p]       K = prefixes
// The vector units reach 69 - 77 TFLOP/s in single precision without packed operations, the matrix units twice that, and
// their instructions run beside the chain work of the other waves.  The products are the same single-precision
// multiply-adds: the forward sweep agrees with the vector kernels bit for bit.
#include <hip/hip_runtime.h>

#include "sig_rows.h"
#include "sig_rows_lanes.h"
#include "sig_launch.h"

namespace sigamd {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kMxMinDim = 33;
constexpr int kMxMaxDim = 4096;

// the tile of a wave: prefixes (r, 64 blk + lane), letters 64 ga ..; all wave-uniform
template <int M>
struct MxTile {
    int ga, blk;
    int64_t r;
    int pu[M - 1];      // the letters of r
    __device__ __forceinline__ MxTile(int64_t w, int d, int nblk, int nga)
    {
        ga = int(w % nga);
        w /= nga;
        blk = int(w % nblk);
        r = w / nblk;
        int64_t q = r;
#pragma unroll
        for (int l = M - 2; l >= 0; --l) {
            pu[l] = __builtin_amdgcn_readfirstlane(int(q % d));     // wave-uniform: say so (64-bit division is vector code)
            q /= d;
        }
    }
};

// ---------------------------------------------------------------------------
// Forward.  Two steps at a time: lane p computes U_t[p] and U_{t+1}[p]; one exchange of half-waves turns the two into
// the left operands (32 prefixes x 2 steps) of two 32x32x2 products per 32 letters, the right operand comes from the
// increments as they lie in memory.  An odd last step is paired with zeros, and its chain is left alone.
// ---------------------------------------------------------------------------
template <int N>
__global__ __launch_bounds__(kBlock, 4) void rows_fwd_mfma_kernel(
    const float* __restrict__ inc, float* __restrict__ out, int64_t batch, int64_t L, int d, int64_t out_stride, int scalar,
    int64_t rows /* d^(N-2) */, int nblk, int nga, int* __restrict__ nonfinite)
{
    using T = float;
    using Tr = Tree<T, -1, N, 1, 1>;
    constexpr int M = N - 1;
    static_assert(M >= 2, "degree 3 and up");
    const int lane = threadIdx.x & (kWave - 1);
    int64_t wave = int64_t(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
    {
        const uint32_t wlo = __builtin_amdgcn_readfirstlane(uint32_t(wave));
        const uint32_t whi = __builtin_amdgcn_readfirstlane(uint32_t(uint64_t(wave) >> 32));
        wave = int64_t((uint64_t(whi) << 32) | wlo);
    }
    const int64_t per_path = rows * nblk * nga;
    const int64_t b = wave / per_path;
    if (b >= batch) return;
    const MxTile<M> tl(wave - b * per_path, d, nblk, nga);
    const int a0 = tl.ga * kWave;
    const int last = tl.blk * kWave + lane;
    const bool active = last < d;
    const int lastc = active ? last : d - 1;        // idle lanes shadow a valid lane: every load stays in bounds
    const int64_t q = tl.r * d + lastc;
    // wave-uniform: whether the tile's second 32 prefixes / letters exist
    const bool p2 = tl.blk * kWave + 32 < d, l2 = a0 + 32 < d;

    Tr S;
#pragma unroll
    for (int l = 0; l < M; ++l) S.c[l] = T(0);
    S.s[0] = T(0);
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i >> 1][i & 1][r] = 0.f;

    // increments [batch][L + 2][d] with a zero row at either end of a path and rows of slack around the array
    const T* zrow = inc + (b * (L + 2) + 1) * d;        // row of the first step
    const int half = lane >> 5, col = lane & 31;
    const int la = half * d + (a0 + col < d ? a0 + col : d - 1);
    const int lb = half * d + (a0 + 32 + col < d ? a0 + 32 + col : d - 1);
    typename Tr::Inc in;
    in.z[0] = T(0);
    in.zs[0] = T(0);
    T pz_next[2][M], za_next, zb_next;
    auto fetch = [&](const T* row) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int l = 0; l < M - 1; ++l) pz_next[s][l] = row[s * d + tl.pu[l]];
            pz_next[s][M - 1] = row[s * d + lastc];
        }
        za_next = row[la];
        zb_next = row[lb];
    };
    auto horner = [&](const T (&pz)[M]) -> T {          // U of the step, and the chain behind it
#pragma unroll
        for (int l = 0; l < M; ++l) in.pz[l] = pz[l];
        if constexpr (Tr::kLockstep) {
            typename Tr::Chain ch;
            S.fwd_step(in, &ch);
            return ch.u[N][M - 1];
        } else {
            T uu[M];
            S.template chain_u<N, M>(in, uu);
            S.fwd_step(in);
            return uu[M - 1];
        }
    };
    // one copy of the loop per form of the tile: a branch around a product would cost copies of its 16 registers
    auto sweep = [&](auto p2_, auto l2_) {
        constexpr bool P2 = decltype(p2_)::value != 0, L2 = decltype(l2_)::value != 0;
        auto products = [&](T u0, T u1, T za, T zb) {
            const auto sw = __builtin_amdgcn_permlane32_swap(unsigned(__float_as_int(u0)), unsigned(__float_as_int(u1)), false, false);
            const T ua = __int_as_float(int(sw[0])), ub = __int_as_float(int(sw[1]));
            acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(ua, za, acc[0][0], 0, 0, 0);
            if constexpr (L2) acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(ua, zb, acc[0][1], 0, 0, 0);
            if constexpr (P2) acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(ub, za, acc[1][0], 0, 0, 0);
            if constexpr (P2 && L2) acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(ub, zb, acc[1][1], 0, 0, 0);
        };
        fetch(zrow);
        for (int64_t t = 0; t + 1 < L; t += 2) {
            T pz[2][M];
#pragma unroll
            for (int l = 0; l < M; ++l) {
                pz[0][l] = pz_next[0][l];
                pz[1][l] = pz_next[1][l];
            }
            const T za = za_next, zb = zb_next;
            const T u0 = horner(pz[0]), u1 = horner(pz[1]);
            // requested once this pair's scalar loads have been used: a wait for one of them is a wait for all
            __builtin_amdgcn_sched_barrier(0);
            zrow += 2 * d;                              // past the last step: the zero row, then the slack
            fetch(zrow);
            __builtin_amdgcn_sched_barrier(0);
            products(u0, u1, za, zb);
        }
        if (L & 1) products(horner(pz_next[0]), T(0), za_next, zb_next);
    };
    if (p2 && l2) sweep(IntC<1>{}, IntC<1>{});
    else if (p2) sweep(IntC<1>{}, IntC<0>{});
    else if (l2) sweep(IntC<0>{}, IntC<1>{});
    else sweep(IntC<0>{}, IntC<0>{});

    T* o = out + b * out_stride;
    if (scalar && tl.r == 0 && tl.blk == 0 && tl.ga == 0 && lane == 0) o[0] = T(1);
    // chk stays 0 while every stored value is finite: x * 0 is NaN for x = NaN or +-Inf
    T chk = T(0);
    int64_t off = scalar ? 1 : 0, size = d;
#pragma unroll
    for (int l = 1; l <= M; ++l) {
        int64_t span = 1;                            // d^(M - l): prefixes of full length below one level-l node
#pragma unroll
        for (int i = l; i < M; ++i) span *= d;
        // a chain node is stored by the lane whose remaining prefix letters are 0, in the first letter tile
        if (active && tl.ga == 0 && q % span == 0) {
            o[off + q / span] = S.c[l - 1];
            chk = fmadd(S.c[l - 1], T(0), chk);
        }
        off += size;
        size *= d;
    }
    T* top = o + off + tl.r * d * d;
#pragma unroll
    for (int ph = 0; ph < 2; ++ph) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int p = tl.blk * kWave + 32 * ph + 8 * (r / 4) + 4 * half + (r & 3);
#pragma unroll
            for (int lh = 0; lh < 2; ++lh) {
                const int a = a0 + 32 * lh + col;
                if (p < d && a < d) {
                    const T v = acc[ph][lh][r];
                    top[int64_t(p) * d + a] = v;
                    chk = fmadd(v, T(0), chk);
                }
            }
        }
    }
    if (nonfinite && !(chk == T(0))) *nonfinite = 1;
}

// ---------------------------------------------------------------------------
// Reverse.  Sixteen steps at a time, per wave:
//   1. red for all of them, 16x16x4 products (steps x letters) (letters x prefixes), through LDS to lane = prefix;
//   2. the steps themselves: chain back, pullback; U_t[p] takes red's place in LDS;
//   3. dz for all of them, (steps x prefixes) (prefixes x letters).
// To degree 4 the products of 1. stand between the pieces of 2. of the sixteen steps before, one by one: the matrix and the
// vector unit of a SIMD, 35 % of the time each when a wave used one at a time, then work side by side in one wave too
// (degree 4, single precision, ms: 64 paths x 128 steps x 64 channels 10.9 -> 10.1, 1 x 399 x 65 2.30 -> 2.02, 8 x 33 x 96
// 5.29 -> 5.01; degree 3: 300 x 49 x 64 0.477 -> 0.440).  At degrees 5 and 6 the steps are most of the work and the next
// steps' operands would not fit the registers (1 x 399 x 34, degree 5: 4.85 -> 4.93), so 1. comes first there.  3. in the
// same manner, as products of four steps (4x4x1), gained nothing more (10.02 -> 10.08).
// The wave holds its tile of G in both operand layouts (128 registers); each product is summed in two halves of K.
// The pieces of a step's gradient row stay in the waves' own LDS until the block adds them up and onto the row.  Thousands
// of blocks add to a row: it is kept in double precision, so that their number costs no accuracy.
// ---------------------------------------------------------------------------
constexpr int kMxSteps = 16;
constexpr int kMxStride = 68;       // words per step: writes of four rows apart and 16-byte reads of 16 rows both spread over all banks
constexpr int kMxBuf = kMxSteps * kMxStride;
constexpr int kMxWaveWords = 3 * kMxBuf;      // red / U of these and of the next steps, pieces
constexpr int kMxGroup = 4;        // steps in a straight line: their red values and increments are loaded together
// Waves per block: two blocks share a CU and drift apart, so that one's products run beside the other's chains (16 paths of
// 200 steps, 64 channels, degree 4, with elements dealt out one by one at the
// end of a chunk: 4.26 ms; one block of eight waves, in step with itself: 4.67).
constexpr int kMxWaves = 4;
constexpr int kMxBwdMaxDim = 256;   // the block's tile of gradient rows stays small beside the waves' own words

template <int N>
__global__ __launch_bounds__((kMxWaves * kWave), 2) void rows_bwd_mfma_kernel(
    const float* __restrict__ inc, const float* __restrict__ sig, const float* __restrict__ gsig,
    double* __restrict__ dzinc, int64_t L, int d, int64_t sig_stride, int scalar, int64_t rows /* d^(N-2) */, int nblk, int nga,
    int64_t blocks_per_path)
{
    using T = float;
    using Tr = Tree<T, -1, N, 1, 1>;
    using Ad = TreeAdj<T, -1, N, 1, 1>;
    constexpr int M = N - 1;
    constexpr int W = kMxWaves;
    constexpr bool kAhead = N <= 4;                     // red of the next steps between the pieces of these
    static_assert(M >= 2, "degree 3 and up");
    const int lane = threadIdx.x & (kWave - 1);
    const int wib = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));

    // The waves of a block belong to one path.  Surplus waves of a path's last block shadow its last tile with all
    // adjoints zero, so that every wave of a block reaches every barrier.
    const int64_t per_path = rows * nblk * nga;
    const int64_t b = int64_t(blockIdx.x) / blocks_per_path;
    const int64_t w = (int64_t(blockIdx.x) - b * blocks_per_path) * W + wib;
    const bool valid = w < per_path;
    const MxTile<M> tl(valid ? w : per_path - 1, d, nblk, nga);
    const int a0 = tl.ga * kWave;
    const int last = tl.blk * kWave + lane;         // this lane's last prefix letter
    const bool active = valid && last < d;
    const int lastc = last < d ? last : d - 1;      // idle lanes shadow a valid lane: every load stays in bounds
    const int64_t q = tl.r * d + lastc;

    Tr S;
    Ad A;
    const T* srow = sig + b * sig_stride;
    const T* grow = gsig + b * sig_stride;
    int64_t leaf_off;
    {
        int64_t off = scalar ? 1 : 0, size = d;      // start and size of level l
#pragma unroll
        for (int l = 1; l <= M; ++l) {
            int64_t span = 1;                        // d^(M - l): prefixes of full length below one level-l node
#pragma unroll
            for (int i = l; i < M; ++i) span *= d;
            const int64_t idx = off + q / span;
            // a chain node's adjoint is seeded in one lane only: the recursion is linear in the adjoint
            const bool owner = active && tl.ga == 0 && (q % span == 0);
            S.c[l - 1] = srow[idx];
            A.gc[l - 1] = owner ? grow[idx] : T(0);
            off += size;
            size *= d;
        }
        leaf_off = off;
    }
    A.gs[0] = T(1);
    S.s[0] = T(0);
    const int g16 = lane >> 4, x16 = lane & 15;
    const T* top = grow + leaf_off + tl.r * d * d;      // G[last prefix letter][letter] of this row of prefixes
    // right operand of red: prefixes 16 i + x16, letters 16 g16 + k
    T gp[4][16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int p = tl.blk * kWave + 16 * i + x16;
        const T* g = top + int64_t(p < d ? p : d - 1) * d;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int a = a0 + 16 * g16 + k;
            const T v = g[a < d ? a : d - 1];
            gp[i][k] = valid && p < d && a < d ? v : T(0);
        }
    }
    // right operand of dz: letters 16 i + x16, prefixes 16 g16 + k
    T gt[4][16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int a = a0 + 16 * i + x16;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int p = tl.blk * kWave + 16 * g16 + k;
            const T v = top[int64_t(p < d ? p : d - 1) * d + (a < d ? a : d - 1)];
            gt[i][k] = valid && p < d && a < d ? v : T(0);
        }
    }

    extern __shared__ f32x4 mx_lds_raw[];               // read four words at a time: aligned by its type
    static_assert(kMxStride % 4 == 0 && kMxWaveWords % 4 == 0, "a step's words start on 16 bytes");
    T* mx_lds = reinterpret_cast<T*>(mx_lds_raw);
    __shared__ int wave_a0[W], wave_l0[W];
    T* mine = mx_lds + wib * kMxWaveWords;              // [step][kMxStride]: red, then U, then the by-letter sums
    T* mine_next = mine + kMxBuf;                       // red of the steps after these
    T* mine_c = mine + 2 * kMxBuf;                      // pieces of the last prefix letter
    T* tile = mx_lds + W * kMxWaveWords;                // [step][d]: pieces of the shared prefix letters
    for (int e = threadIdx.x; e < kMxSteps * d; e += W * kWave) tile[e] = T(0);
    if (lane == 0) {
        wave_a0[wib] = a0;
        wave_l0[wib] = tl.blk * kWave;
    }
    __syncthreads();

    const T* zbase = inc + (b * (L + 2) + 1) * d;       // row of step 0; a zero row in front
    typename Tr::Inc in;
    in.z[0] = T(0);
    // the last prefix letter's increments, requested a group of steps ahead (the last group reads on in front of the path,
    // at most 2 kMxGroup rows: the zero row, other paths' rows or the slack; what it makes of them is not used)
    const T* zlast = zbase + (L - 1) * d + lastc;
    T zl_next[kMxGroup];
    auto fetch_last = [&]() {
#pragma unroll
        for (int k = 0; k < kMxGroup; ++k) {
            zl_next[k] = *zlast;
            zlast -= d;
        }
    };
    fetch_last();
    struct alignas(4) Quad { T v[4]; };                 // the rows have the alignment of an element
    // the rows of the steps from t_first on: rows in front of the path read its zero row; letters beyond the row meet adjoints
    // that are zero
    auto step_row = [&](int64_t t_first) {
        const int64_t t = t_first - x16 < 0 ? int64_t(-1) : t_first - x16;
        return zbase + t * d;
    };
    T pz_shared[M - 1], pz_ahead[M - 1];                // the shared prefix letters: lane s holds those of step t_first - s
    auto all_red = [&](int64_t t_first) {
        const T* zt = step_row(t_first);
#pragma unroll
        for (int l = 0; l < M - 1; ++l) pz_ahead[l] = zt[tl.pu[l]];
        const Quad* zp = reinterpret_cast<const Quad*>(zt + a0 + 16 * g16);
        f32x4 c[4][2];
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
        Quad zq[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) zq[k] = zp[k];
#pragma unroll
        for (int k = 0; k < 16; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                c[i][k >> 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(zq[k >> 2].v[k & 3], gp[i][k], c[i][k >> 3], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) mine[(4 * g16 + r) * kMxStride + 16 * i + x16] = c[i][0][r] + c[i][1][r];
    };
    if constexpr (kAhead) all_red(L - 1);
    int turn = 0;                                       // which of the two buffers is `mine`
    [[maybe_unused]] Quad zq[4];                        // the next steps' increments, left operand of red
    [[maybe_unused]] auto fetch_rows = [&](int64_t t_first) {
        const Quad* zp = reinterpret_cast<const Quad*>(step_row(t_first) + a0 + 16 * g16);
#pragma unroll
        for (int k = 0; k < 4; ++k) zq[k] = zp[k];
    };
    if constexpr (kAhead)
        if (L > kMxSteps) fetch_rows(L - 1 - kMxSteps);
    for (int64_t t_first = L - 1; t_first >= 0; t_first -= kMxSteps) {
        const int n = t_first + 1 < kMxSteps ? int(t_first + 1) : kMxSteps;
        if constexpr (!kAhead) all_red(t_first);
#pragma unroll
        for (int l = 0; l < M - 1; ++l) pz_shared[l] = pz_ahead[l];
        [[maybe_unused]] const T* zt_ahead = step_row(t_first - kMxSteps);
        // four steps; PART >= 0: sixteen prefixes' part of the next steps' red, a product between the pieces of a step
        auto group = [&](int s0, auto part) {
            constexpr int PART = decltype(part)::value;
            constexpr bool AHEAD = PART >= 0;
            constexpr int I = AHEAD ? PART : 0;
            T zl[kMxGroup], red[kMxGroup], dcs[M - 1][kMxGroup];
            [[maybe_unused]] f32x4 c0 = f32x4{0.f, 0.f, 0.f, 0.f}, c1 = c0;
            if constexpr (PART == 3) {
#pragma unroll
                for (int l = 0; l < M - 1; ++l) pz_ahead[l] = zt_ahead[tl.pu[l]];
            }
            auto product = [&](int k) {
                if constexpr (AHEAD) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (k < 8) c0 = __builtin_amdgcn_mfma_f32_16x16x4f32(zq[k >> 2].v[k & 3], gp[I][k], c0, 0, 0, 0);
                    else c1 = __builtin_amdgcn_mfma_f32_16x16x4f32(zq[k >> 2].v[k & 3], gp[I][k], c1, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
#pragma unroll
            for (int k = 0; k < kMxGroup; ++k) {
                zl[k] = zl_next[k];
                red[k] = mine[(s0 + k) * kMxStride + lane];
            }
            fetch_last();
#pragma unroll
            for (int k = 0; k < kMxGroup; ++k) {
#pragma unroll
                for (int l = 0; l < M - 1; ++l) in.pz[l] = lane_value(pz_shared[l], s0 + k);
                in.pz[M - 1] = zl[k];
                in.zs[0] = red[k];
                typename Tr::Chain unmul;
                product(4 * k);
                S.template fwd_step<AllLetters, true>(in, &unmul);
                product(4 * k + 1);
                T u;
                if constexpr (Tr::kLockstep) {
                    typename Tr::Chain ch;
                    S.template chain_all<false>(in, ch, &unmul);
                    u = ch.u[N][M - 1];
                } else {
                    T uu[M];
                    S.template chain_u<N, M>(in, uu);
                    u = uu[M - 1];
                }
                mine[(s0 + k) * kMxStride + lane] = u;
                typename Ad::DInc dz;
                dz.dj[0] = T(0);
                dz.da[0] = T(0);
#pragma unroll
                for (int l = 0; l < M; ++l) dz.dc[l] = T(0);
                product(4 * k + 2);
                A.template pullback<-1, AllLetters>(S, in, dz, Tr::kLockstep ? &unmul : nullptr);
                product(4 * k + 3);
                mine_c[(s0 + k) * kMxStride + lane] = dz.dc[M - 1];
#pragma unroll
                for (int l = 0; l < M - 1; ++l) dcs[l][k] = dz.dc[l];
            }
            // the shared prefix letters: the sums of four steps over the wave end in one row of 16 lanes each
            T piece = T(0);
            int letter = tl.pu[0];
#pragma unroll
            for (int l = 0; l < M - 1; ++l) {
                const T v = row_sum_rows(quarter_sums(half_sums(dcs[l][0], dcs[l][2]), half_sums(dcs[l][1], dcs[l][3])));
                piece = x16 == l ? v : piece;
                letter = x16 == l ? tl.pu[l] : letter;
            }
            if (x16 < M - 1) lds_add_shared(&tile[(s0 + g16) * d + letter], piece);
            if constexpr (AHEAD) {
#pragma unroll
                for (int r = 0; r < 4; ++r) mine_next[(4 * g16 + r) * kMxStride + 16 * I + x16] = c0[r] + c1[r];
            }
        };
        bool ahead = false;
        if constexpr (kAhead) {
            ahead = t_first >= kMxSteps;
            if (ahead) {
                static_for<0, 3>([&](auto part) { group(decltype(part)::value * kMxGroup, part); });
                if (t_first >= 2 * kMxSteps) fetch_rows(t_first - 2 * kMxSteps);
            }
        }
        if (!ahead)
            for (int s0 = 0; s0 < n; s0 += kMxGroup) group(s0, IntC<-1>{});
        {
            f32x4 c[4][2];
#pragma unroll
            for (int i = 0; i < 8; ++i) c[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
            f32x4 uq[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) uq[k] = *reinterpret_cast<const f32x4*>(mine + x16 * kMxStride + 16 * g16 + 4 * k);
#pragma unroll
            for (int k = 0; k < 16; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    c[i][k >> 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(uq[k >> 2][k & 3], gt[i][k], c[i][k >> 3], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) mine[(4 * g16 + r) * kMxStride + 16 * i + x16] = c[i][0][r] + c[i][1][r];
        }
        __syncthreads();
        double* out = dzinc + (b * L + t_first) * d;
        // A wave takes whole steps, its lanes the letters: no division per element, and which waves' tiles hold a letter
        // is found once for all of its steps (16 paths of 200 steps, 64 channels, degree 4: the training call 5.67 ms
        // with the elements of all steps dealt out one by one, 5.44 so).
        for (int a = lane; a < d; a += kWave) {
#pragma unroll 4
            for (int s = wib; s < n; s += W) {
                T v = tile[s * d + a];
                tile[s * d + a] = T(0);
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    const T* wr = mx_lds + k * kMxWaveWords + s * kMxStride;
                    const unsigned ia = unsigned(a - wave_a0[k]), il = unsigned(a - wave_l0[k]);
                    if (ia < unsigned(kWave)) v += wr[turn * kMxBuf + ia];
                    if (il < unsigned(kWave)) v += wr[2 * kMxBuf + il];
                }
                dev_add(&out[a - int64_t(s) * d], double(v));       // step s lies s gradient rows before t_first
            }
        }
        __syncthreads();
        if constexpr (kAhead) {
            T* const other = mine;
            mine = mine_next;
            mine_next = other;
            turn ^= 1;
        }
    }
}

template <int N>
static hipError_t launch_fwd_n(const FwdParams& p)
{
    const int nblk = (p.d + kWave - 1) / kWave;
    int64_t rows = 1;
    for (int i = 0; i < N - 2; ++i) rows *= p.d;
    const int64_t waves = p.batch * rows * nblk * nblk;
    const int64_t blocks = (waves + kWavesPerBlock - 1) / kWavesPerBlock;
    if (blocks < 1 || blocks > kMaxGridX) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((rows_fwd_mfma_kernel<N>), dim3(unsigned(blocks)), dim3(kBlock), 0, p.stream,
                       static_cast<const float*>(p.inc), static_cast<float*>(p.out), p.batch, p.L, p.d, p.out_stride, p.scalar, rows,
                       nblk, nblk, p.nonfinite);
    return hipGetLastError();
}

hipError_t launch_rows_fwd_mfma(const FwdParams& p, int degree)
{
    if (p.nseg != 1 || p.from_points || p.d < kMxMinDim || p.d > kMxMaxDim) return hipErrorInvalidConfiguration;
    switch (degree) {
        case 3: return launch_fwd_n<3>(p);
        case 4: return launch_fwd_n<4>(p);
        case 5: return launch_fwd_n<5>(p);
        case 6: return launch_fwd_n<6>(p);
        case 7: return launch_fwd_n<7>(p);
        default: return hipErrorInvalidConfiguration;
    }
}

template <int N>
static hipError_t launch_bwd_n(const BwdParams& p)
{
    constexpr int W = kMxWaves;
    const int nblk = (p.d + kWave - 1) / kWave;
    int64_t rows = 1;
    for (int i = 0; i < N - 2; ++i) rows *= p.d;
    const int64_t blocks_per_path = (rows * nblk * nblk + W - 1) / W;
    const int64_t blocks = p.batch * blocks_per_path;
    if (blocks < 1 || blocks > kMaxGridX) return hipErrorInvalidConfiguration;
    const size_t lds = (size_t(W) * kMxWaveWords + size_t(kMxSteps) * p.d) * sizeof(float);
    const hipError_t e = allow_lds(rows_bwd_mfma_kernel<N>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((rows_bwd_mfma_kernel<N>), dim3(unsigned(blocks)), dim3(W * kWave), lds, p.stream,
                       static_cast<const float*>(p.inc), static_cast<const float*>(p.sig), static_cast<const float*>(p.gsig),
                       static_cast<double*>(p.dzinc), p.L, p.d, p.sig_stride, p.scalar, rows, nblk, nblk, blocks_per_path);
    return hipGetLastError();
}

bool rows_bwd_mfma_supported(uint64_t d) { return d >= uint64_t(kMxMinDim) && d <= uint64_t(kMxBwdMaxDim); }

hipError_t launch_rows_bwd_mfma(const BwdParams& p, int degree)
{
    if (p.nseg != 1 || p.from_points || !rows_bwd_mfma_supported(uint64_t(p.d))) return hipErrorInvalidConfiguration;
    switch (degree) {
        case 3: return launch_bwd_n<3>(p);
        case 4: return launch_bwd_n<4>(p);
        case 5: return launch_bwd_n<5>(p);
        case 6: return launch_bwd_n<6>(p);
        default: return hipErrorInvalidConfiguration;
    }
}

}  // namespace sigamd
