// Adjoint of the Chen product, both factors in one pass over dC (siglib/cpsig/cp_sig_combine.h:126-176):
//
//   dA_k[u] = dC_k[u] + sum_{m >= 1} sum_{v in d^m} dC_{k+m}[u v] * B_m[v]
//   dB_t[w] = dC_t[w] + sum_{k >= 1} sum_{u in d^k} dC_{k+t}[u w] * A_k[u]
//
// The kernels of sig_chen_stream.h read the top level of dC once for each factor: of the four signature rows that the adjoint moves
// beside the lower levels, one.  Here a word of the top level is x y s, |x| = |y| = 1, |s| = Q = degree - 2, and a block takes, of
// one row, the words whose s begins with one of R letters.  It walks them in memory order, a letter x at a time; a thread owns
// one s, and with it
//   * the sums over x and over x y, whose weights A_1[x], A_2[x y] are uniform (dB_{Q+1}[y s], dB_Q[s]), and its part of dA_1[x];
//   * one word x y s', s' a letter shorter (as many as there are s), once the block has laid the top words of an x in LDS:
//     it reads its D children, sums them against B_1 .. B_Q (one value for each ancestor, which then meet along s') and adds
//     them, times A_{2+j}[x y s'_1..j], to what later becomes dB_t, t < Q.
// Level degree - 1 goes along: a thread's word x y s' is one of its entries.  The levels below come from the item-per-word
// kernels on the signature truncated at Q, launched first; this kernel adds to them at the end, atomically, since the blocks of a
// row meet there.
//
// Partial sums that meet are added up in double precision, and a thread sums the words of an x by themselves: in single precision, one after the other,
// the sums of D * D words cost accuracy (relative to 64 bits, general kernels / one chain / now: 13 channels, degree 4, dB_2 1.0e-7 / 2.2e-7 / 1.0e-7; 16, 5,
// dA_2 1.0e-7 / 1.4e-7 / 1.1e-7; with the items of the truncated problem 3, 8, dA_1 1.0e-7 / 1.8e-7 / 1.0e-7), which takes no time that could be
// measured (74 calls of all plans: 1.006, two runs of the same 1.005).
#pragma once
#include "sig_barrier.h"
#include "sig_chen_stream.h"
#include "sig_kernels.h"

namespace sigamd {

constexpr int kBothNever = 0x7fffffff;

// FROM64, FROM32: rows of a call from which the kernel is the sooner one, in double and in single precision
template <int D_, int Q_, int R_, int PER_SIMD_, int FROM64_, int FROM32_>
struct BothPlan {
    static constexpr int D = D_, Q = Q_, R = R_, N = Q + 2, PER_SIMD = PER_SIMD_, FROM64 = FROM64_, FROM32 = FROM32_;
    static constexpr int PARTS = D / R;                                     // blocks of a row
    static constexpr int S = int(ipow64(D, Q)), SP = S / D;                 // words s, s'
    static constexpr int OWN = S / PARTS, OWNP = SP / PARTS;                // a block's
    static constexpr int THREADS = (OWN + kWave - 1) / kWave * kWave;
    static_assert(Q >= 2 && D % R == 0 && THREADS <= 1024, "a thread owns one s");
    static constexpr int lo(int t) { return int((ipow64(D, t) - D) / (D - 1)); }    // start of level t in a scalar-free row
    static constexpr int LOW = lo(Q + 1);                                   // coefficients of the levels 1 .. Q
    static constexpr int PAD = D % 2 == 0 ? 1 : 0;                          // runs of D children start in different banks
    static constexpr int CHILDREN = OWNP * (D + PAD);
    static constexpr int TILE = D * CHILDREN > lo(Q) ? D * CHILDREN : lo(Q);
    static constexpr int SUMS = (Q - 1) * OWN;                              // ancestors' sums of one x, and once summed over a letter
    static constexpr size_t lds_entries() { return size_t(TILE) + 2 * LOW + SUMS + SUMS / R; }      // beside a sum per wave
};

template <typename T, typename P>
__global__ __launch_bounds__(P::THREADS) __attribute__((amdgpu_waves_per_eu(P::PER_SIMD))) void chen_adjoint_both_kernel(
    const T* __restrict__ dC, T* __restrict__ dA, T* __restrict__ dB, const T* __restrict__ A, const T* __restrict__ B, int64_t items, int64_t stride,
    int off)
{
    constexpr int D = P::D, Q = P::Q, N = P::N, R = P::R, S = P::S, SP = P::SP, OWN = P::OWN, OWNP = P::OWNP;
    extern __shared__ __align__(16) unsigned char both_lds[];
    T* tile = reinterpret_cast<T*>(both_lds);       // [y][own s'][D + PAD]; at the end the sums for dB below level Q
    T* Bl = tile + P::TILE;                         // levels 1 .. Q of B
    T* Ra = Bl + P::LOW;                            // sums for dA, the block's words of a level end to end
    T* sums = Ra + P::LOW;                          // [m - 2][y][own s']
    T* next = sums + P::SUMS;                       // the same with one letter summed over
    __shared__ double part_sum[P::THREADS / kWave];
    const int own_tid = threadIdx.x, lane = own_tid & (kWave - 1);
    const bool live = own_tid < OWN;
    const int mine = live ? own_tid : OWN - 1;      // idle threads do the last one's work again, but for its sums
    // the length of s, hidden from the compiler: multiples of it stay in the scalar part of an address
    int rs = S;
    asm volatile("" : "+s"(rs));
    for (int64_t item = xcd_block(); item < items; item += gridDim.x) {
        const int64_t b = item / P::PARTS;
        const int part = int(item % P::PARTS);
        const T* g = dC + b * stride + off;
        const T* fa = A + b * stride + off;
        const T* fb = B + b * stride + off;
        T* oa = dA + b * stride + off;
        T* ob = dB + b * stride + off;
        if (off && part == 0 && own_tid == 0) { oa[-1] = T(0); ob[-1] = T(0); }
        for (int i = own_tid; i < P::LOW; i += P::THREADS) Bl[i] = fb[i];
        T sum_x[D], sum_xy = T(0), item_x = T(0), low[Q][D], item_low[Q];
#pragma unroll
        for (int y = 0; y < D; ++y) sum_x[y] = T(0);
#pragma unroll
        for (int j = 0; j < Q; ++j) {
            item_low[j] = T(0);
#pragma unroll
            for (int z = 0; z < D; ++z) low[j][z] = T(0);
        }
#pragma unroll 1
        for (int x = 0; x < D; ++x) {
            // indexes are formed again for every x, and B's level Q + 1 is read again: kept, they would fill the registers
            int again = 0, own = mine, tid = own_tid;
            asm volatile("" : "+s"(again), "+v"(own), "+v"(tid));
            const int s = part * OWN + own;
            const uint32_t so = uint32_t(s) * uint32_t(sizeof(T));
            const int yi = own / OWNP, sp = part * OWNP + own % OWNP;       // the thread's word x y s'
            const uint32_t io = uint32_t(yi * SP + sp) * uint32_t(sizeof(T));
            const T a1 = fa[x];
            T k1 = T(0), xy = T(0), e[D], by[D];
#pragma unroll
            for (int y = 0; y < D; ++y) {
                e[y] = load_at(g + P::lo(N) + x * (D * rs) + y * rs, so);
                by[y] = load_at(fb + again + P::lo(Q + 1) + y * rs, so);
            }
            T* ta = oa + P::lo(N) + x * (D * rs);
            T* tb = ob + P::lo(N) + x * (D * rs);
#pragma unroll
            for (int y = 0; y < D; ++y) {
                tile[y * P::CHILDREN + own + P::PAD * (own / D)] = e[y];
                store_at(ta + y * rs, so, e[y]);
                store_at(tb + y * rs, so, e[y]);
                sum_x[y] = fmadd(a1, e[y], sum_x[y]);
                xy = fmadd(fa[D + x * D + y], e[y], xy);
                k1 = fmadd(e[y], by[y], k1);
            }
            sum_xy += xy;
            const T g1 = load_at(g + P::lo(N - 1) + x * rs, io);
            T w[Q];
            w[0] = load_at(fa + D + x * D, uint32_t(yi) * uint32_t(sizeof(T)));
            static_for<1, Q - 1>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                w[j] = load_at(fa + P::lo(2 + j) + x * int(ipow64(D, 1 + j)),
                               uint32_t((yi * SP + sp) / int(ipow64(D, Q - 1 - j))) * uint32_t(sizeof(T)));
            });
            lds_barrier();
            const T* Bx = opaque_lds(Bl);
            const T* children = tile + own * (D + P::PAD);
            T sum_1 = g1, u[Q + 1];
            static_for<2, Q>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                u[m] = g1 * Bx[P::lo(m - 1) + sp % int(ipow64(D, m - 1))];
            });
#pragma unroll
            for (int z = 0; z < D; ++z) {
                const T c = children[z];
                sum_1 = fmadd(c, Bx[z], sum_1);
                static_for<2, Q>([&](auto mc) {
                    constexpr int m = decltype(mc)::value;
                    u[m] = fmadd(c, Bx[P::lo(m) + sp % int(ipow64(D, m - 1)) * D + z], u[m]);
                });
#pragma unroll
                for (int j = 1; j < Q; ++j) low[j][z] = fmadd(w[j], c, low[j][z]);
                if (z % 4 == 3) __builtin_amdgcn_sched_barrier(0);      // few children at a time
            }
            store_at(oa + P::lo(N - 1) + x * rs, io, sum_1);
#pragma unroll
            for (int m = 2; m <= Q; ++m) sums[(m - 2) * OWN + own] = u[m];
            item_x = fmadd(a1, g1, item_x);
#pragma unroll
            for (int j = 0; j + 1 < Q; ++j) item_low[j] = fmadd(w[j], g1, item_low[j]);
            k1 = fmadd(g1, Bx[P::lo(Q) + yi * SP + sp], k1);
            const double block_k1 = wave_sum(live ? double(k1) : 0.0);
            if (lane == 0) part_sum[own_tid / kWave] = block_k1;
            lds_barrier();
            if (own_tid == 0) {
                double v = part_sum[0];
                for (int i = 1; i < P::THREADS / kWave; ++i) v += part_sum[i];
                Ra[x] = T(v);
            }
            // the sums over the last letter, the last two, ...: level N - m takes m - 1 of these steps
            static_for<2, Q>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                constexpr int fan = k == Q ? R : D;             // the first letter of s' is one of the block's
                constexpr int in = OWN / int(ipow64(D, k - 2)), out = in / fan;
                const T* from = (k & 1) ? next : sums;
                T* to = (k & 1) ? sums : next;
                for (int i = tid; i < (Q - k + 1) * out; i += P::THREADS) {
                    const int m = k + i / out, o = i % out;
                    const T* v = from + (m - (k == 2 ? 2 : k - 1)) * in + o * fan;
                    double t = double(v[0]);
#pragma unroll
                    for (int z = 1; z < fan; ++z) t += double(v[z]);
                    if (m == k) Ra[P::lo(N - k) + x * out + o] = T(t);     // level N - k is complete
                    else to[(m - k) * out + o] = T(t);
                }
                lds_barrier();
            });
        }
        // what meets in the lower levels
        const int s = part * OWN + mine, yi = mine / OWNP, sp = part * OWNP + mine % OWNP;
        const uint32_t so = uint32_t(s) * uint32_t(sizeof(T));
        for (int i = own_tid; i < D + D * D; i += P::THREADS) dev_add(oa + i, Ra[i]);
        static_for<1, Q - 2>([&](auto jc) {
            constexpr int j = decltype(jc)::value, run = R * int(ipow64(D, j - 1));     // words x y s'_1..j: runs of a block's
            for (int i = own_tid; i < D * D * run; i += P::THREADS)
                dev_add(oa + P::lo(2 + j) + i / run * int(ipow64(D, j)) + part * run + i % run, Ra[P::lo(2 + j) + i]);
        });
        for (int i = own_tid; i < P::lo(Q); i += P::THREADS) tile[i] = T(0);
#pragma unroll
        for (int y = 0; y < D; ++y) store_at(ob + P::lo(N - 1) + y * rs, so, load_at(g + P::lo(N - 1) + y * rs, so) + sum_x[y]);
        if (live) {
            dev_add(ob + P::lo(Q) + s, sum_xy);
            dev_add(ob + P::lo(Q) + yi * SP + sp, item_x);
        }
        lds_barrier();
        if (live) {
            static_for<1, Q - 1>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                T* at = tile + P::lo(Q - j) + sp % int(ipow64(D, Q - 1 - j)) * D;
#pragma unroll
                for (int z = 0; z < D; ++z) lds_add_shared(at + z, low[j][z]);
            });
            static_for<0, Q - 2>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                lds_add_shared(tile + P::lo(Q - 1 - j) + sp % int(ipow64(D, Q - 1 - j)), item_low[j]);
            });
        }
        lds_barrier();
        for (int i = own_tid; i < P::lo(Q); i += P::THREADS) dev_add(ob + i, tile[i]);
        lds_barrier();
    }
}

}  // namespace sigamd
