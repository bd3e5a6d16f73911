// Adjoint of the Chen product: kernels and their launcher, shared by sig_combine_backprop, sig_join_backprop, the
// tensor logarithm's backward pass and the time-split signature backward.
#include "sig_chen_adjoint.h"

#include <atomic>
#include <type_traits>

#include "sig_kernels.h"
#include "sig_chen_both.h"
#include "sig_chen_stream.h"

namespace sigamd {

// four consecutive elements with the alignment of one
template <typename T>
struct alignas(sizeof(T)) Quad {
    T v[4];
};
constexpr int kCombChunk = 256;
template <typename I>
struct CombBwdPlan {
    int degree;
    I items;                            // work items of one family
    I lo[kCombMaxLevels + 2];           // lo[t]: start of level t in a scalar-free row, t = 1 .. degree + 1
    I item_start[kCombMaxLevels + 2];   // first work item of level t
    I parts[kCombMaxLevels + 2];        // parts per word of level t (>= 1)
    I init_len;                         // coefficients (a prefix of the row) whose levels have several parts
};

template <typename I>
static CombBwdPlan<I> make_comb_plan(uint64_t d, uint64_t degree)
{
    CombBwdPlan<I> p{};
    p.degree = int(degree);
    uint64_t lo = 0, sz = d;
    for (uint64_t t = 1; t <= degree + 1; ++t) {
        p.lo[t] = I(lo);
        lo += sz;
        if (t <= degree) sz *= d;
    }
    uint64_t items = 0;
    p.init_len = 0;
    for (uint64_t t = 1; t <= degree; ++t) {
        const uint64_t s_t = uint64_t(p.lo[degree - t + 1]);          // d + .. + d^(degree - t)
        const uint64_t parts = s_t == 0 ? 1 : (s_t + kCombChunk - 1) / kCombChunk;
        p.item_start[t] = I(items);
        p.parts[t] = I(parts);
        items += parts * (uint64_t(p.lo[t + 1]) - uint64_t(p.lo[t]));
        if (parts > 1) p.init_len = p.lo[t + 1];
    }
    p.item_start[degree + 1] = I(items);
    p.items = I(items);
    return p;
}

template <typename T, typename I>
__global__ __launch_bounds__(kBlock) void sig_combine_bwd_init_kernel(
    const T* __restrict__ dC, T* __restrict__ dA, T* __restrict__ dB, int64_t batch, I init_len, int64_t stride, int off,
    int identity, int64_t dc_share, int64_t dc_stride, int dc_off, int families, int only_b)
{
    for (int64_t b = xcd_block_2d().y; b < batch; b += gridDim.y) {
        for (I r = I(xcd_block_2d().x) * kBlock + threadIdx.x; r < init_len; r += I(gridDim.x) * kBlock) {
            const T v = identity ? dC[(b / dc_share) * dc_stride + dc_off + r] : T(0);
            if (!only_b) dA[b * stride + off + r] = (identity & 1) ? v : T(0);
            if (families > 1 || only_b) dB[b * stride + off + r] = (identity & 2) ? v : T(0);
        }
    }
}

// Acc: what an item sums in
template <typename T, typename I, typename Acc>
__global__ __launch_bounds__(kBlock) void sig_combine_bwd_kernel(
    const T* __restrict__ dC, T* __restrict__ dA, T* __restrict__ dB, const T* __restrict__ A,
    const T* __restrict__ B, int64_t batch, CombBwdPlan<I> plan, int64_t stride, int off, int identity,
    int64_t dc_share, int64_t dc_stride, int dc_off, int families, int only_b)
{
    const int N = plan.degree;
    for (int64_t b = xcd_block_2d().y; b < batch; b += gridDim.y) {
        const T* g = dC + (b / dc_share) * dc_stride + dc_off;
        for (I it = I(xcd_block_2d().x) * kBlock + threadIdx.x; it < I(families) * plan.items; it += I(gridDim.x) * kBlock) {
            const bool fam_b = only_b || it >= plan.items;
            const I i2 = it >= plan.items ? it - plan.items : it;
            int t = 1;
            while (t < N && i2 >= plan.item_start[t + 1]) ++t;
            const I sz_t = plan.lo[t + 1] - plan.lo[t];
            const I local = i2 - plan.item_start[t];
            const I q = local / sz_t;
            const I w = local - q * sz_t;
            const I s_t = plan.lo[N - t + 1];
            const I x0 = q * kCombChunk;
            const I x1 = x0 + kCombChunk < s_t ? x0 + kCombChunk : s_t;
            const T* other = (fam_b ? A : B) + b * stride + off;      // the factor the sum runs over
            Acc s0 = Acc(0), s1 = Acc(0), s2 = Acc(0), s3 = Acc(0);
            for (int m = 1; m <= N - t; ++m) {
                const I seg0 = plan.lo[m] > x0 ? plan.lo[m] : x0;
                const I seg1 = plan.lo[m + 1] < x1 ? plan.lo[m + 1] : x1;
                if (seg0 >= seg1) continue;
                const T* up = g + plan.lo[t + m];                     // level t + m of dC
                if (!fam_b) {
                    const T* blockp = up + w * (plan.lo[m + 1] - plan.lo[m]) - plan.lo[m];    // words w v
                    I x = seg0;
                    for (; x + 4 <= seg1; x += 4) {      // all loads are issued before the first product needs one
                        // a lane walks a block of its own, so every load costs it a cache access of its own: take the
                        // four consecutive entries in wide loads (element alignment is all that is known)
                        const Quad<T> gq = *reinterpret_cast<const Quad<T>*>(blockp + x);
                        const Quad<T> oq = *reinterpret_cast<const Quad<T>*>(other + x);
                        s0 = fmadd(Acc(gq.v[0]), Acc(oq.v[0]), s0);
                        s1 = fmadd(Acc(gq.v[1]), Acc(oq.v[1]), s1);
                        s2 = fmadd(Acc(gq.v[2]), Acc(oq.v[2]), s2);
                        s3 = fmadd(Acc(gq.v[3]), Acc(oq.v[3]), s3);
                    }
                    for (; x < seg1; ++x) s0 = fmadd(Acc(blockp[x]), Acc(other[x]), s0);
                } else {
                    const T* strided = up + w;                         // words u w: index u * d^t + w
                    I x = seg0;
                    for (; x + 4 <= seg1; x += 4) {
                        const T* sp = strided + (x - plan.lo[m]) * sz_t;
                        const T g0 = sp[0], g1 = sp[sz_t], g2 = sp[2 * sz_t], g3 = sp[3 * sz_t];
                        const Quad<T> oq = *reinterpret_cast<const Quad<T>*>(other + x);      // the same four for the whole wave
                        s0 = fmadd(Acc(g0), Acc(oq.v[0]), s0);
                        s1 = fmadd(Acc(g1), Acc(oq.v[1]), s1);
                        s2 = fmadd(Acc(g2), Acc(oq.v[2]), s2);
                        s3 = fmadd(Acc(g3), Acc(oq.v[3]), s3);
                    }
                    for (; x < seg1; ++x) s0 = fmadd(Acc(strided[(x - plan.lo[m]) * sz_t]), Acc(other[x]), s0);
                }
            }
            const I r = plan.lo[t] + w;
            T* dst = (fam_b ? dB : dA) + b * stride + off + r;
            const Acc sum = (s0 + s1) + (s2 + s3);
            if (plan.parts[t] == 1) *dst = T(((identity >> int(fam_b)) & 1 ? Acc(g[r]) : Acc(0)) + sum);
            else dev_add(dst, T(sum));
            if (off && it == 0) {
                if (!only_b) dA[b * stride] = T(0);
                if (families > 1 || only_b) dB[b * stride] = T(0);
            }
        }
    }
}

// test hook (defined in sig_api.hip): 0 = streaming kernels for rows of at least kStreamMinCoef coefficients,
// 1 = streaming kernels wherever they apply, 2 = item-per-word kernels only
extern std::atomic<int> g_chen_adjoint_mode;
constexpr uint64_t kStreamMinCoef = 4096;
constexpr uint64_t kStreamLdsEntries = 6144;      // 48 KB of float64

// the item-per-word kernels on the signature truncated at `degree` (rows keep their stride): both factors, or one
template <typename T, typename Acc = T>
static void launch_combine_bwd_items(const T* dC, T* dA, T* dB, const T* A, const T* B, uint64_t batch, uint64_t dimension,
                                     uint64_t degree, const SigShape& s, hipStream_t stream, int identity,
                                     const SharedRows& dc, int families, int only_b)
{
    launch_indexed(3 * s.n_coef + 1024, 1, batch, [&](auto ix, dim3) {      // 2 * items <= 2 n (1 + degree / kCombChunk)
        using I = decltype(ix);
        const CombBwdPlan<I> plan = make_comb_plan<I>(dimension, degree);
        if (plan.init_len > 0)
            launch_indexed(0, uint64_t(plan.init_len), batch, [&](auto, dim3 grid) {
                hipLaunchKernelGGL((sig_combine_bwd_init_kernel<T, I>), grid, dim3(kBlock), 0, stream, dC, dA, dB,
                                   int64_t(batch), plan.init_len, int64_t(s.stride), s.off, identity, dc.share, dc.stride,
                                   dc.off, families, only_b);
            });
        launch_indexed(0, uint64_t(families) * uint64_t(plan.items), batch, [&](auto, dim3 grid) {
            hipLaunchKernelGGL((sig_combine_bwd_kernel<T, I, Acc>), grid, dim3(kBlock), 0, stream, dC, dA, dB, A, B, int64_t(batch),
                               plan, int64_t(s.stride), s.off, identity, dc.share, dc.stride, dc.off, families, only_b);
        });
    });
}

// LDS of the right factor's kernel when it folds exp(z): one slot per lane and letter
template <typename T>
static bool right_fold_fits(uint64_t dimension)
{
    return dimension * uint64_t(kBlock) * sizeof(T) <= uint64_t(64) << 10;
}

template <typename T, int QL = 0, int REL = 1>
static void launch_right_stream(const RightPlan& rp, const T* dC, T* dB, const T* A, T* sum_rows, uint64_t batch, const SigShape& s,
                                hipStream_t stream, int identity, const SharedRows& dc, const ExpFold<T>* fold)
{
    if constexpr (QL <= kRightMaxLow && REL <= kRightMaxRel) {
        if (rp.qe - 1 != QL) return launch_right_stream<T, QL + 1, REL>(rp, dC, dB, A, sum_rows, batch, s, stream, identity, dc, fold);
        if (rp.rel != REL) return launch_right_stream<T, QL, REL + 1>(rp, dC, dB, A, sum_rows, batch, s, stream, identity, dc, fold);
        const uint64_t waves = (uint64_t(rp.words) + kWave - 1) / kWave;
        const dim3 grid{unsigned((waves + kWavesPerBlock - 1) / kWavesPerBlock), unsigned(std::min<uint64_t>(batch, 65535)), 1};
        FoldScale<T> fs{};
        if (fold) {
            double fact = 1.0;
            for (int t = 1; t <= rp.qe; ++t) fact *= double(t);
            for (int D = 0; D <= REL; ++D) {
                if (D) fact *= double(rp.qe + D);
                fs.inv_level[D] = T(1.0 / double(rp.qe + D));
                fs.inv_fact[D] = T(1.0 / fact);
            }
            hipLaunchKernelGGL((chen_adjoint_right_kernel<T, QL, REL, true>), grid, dim3(kBlock),
                               size_t(rp.d) * kBlock * sizeof(T), stream, dC, dB, A, int64_t(batch), rp, int64_t(s.stride), s.off,
                               identity, dc.share, dc.stride, dc.off, fold->z, fold->dz, fs, sum_rows);
        } else {
            hipLaunchKernelGGL((chen_adjoint_right_kernel<T, QL, REL, false>), grid, dim3(kBlock), 0, stream, dC, dB, A,
                               int64_t(batch), rp, int64_t(s.stride), s.off, identity, dc.share, dc.stride, dc.off,
                               (const T*)nullptr, (T*)nullptr, fs, sum_rows);
        }
    }
}

template <typename T, typename P>
static void launch_both(const T* dC, T* dA, T* dB, const T* A, const T* B, uint64_t batch, const SigShape& s, hipStream_t stream)
{
    constexpr size_t lds = P::lds_entries() * sizeof(T);
    static_assert(lds + P::THREADS / kWave * sizeof(double) <= size_t(160) * 1024, "a row's pieces fit a compute unit");
    if (lds > 64 * 1024)
        SIG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(chen_adjoint_both_kernel<T, P>), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    const uint64_t most = ((uint64_t(1) << 32) - 1) / P::THREADS;      // a launch numbers its threads with 32 bits; further items in the same blocks
    hipLaunchKernelGGL((chen_adjoint_both_kernel<T, P>), dim3(unsigned(std::min<uint64_t>(batch * P::PARTS, most))), dim3(P::THREADS), lds, stream, dC, dA,
                       dB, A, B, int64_t(batch) * P::PARTS, int64_t(s.stride), s.off);
}

template <typename... P>
struct BothPlans {};
template <typename Go, typename... P>
static bool any_of_plans(Go&& go, BothPlans<P...>)
{
    return (go(P()) || ...);
}

// Both factors in one pass over dC, where there is such a kernel.  Blocks of a row (D / R), registers (waves a SIMD) and, per precision, the rows from
// which it takes over were measured for each against the general kernels with the longer words that those take where rows are few
// (right_word_length).  us, general / one pass, double: 1080 rows of 10 channels, degree 5: 1050 / 850; 1806 of 9, 5: 1300 / 810; 4096 of 6, 5: 670 / 320, of
// 5, 6: 1030 / 680, of 3, 7: 620 / 220; 298 of 13, 5: 2990 / 930; 512 of 22, 4: 1542 / 748; single row of 6, 6: 155 / 54.  Where a row's few blocks leave
// the chip idle: 1 row of 20, 4: 63 / 141, 32: 94 / 147, 80: 188 / 200, 96: 213 / 204; 24 of 22, 4: 132 / 167, 28: 179 / 167; 1 of 8, 4: 35 / 43, 512:
// 51 / 50.  Single precision moves half as much and gains sooner: 1 row of 17, 4: 110 / 118 and 106 / 84; 48 of 20, 4: 134 / 148 and 101 / 100.
// 16 channels, degree 5, has one word a thread in 16 blocks of a row, each with 113 KB of LDS in double precision: 123 / 183, 128 rows 1289 / 1567.
// The one pass rounds less at degree 5 (1 row, double, right factor: 14, 5: 3.0e-16 / 1.6e-16; 16, 5: 3.6 / 1.6; degree 4 1.6-2.5 / 1.3-1.7), so no line was
// raised for less than a tenth (1 row of 14, 5: 94 / 101; 256 rows of 4, 5, single: 31 / 30).  Without a plan: 2 channels, degree 11 (0.84 / 1.16 ms), 8, 6 (1.28 / 1.33).
template <typename T>
static bool launch_both_factors(const T* dC, T* dA, T* dB, const T* A, const T* B, uint64_t batch, uint64_t dimension, uint64_t degree,
                                const SigShape& s, hipStream_t stream, const SharedRows& dc)
{
    auto go = [&](auto plan) {
        using P = decltype(plan);
        if (dimension != uint64_t(P::D) || degree != uint64_t(P::N) || (row_forms() != 2 && batch < uint64_t(sizeof(T) == 8 ? P::FROM64 : P::FROM32))) return false;
        launch_combine_bwd_items<T, double>(dC, dA, dB, A, B, batch, dimension, uint64_t(P::Q), s, stream, 3, dc, 2, 0);
        launch_both<T, P>(dC, dA, dB, A, B, batch, s, stream);
        tl_chen_both = 1;
        return true;
    };
    return any_of_plans(go, BothPlans<BothPlan<4, 3, 4, 4, 192, 192>, BothPlan<5, 3, 5, 4, 96, 96>, BothPlan<6, 2, 6, 4, 256, 256>,
                        BothPlan<8, 2, 8, 4, 512, 400>, BothPlan<9, 2, 9, 4, 48, 48>, BothPlan<10, 2, 10, 3, 96, 96>, BothPlan<11, 2, 11, 3, 1, 1>,
                        BothPlan<12, 2, 12, 3, 1, 1>, BothPlan<13, 2, 13, 3, 1, 1>, BothPlan<14, 2, 14, 3, 160, 160>,
                        BothPlan<15, 2, 15, 2, 128, 128>, BothPlan<16, 2, 16, 2, 128, 128>, BothPlan<17, 2, 17, 2, 12, 1>,
                        BothPlan<18, 2, 9, 2, 64, 48>, BothPlan<19, 2, 19, 2, 32, 1>, BothPlan<20, 2, 10, 2, 96, 48>, BothPlan<21, 2, 7, 2, 48, 32>,
                        BothPlan<22, 2, 11, 2, 28, 20>, BothPlan<24, 2, 8, 2, 56, 28>, BothPlan<6, 3, 6, 4, 1, 1>, BothPlan<7, 3, 1, 4, 1, 1>,
                        BothPlan<8, 3, 4, 3, 1, 1>, BothPlan<9, 3, 3, 3, 1, 1>, BothPlan<10, 3, 2, 3, 1, 1>, BothPlan<11, 3, 1, 3, 1, 1>,
                        BothPlan<12, 3, 1, 3, 1, 1>, BothPlan<13, 3, 1, 2, 1, 1>, BothPlan<14, 3, 1, 2, 1, 1>, BothPlan<16, 3, 1, 2, kBothNever, 1>,
                        BothPlan<4, 4, 2, 4, 1, 1>, BothPlan<5, 4, 1, 3, 1, 1>, BothPlan<6, 4, 1, 3, 1, 1>, BothPlan<7, 4, 1, 3, 1, 1>,
                        BothPlan<3, 5, 3, 4, 64, 64>, BothPlan<4, 5, 1, 3, 1, 1>, BothPlan<3, 6, 1, 3, 1, 1>, BothPlan<2, 8, 1, 3, 1, 1>>());
}

// launches the adjoint of the Chen product on `stream`
template <typename T>
void launch_combine_bwd(const T* dC, T* dA, T* dB, const T* A, const T* B, uint64_t batch, uint64_t dimension,
                        uint64_t degree, const SigShape& s, hipStream_t stream, int identity, SharedRows dc, int families,
                        ExpFold<T>* fold)
{
    if (dc.stride < 0) { dc.stride = int64_t(s.stride); dc.off = s.off; }
    if (fold) fold->level = int(degree);
    const int ida = identity & 1, idb = (identity >> 1) & 1;
    if (degree > uint64_t(kCombMaxLevels)) throw std::runtime_error("sig_combine_backprop_cuda: degree too high");
    const int mode = g_chen_adjoint_mode;
    const bool streaming = mode != 2 && (mode == 1 || s.n_coef >= kStreamMinCoef) && dimension >= 2 && degree >= 2 &&
                           degree <= uint64_t(kStreamMaxLevels) && s.n_coef < (uint64_t(1) << 28) &&
                           !g_force_wide_index;
    tl_chen_both = 0;
    if (families == 2 && identity == 3 && !fold && row_forms() != 0 && dc.share == 1 && dc.stride == int64_t(s.stride) && dc.off == s.off &&
        launch_both_factors<T>(dC, dA, dB, A, B, batch, dimension, degree, s, stream, dc))
        return;
    LeftPlan lp;
    RowsPlan wp;
    RightPlan rp;
    const bool rows = streaming && make_rows_plan(wp, dimension, degree, kStreamLdsEntries);
    const bool left = rows || (streaming && make_left_plan(lp, dimension, degree, kStreamLdsEntries));
    const bool right = streaming && families > 1 && make_right_plan(rp, dimension, degree, batch, sizeof(T));
    if (!left && !right) {
        launch_combine_bwd_items<T>(dC, dA, dB, A, B, batch, dimension, degree, s, stream, identity, dc, families, 0);
        return;
    }
    // words shorter than the blocks' own take their low-level terms from the truncated problem first
    auto left_factor = [&] {
        if (!left) {
            launch_combine_bwd_items<T>(dC, dA, dB, A, B, batch, dimension, degree, s, stream, identity, dc, 1, 0);
        } else if (rows) {
            if (wp.np >= 2)
                launch_combine_bwd_items<T>(dC, dA, dB, A, B, batch, dimension, uint64_t(wp.np), s, stream, identity, dc, 1, 0);
            const uint64_t groups = (uint64_t(wp.units) + uint64_t(wp.upb) - 1) / uint64_t(wp.upb);
            const dim3 grid{unsigned(groups), unsigned(std::min<uint64_t>(batch, 65535)), 1};
            const size_t lds = (size_t(wp.bs) + 2 * size_t(wp.targets) + size_t(wp.img)) * sizeof(T);
            const int kt = int((wp.top + kBlock - 1) / kBlock), ks = int((wp.targets + kBlock - 1) / kBlock);
            auto go3 = [&](auto dc_, auto kt_, auto ks_) {
                hipLaunchKernelGGL((chen_adjoint_left_rows_kernel<T, decltype(dc_)::value, decltype(kt_)::value, decltype(ks_)::value>),
                                   grid, dim3(kBlock), lds, stream, dC, dA, B, int64_t(batch), wp, int64_t(s.stride), s.off, ida,
                                   dc.share, dc.stride, dc.off);
            };
            auto go2 = [&](auto dc_, auto ks_) {
                if (kt <= 2) go3(dc_, std::integral_constant<int, 2>(), ks_);
                else if (kt <= 4) go3(dc_, std::integral_constant<int, 4>(), ks_);
                else go3(dc_, std::integral_constant<int, kRowsMaxTop>(), ks_);
            };
            // owned entries per thread: more than one only for few channels (targets ~ top / (d - 1))
            auto go = [&](auto dc_) {
                constexpr int DC = decltype(dc_)::value;
                if (ks <= 1) go2(dc_, std::integral_constant<int, 1>());
                else if constexpr (DC <= 8) {
                    if (ks <= 2) go2(dc_, std::integral_constant<int, 2>());
                    else if constexpr (DC <= 4) go2(dc_, std::integral_constant<int, kRowsMaxLow>());
                    else throw std::logic_error("sig_combine_backprop_cuda: kernel plan");
                } else throw std::logic_error("sig_combine_backprop_cuda: kernel plan");
            };
            const uint64_t d = dimension;
            if (d <= 4) go(std::integral_constant<int, 4>());
            else if (d <= 8) go(std::integral_constant<int, 8>());
            else if (d <= 12) go(std::integral_constant<int, 12>());
            else if (d <= 16) go(std::integral_constant<int, 16>());
            else go(std::integral_constant<int, 32>());
        } else {
            if (lp.np >= 2)
                launch_combine_bwd_items<T>(dC, dA, dB, A, B, batch, dimension, uint64_t(lp.np), s, stream, identity, dc, 1, 0);
            const uint64_t groups = (uint64_t(lp.units) + uint64_t(lp.upb) - 1) / uint64_t(lp.upb);
            const dim3 grid{unsigned(groups), unsigned(std::min<uint64_t>(batch, 65535)), 1};
            const size_t lds = (size_t(lp.xs) + size_t(lp.bs)) * sizeof(T);
            auto go = [&](auto kx) {
                hipLaunchKernelGGL((chen_adjoint_left_kernel<T, decltype(kx)::value>), grid, dim3(kBlock), lds, stream, dC, dA, B,
                                   int64_t(batch), lp, int64_t(s.stride), s.off, ida, dc.share, dc.stride, dc.off);
            };
            const uint32_t per = (lp.xs + kBlock - 1) / kBlock;      // entries of a unit per thread
            if (per <= 4) go(std::integral_constant<int, 4>());
            else if (per <= 8) go(std::integral_constant<int, 8>());
            else if (per <= 12) go(std::integral_constant<int, 12>());
            else if (per <= 16) go(std::integral_constant<int, 16>());
            else go(std::integral_constant<int, 24>());
        }
    };
    auto right_factor = [&] {
        if (!right) {
            launch_combine_bwd_items<T>(dC, dA, dB, A, B, batch, dimension, degree, s, stream, identity, dc, 1, 1);
            return;
        }
        if (rp.qe >= 2)
            launch_combine_bwd_items<T>(dC, dA, dB, A, B, batch, dimension, uint64_t(rp.qe - 1), s, stream, identity, dc, 1, 1);
        const bool folding = fold && idb == 1 && rp.rel >= 1 && right_fold_fits<T>(dimension);
        if (folding) fold->level = rp.qe;
        const dim3 grid{unsigned((rp.lv.lo[rp.qe] + rp.d + kBlock - 1) / kBlock), unsigned(std::min<uint64_t>(batch, 65535)), 1};
        if (rp.longer)
            hipLaunchKernelGGL((right_sums_zero_kernel<T>), grid, dim3(kBlock), 0, stream, dA, int64_t(batch), rp, int64_t(s.stride), s.off);
        launch_right_stream<T>(rp, dC, dB, A, rp.longer ? dA : nullptr, batch, s, stream, idb, dc, folding ? fold : nullptr);
        if (rp.longer)
            hipLaunchKernelGGL((right_sums_add_kernel<T>), grid, dim3(kBlock), 0, stream, dA, dB, folding ? fold->dz : nullptr, int64_t(batch), rp,
                               int64_t(s.stride), s.off);
    };
    if (families < 2) return left_factor();
    if (right && rp.longer) {       // keeps sums in dA
        right_factor();
        left_factor();
    } else {
        left_factor();
        right_factor();
    }
}

template void launch_combine_bwd<float>(const float*, float*, float*, const float*, const float*, uint64_t, uint64_t,
                                        uint64_t, const SigShape&, hipStream_t, int, SharedRows, int, ExpFold<float>*);
template void launch_combine_bwd<double>(const double*, double*, double*, const double*, const double*, uint64_t,
                                         uint64_t, uint64_t, const SigShape&, hipStream_t, int, SharedRows, int,
                                         ExpFold<double>*);

}  // namespace sigamd
