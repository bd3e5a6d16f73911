// Forward sweeps of few channels to high degrees with shared prefix chains.
//
// Where many words hang below a path (3 channels to degree 12: 797 160), the tree kernels of sig_kernels.h spend a large
// part of a step on the chain of Horner values along each lane's prefix, which every lane evaluates for itself, and on
// copies to and from the accumulation registers that a subtree of 121 values needs.  Here a word is cut into a head of H
// letters, a lane's own, and a tail whose letters are the same for a whole wave:
//   * one wave of a block, the producer, evaluates the chains of the block's 64 heads and leaves, per step, the Horner values
//     towards the levels above H in LDS, a chunk of steps ahead of use;
//   * every other wave, a consumer, carries 64 heads x one tail: it goes on from the head's values along M letters and
//     through a subtree of TAIL levels.  Its letters are wave-uniform, so that they and their fractions z / j come as scalar
//     operands from a table that a pass over the increments lays out beforehand, and cost no instruction.
// The values are those of cp_signature.h:464-499 (siglib/cpsig), regrouped per word as in sig_tree.h.
//
// Double precision only: single precision has the registers for larger subtrees in the tree kernels, whose all-vector
// operands it issues faster (3 channels, degree 12, 282 paths of 257 points: tree 3.1 ms, this form 4.9).
// Measured at 3 channels, degree 12, 64 paths of 4096 points: 23.3 -> 14.4-15.3 ms; 74 vector instructions a step and wave for
// 27 top-level values (tree: 455 for 81), four waves a SIMD.  Bound: vector FP64 issue, 80 % of a SIMD's cycles (6.9e6 instructions of four
// cycles in 34.4e6, at 2.3 GHz; counters), beside the scalar cache, whose 36 dwords a step and wave take as long; the rest are waits for scalar operands and
// for the other waves of a block at the end of a chunk.
#include <algorithm>

#include "sig_barrier.h"
#include "sig_heads.h"
#include "sig_kernels.h"

namespace sigamd {

using T = double;

template <int D_, int N_, int H_, int TAIL_, int K_, int C_, int PER_SIMD_, int CS_, int PAD>
struct HeadPlan {
    static constexpr int D = D_, N = N_, H = H_, TAIL = TAIL_, K = K_;
    static constexpr int M = N - H - TAIL;                          // letters between the head and the subtree
    static_assert(M >= 0 && TAIL >= 2 && D % K == 0, "head, letters between, subtree");
    static constexpr bool kAll = K == D;                            // the subtree's first level has all letters
    static constexpr int J = N - H;                                 // levels above the heads
    static constexpr int64_t P = ipow64(D, H);
    static constexpr int GROUPS = int((P + kWave - 1) / kWave);     // groups of 64 heads
    static constexpr int Q = int(ipow64(D, M)) * (D / K);           // tails
    static constexpr int C = C_;                                    // consumers of a block
    static constexpr int PARTS = (Q + C - 1) / C;
    static constexpr int WAVES = (C + PAD) / PAD * PAD;             // ... the producer and waves that stay idle
    static constexpr int PER_SIMD = PER_SIMD_;                      // waves of a SIMD that the registers are cut for
    static constexpr int CS = CS_;                                  // steps of a chunk
    static constexpr int HEADS = CS * J * kWave;                    // elements of a chunk of head values
    // A step's row of the table: its letters; per letter the fractions z / j, j = 1 .. J, of the letters between; per letter
    // the fractions z / j!, j = 1 .. TURN, of the turn (see HeadConsumer)
    static constexpr bool kTurnBetween = kAll && M > 0;
    static constexpr int FRACTIONS = kTurnBetween ? M - 1 : M;      // letters between that take fractions
    static constexpr int TURN = kTurnBetween ? TAIL + 1 : kAll ? 0 : TAIL;
    static constexpr int even(int n) { return (n + 1) / 2 * 2; }
    static constexpr int JP = FRACTIONS > 0 ? even(J) : 0, TP = even(TURN);
    static constexpr int FRACTION0 = even(D), TURN0 = FRACTION0 + D * JP;
    static constexpr int ROW = (TURN0 + D * TP + 7) / 8 * 8;
    __host__ __device__ static constexpr int64_t level(int l) { return (ipow64(D, l) - D) / (D - 1); }     // offset of a level in a row
    // subtree depth e holds K D^(e-1) values from off(e) on
    __host__ __device__ static constexpr int off(int e) { return K * int((ipow64(D, e - 1) - 1) / (D - 1)); }
    static constexpr int SUB = off(TAIL + 1);
    static constexpr size_t kLds = (size_t(2) * HEADS + 2 * CS * D) * sizeof(T);
};

template <typename Plan>
__global__ __launch_bounds__(kBlock) void head_table_kernel(const T* __restrict__ inc, T* __restrict__ table,
                                                            int64_t rows, int64_t L)
{
    const int64_t n = rows * Plan::ROW;
    for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += int64_t(gridDim.x) * kBlock) {
        const int64_t r = i / Plan::ROW;
        const int c = int(i % Plan::ROW);
        int letter = c;
        T by = T(1);
        if (c >= Plan::TURN0) {
            constexpr int TP = Plan::TP > 0 ? Plan::TP : 1;
            letter = (c - Plan::TURN0) / TP;
            for (int j = 2; j <= (c - Plan::TURN0) % TP + 1; ++j) by *= T(j);
        } else if (c >= Plan::FRACTION0) {
            constexpr int JP = Plan::JP > 0 ? Plan::JP : 1;
            letter = (c - Plan::FRACTION0) / JP;
            by = T((c - Plan::FRACTION0) % JP + 1);
        }
        const T z = letter < Plan::D ? inc[((r / L) * (L + 2) + 1 + r % L) * Plan::D + letter] : T(0);
        table[i] = z / by;
    }
}

// values read through the scalar cache: wave-uniform address, never written by the kernel that reads them
template <typename V>
using ScalarPtr = const V __attribute__((address_space(4)))*;

// Horner values on the way down a word come in two scales.  With c = S_k + c' z / (m + 1), m the levels still to go, every letter
// needs its fractions; with e = c / m!, e = S_k / m! + e' z, the letter alone does, at the cost of a product per node and value
// with m >= 2.  The heads and the letters between take the first, a node or two each; the subtree takes the second, since
// scalar operands are what a compute unit runs out of (the cache they come through delivers about one word a cycle to two of
// them).  The letter at the turn takes z / (m + 1)!.

template <typename Plan>
struct HeadConsumer {
    static constexpr int D = Plan::D, M = Plan::M, J = Plan::J, K = Plan::K, TAIL = Plan::TAIL;
    static constexpr int FRACTIONS = Plan::FRACTIONS, TURN = Plan::TURN;

    T c[M > 0 ? M : 1];             // levels H + 1 .. H + M of the tail's own word
    T s[Plan::SUB];                 // subtree
    T h[J];                         // the heads' values of the next step
    T fz[FRACTIONS > 0 ? FRACTIONS : 1][J];     // its fractions of the letters between
    T tz[K][TURN > 0 ? TURN : 1];               // ... and at the turn: of the last letter between, or of the subtree's first ones
    uint32_t letter[M + 1];         // where these lie in a row of the table (bytes)

    struct Letters {
        T z[D];
    };

    __device__ __forceinline__ void load_heads(const T* lds)
    {
#pragma unroll
        for (int t = 0; t < J; ++t) h[t] = lds[t * kWave];
    }
    __device__ __forceinline__ void load_row(ScalarPtr<char> row, Letters& all)
    {
#pragma unroll
        for (int a = 0; a < D; ++a) all.z[a] = ((ScalarPtr<T>)row)[a];
#pragma unroll
        for (int i = 0; i < FRACTIONS; ++i)
#pragma unroll
            for (int j = 0; j < J - i; ++j) fz[i][j] = ((ScalarPtr<T>)(row + letter[i]))[j];
        if constexpr (TURN > 0) {
#pragma unroll
            for (int k = 0; k < (Plan::kAll ? 1 : K); ++k)
#pragma unroll
                for (int j = 0; j < TURN; ++j) tz[k][j] = ((ScalarPtr<T>)(row + letter[M]))[k * Plan::TP + j];
        }
    }

    __device__ __forceinline__ static T over_factorial(T v, int m) {
        T f = T(1);
#pragma unroll
        for (int i = 2; i <= m; ++i) f *= T(i);
        return m <= 1 ? v : v * (T(1) / f);
    }

    // The letters between and the turn, from the heads' values h towards the levels above them.  On return w holds the values
    // that enter the subtree's first level, if that has all letters, and v those that leave each of its K nodes, if not.
    struct Middle {
        T w[J];
        T v[K][TAIL];
    };
    __device__ __forceinline__ void chain(Middle& m)
    {
#pragma unroll
        for (int t = 0; t < J; ++t) m.w[t] = h[t];
#pragma unroll
        for (int i = 0; i < FRACTIONS; ++i) {
#pragma unroll
            for (int t = J - i - 1; t >= 1; --t) m.w[t] = fmadd(m.w[t], fz[i][t], c[i]);
            c[i] = fmadd(m.w[0], fz[i][0], c[i]);
#pragma unroll
            for (int t = 0; t + 1 < J - i; ++t) m.w[t] = m.w[t + 1];
        }
        if constexpr (Plan::kTurnBetween) {
            T& S = c[M - 1];
            T x[TAIL];
#pragma unroll
            for (int t = TAIL; t >= 1; --t) x[t - 1] = fmadd(m.w[t], tz[0][t], over_factorial(S, t));
            S = fmadd(m.w[0], tz[0][0], S);
#pragma unroll
            for (int t = 0; t < TAIL; ++t) m.w[t] = x[t];
        } else if constexpr (Plan::kAll) {
#pragma unroll
            for (int t = 0; t < TAIL; ++t) m.w[t] = over_factorial(m.w[t], t + 1);
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k) {
#pragma unroll
                for (int t = TAIL - 1; t >= 1; --t) m.v[k][t - 1] = fmadd(m.w[t], tz[k][t], over_factorial(s[k], t));
                s[k] = fmadd(m.w[0], tz[k][0], s[k]);
            }
        }
        // all sums of this part stay ahead of the branch that follows, and so of the loads into their operands
#pragma unroll
        for (int i = 0; i < M; ++i) asm volatile("" : "+v"(c[i]));
        if constexpr (Plan::kAll) {
#pragma unroll
            for (int t = 0; t < TAIL; ++t) asm volatile("" : "+v"(m.w[t]));
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                asm volatile("" : "+v"(s[k]));
#pragma unroll
                for (int t = 0; t + 1 < TAIL; ++t) asm volatile("" : "+v"(m.v[k][t]));
            }
        }
    }
    // children, at subtree depth E, of node `idx`; w: the node's values towards the levels from theirs on
    template <int E, int W>
    __device__ __forceinline__ void below(const T (&w)[W], const Letters& all, int idx)
    {
        if constexpr (E <= TAIL) {
            T v[D][TAIL];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                T& S = s[Plan::off(E) + idx * D + a];
#pragma unroll
                for (int t = TAIL - E; t >= 1; --t) v[a][t - 1] = fmadd(w[t], all.z[a], over_factorial(S, t));
                S = fmadd(w[0], all.z[a], S);
            }
#pragma unroll
            for (int a = 0; a < D; ++a) below<E + 1>(v[a], all, idx * D + a);
        }
    }
    __device__ __forceinline__ void subtree(const Middle& m, const Letters& all)
    {
        if constexpr (Plan::kAll) {
            below<1>(m.w, all, 0);
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k) below<2>(m.v[k], all, k);
        }
    }
};

// one struct, so that what is needed only after the sweep can be read again then
struct HeadsArgs {
    const void* inc;
    const void* table;
    void* out;
    int64_t L, out_stride, lseg;
    int* nonfinite;
    int scalar, nseg;
};

__device__ __forceinline__ const HeadsArgs __attribute__((address_space(4))) * kernel_args()
{
    auto p = (const HeadsArgs __attribute__((address_space(4)))*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

template <typename Plan>
__global__ __launch_bounds__(Plan::WAVES * kWave) __attribute__((amdgpu_waves_per_eu(Plan::PER_SIMD))) void heads_fwd_kernel(HeadsArgs)
{
    constexpr int D = Plan::D, N = Plan::N, H = Plan::H, M = Plan::M, J = Plan::J, TAIL = Plan::TAIL, CS = Plan::CS;
    extern __shared__ double heads_lds[];
    T* lds = reinterpret_cast<T*>(heads_lds);       // [2][CS][J][64] head values, [2][CS][D] increments
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const int64_t block = xcd_block();
    const int part = int(block % Plan::PARTS);
    const int group = int(block / Plan::PARTS % Plan::GROUPS);
    const int64_t item = block / (Plan::PARTS * Plan::GROUPS);      // (path, segment)
    const auto* args = kernel_args();
    const int nseg = args->nseg;
    const int64_t L = args->L, lseg = args->lseg;
    const int64_t b = item / nseg, t0 = (item % nseg) * lseg;
    const int ns = int(L - t0 < lseg ? L - t0 : lseg);              // steps, at least one
    const int chunks = (ns + CS - 1) / CS;
    const int64_t q = int64_t(group) * kWave + lane;
    const bool active = q < Plan::P;
    T chk = T(0);               // stays 0 while every value is finite

    if (wave == 0) {
        int p[H];
        {
            int64_t r = active ? q : Plan::P - 1;
#pragma unroll
            for (int l = H - 1; l >= 0; --l) {
                p[l] = int(r % D);
                r /= D;
            }
        }
        T c[H];
#pragma unroll
        for (int l = 0; l < H; ++l) c[l] = T(0);
        T* ring = lds + 2 * Plan::HEADS;
        const T* src = static_cast<const T*>(args->inc) + (b * (L + 2) + 1 + t0) * D;
        constexpr int CHUNK = CS * D, NREG = (CHUNK + kWave - 1) / kWave;
        T regs[NREG];
        // rows of a chunk: the increments continue for more than a chunk past any row (their buffer's slack)
        auto fetch = [&](int k) {
#pragma unroll
            for (int i = 0; i < NREG; ++i) {
                const int e = lane + i * kWave;
                if (e < CHUNK) regs[i] = src[int64_t(k) * CHUNK + e];
            }
        };
        auto commit = [&](int k) {
#pragma unroll
            for (int i = 0; i < NREG; ++i) {
                const int e = lane + i * kWave;
                if (e < CHUNK) ring[(k & 1) * CHUNK + e] = regs[i];
            }
        };
        fetch(0);
        commit(0);
        if (chunks > 1) fetch(1);
        for (int k = 0; k < chunks; ++k) {
            if (k + 1 < chunks) commit(k + 1);
            if (k + 2 < chunks) fetch(k + 2);
            const int n = int(ns - k * CS < CS ? ns - k * CS : CS);
            const T* row = ring + (k & 1) * CHUNK;
            T* dst = lds + (k & 1) * Plan::HEADS + lane;
            T z[H];
#pragma unroll
            for (int l = 0; l < H; ++l) z[l] = row[p[l]];
            for (int i = 0; i < n; ++i) {
                T zn[H];
                const int next = i + 1 < n ? D : 0;
#pragma unroll
                for (int l = 0; l < H; ++l) zn[l] = row[next + p[l]];
                // u[t]: Horner value towards level t along the head
                T u[N + 1];
#pragma unroll
                for (int t = 2; t <= N; ++t) u[t] = fmadd(z[0], rcp<T>(t), c[0]);
                c[0] += z[0];
#pragma unroll
                for (int l = 1; l < H; ++l) {
#pragma unroll
                    for (int t = N; t > l + 1; --t) u[t] = fmadd(u[t], z[l] * rcp<T>(t - l), c[l]);
                    c[l] = fmadd(u[l + 1], z[l], c[l]);
                }
#pragma unroll
                for (int t = 0; t < J; ++t) dst[t * kWave] = u[H + 1 + t];
                dst += J * kWave;
                row += next;
#pragma unroll
                for (int l = 0; l < H; ++l) z[l] = zn[l];
            }
            lds_barrier();
        }
        if (part == 0 && active) {
            const auto* late = kernel_args();
            const int scalar = late->scalar;
            T* o = static_cast<T*>(late->out) + item * late->out_stride + (scalar ? 1 : 0);
            if (scalar && q == 0) o[-1] = T(1);
            int64_t rest = 1;
#pragma unroll
            for (int l = H; l >= 1; --l) {
                if (q % rest == 0) o[Plan::level(l) + q / rest] = c[l - 1];
                chk = fmadd(c[l - 1], T(0), chk);
                rest *= D;
            }
        }
    } else {
        // A block of sixteen with a wave to spare leaves it to the producer's SIMD
        constexpr bool kSpare = Plan::WAVES >= 8 && Plan::WAVES > Plan::C + 1;
        const int consumer = kSpare && wave == 4 ? Plan::C : kSpare && wave > 4 ? wave - 2 : wave - 1;
        const int tail = part * Plan::C + consumer;
        if (consumer >= Plan::C || tail >= Plan::Q) {
            for (int k = 0; k < chunks; ++k) lds_barrier();
            return;
        }
        HeadConsumer<Plan> S;
        {
            int r = tail;
            auto place = [&](int first) {
                uint32_t at = uint32_t(first) * uint32_t(sizeof(T));
                asm volatile("" : "+s"(at));
                return at;
            };
            if (!Plan::kAll) S.letter[M] = place(Plan::TURN0 + r % (D / Plan::K) * Plan::K * Plan::TP);
            r /= D / Plan::K;
#pragma unroll
            for (int i = M - 1; i >= 0; --i) {
                if (i >= Plan::FRACTIONS) S.letter[M] = place(Plan::TURN0 + r % D * Plan::TP);
                else S.letter[i] = place(Plan::FRACTION0 + r % D * Plan::JP);
                r /= D;
            }
        }
#pragma unroll
        for (int i = 0; i < (M > 0 ? M : 1); ++i) S.c[i] = T(0);
#pragma unroll
        for (int i = 0; i < Plan::SUB; ++i) S.s[i] = T(0);
        ScalarPtr<char> row = (ScalarPtr<char>)(ScalarPtr<T>)(static_cast<const T*>(args->table) + (b * L + t0) * Plan::ROW);
        const T* heads = lds + lane;
        typename HeadConsumer<Plan>::Letters la, lb;
        lds_barrier();
        S.load_heads(heads);
        S.load_row(row, la);
        int to_chunk = CS, left = chunks;
        // A step's operands were requested in the step before, as soon as the tail's chain had used that step's.
        auto step = [&](typename HeadConsumer<Plan>::Letters& now, typename HeadConsumer<Plan>::Letters& next) {
            wait_lds();
            typename HeadConsumer<Plan>::Middle m;
            S.chain(m);
            __builtin_amdgcn_sched_barrier(0);
            heads += J * kWave;
            if (--to_chunk == 0) {
                to_chunk = CS;
                if (--left > 0) lds_barrier();
                heads = lds + ((chunks - left) & 1) * Plan::HEADS + lane;
            }
            row += Plan::ROW * sizeof(T);       // after the last step: the row that ends the table, unused
            asm volatile("" : "+s"(row));
            S.load_heads(heads);                // after the last step: unused values from the ring
            S.load_row(row, next);
            __builtin_amdgcn_sched_barrier(0);
            S.subtree(m, now);
        };
        int n = ns;
        for (; n >= 2; n -= 2) {
            step(la, lb);
            step(lb, la);
        }
        if (n) step(la, lb);
        if (active) {
            const auto* late = kernel_args();
            T* o = static_cast<T*>(late->out) + item * late->out_stride + (late->scalar ? 1 : 0);
            constexpr int NG = D / Plan::K;                     // groups of first letters
            const int between = tail / NG;                      // the letters between
            const int64_t node = q * ipow64(D, M) + between;    // the word of level H + M
            int64_t rest = 1;
#pragma unroll
            for (int i = M; i >= 1; --i) {
                if (tail % NG == 0 && between % rest == 0) o[Plan::level(H + i) + node / rest] = S.c[i - 1];
                chk = fmadd(S.c[i - 1], T(0), chk);
                rest *= D;
            }
            static_for<1, TAIL>([&](auto ec) {
                constexpr int E = decltype(ec)::value;
                constexpr int n_e = Plan::K * int(ipow64(D, E - 1));
                T* dst = o + Plan::level(H + M + E) + (node * NG + tail % NG) * n_e;
#pragma unroll
                for (int v = 0; v < n_e; ++v) dst[v] = S.s[Plan::off(E) + v];
            });
#pragma unroll
            for (int v = 0; v < Plan::SUB; ++v) chk = fmadd(S.s[v], T(0), chk);
        }
    }
    if (active && !(chk == T(0))) {
        int* nonfinite = kernel_args()->nonfinite;
        if (nonfinite) *nonfinite = 1;
    }
}

template <typename Plan>
constexpr int64_t kMostBlocks = ((int64_t(1) << 32) - 1) / (Plan::WAVES * kWave);

template <typename Plan>
static hipError_t launch_plan(const HeadsParams& p)
{
    const int64_t rows = p.paths * p.L;
    const int64_t blocks = p.paths * p.nseg * Plan::GROUPS * Plan::PARTS;
    if (blocks < 1 || blocks > kMostBlocks<Plan>) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((head_table_kernel<Plan>), dim3(unsigned(std::min<int64_t>((rows * Plan::ROW + kBlock - 1) / kBlock, 8192))), dim3(kBlock), 0,
                       p.stream, static_cast<const T*>(p.inc), static_cast<T*>(p.table), rows, p.L);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (Plan::kLds > 64 * 1024) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(heads_fwd_kernel<Plan>), hipFuncAttributeMaxDynamicSharedMemorySize, int(Plan::kLds));
        if (e != hipSuccess) return e;
    }
    const HeadsArgs args{p.inc, p.table, p.out, p.L, p.out_stride, p.lseg, p.nonfinite, p.scalar, p.nseg};
    hipLaunchKernelGGL((heads_fwd_kernel<Plan>), dim3(unsigned(blocks)), dim3(Plan::WAVES * kWave), Plan::kLds, p.stream, args);
    return hipGetLastError();
}

// step_ns: a step of as many blocks as a compute unit holds, lone_ns: of few, both measured
template <typename Plan>
static constexpr HeadsEntry entry(int step_ns, int lone_ns)
{
    constexpr int by_waves = 4 * Plan::PER_SIMD / Plan::WAVES, by_lds = int(160 * 1024 / Plan::kLds);
    static_assert(by_waves >= 1 && by_lds >= 1, "a block fits a compute unit");
    static_assert(Plan::GROUPS * Plan::PARTS <= kMostBlocks<Plan> / 64, "a path in as many pieces as the dispatch cuts fits a launch");
    return HeadsEntry{Plan::D, Plan::N, Plan::ROW, Plan::GROUPS * Plan::PARTS, kMostBlocks<Plan>, by_waves < by_lds ? by_waves : by_lds, step_ns, lone_ns,
                      launch_plan<Plan>};
}

// Plans found by a sweep over heads, tails and blocks at full launches (3e7 / D^N x 5 paths of 257 points), kept where they take at most 0.9 of the
// tree kernels' time.  ms before / with: 3 channels, degree 9 .. 14: 2.80 / 1.98, 7.14 / 4.84, 7.58 / 4.92, 6.53 / 4.71, 8.83 / 4.65, 9.61 / 4.66;
// 4, 9 and 10: 4.25 / 3.81, 4.46 / 3.72; 5, 8 and 9: 4.09 / 3.46, 4.55 / 3.38; 6, 7 and 8: 3.14 / 2.77, 3.53 / 2.56; 8, 7: 3.25 / 2.47; 11, 6:
// 3.64 / 2.78; 4, 11 and 12: 5.02 / 4.22, 5.09 / 3.62; 5, 10: 5.33 / 3.51; 6, 9: 3.70 / 2.52; 7, 8: 3.68 / 2.97; 8, 8: 3.25 / 2.31; 10, 7:
// 3.26 / 2.45.  3, 15 and 16, 5, 11, 7, 9 and 9, 8 have no compiled tree kernel (3, 15: 94.0 / 4.89).  12, 7 gains only in
// calls that leave the tree kernel a last round of few waves (2 x 400: 1.84 / 1.70).  2 channels, 9 and 11 at degree 7, and fewer levels than these,
// are faster in the tree kernels (2, 14: 3.9 / 4.3; 7, 6: 2.8 / 3.6).
static const HeadsEntry kHeads[] = {
    entry<HeadPlan<3, 9, 5, 4, 1, 3, 4, 8, 1>>(545, 305),
    entry<HeadPlan<3, 10, 6, 3, 3, 3, 4, 8, 1>>(620, 309),
    entry<HeadPlan<3, 11, 5, 3, 3, 14, 4, 16, 16>>(610, 540),
    entry<HeadPlan<3, 12, 6, 3, 3, 14, 4, 16, 16>>(610, 560),
    entry<HeadPlan<3, 13, 7, 3, 3, 14, 4, 16, 16>>(610, 585),
    entry<HeadPlan<3, 14, 8, 3, 3, 14, 4, 16, 16>>(620, 600),
    entry<HeadPlan<3, 15, 9, 3, 3, 14, 4, 16, 16>>(620, 600),
    entry<HeadPlan<3, 16, 9, 3, 3, 14, 4, 16, 16>>(670, 600),
    entry<HeadPlan<4, 9, 4, 3, 2, 11, 3, 16, 1>>(400, 400),
    entry<HeadPlan<4, 10, 5, 3, 2, 11, 3, 16, 1>>(410, 400),
    entry<HeadPlan<4, 11, 5, 3, 2, 11, 3, 16, 1>>(440, 440),
    entry<HeadPlan<4, 12, 6, 3, 2, 11, 3, 16, 1>>(470, 440),
    entry<HeadPlan<5, 8, 4, 3, 1, 13, 4, 16, 16>>(360, 350),
    entry<HeadPlan<5, 9, 4, 2, 5, 14, 4, 16, 16>>(410, 400),
    entry<HeadPlan<5, 10, 5, 2, 5, 14, 4, 16, 16>>(410, 400),
    entry<HeadPlan<5, 11, 6, 2, 5, 14, 4, 16, 16>>(410, 400),
    entry<HeadPlan<6, 7, 4, 2, 6, 6, 4, 8, 8>>(390, 270),
    entry<HeadPlan<6, 8, 5, 2, 6, 6, 4, 8, 8>>(420, 310),
    entry<HeadPlan<6, 9, 6, 2, 6, 6, 4, 8, 8>>(420, 320),
    entry<HeadPlan<7, 8, 5, 2, 7, 3, 3, 16, 1>>(320, 290),
    entry<HeadPlan<7, 9, 4, 2, 7, 11, 3, 16, 1>>(470, 440),
    entry<HeadPlan<8, 7, 3, 2, 4, 15, 4, 16, 1>>(380, 380),
    entry<HeadPlan<8, 8, 4, 2, 4, 15, 4, 16, 1>>(390, 380),
    entry<HeadPlan<9, 8, 4, 2, 3, 14, 4, 16, 16>>(360, 340),
    entry<HeadPlan<10, 7, 3, 2, 5, 11, 3, 16, 1>>(410, 400),
    entry<HeadPlan<11, 6, 4, 2, 1, 11, 8, 16, 1>>(240, 230),
    entry<HeadPlan<12, 7, 3, 2, 3, 14, 4, 16, 16>>(400, 390),
};

const HeadsEntry* heads_entry(uint64_t d, uint64_t degree)
{
    for (const HeadsEntry& e : kHeads)
        if (uint64_t(e.D) == d && uint64_t(e.N) == degree) return &e;
    return nullptr;
}

}  // namespace sigamd
