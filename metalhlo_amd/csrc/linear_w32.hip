// Linear layers of a few tokens whose parameters are held in fp32:
//   C = act(x . round(W) + round(bias)),  and behind them  x' = round(sum + round(bias)) + x,  h = LayerNorm(x'),
// tensors in a 16-bit type, every parameter rounded to that type where it is used.  The results are those of
// converting the parameters first and launching dot_general, add and LayerNorm one after the other (up to the order of the
// fp32 sums), without the conversion's pass over all weights (GPT-2-small: 117 us for 124 M parameters).
//
// What bounds it: launches (1.6 us each when they depend on one another) and latencies.  A cold matrix answers after about
// 4 us, address translation included, and a compute unit takes no more than about 30 bytes a nanosecond from memory,
// 75 from its L2: [4,768] x [768,768] 5.4 us with W from memory, 4.1 from the memory-side cache, 2.7 from the L2s.  Hence
//   * as in gemm_skinny.hip a workgroup owns a strip of columns, its waves split K, W goes to the operand registers
//     without a stop in LDS and all of it is in flight before anything else;
//   * a layer whose result is added to the residual splits K over the grid too ([37,3072] x [3072,768] 19.5 us in 48
//     workgroups, 7.4 in 192), and the launch that adds the parts up forms the next LayerNorm, whose rows it holds anyway;
//   * workgroups in front of a launch fetch weights that the next launches will read into the L2 of the XCD that
//     will want them (fetch_ahead): [37,768] x [768,2304] 7.3 -> 5.0 us, those workgroups included.
// Workgroups of one XCD take neighbouring strips, so a 128-byte line of W that two strips share is fetched once.
#include <initializer_list>
#include <mutex>
#include <type_traits>

#include "arrive.h"
#include "attention_short.h"
#include "gemm_lds.h"

namespace mhip {
namespace {

constexpr int kAhead = 2, kAheadLoads = 16, kWaves = 8;

struct Band { const float* w; int N, K, cols, wgs; uint32_t magic; };      // cols: what the strips of one XCD will cover; wgs: per XCD

struct LinearArgs {
    const void* x;
    const float *gamma, *beta;        // finish_norm_kernel, and a product that normalises the rows of x; beta may be NULL
    float eps;
    const float* w;
    const float* bias;                // may be NULL
    const void* residual;             // may be NULL
    void* c;
    float* sums;                      // instead of c: fp32 sums [splits][M][N]
    uint64_t *words, tag;             // with sums: the last part to arrive adds them up to c (arrive.h)
    int M, N, K, act, splits;
    int strips, per_xcd, blocks, first;      // first: workgroups in front of the product's
    int part_steps, per;              // k steps of a part and of a wave
    uint32_t by_blocks, by_splits;    // divided(n, .): n / blocks, n / splits
    Band ahead[kAhead];
};

// A launch here is a few hundred instructions a wave, 2 to 3 ns each where nothing overlaps them, and a division is 25 of them: the ones that a
// workgroup needs to find its place are formed by a multiplication (exact for numbers below 2^32 / n; GPT-2-small over 37 tokens 446 -> 436 us).
inline uint32_t divisor(int n) { return n == 1 ? 0 : (uint32_t)((((uint64_t)1 << 32) + n - 1) / n); }
__device__ __forceinline__ int divided(int n, uint32_t by) { return by ? (int)__umulhi((uint32_t)n, by) : n; }

template <typename T>
__device__ __forceinline__ float rounded(float v) { return Elem<T>::to_f32(Elem<T>::from_f32(v)); }
// Workgroup `id` of those in front: kAheadLoads 16-byte pieces per thread of the columns that the strips of its XCD cover.
__device__ __forceinline__ void fetch_ahead(const LinearArgs& g, int id) {
    const int xcd = id % kXcds;
    int j = id / kXcds, r = 0;
    if (j >= g.ahead[0].wgs) { j -= g.ahead[0].wgs; r = 1; }
    const float* w = r ? g.ahead[1].w : g.ahead[0].w;
    const int N = r ? g.ahead[1].N : g.ahead[0].N, K = r ? g.ahead[1].K : g.ahead[0].K, cols = r ? g.ahead[1].cols : g.ahead[0].cols;
    const uint32_t magic = r ? g.ahead[1].magic : g.ahead[0].magic, per_row = (uint32_t)cols / 4;
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(w, (uint32_t)((int64_t)N * K * 4));
    const uint32_t at = (uint32_t)j * (64 * kWaves * kAheadLoads) + threadIdx.x;
    u32x4 v[kAheadLoads];
#pragma unroll
    for (int i = 0; i < kAheadLoads; i++) {
        const uint32_t p = at + i * 64 * kWaves, row = __umulhi(p, magic), col = xcd * cols + (p - row * per_row) * 4;
        v[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)row < K && (int)col < N ? (row * (uint32_t)N + col) * 4 : kOob, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < kAheadLoads; i++) asm volatile("" ::"v"(v[i]));
}

// A strip of 16 columns.  TB: W stored [N, K].  MT = groups of 16 rows, U = steps of 32 k that a wave holds at once; LOOP: it has
// more of them and loads a block ahead.  FORM kArrive: the last part of K to arrive adds the parts up.  kNorm: the rows of x are normalised first, LayerNorm(x) rounded to T, which a workgroup with
// all of K holds anyway: two barriers here instead of a launch (finish_norm_kernel 3.3 us; GPT-2-small's two norms a layer cost 0.7 each).
enum Form { kPlain = 0, kNorm = 1, kArrive = 2 };
template <typename T, bool TB, bool LOOP, int FORM, int MT, int U>
__global__ __launch_bounds__(64 * kWaves, LOOP ? 2 : 4) void linear_w32_kernel(LinearArgs g) {
    constexpr int KS = 32;
    constexpr bool NORM = FORM == kNorm, ARRIVE = FORM == kArrive;
    static_assert(!NORM || (!TB && !LOOP), "all of K in the workgroup");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    // The arguments are asked for together: behind the branches that use them they come in four goes, each of a latency (GPT-2-small over 37 tokens, this
    // and the other kernels of a layer: 436 -> 412 us).
    asm volatile("" ::"s"(g.first), "s"(g.x), "s"(g.w), "s"(g.bias), "s"(g.residual), "s"(g.c), "s"(g.M), "s"(g.N), "s"(g.K), "s"(g.splits), "s"(g.strips), "s"(g.per_xcd),
                 "s"(g.blocks), "s"(g.part_steps), "s"(g.per), "s"(g.by_blocks), "s"(g.by_splits));
    if ((int)blockIdx.x < g.first) {
        fetch_ahead(g, blockIdx.x);
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const uint32_t id = blockIdx.x - (uint32_t)g.first;
    const int xcd = id % kXcds, local = id / kXcds, column = divided(local, g.by_blocks), m0 = (local - column * g.blocks) * (16 * MT);
    const int place = divided(column, g.by_splits), split = column - place * g.splits, strip = xcd * g.per_xcd + place, n0 = strip * 16;
    if (strip >= g.strips) return;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(g.x, (uint32_t)((int64_t)g.M * g.K * 2));
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(g.w, (uint32_t)((int64_t)g.N * g.K * 4));

    // ---- this wave's share of the k steps
    const int all = (g.K + KS - 1) / KS, p0 = split * g.part_steps, p1 = min(all, p0 + g.part_steps), s0 = p0 + wave * g.per, s1 = min(p1, s0 + g.per);
    uint64_t* const word = ARRIVE ? g.words + strip * g.blocks + m0 / (16 * MT) : nullptr;
    uint64_t seen = 0;
    if (ARRIVE && threadIdx.x == 0) seen = arrive_look(word);
    f32x4 ga = {0.f, 0.f, 0.f, 0.f}, be = ga;
    const int gn = threadIdx.x * 4;
    if (NORM && gn < g.K) {
        ga = *reinterpret_cast<const f32x4*>(g.gamma + gn);
        if (g.beta) be = *reinterpret_cast<const f32x4*>(g.beta + gn);
    }
    struct Block {
        f32x4 wt[TB ? U : 1][2];                             // W stored [N, K]: eight k of a column
        float wn[TB ? 1 : U][TB ? 1 : 8];                    // W stored [K, N]: the same, one by one
        u32x4 a[U][MT];
    };
    auto load = [&](Block& b, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = (s + u) * KS + lg * 8;
            const bool live = s + u < s1 && k < g.K;
            const int n = n0 + li;
            if (TB) {
                const uint32_t off = live && n < g.N ? (uint32_t)(((int64_t)n * g.K + k) * 4) : kOob;
#pragma unroll
                for (int h = 0; h < 2; h++) b.wt[TB ? u : 0][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, off + 16 * h, 0, 0));
            } else {
                const uint32_t off = live && n < g.N ? (uint32_t)(((int64_t)k * g.N + n) * 4) : kOob;
#pragma unroll
                for (int j = 0; j < 8; j++)
                    b.wn[TB ? 0 : u][TB ? 0 : j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rw, off + (uint32_t)(j * g.N * 4), 0, 0));
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const int k = (s + u) * KS + lg * 8, m = m0 + mt * 16 + li;
                b.a[u][mt] = __builtin_amdgcn_raw_buffer_load_b128(rx, s + u < s1 && k < g.K && m < g.M ? (uint32_t)((m * g.K + k) * 2) : kOob, 0, 0);
            }
    };
    Block cur;
    load(cur, s0);

    // ---- the epilogue's thread (wave = mt, li, lg) finishes row li of group mt: columns 4 lg .. 4 lg + 3 of the strip
    const int fm = m0 + wave * 16 + li, col = n0 + 4 * lg;
    const bool finisher = wave < MT && fm < g.M;
    f32x4 bias = {0.f, 0.f, 0.f, 0.f};
    u32x2 res = {0, 0};
    if (finisher && col < g.N) {
        if (g.bias) bias = *reinterpret_cast<const f32x4*>(g.bias + col);
        if (g.residual) res = *reinterpret_cast<const u32x2*>(static_cast<const T*>(g.residual) + (int64_t)fm * g.N + col);
    }

    if constexpr (NORM) {
        constexpr int kMostK = kWaves * U * KS;
        float* const stat = reinterpret_cast<float*>(smem);              // [2][wave][row]
        float* const gb = stat + 2 * kWaves * MT * 16;                   // gamma, beta
        if (gn < g.K) {
#pragma unroll
            for (int e = 0; e < 4; e++) { gb[gn + e] = rounded<T>(ga[e]); gb[kMostK + gn + e] = rounded<T>(be[e]); }
        }
        typedef T vec8 __attribute__((ext_vector_type(8)));
        auto over_row = [&](float(&v)[MT], int set) __attribute__((always_inline)) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                v[mt] += __shfl_xor(v[mt], 16, 64);
                v[mt] += __shfl_xor(v[mt], 32, 64);
                if (lg == 0) stat[(set * kWaves + wave) * MT * 16 + mt * 16 + li] = v[mt];
            }
            __syncthreads();
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                v[mt] = 0.f;
#pragma unroll
                for (int w = 0; w < kWaves; w++) v[mt] += stat[(set * kWaves + w) * MT * 16 + mt * 16 + li];
                v[mt] = v[mt] / (float)g.K;                              // (a quotient: a row of equal elements has that mean and no variance)
            }
            // (from here on the operand as 16-bit values only: kept as the fp32 values of this pass they would be spilled)
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int e = 0; e < 4; e++) asm("" : "+v"(cur.a[u][mt][e]));
        };
        float mean[MT], var[MT];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            mean[mt] = 0.f;
#pragma unroll
            for (int u = 0; u < U; u++) {                                // (what is not there reads zero)
                const vec8 v = __builtin_bit_cast(vec8, cur.a[u][mt]);
#pragma unroll
                for (int e = 0; e < 8; e++) mean[mt] += (float)v[e];
            }
        }
        over_row(mean, 0);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            var[mt] = 0.f;
#pragma unroll
            for (int u = 0; u < U; u++) {
                const vec8 v = __builtin_bit_cast(vec8, cur.a[u][mt]);
                if (s0 + u < s1 && (s0 + u) * KS + lg * 8 < g.K)
#pragma unroll
                    for (int e = 0; e < 8; e++) { const float t = (float)v[e] - mean[mt]; var[mt] = fmaf(t, t, var[mt]); }
            }
        }
        over_row(var, 1);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) var[mt] = 1.f / sqrtf(var[mt] + g.eps);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = (s0 + u) * KS + lg * 8;
            if (s0 + u >= s1 || k >= g.K) continue;
            const f32x4 *gs = reinterpret_cast<const f32x4*>(gb + k), *bs = reinterpret_cast<const f32x4*>(gb + kMostK + k);
            const f32x4 g2[2] = {gs[0], gs[1]}, b2[2] = {bs[0], bs[1]};
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const vec8 v = __builtin_bit_cast(vec8, cur.a[u][mt]);
                float o[8];
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = fmaf(((float)v[e] - mean[mt]) * var[mt], g2[e / 4][e % 4], b2[e / 4][e % 4]);
#pragma unroll
                for (int e = 0; e < 4; e++) cur.a[u][mt][e] = round_pair<T>(o[2 * e], o[2 * e + 1]);
            }
        }
        __syncthreads();                                                 // the sums below go where this has been read
    }

    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Block& b, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s + u >= s1) break;
            u32x4 w;
#pragma unroll
            for (int j = 0; j < 4; j++)
                w[j] = TB ? round_pair<T>(b.wt[TB ? u : 0][j / 2][j % 2 * 2], b.wt[TB ? u : 0][j / 2][j % 2 * 2 + 1])
                          : round_pair<T>(b.wn[TB ? 0 : u][TB ? 0 : 2 * j], b.wn[TB ? 0 : u][TB ? 0 : 2 * j + 1]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt] = Tile16<T>::run(w, b.a[u][mt], acc[mt]);
        }
    };
    if (LOOP) {
        for (int s = s0; s < s1; s += U) {
            Block nxt;
            if (s + U < s1) load(nxt, s + U);
            multiply(cur, s);
            if (s + U < s1) cur = nxt;
        }
    } else multiply(cur, s0);
    if (ARRIVE && threadIdx.x == 0) arrive_claim(word, seen, g.tag);

    // ---- the waves' partial sums, in the accumulators' own layout: lane (li, lg) holds row 16 mt + li and, in its four
    // registers, columns 4 lg .. 4 lg + 3
    f32x4* part = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int mt = 0; mt < MT; mt++) part[(wave * MT + mt) * 64 + lane] = acc[mt];
    __syncthreads();
    if (!ARRIVE && wave >= MT) return;
    f32x4 sum = part[(ARRIVE ? min(wave, MT - 1) : wave) * 64 + lane];
#pragma unroll
    for (int w = 1; w < kWaves; w++) sum += part[(w * MT + (ARRIVE ? min(wave, MT - 1) : wave)) * 64 + lane];
    const bool mine = finisher && col < g.N;
    if constexpr (ARRIVE) {
        __shared__ int last;
        const __amdgpu_buffer_rsrc_t rp = parts_rsrc(g.sums);
        if (mine) store_part(rp, (uint32_t)(((split * g.M + fm) * g.N + col) * 4), sum);
        if (!arrive_last(word, g.splits, &last) || !mine) return;
        f32x4 v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = load_part(rp, i < g.splits ? (uint32_t)(((i * g.M + fm) * g.N + col) * 4) : kOob);
        sum = v[0];
#pragma unroll
        for (int i = 1; i < 8; i++) sum += v[i];
    }
    if (!mine) return;
    if (!ARRIVE && g.sums) {
        *reinterpret_cast<f32x4*>(g.sums + ((int64_t)split * g.M + fm) * g.N + col) = sum;
        return;
    }
    T* c = static_cast<T*>(g.c) + (int64_t)fm * g.N + col;
    dispatch_act(g.act, [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
        Pack4<T> o, r = __builtin_bit_cast(Pack4<T>, res);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o.v[e] = Elem<T>::from_f32(apply_act_c<ACT>(sum[e] + rounded<T>(bias[e])));
            // (second rounding on purpose: the same result as a separate add over the stored C)
            if (g.residual) o.v[e] = Elem<T>::from_f32(Elem<T>::to_f32(o.v[e]) + Elem<T>::to_f32(r.v[e]));
        }
        *reinterpret_cast<u32x2*>(c) = __builtin_bit_cast(u32x2, o);
    });
}

// W stored [N, K] where a wave holds its share of the k steps at once (a tied output head: 50304 columns of K 768).  The grid
// is resident and walks the strips: x stays in registers, the next strip's W is on its way while this one is
// multiplied and added up, through two sets of partial sums with one barrier per strip.  One strip per workgroup spends as
// much on x as on W: [37,768] x [50304,768]^T 53 us against 36.7, [128,768] 106 against 58.
template <typename T, int MT, int U>
__global__ __launch_bounds__(64 * kWaves, MT < 2 ? 4 : 2) void linear_w32_stream_kernel(LinearArgs g) {
    constexpr int KS = 32;
    __shared__ f32x4 part[2][kWaves][MT][64];
    asm volatile("" ::"s"(g.x), "s"(g.w), "s"(g.bias), "s"(g.residual), "s"(g.c), "s"(g.M), "s"(g.N), "s"(g.K), "s"(g.act), "s"(g.strips));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int m0 = (int)blockIdx.y * (16 * MT);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(g.x, (uint32_t)((int64_t)g.M * g.K * 2));
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(g.w, (uint32_t)((int64_t)g.N * g.K * 4));
    const int all = (g.K + KS - 1) / KS, per = (all + kWaves - 1) / kWaves, s0 = wave * per, s1 = min(all, s0 + per);
    u32x4 a[U][MT];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int k = (s0 + u) * KS + lg * 8, m = m0 + mt * 16 + li;
            a[u][mt] = __builtin_amdgcn_raw_buffer_load_b128(rx, s0 + u < s1 && k < g.K && m < g.M ? (uint32_t)((m * g.K + k) * 2) : kOob, 0, 0);
        }
    f32x4 w[2][U][2];
    auto load = [&](f32x4(&v)[U][2], int strip) __attribute__((always_inline)) {
        const int n = strip * 16 + li;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = (s0 + u) * KS + lg * 8;
            const uint32_t off = s0 + u < s1 && k < g.K && n < g.N ? (uint32_t)((n * g.K + k) * 4) : kOob;
#pragma unroll
            for (int h = 0; h < 2; h++) v[u][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, off + 16 * h, 0, 0));
        }
    };
    const int fm = m0 + wave * 16 + li;
    const bool finisher = wave < MT && fm < g.M;
    T* c = static_cast<T*>(g.c) + (int64_t)fm * g.N;
    const T* res = static_cast<const T*>(g.residual) + (int64_t)fm * g.N;
    auto strip_of = [&](const f32x4(&v)[U][2], int strip, int set) __attribute__((always_inline)) {
        f32x4 acc[MT];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; u++) {
            const u32x4 b = {round_pair<T>(v[u][0][0], v[u][0][1]), round_pair<T>(v[u][0][2], v[u][0][3]),
                             round_pair<T>(v[u][1][0], v[u][1][1]), round_pair<T>(v[u][1][2], v[u][1][3])};
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt] = Tile16<T>::run(b, a[u][mt], acc[mt]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) part[set][wave][mt][lane] = acc[mt];
        // (a barrier that leaves the loads of W in flight; the set is written again behind the next strip's barrier, which
        // a wave reaches when it has read this one)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (wave >= MT) return;
        f32x4 sum = part[set][0][wave][lane];
#pragma unroll
        for (int i = 1; i < kWaves; i++) sum += part[set][i][wave][lane];
        const int n = strip * 16 + 4 * lg;
        if (!finisher || n >= g.N) return;
        f32x4 bias = {0.f, 0.f, 0.f, 0.f};
        if (g.bias) bias = *reinterpret_cast<const f32x4*>(g.bias + n);
        Pack4<T> r = {};
        if (g.residual) r = *reinterpret_cast<const Pack4<T>*>(res + n);
        dispatch_act(g.act, [&](auto act_tag) {
            constexpr int ACT = decltype(act_tag)::value;
            Pack4<T> o;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o.v[e] = Elem<T>::from_f32(apply_act_c<ACT>(sum[e] + rounded<T>(bias[e])));
                if (g.residual) o.v[e] = Elem<T>::from_f32(Elem<T>::to_f32(o.v[e]) + Elem<T>::to_f32(r.v[e]));
            }
            *reinterpret_cast<Pack4<T>*>(c + n) = o;
        });
    };
    const int stride = (int)gridDim.x;
    int strip = blockIdx.x;
    if (strip >= g.strips) return;
    load(w[0], strip);
    for (;;) {
        if (strip + stride < g.strips) load(w[1], strip + stride);
        strip_of(w[0], strip, 0);
        strip += stride;
        if (strip >= g.strips) break;
        if (strip + stride < g.strips) load(w[0], strip + stride);
        strip_of(w[1], strip, 1);
        strip += stride;
        if (strip >= g.strips) break;
    }
}

// Causal attention of a short prompt and the projection behind it: fp32 sums [part][M][N] of attention(x) . round(W), a part being `group` heads of size 64
// (their 64 group rows of W), for the launch that adds parts up.  Two launches that depend on one another cost 1.6 us between them and a trip of
// the attention's result past the L2s; what it takes to have it in every workgroup, 14 KB of x a head, comes from an L2 while W, which
// is fetched first, is on its way.  (GPT-2-small, against two launches: 37 tokens 453.5 -> 446.4 us, 2 x 20 452.7 -> 442.9.  A workgroup's waves take the heads of a part
// in one turn: with two, 4 x 12 tokens went from 462 to 465.)
// A workgroup owns 32 columns and a part: each wave takes 32 queries of a head, leaves the result in LDS, rounded as the attention kernel
// rounds it, and then takes 32 k of W.
constexpr int kProjectCols = 32, kProjectHead = 64;
template <typename T, int MT>
__global__ __launch_bounds__(64 * kWaves) void attend_project_kernel(FaArgs a, LinearArgs g, int group) {
    constexpr int NF = kProjectCols / 16, kValues = 64 * kProjectHead * 2;      // bytes of values a wave holds at once
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    asm volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.B), "s"(a.H), "s"(a.Sq), "s"(a.Skv), "s"(a.c), "s"(a.negate_q), "s"(a.qs[0]), "s"(a.qs[1]), "s"(a.ks[0]), "s"(a.ks[1]),
                 "s"(a.vs[0]), "s"(a.vs[1]), "s"((int)a.qs[2]), "s"((int)a.ks[2]), "s"((int)a.vs[2]), "s"(g.first), "s"(g.w), "s"(g.sums), "s"(g.M), "s"(g.N), "s"(g.K),
                 "s"(g.splits), "s"(g.per_xcd), "s"(g.by_blocks), "s"(g.by_splits), "s"(group));
    if ((int)blockIdx.x < g.first) {
        fetch_ahead(g, blockIdx.x);
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    // the columns of an XCD's strips are those that fetch_ahead gives its L2
    const uint32_t id = blockIdx.x - (uint32_t)g.first;
    const int xcd = id % kXcds, place = divided(id / kXcds, g.by_splits), part = id / kXcds - place * g.splits;
    const int n0 = xcd * g.per_xcd * 16 + place * kProjectCols, n1 = min(g.N, (xcd + 1) * g.per_xcd * 16);
    if (n0 >= n1) return;
    const int depth = group * kProjectHead, pitch = depth * 2 + 16;
    char* const rows = smem + kWaves * kValues;              // the attention's result, [M][depth]
    const bool active = wave * 32 < depth;

    float wn[NF][8];
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(g.w, (uint32_t)((int64_t)g.N * g.K * 4));
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int n = n0 + 16 * f + li, k = part * depth + wave * 32 + lg * 8;
        const uint32_t off = active && n < n1 ? (uint32_t)(((int64_t)k * g.N + n) * 4) : kOob;
#pragma unroll
        for (int j = 0; j < 8; j++) wn[f][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rw, off + (uint32_t)(j * g.N * 4), 0, 0));
    }

    // (a wave's 32 queries: half of sequence b, head h of the group; by_blocks divides by the sequences)
    const int halves = a.Sq > 32 ? 2 : 1, pair = wave >> (halves - 1), h = divided(pair, g.by_blocks), b = pair - h * a.B, half = wave & (halves - 1);
    if (h < group) {
        auto store = [&](int query, int d, u32x2 v) __attribute__((always_inline)) {
            *reinterpret_cast<u32x2*>(rows + (b * a.Sq + query) * pitch + (h * kProjectHead + d) * 2) = v;
        };
        if (half) short_rows<T, kProjectHead, 2>(a, b * a.H + part * group + h, smem + wave * kValues, store);
        else short_rows<T, kProjectHead, 1>(a, b * a.H + part * group + h, smem + wave * kValues, store);
    }
    __syncthreads();

    // (rows past the last hold whatever LDS held: each is a row of the product of its own, and not stored)
    f32x4* const sums = reinterpret_cast<f32x4*>(smem);      // [wave][MT][NF], where the values were
    if (active) {
        u32x4 w[NF];
#pragma unroll
        for (int f = 0; f < NF; f++)
#pragma unroll
            for (int j = 0; j < 4; j++) w[f][j] = round_pair<T>(wn[f][2 * j], wn[f][2 * j + 1]);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(rows + (mt * 16 + li) * pitch + (wave * 32 + lg * 8) * 2);
#pragma unroll
            for (int f = 0; f < NF; f++) sums[((wave * MT + mt) * NF + f) * 64 + lane] = Tile16<T>::run(w[f], x, f32x4{0.f, 0.f, 0.f, 0.f});
        }
    }
    __syncthreads();
    if (wave >= MT * NF) return;
    const int mt = wave / NF, f = wave % NF, m = mt * 16 + li, n = n0 + 16 * f + 4 * lg;
    f32x4 sum = sums[(mt * NF + f) * 64 + lane];
    for (int i = 1; i < depth / 32; i++) sum += sums[((i * MT + mt) * NF + f) * 64 + lane];
    if (m < g.M && n < n1) *reinterpret_cast<f32x4*>(g.sums + ((int64_t)part * g.M + m) * g.N + n) = sum;
}

// The same for up to 32 rows with all heads in a workgroup, a wave for one head of a sequence or two: 16 columns of c = round(attention(x) . round(W) + round(bias)) +
// residual, and no launch that adds parts up.  The wave of head h then takes its 64 rows of W.
// (GPT-2-small, against two launches: 4 tokens 331 -> 298 us, 8 tokens 335 -> 307, 16 tokens 348 -> 323, 32 tokens 405 -> 400.)
constexpr int kLayerWaves = 16, kLayerRows = 32;
template <typename T, int MT>
__global__ __launch_bounds__(64 * kLayerWaves) void attend_project_layer_kernel(FaArgs a, LinearArgs g) {
    constexpr int kValues = kLayerRows * kProjectHead * 2, kSteps = kProjectHead / 32;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    asm volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.B), "s"(a.H), "s"(a.Sq), "s"(a.Skv), "s"(a.c), "s"(a.negate_q), "s"(a.qs[0]), "s"(a.qs[1]), "s"(a.ks[0]), "s"(a.ks[1]),
                 "s"(a.vs[0]), "s"(a.vs[1]), "s"((int)a.qs[2]), "s"((int)a.ks[2]), "s"((int)a.vs[2]), "s"(g.first), "s"(g.w), "s"(g.bias), "s"(g.residual), "s"(g.c), "s"(g.M),
                 "s"(g.N), "s"(g.K), "s"(g.strips), "s"(g.per_xcd), "s"(g.by_blocks));
    if ((int)blockIdx.x < g.first) {
        if (threadIdx.x < 64 * kWaves) fetch_ahead(g, blockIdx.x);
        return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const uint32_t id = blockIdx.x - (uint32_t)g.first;
    const int strip = id % kXcds * g.per_xcd + id / kXcds, n0 = strip * 16, pitch = g.K * 2 + 16;
    if (strip >= g.strips) return;
    char* const rows = smem + waves * kValues;               // the attention's result, [M][K]
    const bool active = wave < a.H;

    float wn[kSteps][8];
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(g.w, (uint32_t)((int64_t)g.N * g.K * 4));
#pragma unroll
    for (int u = 0; u < kSteps; u++) {
        const int n = n0 + li, k = wave * kProjectHead + u * 32 + lg * 8;
        const uint32_t off = active && n < g.N ? (uint32_t)(((int64_t)k * g.N + n) * 4) : kOob;
#pragma unroll
        for (int j = 0; j < 8; j++) wn[u][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rw, off + (uint32_t)(j * g.N * 4), 0, 0));
    }
    const int fm = wave * 16 + li, col = n0 + 4 * lg;
    const bool mine = wave < MT && fm < g.M && col < g.N;
    f32x4 bias = {0.f, 0.f, 0.f, 0.f};
    u32x2 res = {0, 0};
    if (mine && g.bias) bias = *reinterpret_cast<const f32x4*>(g.bias + col);
    if (mine && g.residual) res = *reinterpret_cast<const u32x2*>(static_cast<const T*>(g.residual) + (int64_t)fm * g.N + col);

    // (by_blocks divides by the sequences)
    for (int pair = wave; pair < a.B * a.H; pair += waves) {
        const int h = divided(pair, g.by_blocks), b = pair - h * a.B;
        short_rows<T, kProjectHead, 1>(a, b * a.H + h, smem + wave * kValues, [&](int query, int d, u32x2 v) __attribute__((always_inline)) {
            *reinterpret_cast<u32x2*>(rows + (b * a.Sq + query) * pitch + (h * kProjectHead + d) * 2) = v;
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the next turn's values come to the same place)
    }
    __syncthreads();

    // (rows past the last hold whatever LDS held: each is a row of the product of its own, and not stored)
    f32x4* const sums = reinterpret_cast<f32x4*>(smem);      // [head][MT], where the values were
    if (active) {
        f32x4 acc[MT];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < kSteps; u++) {
            u32x4 w;
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = round_pair<T>(wn[u][2 * j], wn[u][2 * j + 1]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                acc[mt] = Tile16<T>::run(w, *reinterpret_cast<const u32x4*>(rows + (mt * 16 + li) * pitch + (wave * kProjectHead + u * 32 + lg * 8) * 2), acc[mt]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) sums[(wave * MT + mt) * 64 + lane] = acc[mt];
    }
    __syncthreads();
    if (!mine) return;
    f32x4 sum = sums[wave * 64 + lane];
#pragma unroll 4
    for (int i = 1; i < a.H; i++) sum += sums[(i * MT + wave) * 64 + lane];
    Pack4<T> o, r = __builtin_bit_cast(Pack4<T>, res);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        o.v[e] = Elem<T>::from_f32(sum[e] + rounded<T>(bias[e]));
        if (g.residual) o.v[e] = Elem<T>::from_f32(Elem<T>::to_f32(o.v[e]) + Elem<T>::to_f32(r.v[e]));
    }
    *reinterpret_cast<u32x2*>(static_cast<T*>(g.c) + (int64_t)fm * g.N + col) = __builtin_bit_cast(u32x2, o);
}

// A row per workgroup: x = round(sum of the parts + bias) + residual (or, without parts, the residual itself), stored to c
// when that is given, and h = LayerNorm(x).  Latency-bound: two memory latencies, two barriers.
constexpr int kFinishPieces = 4;      // four columns each, 256 threads: N <= 4096
template <typename T, int PIECES>
__global__ __launch_bounds__(256) void finish_norm_kernel(LinearArgs g, T* h) {
    __shared__ float red[2][4];
    asm volatile("" ::"s"(g.gamma), "s"(g.beta), "s"(g.eps), "s"(g.bias), "s"(g.residual), "s"(g.c), "s"(g.sums), "s"(g.M), "s"(g.N), "s"(g.splits), "s"(h));
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    f32x4 v[PIECES];
    u32x2 x[PIECES];
    f32x4 ga[PIECES], be[PIECES];
    float s = 0.f;
#pragma unroll
    for (int p = 0; p < PIECES; p++) {
        const int n = (p * 256 + (int)threadIdx.x) * 4;
        v[p] = f32x4{0.f, 0.f, 0.f, 0.f};
        x[p] = u32x2{0, 0};
        if (n >= g.N) continue;
        const int64_t at = row * g.N + n;
        ga[p] = *reinterpret_cast<const f32x4*>(g.gamma + n);
        be[p] = g.beta ? *reinterpret_cast<const f32x4*>(g.beta + n) : f32x4{0.f, 0.f, 0.f, 0.f};
        if (g.residual) x[p] = *reinterpret_cast<const u32x2*>(static_cast<const T*>(g.residual) + at);
        if (g.splits) {
            f32x4 b = f32x4{0.f, 0.f, 0.f, 0.f};
            if (g.bias) b = *reinterpret_cast<const f32x4*>(g.bias + n);
            // (four parts asked for at a time, the last one again where there are fewer: one by one each is a latency.  GPT-2-small over 37 tokens
            // 413 -> 397 us, 64 tokens 462 -> 445, 2 x 100 tokens 635 -> 622)
            for (int i = 0; i < g.splits; i += 4) {
                f32x4 t[4];
#pragma unroll
                for (int j = 0; j < 4; j++) t[j] = *reinterpret_cast<const f32x4*>(g.sums + (int64_t)min(i + j, g.splits - 1) * g.M * g.N + at);
                asm volatile("" : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]));
#pragma unroll
                for (int j = 0; j < 4; j++) v[p] += i + j < g.splits ? t[j] : f32x4{0.f, 0.f, 0.f, 0.f};
            }
            Pack4<T> r = __builtin_bit_cast(Pack4<T>, x[p]), o;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o.v[e] = Elem<T>::from_f32(v[p][e] + rounded<T>(b[e]));
                if (g.residual) o.v[e] = Elem<T>::from_f32(Elem<T>::to_f32(o.v[e]) + Elem<T>::to_f32(r.v[e]));
            }
            x[p] = __builtin_bit_cast(u32x2, o);
        }
        if (g.c) *reinterpret_cast<u32x2*>(static_cast<T*>(g.c) + at) = x[p];
        const Pack4<T> t = __builtin_bit_cast(Pack4<T>, x[p]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[p][e] = Elem<T>::to_f32(t.v[e]);
            s += v[p][e];
        }
    }
    auto over_row = [&](float t, int set) {
        t = wave_sum(t);
        if (lane == 0) red[set][wave] = t;
        __syncthreads();
        return (red[set][0] + red[set][1]) + (red[set][2] + red[set][3]);
    };
    // (quotients: a row of equal elements has that mean and no variance)
    const float mean = over_row(s, 0) / (float)g.N;
    float q = 0.f;
#pragma unroll
    for (int p = 0; p < PIECES; p++)
        if ((p * 256 + (int)threadIdx.x) * 4 < g.N)
#pragma unroll
            for (int e = 0; e < 4; e++) { v[p][e] -= mean; q = fmaf(v[p][e], v[p][e], q); }
    const float rstd = 1.f / sqrtf(over_row(q, 1) / (float)g.N + g.eps);
#pragma unroll
    for (int p = 0; p < PIECES; p++) {
        const int n = (p * 256 + (int)threadIdx.x) * 4;
        if (n >= g.N) continue;
        Pack4<T> o;
#pragma unroll
        for (int e = 0; e < 4; e++) o.v[e] = Elem<T>::from_f32(fmaf(v[p][e] * rstd, rounded<T>(ga[p][e]), rounded<T>(be[p][e])));
        *reinterpret_cast<u32x2*>(h + row * g.N + n) = __builtin_bit_cast(u32x2, o);
    }
}

// The workgroups that fetch g.ahead, in front of a launch's own.
void plan_ahead(LinearArgs& g) {
    g.first = 0;
    for (Band& a : g.ahead) {
        a.cols = ((a.N + 15) / 16 + kXcds - 1) / kXcds * 16;
        const int64_t pieces = (int64_t)a.cols / 4 * a.K, per_wg = 64 * kWaves * kAheadLoads;
        a.wgs = a.w ? (int)((pieces + per_wg - 1) / per_wg) : 0;
        a.magic = a.w ? (uint32_t)((((uint64_t)1 << 32) + a.cols / 4 - 1) / (a.cols / 4)) : 0;
        g.first += kXcds * a.wgs;
    }
}

template <typename T, bool TB, bool LOOP, int FORM, int MT, int U>
int launch_one(hipStream_t s, LinearArgs g) {
    auto kern = linear_w32_kernel<T, TB, LOOP, FORM, MT, U>;
    constexpr int kShares = kWaves * MT * 1024, kStats = FORM == kNorm ? 2 * kWaves * MT * 64 + 2 * kWaves * U * 32 * 4 : 0, kSums = kShares > kStats ? kShares : kStats;
    static_assert(kSums < 64 * 1024, "more LDS than a launch gets unasked");
    g.blocks = (g.M + 16 * MT - 1) / (16 * MT);
    g.strips = (g.N + 15) / 16;
    g.per_xcd = (g.strips + kXcds - 1) / kXcds;
    plan_ahead(g);
    g.part_steps = ((g.K + 31) / 32 + g.splits - 1) / g.splits;
    g.per = (g.part_steps + kWaves - 1) / kWaves;
    g.by_blocks = divisor(g.blocks);
    g.by_splits = divisor(g.splits);
    const int64_t grid = g.first + (int64_t)kXcds * g.per_xcd * g.blocks * g.splits;
    if (grid > 0x7FFFFFFFLL) return fail(MHIP_ERR_UNSUPPORTED, "linear_w32: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * kWaves), kSums, s, g);
    return check_launch("linear_w32");
}

template <typename T, int MT>
int launch_rows(hipStream_t s, const LinearArgs& g, bool tb) {
    const bool loop = ((g.K + 31) / 32 + g.splits - 1) / g.splits > 3 * kWaves;
    if (tb && !loop && !g.sums) {
        LinearArgs t = g;
        t.strips = (g.N + 15) / 16;
        const int blocks = (g.M + 16 * MT - 1) / (16 * MT), room = (MT < 2 ? 2 : 1) * compute_units() / blocks;
        hipLaunchKernelGGL((linear_w32_stream_kernel<T, MT, 3>), dim3((unsigned)(t.strips < room ? t.strips : room), (unsigned)blocks), dim3(64 * kWaves), 0, s, t);
        return check_launch("linear_w32_stream");
    }
    if (tb) return launch_one<T, true, true, kPlain, MT, 3>(s, g);
    if constexpr (MT <= 2) {
        if (g.gamma) return launch_one<T, false, false, kNorm, MT, 3>(s, g);
        if (g.words) return loop ? launch_one<T, false, true, kArrive, MT, 3>(s, g) : launch_one<T, false, false, kArrive, MT, 3>(s, g);
    }
    return loop ? launch_one<T, false, true, kPlain, MT, 3>(s, g) : launch_one<T, false, false, kPlain, MT, 3>(s, g);
}

template <typename T>
int launch_type(hipStream_t s, const LinearArgs& g, bool tb) {
    // blocks of up to 64 rows, of one size
    const int blocks = (g.M + 63) / 64;
    switch (((g.M + blocks - 1) / blocks + 15) / 16) {
        case 1: return launch_rows<T, 1>(s, g, tb);
        case 2: return launch_rows<T, 2>(s, g, tb);
        case 3: return launch_rows<T, 3>(s, g, tb);
        default: return launch_rows<T, 4>(s, g, tb);
    }
}

bool aligned16(std::initializer_list<const void*> ps) {
    uintptr_t all = 0;
    for (const void* p : ps) all |= reinterpret_cast<uintptr_t>(p);
    return (all & 15) == 0;
}

}  // namespace
}  // namespace mhip

using namespace mhip;

extern "C" int mhip_linear_w32_ok(int64_t M, int64_t N, int64_t K, int dtype) {
    if (dtype != MHIP_BF16 && dtype != MHIP_F16) return 0;
    if (M < 1 || M > 192 || N < 1 || K < 1 || N % 8 != 0 || K % 8 != 0 || N > (1 << 24) || K > (1 << 24)) return 0;
    // (x and w each inside one descriptor, whose last byte lies below kOob)
    return (N + 64) * (K + 64) * 4 < 0x7FFFFFFFLL && M * K * 2 < 0x7FFFFFFFLL;
}

// Parts of K: about 768 k, at most two workgroups per compute unit.
extern "C" int mhip_linear_w32_parts(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = (N + 15) / 16 * ((M + 63) / 64), room = tiles > 0 ? 512 / tiles : 1, want = (K + 384) / 768;
    const int64_t n = room < want ? room : want;
    return n < 2 ? 1 : n > 8 ? 8 : (int)n;
}

namespace mhip {
namespace {
// The matrices that can be fetched ahead; the others are left to the calls that read them.
void take_ahead(LinearArgs& g, int n_ahead, const mhip_weights* ahead) {
    for (int i = 0; i < n_ahead; i++)
        if (ahead[i].w && ahead[i].N > 0 && ahead[i].K > 0 && ahead[i].N % 8 == 0 && ahead[i].N <= (1 << 16) && ahead[i].K <= (1 << 16) &&
            ahead[i].N * ahead[i].K <= (1 << 23) && aligned16({ahead[i].w})) {
            g.ahead[i].w = ahead[i].w; g.ahead[i].N = (int)ahead[i].N; g.ahead[i].K = (int)ahead[i].K;
        }
}

// Heads a part of attend_project_kernel, 0 where it does not serve: a divisor of the heads of which up to four parts come, or eight where they are many;
// 64 rows, and a wave for every 32 of a head's.
int project_group(int64_t B, int64_t S, int64_t H) {
    if (B < 1 || S < 1 || H < 1 || H > 32 || S > 64 || B * S > 64) return 0;
    int group = 0;
    for (int n = 1; n <= 4 && !group; n++)
        if (H % n == 0 && H / n <= 4) group = n;
    if (!group && H % 4 == 0) group = 4;
    return group && group * B * ((S + 31) / 32) <= kWaves ? group : 0;
}

template <typename T, int MT>
int launch_project(hipStream_t s, const FaArgs& a, LinearArgs g, int group) {
    auto kern = attend_project_kernel<T, MT>;
    constexpr int kMost = kWaves * 64 * kProjectHead * 2 + 64 * (4 * kProjectHead * 2 + 16);
    static_assert(kWaves * MT * kProjectCols / 16 * 1024 <= kWaves * 64 * kProjectHead * 2, "the sums lie where the values were");
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMost); });
    if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "attend_project: cannot reserve %d bytes of LDS: %s", kMost, hipGetErrorString(err));
    const int lds = kWaves * 64 * kProjectHead * 2 + MT * 16 * (group * kProjectHead * 2 + 16);
    g.per_xcd = ((g.N + 15) / 16 + kXcds - 1) / kXcds;
    plan_ahead(g);
    g.by_splits = divisor(g.splits);
    g.by_blocks = divisor(a.B);
    const int64_t grid = g.first + (int64_t)kXcds * ((g.per_xcd + 1) / 2) * g.splits;
    if (grid > 0x7FFFFFFFLL) return fail(MHIP_ERR_UNSUPPORTED, "attend_project: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * kWaves), lds, s, a, g, group);
    return check_launch("attend_project");
}

template <typename T, int MT>
int launch_project_layer(hipStream_t s, const FaArgs& a, LinearArgs g) {
    auto kern = attend_project_layer_kernel<T, MT>;
    constexpr int kValues = kLayerRows * kProjectHead * 2, kMost = kLayerWaves * kValues + 16 * MT * (kLayerWaves * kProjectHead * 2 + 16);
    static_assert(MT * 1024 <= kValues, "the sums lie where the values were");
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMost); });
    if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "attend_project_layer: cannot reserve %d bytes of LDS: %s", kMost, hipGetErrorString(err));
    const int pairs = a.B * a.H, turns = (pairs + kLayerWaves - 1) / kLayerWaves, deal = (pairs + turns - 1) / turns;
    const int least = a.H < kWaves ? kWaves : a.H, waves = deal < least ? least : deal;      // (a wave for each head's rows of W; a workgroup in front is kWaves of them)
    g.strips = (g.N + 15) / 16;
    g.per_xcd = (g.strips + kXcds - 1) / kXcds;
    plan_ahead(g);
    g.by_blocks = divisor(a.B);
    hipLaunchKernelGGL(kern, dim3((unsigned)(g.first + kXcds * g.per_xcd)), dim3(64 * waves), waves * kValues + 16 * MT * (g.K * 2 + 16), s, a, g);
    return check_launch("attend_project_layer");
}

template <typename T>
int project_type(hipStream_t s, const FaArgs& a, const LinearArgs& g, int group) {
    switch ((g.M + 15) / 16) {
        case 1: return launch_project<T, 1>(s, a, g, group);
        case 2: return launch_project<T, 2>(s, a, g, group);
        case 3: return launch_project<T, 3>(s, a, g, group);
        default: return launch_project<T, 4>(s, a, g, group);
    }
}

int linear_entry(void* stream, const void* x, const float* w, const float* bias, const void* residual, void* c, int64_t M, int64_t N, int64_t K, int trans_b,
                 int activation, int dtype, const float* gamma, const float* beta, float eps, float* sums, uint64_t* words, int parts, int n_ahead,
                 const mhip_weights* ahead) {
    if (activation < MHIP_ACT_NONE || activation > MHIP_ACT_GELU_ERF)
        return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_linear_w32: unknown activation %d", activation);
    if (!x || !w || (!c && !sums)) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_linear_w32: NULL matrix pointer");
    if (sums && !words ? (parts < 1 || parts > 8 || c || bias || residual || activation != MHIP_ACT_NONE) : !words && parts != 1)
        return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_linear_w32: parts of K come as plain sums, eight at most");
    if (!mhip_linear_w32_ok(M, N, K, dtype))
        return fail(MHIP_ERR_UNSUPPORTED, "mhip_linear_w32: [%lld,%lld] x K %lld, dtype %d is not served", (long long)M, (long long)N, (long long)K, dtype);
    if (!aligned16({x, w, bias, residual, c, sums, gamma, beta})) return fail(MHIP_ERR_UNSUPPORTED, "mhip_linear_w32: tensors must be 16-byte aligned");
    if (n_ahead < 0 || n_ahead > kAhead || (n_ahead > 0 && !ahead)) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_linear_w32: up to %d matrices ahead", kAhead);
    LinearArgs g = {};
    g.x = x; g.w = w; g.bias = bias; g.residual = residual; g.c = c; g.sums = sums;
    g.M = (int)M; g.N = (int)N; g.K = (int)K; g.act = activation; g.splits = parts;
    g.gamma = gamma; g.beta = beta; g.eps = eps; g.words = words; g.tag = words ? launch_tag() : 0;
    take_ahead(g, n_ahead, ahead);
    return dtype == MHIP_BF16 ? launch_type<bf16_t>(as_stream(stream), g, trans_b != 0) : launch_type<f16_t>(as_stream(stream), g, trans_b != 0);
}

int64_t part_bytes(int64_t M, int64_t N, int parts) { return (parts * M * N * 4 + 255) / 256 * 256; }
}  // namespace
}  // namespace mhip

extern "C" int mhip_linear_w32(void* stream, const void* x, const float* w, const float* bias, const void* residual, void* c, int64_t M,
                               int64_t N, int64_t K, int trans_b, int activation, int dtype, float* sums, int parts, int n_ahead,
                               const mhip_weights* ahead) {
    return linear_entry(stream, x, w, bias, residual, c, M, N, K, trans_b, activation, dtype, nullptr, nullptr, 0.f, sums, nullptr, parts, n_ahead, ahead);
}

// Up to 32 rows: every workgroup normalises all of them, 10 operations an element, 0.7 us for 16 rows and 2.3 for 48.  GPT-2-small, us, so | normalised by finish_norm_kernel behind
// attend_project: 16 tokens 322 | 355, 17 363 | 358, 24 380 | 363, 32 399 | 368, 2 x 8 336 | 352, 2 x 12 392 | 365, 2 x 16 403 | 370; 3 x 5 342 | 400, 3 x 8 390 | 400, 4 x 8 402 | 404.
// The line is the one from before attend_project; from 17 rows on the other form is the faster one for one or two sequences.
extern "C" int mhip_linear_w32_norm_ok(int64_t M, int64_t N, int64_t K, int dtype) { return mhip_linear_w32_ok(M, N, K, dtype) && M <= 32 && K <= kWaves * 3 * 32; }

extern "C" int64_t mhip_linear_w32_workspace(int64_t M, int64_t N, int64_t K) {
    const int parts = mhip_linear_w32_parts(M, N, K);
    return parts == 1 || M < 1 || M > 32 ? 0 : part_bytes(M, N, parts) + (N + 15) / 16 * ((M + 63) / 64) * 8;
}

extern "C" int mhip_linear_w32_layer(void* stream, const void* x, const float* gamma, const float* beta, float eps, const float* w, const float* bias,
                                     const void* residual, void* c, int64_t M, int64_t N, int64_t K, int activation, int dtype, void* workspace,
                                     int64_t workspace_bytes, int n_ahead, const mhip_weights* ahead) {
    if (!c) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_linear_w32_layer: NULL result");
    if (gamma && !mhip_linear_w32_norm_ok(M, N, K, dtype))
        return fail(MHIP_ERR_UNSUPPORTED, "mhip_linear_w32_layer: rows of %lld are not normalised", (long long)K);
    // (normalised rows need all of K in a workgroup)
    const int64_t need = mhip_linear_w32_workspace(M, N, K);
    const bool split = !gamma && need > 0 && workspace && workspace_bytes >= need;
    const int parts = split ? mhip_linear_w32_parts(M, N, K) : 1;
    char* ws = static_cast<char*>(workspace);
    return linear_entry(stream, x, w, bias, residual, c, M, N, K, 0, activation, dtype, gamma, beta, eps, split ? reinterpret_cast<float*>(ws) : nullptr,
                        split ? reinterpret_cast<uint64_t*>(ws + part_bytes(M, N, parts)) : nullptr, parts, n_ahead, ahead);
}

extern "C" int mhip_finish_norm(void* stream, const float* sums, int parts, const float* bias, const void* residual, void* c,
                                const float* gamma, const float* beta, float eps, void* h, int64_t M, int64_t N, int dtype) {
    if (M < 0 || N < 1 || parts < 0 || (parts > 0) != (sums != nullptr) || !gamma || !h || (parts == 0 && !residual))
        return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_finish_norm: bad argument");
    if (M == 0) return MHIP_OK;
    if ((dtype != MHIP_BF16 && dtype != MHIP_F16) || N % 8 != 0 || N > 1024 * kFinishPieces || M > 0x7FFFFFFF || !aligned16({sums, bias, residual, c, gamma, beta, h}))
        return fail(MHIP_ERR_UNSUPPORTED, "mhip_finish_norm: rows of %lld, dtype %d", (long long)N, dtype);
    LinearArgs g = {};
    g.sums = const_cast<float*>(sums); g.splits = parts; g.bias = bias; g.residual = residual; g.c = c; g.gamma = gamma; g.beta = beta;
    g.eps = eps; g.M = (int)M; g.N = (int)N;
    auto launch = [&](auto* to, auto pieces) {
        hipLaunchKernelGGL((finish_norm_kernel<std::remove_pointer_t<decltype(to)>, decltype(pieces)::value>), dim3((unsigned)M), dim3(256), 0, as_stream(stream), g, to);
    };
    auto type = [&](auto* to) {
        if (N <= 1024) launch(to, std::integral_constant<int, 1>{});
        else launch(to, std::integral_constant<int, kFinishPieces>{});
    };
    if (dtype == MHIP_BF16) type(static_cast<bf16_t*>(h));
    else type(static_cast<f16_t*>(h));
    return check_launch("finish_norm");
}

extern "C" int mhip_attend_project_parts(int64_t B, int64_t S, int64_t H, int64_t D, int64_t N, int dtype) {
    const int group = D == kProjectHead && (dtype == MHIP_BF16 || dtype == MHIP_F16) && N >= 1 && N % 8 == 0 ? project_group(B, S, H) : 0;
    return group && (N + 64) * H * D * 4 < 0x7FFFFFFFLL ? (int)H / group : 0;
}

namespace mhip {
namespace {
// The operands of causal attention over a projection [B S, 3 H D], and its product with W.
void project_args(FaArgs& a, LinearArgs& g, const void* qkv, const float* w, int64_t B, int64_t S, int64_t H, int64_t D, int64_t N) {
    const int64_t d = H * D;
    a.q = qkv;
    a.k = static_cast<const char*>(qkv) + d * 2;
    a.v = static_cast<const char*>(qkv) + 2 * d * 2;
    a.B = (int)B; a.H = (int)H; a.Sq = a.Skv = (int)S; a.D = (int)D;
    a.scale = (float)(1.0 / sqrt((double)D));
    a.c = a.scale * kLog2e;
    a.is_causal = 1;
    for (int64_t* st : {a.qs, a.ks, a.vs}) { st[0] = S * 3 * d; st[1] = D; st[2] = 3 * d; }
    g.w = w;
    g.M = (int)(B * S); g.N = (int)N; g.K = (int)d;
}
}  // namespace
}  // namespace mhip

// Two turns of the waves up to 16 rows only (GPT-2-small, in one launch and in two: 2 x 4 tokens 324 and 334 us, 2 x 8 336 and 344, 2 x 12 395 and 392, 2 x 16 413 and 404; past 16
// rows the form with finish_norm is faster than both, see mhip_linear_w32_norm_ok).
extern "C" int mhip_attend_project_layer_ok(int64_t B, int64_t S, int64_t H, int64_t D, int64_t N, int dtype) {
    if (D != kProjectHead || (dtype != MHIP_BF16 && dtype != MHIP_F16) || N < 1 || N % 8 != 0 || N > (1 << 24)) return 0;
    if (B < 1 || H < 1 || S < 1 || B > kLayerRows || H > kLayerWaves || S > kLayerRows || B * H > (B * S <= 16 ? 2 : 1) * kLayerWaves || B * S > kLayerRows) return 0;
    return (N + 64) * H * D * 4 < 0x7FFFFFFFLL;
}

extern "C" int mhip_attend_project_layer(void* stream, const void* qkv, const float* w, const float* bias, const void* residual, void* c, int64_t B, int64_t S, int64_t H,
                                         int64_t D, int64_t N, int dtype, int n_ahead, const mhip_weights* ahead) {
    if (!qkv || !w || !c) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_attend_project_layer: NULL pointer");
    if (n_ahead < 0 || n_ahead > kAhead || (n_ahead > 0 && !ahead)) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_attend_project_layer: up to %d matrices ahead", kAhead);
    if (!mhip_attend_project_layer_ok(B, S, H, D, N, dtype) || !aligned16({qkv, w, bias, residual, c}))
        return fail(MHIP_ERR_UNSUPPORTED, "mhip_attend_project_layer: [%lld,%lld], %lld heads of %lld, %lld columns, dtype %d, or pointers off 16 bytes", (long long)B,
                    (long long)S, (long long)H, (long long)D, (long long)N, dtype);
    FaArgs a = {};
    LinearArgs g = {};
    project_args(a, g, qkv, w, B, S, H, D, N);
    g.bias = bias; g.residual = residual; g.c = c;
    take_ahead(g, n_ahead, ahead);
    const hipStream_t s = as_stream(stream);
    if (g.M <= 16) return dtype == MHIP_BF16 ? launch_project_layer<bf16_t, 1>(s, a, g) : launch_project_layer<f16_t, 1>(s, a, g);
    return dtype == MHIP_BF16 ? launch_project_layer<bf16_t, 2>(s, a, g) : launch_project_layer<f16_t, 2>(s, a, g);
}

extern "C" int mhip_attend_project(void* stream, const void* qkv, const float* w, float* sums, int64_t B, int64_t S, int64_t H, int64_t D, int64_t N, int dtype,
                                   int n_ahead, const mhip_weights* ahead) {
    if (!qkv || !w || !sums) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_attend_project: NULL pointer");
    if (n_ahead < 0 || n_ahead > kAhead || (n_ahead > 0 && !ahead)) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_attend_project: up to %d matrices ahead", kAhead);
    const int parts = mhip_attend_project_parts(B, S, H, D, N, dtype);
    if (!parts || !aligned16({qkv, w, sums}))
        return fail(MHIP_ERR_UNSUPPORTED, "mhip_attend_project: [%lld,%lld], %lld heads of %lld, %lld columns, dtype %d, or pointers off 16 bytes", (long long)B,
                    (long long)S, (long long)H, (long long)D, (long long)N, dtype);
    FaArgs a = {};
    LinearArgs g = {};
    project_args(a, g, qkv, w, B, S, H, D, N);
    g.sums = sums; g.splits = parts;
    take_ahead(g, n_ahead, ahead);
    return dtype == MHIP_BF16 ? project_type<bf16_t>(as_stream(stream), a, g, (int)H / parts) : project_type<f16_t>(as_stream(stream), a, g, (int)H / parts);
}
