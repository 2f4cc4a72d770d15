// dot_general with few rows: C = act(A . op(B) + bias) (+ residual) for M <= 64, fp32 also in blocks of rows up
// to 192 (a decode step, a short prompt, a small batch), where the product costs nothing and the time is that of reading B once.
//
// A tile kernel leaves such a problem on a handful of workgroups ([4,4096] x [4096,4096]: 32 tiles of
// 128 columns on 256 compute units, each walking K through LDS one load latency at a time).  Here
//   * a workgroup owns a strip of 16 to 64 columns and ALL of K, its waves split K between them: every wave
//     has a block of loads in flight from its first instruction on, and the partial sums meet in LDS;
//   * B goes from memory straight to the operand registers, no LDS, no barrier in the loop.  The matrix
//     instruction wants eight consecutive k of one column per lane.  Stored [N, K] that is one 16-byte
//     load.  Stored [K, N] a lane loads VE neighbouring columns of its eight k rows, and one byte
//     permute per register pairs two k of one column: lane i then owns columns VE*i .. VE*i + VE-1 of the
//     strip, one per operand f, which only changes where the results go;
//   * the product is formed transposed (B as first operand), rows of A beyond M are duplicates of the last
//     row whose results are dropped, k beyond K reads zero through the buffer bounds.
// fp32 operands take the same path on v_mfma_f32_16x16x4_f32; operands whose rows are not aligned for
// vector loads (odd K or N) load element by element (VEC = false), still with every load in flight.
#include <mutex>

#include "arrive.h"

namespace mhip {

bool gemm_strip_wanted(int64_t M, int64_t N, int64_t K, int64_t batch, int trans_b);          // gemm_strip.hip
int launch_gemm_strip(hipStream_t s, const GemmArgs& g, int64_t batch, int dtype);

namespace {

template <typename T> struct Mfma16;
template <> struct Mfma16<bf16_t> {
    static constexpr int kKpl = 8;                   // consecutive k per lane and operand
    typedef u32x4 frag;
    __device__ static f32x4 run(frag b, frag a, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
    }
};
template <> struct Mfma16<f16_t> {
    static constexpr int kKpl = 8;
    typedef u32x4 frag;
    __device__ static f32x4 run(frag b, frag a, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, b), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
    }
};
template <> struct Mfma16<float> {
    static constexpr int kKpl = 4;                   // four issues of k = 4: lane group g supplies k = 4 g + p to issue p
    typedef u32x4 frag;
    __device__ static f32x4 run(frag b, frag a, f32x4 c) {
#pragma unroll
        for (int p = 0; p < 4; p++)
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(f32x4, b)[p], __builtin_bit_cast(f32x4, a)[p], c, 0, 0, 0);
        return c;
    }
};

__device__ inline __amdgpu_buffer_rsrc_t skinny_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// 16 bytes of consecutive elements at element offset `off` of which `n` exist (n <= 0: none).
template <typename T, bool VEC>
__device__ inline u32x4 load_run(__amdgpu_buffer_rsrc_t r, int64_t off, int n) {
    if (VEC) return __builtin_amdgcn_raw_buffer_load_b128(r, n > 0 ? (uint32_t)(off * (int)sizeof(T)) : kOob, 0, 0);
    u32x4 v;
    if (sizeof(T) == 4) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = __builtin_amdgcn_raw_buffer_load_b32(r, e < n ? (uint32_t)((off + e) * 4) : kOob, 0, 0);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t lo = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, 2 * e < n ? (uint32_t)((off + 2 * e) * 2) : kOob, 0, 0);
            const uint32_t hi = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, 2 * e + 1 < n ? (uint32_t)((off + 2 * e + 1) * 2) : kOob, 0, 0);
            v[e] = lo | (hi << 16);
        }
    }
    return v;
}

// VE consecutive elements (as dwords; one 16-bit pair per dword) of one row of B stored [K, N].
template <typename T, int VE, bool VEC> struct RowPiece {
    static constexpr int kDw = (int)(VE * sizeof(T) / 4);
    uint32_t w[kDw];
    __device__ void load(__amdgpu_buffer_rsrc_t r, int64_t off, int n) {
        if (VEC) {
            const uint32_t o = n > 0 ? (uint32_t)(off * (int)sizeof(T)) : kOob;
            if (kDw == 1) w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0);
            else if (kDw == 3) {
                const auto t = __builtin_amdgcn_raw_buffer_load_b96(r, o, 0, 0);
                w[0] = t[0]; w[1 % kDw] = t[1]; w[kDw - 1] = t[2];
            } else {
                const u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0);
                w[0] = t.x; w[kDw - 1] = t.y;
            }
        } else if (sizeof(T) == 4) {
#pragma unroll
            for (int e = 0; e < kDw; e++) w[e] = __builtin_amdgcn_raw_buffer_load_b32(r, e < n ? (uint32_t)((off + e) * 4) : kOob, 0, 0);
        } else {
#pragma unroll
            for (int e = 0; e < kDw; e++) {
                const uint32_t lo = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, 2 * e < n ? (uint32_t)((off + 2 * e) * 2) : kOob, 0, 0);
                const uint32_t hi = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, 2 * e + 1 < n ? (uint32_t)((off + 2 * e + 1) * 2) : kOob, 0, 0);
                w[e] = lo | (hi << 16);
            }
        }
    }
};

// Whether neighbouring strips go to one XCD: rows of a strip that are half a line or less, whose other half the same L2 then holds for the
// neighbour.  us, without | with: [1,6720] x K 832 bf16 5.9 | 5.0, [8,1024] x K 4096 bf16 9.3 | 8.8, [16,6720] x K 832 fp32
// 10.4 | 9.0; strips of 128 or 192 bytes lose by it, [4,4096] x K 4096 bf16 11.0 | 11.3, [128,3072] x K 768 fp32 11.5 | 12.0, and
// so do blocks of 32 fp32 rows, [100,512] x K 2048 11.8 | 12.2, [190,256] x K 2048 12.0 | 12.6.
template <typename T, bool TB, int NF, int MT>
constexpr bool strip_order() { return !TB && 16 * NF * (int)sizeof(T) < 128 && (sizeof(T) == 2 || MT == 1); }

// NF = operands (groups of 16 columns) per strip, MT = groups of 16 rows, U = k steps loaded as one block.  PARTS: K is split over the grid too,
// a kernel of its own: compiled into the others the arrivals cost up to 8 %, [128,768] x K 768 fp32 6.9 -> 7.5 us.
template <typename T, bool TB, bool VEC, int NF, int MT, int U, int WAVES, bool PARTS>
__global__ __launch_bounds__(64 * WAVES) void gemm_skinny_kernel(GemmArgs g) {
    constexpr int KPL = Mfma16<T>::kKpl, KS = 4 * KPL;      // k per step
    constexpr int VE = NF, NS = 16 * NF;                     // (stored [K, N]: NF consecutive columns per lane)
    constexpr int kDw = (int)(VE * sizeof(T) / 4);
    extern __shared__ __attribute__((aligned(16))) float part[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int strip = strip_order<T, TB, NF, MT>() ? (int)(blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds) : (int)blockIdx.x, n0 = strip * NS;
    if (strip_order<T, TB, NF, MT>() && n0 >= g.N) return;
    int batch_i = blockIdx.y, m0 = 0;
    if (g.tiles_m > 1) { m0 = batch_i % g.tiles_m * (16 * MT); batch_i /= g.tiles_m; }
    const int64_t batch = batch_i;
    const T* a = static_cast<const T*>(g.a) + batch * g.sa;
    const T* b = static_cast<const T*>(g.b) + batch * g.sb;
    const __amdgpu_buffer_rsrc_t ra = skinny_rsrc(a, (uint32_t)((int64_t)g.M * g.lda * sizeof(T)));
    const __amdgpu_buffer_rsrc_t rb = skinny_rsrc(b, (uint32_t)((int64_t)(TB ? g.N : g.K) * g.ldb * sizeof(T)));

    uint64_t* const word = PARTS ? g.words + (int64_t)blockIdx.y * gridDim.x + blockIdx.x : nullptr;
    uint64_t seen = 0;
    if (PARTS && threadIdx.x == 0) seen = arrive_look(word);
    // this workgroup's k steps (all of them, or one split's), and this wave's share of them
    const int all_steps = (g.K + KS - 1) / KS, per_split = (all_steps + (int)gridDim.z - 1) / (int)gridDim.z;
    const int first = (int)blockIdx.z * per_split, steps = min(all_steps - first, per_split), per = (steps + waves - 1) / waves;
    const int s0 = first + wave * per, s1 = min(first + steps, s0 + per);
    const int kend = min(g.K, s1 * KS);

    uint32_t arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) arow[mt] = (uint32_t)(min(m0 + mt * 16 + li, g.M - 1) * g.lda);

    f32x4 acc[NF][MT];
#pragma unroll
    for (int f = 0; f < NF; f++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[f][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

    struct Block {
        u32x4 a[U][MT];
        u32x4 bt[TB ? U : 1][NF];                            // B stored [N, K]
        RowPiece<T, VE, VEC> bn[TB ? 1 : U][KPL];            // B stored [K, N]
    };
    auto load = [&](Block& blk, int s) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = (s + u) * KS + lg * KPL;
            if (TB) {
#pragma unroll
                for (int f = 0; f < NF; f++) {
                    const int n = n0 + 16 * f + li;
                    blk.bt[TB ? u : 0][f] = load_run<T, VEC>(rb, (int64_t)n * g.ldb + k, n < g.N ? kend - k : 0);
                }
            } else {
                const int n = n0 + VE * li;
#pragma unroll
                for (int j = 0; j < KPL; j++)
                    blk.bn[TB ? 0 : u][j].load(rb, (int64_t)(k + j) * g.ldb + n, k + j < kend ? g.N - n : 0);
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) blk.a[u][mt] = load_run<T, VEC>(ra, (int64_t)arow[mt] + k, kend - k);
        }
    };
    auto multiply = [&](const Block& blk) {
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int f = 0; f < NF; f++) {
                u32x4 bf;
                if (TB) bf = blk.bt[TB ? u : 0][f];
                else if (sizeof(T) == 4) {
#pragma unroll
                    for (int j = 0; j < 4; j++) bf[j] = blk.bn[TB ? 0 : u][j].w[f < kDw ? f : 0];
                } else {
                    // column f of rows 2j and 2j + 1 as one register: bytes of the second operand are 0..3
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        bf[j] = __builtin_amdgcn_perm(blk.bn[TB ? 0 : u][(2 * j + 1) % KPL].w[(f / 2) % kDw], blk.bn[TB ? 0 : u][(2 * j) % KPL].w[(f / 2) % kDw],
                                                      (f & 1) ? 0x07060302u : 0x05040100u);
                }
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[f][mt] = Mfma16<T>::run(bf, blk.a[u][mt], acc[f][mt]);
            }
        }
    };
    if (s0 < s1) {
        Block cur;
        load(cur, s0);
        for (int s = s0; s < s1; s += U) {
            Block nxt;
            if (s + U < s1) load(nxt, s + U);
            multiply(cur);
            if (s + U < s1) cur = nxt;
        }
    }

    if (PARTS && threadIdx.x == 0) arrive_claim(word, seen, g.tag);
    // ---- the waves' partial sums, in the accumulators' own layout: lane (li, lg) holds row 16 mt + li and,
    // in its four registers, operand rows 4 lg .. 4 lg + 3
#pragma unroll
    for (int f = 0; f < NF; f++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
            *reinterpret_cast<f32x4*>(part + (((wave * NF + f) * MT + mt) * 64 + lane) * 4) = acc[f][mt];
    __syncthreads();
    const T* bias = static_cast<const T*>(g.bias);
    const T* res = g.residual ? static_cast<const T*>(g.residual) + batch * g.sc : nullptr;
    T* c = static_cast<T*>(g.c) + batch * g.sc;
    const int total = min(g.M - m0, 16 * MT) * NS;
    auto sum_of = [&](int m, int nl) {
        const int f = TB ? nl / 16 : nl % VE, i = TB ? nl % 16 : nl / VE;
        const float* p = part + ((f * MT + m / 16) * 64 + (i >> 2) * 16 + (m & 15)) * 4 + (i & 3);
        float v = 0.f;
        for (int w = 0; w < waves; w++) v += p[w * (NF * MT * 256)];
        return v;
    };
    if constexpr (PARTS) {
        // one split's sums; the last split to arrive goes on with all of them
        for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
            const int m = idx / NS, nl = idx % NS;
            if (n0 + nl < g.N) store_part(g.partial + ((int64_t)blockIdx.z * g.M + m0 + m) * g.N + n0 + nl, sum_of(m, nl));
        }
        // (the flag where the sums were, which nobody reads behind the arrival's barrier: a word beside 64 KB is more than a launch gets unasked)
        if (!arrive_last(word, (int)gridDim.z, reinterpret_cast<int*>(part))) return;
    }
    auto finish = [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
        for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
            const int m = idx / NS, nl = idx % NS, n = n0 + nl;
            if (n >= g.N) continue;
            const int64_t at = (int64_t)(m0 + m) * g.N + n;
            float v = 0.f;
            if (PARTS) {
                const int64_t mn = (int64_t)g.M * g.N;
                float t[8];                                  // (eight splits at most, their loads in flight together)
#pragma unroll
                for (int s = 0; s < 8; s++) t[s] = load_part(g.partial + min(s, (int)gridDim.z - 1) * mn + at);
#pragma unroll
                for (int s = 0; s < 8; s++) if (s < (int)gridDim.z) v += t[s];
            } else v = sum_of(m, nl);
            if (bias) v += Elem<T>::to_f32(bias[n]);
            v = sizeof(T) == 4 ? apply_act(v, ACT) : apply_act_c<ACT>(v);
            T o = Elem<T>::from_f32(v);
            // (second rounding on purpose: the same result as a separate add over the stored C)
            if (res) o = Elem<T>::from_f32(Elem<T>::to_f32(o) + Elem<T>::to_f32(res[at]));
            c[at] = o;
        }
    };
    dispatch_act(g.act, finish);
}

template <typename T, bool TB, bool VEC, int NF, int MT, int U, bool PARTS>
int launch_kernel(hipStream_t s, GemmArgs g, int64_t batch) {
    constexpr int KS = 4 * Mfma16<T>::kKpl, WAVES = 8;
    auto kern = gemm_skinny_kernel<T, TB, VEC, NF, MT, U, WAVES, PARTS>;
    constexpr int kLds = WAVES * NF * MT * 1024;
    if (kLds > 64 * 1024) {
        static std::once_flag once;
        static hipError_t err = hipSuccess;
        std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds); });
        if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "gemm: cannot reserve %d bytes of LDS: %s", kLds, hipGetErrorString(err));
    }
    // a wave takes at least one block of loads
    const int steps = ((g.K + KS - 1) / KS + g.splits - 1) / g.splits, want = (steps + U - 1) / U;
    const int waves = want < 1 ? 1 : want > WAVES ? WAVES : want;
    const int64_t strips = (g.N + 16 * NF - 1) / (16 * NF);
    g.tiles_m = (g.M + 16 * MT - 1) / (16 * MT);
    const int64_t grid = strip_order<T, TB, NF, MT>() ? (strips + kXcds - 1) / kXcds * kXcds : strips;
    if (grid > 0x7FFFFFFFLL || batch * g.tiles_m > 65535) return fail(MHIP_ERR_UNSUPPORTED, "gemm: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)grid, (unsigned)(batch * g.tiles_m), (unsigned)g.splits), dim3(64 * waves), waves * NF * MT * 1024, s, g);
    return check_launch("gemm_skinny");
}

template <typename T, bool TB, bool VEC, int NF, int MT, int U>
int launch_one(hipStream_t s, const GemmArgs& g, int64_t batch) {
    return g.splits > 1 ? launch_kernel<T, TB, VEC, NF, MT, U, true>(s, g, batch) : launch_kernel<T, TB, VEC, NF, MT, U, false>(s, g, batch);
}

// Strip width: narrow strips put a small weight matrix on as many compute units as it has columns for, wide
// ones read whole 128-byte lines per row.  Stored [K, N], us narrow / wide: [4,4096] x [4096,4096] 14.4 / 13.0,
// [4,3072] x [3072,768] 5.8 / 9.4.  Stored [N, K] every strip reads whole lines and the wide one only saves reads
// of A: [16,8192] x [8192,16384] 67.7 / 62.9, [4,768] x [768,50304] 16.1 / 17.4.
bool wide_strips(int64_t N, int64_t K, int64_t batch, bool tb) {
    const int64_t strips = (N + 63) / 64 * batch;
    return tb ? strips >= 128 && K >= 2048 : strips >= 128 || (strips >= 64 && K >= 2048);
}

// K split over the grid as well (fp32 sums in a workspace, added up by the last split of a block to arrive: 2 to 3 us less than by a launch
// of its own, with which the lines below were drawn; fp32 [4,1024] x K 4096 12.3 -> 9.7, [64,768] x K 3072 12.5 -> 10.5): parts of about 1024 k, at most one
// workgroup per compute unit.  From which K on that pays for the launch was swept with weights from memory, M 1 to 64, N 256 to
// 4096; time in parts over time whole, the range over N:
//   16-bit [K, N], up to 32 rows   K 2048 0.86 to 1.26   K 2560 0.71 to 1.02   K 3064 0.66 to 0.96
//   16-bit [N, K], up to 16 rows   K 2560 1.02 to 1.31   K 3064 1.12 to 1.39   K 3584 0.85 to 1.18   (whole lines: it is the shorter
//   16-bit [N, K], 32 rows         K 2048 1.05           K 2560 0.88 to 0.99   K 3064 0.87 to 0.98    product to begin with)
//   fp32, up to 32 rows            K 2048 0.82 to 1.31   K 2560 0.70 to 1.08   K 3064 0.66 to 1.02
//   fp32, 64 rows                  K 2560 0.87 to 1.38   K 3064 0.82 to 1.26   K 3584 0.69 to 1.14
// Blocks of more than 64 rows (fp32) fill the device earlier ([128,3072] x [3072,768] 16.4 us whole, 20.5) and keep 2048 k.
//
// fp32 of 33 to 64 rows from K 3000 on, of more from K 3500 on: the block, 16 x 48 or 32 x 32, whose number times the parts comes
// closest to one workgroup per compute unit, if that leaves few of them idle.  us, before | 16 x 48 / parts (workgroups) | 32 x 32 / parts:
//   [48,768] x K 3072  15.2 | 11.9 / 4 (192) | 13.1 / 4 (192)      [128,1024] x K 4096 24.3 | 24.6 / 1 (176) | 19.8 / 2 (256)
//   [64,1024] x K 4096 17.0 | -              | 14.8 / 4 (256)      [70,1024] x K 4096  23.4 | 21.8 / 2 (220) | 19.7 / 2 (192)
// Shorter: [40,2048] x K 2048 12.3 | 14.4, [60,3000] x K 2500 22.4 | 24.1, [150,512] x K 2048 11.9 | 12.6, [128,768] x K 3072 16.6 | 15.1
// (all of these with a launch of its own for the parts, when the lines were drawn); below 216 workgroups: [160,640] x K 2560 15.0 whole | - | 15.9 / 2 (200).
struct RowsPlan { int rows = 0, cols = 0, splits = 1; };
RowsPlan rows_plan(int64_t M, int64_t N, int64_t K, int64_t batch, bool tb) {
    RowsPlan best;
    if (batch != 1 || M <= 32 || K < (M <= 64 ? 3000 : 3500)) return best;
    int64_t most = 215;
    auto consider = [&](int rows, int cols) {
        const int64_t blocks = (M + rows - 1) / rows * ((N + cols - 1) / cols), room = 256 / blocks, parts = room < K / 512 ? room : K / 512;
        const int64_t s = parts > 8 ? 8 : parts;
        if (s >= 2 && blocks * s > most) { most = blocks * s; best.rows = rows; best.cols = cols; best.splits = (int)s; }
    };
    if (!tb && K % 4 == 0 && N % 4 == 0) consider(16, 48);
    consider(32, 32);
    return best;
}

// (The strip kernel, which holds all of K, takes 16-bit operands on 16 bytes only: `vec`.  Others of its sizes are split: [8,256] x K 4096 two
// bytes off 48.9 us whole, 17.5.)
int skinny_splits(int64_t M, int64_t N, int64_t K, int64_t batch, int trans_b, bool is16, bool vec) {
    if (batch != 1 || M * N > (1 << 20) || (is16 && vec && gemm_strip_wanted(M, N, K, batch, trans_b))) return 1;
    if (!is16 && rows_plan(M, N, K, batch, trans_b != 0).splits > 1) return rows_plan(M, N, K, batch, trans_b != 0).splits;
    const int64_t width = wide_strips(N, K, 1, trans_b != 0) ? (trans_b ? 32 : 64) : (trans_b ? 16 : 32);
    const int64_t from = is16 ? (trans_b && M <= 16 ? 3584 : 2560) : (M > 32 ? 3072 : 2560);
    const int64_t want = M > 64 ? K / 2048 + (K % 2048 > 1024) : K >= from ? (K + 512) / 1024 : 1;
    const int64_t room = 256 / ((N + width - 1) / width), n = room < want ? room : want;
    return n < 2 ? 1 : n > 8 ? 8 : (int)n;
}

template <typename T, bool TB, bool VEC>
int launch_shape(hipStream_t s, const GemmArgs& g, int64_t batch) {
    constexpr bool k16 = sizeof(T) == 2;
    const bool wide = wide_strips(g.N, g.K, batch, TB);
    if constexpr (!k16) {
        // fp32 from 33 rows on: the block of rows by columns that leaves no compute unit a second turn, since a unit takes about 30
        // bytes a nanosecond of a matrix from memory; beyond that 32 by 32, unless the strips are wide, whose blocks of 64 rows
        // read B half as often.  Weights from memory, us (workgroups):
        //                        32 x 16       16 x 48       32 x 32       32 x 48
        //   [128,768] x K 768      7.0 (192)     8.0 (128)     9.3 (96)     11.2 (64)
        //   [100,1536] x K 512     7.9 (384)     6.5 (224)     7.4 (192)     8.9 (128)
        //   [64,3072] x K 1024    12.9 (384)     9.7 (256)    11.0 (192)    13.4 (128)
        //   [192,768] x K 3072    28.6 (288)    19.0 (192)    22.4 (144)    28.3 (96)
        //   [100,2048] x K 512     8.0 (512)    10.1 (301)     7.5 (256)     9.7 (172)
        //   [128,2304] x K 768    13.6 (576)    11.8 (384)    13.9 (288)    11.3 (192)
        //   [128,3072] x K 1024   17.2 (768)    14.9 (512)    17.4 (384)    13.5 (256)
        //   [192,2304] x K 768    16.5 (864)    16.3 (576)    14.4 (432)    17.5 (288)
        // Wide: [64,8192] x K 4096 59.1 in 32 x 32, 52.3 in 64 rows.  Up to 64 rows a split K fills the device as it is:
        // [36,768] x K 8192 24.4 in 32 x 16, 20.8 in 64 rows.  (Stored [K, N] a strip of 48 columns is three per lane.)
        const RowsPlan plan = rows_plan(g.M, g.N, g.K, batch, TB);
        if (g.splits > 1 && plan.splits == g.splits) {
            if constexpr (VEC && !TB) if (plan.cols == 48) return launch_one<T, TB, VEC, 3, 1, 2>(s, g, batch);
            return launch_one<T, TB, VEC, 2, 2, 2>(s, g, batch);
        }
        if (g.M > 32 && (g.M > 64 || g.splits == 1)) {
            auto blocks = [&](int rows, int cols) { return (int64_t)((g.M + rows - 1) / rows) * ((g.N + cols - 1) / cols) * batch; };
            constexpr bool k48 = VEC && !TB;
            if (blocks(32, 16) <= 256) return launch_one<T, TB, VEC, 1, 2, 2>(s, g, batch);
            // (48 columns where rows start on lines: [60,3000] x K 2500 22.5 in 32 x 32, 24.1)
            if constexpr (k48) if (g.N % 32 == 0 && blocks(16, 48) <= 256) return launch_one<T, TB, VEC, 3, 1, 2>(s, g, batch);
            if constexpr (k48) if (g.N % 32 == 0 && blocks(32, 32) > 256 && blocks(32, 48) <= 256) return launch_one<T, TB, VEC, 3, 2, 2>(s, g, batch);
            if (!wide) return launch_one<T, TB, VEC, 2, 2, 2>(s, g, batch);
        }
    }
    if (g.M <= 16) {
        if (wide) return k16 || TB ? launch_one<T, TB, VEC, TB ? 2 : 4, 1, 2>(s, g, batch) : launch_one<T, TB, VEC, 2, 1, 2>(s, g, batch);
        return launch_one<T, TB, VEC, TB ? 1 : k16 ? 2 : 1, 1, 4>(s, g, batch);
    }
    // (16-bit rows without vector alignment: gemm_any.hip takes them from 17 rows on)
    if constexpr (k16 && !VEC) return fail(MHIP_ERR_UNSUPPORTED, "gemm: more than 16 unaligned rows");
    else {
        if (g.M <= 32) {
            if (wide) return k16 || TB ? launch_one<T, TB, VEC, TB ? 2 : 4, 2, 2>(s, g, batch) : launch_one<T, TB, VEC, 2, 2, 2>(s, g, batch);
            return launch_one<T, TB, VEC, TB ? 1 : k16 ? 2 : 1, 2, 2>(s, g, batch);
        }
        // 33 to 64 rows of a small 16-bit weight matrix: two blocks of 32 rows (one of 64 takes 8.2 us where they take 6.7)
        if constexpr (k16) return launch_one<T, TB, VEC, TB ? 1 : 2, 2, 2>(s, g, batch);
        else {
            if (wide) return launch_one<T, TB, VEC, 2, 4, 1>(s, g, batch);
            return launch_one<T, TB, VEC, 1, 4, 2>(s, g, batch);
        }
    }
}

bool on_16_bytes(const GemmArgs& g, int dtype) {
    const int per16 = dtype == MHIP_F32 ? 4 : 8;
    return g.lda % per16 == 0 && g.ldb % per16 == 0 && g.sa % per16 == 0 && g.sb % per16 == 0 &&
           ((reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b)) & 15) == 0;
}

int dtype_launch(hipStream_t s, const GemmArgs& g, int64_t batch, int trans_b, int dtype) {
    const bool vec = on_16_bytes(g, dtype);
    if (vec && dtype != MHIP_F32 && gemm_strip_wanted(g.M, g.N, g.K, batch, trans_b)) return launch_gemm_strip(s, g, batch, dtype);
#define MHIP_SKINNY(T)                                                                                              \
    (vec ? (trans_b ? launch_shape<T, true, true>(s, g, batch) : launch_shape<T, false, true>(s, g, batch))         \
         : (trans_b ? launch_shape<T, true, false>(s, g, batch) : launch_shape<T, false, false>(s, g, batch)))
    switch (dtype) {
        case MHIP_F32: return MHIP_SKINNY(float);
        case MHIP_BF16: return MHIP_SKINNY(bf16_t);
        default: return MHIP_SKINNY(f16_t);
    }
#undef MHIP_SKINNY
}

}  // namespace

// What this kernel takes: A stored [M, K], at most 64 rows (fp32: 192, in blocks), operands that one buffer descriptor spans.
bool gemm_skinny_eligible(const GemmArgs& g, int trans_a, int elem_bytes) {
    return !trans_a && g.M <= (elem_bytes == 4 ? 192 : 64) && g.K > 0 && g.ldc == 0 && (int64_t)g.M * g.lda * elem_bytes < 0x7FFFFFFFLL &&
           ((int64_t)g.N + 64) * g.K * elem_bytes < 0x7FFFFFFFLL && ((int64_t)g.K + 64) * g.N * elem_bytes < 0x7FFFFFFFLL;
}

// The splits' sums, and a word for each block of at least 16 columns and 16 rows (strips in multiples of eight).
static int64_t parts_bytes(int64_t M, int64_t N, int n) { return (M * N * 4 * n + 255) / 256 * 256; }
static int64_t words_bytes(int64_t M, int64_t N) { return ((N + 15) / 16 + kXcds) * ((M + 15) / 16) * 8; }
int64_t gemm_skinny_workspace(int64_t M, int64_t N, int64_t K, int64_t batch, int trans_b, bool is16) {
    // (from the sizes: the pointers may lie anywhere)
    const int n = skinny_splits(M, N, K, batch, trans_b, is16, false);
    return n == 1 ? 0 : parts_bytes(M, N, n) + words_bytes(M, N);
}

int launch_gemm_skinny(hipStream_t s, GemmArgs g, int64_t batch, int trans_b, int dtype, int64_t workspace_bytes) {
    g.splits = g.partial ? skinny_splits(g.M, g.N, g.K, batch, trans_b, dtype != MHIP_F32, on_16_bytes(g, dtype)) : 1;
    if (g.splits > 1 && parts_bytes(g.M, g.N, g.splits) + words_bytes(g.M, g.N) > workspace_bytes) g.splits = 1;
    if (g.splits == 1) g.partial = nullptr;
    else {
        g.words = reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(g.partial) + parts_bytes(g.M, g.N, g.splits));
        g.tag = launch_tag();
    }
    return dtype_launch(s, g, batch, trans_b, dtype);
}

}  // namespace mhip
