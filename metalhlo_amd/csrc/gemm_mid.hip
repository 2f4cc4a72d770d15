// dot_general on tiles of 32 to 128 rows and columns for problems that do not fill the device with the
// 256-row tiles of gemm256.hip: few tiles, ragged sizes, a short or a very long contraction.
//
// Such a problem runs one or two workgroups per compute unit, so nothing hides a load latency but the
// workgroup itself.  Operand tiles therefore come through a ring of S LDS stages of 64 k that buffer loads
// fill directly (no register stop); the loads of S - 1 stages are in flight while one is multiplied, and
// one barrier per stage both publishes the stage that landed and frees the one before it.  Stage layouts,
// swizzles and operand reads are those of gemm.hip's register-staged kernel (which re-exposed the latency
// of every stage: 1.2 us per 64 k against 0.25 us of matrix instructions); the swizzle is applied by
// choosing the global chunk each lane asks for.  With one group of waves the k
// order of every sum is the same too, so results are bit for bit those of the other 16-bit kernels.
//
// Where even that leaves units idle (a weight gradient: 768 x 3072 out of 8192) the grid also splits K: each
// part writes its fp32 sums to a workspace of the caller's, and gemm_finish_kernel adds them in order and
// applies bias, activation, rounding and residual.
#include <mutex>

#include "gemm_lds.h"

namespace mhip {

bool gemm256_eligible(const GemmArgs& g, int64_t batch, int trans_a, int trans_b, int dtype, int bw, bool any_tile_count);
int launch_gemm192(hipStream_t s, const GemmArgs& g, int64_t batch, int trans_a, int trans_b, int dtype);

namespace {

// One operand's loads: the wave-wide load i of wave w fills the KB number i * 4 + w of the stage's tile.
template <int ROWS, bool KMAJOR>
struct StageLoader {
    static constexpr int kLoads = ROWS * kRowBytes / 1024 / 4;
    uint32_t off[kLoads];      // byte offset at k0 = 0, kOob when the row / column does not exist
    int k[kLoads];             // first k of the chunk inside the stage
    uint32_t step;             // bytes from one stage to the next
    __device__ void init(int row0, int rows_total, int ld, int wave, int lane) {
        step = KMAJOR ? (uint32_t)(kBK * 2) : (uint32_t)((int64_t)kBK * ld * 2);
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const int p = (i * 4 + wave) * 64 + lane;                   // 16-byte slot of the tile
            if (KMAJOR) {
                const int r = p >> 3, c = (p & 7) ^ swz(r);
                k[i] = c * 8;
                off[i] = row0 + r < rows_total ? (uint32_t)(((int64_t)(row0 + r) * ld + c * 8) * 2) : kOob;
            } else {
                constexpr int kCpr = ROWS / 8;
                const int kk = p / kCpr, c = (p % kCpr) ^ mn_swz<ROWS>(kk);
                k[i] = kk;
                off[i] = row0 + c * 8 < rows_total ? (uint32_t)(((int64_t)kk * ld + row0 + c * 8) * 2) : kOob;
            }
        }
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, uint32_t tile, int wave, int k0, int kend) const {
        const uint32_t at = (uint32_t)(k0 / kBK) * step;
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const bool ok = off[i] != kOob && k0 + k[i] < kend;
            load_to_lds(rsrc, tile + (uint32_t)(i * 4 + wave) * 1024u, ok ? off[i] + at : kOob);
        }
    }
};

// KG groups of four waves: a stage is KG x 64 k, group q multiplies its 64, the groups' sums meet in LDS at the
// end.  S stages in the ring.
// SUMS: each part's sums by row for mhip_gemm_sums, a kernel of its own (as an argument it cost the others 0.1 us a launch).
template <typename T, int BM, int BN, int WGM, bool TA, bool TB, int KG, int S, bool AHEAD, bool SUMS>
__global__ __launch_bounds__(256 * KG) void gemm_mid_kernel(GemmArgs g) {
    constexpr int WGN = 4 / WGM, WTM = BM / WGM, WTN = BN / WGN, TM = WTM / 32, TN = WTN / 32;
    constexpr int kATile = BM * kRowBytes, kPart = (BM + BN) * kRowBytes, kStage = KG * kPart;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    int tm, tn;
    tile_of(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int64_t batch = blockIdx.y;
    const T* a = static_cast<const T*>(g.a) + batch * g.sa;
    const T* b = static_cast<const T*>(g.b) + batch * g.sb;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a, (uint32_t)((int64_t)(TA ? g.K : g.M) * g.lda * 2));
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(b, (uint32_t)((int64_t)(TB ? g.N : g.K) * g.ldb * 2));
    const int lane = threadIdx.x & 63, wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int group = wave_id / 4, wave = wave_id % 4;
    const int wm = wave / WGN, wn = wave % WGN, lrow = lane & 31;

    // this workgroup's stages: all of K, or one split's
    const int all = (g.K + KG * kBK - 1) / (KG * kBK), per = (all + g.splits - 1) / g.splits;
    const int kt0 = (int)blockIdx.z * per, kt1 = min(all, kt0 + per), kend = min(g.K, kt1 * KG * kBK);
    StageLoader<BM, !TA> la;
    StageLoader<BN, TB> lb;
    la.init(m0, g.M, g.lda, wave, lane);
    lb.init(n0, g.N, g.ldb, wave, lane);
    constexpr int kLoads = StageLoader<BM, !TA>::kLoads + StageLoader<BN, TB>::kLoads;
    // (a stage behind the last one is loaded all the same, with every chunk out of bounds: the waits
    // count loads, so every step issues the same number)
    const uint32_t ring = lds_address(smem) + (uint32_t)group * kPart;
    auto load = [&](int kt) {
        const uint32_t st = ring + (uint32_t)((kt - kt0) % S) * kStage;
        la.load(ra, st, wave, (kt * KG + group) * kBK, kend);
        lb.load(rb, st + kATile, wave, (kt * KG + group) * kBK, kend);
    };

    // (two groups of waves, few stages each: behind the loop)
    constexpr bool kAhead = KG == 1 && !SUMS;
    TileBias<T, TN> bias;
    if (kAhead) bias.load(g, n0 + wn * WTN, lane);
    TileResidual<T, TM, TN> residual;
    const bool early = kAhead && g.residual && !g.partial && residual.kPasses == residual.kAtOnce && g.N >= 8;
    if (early) residual.load(g, static_cast<const T*>(g.residual) + batch * g.sc, m0 + wm * WTM, n0 + wn * WTN, lane, 0);
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    auto stage_at = [&](int kt) { return smem + ((kt - kt0) % S) * kStage + group * kPart; };
    auto read = [&](const char* at, int s, u32x4(&fa)[TM], u32x4(&fb)[TN]) {
        const char* bt = at + kATile;
#pragma unroll
        for (int i = 0; i < TM; i++)
            fa[i] = TA ? frag_mn<BM>(at, wm * WTM + i * 32, s, lane) : frag_kmajor(at, wm * WTM + i * 32, s, lane);
#pragma unroll
        for (int j = 0; j < TN; j++)
            fb[j] = TB ? frag_kmajor(bt, wn * WTN + j * 32, s, lane) : frag_mn<BN>(bt, wn * WTN + j * 32, s, lane);
    };
    // AHEAD: the first operands of a stage are read while the one before it is multiplied; a lone wave per SIMD otherwise
    // waits out an LDS latency behind every barrier.
    static_assert(!AHEAD || S >= 4, "two stages have to have landed");
    u32x4 af[2][TM], bf[2][TN];
#pragma unroll
    for (int p = 0; p < S - 1; p++) load(kt0 + p);
    if (AHEAD) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * kLoads) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read(stage_at(kt0), 0, af[0], bf[0]);
    }
    for (int kt = kt0; kt < kt1; kt++) {
        // stage kt (AHEAD: and kt + 1) has landed when only the stages behind it are in flight; past the barrier that
        // holds for every wave's share, and every wave has read stage kt - 1, whose place is reused
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((AHEAD ? S - 3 : S - 2) * kLoads) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load(kt + S - 1);
        const char* at = stage_at(kt);
        if (!AHEAD) read(at, 0, af[0], bf[0]);
#pragma unroll
        for (int s = 0; s < kBK / 16; s++) {
            if (s + 1 < kBK / 16) read(at, s + 1, af[(s + 1) & 1], bf[(s + 1) & 1]);
            else if (AHEAD) read(stage_at(kt + 1), 0, af[0], bf[0]);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = Mfma32<T>::run(bf[s & 1][j], af[s & 1][i], acc[i][j]);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may land in LDS that the epilogue uses, or after the end
    __syncthreads();                                        // every wave has read the last stage: the ring is free
    if (KG > 1) {
        // in pairs, halving the groups: the upper half leaves its sums, the lower half adds them
        f32x4* sums = reinterpret_cast<f32x4*>(smem);
#pragma unroll
        for (int half = KG / 2; half >= 1; half /= 2) {
            if (group >= half && group < 2 * half) {
#pragma unroll
                for (int x = 0; x < TM * TN * 4; x++) {
                    const f32x16& t = acc[x / 4 / TN][x / 4 % TN];
                    sums[((group - half) * TM * TN * 4 + x) * 256 + wave * 64 + lane] = f32x4{t[4 * (x % 4)], t[4 * (x % 4) + 1], t[4 * (x % 4) + 2], t[4 * (x % 4) + 3]};
                }
            }
            __syncthreads();
            if (group < half) {
#pragma unroll
                for (int x = 0; x < TM * TN * 4; x++) {
                    const f32x4 t = sums[(group * TM * TN * 4 + x) * 256 + wave * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[x / 4 / TN][x / 4 % TN][4 * (x % 4) + e] += t[e];
                }
            }
            __syncthreads();
        }
        if (group > 0) return;
    }
    if constexpr (SUMS) {
        // [part][M][N]: a lane's row, four columns per store (two lanes' stores are 32 consecutive bytes)
        float* p = g.partial + (int64_t)blockIdx.z * g.M * g.N;
#pragma unroll
        for (int x = 0; x < TM * TN * 4; x++) {
            const f32x16& t = acc[x / 4 / TN][x / 4 % TN];
            const int m = m0 + wm * WTM + x / 4 / TN * 32 + lrow, n = n0 + wn * WTN + x / 4 % TN * 32 + 8 * (x % 4) + 4 * (lane >> 5);
            if (m < g.M && n < g.N) *reinterpret_cast<f32x4*>(p + (int64_t)m * g.N + n) = f32x4{t[4 * (x % 4)], t[4 * (x % 4) + 1], t[4 * (x % 4) + 2], t[4 * (x % 4) + 3]};
        }
        return;
    }
    if (!SUMS && g.partial) {
        // the block's registers as they are, 1 KB per store: block (i, j) of wave w of tile t, register group q
        f32x4* dst = reinterpret_cast<f32x4*>(g.partial) + ((((int64_t)blockIdx.z * g.tiles_m * g.tiles_n + tm * g.tiles_n + tn) * 4 + wave) * TM * TN) * 256 + lane;
#pragma unroll
        for (int x = 0; x < TM * TN * 4; x++) {
            const f32x16& t = acc[x / 4 / TN][x / 4 % TN];
            dst[x * 64] = f32x4{t[4 * (x % 4)], t[4 * (x % 4) + 1], t[4 * (x % 4) + 2], t[4 * (x % 4) + 3]};
        }
        return;
    }
    if (!SUMS && !kAhead) bias.load(g, n0 + wn * WTN, lane);
    if constexpr (!SUMS) store_tile<T, TM, TN>(g, acc, bias, residual, early, smem + wave * (WTM * (WTN * 2 + 16)), m0 + wm * WTM, n0 + wn * WTN, batch, lane);
}

// C from the splits' sums in the accumulators' own layout (tiles of BM x BN, WGM x 4 / WGM waves): a wave of
// this kernel takes one 32x32 block, a lane row lrow and per register group q columns 8 q + 4 (lane / 32) .. + 3.
template <typename T, int BM, int BN, int WGM>
__global__ __launch_bounds__(256) void gemm_finish_tiles_kernel(GemmArgs g) {
    constexpr int WGN = 4 / WGM, WTM = BM / WGM, WTN = BN / WGN, TM = WTM / 32, TN = WTN / 32;
    const int lane = threadIdx.x & 63, blk = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles = g.tiles_m * g.tiles_n;
    if (blk >= tiles * 4 * TM * TN) return;
    const int tile = blk / (4 * TM * TN), wave = blk / (TM * TN) % 4, i = blk / TN % TM, j = blk % TN;
    const int m = tile / g.tiles_n * BM + wave / WGN * WTM + i * 32 + (lane & 31);
    const int n0 = tile % g.tiles_n * BN + wave % WGN * WTN + j * 32;
    if (n0 >= g.N) return;
    const f32x4* p = reinterpret_cast<const f32x4*>(g.partial) + (int64_t)blk * 256 + lane;
    f32x4 v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    // (four splits' loads in flight: one at a time the loop takes a memory latency per split, 7.6 us for eight)
#pragma unroll 4
    for (int s = 0; s < g.splits; s++) {
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] += p[q * 64];
        p += (int64_t)tiles * 4 * TM * TN * 256;
    }
    const T* bias = static_cast<const T*>(g.bias);
    const T* res = static_cast<const T*>(g.residual);
    T* c = static_cast<T*>(g.c);
    const bool vec = g.N % 8 == 0 && ((reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(res)) & 15) == 0;
    dispatch_act(g.act, [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int n = n0 + 8 * q + 4 * (lane >> 5) + e;
                if (bias && n < g.N) v[q][e] += Elem<T>::to_f32(bias[n]);
                v[q][e] = sizeof(T) == 4 ? apply_act(v[q][e], ACT) : apply_act_c<ACT>(v[q][e]);
            }
    });
    if (sizeof(T) == 2 && vec) {
        // the two halves of the wave trade register groups: eight consecutive columns per lane, 16 bytes per store
#pragma unroll
        for (int h = 0; h < 2; h++) {
            Pack4<T> lo, hi;
#pragma unroll
            for (int e = 0; e < 4; e++) { lo.v[e] = Elem<T>::from_f32(v[2 * h][e]); hi.v[e] = Elem<T>::from_f32(v[2 * h + 1][e]); }
            const u32x2 a = __builtin_bit_cast(u32x2, *reinterpret_cast<Pack4<bf16_t>*>(&lo)), b = __builtin_bit_cast(u32x2, *reinterpret_cast<Pack4<bf16_t>*>(&hi));
            const auto x = __builtin_amdgcn_permlane32_swap(a.x, b.x, false, false);
            const auto y = __builtin_amdgcn_permlane32_swap(a.y, b.y, false, false);
            u32x4 w = {x[0], y[0], x[1], y[1]};
            const int n = n0 + 16 * h + 8 * (lane >> 5);
            if (m < g.M && n < g.N) {
                const int64_t at = (int64_t)m * g.N + n;
                if constexpr (sizeof(T) == 2) if (res) w = add_chunk<T>(w, *reinterpret_cast<const u32x4*>(res + at));
                *reinterpret_cast<u32x4*>(c + at) = w;
            }
        }
        return;
    }
    if (m >= g.M) return;
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int n = n0 + 8 * q + 4 * (lane >> 5) + e;
            if (n >= g.N) continue;
            const int64_t at = (int64_t)m * g.N + n;
            T o = Elem<T>::from_f32(v[q][e]);
            // (second rounding on purpose: the same result as a separate add over the stored C)
            if (res) o = Elem<T>::from_f32(Elem<T>::to_f32(o) + Elem<T>::to_f32(res[at]));
            c[at] = o;
        }
}

// C from row-major sums [split][M][N], four columns per thread.
template <typename T>
__global__ __launch_bounds__(256) void gemm_finish_kernel(GemmArgs g) {
    const int64_t mn = (int64_t)g.M * g.N, i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i0 >= mn) return;
    const int n_here = (int)min((int64_t)4, mn - i0);
    const bool vec = n_here == 4 && g.N % 4 == 0;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = 0; s < g.splits; s++) {
        const float* p = g.partial + s * mn + i0;
        if (vec) {
            const f32x4 t = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += t[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) if (e < n_here) v[e] += p[e];
        }
    }
    const T* bias = static_cast<const T*>(g.bias);
    const T* res = static_cast<const T*>(g.residual);
    T* c = static_cast<T*>(g.c);
    int next = (int)(i0 % g.N);           // (four elements cover up to four rows: N may be 1)
    dispatch_act(g.act, [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
        T o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int col = next;
            next = col + 1 == g.N ? 0 : col + 1;
            o[e] = Elem<T>::from_f32(0.f);
            if (e >= n_here) continue;
            float x = v[e];
            if (bias) x += Elem<T>::to_f32(bias[col]);
            x = sizeof(T) == 4 ? apply_act(x, ACT) : apply_act_c<ACT>(x);
            o[e] = Elem<T>::from_f32(x);
            // (second rounding on purpose: the same result as a separate add over the stored C)
            if (res) o[e] = Elem<T>::from_f32(Elem<T>::to_f32(o[e]) + Elem<T>::to_f32(res[i0 + e]));
        }
        const bool al = vec && (reinterpret_cast<uintptr_t>(c) & (4 * sizeof(T) - 1)) == 0;
        if (al && sizeof(T) == 2) *reinterpret_cast<u32x2*>(c + i0) = __builtin_bit_cast(u32x2, *reinterpret_cast<Pack4<bf16_t>*>(o));
        else {
#pragma unroll
            for (int e = 0; e < 4; e++) if (e < n_here) c[i0 + e] = o[e];
        }
    });
}

template <typename T, int BM, int BN, int WGM, bool TA, bool TB, bool SUMS, int KG, int S, bool AHEAD = false>
int launch_tile(hipStream_t s, GemmArgs g, int64_t batch) {
    constexpr int kStage = KG * (BM + BN) * kRowBytes, kRing = S * kStage, kSums = KG / 2 * BM * BN * 4, kOut = 4 * (BM / WGM) * ((BN / (4 / WGM)) * 2 + 16);
    constexpr int kUse = kRing > kOut ? kRing : kOut, kSmem = kUse > kSums ? kUse : kSums;
    static_assert(kSmem <= 160 * 1024, "ring larger than LDS");
    auto kern = gemm_mid_kernel<T, BM, BN, WGM, TA, TB, KG, S, AHEAD, SUMS>;
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kSmem); });
    if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "gemm: cannot reserve %d bytes of LDS: %s", kSmem, hipGetErrorString(err));
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n;
    if (tiles > 0x7FFFFFFFLL || batch > 65535) return fail(MHIP_ERR_UNSUPPORTED, "gemm: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)batch, (unsigned)g.splits), dim3(256 * KG), kSmem, s, g);
    return check_launch("gemm_mid");
}

// The forms of this file and the 128x192 ring kernel of gemm_twoset.hip, with what a launch of each costs
// in microseconds: `lone` per 128 k for a workgroup that has its compute unit's L1 to itself (the unit
// fetches 70 to 95 GB/s, which is what binds, not the matrix instructions), no less than all workgroups
// together take from the L2s at 15 TB/s; `ends` for prologue and epilogue of a workgroup.  Fitted to 24
// shapes from [37,768] x K 768 to [2048,2048] x K 2048 and [512,512] x K 16384, each within about 15 %.
struct Form { int bm, bn; float lone, ends; bool in_order; };
constexpr Form kForms[] = {{64, 64, 0.40f, 0.7f, false}, {64, 128, 0.60f, 1.0f, false}, {128, 128, 0.92f, 1.4f, false},   // two groups of waves
                           {64, 64, 0.53f, 0.7f, true}, {64, 128, 0.77f, 1.0f, true}, {128, 128, 1.20f, 1.4f, true},     // one group
                           {128, 192, 0.88f, 2.0f, true}};
constexpr int kRing192 = 6, kMaxSplits = 8;

struct MidPlan { int form = 0, splits = 1; };

float form_cost(const Form& f, int64_t M, int64_t N, int64_t K, int64_t batch, int splits) {
    const int64_t wgs = ((M + f.bm - 1) / f.bm) * ((N + f.bn - 1) / f.bn) * batch * splits;
    const int64_t rounds = (wgs + 255) / 256, at_once = wgs < 256 ? wgs : 256;
    const float bytes = (float)(f.bm + f.bn) * 256.f, l2 = (float)at_once * bytes / 15e6f;
    const float iters = (float)((K / splits + 127) / 128);
    // (two workgroups of the one-group 64x64 form share a compute unit: up to two rounds of it take 1.25 to 1.45 times one,
    // [1500,1024] x K 2048 15.8 us where 64x128 tiles take 16.7, [512,2304] x K 768 8.2 and 8.6)
    const float turns = f.in_order && f.bn == 64 && rounds == 2 ? 1.4f : (float)rounds;
    float t = 3.3f + turns * (iters * (f.lone > l2 ? f.lone : l2) + f.ends);
    // the sums go out and come back (5 TB/s), one more launch
    if (splits > 1) t += 3.f + (float)(M * N) * 8e-6f * (float)splits / 5.f;
    return t;
}

// Smallest estimate.  Two groups of waves and a split K add a sum up in parts, and how many depends on M: the last
// bits of a row may then change with the rows beside it.  That is so up to 192 rows and from K 4096 on, where the parts
// are worth a factor; in between every sum keeps the order of the large tiles, and a sequence its bits in any batch
// (gemm_skinny.hip, gemm_any.hip and gemm_f32.hip have the same limits).  K goes to a workspace in parts only for a
// clear gain.
// `sum_k`: K without the zeros behind it that copied operands have (gemm_any.hip).
MidPlan plan_mid(int64_t M, int64_t N, int64_t K, int64_t sum_k, int64_t batch, bool ring_ok, bool may_split) {
    MidPlan best;
    float t_best = 1e30f;
    const bool in_order = M > 192 && sum_k < 4096;
    for (int f = 0; f <= (ring_ok ? kRing192 : kRing192 - 1); f++) {
        if (in_order && !kForms[f].in_order) continue;
        for (int s = 1; s <= (may_split && batch == 1 && !in_order ? kMaxSplits : 1); s++) {
            if (s > 1 && K / s < 256) break;
            float t = form_cost(kForms[f], M, N, K, batch, s);
            if (f == kRing192 && K % 32 != 0) t += 1.5f;             // (the rest of K: one load latency more)
            if (s > 1) t *= 1.08f;
            if (t < t_best) { t_best = t; best.form = f; best.splits = s; }
        }
    }
    return best;
}

// The same for sums that another launch adds up in any case (mhip_gemm_sums): no order to keep, no launch of its own.
MidPlan plan_sums(int64_t M, int64_t N, int64_t K, int parts) {
    MidPlan best;
    float t_best = 1e30f;
    for (int f = 0; f < kRing192; f++)
        for (int s = parts ? parts : 1; s <= (parts ? parts : kMaxSplits); s++) {
            if (!parts && s > 1 && K / s < 256) break;
            const float t = form_cost(kForms[f], M, N, K, 1, s) + (s == 1 ? (float)(M * N) * 8e-6f / 5.f : -3.f);
            if (t < t_best) { t_best = t; best.form = f; best.splits = s; }
        }
    return best;
}

int64_t plan_bytes(const MidPlan& p, int64_t M, int64_t N) {
    const Form& f = kForms[p.form];
    return p.splits == 1 ? 0 : ((M + f.bm - 1) / f.bm) * ((N + f.bn - 1) / f.bn) * f.bm * f.bn * 4 * p.splits;
}

template <typename T, bool TA, bool TB, bool SUMS = false>
int launch_form(hipStream_t s, const GemmArgs& g, int64_t batch, int form) {
    // one workgroup per compute unit or fewer: all of LDS for a ring of four that reads ahead; otherwise the ring that two
    // workgroups of a unit share ([2000,2000] x K 2000, 256 of 128x128, 29.7 -> 26.6 us; [1000,3000] x K 1000, 384 of 64x128,
    // 16.4 against 20.2; tiles of 64x64 lose by it, [1000,1000] x K 1000 7.9 against 8.6)
    const Form& f = kForms[form];
    const bool one_each = ((g.M + f.bm - 1) / f.bm) * (int64_t)((g.N + f.bn - 1) / f.bn) * batch * g.splits <= 256;
    switch (form) {
        case 0: return launch_tile<T, 64, 64, 2, TA, TB, SUMS, 2, 3>(s, g, batch);
        case 1: return launch_tile<T, 64, 128, 2, TA, TB, SUMS, 2, 3>(s, g, batch);
        case 2: return launch_tile<T, 128, 128, 2, TA, TB, SUMS, 2, 2>(s, g, batch);
        case 3: return launch_tile<T, 64, 64, 2, TA, TB, SUMS, 1, 4>(s, g, batch);
        case 4: return one_each ? launch_tile<T, 64, 128, 2, TA, TB, SUMS, 1, 4, true>(s, g, batch) : launch_tile<T, 64, 128, 2, TA, TB, SUMS, 1, 3>(s, g, batch);
        default: return one_each ? launch_tile<T, 128, 128, 2, TA, TB, SUMS, 1, 4, true>(s, g, batch) : launch_tile<T, 128, 128, 2, TA, TB, SUMS, 1, 2>(s, g, batch);
    }
}

template <typename T, int BM, int BN>
int launch_finish(hipStream_t s, GemmArgs g) {
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int64_t waves = (int64_t)g.tiles_m * g.tiles_n * (BM / 32) * (BN / 32);
    hipLaunchKernelGGL((gemm_finish_tiles_kernel<T, BM, BN, 2>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, g);
    return check_launch("gemm_finish");
}

template <typename T>
int launch_plan(hipStream_t s, GemmArgs g, int64_t batch, int ta, int tb, int dtype, const MidPlan& p) {
    g.splits = p.splits;
    if (p.splits == 1) g.partial = nullptr;
    GemmArgs k = g;                       // (a split stores sums: bias and residual are the finish kernel's)
    if (p.splits > 1) k.bias = k.residual = nullptr;
    int st;
    if (p.form == kRing192) st = launch_gemm192(s, k, batch, ta, tb, dtype);
    else if (!ta && !tb) st = launch_form<T, false, false>(s, k, batch, p.form);
    else if (!ta) st = launch_form<T, false, true>(s, k, batch, p.form);
    else if (!tb) st = launch_form<T, true, false>(s, k, batch, p.form);
    else st = launch_form<T, true, true>(s, k, batch, p.form);
    if (st != MHIP_OK || p.splits == 1) return st;
    switch (p.form) {
        case 0: case 3: return launch_finish<T, 64, 64>(s, g);
        case 1: case 4: return launch_finish<T, 64, 128>(s, g);
        case 2: case 5: return launch_finish<T, 128, 128>(s, g);
        default: return launch_finish<T, 128, 192>(s, g);
    }
}

}  // namespace

// Bytes of workspace the choice for this problem can use (0 = none); a function of the sizes alone.
int64_t gemm_mid_workspace(int64_t M, int64_t N, int64_t K, int64_t sum_k, int64_t batch, int trans_a, int trans_b) {
    return plan_bytes(plan_mid(M, N, K, sum_k, batch, K >= 32 && (K % 32 == 0 || (trans_a && !trans_b)), true), M, N);
}

// 16-bit operands with 16-byte-aligned rows (the caller has checked).  `workspace` (g.partial) may be absent or
// smaller than asked for: then K is not split.
int launch_gemm_mid(hipStream_t s, const GemmArgs& g, int64_t batch, int trans_a, int trans_b, int dtype, int64_t workspace_bytes, int64_t sum_k) {
    const bool ring = gemm256_eligible(g, batch, trans_a, trans_b, dtype, 192, true);
    MidPlan p = plan_mid(g.M, g.N, g.K, sum_k, batch, ring, g.partial != nullptr);
    if (plan_bytes(p, g.M, g.N) > workspace_bytes) p = plan_mid(g.M, g.N, g.K, sum_k, batch, ring, false);
    return dtype == MHIP_BF16 ? launch_plan<bf16_t>(s, g, batch, trans_a, trans_b, dtype, p) : launch_plan<f16_t>(s, g, batch, trans_a, trans_b, dtype, p);
}

// C from the row-major sums [g.splits][M][N] in g.partial.
int launch_gemm_finish(hipStream_t s, const GemmArgs& g, int dtype) {
    const unsigned grid = (unsigned)(((int64_t)g.M * g.N + 1023) / 1024);
    if (dtype == MHIP_F32) hipLaunchKernelGGL((gemm_finish_kernel<float>), dim3(grid), dim3(256), 0, s, g);
    else if (dtype == MHIP_BF16) hipLaunchKernelGGL((gemm_finish_kernel<bf16_t>), dim3(grid), dim3(256), 0, s, g);
    else hipLaunchKernelGGL((gemm_finish_kernel<f16_t>), dim3(grid), dim3(256), 0, s, g);
    return check_launch("gemm_finish");
}

}  // namespace mhip

using namespace mhip;

extern "C" int mhip_gemm_sums_parts(int64_t M, int64_t N, int64_t K, int dtype) {
    if ((dtype != MHIP_BF16 && dtype != MHIP_F16) || M < 1 || N < 1 || K < 1 || N % 8 != 0 || K % 8 != 0) return 0;
    if (M > 0x7FFFFFFF || N > 0x7FFFFFFF || K > 0x7FFFFFFF || M * K * 2 >= 0x7FFFFFFFLL || N * K * 2 >= 0x7FFFFFFFLL) return 0;
    return plan_sums(M, N, K, 0).splits;
}

extern "C" int mhip_gemm_sums(void* stream, const void* a, const void* b, float* sums, int64_t M, int64_t N, int64_t K, int dtype, int parts) {
    if (!a || !b || !sums || parts < 1 || parts > kMaxSplits) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_gemm_sums: NULL pointer, or not 1 to 8 parts");
    if (!mhip_gemm_sums_parts(M, N, K, dtype) || ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(sums)) & 15) != 0)
        return fail(MHIP_ERR_UNSUPPORTED, "mhip_gemm_sums: [%lld,%lld] x K %lld, dtype %d, or pointers off 16 bytes", (long long)M, (long long)N, (long long)K, dtype);
    GemmArgs g = {};
    g.a = a; g.b = b; g.partial = sums;
    g.M = (int)M; g.N = (int)N; g.K = (int)K; g.lda = (int)K; g.ldb = (int)N;
    const MidPlan p = plan_sums(M, N, K, parts);
    g.splits = p.splits;
    return dtype == MHIP_BF16 ? launch_form<bf16_t, false, false, true>(as_stream(stream), g, 1, p.form) : launch_form<f16_t, false, false, true>(as_stream(stream), g, 1, p.form);
}
