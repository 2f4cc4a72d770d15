// dot_general of a few rows (a decode step) on 16-bit operands with 16-byte aligned rows: C = act(A . op(B) + bias) (+ residual), where
// the time is that of reading B once.
//
// What bounds it: how many bytes of a cold matrix a compute unit has in flight, how far apart they are, and every further launch.
// Loads that stop in registers leave 64 KB of B in flight a unit, and parts of K that a second launch adds up cost 3 to 5 us
// ([4,4096] x [4096,4096]: 7.9 us and that launch, 11.3 in all with B in the memory-side cache).  Here B lands in LDS, which takes no
// registers, 64 to 128 KB a unit from the first instruction on, every row of a piece a whole 128-byte line; the waves split K and each
// walks its share behind its own loads, without a barrier, A's fragments in registers before the first piece arrives.
//   * gemm_strip_kernel: B stored [N, K], up to 16 rows, a workgroup owns 16 columns and all of K;
//   * gemm_parts_kernel: up to 32 rows, strips of 64 columns and parts of 512 k; the last workgroup of a strip to arrive adds its parts up
//     (arrive.h): 13.3 -> 10.2 us from memory.
// Tried: all of K in strips of 16 columns where B is stored [K, N]: rows of 32 bytes over the whole matrix, 17 us; parts of 1024 k or
// strips of 128 columns 10.8 to 11.6.
#include <mutex>

#include "arrive.h"
#include "gemm_lds.h"

namespace mhip {
namespace {

constexpr int kStripWaves = 8;

// PIECES = pieces of 64 k per wave, all of them in flight.
template <typename T, int PIECES>
__global__ __launch_bounds__(64 * kStripWaves) void gemm_strip_kernel(GemmArgs g) {
    constexpr int kPiece = 16 * kRowBytes;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int n0 = (int)blockIdx.x * 16;
    const int64_t batch = blockIdx.y;
    const T* a = static_cast<const T*>(g.a) + batch * g.sa;
    const T* b = static_cast<const T*>(g.b) + batch * g.sb;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a, (uint32_t)((int64_t)g.M * g.lda * 2));
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(b, (uint32_t)((int64_t)g.N * g.ldb * 2));

    // this wave's share of the pieces
    const int pieces = (g.K + kBK - 1) / kBK, per = (pieces + kStripWaves - 1) / kStripWaves;
    const int s0 = wave * per, s1 = min(pieces, s0 + per);
    u32x4 af[PIECES][2];
#pragma unroll
    for (int i = 0; i < PIECES; i++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int k = (s0 + i) * kBK + h * 32 + lg * 8;
            af[i][h] = __builtin_amdgcn_raw_buffer_load_b128(ra, s0 + i < s1 && k < g.K && li < g.M ? (uint32_t)((li * g.lda + k) * 2) : kOob, 0, 0);
        }
    asm volatile("" ::: "memory");
    char* const mine = smem + wave * (PIECES * kPiece);
    const uint32_t at = lds_address(smem) + (uint32_t)wave * (PIECES * kPiece);
    // (loads also of a piece behind the share's end, whose lanes are all out of bounds: the waits count them)
#pragma unroll
    for (int i = 0; i < PIECES; i++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int r = h * 8 + (lane >> 3), n = n0 + r, k = (s0 + i) * kBK + ((lane & 7) ^ swz(r)) * 8;
            load_to_lds(rb, at + (uint32_t)(i * kPiece + h * 1024), n < g.N && k < g.K && s0 + i < s1 ? (uint32_t)(((int64_t)n * g.ldb + k) * 2) : kOob);
        }

    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < PIECES; i++) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((PIECES - 1 - i) * 2) : "memory");
#pragma unroll
        for (int h = 0; h < 2; h++)
            acc = Tile16<T>::run(*reinterpret_cast<const u32x4*>(mine + i * kPiece + lds_off(li, 4 * h + lg)), af[i][h], acc);
    }

    // ---- the waves' sums, in the accumulators' layout: lane (li, lg) holds row li, columns 16 f + 4 lg .. + 3
    __syncthreads();
    f32x4* part = reinterpret_cast<f32x4*>(smem);
    part[wave * 64 + lane] = acc;
    __syncthreads();
    const int n = n0 + 4 * lg;
    if (wave > 0 || li >= g.M || n >= g.N) return;
    f32x4 sum = part[lane];
#pragma unroll
    for (int w = 1; w < kStripWaves; w++) sum += part[w * 64 + lane];
    const T* bias = static_cast<const T*>(g.bias);
    const T* res = static_cast<const T*>(g.residual);
    const int64_t to = batch * g.sc + (int64_t)li * g.N + n;
    T* c = static_cast<T*>(g.c) + to;
    const int live = min(4, g.N - n);
    dispatch_act(g.act, [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
        Pack4<T> o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o.v[e] = Elem<T>::from_f32(apply_act_c<ACT>(sum[e] + (bias && e < live ? Elem<T>::to_f32(bias[n + e]) : 0.f)));
            // (second rounding on purpose: the same result as a separate add over the stored C)
            if (res && e < live) o.v[e] = Elem<T>::from_f32(Elem<T>::to_f32(o.v[e]) + Elem<T>::to_f32(res[to + e]));
        }
        if (live == 4 && (reinterpret_cast<uintptr_t>(c) & 7) == 0) *reinterpret_cast<u32x2*>(c) = __builtin_bit_cast(u32x2, o);
        else
#pragma unroll
            for (int e = 0; e < 4; e++) if (e < live) c[e] = o.v[e];
    });
}

// Strips of 64 columns and parts of 512 k that are in flight as a whole.  MT = groups of 16 rows of A.
constexpr int kPartCols = 64, kPartSteps = 2, kPartK = kStripWaves * kPartSteps * 32;
template <typename T, bool TB, int MT>
__global__ __launch_bounds__(64 * kStripWaves) void gemm_parts_kernel(GemmArgs g, uint64_t* words, uint64_t tag) {
    constexpr int NS = kPartCols, NF = NS / 16, kRow = 2 * NS, kPiece = 32 * kRow, kRows = 8, kLoads = kPiece / 1024;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ int last;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int n0 = (int)blockIdx.x * NS, split = blockIdx.y, parts = gridDim.y;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(g.a, (uint32_t)((int64_t)g.M * g.lda * 2));
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(g.b, (uint32_t)((int64_t)(TB ? g.N : g.K) * g.ldb * 2));
    const int k0 = split * kPartK + wave * (kPartSteps * 32);
    uint64_t seen = 0;
    if (threadIdx.x == 0) seen = arrive_look(words + blockIdx.x);
    u32x4 af[kPartSteps][MT];
#pragma unroll
    for (int i = 0; i < kPartSteps; i++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int k = k0 + i * 32 + lg * 8, m = mt * 16 + li;
            af[i][mt] = __builtin_amdgcn_raw_buffer_load_b128(ra, k < g.K && m < g.M ? (uint32_t)((m * g.lda + k) * 2) : kOob, 0, 0);
        }
    asm volatile("" ::: "memory");
    char* const mine = smem + wave * (kPartSteps * kPiece);
    const uint32_t at = lds_address(smem) + (uint32_t)wave * (kPartSteps * kPiece);
#pragma unroll
    for (int i = 0; i < kPartSteps; i++)
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            // [K, N]: 32 k x 64 columns a step; [N, K]: 64 columns x 64 k for both steps, half of the columns with each
            const int r = (TB ? i * 32 : 0) + j * kRows + lane / 8, c = (lane % 8 ^ (TB ? swz(r) : mn_swz<NS>(r))) * 8;
            const int k = k0 + (TB ? c : i * 32 + r), n = n0 + (TB ? r : c);
            load_to_lds(rb, at + (uint32_t)(i * kPiece + j * 1024), k < g.K && n < g.N ? (uint32_t)((TB ? (int64_t)n * g.ldb + k : (int64_t)k * g.ldb + n) * 2) : kOob);
        }
    f32x4 acc[MT][NF];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int f = 0; f < NF; f++) acc[mt][f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kPartSteps; i++) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(TB ? 0 : (kPartSteps - 1 - i) * kLoads) : "memory");
#pragma unroll
        for (int f = 0; f < NF; f++) {
            u32x4 bf;
            if (TB) bf = *reinterpret_cast<const u32x4*>(mine + lds_off(16 * f + li, 4 * i + lg));
            else {
                const int k = 8 * lg + (li >> 2), mn = 16 * f + 4 * (li & 3);
                const char* p = mine + i * kPiece + k * kRow + (((mn >> 3) ^ mn_swz<NS>(k)) << 4) + (mn & 7) * 2;
                const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
                const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * kRow)));
                bf = u32x4{lo.x, lo.y, hi.x, hi.y};
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt][f] = Tile16<T>::run(bf, af[i][mt], acc[mt][f]);
        }
    }
    if (threadIdx.x == 0) arrive_claim(words + blockIdx.x, seen, tag);

    // ---- the waves' sums, in the accumulators' layout: lane (li, lg) holds row 16 mt + li, columns 16 f + 4 lg .. + 3; a wave
    // adds up one of the NF groups of every second group of rows
    const __amdgpu_buffer_rsrc_t rp = parts_rsrc(g.partial);
    f32x4* part = reinterpret_cast<f32x4*>(smem);
    constexpr int kOnce = MT < 2 ? 1 : 2;
#pragma unroll
    for (int m0 = 0; m0 < MT; m0 += kOnce) {
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < kOnce; mt++)
#pragma unroll
            for (int f = 0; f < NF; f++) part[((mt * NF + f) * kStripWaves + wave) * 64 + lane] = acc[m0 + mt][f];
        __syncthreads();
        const int m = (m0 + wave / NF) * 16 + li, n = n0 + wave % NF * 16 + 4 * lg;
        if (wave >= kOnce * NF || m >= g.M || n >= g.N) continue;
        f32x4 sum = part[wave * kStripWaves * 64 + lane];
#pragma unroll
        for (int w = 1; w < kStripWaves; w++) sum += part[(wave * kStripWaves + w) * 64 + lane];
        store_part(rp, (uint32_t)(((split * g.M + m) * g.N + n) * 4), sum);
    }
    if (!arrive_last(words + blockIdx.x, parts, &last)) return;

    // ---- the last part of the strip to arrive: four columns a thread, eight parts' loads in flight
    const T* bias = static_cast<const T*>(g.bias);
    const T* res = static_cast<const T*>(g.residual);
    for (int idx = threadIdx.x; idx < g.M * (NS / 4); idx += 64 * kStripWaves) {
        const int m = idx / (NS / 4), n = n0 + idx % (NS / 4) * 4;
        if (n >= g.N) continue;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < parts; s += 8) {
            f32x4 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = load_part(rp, s + u < parts ? (uint32_t)((((s + u) * g.M + m) * g.N + n) * 4) : kOob);
#pragma unroll
            for (int u = 0; u < 8; u++) sum += v[u];
        }
        const int64_t to = (int64_t)m * g.N + n;
        T* c = static_cast<T*>(g.c) + to;
        dispatch_act(g.act, [&](auto act_tag) {
            constexpr int ACT = decltype(act_tag)::value;
            Pack4<T> o;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o.v[e] = Elem<T>::from_f32(apply_act_c<ACT>(sum[e] + (bias ? Elem<T>::to_f32(bias[n + e]) : 0.f)));
                // (second rounding on purpose: the same result as a separate add over the stored C)
                if (res) o.v[e] = Elem<T>::from_f32(Elem<T>::to_f32(o.v[e]) + Elem<T>::to_f32(res[to + e]));
            }
            if ((reinterpret_cast<uintptr_t>(c) & 7) == 0) *reinterpret_cast<u32x2*>(c) = __builtin_bit_cast(u32x2, o);
            else
#pragma unroll
                for (int e = 0; e < 4; e++) c[e] = o.v[e];
        });
    }
}

int64_t part_count(int64_t K) { return (K + kPartK - 1) / kPartK; }
int64_t part_bytes(int64_t M, int64_t N, int64_t K) { return (part_count(K) * M * N * 4 + 255) / 256 * 256; }

template <typename T, bool TB, int MT>
int launch_parts(hipStream_t s, const GemmArgs& g) {
    static_assert(kStripWaves * kPartSteps * 32 * kPartCols * 2 == 64 * 1024, "with the word beside it more than a launch gets unasked");
    auto kern = gemm_parts_kernel<T, TB, MT>;
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024); });
    if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "gemm: cannot reserve 64 KB of LDS: %s", hipGetErrorString(err));
    uint64_t* words = reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(g.partial) + part_bytes(g.M, g.N, g.K));
    hipLaunchKernelGGL(kern, dim3((unsigned)((g.N + kPartCols - 1) / kPartCols), (unsigned)part_count(g.K)), dim3(64 * kStripWaves), 64 * 1024, s, g, words, launch_tag());
    return check_launch("gemm_parts");
}

template <typename T, int PIECES>
int launch_pieces(hipStream_t s, const GemmArgs& g, int64_t batch) {
    constexpr int kLds = kStripWaves * PIECES * 16 * kRowBytes;
    auto kern = gemm_strip_kernel<T, PIECES>;
    if (kLds > 64 * 1024) {
        static std::once_flag once;
        static hipError_t err = hipSuccess;
        std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds); });
        if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "gemm: cannot reserve %d bytes of LDS: %s", kLds, hipGetErrorString(err));
    }
    const int64_t strips = (g.N + 15) / 16;
    if (strips > 0x7FFFFFFFLL || batch > 65535) return fail(MHIP_ERR_UNSUPPORTED, "gemm: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)strips, (unsigned)batch), dim3(64 * kStripWaves), kLds, s, g);
    return check_launch("gemm_strip");
}

template <typename T>
int launch_type(hipStream_t s, const GemmArgs& g, int64_t batch) {
    const int per = ((g.K + kBK - 1) / kBK + kStripWaves - 1) / kStripWaves;
    if (per <= 2) return launch_pieces<T, 2>(s, g, batch);
    if (per <= 4) return launch_pieces<T, 4>(s, g, batch);
    if (per <= 6) return launch_pieces<T, 6>(s, g, batch);
    return launch_pieces<T, 8>(s, g, batch);
}

}  // namespace

// Stored [N, K], all of K in one workgroup.  us, before | here | in parts of 512 k (below), weights from memory:
//   [1,1024] x K 4096 8.2 | 4.5 | 5.6     [4,512] x K 4096 7.9 | 5.1 | 5.2      [4,2048] x K 3072 7.1 | 5.7 | 6.8
//   [4,4096] x K 4096 9.1 | 9.0 | 9.8     [4,1024] x K 2048 4.9 | 4.3 | 5.2     [4,1024] x K 8192 9.6 | 10.5 | 8.5
//   [16,1024] x K 2048 6.1 | 4.8 | 5.4    [16,768] x K 3072 7.8 | 5.9 | 5.6     [16,1024] x K 4096 8.2 | 7.1 | 6.0
// (fewer columns than a strip has: as before);
// and larger matrices keep the few-row kernel's wide strips, [4,6144] x K 4096 13.7 | 14.3, [1,7168] x K 4096 13.1 | - | 16.3.
bool gemm_strip_wanted(int64_t M, int64_t N, int64_t K, int64_t batch, int trans_b) {
    return trans_b && M <= 16 && N >= 16 && K <= (M <= 8 ? 4096 : 2048) && K % 8 == 0 && N * batch <= 16384 && N * K <= (16 << 20);
}

// K in parts of 512.  us, the few-row kernel (from K 2560 on with a launch of its own for the parts' sum) or 64-row tiles | here, weights
// from memory; stored [K, N]:
//   [4,4096] x K 4096 13.2 | 10.2   [4,1024] x K 4096 8.7 | 5.6    [4,768] x K 3072 8.3 | 5.2    [1,4096] x K 1152 6.1 | 5.4
//   [4,8192] x K 4096 18.2 | 16.6   [16,4096] x K 2048 12.9 | 7.6  [32,4096] x K 4096 16.2 | 12.6  [20,1024] x K 1152 6.7 | 5.8
//   [1,1024] x K 1024 4.6 | 5.2     [1,8192] x K 8192 30.1 | 30.7  [1,14336] x K 4096 24.9 | 26.8
//   [48,8192] x K 1536 11.8 | 14.5  [64,4096] x K 4096 16.0 | 17.3 (four groups of rows, not built)
// Stored [N, K], where the few-row kernel reads whole lines too: [4,2048] x K 8192 13.4 | 11.8, [16,512] x K 4096 8.2 | 5.7,
// [16,7168] x K 4096 18.3 | 17.4, [32,4096] x K 4096 15.2 | 11.7, [20,2048] x K 1536 6.1 | 6.1, [20,1024] x K 1152 5.2 | 5.8.
bool gemm_parts_wanted(int64_t M, int64_t N, int64_t K, int64_t batch, int trans_a, int trans_b) {
    // (narrower: [4,264] x K 2552, five strips, is left to the few-row kernel, which puts such a matrix on more units)
    if (trans_a || batch != 1 || M > 32 || N < 512 || N % 8 != 0 || K % 8 != 0 || N > 16384 || K > 16384 || N * K > (32 << 20)) return false;
    return trans_b ? K > (M <= 8 ? 4096 : M <= 16 ? 2048 : 1535) : K > 1024 && N <= 8192;
}
int64_t gemm_parts_workspace(int64_t M, int64_t N, int64_t K) { return part_bytes(M, N, K) + (N + kPartCols - 1) / kPartCols * 8; }

template <typename T>
int launch_parts_type(hipStream_t s, const GemmArgs& g, int trans_b) {
    if (trans_b) return g.M <= 16 ? launch_parts<T, true, 1>(s, g) : launch_parts<T, true, 2>(s, g);
    return g.M <= 16 ? launch_parts<T, false, 1>(s, g) : launch_parts<T, false, 2>(s, g);
}
int launch_gemm_parts(hipStream_t s, const GemmArgs& g, int trans_b, int dtype) {
    return dtype == MHIP_BF16 ? launch_parts_type<bf16_t>(s, g, trans_b) : launch_parts_type<f16_t>(s, g, trans_b);
}

int launch_gemm_strip(hipStream_t s, const GemmArgs& g, int64_t batch, int dtype) {
    return dtype == MHIP_BF16 ? launch_type<bf16_t>(s, g, batch) : launch_type<f16_t>(s, g, batch);
}

}  // namespace mhip
