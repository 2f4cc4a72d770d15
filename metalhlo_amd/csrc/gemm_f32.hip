// fp32 GEMM on the matrix cores of gfx950: v_mfma_f32_32x32x2_f32 (fp32 operands, fp32
// accumulate -- the products are exact fp32 products, so the 1e-5 bar of fp32 programs holds).
//
// Operands that one buffer descriptor spans go through the ring further down; this kernel takes the larger ones.
//
// One workgroup = a 64x64 tile of C, four waves (2 x 2), one 32x32 accumulator each (or a
// 128x128 tile, 2 x 2 accumulators per wave).  K advances in steps of 16 through two LDS stage buffers: while a
// step is multiplied, the next step's operands travel global -> registers, and are written to
// the other buffer after the step (one barrier per step).  Both operands lie in LDS as
// [rows or columns][16 k] with rows padded to 20 floats, whatever their layout in memory:
// an operand whose k axis is contiguous in memory is copied with 16-byte accesses, the other
// one is transposed on the way in (16-byte global reads along m / n, scalar LDS writes).
//
// The instruction sums two k per issue: lanes 0..31 supply k = 0, lanes 32..63 k = 1.  Which
// two of the step's sixteen k a given issue takes is free as long as both operands agree, so
// issue p takes k = p (lower half) and k = 8 + p (upper half): a lane then needs eight
// CONSECUTIVE k of its row -- two 16-byte LDS reads per fragment and step.
//
// The product is issued as (B, A), so an accumulator comes out transposed: a lane holds one
// row m of the block and, per register group of four, four consecutive columns -- rows of C
// are written with 16-byte stores.
#include <mutex>
#include <type_traits>

#include "gemm_lds.h"

namespace mhip {

int launch_gemm_finish(hipStream_t s, const GemmArgs& g, int dtype);     // gemm_mid.hip

namespace {

constexpr int kStep = 16;       // k per stage
constexpr int kPad = 20;        // floats per LDS row (16 + 4: rows stay 16-byte aligned, banks spread)
// Start of row r of a stage: 20 floats per row and four more after every sixteenth row.  The
// transposing store below has the lanes of a wave sixteen row groups apart in steps of four
// rows: 4 x 20 floats are 16 banks, so without the extra step lanes i and i + 4 (rows 16 apart
// = 320 floats = five times around the 64 banks) would land on the same bank, four deep.
__device__ __forceinline__ constexpr int lds_row(int r) { return r * kPad + 4 * (r >> 4); }
constexpr int lds_floats(int rows) { return rows * kPad + 4 * (rows / 16); }

// Copies this thread's share (NF = TILE / 16 floats) of one operand's [TILE x 16] stage into
// registers.  K_CONTIG: element (row, k) at p[row * ld + k]; otherwise at p[k * ld + row].
// Out-of-range rows / k read as zero.  (A global load of 16 bytes needs no alignment.)
template <bool K_CONTIG, int NF>
__device__ inline void stage_load(const float* __restrict__ p, int ld, int row0, int rows, int k0, int K, float (&r)[NF]) {
    const int t = threadIdx.x;
    constexpr int TPR = 16 / NF;           // threads per row of a k-contiguous stage
    if (K_CONTIG) {
        const int row = row0 + t / TPR, k = k0 + (t % TPR) * NF;
#pragma unroll
        for (int h = 0; h < NF / 4; h++) {
            const int kk = k + 4 * h;
            if (row < rows && kk + 4 <= K) {
                f32x4 v;
                __builtin_memcpy(&v, p + (int64_t)row * ld + kk, 16);
                r[4 * h + 0] = v[0]; r[4 * h + 1] = v[1]; r[4 * h + 2] = v[2]; r[4 * h + 3] = v[3];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) r[4 * h + e] = (row < rows && kk + e < K) ? p[(int64_t)row * ld + kk + e] : 0.f;
            }
        }
    } else {
        const int k = k0 + (t >> 4), row = row0 + (t & 15) * NF;
#pragma unroll
        for (int h = 0; h < NF / 4; h++) {
            const int rr = row + 4 * h;
            if (k < K && rr + 4 <= rows) {
                f32x4 v;
                __builtin_memcpy(&v, p + (int64_t)k * ld + rr, 16);
                r[4 * h + 0] = v[0]; r[4 * h + 1] = v[1]; r[4 * h + 2] = v[2]; r[4 * h + 3] = v[3];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) r[4 * h + e] = (k < K && rr + e < rows) ? p[(int64_t)k * ld + rr + e] : 0.f;
            }
        }
    }
}

template <bool K_CONTIG, int NF>
__device__ inline void stage_store(float* lds, const float (&r)[NF]) {
    const int t = threadIdx.x;
    constexpr int TPR = 16 / NF;
    if (K_CONTIG) {
        float* d = lds + lds_row(t / TPR) + (t % TPR) * NF;
#pragma unroll
        for (int h = 0; h < NF / 4; h++) *reinterpret_cast<f32x4*>(d + 4 * h) = f32x4{r[4 * h], r[4 * h + 1], r[4 * h + 2], r[4 * h + 3]};
    } else {
        const int k = t >> 4, row = (t & 15) * NF;
#pragma unroll
        for (int e = 0; e < NF; e++) lds[lds_row(row + e) + k] = r[e];
    }
}

// The wave's (32 WB) x (32 WB) block at (row0, col0) of C, or of this split's sums.
template <int WB>
__device__ __forceinline__ void store_f32(const GemmArgs& g, const f32x16 (&acc)[WB][WB], int row0, int col0, int64_t batch, int lane) {
    const int lrow = lane & 31, lhalf = lane >> 5;
    float* c = g.partial ? g.partial + (int64_t)blockIdx.z * g.M * g.N : static_cast<float*>(g.c) + batch * g.sc;
    const float* res = g.residual && !g.partial ? static_cast<const float*>(g.residual) + batch * g.sc : nullptr;
    // lane = row m of the block; register 4q + e = column 8q + 4 * lhalf + e
    const float* bias = g.partial ? nullptr : static_cast<const float*>(g.bias);
    const int act = g.partial ? MHIP_ACT_NONE : g.act;
    const bool rows_vec = g.N % 4 == 0 && (reinterpret_cast<uintptr_t>(c) & 15) == 0 &&
                          (!res || (reinterpret_cast<uintptr_t>(res) & 15) == 0);
#pragma unroll
    for (int i = 0; i < WB; i++) {
        const int m = row0 + i * 32 + lrow;
#pragma unroll
        for (int j = 0; j < WB; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int n = col0 + j * 32 + 8 * q + 4 * lhalf;
                if (m >= g.M || n >= g.N) continue;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float x = acc[i][j][4 * q + e];
                    if (bias && n + e < g.N) x += bias[n + e];
                    if (act != MHIP_ACT_NONE) x = apply_act(x, act);
                    v[e] = x;
                }
                float* dst = c + (int64_t)m * g.N + n;
                if (rows_vec && n + 4 <= g.N) {
                    f32x4 o = {v[0], v[1], v[2], v[3]};
                    if (res) {
                        const f32x4 r = *reinterpret_cast<const f32x4*>(res + (int64_t)m * g.N + n);
                        o += r;
                    }
                    *reinterpret_cast<f32x4*>(dst) = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (n + e < g.N) dst[e] = res ? v[e] + res[(int64_t)m * g.N + n + e] : v[e];
                }
            }
    }
}

// WB = 32x32 accumulator blocks per wave and side: tile = (64 WB) x (64 WB)
template <bool TA, bool TB, int WB>
__global__ __launch_bounds__(256, 2) void gemm_f32_mfma_kernel(GemmArgs g) {
    constexpr int kTile = 64 * WB, NF = kTile / 16;
    __shared__ __attribute__((aligned(16))) float lds[2][2][lds_floats(kTile)];   // [stage][A | B]
    int tm, tn;
    tile_of(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * kTile, n0 = tn * kTile;
    const int64_t batch = blockIdx.y;
    const float* a = static_cast<const float*>(g.a) + batch * g.sa;
    const float* b = static_cast<const float*>(g.b) + batch * g.sb;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lrow = lane & 31, lhalf = lane >> 5;

    f32x16 acc[WB][WB];
#pragma unroll
    for (int i = 0; i < WB; i++)
#pragma unroll
        for (int j = 0; j < WB; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;

    float ra[NF], rb[NF];
    // A in memory: [M, K] (k contiguous) unless TA; B in memory: [K, N] (n contiguous) unless TB
    stage_load<!TA, NF>(a, g.lda, m0, g.M, 0, g.K, ra);
    stage_load<TB, NF>(b, g.ldb, n0, g.N, 0, g.K, rb);
    stage_store<!TA, NF>(lds[0][0], ra);
    stage_store<TB, NF>(lds[0][1], rb);
    __syncthreads();
    const int steps = (g.K + kStep - 1) / kStep;
    for (int t = 0; t < steps; t++) {
        const int cur = t & 1;
        if (t + 1 < steps) {
            stage_load<!TA, NF>(a, g.lda, m0, g.M, (t + 1) * kStep, g.K, ra);
            stage_load<TB, NF>(b, g.ldb, n0, g.N, (t + 1) * kStep, g.K, rb);
        }
        f32x4 fa[WB][2], fb[WB][2];
#pragma unroll
        for (int i = 0; i < WB; i++) {
            const float* pa = lds[cur][0] + lds_row(wm * 32 * WB + i * 32 + lrow) + lhalf * 8;
            const float* pb = lds[cur][1] + lds_row(wn * 32 * WB + i * 32 + lrow) + lhalf * 8;
            fa[i][0] = *reinterpret_cast<const f32x4*>(pa);
            fa[i][1] = *reinterpret_cast<const f32x4*>(pa + 4);
            fb[i][0] = *reinterpret_cast<const f32x4*>(pb);
            fb[i][1] = *reinterpret_cast<const f32x4*>(pb + 4);
        }
#pragma unroll
        for (int p = 0; p < 8; p++)
#pragma unroll
            for (int i = 0; i < WB; i++)
#pragma unroll
                for (int j = 0; j < WB; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j][p >> 2][p & 3], fa[i][p >> 2][p & 3], acc[i][j], 0, 0, 0);
        if (t + 1 < steps) {
            stage_store<!TA, NF>(lds[cur ^ 1][0], ra);
            stage_store<TB, NF>(lds[cur ^ 1][1], rb);
        }
        __syncthreads();
    }

    store_f32<WB>(g, acc, m0 + wm * 32 * WB, n0 + wn * 32 * WB, batch, lane);
}

// ---- a ring of LDS stages filled by the loads themselves ----
//
// With one stage of 16 k in flight a problem that does not fill the device waits out a load latency per stage
// (0.55 us; the stage's matrix instructions take 0.21).  [2048,2048] x K 2048 173 -> 143 us (120 TFLOP/s),
// [512,768] x K 768 26.7 -> 19.7, 4096^3 1183 -> 1038 (132).  Here S stages of 32 k come straight into LDS (no
// register stop), S - 1 of them in flight, one barrier per stage.  A k-contiguous operand lies there as rows of
// 128 bytes (lane = row, 16 bytes = four consecutive k), the other one as it lies in memory, [32 k][rows], read
// one float per lane with the rows k and k + 4 that one issue takes on different halves of the banks.
// An issue sums k = 8 s + e (lower half of the wave) and 8 s + 4 + e (upper half).
// W = bytes per lane and load: 16, or 4 where a row does not start on 16 bytes (four times the loads, sixteen beside sixteen
// matrix instructions of 64 cycles; the same tile).  us, register-staged | W = 4: [890,712] x K 1536 with A stored [K, M]
// 80.2 | 47.2, [1001,777] x K 1500 60.4 | 49.2, [2047,2047] x K 2047 192 | 178, [300,333] x K 999 43.0 | 32.8.
template <int ROWS, bool KMAJOR, int W>
struct RingLoader {
    static constexpr int kLoads = ROWS * kRowBytes / (64 * W) / 4;  // wave-wide loads per stage and wave
    uint32_t off[kLoads];      // byte offset in stage 0, kOob where the row / column does not exist
    int k[kLoads];             // first k of the piece inside the stage
    uint32_t step;
    __device__ void init(int row0, int rows_total, int ld, int wave, int lane) {
        step = (uint32_t)(KMAJOR ? 128 : (int64_t)32 * ld * 4);
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            // 16-byte slot of the tile, and the element in it
            const int lin = (i * 4 + wave) * 64 + lane, p = W == 16 ? lin : lin >> 2, e = W == 16 ? 0 : lin & 3;
            if (KMAJOR) {
                const int r = p >> 3, c = (p & 7) ^ swz(r);
                k[i] = c * 4 + e;
                off[i] = row0 + r < rows_total ? (uint32_t)(((int64_t)(row0 + r) * ld + k[i]) * 4) : kOob;
            } else {
                constexpr int kCpr = ROWS / 4;
                const int kk = p / kCpr, c = (p % kCpr) ^ (kk >> 2 & 1) << 3, col = row0 + c * 4 + e;
                k[i] = kk;
                off[i] = col < rows_total ? (uint32_t)(((int64_t)kk * ld + col) * 4) : kOob;
            }
        }
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, uint32_t tile, int wave, int kt, int K) const {
        const uint32_t at = (uint32_t)kt * step;
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const bool ok = off[i] != kOob && kt * 32 + k[i] < K;
            if (W == 16) load_to_lds(rsrc, tile + (uint32_t)(i * 4 + wave) * 1024u, ok ? off[i] + at : kOob);
            else load_dword_to_lds(rsrc, tile + (uint32_t)(i * 4 + wave) * 256u, ok ? off[i] + at : kOob);
        }
    }
};

// The four k of this lane's half in step s (of eight k) of one 32-row block.
template <int ROWS, bool KMAJOR>
__device__ __forceinline__ f32x4 ring_frag(const char* tile, int row0, int s, int lane) {
    const int r = row0 + (lane & 31), h = lane >> 5;
    if (KMAJOR) return *reinterpret_cast<const f32x4*>(tile + lds_off(r, 2 * s + h));
    const char* p = tile + (8 * s + 4 * h) * (ROWS * 4) + ((r ^ h << 5) << 2);
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = *reinterpret_cast<const float*>(p + e * (ROWS * 4));
    return v;
}

template <bool TA, bool TB, int WB, int S, int W>
__global__ __launch_bounds__(256) void gemm_f32_ring_kernel(GemmArgs g) {
    constexpr int kTile = 64 * WB, kBytes = kTile * kRowBytes, kStage = 2 * kBytes;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    int tm, tn;
    tile_of(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * kTile, n0 = tn * kTile;
    const int64_t batch = blockIdx.y;
    const float* a = static_cast<const float*>(g.a) + batch * g.sa;
    const float* b = static_cast<const float*>(g.b) + batch * g.sb;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a, (uint32_t)((int64_t)g.M * g.K * 4)), rb = make_rsrc(b, (uint32_t)((int64_t)g.N * g.K * 4));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    // this workgroup's stages: one part of K, or all parts one after the other
    const int all = (g.K + 31) / 32, per = (all + g.splits - 1) / g.splits;
    const int kt0 = (int)blockIdx.z * per, kt1 = g.partial ? min(all, kt0 + per) : all, kend = min(g.K, kt1 * 32);
    RingLoader<kTile, !TA, W> la;
    RingLoader<kTile, TB, W> lb;
    la.init(m0, g.M, g.lda, wave, lane);
    lb.init(n0, g.N, g.ldb, wave, lane);
    constexpr int kLoads = 2 * RingLoader<kTile, !TA, W>::kLoads;
    // (a stage behind the last one is loaded all the same, out of bounds: the waits count loads)
    const uint32_t ring = lds_address(smem);
    auto load = [&](int kt) {
        const uint32_t st = ring + (uint32_t)((kt - kt0) % S) * kStage;
        la.load(ra, st, wave, kt, kend);
        lb.load(rb, st + kBytes, wave, kt, kend);
    };

    // (sum: the parts that are done, added in their order: the bits of the launch that has a workgroup for each)
    f32x16 acc[WB][WB], sum[WB][WB];
#pragma unroll
    for (int i = 0; i < WB; i++)
#pragma unroll
        for (int j = 0; j < WB; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = sum[i][j][e] = 0.f;
    auto close_part = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WB; i++)
#pragma unroll
            for (int j = 0; j < WB; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) { sum[i][j][e] += acc[i][j][e]; acc[i][j][e] = 0.f; }
    };
#pragma unroll
    for (int p = 0; p < S - 1; p++) load(kt0 + p);
    // A loop for the stages of each part: with the end of a part tested in one loop over all stages a stage took 0.07 us more,
    // [512,768] x K 768 stored [N, K] 20.9 -> 19.4 us, [476,1232] x K 264 13.9 -> 13.3, [1000,1000] x K 500 16.6 -> 15.5.
    // Small tiles add a part up in the next one's first stage, where the barrier and the LDS reads give its last products time.
    // us, behind its last stage | in the next one's first: [2048,768] x K 3072 112.3 | 110.8, [3782,1120] x K 2048 175.0 | 172.7, x^T dy [768,3072]
    // over 8192 404 | 398; without parts 111.3, 173.7 and 405; few stages a part: [512,768] x K 768 19.8 | 19.4, stored [N, K] 19.5 | 19.6.
    // (The other forms have no registers for a stage of its own: 228 -> 264 with 128x128 tiles, one workgroup a unit instead of two.)
    constexpr bool kLate = WB == 1 && W == 16;
    auto stage = [&](int kt, auto first) __attribute__((always_inline)) {
        // stage kt has landed when only the S - 2 stages behind it are in flight; past the barrier that holds for
        // every wave's share, and every wave has read stage kt - 1, whose place is reused
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * kLoads) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load(kt + S - 1);
        const char* at = smem + ((kt - kt0) % S) * kStage;
        f32x4 af[2][WB], bf[2][WB];
        auto read = [&](int s, f32x4(&fa)[WB], f32x4(&fb)[WB]) {
#pragma unroll
            for (int i = 0; i < WB; i++) {
                fa[i] = ring_frag<kTile, !TA>(at, (wm * WB + i) * 32, s, lane);
                fb[i] = ring_frag<kTile, TB>(at + kBytes, (wn * WB + i) * 32, s, lane);
            }
        };
        read(0, af[0], bf[0]);
        if (first) close_part();
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s < 3) read(s + 1, af[(s + 1) & 1], bf[(s + 1) & 1]);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < WB; i++)
#pragma unroll
                    for (int j = 0; j < WB; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[s & 1][j][e], af[s & 1][i][e], acc[i][j], 0, 0, 0);
        }
    };
    for (int k0 = kt0; k0 < kt1; k0 += per) {
        const int k1 = min(kt1, k0 + per);
        if (kLate) stage(k0, std::true_type{});
        for (int kt = k0 + kLate; kt < k1; kt++) stage(kt, std::false_type{});
        if (!kLate) close_part();
    }
    if (kLate) close_part();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may land in LDS after the workgroup ends
    store_f32<WB>(g, sum, m0 + wm * 32 * WB, n0 + wn * 32 * WB, batch, lane);
}

template <bool TA, bool TB, int WB>
int launch_tile(hipStream_t s, GemmArgs g, int64_t batch) {
    constexpr int kTile = 64 * WB;
    g.tiles_m = (g.M + kTile - 1) / kTile;
    g.tiles_n = (g.N + kTile - 1) / kTile;
    const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n;
    if (tiles > 0x7FFFFFFFLL || batch > 65535) return fail(MHIP_ERR_UNSUPPORTED, "gemm: grid too large");
    hipLaunchKernelGGL((gemm_f32_mfma_kernel<TA, TB, WB>), dim3((unsigned)tiles, (unsigned)batch), dim3(256), 0, s, g);
    return check_launch("gemm_f32_mfma");
}

template <bool TA, bool TB, int WB, int S, int W>
int launch_ring(hipStream_t s, GemmArgs g, int64_t batch) {
    constexpr int kTile = 64 * WB, kSmem = S * 2 * kTile * kRowBytes;
    auto kern = gemm_f32_ring_kernel<TA, TB, WB, S, W>;
    if (kSmem > 64 * 1024) {
        static std::once_flag once;
        static hipError_t err = hipSuccess;
        std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kSmem); });
        if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "gemm: cannot reserve %d bytes of LDS: %s", kSmem, hipGetErrorString(err));
    }
    g.tiles_m = (g.M + kTile - 1) / kTile;
    g.tiles_n = (g.N + kTile - 1) / kTile;
    const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n;
    if (tiles > 0x7FFFFFFFLL || batch > 65535) return fail(MHIP_ERR_UNSUPPORTED, "gemm: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)batch, g.partial ? (unsigned)g.splits : 1u), dim3(256), kSmem, s, g);
    return check_launch("gemm_f32_ring");
}

int64_t large_tiles(int64_t M, int64_t N, int64_t batch) { return ((M + 127) / 128) * ((N + 127) / 128) * batch; }

// 128x128 tiles once there are enough of them for a round and a quarter of three per compute unit, 64x64 tiles (five
// per compute unit) below that.  Measured with the ring (us, 64 | 128): 4096^3 1060 | 1038, 2048^3 143 | 157,
// [8192,768] x K 3072 308 | 405; register-staged 1183 at 4096^3 (128), 173 at 2048^3 and 382 (64).  Rings of
// three and four stages are 2 to 8 % behind two: the workgroups of a unit hide each other's latency.
// Four-byte loads keep the 64x64 tiles: 128x128 ones take 272 to 308 registers, one workgroup a unit (us, 64 | 128 | register-staged
// 128): [4095,4095] x K 1023 366 | 467 | 425, [16383,1027] x K 771 stored [N, K] 309 | 449 | 333, [8191,2047] x K 2047 707 | 844 | 687,
// [6001,3001] x K 3001 1133 | 1442 | 1203, [4093,4097] x K 4099 with A stored [K, M] 1403 | 1766 | 1599.
template <bool TA, bool TB>
int launch(hipStream_t s, const GemmArgs& g, int64_t batch, bool ring, bool wide) {
    const bool large = large_tiles(g.M, g.N, batch) >= 960 && !g.partial;
    if (ring && wide) return large ? launch_ring<TA, TB, 2, 2, 16>(s, g, batch) : launch_ring<TA, TB, 1, 2, 16>(s, g, batch);
    if (ring) return launch_ring<TA, TB, 1, 2, 4>(s, g, batch);
    return large ? launch_tile<TA, TB, 2>(s, g, batch) : launch_tile<TA, TB, 1>(s, g, batch);
}

// The parts in which a sum over K is formed: about 256 k each, eight at most, from K alone, so that a row has the same bits
// whether the parts have workgroups of their own (fp32 sums in a workspace, one more launch) or one that takes them in turn.
int ring_parts(int64_t K) { return K < 512 ? 1 : K < 2048 ? (int)(K / 256) : 8; }

// Workgroups of their own while tiles of 64x64 leave half of the compute units idle, for short K only if all parts then
// find an idle one (us, whole | in parts, weights from memory): 48 tiles [256,768] x K 768 19.6 | 13.7 and K 3072 65 | 23.5,
// 54 tiles [568,384] x K 1016 24.5 | 16.0, 96 tiles [512,768] x K 768 19.6 | 18.9 and K 3072 65 | 31, 121 tiles of K 700 18.2 | 16.5,
// 144 tiles of K 768 19.8 | 20.3, 256 tiles of K 1024 25.1 | 31.
bool ring_split(int64_t M, int64_t N, int64_t K, int64_t batch) {
    const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64), n = ring_parts(K);
    return batch == 1 && n > 1 && tiles <= 128 && (tiles * n <= 256 || K >= 1024);
}

bool ring_sizes(int64_t M, int64_t N, int64_t K) { return M * K < 0x1FFFFFFF && N * K < 0x1FFFFFFF; }

}  // namespace

// fp32 problems with enough work for a 64x64 tile to pay (smaller ones keep the plain kernel:
// it wastes nothing on a 20x24 product).  MHIP_GEMM_F32_MFMA = 2 turns the kernel off, = 3
// takes it for every fp32 problem.
bool gemm_f32_mfma_wanted(const GemmArgs& g) {
    const int mode = tune_int("MHIP_GEMM_F32_MFMA", 1);
    if (mode == 2 || g.K < 1) return false;
    return mode == 3 || ((int64_t)g.M * g.N >= 48 * 48 && g.K >= 16);
}

int64_t gemm_f32_workspace(int64_t M, int64_t N, int64_t K, int64_t batch, int trans_a, int trans_b) {
    if (!ring_sizes(M, N, K)) return 0;
    return ring_split(M, N, K, batch) ? M * N * 4 * ring_parts(K) : 0;
}

// Without the workspace (g.partial), or with a smaller one, K is not split.
int launch_gemm_f32_mfma(hipStream_t s, GemmArgs g, int64_t batch, int trans_a, int trans_b, int64_t workspace_bytes) {
    const bool ring = ring_sizes(g.M, g.N, g.K);
    const bool wide = g.lda % 4 == 0 && g.ldb % 4 == 0 && g.sa % 4 == 0 && g.sb % 4 == 0 &&
                      ((reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b)) & 15) == 0;
    g.splits = ring_parts(g.K);
    if (!ring || !ring_split(g.M, g.N, g.K, batch) || (int64_t)g.M * g.N * 4 * g.splits > workspace_bytes) g.partial = nullptr;
    const int st = !trans_a ? (!trans_b ? launch<false, false>(s, g, batch, ring, wide) : launch<false, true>(s, g, batch, ring, wide))
                            : (!trans_b ? launch<true, false>(s, g, batch, ring, wide) : launch<true, true>(s, g, batch, ring, wide));
    return st != MHIP_OK || !g.partial ? st : launch_gemm_finish(s, g, MHIP_F32);
}

}  // namespace mhip
