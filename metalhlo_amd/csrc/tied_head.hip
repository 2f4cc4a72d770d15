// The output head of a short prompt: c = x . round(W)^T with W [N, K] held in fp32 (a tied embedding), up to 768 rows of x in a
// 16-bit type.
//
// What bounds it is reading W once (GPT-2-small: 50304 x 768, 154 MB): the fp32 rows come through a ring in LDS straight
// from memory, sixteen columns of C at a time, are rounded on the way to the operand registers, and x never moves: eight
// waves hold up to 256 rows of it in registers (32 rows x 768 k are 192 of a wave's 256), so nothing is read twice within
// a block of 256 rows.  Sixteen rows of W are 48 KB; two of the ring's three stages are in flight while one is
// multiplied, 96 KB a compute unit where 30 bytes a nanosecond over 2 us need 60.  LDS reads take 1.3 us a stage, the
// fetch 1.6.  Blocks of 256 rows are the grid's second axis: their workgroups lie on the same XCD and read a stage of W
// from its L2 where another block fetched it.  [M,768] x [50304,768]^T, us, against converting W (36) and multiplying: M 150 46.6
// | 36 + 28, 256 52 | 36 + 29, 300 61 | 36 + 50, 576 89 | 36 + 76, 768 95 | 36 + 81; M 1 takes 31 (the 154 MB 24).  (Holding a
// row's 32-byte pieces until a 128-byte line is whole costs the registers of the read-ahead: 300 rows 82.)
#include <mutex>

#include "gemm_lds.h"

namespace mhip {
namespace {

constexpr int kHeadWaves = 8, kHeadSteps = 24, kHeadCols = 16, kHeadStages = 3;
constexpr int kHeadRow = kHeadSteps * 32 * 4, kHeadStage = kHeadCols * kHeadRow;      // bytes of a row of W, of sixteen
constexpr int kHeadRows = kHeadWaves * 32, kHeadMaxRows = 3 * kHeadRows;
constexpr int kHeadLoads = kHeadStage / 1024 / kHeadWaves, kHeadStores = 2;           // per wave and stage

struct HeadArgs {
    const void* x;
    const float* w;
    void* c;
    int M, N, K;
    int rows;             // of x per block
    int strips, per;      // sixteen columns each; strips per workgroup
};

template <typename T>
__global__ __launch_bounds__(64 * kHeadWaves) void tied_head_kernel(HeadArgs g) {
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    // (the arguments in one go)
    asm volatile("" ::"s"(g.x), "s"(g.w), "s"(g.c), "s"(g.M), "s"(g.N), "s"(g.K), "s"(g.rows), "s"(g.strips), "s"(g.per));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lg = lane >> 4;
    const int first = (int)blockIdx.x * g.per, last = min(g.strips, first + g.per);
    if (first >= last) return;
    const int m0 = (int)blockIdx.y * g.rows, rows = min(g.rows, g.M - m0), groups = (rows + 15) / 16;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(g.x, (uint32_t)((int64_t)g.M * g.K * 2)), rw = make_rsrc(g.w, (uint32_t)((int64_t)g.N * g.K * 4));
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(g.c, (uint32_t)((int64_t)g.M * g.N * 2));
    const uint32_t lds = lds_address(smem);

    // ---- sixteen rows of W as they lie in memory, the 16-byte chunks of row r XORed with r inside each run of sixteen (the
    // sixteen rows that one read touches fall on different banks).  A strip behind the last one is loaded all the
    // same, out of bounds: the waits count loads.
    auto load = [&](int strip, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kHeadLoads; j++) {
            const int q = j * kHeadWaves + wave, r = q / 3, pos = q % 3 * 64 + lane, chunk = (pos & ~15) | ((pos ^ r) & 15), n = strip * kHeadCols + r;
            const bool live = strip < last && n < g.N && chunk * 4 < g.K;
            load_to_lds(rw, lds + (uint32_t)(slot * kHeadStage + q * 1024), live ? (uint32_t)(((int64_t)n * g.K + chunk * 4) * 4) : kOob);
        }
    };
    load(first, 0);
    load(first + 1, 1);

    // ---- x: groups `wave` and `wave` + 8 of sixteen rows; step s holds k = 32 s + 8 lg .. + 7 of row li
    u32x4 a[2][kHeadSteps];
    int row[2];
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const int r = (wave + b * kHeadWaves) * 16 + li;
        row[b] = r < rows ? m0 + r : -1;
#pragma unroll
        for (int s = 0; s < kHeadSteps; s++) {
            const int k = 32 * s + 8 * lg;
            a[b][s] = __builtin_amdgcn_raw_buffer_load_b128(rx, row[b] >= 0 && k < g.K ? (uint32_t)((row[b] * g.K + k) * 2) : kOob, 0, 0);
        }
    }
    uint32_t at[2][2];        // chunk 8 (s & 1) + 2 lg + h of row li
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int h = 0; h < 2; h++) at[p][h] = (uint32_t)(li * kHeadRow + ((8 * p + 2 * lg + h) ^ li) * 16);
    __builtin_amdgcn_s_waitcnt(0x0F70);                     // vmcnt(0), in a form that the compiler counts by: no waits for x in the loop

    int slot = 0;
    for (int strip = first; strip < last; strip++) {
        // this strip's loads are older than the stores of two strips and the loads of one; past the barrier every wave has read
        // the strip before, whose place is loaded again
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kHeadLoads + 2 * kHeadStores) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load(strip + 2, slot == 0 ? 2 : slot - 1);
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        if (wave < groups) {
            const char* tile = smem + slot * kHeadStage;
            f32x4 raw[2][2];
            auto read = [&](int s) __attribute__((always_inline)) {
#pragma unroll
                for (int h = 0; h < 2; h++) raw[s & 1][h] = *reinterpret_cast<const f32x4*>(tile + at[s & 1][h] + (s >> 1) * 256);
            };
            read(0);
#pragma unroll
            for (int s = 0; s < kHeadSteps; s++) {
                if (s + 1 < kHeadSteps) read(s + 1);
                __builtin_amdgcn_sched_barrier(0);           // (left alone the compiler moves the reads down to their use)
                const f32x4 lo = raw[s & 1][0], hi = raw[s & 1][1];
                const u32x4 b = {round_pair<T>(lo[0], lo[1]), round_pair<T>(lo[2], lo[3]), round_pair<T>(hi[0], hi[1]), round_pair<T>(hi[2], hi[3])};
                acc[0] = Tile16<T>::run(b, a[0][s], acc[0]);
                acc[1] = Tile16<T>::run(b, a[1][s], acc[1]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // a lane holds columns 4 lg .. + 3 of row li of each group.  (Every wave issues both stores: the waits count them.)
        const int n = strip * kHeadCols + 4 * lg;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const u32x2 v = {round_pair<T>(acc[b][0], acc[b][1]), round_pair<T>(acc[b][2], acc[b][3])};
            __builtin_amdgcn_raw_buffer_store_b64(v, rc, row[b] >= 0 && n < g.N ? (uint32_t)(((int64_t)row[b] * g.N + n) * 2) : kOob, 0, 0);
        }
        slot = slot == 2 ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may land in LDS after the workgroup ends
}

template <typename T>
int launch_head(hipStream_t s, HeadArgs g) {
    auto kern = tied_head_kernel<T>;
    constexpr int kLds = kHeadStages * kHeadStage;
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [&] { err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds); });
    if (err != hipSuccess) return fail(MHIP_ERR_LAUNCH, "tied_head: cannot reserve %d bytes of LDS: %s", kLds, hipGetErrorString(err));
    // blocks of rows of one size; the workgroups of a column range a multiple of eight apart (one XCD)
    const int blocks = (g.M + kHeadRows - 1) / kHeadRows, wgs = compute_units() / blocks / kXcds * kXcds;
    g.rows = ((g.M + blocks - 1) / blocks + 15) / 16 * 16;
    g.strips = (g.N + kHeadCols - 1) / kHeadCols;
    g.per = (g.strips + (wgs > 0 ? wgs : 1) - 1) / (wgs > 0 ? wgs : 1);
    const int used = (g.strips + g.per - 1) / g.per;
    hipLaunchKernelGGL(kern, dim3((unsigned)((used + kXcds - 1) / kXcds * kXcds), (unsigned)blocks), dim3(64 * kHeadWaves), kLds, s, g);
    return check_launch("tied_head");
}

}  // namespace
}  // namespace mhip

using namespace mhip;

extern "C" int mhip_tied_head_ok(int64_t M, int64_t N, int64_t K, int dtype) {
    if (dtype != MHIP_BF16 && dtype != MHIP_F16) return 0;
    return M >= 1 && M <= kHeadMaxRows && N >= 1 && N % 8 == 0 && K >= 32 && K % 32 == 0 && K <= 32 * kHeadSteps && (N + 64) * K * 4 < 0x7FFFFFFFLL && M * N * 2 < 0x7FFFFFFFLL;
}

extern "C" int mhip_tied_head(void* stream, const void* x, const float* w, void* c, int64_t M, int64_t N, int64_t K, int dtype) {
    if (!x || !w || !c) return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_tied_head: NULL matrix pointer");
    if (!mhip_tied_head_ok(M, N, K, dtype) || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(c)) & 15) != 0)
        return fail(MHIP_ERR_UNSUPPORTED, "mhip_tied_head: [%lld,%lld] x K %lld, dtype %d, or pointers off 16 bytes", (long long)M, (long long)N, (long long)K, dtype);
    HeadArgs g = {};
    g.x = x; g.w = w; g.c = c; g.M = (int)M; g.N = (int)N; g.K = (int)K;
    return dtype == MHIP_BF16 ? launch_head<bf16_t>(as_stream(stream), g) : launch_head<f16_t>(as_stream(stream), g);
}
