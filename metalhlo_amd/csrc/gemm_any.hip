// dot_general for 16-bit operands that the vector kernels cannot address: rows that start at odd elements (a
// vocabulary of 50257, 4095 tokens), views at odd addresses, matrices beyond one 2 GB buffer descriptor.
//
// Global loads of 16 bytes need no alignment on this device, only a place inside the allocation.  A tile is
// therefore staged as in gemm.hip (64 k per stage, two LDS buffers, the same swizzles and operand reads), with
// plain loads at whatever address a row begins: rows beyond the matrix repeat its last one (what they give is
// never stored), a piece that leaves its row reads on into the next one, and only in the last stage, behind
// which nothing may be read, is a piece moved to where its row ends.  Two stages of loads are in flight in registers.
//
// 64x64 tiles (five workgroups per compute unit) until 128x128 ones fill the device; a long K is split over the
// grid where a workspace takes the parts.  bf16 [2047,2047] x K 2047 1077 -> 54 us, x^T dy of 769 x 3071 over 8192 tokens
// 2707 -> 129, [4096,4097] x K 4096 8662 -> 231 (595 TFLOP/s; the loads of unaligned rows touch two lines each).
//
// Large ones are copied to rows on 16-byte boundaries instead (gemm_pack_kernel, about 4.5 TB/s of reads and writes) and take the
// kernels for aligned operands; gemm.hip says from where on.
#include "gemm_lds.h"

namespace mhip {

int launch_gemm_finish(hipStream_t s, const GemmArgs& g, int dtype);     // gemm_mid.hip

namespace {

__device__ __forceinline__ u32x4 load_piece(const uint16_t* p) {
    u32x4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
// The last n (1 .. 8) elements of a piece at its front, zeros behind them; n <= 0: zeros.
__device__ __forceinline__ u32x4 keep_last(u32x4 v, int n) {
    const uint64_t lo = v.x | (uint64_t)v.y << 32, hi = v.z | (uint64_t)v.w << 32;
    const int sh = 16 * (8 - n);
    const uint64_t l = sh == 0 ? lo : sh < 64 ? lo >> sh | hi << (64 - sh) : hi >> (sh & 63), h = sh < 64 ? hi >> sh : 0;
    const u32x4 r = {(uint32_t)l, (uint32_t)(l >> 32), (uint32_t)h, (uint32_t)(h >> 32)};
    return n > 0 ? r : u32x4{0u, 0u, 0u, 0u};
}
// The first n (0 .. 7) elements at p, zeros behind them.
__device__ inline u32x4 load_part(const uint16_t* p, int n) {
    u32x4 v = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < 7; e++)
        if (e < n) v[e >> 1] |= (uint32_t)p[e] << (16 * (e & 1));
    return v;
}

// One operand's share of a stage per thread (256 threads).  KMAJOR: element (row, k) at p[row * ld + k],
// otherwise at p[k * ld + row].
template <int ROWS, bool KMAJOR>
struct AnyLoader {
    static constexpr int kCpr = KMAJOR ? 8 : ROWS / 8;       // pieces of eight elements per LDS row
    static constexpr int kLoads = ROWS * 8 / 256;
    const uint16_t* base;
    const uint16_t* src[kLoads];       // this thread's pieces of stage 0, inside the matrix
    int64_t step;                      // elements from one stage to the next
    int rest;                          // k-slow: columns from this thread's piece to the end of the row
    __device__ void init(const uint16_t* p, int row0, int rows, int ld) {
        const int t = threadIdx.x;
        base = p;
        step = KMAJOR ? (int64_t)kBK : (int64_t)kBK * ld;
        rest = KMAJOR ? 0 : rows - (row0 + t % kCpr * 8);
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const int line = t / kCpr + i * (256 / kCpr), c = t % kCpr * 8;
            src[i] = KMAJOR ? p + (int64_t)min(row0 + line, rows - 1) * ld + c : p + (int64_t)line * ld + min(row0 + c, rows - 1);
        }
    }
    // Stage kt whose pieces all lie inside the allocation: K-contiguous rows with 64 k left, k rows with eight
    // elements behind them.
    __device__ static bool inside(int kt, int K, int ld) {
        return KMAJOR ? (kt + 1) * kBK <= K : (int64_t)(K - (kt + 1) * kBK) * ld >= 8;
    }
    __device__ __forceinline__ void load(u32x4 (&r)[kLoads], int kt, int K, int ld) const {
        const int64_t at = kt * step;
        if (inside(kt, K, ld)) {
#pragma unroll
            for (int i = 0; i < kLoads; i++) r[i] = load_piece(src[i] + at);
        } else {
            auto here = [&](int i) {           // how many elements of piece i exist
                const int t = threadIdx.x, left = K - kt * kBK - (KMAJOR ? t % kCpr * 8 : t / kCpr + i * (256 / kCpr));
                return left <= 0 ? 0 : min(8, max(0, KMAJOR ? left : rest));
            };
            if (ld >= 8) {
                // the piece that ends where the elements do, in the same row, moved to the front
#pragma unroll
                for (int i = 0; i < kLoads; i++) r[i] = load_piece(here(i) > 0 ? src[i] + at - (8 - here(i)) : base);
#pragma unroll
                for (int i = 0; i < kLoads; i++) r[i] = keep_last(r[i], here(i));
            } else {
#pragma unroll
                for (int i = 0; i < kLoads; i++) {
                    r[i] = load_part(src[i] + at, here(i));
                    __builtin_amdgcn_sched_barrier(0);       // (one piece's elements in registers at a time)
                }
            }
        }
    }
    __device__ __forceinline__ void store(char* tile, const u32x4 (&r)[kLoads]) const {
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const int t = threadIdx.x, line = t / kCpr + i * (256 / kCpr), c = t % kCpr;
            const uint32_t at = KMAJOR ? lds_off(line, c) : (uint32_t)(line * (ROWS * 2) + ((c ^ mn_swz<ROWS>(line)) << 4));
            *reinterpret_cast<u32x4*>(tile + at) = r[i];
        }
    }
};

template <typename T, int TILE, bool TA, bool TB>
__global__ __launch_bounds__(256, 2) void gemm_any_kernel(GemmArgs g) {
    constexpr int WT = TILE / 2, TM = WT / 32, kTile = TILE * kRowBytes, kStage = 2 * kTile;
    constexpr int kOut = 4 * WT * (WT * 2 + 16), kSmem = 2 * kStage > kOut ? 2 * kStage : kOut;
    __shared__ __attribute__((aligned(1024))) char smem[kSmem];
    int tm, tn;
    tile_of(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * TILE, n0 = tn * TILE;
    const int64_t batch = blockIdx.y;
    const uint16_t* a = static_cast<const uint16_t*>(g.a) + batch * g.sa;
    const uint16_t* b = static_cast<const uint16_t*>(g.b) + batch * g.sb;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // this workgroup's stages: all of K, or one split's
    const int all = (g.K + kBK - 1) / kBK, per = (all + g.splits - 1) / g.splits;
    const int kt0 = (int)blockIdx.z * per, kt1 = min(all, kt0 + per);
    typedef AnyLoader<TILE, !TA> LoadA;
    typedef AnyLoader<TILE, TB> LoadB;
    LoadA la;
    LoadB lb;
    la.init(a, m0, g.M, g.lda);
    lb.init(b, n0, g.N, g.ldb);
    u32x4 ra[2][LoadA::kLoads], rb[2][LoadB::kLoads];

    f32x16 acc[TM][TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    if (kt0 < kt1) {
        la.load(ra[0], kt0, g.K, g.lda);
        lb.load(rb[0], kt0, g.K, g.ldb);
        if (kt0 + 1 < kt1) {
            la.load(ra[1], kt0 + 1, g.K, g.lda);
            lb.load(rb[1], kt0 + 1, g.K, g.ldb);
        }
        la.store(smem, ra[0]);
        lb.store(smem + kTile, rb[0]);
    }
    __syncthreads();
    // set u of the registers holds the stages of parity u (counted from kt0), buffer u of LDS likewise
    for (int kt = kt0; kt < kt1; kt += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (kt + u >= kt1) break;
            if (kt + u + 2 < kt1) {
                la.load(ra[u], kt + u + 2, g.K, g.lda);
                lb.load(rb[u], kt + u + 2, g.K, g.ldb);
            }
            const char* at = smem + u * kStage;
            const char* bt = at + kTile;
            u32x4 af[2][TM], bf[2][TM];
            auto read = [&](int s, u32x4(&fa)[TM], u32x4(&fb)[TM]) {
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    fa[i] = TA ? frag_mn<TILE>(at, wm * WT + i * 32, s, lane) : frag_kmajor(at, wm * WT + i * 32, s, lane);
                    fb[i] = TB ? frag_kmajor(bt, wn * WT + i * 32, s, lane) : frag_mn<TILE>(bt, wn * WT + i * 32, s, lane);
                }
            };
            read(0, af[0], bf[0]);
#pragma unroll
            for (int s = 0; s < kBK / 16; s++) {
                if (s + 1 < kBK / 16) read(s + 1, af[(s + 1) & 1], bf[(s + 1) & 1]);
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TM; j++) acc[i][j] = Mfma32<T>::run(bf[s & 1][j], af[s & 1][i], acc[i][j]);
            }
            if (kt + u + 1 < kt1) {
                la.store(smem + (u ^ 1) * kStage, ra[u ^ 1]);
                lb.store(smem + (u ^ 1) * kStage + kTile, rb[u ^ 1]);
            }
            __syncthreads();
        }
    }

    if (g.partial) {
        // row-major sums of this split
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int m = m0 + wm * WT + i * 32 + (lane & 31);
            if (m >= g.M) continue;
            float* dst = g.partial + ((int64_t)blockIdx.z * g.M + m) * g.N;
#pragma unroll
            for (int j = 0; j < TM; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int n = n0 + wn * WT + j * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (n < g.N) dst[n] = acc[i][j][r];
                }
        }
        return;
    }
    TileBias<T, TM> bias;
    bias.load(g, n0 + wn * WT, lane);
    TileResidual<T, TM, TM> residual;
    store_tile<T, TM, TM>(g, acc, bias, residual, false, smem + wave * (WT * (WT * 2 + 16)), m0 + wm * WT, n0 + wn * WT, batch, lane);
}

bool large_tiles(int64_t M, int64_t N, int64_t batch) {
    return ((M + 127) / 128) * ((N + 127) / 128) * batch >= 256;
}

// Parts of K: up to two workgroups per compute unit, each with at least 512 k.  As in gemm_mid.hip a sum is
// left in one piece from 193 rows on unless K is 4096 or more: in that range more rows do not change a row's bits.
int any_splits(int64_t M, int64_t N, int64_t K, int64_t batch) {
    if (batch != 1 || (M > 192 && K < 4096) || large_tiles(M, N, batch)) return 1;
    const int64_t room = 512 / (((M + 63) / 64) * ((N + 63) / 64)), most = K / 512;
    const int64_t n = room < most ? room : most;
    return n < 2 ? 1 : n > 8 ? 8 : (int)n;
}

template <typename T, int TILE>
int launch_tile(hipStream_t s, GemmArgs g, int64_t batch, int ta, int tb) {
    g.tiles_m = (g.M + TILE - 1) / TILE;
    g.tiles_n = (g.N + TILE - 1) / TILE;
    const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n;
    if (tiles > 0x7FFFFFFFLL || batch > 65535) return fail(MHIP_ERR_UNSUPPORTED, "gemm: grid too large");
    const dim3 grid((unsigned)tiles, (unsigned)batch, (unsigned)g.splits);
    if (!ta && !tb) hipLaunchKernelGGL((gemm_any_kernel<T, TILE, false, false>), grid, dim3(256), 0, s, g);
    else if (!ta) hipLaunchKernelGGL((gemm_any_kernel<T, TILE, false, true>), grid, dim3(256), 0, s, g);
    else if (!tb) hipLaunchKernelGGL((gemm_any_kernel<T, TILE, true, false>), grid, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((gemm_any_kernel<T, TILE, true, true>), grid, dim3(256), 0, s, g);
    return check_launch("gemm_any");
}

// ---- copies with rows on 16-byte boundaries ----
struct PackArgs {
    const uint16_t* src[2];
    uint16_t* dst[2];
    int rows[2], cols[2];              // what exists
    int dst_rows[2], dst_cols[2];      // zeros behind it; columns a multiple of eight
    unsigned blocks0;                  // workgroups of the first matrix
};
constexpr int kPackPieces = 4;         // 16 bytes each, per thread

__global__ __launch_bounds__(256) void gemm_pack_kernel(PackArgs p) {
    const int o = blockIdx.x >= p.blocks0 ? 1 : 0;
    const int rows = p.rows[o], cols = p.cols[o], cpr = p.dst_cols[o] / 8;
    const int64_t all = (int64_t)p.dst_rows[o] * cpr, first = (int64_t)(blockIdx.x - (o ? p.blocks0 : 0)) * (256 * kPackPieces) + threadIdx.x;
    u32x4 v[kPackPieces];
#pragma unroll
    for (int i = 0; i < kPackPieces; i++) {
        const int64_t at = first + i * 256;
        v[i] = u32x4{0u, 0u, 0u, 0u};
        if (at >= all) continue;
        const int64_t row = at / cpr;
        const int c = (int)(at - row * cpr) * 8, n = row < rows ? min(8, cols - c) : 0;
        if (n <= 0) continue;
        const uint16_t* s = p.src[o] + row * cols + c;
        if (n == 8) v[i] = load_piece(s);
        else if (cols >= 8) v[i] = keep_last(load_piece(s - (8 - n)), n);      // (the piece that ends where the row does)
        else v[i] = load_part(s, n);
    }
#pragma unroll
    for (int i = 0; i < kPackPieces; i++)
        if (first + i * 256 < all) *reinterpret_cast<u32x4*>(p.dst[o] + (first + i * 256) * 8) = v[i];
}

}  // namespace

// How an unaligned problem becomes an aligned one: a copy of each operand whose rows need it; k is padded with zeros to
// whole stages where both are copied, and where k is the row of one, both are.
GemmPack gemm_pack_plan(const GemmArgs& g, int trans_a, int trans_b, bool a_off, bool b_off) {
    GemmPack p;
    p.a = a_off || g.K % 8 != 0;
    p.b = b_off || g.K % 8 != 0;
    const int64_t k = p.a && p.b ? (g.K + 31) / 32 * 32 : g.K;
    p.K = (int)k;
    const int64_t m = (g.M + 7) / 8 * 8, n = (g.N + 7) / 8 * 8;
    p.lda = !p.a ? g.lda : (int)(trans_a ? m : k);
    p.ldb = !p.b ? g.ldb : (int)(trans_b ? k : n);
    p.a_bytes = p.a ? (trans_a ? k * m : (int64_t)g.M * k) * 2 : 0;
    p.b_bytes = p.b ? (trans_b ? (int64_t)g.N * k : k * n) * 2 : 0;
    p.a_bytes = (p.a_bytes + 255) / 256 * 256;
    p.b_bytes = (p.b_bytes + 255) / 256 * 256;
    return p;
}

int launch_gemm_pack(hipStream_t s, const GemmArgs& g, const GemmPack& p, int trans_a, int trans_b, char* to) {
    PackArgs w = {};
    int n = 0;
    int64_t blocks[2] = {0, 0};
    auto add = [&](const void* src, char* dst, int rows, int cols, int dst_rows, int dst_cols) {
        w.src[n] = static_cast<const uint16_t*>(src); w.dst[n] = reinterpret_cast<uint16_t*>(dst);
        w.rows[n] = rows; w.cols[n] = cols; w.dst_rows[n] = dst_rows; w.dst_cols[n] = dst_cols;
        blocks[n] = ((int64_t)dst_rows * (dst_cols / 8) + 256 * kPackPieces - 1) / (256 * kPackPieces);
        n++;
    };
    if (p.a) add(g.a, to, trans_a ? g.K : g.M, trans_a ? g.M : g.K, trans_a ? p.K : g.M, p.lda);
    if (p.b) add(g.b, to + p.a_bytes, trans_b ? g.N : g.K, trans_b ? g.K : g.N, trans_b ? g.N : p.K, p.ldb);
    w.blocks0 = (unsigned)blocks[0];
    if (blocks[0] + blocks[1] > 0x7FFFFFFFLL) return fail(MHIP_ERR_UNSUPPORTED, "gemm: grid too large");
    hipLaunchKernelGGL(gemm_pack_kernel, dim3((unsigned)(blocks[0] + blocks[1])), dim3(256), 0, s, w);
    return check_launch("gemm_pack");
}

int64_t gemm_any_workspace(int64_t M, int64_t N, int64_t K, int64_t batch) {
    const int n = any_splits(M, N, K, batch);
    return n == 1 ? 0 : M * N * 4 * n;
}

// Any 16-bit problem.  Without the workspace (g.partial), or with a smaller one, K is not split.
int launch_gemm_any(hipStream_t s, GemmArgs g, int64_t batch, int trans_a, int trans_b, int dtype, int64_t workspace_bytes) {
    g.splits = g.partial ? any_splits(g.M, g.N, g.K, batch) : 1;
    if ((int64_t)g.M * g.N * 4 * g.splits > workspace_bytes) g.splits = 1;
    if (g.splits == 1) g.partial = nullptr;
    const bool bf = dtype == MHIP_BF16, large = large_tiles(g.M, g.N, batch);
    const int st = large ? (bf ? launch_tile<bf16_t, 128>(s, g, batch, trans_a, trans_b) : launch_tile<f16_t, 128>(s, g, batch, trans_a, trans_b))
                         : (bf ? launch_tile<bf16_t, 64>(s, g, batch, trans_a, trans_b) : launch_tile<f16_t, 64>(s, g, batch, trans_a, trans_b));
    return st != MHIP_OK || g.splits == 1 ? st : launch_gemm_finish(s, g, dtype);
}

}  // namespace mhip
