// LDS tiles of 16-bit operands and the tile store, shared by the register-staged and the ring-staged
// MFMA kernels.
#pragma once
#include "gemm_common.h"

namespace mhip {

// Swizzle of the 16-byte chunk index inside a 128-byte LDS row.  Rows r..r+15
// (r % 16 == 0) map one chunk column onto 16 distinct bank groups.
__device__ inline int swz(int row) { return ((row >> 1) ^ (row >> 4)) & 7; }

__device__ inline uint32_t lds_off(int row, int chunk) {
    return (uint32_t)(row * kRowBytes + ((chunk ^ swz(row)) << 4));
}

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// Buffer load of 16 bytes per lane straight into LDS: lane l lands at byte lds + 16 l (lds uniform, a
// multiple of 16).  As inline assembly because the compiler puts a wait for ALL outstanding loads in
// front of any LDS read that it cannot tell apart from the builtin's target, which is every read of
// another stage of a ring; the kernels count their loads and wait themselves.  (M0 is a reserved register
// that cannot be named as clobbered; nothing else in these kernels uses it.)
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(off), "s"(rsrc) : "memory");
}
// The same with 4 bytes per lane (lds a multiple of 4), for rows that start on no 16-byte boundary.
__device__ __forceinline__ void load_dword_to_lds(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds), "v"(off), "s"(rsrc) : "memory");
}
// LDS address of a shared-memory pointer, as those loads take it.
__device__ __forceinline__ uint32_t lds_address(const char* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

// c + 16 x 32 . 32 x 16 on operands of a 16-bit type, eight k a lane; b's side comes out in the four registers.
template <typename T> struct Tile16;
template <> struct Tile16<bf16_t> {
    __device__ static f32x4 run(u32x4 b, u32x4 a, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
    }
};
template <> struct Tile16<f16_t> {
    __device__ static f32x4 run(u32x4 b, u32x4 a, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, b), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
    }
};
// Two fp32 values rounded to T, the first one in the low half.
template <typename T>
__device__ __forceinline__ uint32_t round_pair(float lo, float hi) {
    typedef T pair __attribute__((ext_vector_type(2)));
    const pair p = {Elem<T>::from_f32(lo), Elem<T>::from_f32(hi)};
    return __builtin_bit_cast(uint32_t, p);
}

typedef u32x2 u32x2_any __attribute__((aligned(2)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// MFMA operand (32 mn x 16 k) for k-step `s` out of a k-major tile.
__device__ inline u32x4 frag_kmajor(const char* tile, int row0, int s, int lane) {
    return *reinterpret_cast<const u32x4*>(tile + lds_off(row0 + (lane & 31), 2 * s + (lane >> 5)));
}
// chunk swizzle of an operand tile that lies [64 k][ROWS] in LDS: the four k rows that a transposing read
// touches must fall on different banks (rows of 64, 128, 256 bytes)
template <int ROWS>
__device__ __forceinline__ int mn_swz(int k) { return ROWS >= 128 ? ((k & 3) << 2) : ROWS == 64 ? (((k >> 1) & 1) << 2) : 0; }

template <int ROWS>
__device__ inline u32x4 frag_mn(const char* tile, int mn0, int s, int lane) {
    const int i = lane & 15, g = lane >> 4;
    const int mn = mn0 + 16 * (g & 1) + 4 * (i & 3);
    const int k = 16 * s + 8 * (g >> 1) + (i >> 2);
    const char* p0 = tile + k * (ROWS * 2) + (((mn >> 3) ^ mn_swz<ROWS>(k)) << 4) + (mn & 7) * 2;
    // (four k further: the same swizzle, four rows down)
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p0 + 4 * ROWS * 2));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2.x, l2.y, h2.x, h2.y};
}

// The bias of a wave's 32 TN columns from col0 on, as its lanes need it in store_tile: asked for without a branch and all at once, in front of
// the loop over K where the kernel can (group by group at the store each waited out a latency: [1000,3000] x K 1000 with GELU 16.45 -> 15.7 us).
template <typename T, int TN>
struct TileBias {
    Pack4<T> v[TN][4];
    __device__ __forceinline__ void load(const GemmArgs& g, int col0, int lane) {
        const T* bias = static_cast<const T*>(g.bias);
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) v[j][q] = __builtin_bit_cast(Pack4<T>, u32x2{0, 0});
        if (!bias) return;
        const int n0 = col0 + 4 * (lane >> 5);
        if (g.N % 4 == 0) {                              // (a group of four columns past the end is another one's, and not stored)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) v[j][q] = __builtin_bit_cast(Pack4<T>, *reinterpret_cast<const u32x2_any*>(bias + min(n0 + 32 * j + 8 * q, g.N - 4)));
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++) v[j][q].v[e] = bias[min(n0 + 32 * j + 8 * q + e, g.N - 1)];
        }
    }
};

// Chunks of 16 bytes of the residual of a wave's tile, in the order of store_tile's stores, kAtOnce of them on their way together (one behind the
// other, each between two stores that may alias it, they took a latency each: [1000,3000] x K 1000 22.8 us, 18.6 asked for while
// the tile is activated, 18.4 in front of the loop over K).
template <typename T, int TM, int TN>
struct TileResidual {
    static constexpr int kCpr = 4 * TN, kRowsPerPass = 64 / kCpr, kPasses = 32 * TM / kRowsPerPass, kAtOnce = kPasses < 8 ? kPasses : 8;
    static_assert(kPasses % kAtOnce == 0, "whole groups of chunks");
    u32x4 v[kAtOnce];
    __device__ __forceinline__ void load(const GemmArgs& g, const T* res, int row0, int col0, int lane, int p0) {
        const int cc = lane % kCpr, rr = lane / kCpr;
#pragma unroll
        for (int p = 0; p < kAtOnce; p++)
            v[p] = *reinterpret_cast<const u32x4_any*>(res + (int64_t)min(row0 + (p0 + p) * kRowsPerPass + rr, g.M - 1) * g.N + min(col0 + cc * 8, g.N - 8));
    }
};

// The wave's (32 TM) x (32 TN) sub-tile at (row0, col0) of C: bias, activation, rounding, residual, store.
// `stage` is this wave's LDS area of 32 TM rows of 64 TN + 16 bytes.
template <typename T, int TM, int TN>
__device__ __forceinline__ void store_tile(const GemmArgs& g, const f32x16 (&acc)[TM][TN], const TileBias<T, TN>& bias, TileResidual<T, TM, TN>& rv, bool have_residual, char* stage, int row0, int col0, int64_t batch, int lane) {
    constexpr int WTM = 32 * TM, WTN = 32 * TN;
    const int lrow = lane & 31, lhalf = lane >> 5;
    T* c = static_cast<T*>(g.c) + batch * g.sc;
    const T* res = g.residual ? static_cast<const T*>(g.residual) + batch * g.sc : nullptr;
    // Epilogue.  The MFMAs were issued as (B-fragment, A-fragment), so each
    // 32x32 accumulator tile is held transposed: a lane owns row m = lrow and,
    // in register group q = r/4, the four consecutive columns 8q + 4*lhalf + r%4.
    using Res = TileResidual<T, TM, TN>;
    constexpr int kCpr = Res::kCpr, kRowsPerPass = Res::kRowsPerPass, kPasses = Res::kPasses, kAtOnce = Res::kAtOnce;
    const int cc = lane % kCpr, rr = lane / kCpr;
    if (!have_residual && res && g.N >= 8) rv.load(g, res, row0, col0, lane, 0);
    // Stage the wave's sub-tile in LDS as rounded 16-bit rows (padded by 16 bytes
    // against bank conflicts); the rows then go out with lanes running along n, so
    // every store instruction writes whole contiguous row segments.
    constexpr int kRowPad = WTN * 2 + 16;
    dispatch_act(g.act, [&](auto act_tag) {
    constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int nl = j * 32 + 8 * q + 4 * lhalf;          // column inside the wave tile
            float bv[4];
#pragma unroll
            for (int e = 0; e < 4; e++) bv[e] = Elem<T>::to_f32(bias.v[j][q].v[e]);
#pragma unroll
            for (int i = 0; i < TM; i++) {
                Pack4<T> o;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float v = acc[i][j][4 * q + e] + bv[e];
                    v = apply_act_c<ACT>(v);
                    o.v[e] = Elem<T>::from_f32(v);
                }
                *reinterpret_cast<u32x2*>(stage + (i * 32 + lrow) * kRowPad + nl * 2) =
                    __builtin_bit_cast(u32x2, o);
            }
        }
    }
    });
    // each wave only re-reads what it wrote itself
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // (rows of any alignment in chunks of 16 bytes, which global memory takes; what is left of a row, up to seven elements, one by one:
    // element by element [5000,1001] x K 1000 with a residual 55.5 us, 30.4 so, [1500,1500] x K 1500 stored [N, K] 25.8, 24.7)
#pragma unroll
    for (int p0 = 0; p0 < kPasses; p0 += kAtOnce) {
        if (p0 > 0 && res && g.N >= 8) rv.load(g, res, row0, col0, lane, p0);
#pragma unroll
        for (int p = 0; p < kAtOnce; p++) {
            const int ml = (p0 + p) * kRowsPerPass + rr;
            const int m = row0 + ml, n = col0 + cc * 8;
            if (m >= g.M || n >= g.N) continue;
            u32x4 w = *reinterpret_cast<const u32x4*>(stage + ml * kRowPad + cc * 16);
            T* to = c + (int64_t)m * g.N + n;
            if (n + 8 <= g.N) {
                if (res) w = add_chunk<T>(w, rv.v[p]);
                *reinterpret_cast<u32x4_any*>(to) = w;
            } else {
                const Vec16<T> t = __builtin_bit_cast(Vec16<T>, w);
                const T* from = res + (int64_t)m * g.N + n;
#pragma unroll
                for (int e = 0; e < 7; e++)
                    if (n + e < g.N) to[e] = res ? Elem<T>::from_f32(Elem<T>::to_f32(t.v[e]) + Elem<T>::to_f32(from[e])) : t.v[e];
            }
        }
    }
}

}  // namespace mhip
