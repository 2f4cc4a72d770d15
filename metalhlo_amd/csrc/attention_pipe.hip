// Flash-attention forward, pipelined variant for head size 128 (bf16 / f16, no mask operand):
// one workgroup of four waves (one per SIMD) owns 256 query rows of one (batch, head);
// each wave owns 64 of them as two 32-row query blocks.
//
// Against the two-workgroups-per-CU kernel (attention.hip) this halves the LDS bytes
// read and the global -> LDS bytes moved per FLOP (every K / V fragment a wave reads
// serves two query blocks), and it overlaps the matrix and the softmax work inside one
// wave instead of relying on a second wave.  A wave alone on its SIMD issues roughly six
// instructions in the time one MFMA occupies the matrix pipe, so all work on key blocks
// is hand-scheduled (fa_loop.inc, generated by gen_fa_loop.py) with softmax arithmetic
// behind every MFMA:
//
//   step j:   O += V(j-1)^T . P(j-1)^T   | MFMA   first half of softmax(j)   | VALU
//             O *= alpha(j)  where a row's reference maximum moved (rare)
//             barrier; K(j+4), V(j+3) -> the buffers just released
//             S(j+1) = K(j+1) . Q^T      | MFMA   second half of softmax(j)  | VALU
//
// This file keeps what surrounds the steps: operand set-up, the prologue loads, the
// choice of how many unmasked steps a wave runs, the masked last step (causal diagonal or
// the block holding the last key), the barrier / load sequence a finished wave keeps up
// for the others, and the epilogue.
//
// Scores are computed transposed (S^T = K . Q^T) so that a lane holds 16 keys of one
// query column per accumulator: row statistics are per-lane loops plus one exchange
// between the two 32-lane halves, and P feeds the second product without any
// cross-lane movement.  K and V blocks of 64 keys go global -> LDS directly (rings
// of four 16 KB buffers each, filled three blocks ahead of their use); V is
// read with transposing LDS reads.  Softmax state and both accumulations are fp32;
// the output is rounded once.  A causal workgroup takes two query tiles, one from each
// end of the sequence, so that all workgroups carry the same load.
#include <mutex>
#include <type_traits>

#include "attention_common.h"

namespace mhip {

typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));

#include "fa_loop.inc"

namespace {

// The hand-scheduled pieces by element type.
template <typename T> struct PipeAsm;
#define MHIP_PIPE_ASM(T, sfx)                                                                                          \
    template <> struct PipeAsm<T> {                                                                                    \
        template <typename... A> __device__ __forceinline__ static void scores0(A&&... a) { fa_pipe_scores0_##sfx(a...); } \
        template <typename... A> __device__ __forceinline__ static void loop(A&&... a) { fa_pipe_loop_##sfx(a...); }       \
        template <typename... A> __device__ __forceinline__ static void final_step(A&&... a) { fa_pipe_final_##sfx(a...); } \
        template <typename... A> __device__ __forceinline__ static void pv(A&&... a) { fa_pipe_pv_##sfx(a...); }           \
    };
MHIP_PIPE_ASM(bf16_t, bf16)
MHIP_PIPE_ASM(f16_t, f16)
#undef MHIP_PIPE_ASM

constexpr int kPD = 128;                    // head size
constexpr int kPTile = kBKV * kPD * 2;      // bytes of one K (or V) block in LDS
constexpr int kPRing = 4;                   // ring depth of each of K and V
constexpr int kPBQ = 256;                   // query rows per workgroup

template <typename T, bool CAUSAL>
__global__ __launch_bounds__(256, 1) void fa_pipe_kernel(FaArgs a) {
    constexpr int D = kPD, CPR = D / 8;
    extern __shared__ __attribute__((aligned(1024))) char psmem[];   // K ring, then V ring
    char* const kring = psmem;
    char* const vring = psmem + kPRing * kPTile;

    // A causal workgroup takes two query tiles, one from each end of the sequence, so that
    // every workgroup walks the same number of key blocks (when there are enough workgroups to
    // fill the chip that way); otherwise one tile per workgroup, long causal rows first.
    const bool paired = CAUSAL && a.pair_tiles;
    const int slots = paired ? (a.nqb + 1) / 2 : a.nqb;
    int bh, slot;
    {
        // an XCD (ids go round-robin over the eight) takes every eighth head; the up to seven that are left over are dealt out by tiles
        const int id = blockIdx.x, xcd = id & 7, local = id >> 3, heads = (a.B * a.H) >> 3;
        const int rest = id - 8 * heads * slots;
        bh = rest < 0 ? (local / slots) * 8 + xcd : 8 * heads + rest / slots;
        slot = rest < 0 ? local % slots : rest % slots;
    }
    const int npass = (paired && slot != a.nqb - 1 - slot) ? 2 : 1;
#pragma nounroll
    for (int pass = 0; pass < npass; pass++) {
    const int qb = pass == 0 ? a.nqb - 1 - slot : slot;
    // Per-lane values are derived again in every pass: kept across the hand-scheduled pieces, which
    // pin nearly the whole register file, they would be spilled (the empty asm hides that they
    // do not change).
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = tid >> 6;
    const int lrow = lane & 31, lhalf = lane >> 5;
    const int qblk0 = qb * kPBQ;
    const int qw = qblk0 + wave * 64;          // first query row of this wave

    const T* qp = static_cast<const T*>(a.q) + (int64_t)bh * a.Sq * D;
    const T* kp = static_cast<const T*>(a.k) + (int64_t)bh * a.Skv * D;
    const T* vp = static_cast<const T*>(a.v) + (int64_t)bh * a.Skv * D;
    T* op = static_cast<T*>(a.o) + (int64_t)bh * a.Sq * D;
    const __amdgpu_buffer_rsrc_t rq = fa_rsrc(qp, (uint32_t)((int64_t)a.Sq * D * 2));
    const __amdgpu_buffer_rsrc_t rk = fa_rsrc(kp, (uint32_t)((int64_t)a.Skv * D * 2));
    const __amdgpu_buffer_rsrc_t rv = fa_rsrc(vp, (uint32_t)((int64_t)a.Skv * D * 2));

    int nkv = (a.Skv + kBKV - 1) / kBKV;
    if (CAUSAL) {
        const int last_q = min(qblk0 + kPBQ, a.Sq) - 1;
        nkv = min(nkv, last_q / kBKV + 1);
    }

    // ---- global -> LDS: a wave-wide load fills 1 KB of a block (4 rows of 256 bytes);
    // lane l lands at byte 16*l of it, the swizzle is the choice of the chunk it asks for.
    // Keys past the end read as zero.
    const int ld_row = lane / CPR, ld_pos = lane % CPR;
    auto load_k = [&](int blk_i) __attribute__((always_inline)) {
        const int kv0 = blk_i * kBKV;
        char* dst = kring + (blk_i & (kPRing - 1)) * kPTile;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kb = i * 4 + wave;
            const int row = kb * 4 + ld_row;
            const int key = kv0 + row;
            const uint32_t off = key < a.Skv ? (uint32_t)((key * D + ((ld_pos ^ k_swz<D>(row)) << 3)) * 2) : kOobA;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (fa_lds_void*)(dst + kb * 1024), 16, off, 0, 0, 0);
        }
    };
    auto load_v = [&](int blk_i) __attribute__((always_inline)) {
        const int kv0 = blk_i * kBKV;
        char* dst = vring + (blk_i & (kPRing - 1)) * kPTile;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kb = i * 4 + wave;
            const int row = kb * 4 + ld_row;
            const int key = kv0 + row;
            const uint32_t off = key < a.Skv ? (uint32_t)((key * D + ((ld_pos ^ v_swz<D>(row)) << 3)) * 2) : kOobA;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (fa_lds_void*)(dst + kb * 1024), 16, off, 0, 0, 0);
        }
    };

    // ---- Q^T operands: lane = query column, 8 consecutive d per k-step --------------
    u32x4 qf[2][8];
#pragma unroll
    for (int qi = 0; qi < 2; qi++) {
        const int qpos = qw + 32 * qi + lrow;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const uint32_t off = qpos < a.Sq ? (uint32_t)((qpos * D + 16 * s + 8 * lhalf) * 2) : kOobA;
            qf[qi][s] = __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, 0);
        }
    }
    // ---- prologue: K(0), then the pairs [K(1), V(0)] .. [K(3), V(2)], BEHIND the Q loads: loads
    // land in program order and the first step waits only for what it needs (Q, K(0), and pair 1,
    // whose K fragments the first body reads before its barrier), i.e. it leaves the 16 loads of
    // pairs 2 and 3 in flight.  The empty asm and the scheduling barrier keep the compiler from
    // moving a Q load behind them.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    load_k(0);
    load_k(1); load_v(0);
    load_k(2); load_v(1);
    load_k(3); load_v(2);
    if (a.negate_q) {
#pragma unroll
        for (int qi = 0; qi < 2; qi++)
#pragma unroll
            for (int s = 0; s < 8; s++) {
                qf[qi][s].x ^= 0x80008000u; qf[qi][s].y ^= 0x80008000u;
                qf[qi][s].z ^= 0x80008000u; qf[qi][s].w ^= 0x80008000u;
            }
    }

    // V^T fragment addresses: lane i of a 16-lane group supplies key row i/4 and
    // d columns 4*(i%4)..+3 of its group's 16-column block.
    const int ti = lane & 15, tg = lane >> 4;
    const int v_row0 = 4 * (tg >> 1) + (ti >> 2);
    const int v_d0 = 16 * (tg & 1) + 4 * (ti & 3);

    // loads land in program order: pair i = [K(i), V(i-1)] is needed by step i; the wait in
    // front of it may leave the two younger pairs (2 x 8 loads) in flight
    // A plain barrier instruction: __syncthreads() carries a fence, in front of which the compiler
    // waits for ALL loads in flight -- a finished wave that keeps up the sequence for the others
    // would then reach every barrier a full memory latency late and hold the working waves up.
    auto sync_blocks = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        __builtin_amdgcn_s_barrier();
    };

    // ---- operands of the hand-scheduled pieces (fa_loop.inc pins each to its registers) ----
    u32x32 q32[2];
#pragma unroll
    for (int qi = 0; qi < 2; qi++)
#pragma unroll
        for (int st = 0; st < 8; st++) {
            q32[qi][4 * st + 0] = qf[qi][st].x; q32[qi][4 * st + 1] = qf[qi][st].y;
            q32[qi][4 * st + 2] = qf[qi][st].z; q32[qi][4 * st + 3] = qf[qi][st].w;
        }
    f32x32 o[4], s32[4];
    u32x32 px, py;
#pragma unroll
    for (int r = 0; r < 32; r++) {
        o[0][r] = 0.f; o[1][r] = 0.f; o[2][r] = 0.f; o[3][r] = 0.f;
        py[r] = 0u;                                  // "P(-1)": block 0 adds nothing to O
    }
    f32x4 state = {-INFINITY, -INFINITY, 0.f, 0.f};         // reference maxima, running sums
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)psmem;
    u32x8 kaddr;
    u32x4 vaddr0;
#pragma unroll
    for (int st = 0; st < 8; st++) kaddr[st] = lds0 + k_off<D>(lrow, 2 * st + lhalf);
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
        vaddr0[dt] = lds0 + kPRing * kPTile + v_off<D>(v_row0, (32 * dt + v_d0) >> 3) + (v_d0 & 7) * 2;
    const uint32_t m0b = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)wave * 1024u);
    const int row0 = 4 * wave + ld_row;                      // this thread's row in row group 0 of a block
    u32x2 goff;                                              // its chunk of K(4) and of V(3)
    goff.x = (uint32_t)(((4 * kBKV + row0) * D + ((ld_pos ^ k_swz<D>(row0)) << 3)) * 2);
    goff.y = (uint32_t)(((3 * kBKV + row0) * D + ((ld_pos ^ v_swz<D>(row0)) << 3)) * 2);

    // "V(-1)" must be finite: clear the buffer block 0's product reads
    {
        const u32x4 z = {0u, 0u, 0u, 0u};
        char* dst = vring + 3 * kPTile + tid * 64;
#pragma unroll
        for (int i = 0; i < 4; i++) *reinterpret_cast<u32x4*>(dst + 16 * i) = z;
    }

    // Q, K(0), K(1), V(0) have landed and the cleared buffer is written; pairs 2 and 3 may still be
    // in flight (the waits of the steps count loads from here on)
    asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();

    // a causal wave stops at the block that holds its last query row; the workgroup's count
    // is that of its last wave.  Only a wave's last block can need masking (the causal
    // diagonal, or the block that holds the last key).
    int nkv_w = nkv;
    if (CAUSAL) nkv_w = min(nkv, (min(qw + 64, a.Sq) - 1) / kBKV + 1);
    if (nkv_w < 1) nkv_w = 1;
    const int jl = __builtin_amdgcn_readfirstlane(nkv_w - 1);          // uniform within the wave

    PipeAsm<T>::scores0(s32[0], s32[1], q32[0], q32[1], kaddr);
    if (jl > 0) {
        PipeAsm<T>::loop(o[0], o[1], o[2], o[3], s32[0], s32[1], s32[2], s32[3], px, py, state, goff, q32[0], q32[1],
                          kaddr, vaddr0, rk, rv, a.c, m0b, (uint32_t)jl);
        if (jl & 1) {
            s32[0] = s32[2];
            s32[1] = s32[3];
            py = px;
        }
    }
    {
        u32x2 lim;
        u32x4 va;
#pragma unroll
        for (int qi = 0; qi < 2; qi++) {
            const int qpos = qw + 32 * qi + lrow;
            const int last = CAUSAL ? min(qpos, a.Skv - 1) : a.Skv - 1;
            lim[qi] = (uint32_t)(last - jl * kBKV - 4 * lhalf);
        }
#pragma unroll
        for (int dt = 0; dt < 4; dt++) va[dt] = vaddr0[dt] + (uint32_t)(((jl + 3) & 3) * kPTile);
        PipeAsm<T>::final_step(o[0], o[1], o[2], o[3], s32[0], s32[1], px, py, state, va, lim, a.c);
        // everyone has read K(jl) and V(jl-1): their buffers take K(jl+4) and V(jl+3)
        sync_blocks();
        load_k(jl + 4);
        load_v(jl + 3);
#pragma unroll
        for (int dt = 0; dt < 4; dt++) va[dt] = vaddr0[dt] + (uint32_t)((jl & 3) * kPTile);
        PipeAsm<T>::pv(o[0], o[1], o[2], o[3], px, va);
    }
    // blocks only later waves of the workgroup need: keep the barrier and load sequence
    for (int j = jl + 1; j < nkv; j++) {
        sync_blocks();
        load_k(j + 4);
        load_v(j + 3);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // nothing may land in LDS after the tile ends

    // ---- normalise and store: lane holds 4 consecutive d per register group ----------
#pragma unroll
    for (int qi = 0; qi < 2; qi++) {
        const int qpos = qw + 32 * qi + lrow;
        const float l_tot = half_sum(state[2 + qi]);
        const float inv = l_tot > 1e-10f ? 1.f / l_tot : 0.f;
        if (qpos < a.Sq) {
            T* orow = op + (int64_t)qpos * D;
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x32& acc = o[2 * qi + dt / 2];
                    const int b = 16 * (dt % 2) + 4 * g;
                    u32x2 w;
                    w.x = Mfma32A<T>::pack2(acc[b + 0] * inv, acc[b + 1] * inv);
                    w.y = Mfma32A<T>::pack2(acc[b + 2] * inv, acc[b + 3] * inv);
                    *reinterpret_cast<u32x2*>(orow + 32 * dt + 8 * g + 4 * lhalf) = w;
                }
        }
    }
    if (pass + 1 < npass) __syncthreads();                  // the rings are refilled for the next tile
    }
}

template <typename T, bool CAUSAL>
int launch_pipe(hipStream_t s, FaArgs a, int pair) {
    constexpr int kSmem = 2 * kPRing * kPTile;
    auto kern = fa_pipe_kernel<T, CAUSAL>;
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [&] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kSmem);
    });
    if (attr_err != hipSuccess)
        return fail(MHIP_ERR_LAUNCH, "flash_attention: cannot reserve %d bytes of LDS: %s", kSmem,
                    hipGetErrorString(attr_err));
    a.nqb = (a.Sq + kPBQ - 1) / kPBQ;
    const int64_t bh = (int64_t)a.B * a.H;
    // pairing halves the number of workgroups: only when they still fill the chip
    const int pair_env = pair >= 0 ? pair : tune_int("MHIP_FA_PAIR", -1);
    a.pair_tiles = CAUSAL && (pair_env >= 0 ? pair_env != 0 : bh * ((a.nqb + 1) / 2) >= 256);
    const int64_t grid = bh * (a.pair_tiles ? (a.nqb + 1) / 2 : a.nqb);
    if (grid > 0x7FFFFFFFLL) return fail(MHIP_ERR_UNSUPPORTED, "flash_attention: grid too large");
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), kSmem, s, a);
    return check_launch("flash_attention_pipe");
}

}  // namespace

// Head size 128, bf16 or f16, no mask operand, and enough 256-row query tiles to give every CU one
// (with fewer, the 128-row kernel's smaller workgroups spread better).  MHIP_FA_PIPE=2 turns
// the kernel off, MHIP_FA_PIPE=3 takes it whenever the shape allows.
// `variant`: 0 = decide here; 1 = the 128-row kernel; 2 / 3 = this kernel (unpaired / paired causal tiles) whenever
// the shape allows it -- what a tuning pass recorded or is timing.
bool fa_pipe_eligible(const FaArgs& a, int64_t D, int dtype, bool has_mask, int variant) {
    const int mode = tune_int("MHIP_FA_PIPE", 1);
    if (has_mask || D != kPD || (dtype != MHIP_BF16 && dtype != MHIP_F16) || a.Sq < kPBQ || a.Skv < 1) return false;
    if (variant) return variant != 1;
    if (mode == 2) return false;
    const int64_t tiles = (int64_t)a.B * a.H * ((a.Sq + kPBQ - 1) / kPBQ);
    return mode == 3 || tiles >= 256;
}

// `pair`: -1 = decide here, 0 / 1 = causal tiles unpaired / paired
int launch_fa_pipe(hipStream_t s, const FaArgs& a, int dtype, bool causal, int pair) {
    if (dtype == MHIP_BF16) return causal ? launch_pipe<bf16_t, true>(s, a, pair) : launch_pipe<bf16_t, false>(s, a, pair);
    if (dtype == MHIP_F16) return causal ? launch_pipe<f16_t, true>(s, a, pair) : launch_pipe<f16_t, false>(s, a, pair);
    return fail(MHIP_ERR_UNSUPPORTED, "flash_attention: pipelined kernel takes 16-bit types only");
}

}  // namespace mhip
