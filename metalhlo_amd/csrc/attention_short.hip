// Causal attention of up to 64 queries over up to 64 keys without a mask operand, 16-bit types, head sizes 64 and 128: a short prompt.
//
// What bounds it: latencies.  The kernels for longer sequences walk blocks of 64 keys through LDS behind barriers, which for one
// block is 2 us of latencies one after the other ([1,12,37,64] 4.4 us in a graph, of which a launch is 2.2).  Here a wave owns 32 query rows and
// asks for every query, key and value it will need in its first instructions, queries and keys straight into matrix operands, values
// into LDS of its own: neither a barrier nor a running maximum, 3.3 us.
//
// The products and sums are those of attention.hip's fa_fwd_kernel over one block of keys, in its order: a row has the same bits
// whether its sequence ends here or goes on.  (The 16x16x32 instruction, 16 rows a wave, adds up in another order; us, so | here:
// [1,12,37,64] 3.0 | 3.3, [8,32,64,64] 4.6 | 4.5, [64,32,64,64] 15.9 | 14.6, head size 128 [1,32,40] 4.0 | 4.3, [8,32,64] 6.6 | 6.2.)
#include "attention_short.h"

namespace mhip {
namespace {

constexpr int kRows = 32, kMostWaves = 2;

template <typename T, int D>
__global__ __launch_bounds__(64 * kMostWaves) void fa_short_kernel(FaArgs a) {
    __shared__ __attribute__((aligned(1024))) char smem[(1 + 2) * kRows * D * 2];
    const int bh = blockIdx.x;
    T* const o = static_cast<T*>(a.o) + bh / a.H * a.os[0] + bh % a.H * a.os[1];
    auto store = [&](int query, int d, u32x2 w) __attribute__((always_inline)) { *reinterpret_cast<u32x2*>(o + (int64_t)query * a.os[2] + d) = w; };
    // (a wave that sees half of the keys has half of the work, and is alone where there are no more rows)
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0) short_rows<T, D, 1>(a, bh, smem, store);
    else short_rows<T, D, 2>(a, bh, smem + kRows * D * 2, store);
}

template <typename T>
int launch_type(hipStream_t s, const FaArgs& a, int64_t D) {
    const dim3 grid((unsigned)(a.B * a.H)), block(64 * ((a.Sq + kRows - 1) / kRows));
    if (D == 128) hipLaunchKernelGGL((fa_short_kernel<T, 128>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fa_short_kernel<T, 64>), grid, block, 0, s, a);
    return check_launch("flash_attention_short");
}

}  // namespace

// us, fa_fwd_kernel | here, in a graph, up to 16 states in turn, D 64: [1,12,16] 4.1 | 2.7, [1,12,64] 4.5 | 3.5, [8,32,64] 5.9 | 4.5, [64,32,64] 17.7 | 14.6;
// D 128: [1,32,40] 5.7 | 4.3, [8,32,64] 8.1 | 6.2, [32,32,64] 18.8 | 16.2.  (GPT-2 launches this where attend_project does not serve: more than 64 tokens in all, or more heads times sequences than its waves.)
// Past 64 keys or without the causal rule 16 rows a wave were tried: they read the keys again for every 16 rows ([8,32,100] 6.9 | 7.8, every
// key for every query D 128 [16,32,64] 10.4 | 11.5).
bool fa_short_wanted(const FaArgs& a) { return a.is_causal && a.Sq <= kRows * kMostWaves && a.Skv <= 64; }

int launch_fa_short(hipStream_t s, const FaArgs& a, int64_t D, int dtype) {
    return dtype == MHIP_BF16 ? launch_type<bf16_t>(s, a, D) : launch_type<f16_t>(s, a, D);
}

}  // namespace mhip
