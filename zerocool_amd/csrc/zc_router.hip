// Router logits of long batches (reference: qwen.metal:512-534, metal.mm:818-822): sixteen contiguous K partitions of a row, a
// k-ascending multiply-accumulate chain in each, partials added 0..15.
#include "zc_kernels.hpp"
#include "zc_device.hpp"
#include "zc_affine_matrix.hpp"   // matrix_chain_step

namespace zc {

// The chains run on the matrix cores (rows a multiple of 128 long): a v_mfma_f32_4x4x1_16b_f32 is one fused multiply-add for each of
// sixteen partitions, four tokens and four experts, rounded as the chains' own.  A wave owns 4 TQ tokens x 4 EQ experts, a workgroup two
// waves of either.  Sixteen elements of every partition at a time go through LDS, so that a row's line is looked up once or twice per
// workgroup and not once for every sixteen bytes of it (a lane's pieces lie a partition apart), and the next sixteen wait in
// registers.  A piece of four fp32 elements stands at (quad of rows, lane that multiplies it, piece), turned by the lane so that sixteen
// lanes' reads meet all banks.
template <uint32_t TQ, uint32_t EQ>
__global__ __launch_bounds__(256, TQ * EQ == 16 ? 2 : 3) void router_matrix_kernel(const uint16_t* __restrict__ w, const float* __restrict__ x, uint32_t T, uint32_t K, uint32_t E,
                                                               const float* __restrict__ offsets, float* __restrict__ out) {
    constexpr uint32_t kTokens = 8 * TQ, kExperts = 8 * EQ, kSums = 16 * EQ;   // kSums: outputs of a wave's quad of tokens
    static_assert((kTokens + kExperts) * 64 * 4 >= 4 * kSums * 17);
    __shared__ __align__(16) uint4 lds[(kTokens + kExperts) * 64];
    uint4 *xs = lds, *ws = lds + kTokens * 64;
    // Neighbouring expert blocks of one token block share its rows: every die gets one stretch of the (token block, expert block) list.
    const uint32_t columns = (E + kExperts - 1) / kExperts, blocks = (T + kTokens - 1) / kTokens * columns, share = (blocks + 7) / 8;
    const uint32_t turn = blockIdx.x / 8, block = blockIdx.x % 8 * share + turn;
    if (turn >= share || block >= blocks) return;
    const uint32_t t0 = block / columns * kTokens, e0 = block % columns * kExperts, P = K / 16;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, j = lane & 3u, split = lane >> 2;
    const uint32_t tq0 = wave / 2 * TQ, eq0 = wave % 2 * EQ;
    // A thread moves, of every sixteen elements, piece tid % 4 of partition tid / 4 % 16 of four rows' inputs at a time, half tid % 2 of
    // partition tid / 2 % 16 of eight experts'.  (Past a partition's end: its last piece again, not used.)
    uint4 x_next[kTokens / 4], w_next[kExperts / 8];
    const uint32_t xq = tid % 4, xp = tid / 4 % 16, xr = tid / 64, wq = tid % 2, wp = tid / 2 % 16, wr = tid / 32;
    auto fetch = [&](uint32_t i0) {
#pragma unroll
        for (uint32_t u = 0; u < kTokens / 4; ++u) x_next[u] = ldg_u4(x + uint64_t(min(t0 + 4 * u + xr, T - 1)) * K + xp * P + min(i0 + 4 * xq, P - 4));
#pragma unroll
        for (uint32_t u = 0; u < kExperts / 8; ++u) w_next[u] = ldg_u4(w + uint64_t(min(e0 + 8 * u + wr, E - 1)) * K + wp * P + min(i0 + 8 * wq, P - 8));
    };
    auto place = [](uint32_t row, uint32_t part, uint32_t q) {
        const uint32_t l = part * 4 + row % 4;
        return (row / 4 * 64 + l) * 4 + (q + l / 4) % 4;
    };
    f32x4 c[TQ][EQ];
#pragma unroll
    for (uint32_t t = 0; t < TQ; ++t)
#pragma unroll
        for (uint32_t e = 0; e < EQ; ++e) c[t][e] = f32x4{0, 0, 0, 0};
    fetch(0);
    for (uint32_t i0 = 0; i0 < P; i0 += 16) {
        lds_barrier();   // the sixteen before have been read
#pragma unroll
        for (uint32_t u = 0; u < kTokens / 4; ++u) xs[place(4 * u + xr, xp, xq)] = x_next[u];
#pragma unroll
        for (uint32_t u = 0; u < kExperts / 8; ++u) {
            const uint4 v = w_next[u];
            ws[place(8 * u + wr, wp, 2 * wq)] = make_uint4(v.x << 16, v.x & 0xffff0000u, v.y << 16, v.y & 0xffff0000u);
            ws[place(8 * u + wr, wp, 2 * wq + 1)] = make_uint4(v.z << 16, v.z & 0xffff0000u, v.w << 16, v.w & 0xffff0000u);
        }
        lds_barrier();
        if (i0 + 16 < P) fetch(i0 + 16);
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {   // four elements of every partition
            if (q == 2 && i0 + 8 >= P) break;
            uint4 wv[EQ], xv[TQ];
#pragma unroll
            for (uint32_t e = 0; e < EQ; ++e) wv[e] = ws[((eq0 + e) * 64 + lane) * 4 + (q + lane / 4) % 4];
#pragma unroll
            for (uint32_t t = 0; t < TQ; ++t) xv[t] = xs[((tq0 + t) * 64 + lane) * 4 + (q + lane / 4) % 4];
            auto element = [](const uint4& v, int k) { return __uint_as_float(k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w); };
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (uint32_t t = 0; t < TQ; ++t)
#pragma unroll
                    for (uint32_t e = 0; e < EQ; ++e) c[t][e] = matrix_chain_step(element(xv[t], k), element(wv[e], k), c[t][e]);
        }
    }
    lds_barrier();
    // the partials added 0..15, four tokens at a time; register r of a lane: token r, expert j
    float* partial = reinterpret_cast<float*>(lds) + wave * (kSums * 17);
#pragma unroll
    for (uint32_t t = 0; t < TQ; ++t) {
#pragma unroll
        for (uint32_t e = 0; e < EQ; ++e)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) partial[(r * 4 * EQ + 4 * e + j) * 17 + split] = c[t][e][r];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < 16; ++i) sum += partial[min(lane, kSums - 1) * 17 + i];
        const uint32_t token = t0 + (tq0 + t) * 4 + lane / (4 * EQ), expert = e0 + eq0 * 4 + lane % (4 * EQ);
        if (lane < kSums && token < T && expert < E) out[uint64_t(token) * E + expert] = offsets ? sum + offsets[expert] : sum;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}
// Blocks are few, and all of one cost: what counts is how many of them the fullest compute unit gets.  A round of one block on each
// of the 256 takes, behind the 4.6 us of a launch's first loads and last sums, 4.2 us with 16 x 16 tokens and experts of 2048 inputs, 7.2 with 16 x
// 32 and 13.5 with 32 x 32, and the block is the one with the cheapest rounds.  us before (chains on the vector unit) -> here, 512
// experts, 2048 inputs: 96 tokens 28.5 -> 9.0, 300 32 -> 17.4, 512 36 -> 18.8, 800 61 -> 30, 1500 93 -> 45, 2048 122 -> 58; 3072
// inputs, 1500 tokens 118 -> 65.  The instructions alone, back to back at 4.3 ns each, are 35 of the 58 us.
void launch_router_batch(hipStream_t s, const void* w, const float* x, uint32_t T, uint32_t K, uint32_t E, const float* offsets, float* out) {
    auto blocks_of = [&](uint32_t tokens, uint32_t experts) { return ((T + tokens - 1) / tokens) * ((E + experts - 1) / experts); };
    auto cost_of = [&](uint32_t blocks, uint32_t round) { return uint64_t(blocks + 255) / 256 * round; };
    const uint32_t small = blocks_of(16, 16), middle = blocks_of(16, 32), large = blocks_of(32, 32);
    const uint64_t cost_small = cost_of(small, 42), cost_middle = cost_of(middle, 72), cost_large = cost_of(large, 135);
#define ZC_ROUTER(TQ, EQ, blocks) hipLaunchKernelGGL((router_matrix_kernel<TQ, EQ>), dim3((blocks + 7) / 8 * 8), dim3(256), 0, s, (const uint16_t*)w, x, T, K, E, offsets, out)
    if (cost_small <= cost_middle && cost_small <= cost_large) ZC_ROUTER(2, 2, small);
    else if (cost_middle < cost_large) ZC_ROUTER(2, 4, middle);
    else ZC_ROUTER(4, 4, large);
#undef ZC_ROUTER
}

}  // namespace zc
