// Prefill path of the MoE layer: tokens sorted by expert, then a grouped GEMM on the bf16 matrix cores with
// fp32 accumulation (the reference batches the same work per expert in encode_expert_rows, src/engine/pipeline.cpp:7-31,
// over q4_mm / q4_gate_up, kernels/metal/qwen.metal:289-376).
//
// Arithmetic.  The reference evaluates, per 16-element block, scale * sum(x q) + bias * sum'(x) with sum' the
// BF16-rounded sum-of-four chain (qwen.metal:46-62).  Here the products x * q run on v_mfma_f32_16x16x32_bf16: x is
// BF16-valued (exact as a bf16 operand), products are exact and accumulate in fp32 over one scale group of 64; per group
// the accumulator is folded as  total += scale * dot.  The bias half, sum over the groups of bias * chain sum, is a product
// over the group index and runs on the matrix cores too, four groups at a time between their dots, the chain sums cut into
// three bf16 pieces that add up to them exactly.  Only the order of the fp32 additions
// differs from the reference, so results agree to a few fp32 steps before the BF16 rounding of the outputs.  Every sum
// that lands within prefill_margin(K) of its term magnitudes of a BF16 rounding boundary is then recomputed with the reference's exact
// lane arithmetic (0.2 to 0.5 % of the sums up to 2048 inputs, 1.1 % at 4096; a gate/up element has two), which removes the rounding flips in practice; the path is still
// specified by a tolerance (max relative error 2e-3 of the layer output), not as bit-exact.  Routing, dispatch and the
// combine use the exact kernels.
//
// Codes as operands.  A nibble, read as an 8-bit float of four exponent and three mantissa bits, is the number code * 2^-9: one
// conversion instruction makes two bf16 codes of two of them and takes the 2^9 back.  Bytes go over floats, three instructions per
// two codes.  (The bit pattern of a code is the bf16 number code * 2^-133, which the matrix cores take at full precision without
// any conversion.  But an instruction drops what lies 24 bits below its largest sum of exponents, and a subnormal operand
// counts there as 2^-126, up to seven bits above its value: beside a large input that met a small code the other products
// lost those bits.  Rows with one input of 2^10 per group on codes 1 to 3, 2048 inputs, root mean square error in 2^-24 of the
// terms' magnitudes: nibbles 1.67, bytes 19.5; converted 0.48 and 0.46.  The layer of 2048 tokens of hidden 2048
// takes 626 us with either, 1500 tokens of hidden 3072 1195 us with the conversion and 1197 without, 300 of the mixed artifact 389 and 390.)
// The even nibbles of a word share one mask and the odd ones another, so the rows are stored with every eight elements in the
// order 0 2 4 6 1 3 5 7.  Groups whose sums could leave the range of exact products (|x| >= 2^100, all below 2^-60, inf, NaN) get a
// NaN chain sum: every output of such a row is then recomputed with the lane arithmetic.
//
// Tiling.  One workgroup (4 waves) owns up to 48 sorted token rows of ONE expert and 128 weight rows (gate/up: 64 gate rows
// and the 64 up rows of the same indices, so SwiGLU is fused in registers), and walks K in steps of 128 = two scale
// groups.  Each wave multiplies all (one to three) 16-row blocks of the tokens by 2 of the 8 column tiles: the codes
// and scales of its 32 weight rows go from memory straight into the lanes that use them, the token rows are
// gathered into LDS as bf16, double-buffered, and chain sums and biases of all groups are brought into LDS once.  An expert's
// rows are cut into tiles of 32, except
// that a run of up to 48 rows (a whole expert with few rows, or the last rows of a longer run) is ONE tile: with about
// forty rows per expert -- an unskewed router at 2048 tokens -- every expert's codes are then expanded once, not twice.
#include <algorithm>
#include <type_traits>
#include "zc_kernels.hpp"
#include "zc_prefill_tiles.hpp"
#include "zc_device.hpp"
#include "zc_decode_common.hpp"   // lds_barrier; route_token: top-k + softmax of one token by one wavefront

namespace zc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kPitch = 136;   // LDS row pitch in bf16 elements: 128 elements of a row, sixteen rows on different banks

// What the matrix-core products and the recomputation need of their token rows, from fp32 rows holding BF16 values (F32)
// or from bf16 rows in the operand's order (the SwiGLU activations): a thread takes four neighbouring elements, so loads and stores are whole runs.
//   xb      the row as bf16 (F32 only, and only for the router on bounds)
//   xp      the row as bf16, every eight elements in the order 0 2 4 6 1 3 5 7: the matrix-core operand (F32 only: the product kernel leaves the
//           activations in that order)
//   planes  per (row, group of 64) the group's input sum as three bf16 pieces, [row][piece][prefill_pitch(K)]: the four
//           blocks' BF16-rounded sum-of-four chains (Q4 lanes), NaN where the group leaves the operand's exact range
//   plain   the same of the plain fp32 sums (Q8 lanes, qwen.metal:112-125: sum += v, element by element in blocks of eight)
// status bit 4: a value was not BF16-valued.
__device__ __forceinline__ void store_pieces(uint16_t* at, uint32_t pitch, float v) {
    const uint32_t hi = __float_as_uint(v) & 0xffff0000u;
    const float rest = v - __uint_as_float(hi);
    const uint32_t mid = __float_as_uint(rest) & 0xffff0000u;
    at[0] = uint16_t(hi >> 16); at[pitch] = uint16_t(mid >> 16); at[2 * pitch] = uint16_t(__float_as_uint(rest - __uint_as_float(mid)) >> 16);
}
//
// The workgroups behind the rows', if norm_rows is not 0, leave |row| of the router's rows for the router on bounds, one wavefront a row.
// |row| is rounded up a little.  A row so small that its squares leave the normal range has no usable norm: +inf makes the router
// recompute everything.
__device__ __forceinline__ float squares_of(uint4 v, float sum) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float lo = __uint_as_float(w[q] << 16), hi = __uint_as_float(w[q] & 0xffff0000u);
        sum = __builtin_fmaf(lo, lo, sum); sum = __builtin_fmaf(hi, hi, sum);
    }
    return sum;
}
__device__ __forceinline__ float row_norm(float lane_squares) {
#pragma unroll
    for (int o = 32; o; o >>= 1) lane_squares += __shfl_xor(lane_squares, o);
    return lane_squares < 0x1p-100f ? __uint_as_float(0x7f800000u) : sqrtf(lane_squares) * 1.0001f;
}
template <bool F32>
__global__ __launch_bounds__(256) void prefill_rows_kernel(const void* x, uint32_t rows, uint32_t K, uint16_t* xb, uint16_t* xp, uint16_t* planes, uint16_t* plain,
                                                           int32_t* status, const uint16_t* norm_of, uint32_t norm_rows, float* norms) {
    const uint32_t quads = K / 4, i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63u;
    if constexpr (F32) {
        const uint32_t before = (rows * quads + 255) / 256;
        if (blockIdx.x >= before) {
            const uint32_t row = (blockIdx.x - before) * 4 + threadIdx.x / 64;
            if (row >= norm_rows) return;
            float sum = 0;
            for (uint32_t k = lane * 8; k < K; k += 512) sum = squares_of(ldg_u4(norm_of + uint64_t(row) * K + k), sum);
            const float norm = row_norm(sum);
            if (lane == 0) norms[row] = norm;
            return;
        }
    }
    if (i >= rows * quads) return;               // (whole groups of sixteen lanes: K is a multiple of 128)
    const uint32_t r = i / quads, c = i % quads, pitch = prefill_pitch(K);
    float v[4];
    if constexpr (F32) {
        const float4 q = reinterpret_cast<const float4*>(x)[i];
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        uint32_t low = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) low |= __float_as_uint(v[k]) & 0xffffu;
        if (low) atomicOr(status, 4);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = __uint_as_float(__float_as_uint(v[k]) & 0xffff0000u);
        if (xb) reinterpret_cast<uint2*>(xb)[i] = make_uint2((__float_as_uint(v[0]) >> 16) | __float_as_uint(v[1]), (__float_as_uint(v[2]) >> 16) | __float_as_uint(v[3]));
    } else {
        const uint2 q = reinterpret_cast<const uint2*>(x)[i];   // a pair's even lane: elements 0 2 | 4 6, the odd one 1 3 | 5 7
        const bool odd = lane & 1u;
        const uint32_t other = uint32_t(__shfl_xor(int(odd ? q.x : q.y), 1)), even = odd ? other : q.x, uneven = odd ? q.y : other;
        v[0] = __uint_as_float(even << 16); v[1] = __uint_as_float(uneven << 16); v[2] = __uint_as_float(even & 0xffff0000u); v[3] = __uint_as_float(uneven & 0xffff0000u);
    }
    uint32_t largest = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) largest = max(largest, __float_as_uint(v[k]) & 0x7fffffffu);
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) largest = max(largest, uint32_t(__shfl_xor(int(largest), o)));
    const bool strange = largest >= 0x71800000u || (largest != 0 && largest < 0x21800000u);   // 2^100, 2^-60
    if constexpr (F32) {   // lane 2m of a pair holds elements 0..3, lane 2m + 1 elements 4..7: 0 2 4 6 | 1 3 5 7
        const uint32_t even = (__float_as_uint(v[0]) >> 16) | __float_as_uint(v[2]), uneven = (__float_as_uint(v[1]) >> 16) | __float_as_uint(v[3]);
        const bool odd = lane & 1u;
        const uint32_t other = uint32_t(__shfl_xor(int(odd ? even : uneven), 1));
        reinterpret_cast<uint2*>(xp)[i] = odd ? make_uint2(other, uneven) : make_uint2(even, other);
    }
    const uint32_t group = r * (3 * pitch) + c / 16, base = lane & ~15u;
    if (planes) {
        const float quad = bf(bf(bf(v[0] + v[1]) + v[2]) + v[3]);
        float sum = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) sum += __shfl(quad, int((lane & ~3u) + uint32_t(k)));
        float total = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) total += __shfl(sum, int(base + 4u * uint32_t(k)));
        if ((lane & 15u) == 0) store_pieces(planes + group, pitch, strange ? __uint_as_float(0x7fc00000u) : total);
    }
    if (plain) {
        const float head = (((0.0f + v[0]) + v[1]) + v[2]) + v[3], before = __shfl_xor(head, 1);
        const float eight = (((before + v[0]) + v[1]) + v[2]) + v[3];       // (of odd lanes)
        float total = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) total += __shfl(eight, int(base + 2u * uint32_t(k) + 1u));
        if ((lane & 15u) == 0) store_pieces(plain + group, pitch, strange ? __uint_as_float(0x7fc00000u) : total);
    }
}

// Work list: tile t = (expert, first sorted position, rows).  offsets[e] .. offsets[e+1] are the expert's sorted
// positions (the dispatch kernel's output); a null offsets pointer means ONE group of `rows` rows (the shared expert).
__global__ __launch_bounds__(1024) void prefill_tiles_kernel(const int32_t* offsets, uint32_t experts, uint32_t rows, int32_t* tile_expert,
                                                            int32_t* tile_first, int32_t* tile_rows, int32_t* tile_count) {
    __shared__ int32_t scan[1024];
    const uint32_t e = threadIdx.x;
    const int32_t first = offsets ? (e < experts ? offsets[e] : 0) : 0, count = offsets ? (e < experts ? offsets[e + 1] - offsets[e] : 0) : (e == 0 ? int32_t(rows) : 0);
    const int32_t tiles = prefill_tiles_of(count);
    scan[e] = tiles;
    __syncthreads();
    for (uint32_t step = 1; step < 1024; step <<= 1) {
        const int32_t add = e >= step ? scan[e - step] : 0;
        __syncthreads();
        scan[e] += add;
        __syncthreads();
    }
    const int32_t begin = scan[e] - tiles;
    for (int32_t t = 0; t < tiles; ++t) {
        tile_expert[begin + t] = int32_t(e); tile_first[begin + t] = first + t * int32_t(kTileRows);
        tile_rows[begin + t] = t + 1 < tiles ? int32_t(kTileRows) : count - t * int32_t(kTileRows);   // the last tile takes what is left (at most 48)
    }
    if (e == 1023) *tile_count = scan[1023];
}

// The dispatch sort of a long batch and the routed experts' work list in ONE launch (the decode path's three dispatch
// kernels and prefill_tiles_kernel hold the same steps as four launches in a row, each of them short: what they cost was
// the four launches).  A workgroup = sixteen experts (one per wave) x one of kDispatchParts stretches of the slots.  Every
// workgroup counts ALL the slots' experts, per stretch, into a table in LDS and keeps its own stretch of the ids there;
// it scans the table (sorted offsets and tile counts of every expert), and each wave then places its expert's slots of
// the workgroup's stretch in ascending slot order, starting where the earlier stretches' slots of that expert end.  The
// workgroups of the first stretch also write their experts' tiles, workgroup (0, 0) the offsets.  Same results as
// launch_dispatch followed by launch_prefill_tiles; the list of selected experts is not written (nothing here reads it).
// (Workgroups of sixteen waves and not of four: 20480 slots 23 -> 17.6 us beside the shared expert's product, 17.4 -> 13.2 alone.)
// ids sixteen-byte aligned; stretch: slots per stretch, a multiple of 1024.
constexpr uint32_t kDispatchParts = 4, kDispatchThreads = 1024;
__global__ __launch_bounds__(kDispatchThreads) void prefill_dispatch_kernel(const int32_t* __restrict__ ids, uint32_t n, uint32_t topk, uint32_t E, uint32_t stretch,
                                                               int32_t* __restrict__ offsets, int32_t* __restrict__ slots, int32_t* __restrict__ rows, int32_t* status,
                                                               int32_t* tile_expert, int32_t* tile_first, int32_t* tile_rows, int32_t* tile_count) {
    extern __shared__ __align__(16) int32_t table[];   // [parts][E] counts, [E + 1] offsets, [E + 1] tiles before, then the stretch's ids
    __shared__ int32_t wave_sum[2][kDispatchThreads / 64];
    int32_t* cnt = table; int32_t* off = table + kDispatchParts * E; int32_t* tiles_before = off + E + 1;
    int32_t* copy = table + ((kDispatchParts + 2) * E + 2 + 3) / 4 * 4;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, part = blockIdx.y, first = part * stretch;
    for (uint32_t i = tid; i < kDispatchParts * E; i += kDispatchThreads) cnt[i] = 0;
    __syncthreads();
    {
        int bad = 0;
        constexpr int kSteps = 5;                                       // steps' loads in flight: 20480 slots in one go
        for (uint32_t b0 = 0; b0 < n; b0 += kSteps * 4 * kDispatchThreads) {
            int4 batch[kSteps];
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                const uint32_t p = b0 + (u * kDispatchThreads + tid) * 4;
                int4 v = make_int4(-1, -1, -1, -1);   // (-1: past the end)
                if (p + 3 < n) v = *reinterpret_cast<const int4*>(ids + p);
                else { if (p < n) v.x = ids[p]; if (p + 1 < n) v.y = ids[p + 1]; if (p + 2 < n) v.z = ids[p + 2]; }
                batch[u] = v;
            }
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                const uint32_t p = b0 + (u * kDispatchThreads + tid) * 4, at = (p >= stretch ? 1u : 0u) + (p >= 2 * stretch ? 1u : 0u) + (p >= 3 * stretch ? 1u : 0u);   // its stretch
                if (p >= (n + 255) / 256 * 256) break;   // (the last 256 slots are looked at as a whole: -1 past the end)
                const int32_t four[4] = {batch[u].x, batch[u].y, batch[u].z, batch[u].w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (p + j >= n) continue;
                    if (four[j] < 0 || four[j] >= int32_t(E)) bad = 1; else atomicAdd(&cnt[at * E + uint32_t(four[j])], 1);
                }
                if (at == part) *reinterpret_cast<int4*>(copy + (p - first)) = batch[u];
            }
        }
        if (bad && blockIdx.x == 0 && part == 0) atomicOr(status, 1);
    }
    __syncthreads();
    auto count_of = [&](uint32_t e) { int32_t c = 0; for (uint32_t q = 0; q < kDispatchParts; ++q) c += cnt[q * E + e]; return c; };
    {   // exclusive scans over the experts, one a thread
        const int32_t c = tid < E ? count_of(tid) : 0, mine[2] = {c, prefill_tiles_of(c)};
        int32_t incl[2] = {mine[0], mine[1]};
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
#pragma unroll
            for (int v = 0; v < 2; ++v) { const int32_t up = __shfl_up(incl[v], o); if (int(lane) >= o) incl[v] += up; }
        if (lane == 63) { wave_sum[0][wave] = incl[0]; wave_sum[1][wave] = incl[1]; }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            int32_t at = incl[v] - mine[v];
            for (uint32_t w = 0; w < wave; ++w) at += wave_sum[v][w];
            int32_t* to = v ? tiles_before : off;
            if (tid < E) to[tid] = at;
            if (tid + 1 == E) to[E] = at + mine[v];
        }
        __syncthreads();
    }
    if (blockIdx.x == 0 && part == 0) {
        for (uint32_t e = tid; e <= E; e += kDispatchThreads) offsets[e] = off[e];
        if (tid == 0) *tile_count = tiles_before[E];
    }
    const uint32_t e = blockIdx.x * (kDispatchThreads / 64) + wave;
    if (e >= E) return;
    const int32_t count = count_of(e);
    if (count == 0) return;
    if (part == 0) {   // the expert's tiles: whole tiles of 32 rows, the last one takes what is left (at most 48)
        const int32_t tiles = tiles_before[e + 1] - tiles_before[e], begin = tiles_before[e];
        for (int32_t t = int32_t(lane); t < tiles; t += 64) {
            tile_expert[begin + t] = int32_t(e); tile_first[begin + t] = off[e] + t * int32_t(kTileRows);
            tile_rows[begin + t] = t + 1 < tiles ? int32_t(kTileRows) : count - t * int32_t(kTileRows);
        }
    }
    int32_t pos = off[e];
    for (uint32_t q = 0; q < part; ++q) pos += cnt[q * E + e];
    const int32_t end = pos + cnt[part * E + e];
    const uint64_t below = (1ull << lane) - 1;
    const float inverse = 1.0f / float(topk);
    // 256 slots per step, in order: four neighbouring slots per lane, slots of lower lanes first, then the lane's own
    for (uint32_t q0 = first; q0 < n && q0 < first + stretch && pos < end; q0 += 256) {
        const uint32_t p = q0 + 4 * lane;
        const int4 v = *reinterpret_cast<const int4*>(copy + (p - first));
        const bool m[4] = {v.x == int32_t(e), v.y == int32_t(e), v.z == int32_t(e), v.w == int32_t(e)};
        const uint64_t mask[4] = {__ballot(m[0]), __ballot(m[1]), __ballot(m[2]), __ballot(m[3])};
        if ((mask[0] | mask[1] | mask[2] | mask[3]) == 0) continue;   // uniform: none of these 256 slots is the expert's
        int32_t at = pos + __popcll(mask[0] & below) + __popcll(mask[1] & below) + __popcll(mask[2] & below) + __popcll(mask[3] & below);
        // token and rank of slot p (p < 2^24: the rounded quotient is off by one at most)
        uint32_t token = uint32_t(float(p) * inverse);
        int32_t rest = int32_t(p) - int32_t(token * topk);
        if (rest < 0) { --token; rest += int32_t(topk); } else if (rest >= int32_t(topk)) { ++token; rest -= int32_t(topk); }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (m[j]) { slots[at] = int32_t(p + j); if (rows) rows[at] = int32_t(token); ++at; }
            if (++rest == int32_t(topk)) { rest = 0; ++token; }
        }
        pos += __popcll(mask[0]) + __popcll(mask[1]) + __popcll(mask[2]) + __popcll(mask[3]);
    }
}

// codes -> matrix-core operand, element order 0 2 4 6 1 3 5 7: eight nibbles of a word, or eight bytes of two words
__device__ __forceinline__ bf16x8 nibble_operand(uint32_t word) {
    const uint32_t even = word & 0x0f0f0f0fu, odd = (word >> 4) & 0x0f0f0f0fu;
    auto two = [](bf16x2 v) { return __builtin_bit_cast(uint32_t, v); };
    return __builtin_bit_cast(bf16x8, make_uint4(two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 512.0f, false)), two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 512.0f, true)),
                                                 two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 512.0f, false)), two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 512.0f, true))));
}
__device__ __forceinline__ bf16x8 byte_operand(uint32_t lo, uint32_t hi) {
    auto two = [](uint32_t word, int i) {   // bytes i and i + 2: whole numbers up to 255 have all their bits in a float's upper half
        return __builtin_amdgcn_perm(__float_as_uint(float((word >> (8 * i + 16)) & 0xffu)), __float_as_uint(float((word >> (8 * i)) & 0xffu)), 0x07060302u);
    };
    return __builtin_bit_cast(bf16x8, make_uint4(two(lo, 0), two(hi, 0), two(lo, 1), two(hi, 1)));
}
// A sum v, terms of magnitude m, close to a BF16 rounding boundary could round
// the other way under the reference's order of additions: it is marked for exact recomputation if v - e and v + e round apart, e
// the margin and what forming v - e and v + e may lose.  Where they do not, both are v's BF16 value.  (A magnitude that is not
// finite, of a row or group that left the operand's range, marks the sum.)
// (Seven instructions a sum; a rounding of its own and the distance from it were sixteen, a layer of 2048 tokens of hidden 2048 582 -> 572 us,
// 1500 of hidden 3072 1053 -> 1043.)
__device__ __forceinline__ uint32_t prefill_round(float v, float m, float margin, bool& near) {
    const float e = __builtin_fmaf(fabsf(v), 0x1p-24f, m * margin), low = v - e, high = v + e;
    const uint32_t both = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{low, high}, bf16x2));
    near = !(low <= high) || (both & 0xffffu) != both >> 16;
    return both << 16;
}
// One tile: up to 16 NB rows of one expert x 128 weight rows.  BITS: 4 (nibble codes) or 8 (byte codes; the planes are then
// the plain sums of the Q8 lanes).  The number of row blocks is a compile-time value, so that the walk over K is straight-line
// code: as a run-time bound it cut every step into short blocks that each waited for its own LDS reads.
//
// The walk goes two scale groups (128 elements) at a time, weights and token rows one such pair ahead.  What bounds it is
// the SIMDs' issue: per wave and pair, three row blocks, Q4, 27 matrix-core instructions (7.7 ns each) and 171 vector ones (1.0 to
// 1.5 ns; the listing of the loop: 54 and 342 per two pairs),
// which overlap only in part -- weights and rows read from a warm cache leave the time of the walk unchanged.  A wave
// alone issues one vector instruction every five clocks, so the registers are kept to what three waves per SIMD allow
// (Q4: 156 and 160 of 168; with a second set of token rows or four pairs of weights in flight two waves fit, and the layer of
// hidden 2048 took 680 us at 2048 tokens where it took 621 then).  At that size the routed gate/up product takes 240 us (369 with a run-time number of
// row blocks, codes converted one by one and the scales staged through LDS); the down product of its rows of 512 is prefill_short_tile's.
template <bool GATED, int BITS, int NB>
__device__ __forceinline__ void prefill_tile(const PrefillGemm& p, uint16_t* a_s, uint16_t* marks_s, uint16_t* bias_s, uint32_t expert, uint32_t first, uint32_t rows, uint32_t n0) {
    constexpr int kAhead = 2, kRegs = BITS;       // pairs of groups in flight; dwords of a column tile's pair per lane
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, j = lane & 15u, g4 = lane >> 4;
    const uint32_t K = p.K, N = p.N, groups = K / 64, pairs = K / 128;
    const uint8_t* record = p.records + uint64_t(expert) * p.stride;
    // What a workgroup needs before its walk is requested in one go, the indices of its rows first: loads return in the order they were
    // sent, and only the rows have to wait for an answer.  (Indices, rows, biases and chain sums one after the other were four more
    // latencies of a workgroup that lives about ten.  us a layer: 2048 tokens of hidden 2048 642 -> 618, 700 397 -> 377, 300 of the mixed artifact 365 ->
    // 342, 1500 of hidden 3072 1190 -> 1143.  With that the bytes in flight are enough: tiles of sixteen rows in a kernel with four pairs
    // of weights in flight and four waves a SIMD took 304 us for 200 tokens where this takes 302, and 433 where this takes 369, 300 tokens of
    // hidden 3072 behind Zipf(1.1) offsets.)
    // Row of `a` for row m of the tile; rows past the end repeat the last one (never stored).  Thread: sixteen bytes of one row of every block.
    uint32_t a_row[NB];
#pragma unroll
    for (int rb = 0; rb < NB; ++rb) {
        const uint32_t pos = first + min(16 * uint32_t(rb) + (tid >> 4), rows - 1);
        a_row[rb] = pos;
        if constexpr (GATED) {   // (without a list of rows: a word that is there, not used)
            const uint32_t listed = *as_global<uint32_t>(p.a_rows ? p.a_rows + pos : p.tile_count);
            a_row[rb] = p.a_rows ? listed : pos;
        }
    }
    // The wave's two column tiles (rows of the workgroup's 128 weight rows) for every block of sixteen token rows; gate/up:
    // a gate tile and the up tile of the same rows.  The codes go from memory straight into the lanes that feed them to
    // the matrix cores, whole 64-byte pieces of a row per load.
    // (Bases are the same in every lane, lanes add 32-bit offsets.)
    const uint8_t *codes_of[2], *scales_of[2], *biases_of[2];
    uint32_t b_at[2], m_at[2];                   // the lane's weight row: bytes from the bases
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint32_t proj = GATED ? uint32_t(q) : 0u, n = n0 + (GATED ? wave * 16u : (2 * wave + uint32_t(q)) * 16u) + j;
        codes_of[q] = record + p.off[proj * 3]; scales_of[q] = record + p.off[proj * 3 + 1]; biases_of[q] = record + p.off[proj * 3 + 2];
        b_at[q] = n * (K * BITS / 8) + g4 * 16; m_at[q] = n * groups * 2;
    }
    u32x4 ring[kAhead][2][kRegs / 4];
    auto fetch_b = [&](uint32_t pair, u32x4 (&to)[2][kRegs / 4]) {
        const uint32_t at = min(pair, pairs - 1) * (16 * BITS);   // (past the end: the last pair again, not used)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int h = 0; h < kRegs / 4; ++h) to[q][h] = *as_global<u32x4>(codes_of[q] + (b_at[q] + at + 64u * uint32_t(h)));
    };
#pragma unroll
    for (int d = 0; d + 1 < kAhead; ++d) fetch_b(uint32_t(d), ring[d]);
    // The scales of the lane's two weight rows, four groups per load (the four lanes of a row fetch the same bytes), one load
    // ahead.  (In LDS, filled by a loop of dependent loads and stores before the walk, they cost 11 us of a workgroup's
    // 29: nearly as much as the walk.)  A row's last load may run into the rows behind it, which the biases always follow.
    uint32_t scales[2][2], scales_next[2][2];
    auto fetch_s = [&](uint32_t g) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint2 v = ldg_u2_by_words(scales_of[q] + (m_at[q] + min(g, (groups - 1) / 4 * 4) * 2));
            scales_next[q][0] = v.x; scales_next[q][1] = v.y;
        }
    };
    fetch_s(0);
    // biases of eight groups of the lane's two weight rows, for up to 64 groups (past the end: not used)
    const uint32_t pitch = prefill_pitch(K);
    uint4 bias_first[2][2];
    auto fetch_biases = [&](int part) {
        const uint32_t mine = 32 * uint32_t(part) + 8 * g4;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (groups % 8 == 0) bias_first[part][q] = ldg_u4_by_words(biases_of[q] + (m_at[q] + min(mine, groups - 8) * 2));
            else {
                uint32_t w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] = ldg_u32(biases_of[q] + (m_at[q] + min(mine + 2 * uint32_t(i), groups - 2) * 2));
                bias_first[part][q] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
    };
    fetch_biases(0);
    if (groups > 32) fetch_biases(1);
    const uint16_t* a_src[NB];
    const uint32_t a_at = (tid >> 4) * kPitch + (tid & 15u) * 8;
#pragma unroll
    for (int rb = 0; rb < NB; ++rb) a_src[rb] = p.a + uint64_t(a_row[rb]) * K + (tid & 15u) * 8;
    u32x4 a_next[NB];
    auto fetch_a = [&](uint32_t pair, u32x4 (&to)[NB]) {
#pragma unroll
        for (int rb = 0; rb < NB; ++rb) to[rb] = *as_global<u32x4>(a_src[rb] + min(pair, pairs - 1) * 128);
    };
    auto stash_a = [&](uint32_t buf, const u32x4 (&from)[NB]) {
#pragma unroll
        for (int rb = 0; rb < NB; ++rb) *reinterpret_cast<u32x4*>(a_s + (buf * kTileRowsMax + 16 * uint32_t(rb)) * kPitch + a_at) = from[rb];
    };
    u32x4 a_first[NB];
    fetch_a(0, a_first); fetch_a(1, a_next);
    // chain sums: the rows' pieces as they lie in memory, sixteen threads a row
    const uint32_t octets = pitch / 8, row_octets = 3 * octets;
    uint4 sums_first[2][NB];
    auto fetch_sums = [&](int part) {
#pragma unroll
        for (int rb = 0; rb < NB; ++rb) sums_first[part][rb] = ldg_u4(p.planes + uint64_t(a_row[rb]) * (3 * pitch) + min(16 * uint32_t(part) + (tid & 15u), row_octets - 1) * 8);
    };
    fetch_sums(0);
    if (groups > 32) fetch_sums(1);
    f32x4 total[NB][2], mag[NB][2];   // mag: sum of the magnitudes of the folded terms, the scale of the rounding error
#pragma unroll
    for (int rb = 0; rb < NB; ++rb)
#pragma unroll
        for (int q = 0; q < 2; ++q) total[rb][q] = mag[rb][q] = f32x4{0, 0, 0, 0};
    // The bias half of the totals, sum over the groups of bias * chain sum, runs on the matrix cores, four groups per
    // instruction: quarter g4 of the operand holds piece g4 of the chain sums (the last one zeros).  A group's bias half mostly
    // cancels its dot, so the four are added in the middle of the same groups' dots: the running totals, which the rounding
    // errors go with, stay small.  Root mean square error against 64 bits in 2^-24 of the terms' magnitudes, biases of -8 scales,
    // 512, 2048 and 4096 inputs: 0.19, 0.14, 0.13; a multiply-add per group, the order that errs least, 0.19, 0.15, 0.14; all of the
    // bias half in front of the walk 0.22, 0.23, 0.24.  (Eight groups at once in front of their dots 0.22, 0.17, 0.15.)  The layer of
    // 2048 tokens of hidden 2048 takes 628 us, with all of it in front of the walk 620; 1500 tokens of hidden 3072 1166 and 1192.
    // Chain sums and biases wait in LDS, zeros behind the last group.
    uint16_t *planes_s = bias_s + 8, *biases_s = planes_s + kTileRowsMax * 3 * pitch;
    const uint32_t col[2] = {(GATED ? wave : 2 * wave) * 16 + j, (GATED ? 4 + wave : 2 * wave + 1) * 16 + j};
    if (tid < 4) reinterpret_cast<uint32_t*>(bias_s)[tid] = 0;
    auto store = [&](uint16_t* at, uint4 v, uint32_t g) {   // of the groups g .. g + 7
        *reinterpret_cast<uint4*>(at) = make_uint4(v.x, g + 2 < groups ? v.y : 0u, g + 4 < groups ? v.z : 0u, g + 6 < groups ? v.w : 0u);
    };
    auto store_first = [&](int part) {
        const uint32_t mine = 32 * uint32_t(part) + 8 * g4, i = 16 * uint32_t(part) + (tid & 15u), piece = (i >= octets ? 1u : 0u) + (i >= 2 * octets ? 1u : 0u);
        if (mine < pitch) {
#pragma unroll
            for (int q = 0; q < 2; ++q) store(biases_s + col[q] * pitch + mine, bias_first[part][q], mine);
        }
        if (i < row_octets) {
#pragma unroll
            for (int rb = 0; rb < NB; ++rb) store(planes_s + (16 * uint32_t(rb) + (tid >> 4)) * (3 * pitch) + i * 8, sums_first[part][rb], (i - piece * octets) * 8);
        }
    };
    store_first(0);
    if (groups > 32) store_first(1);
    auto from_lds = [](const uint16_t* at) { return *reinterpret_cast<const uint4*>(at); };
    const uint16_t* sums_at = bias_s + (g4 < 3 ? 8 + (j * 3 + g4) * pitch : 0u);
    const uint32_t sums_rb = g4 < 3 ? 48 * pitch : 0u;
    auto add_biases = [&](uint32_t g) {          // of the groups g .. g + 3
        s16x4 bias[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) bias[q] = *reinterpret_cast<const s16x4*>(biases_s + col[q] * pitch + g);
#pragma unroll
        for (uint32_t rb = 0; rb < NB; ++rb) {
            const s16x4 sums = *reinterpret_cast<const s16x4*>(sums_at + (rb * sums_rb + (g4 < 3 ? g : 0u)));
#pragma unroll
            for (int q = 0; q < 2; ++q) total[rb][q] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(sums, bias[q], total[rb][q], 0, 0, 0);
        }
    };
    // Their share of the magnitudes, 32 groups per instruction: the first piece is the chain sum cut off to bf16, made up for
    // by the factor (the magnitudes only scale a margin).
    auto add_bias_sizes = [&] {
        for (uint32_t g = 0; g < groups; g += 32) {
            const uint32_t at = min(g + 8 * g4, pitch - 8), M = g + 8 * g4 < groups ? 0x7fff7fffu : 0u;
            auto size = [&](const uint16_t* from) { const uint4 v = from_lds(from + at); return __builtin_bit_cast(bf16x8, make_uint4(v.x & M, v.y & M, v.z & M, v.w & M)); };
            const bf16x8 bias[2] = {size(biases_s + col[0] * pitch), size(biases_s + col[1] * pitch)};
#pragma unroll
            for (uint32_t rb = 0; rb < NB; ++rb) {
                const bf16x8 sums = size(planes_s + (rb * 16 + j) * 3 * pitch);
#pragma unroll
                for (int q = 0; q < 2; ++q) mag[rb][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sums, bias[q], mag[rb][q], 0, 0, 0);
            }
        }
#pragma unroll
        for (int rb = 0; rb < NB; ++rb)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) mag[rb][q][r] *= 1.0078125f;
    };
    // elements of a group that lane (j, g4) multiplies, from this one on: sixteen of them.  Q4: a load brings the four
    // lanes of a row the four quarters of two groups; a swap between the half waves gives every lane its share of either
    const uint32_t koff = BITS == 4 ? (g4 & 1u) * 32u + (g4 >> 1) * 16u : g4 * 16u;
    const uint16_t* a_lane = a_s + j * kPitch + koff;
    auto work = [&](uint32_t pair, const u32x4 (&slot)[2][kRegs / 4], u32x4 (&last)[2][kRegs / 4], const int odd) {   // odd: pair % 2, known at compile time
        const uint32_t buf = pair & 1u;
        // Loads return in the order they were sent, so a wait for token rows is a wait for all weights requested before them:
        // the rows are requested two pairs before they go to LDS, ahead of the pair's weight request.
        stash_a(buf ^ 1u, a_next);
        fetch_a(pair + 2, a_next);
        // (into the slot of the pair before, which nothing reads any more: loaded behind its own uses, the loop's last slot
        // got other registers, and the copies at the loop's end waited for every load in flight)
        fetch_b(pair + kAhead - 1, last);
        uint32_t codes[2][kRegs];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int w = 0; w < kRegs; ++w) codes[q][w] = slot[q][w / 4][w % 4];
        if constexpr (BITS == 4) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    const auto both = __builtin_amdgcn_permlane32_swap(codes[q][w], codes[q][w + 2], false, false);
                    codes[q][w] = both[0]; codes[q][w + 2] = both[1];
                }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            bf16x8 b[2][2];   // [tile][half of the lane's sixteen codes]
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
                    if constexpr (BITS == 4) b[q][kk] = nibble_operand(codes[q][2 * h + kk]);
                    else b[q][kk] = byte_operand(codes[q][4 * h + 2 * kk], codes[q][4 * h + 2 * kk + 1]);
                }
            float scale[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) scale[q] = __uint_as_float(h ? scales[q][odd] & 0xffff0000u : scales[q][odd] << 16);
            bf16x8 a[NB][2];
#pragma unroll
            for (int rb = 0; rb < NB; ++rb)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk)
                    a[rb][kk] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(a_lane + (buf * kTileRowsMax + 16 * uint32_t(rb)) * kPitch + 64 * h + 8 * kk));
#pragma unroll
            for (int rb = 0; rb < NB; ++rb) {
                f32x4 dot[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) dot[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rb][0], b[q][0], f32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 2; ++q) dot[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rb][1], b[q][1], dot[q], 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        total[rb][q][r] = __builtin_fmaf(scale[q], dot[q][r], total[rb][q][r]);
                        mag[rb][q][r] = __builtin_fmaf(fabsf(scale[q]), fabsf(dot[q][r]), mag[rb][q][r]);
                    }
            }
        }
        lds_barrier();
    };
    stash_a(0, a_first);
    lds_barrier();
    auto next_scales = [&](uint32_t g) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < 2; ++i) scales[q][i] = scales_next[q][i];
        fetch_s(g);
    };
    // (An odd pair stands behind the loop: a way round the second half would leave the first half's loads pending at the
    // loop's head, which then waited for all of them.)
    uint32_t pair = 0;
    for (; pair + 1 < pairs; pair += 2) {
        next_scales(2 * pair + 4);
        work(pair, ring[0], ring[1], 0);
        add_biases(2 * pair);
        work(pair + 1, ring[1], ring[0], 1);
    }
    if (pair < pairs) {
        next_scales(2 * pair);
        add_biases(2 * pair);
        work(pair, ring[0], ring[1], 0);
    }
    uint32_t out_row[NB];                        // (asked for here, the answer is back when the outputs are)
#pragma unroll
    for (int rb = 0; rb < NB; ++rb) {
        const uint32_t pos = first + min(16 * uint32_t(rb) + (tid >> 4), rows - 1);
        out_row[rb] = pos;
        if constexpr (!GATED) { if (p.out_rows) out_row[rb] = ldg_u32(p.out_rows, pos); }
    }
    add_bias_sizes();
    // epilogue: row m of the tile is sorted position first + m
    const float margin = p.near_margin;
    // Outputs and marks (one bit per sum: [sorted position][gate, up][N / 32] words, or [sorted position][N / 32]) cross through LDS, so that they leave in
    // whole pieces of a row: two-byte stores straight from the accumulators' lanes took longer than the walk of a short row.
    constexpr uint32_t kCols = GATED ? 64u : 128u, kOutPitch = kPitch;
    uint16_t* out_s = a_s;                       // (every wave has passed the walk's last barrier)
#pragma unroll
    for (int rb = 0; rb < NB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t m = 16 * uint32_t(rb) + 4 * g4 + uint32_t(r);
#pragma unroll
            for (int q = 0; q < (GATED ? 1 : 2); ++q) {
                const uint32_t col = GATED ? wave * 16 : (2 * wave + uint32_t(q)) * 16;
                bool near;
                float value = __uint_as_float(prefill_round(total[rb][q][r], mag[rb][q][r], margin, near));
                const uint64_t marks = __ballot(near);
                if (j == 0) marks_s[m * 8 + col / 16] = uint16_t(marks >> (16 * g4));
                if constexpr (GATED) {   // where one of the two is marked the other waits in the output's place
                    bool up_near;
                    const float up = __uint_as_float(prefill_round(total[rb][1][r], mag[rb][1][r], margin, up_near));
                    const uint64_t up_marks = __ballot(up_near);
                    if (j == 0) marks_s[m * 8 + 4 + col / 16] = uint16_t(up_marks >> (16 * g4));
                    value = near ? up : up_near ? value : swiglu_rounded(value, up);
                }
                out_s[m * kOutPitch + col + j] = uint16_t(__float_as_uint(value) >> 16);
            }
        }
    lds_barrier();
#pragma unroll
    for (uint32_t i = 0; i < 16u * NB * (kCols / 8) / 256u + (16u * NB * (kCols / 8) % 256u ? 1u : 0u); ++i) {
        const uint32_t piece = i * 256 + tid, m = piece / (kCols / 8), c = piece % (kCols / 8);
        if (m >= rows) continue;
        const uint32_t pos = first + m;
        const uint4 v = *reinterpret_cast<const uint4*>(out_s + m * kOutPitch + c * 8);
        if constexpr (GATED) {
            *reinterpret_cast<uint4*>(p.out_b + uint64_t(pos) * N + n0 + c * 8) =   // in the operand's order
                make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
                           __builtin_amdgcn_perm(v.y, v.x, 0x07060302u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u));
            if (c < 2) *reinterpret_cast<uint2*>(p.near_bits + (uint64_t(pos) * 2 * N + c * N + n0) / 32) = *reinterpret_cast<const uint2*>(marks_s + m * 8 + c * 4);
        } else {
            const uint64_t at = uint64_t(out_row[i]) * N + n0 + c * 8;   // (a piece's row is the thread's row of block i)
            if (p.out_h) *reinterpret_cast<uint4*>(p.out_h + at) = v;
            else {
                *reinterpret_cast<float4*>(p.out_f + at) = make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
                *reinterpret_cast<float4*>(p.out_f + at + 4) = make_float4(__uint_as_float(v.z << 16), __uint_as_float(v.z & 0xffff0000u), __uint_as_float(v.w << 16), __uint_as_float(v.w & 0xffff0000u));
            }
            if (c == 0) *reinterpret_cast<uint4*>(p.near_bits + (uint64_t(pos) * N + n0) / 32) = *reinterpret_cast<const uint4*>(marks_s + m * 8);
        }
    }
}
template <bool GATED, int BITS>
__global__ __launch_bounds__(256, BITS == 4 ? 3 : 2) void prefill_gemm_kernel(PrefillGemm p) {
    __shared__ __align__(16) uint16_t a_s[2 * kTileRowsMax * kPitch], marks_s[kTileRowsMax * 8];
    extern __shared__ __align__(16) uint16_t bias_s[];   // eight zeros, chain sums [48][3][pitch], biases [128][pitch]
    // The workgroups of one tile (neighbours in column block) share its token rows: they go to one of the eight dies, whose
    // L2 then fetches the rows once.
    const uint32_t columns = GATED ? p.N / 64u : p.N / 128u, turn = blockIdx.x / 8u;
    const uint32_t tile = turn / columns * 8u + blockIdx.x % 8u, n0 = turn % columns * (GATED ? 64u : 128u);
    // (requested together: the lists have room for the grid's last tiles)
    const uint32_t count = uint32_t(*p.tile_count), expert = uint32_t(p.tile_expert[tile]), first = uint32_t(p.tile_first[tile]), rows = uint32_t(p.tile_rows[tile]);
    if (tile >= count) return;
    if (rows <= 16) prefill_tile<GATED, BITS, 1>(p, a_s, marks_s, bias_s, expert, first, rows, n0);
    else if (rows <= 32) prefill_tile<GATED, BITS, 2>(p, a_s, marks_s, bias_s, expert, first, rows, n0);
    else prefill_tile<GATED, BITS, 3>(p, a_s, marks_s, bias_s, expert, first, rows, n0);
}

// The down product of rows of 512.  prefill_tile walks four pairs of groups there, and a workgroup is mostly its requests
// before the walk and its epilogue behind it (60 of 145 us at 2048 tokens).  Here a workgroup stages its tile's rows once, whole, and takes several
// blocks of 128 weight rows in turn: a wave multiplies its 32 weight rows of a block without waiting for any other, and asks for the next
// block's codes, scales and biases as it uses up this one's, so that loads are in flight during the epilogue too.  Sums, marks and outputs are
// prefill_tile's, added in the same order.  2048 weight rows, routed product alone: 2048 tokens 141 -> 123 us, 300 tokens with byte codes 130 ->
// 108; a layer 551 -> 534 and 332 -> 320.  (Rows of 640, whose LDS and registers leave as many waves: a layer of 300 tokens of hidden 2560 408 -> 402 us, but
// 600 503 -> 509 and 1000 612 -> 621.  Longer rows, where a tile has three blocks of them, leave one workgroup a compute unit.  Rows of 128 to 384 have not been
// tried.)
constexpr uint32_t kShortK = 512, kShortPitch = kShortK + 8, kShortOutPitch = 40;   // pitches in bf16 elements: sixteen rows on different banks
constexpr uint32_t kShortLds = 2 * (8 + kTileRowsMax * (kShortPitch + 3 * prefill_pitch(kShortK)) + 4 * 16 * kShortOutPitch);
template <int BITS, int NB>
__device__ __forceinline__ void prefill_short_tile(const PrefillGemm& p, uint16_t* lds, uint32_t expert, uint32_t first, uint32_t rows, uint32_t block0, uint32_t block1) {
    constexpr uint32_t K = kShortK, groups = K / 64, pitch = prefill_pitch(K), kPitchX = kShortPitch;
    constexpr int PAIRS = K / 128, kRegs = BITS, kQuads = groups / 4;   // kRegs: dwords of a column tile's pair per lane; kQuads: loads of four groups' scales
    static_assert(groups == 8 && pitch == groups);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, j = lane & 15u, g4 = lane >> 4, N = p.N;
    const uint8_t* record = p.records + uint64_t(expert) * p.stride;
    const uint8_t *codes_of = record + p.off[0], *scales_of = record + p.off[1], *biases_of = record + p.off[2];
    uint16_t *zeros_s = lds, *planes_s = lds + 8, *x_s = planes_s + kTileRowsMax * 3 * pitch, *out_s = x_s + kTileRowsMax * kPitchX + wave * (16 * kShortOutPitch);
    // (Bases are the same in every lane, lanes add 32-bit offsets; past the last block: it again, not used.)
    auto lane_row = [&](int q) { return (2 * wave + uint32_t(q)) * 16 + j; };
    u32x4 ring[PAIRS][2][kRegs / 4];
    auto fetch_b = [&](uint32_t block, int pair, uint32_t none) {
        const uint8_t* from = codes_of + uint64_t(min(block, block1 - 1)) * (128 * (K * BITS / 8));
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int h = 0; h < kRegs / 4; ++h) ring[pair][q][h] = *as_global<u32x4>(from + (lane_row(q) * (K * BITS / 8) + g4 * 16 + none + uint32_t(pair) * (16 * BITS) + 64u * uint32_t(h)));
    };
    uint2 scales_next[2][kQuads], biases_next[2][kQuads];
    auto fetch_s = [&](uint32_t block, uint32_t none) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < kQuads; ++i) {
                const uint64_t from = uint64_t(min(block, block1 - 1)) * (128 * groups * 2);
                const uint32_t at = (lane_row(q) * groups + 4u * uint32_t(i)) * 2 + none;
                scales_next[q][i] = ldg_u2_by_words(scales_of + from + at); biases_next[q][i] = ldg_u2_by_words(biases_of + from + at);
            }
    };
    // the tile's rows and their chain sums; rows past the end repeat the last one (never stored)
    uint4 row[NB][PAIRS], sums[NB];
#pragma unroll
    for (int rb = 0; rb < NB; ++rb) {
        const uint32_t pos = first + min(16 * uint32_t(rb) + (tid >> 4), rows - 1);
        sums[rb] = ldg_u4(p.planes + uint64_t(pos) * (3 * pitch) + min(tid & 15u, 3 * pitch / 8 - 1) * 8);
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) row[rb][i] = ldg_u4(p.a + uint64_t(pos) * K + ((tid & 15u) + 16 * uint32_t(i)) * 8);
    }
    fetch_s(block0, 0);
#pragma unroll
    for (int u = 0; u < PAIRS; ++u) fetch_b(block0, u, 0);
    uint32_t out_row[NB];
#pragma unroll
    for (int rb = 0; rb < NB; ++rb) {
        const uint32_t pos = first + min(16 * uint32_t(rb) + lane / 4, rows - 1);
        out_row[rb] = p.out_rows ? ldg_u32(p.out_rows, pos) : pos;
    }
    if (tid < 4) reinterpret_cast<uint32_t*>(zeros_s)[tid] = 0;
#pragma unroll
    for (int rb = 0; rb < NB; ++rb) {
        const uint32_t r = 16 * uint32_t(rb) + (tid >> 4), c = tid & 15u;
        if (c < 3 * pitch / 8)
            *reinterpret_cast<uint4*>(planes_s + r * (3 * pitch) + c * 8) = sums[rb];
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) *reinterpret_cast<uint4*>(x_s + r * kPitchX + (c + 16 * uint32_t(i)) * 8) = row[rb][i];
    }
    lds_barrier();
    const uint32_t koff = BITS == 4 ? (g4 & 1u) * 32u + (g4 >> 1) * 16u : g4 * 16u;   // (as in prefill_tile)
    const uint16_t* x_lane = x_s + j * kPitchX + koff;
    const uint16_t* sums_at = g4 < 3 ? planes_s + (j * 3 + g4) * pitch : zeros_s;
    const uint32_t sums_rb = g4 < 3 ? 48 * pitch : 0u, sums_g = g4 < 3 ? 1u : 0u;
    for (uint32_t block = block0; block < block1; ++block) {
        uint32_t none = 0;                       // (a zero that the compiler does not know: it would form every address and read the rows once, in front of the loop, into registers that are not there)
        asm volatile("" : "+v"(none));
        uint2 scales[2][kQuads], biases[2][kQuads];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < kQuads; ++i) { scales[q][i] = scales_next[q][i]; biases[q][i] = biases_next[q][i]; }
        fetch_s(block + 1, none);
        f32x4 total[NB][2], mag[NB][2];
#pragma unroll
        for (int rb = 0; rb < NB; ++rb)
#pragma unroll
            for (int q = 0; q < 2; ++q) total[rb][q] = mag[rb][q] = f32x4{0, 0, 0, 0};
        auto add_biases = [&](int i) {           // of the groups 4 i .. 4 i + 3
#pragma unroll
            for (uint32_t rb = 0; rb < NB; ++rb) {
                const s16x4 piece = *reinterpret_cast<const s16x4*>(sums_at + (rb * sums_rb + sums_g * 4 * uint32_t(i) + none));
#pragma unroll
                for (int q = 0; q < 2; ++q) total[rb][q] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(piece, __builtin_bit_cast(s16x4, biases[q][i]), total[rb][q], 0, 0, 0);
            }
        };
#pragma unroll
        for (int pair = 0; pair < PAIRS; ++pair) {
            uint32_t codes[2][kRegs];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int w = 0; w < kRegs; ++w) codes[q][w] = ring[pair][q][w / 4][w % 4];
            if constexpr (BITS == 4) {
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        const auto both = __builtin_amdgcn_permlane32_swap(codes[q][w], codes[q][w + 2], false, false);
                        codes[q][w] = both[0]; codes[q][w + 2] = both[1];
                    }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                bf16x8 b[2][2];
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) {
                        if constexpr (BITS == 4) b[q][kk] = nibble_operand(codes[q][2 * h + kk]);
                        else b[q][kk] = byte_operand(codes[q][4 * h + 2 * kk], codes[q][4 * h + 2 * kk + 1]);
                    }
                float scale[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const uint32_t two = pair % 2 ? scales[q][pair / 2].y : scales[q][pair / 2].x;
                    scale[q] = __uint_as_float(h ? two & 0xffff0000u : two << 16);
                }
#pragma unroll
                for (int rb = 0; rb < NB; ++rb) {
                    bf16x8 a[2];
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) a[kk] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(x_lane + (none + 16 * uint32_t(rb) * kPitchX + 128 * uint32_t(pair) + 64 * uint32_t(h) + 8 * uint32_t(kk))));
                    f32x4 dot[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q) dot[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[q][0], f32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 2; ++q) dot[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[q][1], dot[q], 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            total[rb][q][r] = __builtin_fmaf(scale[q], dot[q][r], total[rb][q][r]);
                            mag[rb][q][r] = __builtin_fmaf(fabsf(scale[q]), fabsf(dot[q][r]), mag[rb][q][r]);
                        }
                }
            }
            fetch_b(block + 1, pair, none);
            if (pair % 2 == 0) add_biases(pair / 2);
            // (the pair is done here: the compiler would put its last multiply-adds off to where the sums are used, and keep all dots until then)
#pragma unroll
            for (int rb = 0; rb < NB; ++rb)
#pragma unroll
                for (int q = 0; q < 2; ++q) asm volatile("" : "+v"(total[rb][q]), "+v"(mag[rb][q]));
            __builtin_amdgcn_sched_barrier(0);
        }
        // the biases' share of the magnitudes: the operand's first quarter holds the eight groups, the others zeros
        const uint32_t M = g4 == 0 ? 0x7fff7fffu : 0u;
        bf16x8 size[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) size[q] = __builtin_bit_cast(bf16x8, make_uint4(biases[q][0].x & M, biases[q][0].y & M, biases[q][1].x & M, biases[q][1].y & M));
        const uint32_t n0 = block * 128 + wave * 32;
#pragma unroll
        for (uint32_t rb = 0; rb < NB; ++rb) {
            const uint4 v = *reinterpret_cast<const uint4*>(planes_s + ((rb * 16 + j) * 3 * pitch + none));
            const bf16x8 sums_of = __builtin_bit_cast(bf16x8, make_uint4(v.x & M, v.y & M, v.z & M, v.w & M));
#pragma unroll
            for (int q = 0; q < 2; ++q) mag[rb][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sums_of, size[q], mag[rb][q], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t m = 4 * g4 + uint32_t(r), pos = first + 16 * rb + m + none;
                uint64_t marks[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    bool near;
                    const uint32_t value = prefill_round(total[rb][q][r], mag[rb][q][r] * 1.0078125f, p.near_margin, near);
                    marks[q] = __ballot(near);
                    out_s[m * kShortOutPitch + uint32_t(q) * 16 + j] = uint16_t(value >> 16);
                }
                if (j == 0 && 16 * rb + m < rows) p.near_bits[(uint64_t(pos) * N + n0) / 32] = (uint32_t(marks[0] >> (16 * g4)) & 0xffffu) | uint32_t(marks[1] >> (16 * g4)) << 16;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const uint4 o = *reinterpret_cast<const uint4*>(out_s + lane / 4 * kShortOutPitch + lane % 4 * 8);
            if (16 * rb + lane / 4 < rows) {
                const uint64_t at = uint64_t(out_row[rb] + none) * N + n0 + lane % 4 * 8;
                if (p.out_h) *reinterpret_cast<uint4*>(p.out_h + at) = o;
                else {
                    *reinterpret_cast<float4*>(p.out_f + at) = make_float4(__uint_as_float(o.x << 16), __uint_as_float(o.x & 0xffff0000u), __uint_as_float(o.y << 16), __uint_as_float(o.y & 0xffff0000u));
                    *reinterpret_cast<float4*>(p.out_f + at + 4) = make_float4(__uint_as_float(o.z << 16), __uint_as_float(o.z & 0xffff0000u), __uint_as_float(o.w << 16), __uint_as_float(o.w & 0xffff0000u));
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
}
template <int BITS>
__global__ __launch_bounds__(256, 2) void prefill_short_kernel(PrefillGemm p, uint32_t share) {   // share: blocks of a workgroup
    extern __shared__ __align__(16) uint16_t short_lds[];
    const uint32_t blocks = p.N / 128u, shares = (blocks + share - 1) / share, turn = blockIdx.x / 8u;   // (a tile's workgroups on one die, as in prefill_gemm_kernel)
    const uint32_t tile = turn / shares * 8u + blockIdx.x % 8u, block0 = turn % shares * share, block1 = min(block0 + share, blocks);
    const uint32_t count = uint32_t(*p.tile_count), expert = uint32_t(p.tile_expert[tile]), first = uint32_t(p.tile_first[tile]), rows = uint32_t(p.tile_rows[tile]);
    if (tile >= count) return;
    if (rows <= 16) prefill_short_tile<BITS, 1>(p, short_lds, expert, first, rows, block0, block1);
    else if (rows <= 32) prefill_short_tile<BITS, 2>(p, short_lds, expert, first, rows, block0, block1);
    else if constexpr (BITS == 4) prefill_short_tile<BITS, 3>(p, short_lds, expert, first, rows, block0, block1);
    else {   // (three blocks of rows beside twice the codes do not fit the registers)
        prefill_short_tile<BITS, 2>(p, short_lds, expert, first, 32, block0, block1);
        lds_barrier();
        prefill_short_tile<BITS, 1>(p, short_lds, expert, first + 32, rows - 32, block0, block1);
    }
}

// Exact recomputation of the marked elements: one group of 32 lanes plays the reference's 32 lanes for one element
// (qwen.metal:46-62: lane width 16 when K % 512 == 0 and N % 8 == 0, else 8; xor-butterfly lane sum).
// BITS 8: the affine Q8 lanes (qwen.metal:112-125: lane width 8 when K % 512 == 0 and N % 8 == 0, else 4; the input sum is the
// plain fp32 sum, the dot a multiply-add chain element by element).
// A workgroup has the elements of a few positions: it fetches those rows of inputs and forms their blocks' input sums in LDS once, beside
// the look at the marks; its eight groups of lanes then take the marked elements in turn.  Of a gate/up element only the marked sum is formed
// again (both are marked in one element of some hundreds): the product kernel left the other one in the output's place.
// AHEAD: blocks of a lane that are fetched together: one memory latency, not several; no more than a lane has (a row of 512 has one).
// What bounds it is the vector unit, about 70 instructions a block of sixteen, with the latencies of a workgroup's few turns.  Gate/up and
// down, us, with every element's rows fetched by its own lanes, both sums of a gate/up element and four blocks at a time whatever the row -> here: 2048 tokens
// of hidden 2048 92 + 38 -> 72 + 36, 1500 of hidden 3072 247 + 67 -> 168 + 55, 300 of the mixed artifact 26 + 12 -> 20 + 12.
constexpr uint32_t kPatchRows = 16, kPatchLds = 24 * 1024;
template <int WIDTH, bool GATED, int BITS, int AHEAD>
__global__ __launch_bounds__(256) void prefill_patch_kernel(PrefillGemm p, uint32_t rows_per) {
    extern __shared__ __align__(16) uint4 patch_x[];   // [rows][K / 8] inputs, [rows][K / WIDTH] input sums, then the marked elements: n | row << 12 (| sums << 16)
    __shared__ uint32_t found_count;
    __shared__ uint32_t expert_s[kPatchRows];
    static_assert(WIDTH * BITS >= 32);
    const uint32_t tid = threadIdx.x, lane = tid & 31u, K = p.K, N = p.N, groups = K / 64, pieces = K / 8, blocks = K / WIDTH, row_words = N / 32u;
    float* sums = reinterpret_cast<float*>(patch_x + rows_per * pieces);
    using Found = std::conditional_t<GATED, uint32_t, uint16_t>;
    Found* found = reinterpret_cast<Found*>(sums + rows_per * blocks);
    // Only the map words of covered positions were written by the product kernel: a word past them holds whatever the
    // buffer held before.  N is a multiple of 32, so a word never straddles two positions.
    const uint32_t positions = p.near_words / ((GATED ? 2 : 1) * row_words);
    const uint32_t covered = p.covered ? min(uint32_t(max(*p.covered, 0)), positions) : positions;
    const uint32_t first = blockIdx.x * rows_per;
    if (first >= covered) return;
    const uint32_t rows = min(rows_per, covered - first);
    const uint32_t mark_row = tid / row_words, mark_word = tid - mark_row * row_words;
    uint32_t marks[2] = {0, 0};
    if (mark_row < rows)
#pragma unroll
        for (int proj = 0; proj < (GATED ? 2 : 1); ++proj) marks[proj] = p.near_bits[((first + mark_row) * (GATED ? 2 : 1) + proj) * row_words + mark_word];
    if (tid == 0) found_count = 0;
    if (tid < rows) expert_s[tid] = p.ids ? uint32_t(p.ids[p.slots[first + tid]]) : 0u;
    // (a block of sixteen is two pieces: they stand turned by their block, so that sixteen lanes' reads meet all banks)
    auto place = [](uint32_t piece) { return WIDTH == 16 ? piece ^ (piece >> 4 & 1u) : piece; };
    for (uint32_t i0 = tid; i0 < rows * pieces; i0 += 1024) {
        uint4 v[4];
        uint32_t at[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t i = min(i0 + 256 * u, rows * pieces - 1), r = i / pieces, c = i - r * pieces;
            const uint32_t a_row = p.a_rows ? uint32_t(p.a_rows[first + r]) : first + r;
            const uint4 q = reinterpret_cast<const uint4*>(p.a + uint64_t(a_row) * K)[c];   // 0 2 | 4 6 | 1 3 | 5 7
            v[u] = make_uint4(__builtin_amdgcn_perm(q.z, q.x, 0x05040100u), __builtin_amdgcn_perm(q.z, q.x, 0x07060302u),
                              __builtin_amdgcn_perm(q.w, q.y, 0x05040100u), __builtin_amdgcn_perm(q.w, q.y, 0x07060302u));
            at[u] = r * pieces + place(c);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t i = i0 + 256 * u, w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
            const bool inside = i < rows * pieces;
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) x[k] = __uint_as_float((k & 1) ? w[k / 2] & 0xffff0000u : w[k / 2] << 16);
            if (inside) patch_x[at[u]] = v[u];
            if constexpr (BITS == 4) {
                const float low = bf(bf(bf(x[0] + x[1]) + x[2]) + x[3]), high = bf(bf(bf(x[4] + x[5]) + x[6]) + x[7]);
                const float half = (0.0f + low) + high;
                if constexpr (WIDTH == 8) { if (inside) sums[i] = half; }
                else {   // (a row has an even number of pieces: a block's two are neighbouring lanes')
                    const float before = __shfl_xor(half, 1);
                    if (inside && (i & 1u)) sums[i / 2] = (before + low) + high;
                }
            } else if constexpr (WIDTH == 8) {
                float sum = 0;
#pragma unroll
                for (int k = 0; k < 8; ++k) sum += x[k];
                if (inside) sums[i] = sum;
            } else {
                float low = 0, high = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) { low += x[k]; high += x[4 + k]; }
                if (inside) { sums[2 * i] = low; sums[2 * i + 1] = high; }
            }
        }
    }
    __syncthreads();
    if (uint32_t either = marks[0] | marks[1]) {
        const uint32_t base = mark_row << 12 | mark_word * 32u;
        uint32_t at = atomicAdd(&found_count, uint32_t(__popc(either)));
        for (; either; either &= either - 1) {
            const uint32_t bit = uint32_t(__ffs(either) - 1);
            if constexpr (GATED) found[at++] = (base + bit) | (marks[0] >> bit & 1u) << 16 | (marks[1] >> bit & 1u) << 17;
            else found[at++] = Found(base + bit);
        }
    }
    __syncthreads();
    const uint32_t listed = found_count;
    for (uint32_t item = tid >> 5; item < listed; item += 8) {
        const uint32_t element = found[item], row = element >> 12 & 15u, n = element & 4095u, pos = first + row, expert = expert_s[row];
        if (p.ids && expert >= p.experts) continue;   // an id the router could not give (reported through the status word)
        const uint8_t* record = p.records + uint64_t(expert) * p.stride;
        constexpr int DW = WIDTH * BITS / 32;
        auto lanes_sum = [&](const uint64_t* off) {
        float result = 0;
        for (uint32_t b0 = lane; b0 < blocks; b0 += 32 * AHEAD) {
            uint32_t words[AHEAD][DW];
            uint16_t scale_bits[AHEAD], bias_bits[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const uint32_t b = min(b0 + 32u * u, blocks - 1);   // past the end: the last block again, not used
                const uint32_t g = n * groups + (b * WIDTH) / 64;
                const uint32_t* src = reinterpret_cast<const uint32_t*>(record + off[0] + uint64_t(n) * (K * BITS / 8)) + b * DW;
#pragma unroll
                for (int i = 0; i < DW; ++i) words[u][i] = src[i];
                scale_bits[u] = reinterpret_cast<const uint16_t*>(record + off[1])[g];
                bias_bits[u] = reinterpret_cast<const uint16_t*>(record + off[2])[g];
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const uint32_t b = b0 + 32u * u;
                if (b >= blocks) break;
                uint32_t xw[WIDTH / 2];   // the block's inputs, two a word
                if constexpr (WIDTH >= 8) {
#pragma unroll
                    for (int i = 0; i < WIDTH / 8; ++i) {
                        const uint4 v = patch_x[row * pieces + place(b * (WIDTH / 8) + uint32_t(i))];
                        xw[4 * i] = v.x; xw[4 * i + 1] = v.y; xw[4 * i + 2] = v.z; xw[4 * i + 3] = v.w;
                    }
                } else {
                    const uint2 v = reinterpret_cast<const uint2*>(patch_x)[row * (2 * pieces) + b];
                    xw[0] = v.x; xw[1] = v.y;
                }
                float x[WIDTH];
#pragma unroll
                for (int i = 0; i < WIDTH; ++i) x[i] = __uint_as_float((i & 1) ? xw[i / 2] & 0xffff0000u : xw[i / 2] << 16);
                float dot = 0;
                if constexpr (BITS == 8) {
                    // (a BF16 value times a byte code is exact in fp32: the fused multiply-add rounds as the reference's multiply and add)
#pragma unroll
                    for (int i = 0; i < WIDTH; ++i) dot = __builtin_fmaf(x[i], float((words[u][i / 4] >> (8 * (i % 4))) & 0xffu), dot);
                } else
#pragma unroll
                for (int i = 0; i < WIDTH; i += 8) {
                    // nibble j of a word is element j: the even ones and the odd ones as bytes, which are 8-bit floats of code * 2^-9: two
                    // converted by one instruction
                    const uint32_t even = words[u][i / 8] & 0x0f0f0f0fu, odd = (words[u][i / 8] >> 4) & 0x0f0f0f0fu;
                    const f32x2 c02 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, false), c46 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, true);
                    const f32x2 c13 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, false), c57 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, true);
                    // (a BF16 value times a 4-bit code is exact in fp32, so a fused multiply-add rounds as the reference's
                    // multiply and add do: ((p0 + p1) + p2) + p3, then onto the block's sum)
                    dot += __builtin_fmaf(x[i + 3], c13.y, __builtin_fmaf(x[i + 2], c02.y, __builtin_fmaf(x[i + 1], c13.x, x[i] * c02.x)));
                    dot += __builtin_fmaf(x[i + 7], c57.y, __builtin_fmaf(x[i + 6], c46.y, __builtin_fmaf(x[i + 5], c57.x, x[i + 4] * c46.x)));
                }
                result += b16(scale_bits[u]) * dot + sums[row * blocks + b] * b16(bias_bits[u]);
            }
        }
        return lane_sum32(result);
        };
        if constexpr (GATED) {
            uint16_t* out = p.out_b + uint64_t(pos) * N + ((n & ~7u) | (n & 1u) << 2 | (n & 7u) >> 1);   // in the operand's order
            const bool up_first = !(element >> 16 & 1u);
            float other = b16(*out);
            const float marked = lanes_sum(p.off + (up_first ? 3 : 0));
            if (element >> 16 == 3u) other = lanes_sum(p.off + 3);
            if (lane == 0) *out = uint16_t(__float_as_uint(up_first ? swiglu_bf(other, marked) : swiglu_bf(marked, other)) >> 16);
        } else {
            const float value = bf(lanes_sum(p.off));
            if (lane == 0) {
                const uint64_t at = uint64_t(p.out_rows ? uint32_t(p.out_rows[pos]) : pos) * N + n;
                if (p.out_h) p.out_h[at] = uint16_t(__float_as_uint(value) >> 16); else p.out_f[at] = value;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------
// Router logits of a long batch without the exact chains for every (token, expert): a bf16 matrix-core product gives
// every logit to within a bound that holds whatever the order of its additions, the top-k can only come from the
// logits within that bound of the k-th largest, and only those are recomputed with the reference's chains
// (qwen.metal:512-534: sixteen contiguous K partitions, a k-ascending multiply-accumulate chain in each, partials added
// 0..15).  The other logits are written as -inf, so the exact selection kernel that follows picks what it would pick from
// all the exact logits: ids and softmax weights are the reference's bits.
//
// The bound.  Inputs and router weights are BF16-valued, so every product is exact in fp32.  Two fp32 sums of the same n
// exact products, each formed with at most n additions that round or truncate to fp32, differ by at most
// n * 2^-22 * sum |x_k w_k| (n * 2^-23 for a truncating accumulator plus n * 2^-24 for the reference's rounded chain
// leaves a factor 1.3), and sum |x_k w_k| <= |x| |w| (Cauchy-Schwarz).  Adding the expert's offset rounds both once more:
// 2^-22 |logit| on top.  With lower bounds a - m and upper bounds a + m of the exact logits: the k-th largest exact logit
// is at least the k-th largest lower bound, which is at least the k-th largest of the 64 lanes' largest lower bounds; an
// expert whose upper bound is below that cannot be among the top k, ties included.  A token with a logit that is not
// finite has every expert recomputed.
// ---------------------------------------------------------------------------------------------------------------------
constexpr uint32_t kRouterPitch = 72;   // in bf16 elements (144 bytes)
// approx[t][e] = sum_k a[t][k] b[e][k] (+ offsets[e]): 64 tokens x 64 experts per workgroup, a wave a 32 x 32 block on
// v_mfma_f32_32x32x16_bf16, K in steps of 64 through LDS (rows padded to 144 bytes), the next step's rows in registers.
__global__ __launch_bounds__(256) void router_product_kernel(const uint16_t* a, const uint16_t* b, uint32_t T, uint32_t E, uint32_t K,
                                                             const float* offsets, float* approx) {
    __shared__ __align__(16) uint16_t a_s[2][64 * kRouterPitch], b_s[2][64 * kRouterPitch];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, m = lane & 31u, h = lane >> 5;
    // Every die gets one stretch of the (token block, expert block) list: neighbours on it share their token rows in the die's L2.
    const uint32_t columns = (E + 63) / 64, blocks = (T + 63) / 64 * columns, share = (blocks + 7) / 8, block = blockIdx.x % 8 * share + blockIdx.x / 8;
    if (blockIdx.x / 8 >= share || block >= blocks) return;
    const uint32_t t0 = block / columns * 64, e0 = block % columns * 64;
    const uint32_t r = tid >> 3, c8 = tid & 7u;   // a thread moves rows r and r + 32, sixteen bytes each, of both operands
    const uint16_t* a_src0 = a + uint64_t(min(t0 + r, T - 1)) * K + c8 * 8;
    const uint16_t* a_src1 = a + uint64_t(min(t0 + r + 32, T - 1)) * K + c8 * 8;
    const uint16_t* b_src0 = b + uint64_t(min(e0 + r, E - 1)) * K + c8 * 8;
    const uint16_t* b_src1 = b + uint64_t(min(e0 + r + 32, E - 1)) * K + c8 * 8;
    uint4 ra0, ra1, rb0, rb1;
    auto fetch = [&](uint32_t g) {
        ra0 = *reinterpret_cast<const uint4*>(a_src0 + g * 64); ra1 = *reinterpret_cast<const uint4*>(a_src1 + g * 64);
        rb0 = *reinterpret_cast<const uint4*>(b_src0 + g * 64); rb1 = *reinterpret_cast<const uint4*>(b_src1 + g * 64);
    };
    auto stash = [&](uint32_t buf) {
        *reinterpret_cast<uint4*>(&a_s[buf][r * kRouterPitch + c8 * 8]) = ra0; *reinterpret_cast<uint4*>(&a_s[buf][(r + 32) * kRouterPitch + c8 * 8]) = ra1;
        *reinterpret_cast<uint4*>(&b_s[buf][r * kRouterPitch + c8 * 8]) = rb0; *reinterpret_cast<uint4*>(&b_s[buf][(r + 32) * kRouterPitch + c8 * 8]) = rb1;
    };
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    const uint32_t steps = K / 64, row_a = (wave >> 1) * 32 + m, row_b = (wave & 1u) * 32 + m;
    fetch(0); stash(0);
    __syncthreads();
    for (uint32_t g = 0; g < steps; ++g) {
        const uint32_t buf = g & 1u;
        if (g + 1 < steps) fetch(g + 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bf16x8 av = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&a_s[buf][row_a * kRouterPitch + q * 16 + h * 8]));
            const bf16x8 bv = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&b_s[buf][row_b * kRouterPitch + q * 16 + h * 8]));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc, 0, 0, 0);
        }
        if (g + 1 < steps) stash(buf ^ 1u);
        __syncthreads();
    }
    const uint32_t e = e0 + (wave & 1u) * 32 + m;
    const float offset = (offsets && e < E) ? offsets[e] : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t t = t0 + (wave >> 1) * 32 + 8 * uint32_t(i / 4) + 4 * h + uint32_t(i % 4);
        if (t < T && e < E) approx[uint64_t(t) * E + e] = offsets ? acc[i] + offset : acc[i];
    }
}
// One wavefront per token: bounds, the experts that can be among the top k, their exact logits; everything else -inf.
// (A whole workgroup per token, each wavefront taking a quarter of the list, measured slower: 35 against 29 us.)
// ids / weights not null (topk <= 64): the wavefront also selects its token's top k and forms the softmax weights from the
// row it holds in LDS (route_token, the selection of the decode kernels: the same ids and weights as route_kernel's), and
// the row itself is not written out.
constexpr int kRefinePerLane = 16;   // experts <= 1024
struct RefineLds { uint32_t x, w, row, list, bytes; };   // bytes from the start, of one wavefront's share
__host__ __device__ inline RefineLds refine_lds(uint32_t K, uint32_t E) {
    RefineLds l{};
    l.w = 2 * (K + 128); l.row = l.w + 8192; l.list = l.row + (E + 3) / 4 * 16; l.bytes = l.list + (E + 7) / 8 * 16;
    return l;
}
__global__ __launch_bounds__(256) void router_refine_kernel(const uint16_t* xb, const uint16_t* w, const float* offsets, const float* norms,
                                                            uint32_t T, uint32_t E, uint32_t K, uint32_t topk, float* logits,
                                                            int32_t* ids, float* weights) {
    __shared__ uint32_t pick_s[4][128];                      // route_token's scratch
    __shared__ int32_t ids_s[4][64]; __shared__ float weights_s[4][64];
    extern __shared__ __align__(16) uint8_t refine_s[];
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x & 63u, t = blockIdx.x * 4 + wave, P = K / 16;
    if (t >= T) return;
    const RefineLds at_s = refine_lds(K, E);
    uint8_t* mine_s = refine_s + wave * at_s.bytes;
    uint16_t* x_row = reinterpret_cast<uint16_t*>(mine_s);   // the token's input row (BF16-valued, so the bf16 copy is the input), eight elements behind every partition
    uint4* w_s = reinterpret_cast<uint4*>(mine_s + at_s.w);  // 64 elements of every partition of four experts
    float* row_s = reinterpret_cast<float*>(mine_s + at_s.row);
    uint16_t* list_s = reinterpret_cast<uint16_t*>(mine_s + at_s.list);
    float squares = 0;
    for (uint32_t i = lane * 8; i < K; i += 512) {
        const uint4 v = ldg_u4(xb + uint64_t(t) * K + i);
        *reinterpret_cast<uint4*>(x_row + i + i / P * 8) = v;
        squares = squares_of(v, squares);
    }
    const float ninf = __uint_as_float(0xff800000u);
    float* row = logits + uint64_t(t) * E;
    const float reach = float(K) * 0x1p-22f * row_norm(squares);
    float upper[kRefinePerLane], best_lower = ninf;
    bool strange = false;
#pragma unroll
    for (int i = 0; i < kRefinePerLane; ++i) {
        const uint32_t e = lane + 64u * uint32_t(i);
        upper[i] = ninf;
        if (e < E) {
            const float a = row[e], bound = reach * norms[e] + 0x1p-22f * fabsf(a);
            strange = strange || !(fabsf(a) < __uint_as_float(0x7f800000u)) || !(bound < __uint_as_float(0x7f800000u));
            upper[i] = a + bound;
            best_lower = fmaxf(best_lower, a - bound);
        }
    }
    // the k-th largest of the lanes' largest lower bounds (fewer than k lanes with an expert: nothing can be ruled out)
    float threshold = ninf;
    bool all = __ballot(strange) != 0;
    {
        float mine = best_lower;
        for (uint32_t j = 0; j < topk && !all; ++j) {
            const float top = wave_max_f32(mine);
            if (!(top > ninf)) { all = true; break; }
            threshold = top;
            const uint64_t holders = __ballot(mine == top);
            if (lane == uint32_t(__ffsll((long long)holders) - 1)) mine = ninf;
        }
    }
    // the list of experts to recompute, in any order
    uint32_t count = 0;
#pragma unroll
    for (int i = 0; i < kRefinePerLane; ++i) {
        const uint32_t e = lane + 64u * uint32_t(i);
        const bool take = e < E && (all || upper[i] >= threshold);
        const uint64_t takers = __ballot(take);
        if (take) list_s[count + uint32_t(__popcll(takers & ((1ull << lane) - 1)))] = uint16_t(e);
        count += uint32_t(__popcll(takers));
        if (e < E) row_s[e] = ninf;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // four experts at a time: sixteen lanes run an expert's sixteen partition chains (router_kernel's arithmetic), 64 elements of every
    // partition after the other.  Eight lanes fetch the 128 bytes of one partition, so that a load looks eight lines up and not 64, and the pieces
    // change lanes in LDS, turned by their partition so that sixteen lanes' reads meet all banks.  The next 64 elements -- of these experts
    // or of the next four -- are requested before the current ones are used.
    const uint32_t split = lane % 16, base = lane & ~15u;
    const uint16_t* xr = x_row + split * (P + 8);
    const uint32_t batches = (P + 63) / 64, total = (count + 3) / 4 * batches;
    uint4 ahead[8];
    auto request = [&](uint32_t index) {
        const uint32_t i = min(index % batches * 64 + lane % 8 * 8, P - 8);   // (past a partition's end: its last piece again, not used)
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) {
            const uint32_t e = uint32_t(__builtin_amdgcn_readfirstlane(int(list_s[min(index / batches * 4 + q / 2, count - 1)])));
            ahead[q] = ldg_u4(w + uint64_t(e) * K + (q % 2 * 8 + lane / 8) * P + i);
        }
    };
    if (total) request(0);
    float c = 0;
    for (uint32_t index = 0; index < total; ++index) {
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) w_s[(q * 8 + lane / 8) * 8 + (lane + (q * 8 + lane / 8) % 16 / 2) % 8] = ahead[q];
        if (index + 1 < total) request(index + 1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint32_t i0 = index % batches * 64;
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) {
            if (i0 + 8 * q >= P) break;
            const uint4 xv4 = *reinterpret_cast<const uint4*>(xr + i0 + 8 * q), wv4 = w_s[lane * 8 + (q + split / 2) % 8];
            const uint32_t ww[4] = {wv4.x, wv4.y, wv4.z, wv4.w}, xw[4] = {xv4.x, xv4.y, xv4.z, xv4.w};
#pragma unroll
            for (int k = 0; k < 8; ++k)
                c = __builtin_fmaf(__uint_as_float((k & 1) ? (xw[k / 2] & 0xffff0000u) : (xw[k / 2] << 16)),
                                   __uint_as_float((k & 1) ? (ww[k / 2] & 0xffff0000u) : (ww[k / 2] << 16)), c);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (index % batches + 1 == batches) {   // the expert's chains are complete: partials added 0..15, then the offset
            const uint32_t at = index / batches * 4 + lane / 16;
            float sum = 0;
            for (uint32_t sidx = 0; sidx < 16; ++sidx) sum += __shfl(c, base + sidx);
            if (split == 0 && at < count) { const uint32_t e = list_s[at]; row_s[e] = offsets ? sum + offsets[e] : sum; }
            c = 0;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (!ids) { for (uint32_t e = lane; e < E; e += 64) row[e] = row_s[e]; return; }
    auto fetch = [&](auto& cand, uint32_t per) {
        constexpr int PER = int(sizeof(cand) / sizeof(float));
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint32_t e = lane * per + uint32_t(i);
            cand[i] = (uint32_t(i) < per && e < E) ? row_s[e] : ninf;
        }
    };
    if (E == 512) route_token<8>(fetch, E, topk, lane, ids_s[wave], weights_s[wave], pick_s[wave], []() {}, []() {});
    else route_token<16>(fetch, E, topk, lane, ids_s[wave], weights_s[wave], pick_s[wave], []() {}, []() {});
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < topk) { ids[uint64_t(t) * topk + lane] = ids_s[wave][lane]; weights[uint64_t(t) * topk + lane] = weights_s[wave][lane]; }
}
// Router logits for the selection that follows: exact where it can matter, -inf elsewhere.  xb: the inputs as bf16 rows;
// norms: those of the router's rows (launch_prefill_rows).  K % 128 == 0, experts <= 1024.
void launch_prefill_router(hipStream_t s, const uint16_t* xb, const void* w, const float* offsets, uint32_t T, uint32_t K,
                           uint32_t E, uint32_t topk, const float* norms, float* logits, int32_t* ids, float* weights) {
    const uint16_t* wb = static_cast<const uint16_t*>(w);
    const uint32_t blocks = ((E + 63) / 64) * ((T + 63) / 64), lds = 4 * refine_lds(K, E).bytes;
    hipLaunchKernelGGL(router_product_kernel, dim3((blocks + 7) / 8 * 8), dim3(256), 0, s, xb, wb, T, E, K, offsets, logits);
    // (the most that any shape asks for: the same whoever calls)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(router_refine_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(4 * refine_lds(4096, 1024).bytes));
    hipLaunchKernelGGL(router_refine_kernel, dim3((T + 3) / 4), dim3(256), lds, s, xb, wb, offsets, norms, T, E, K, topk, logits, ids, weights);
}

void launch_prefill_rows(hipStream_t s, const float* x, uint32_t rows, uint32_t K, uint16_t* xb, uint16_t* xp, uint16_t* planes, uint16_t* plain, int32_t* status,
                         const void* norm_of, uint32_t norm_rows, float* norms) {
    hipLaunchKernelGGL((prefill_rows_kernel<true>), dim3((rows * (K / 4) + 255) / 256 + (norm_rows + 3) / 4), dim3(256), 0, s, x, rows, K, xb, xp, planes, plain, status,
                       static_cast<const uint16_t*>(norm_of), norm_rows, norms);
}
void launch_prefill_acts(hipStream_t s, const uint16_t* xp, uint32_t rows, uint32_t K, uint16_t* planes, uint16_t* plain) {
    hipLaunchKernelGGL((prefill_rows_kernel<false>), dim3((rows * (K / 4) + 255) / 256), dim3(256), 0, s, xp, rows, K, nullptr, nullptr, planes, plain, nullptr, nullptr, 0u, nullptr);
}
void launch_prefill_tiles(hipStream_t s, const int32_t* offsets, uint32_t experts, uint32_t rows, int32_t* tile_expert, int32_t* tile_first,
                          int32_t* tile_rows, int32_t* tile_count) {
    hipLaunchKernelGGL(prefill_tiles_kernel, dim3(1), dim3(1024), 0, s, offsets, experts, rows, tile_expert, tile_first, tile_rows, tile_count);
}
void launch_prefill_dispatch(hipStream_t s, const int32_t* ids, uint32_t tokens, uint32_t topk, uint32_t E, int32_t* offsets, int32_t* slots, int32_t* rows,
                             int32_t* status, int32_t* tile_expert, int32_t* tile_first, int32_t* tile_rows, int32_t* tile_count) {
    const uint32_t n = tokens * topk, stretch = ((n + kDispatchParts - 1) / kDispatchParts + 1023) / 1024 * 1024;
    const size_t lds = size_t(((kDispatchParts + 2) * E + 2 + 3) / 4 * 4 + stretch) * 4;
    if (lds > 48 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(prefill_dispatch_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    hipLaunchKernelGGL(prefill_dispatch_kernel, dim3((E + kDispatchThreads / 64 - 1) / (kDispatchThreads / 64), kDispatchParts), dim3(kDispatchThreads), lds, s, ids, n, topk, E, stretch, offsets, slots, rows, status,
                       tile_expert, tile_first, tile_rows, tile_count);
}
// whether launch_prefill_dispatch takes this batch (else: launch_dispatch and launch_prefill_tiles)
bool prefill_dispatch_fits(const int32_t* ids, uint32_t tokens, uint32_t topk, uint32_t E) {
    const uint64_t n = uint64_t(tokens) * topk;
    return reinterpret_cast<uintptr_t>(ids) % 16 == 0 && n > 1024 && n < (1u << 24) && E <= 1024 && n / kDispatchParts + 1024 <= 24 * 1024;
}
void launch_prefill_gemm(hipStream_t s, const PrefillGemm& p, bool gated, uint32_t max_tiles) {
    if (!gated && p.K == kShortK) {
        // (a shared expert's few tiles, and a short batch's, need more workgroups than four blocks each leave)
        const uint32_t tiles = (max_tiles + 7) / 8 * 8, blocks = p.N / 128, share = prefill_short_share(tiles, blocks);
        const dim3 grid(tiles * ((blocks + share - 1) / share));
        auto go = [&](auto kernel) {
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(kShortLds));
            hipLaunchKernelGGL(kernel, grid, dim3(256), kShortLds, s, p, share);
        };
        if (p.bits == 8) go(prefill_short_kernel<8>); else go(prefill_short_kernel<4>);
        return;
    }
    const dim3 grid((max_tiles + 7) / 8 * 8 * (gated ? p.N / 64 : p.N / 128));
    const uint32_t lds = (8 + (kTileRowsMax * 3 + 128) * prefill_pitch(p.K)) * 2;
    if (p.bits == 8) {
        if (gated) hipLaunchKernelGGL((prefill_gemm_kernel<true, 8>), grid, dim3(256), lds, s, p);
        else hipLaunchKernelGGL((prefill_gemm_kernel<false, 8>), grid, dim3(256), lds, s, p);
    } else {
        if (gated) hipLaunchKernelGGL((prefill_gemm_kernel<true, 4>), grid, dim3(256), lds, s, p);
        else hipLaunchKernelGGL((prefill_gemm_kernel<false, 4>), grid, dim3(256), lds, s, p);
    }
}
void launch_prefill_patch(hipStream_t s, const PrefillGemm& p, bool gated) {
    const bool wide = p.K % 512 == 0 && p.N % 8 == 0;     // the reference's lane-width rule (metal.mm:649-674); the Q8 lanes are half as wide
    const uint32_t width = (wide ? 16 : 8) / (p.bits / 4), row_bytes = 2 * p.K + 4 * (p.K / width);
    const uint32_t rows = std::max(1u, std::min({(gated ? 2048u : 8192u) / p.N, kPatchRows, kPatchLds / row_bytes}));
    const uint32_t lds = rows * (row_bytes + (gated ? 4 : 2) * p.N), positions = p.near_words / (p.N / 32 * (gated ? 2 : 1));
    const dim3 grid((positions + rows - 1) / rows);
    // (a lane's blocks in as few turns as four at a time allow, no more of them a turn than that takes)
    const uint32_t each = (p.K / width + 31) / 32, turns = (each + 3) / 4, ahead = (each + turns - 1) / turns;
#define ZC_PATCH(W, G, B, A) hipLaunchKernelGGL((prefill_patch_kernel<W, G, B, A>), grid, dim3(256), lds, s, p, rows)
#define ZC_PATCH4(W, G) do { if (ahead == 1) ZC_PATCH(W, G, 4, 1); else if (ahead == 2) ZC_PATCH(W, G, 4, 2); else if (ahead == 3) ZC_PATCH(W, G, 4, 3); else ZC_PATCH(W, G, 4, 4); } while (0)
#define ZC_PATCH8(W, G) do { if (ahead <= 2) ZC_PATCH(W, G, 8, 2); else ZC_PATCH(W, G, 8, 4); } while (0)
    if (p.bits == 8) {
        if (gated) { if (wide) ZC_PATCH8(8, true); else ZC_PATCH8(4, true); }
        else { if (wide) ZC_PATCH8(8, false); else ZC_PATCH8(4, false); }
    } else if (gated) { if (wide) ZC_PATCH4(16, true); else ZC_PATCH4(8, true); }
    else { if (wide) ZC_PATCH4(16, false); else ZC_PATCH4(8, false); }
#undef ZC_PATCH8
#undef ZC_PATCH4
#undef ZC_PATCH
}
// (hidden and intermediate sizes up to 4096: the margins of the recomputation are measured up to there)
bool prefill_shape(uint32_t hidden, uint32_t inter, uint32_t experts) {
    return hidden % 128 == 0 && inter % 128 == 0 && hidden <= 4096 && inter <= 4096 && experts <= 1024;
}

}  // namespace zc
