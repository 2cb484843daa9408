// The reference's lanes of the affine products, literally: the device code that the operator kernels and the layer's expert kernels share.
#pragma once
#include <type_traits>
#include "zc_device.hpp"
#include "zc_decode_common.hpp"   // lds_barrier

namespace zc {

// ---------------------------------------------------------------------------
// Affine Q4 / Q8 rows (reference: qwen.metal:46-81, 112-144)
//
// A half wave plays the 32 reference lanes of one output row: lane l takes the row's blocks l, l + 32, ... of WIDTH elements
// (Q4 16|8, Q8 8|4: one or two dwords of codes) in order.  It walks two rows at a time (gate and up, or two rows of the one
// matrix), so that an input block read from LDS serves two rows, and up to two tokens, so that a code is unpacked once for
// four products.  The walk over (row tile, block step) is one flat loop: the codes and scales of its next three steps are in
// flight, across row tiles too, and the first three are requested before the input rows are staged.
//
// The products x * q of a BF16-valued row (zeros and magnitudes from 2^-100 to 2^100) are exact in fp32, so a fused multiply-add
// rounds as the reference's multiply and add do, also when all of it is scaled by a power of two: such rows multiply codes
// that were never converted (affine_halves).  Rows that hold anything else, infinities and NaN among them, keep converted codes
// and separate operations.
//
// What bounds it: with one token per row, the latency of the chain job -> row index -> input row -> LDS -> codes (a launch
// of a few us); with several, vector instructions, a wave's at four clocks each: 24 per block of sixteen weights and token, 14
// to unpack the block (the listing's 49 and 28 for the two rows), and the finish of a row.  Per layer of hidden 2560 and intermediate 640, gate/up and down: 40 tokens 144
// and 116 us, one token 11.9 and 8.7 us.  With codes converted to floats, addresses formed per lane and four tokens per
// workgroup it was 172 and 132, 12.5 and 9.2 us.  (One token's gate/up that makes its picks takes 13.2 us, down 7.0; 40 tokens now go to the
// matrix cores, 105 and 105 us: zc_affine_matrix.hpp.)  Four tokens per workgroup take 159 and 112 us: most experts have one or two
// tokens, and the LDS of four leaves room for three workgroups on a compute unit where two leave six (decoding stacks of
// hidden 2048 and 3072 at 2 to 64 tokens lost 5 to 25 %).  One token at a time, codes requested step by step behind the staging,
// sums through LDS permutes and the shared expert in launches of its own took 397 and 310, 20.2 and 14.3 us.
// ---------------------------------------------------------------------------
constexpr uint32_t kAffineTokens = 2;                                            // tokens a workgroup multiplies at once, at most
struct AffineMatrix { const uint8_t* w; const uint16_t *s, *b; };

// Input rows in LDS: a block's WIDTH elements and its bias sum behind them, WIDTH / 4 words further apart than the elements
// need (20, 10 or 5 words: the blocks of neighbouring lanes meet different banks), so that a lane adds one offset per token.
template <int WIDTH> __host__ __device__ constexpr uint32_t affine_token_bytes(uint32_t K) { return (K * 5 + 15) / 16 * 16; }
template <int WIDTH> struct AffineBlock { static constexpr uint32_t kBytes = WIDTH * 5, kPiece = WIDTH == 16 ? 4 : WIDTH == 8 ? 2 : 1; };
template <int WIDTH>
__device__ __forceinline__ void affine_inputs(const uint8_t* at, float* x, float& sum) {
    typedef float piece __attribute__((ext_vector_type(AffineBlock<WIDTH>::kPiece)));
    constexpr int P = AffineBlock<WIDTH>::kPiece;
#pragma unroll
    for (int i = 0; i < WIDTH; i += P) {
        const piece v = *reinterpret_cast<const piece*>(at + 4 * i);
#pragma unroll
        for (int k = 0; k < P; ++k) x[i + k] = v[k];
    }
    sum = *reinterpret_cast<const float*>(at + 4 * WIDTH);
}

// Addresses: the bases are the same in every lane and move with tile and step, the lanes' 32-bit offsets are those of their row
// and block in the tile.  wide: rows are whole steps (K % 512 == 0), else the last step's idle lanes repeat the last block.
// Streams: the matrix rows a half wave walks at once, gate and up of one row or two rows of the one matrix.  (Four streams, which
// halve the reads of LDS, took 130 registers: three waves per SIMD.  S-sized layers took 5 % longer, hidden 3072 the same.)
template <int BITS, int WIDTH, bool GATED, uint32_t TOKENS>
struct AffineStream {
    static constexpr int kStreams = 2, kRows = GATED ? kStreams / 2 : kStreams;   // kRows: output rows of a half wave per tile
    static constexpr uint32_t kAhead = TOKENS == 1 ? 3 : 2;   // steps in flight (three for two tokens: 93 registers, four waves per SIMD instead of five, 5 % longer)
    static constexpr int DW = WIDTH * BITS / 32;
    static constexpr bool kWide = WIDTH * BITS == 64;
    struct Slot { uint32_t q[kStreams][DW]; uint32_t s[kStreams], b[kStreams]; };
    static constexpr uint32_t kTileRows = 8 * kRows;   // of a workgroup: eight half waves
    uint32_t K, N, blocks, groups, shift, steps, lane, half, tile, end, step;   // tile, step: the next one to request
    AffineMatrix m[2];
    uint32_t w_at[kRows], g_at[kRows];
    __device__ __forceinline__ uint32_t row(uint32_t t, uint32_t i) const { return t * kTileRows + i * 8 + half; }
    __device__ __forceinline__ void aim() {
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const uint32_t r = min(row(tile, uint32_t(i)), N - 1) - tile * kTileRows;
            w_at[i] = r * (K / 8 * BITS) + (kWide ? lane * (DW * 4) : 0u);
            g_at[i] = (r * groups + (kWide ? (lane * WIDTH) >> shift : 0u)) * 2;
        }
    }
    __device__ __forceinline__ void fetch(Slot& slot) {   // past the end: the last tile again, not used
        const uint64_t first = uint64_t(tile) * kTileRows;
        const uint32_t at = kWide ? 0u : min(lane, blocks - 1 - step * 32), g = ((step * 32 * WIDTH) >> shift) * 2;
#pragma unroll
        for (int q = 0; q < kStreams; ++q) {
            const AffineMatrix& a = m[GATED ? q % 2 : 0];
            const int i = GATED ? q / 2 : q;
            const uint8_t* w = a.w + (first * (K / 8 * BITS) + step * (32 * DW * 4));
            const uint32_t w_lane = w_at[i] + (kWide ? 0u : at * (DW * 4)), g_lane = g_at[i] + (kWide ? 0u : ((at * WIDTH) >> shift) * 2);
            if constexpr (DW == 2) { const uint2 v = ldg_u2_by_words(w + w_lane); slot.q[q][0] = v.x; slot.q[q][DW - 1] = v.y; }
            else slot.q[q][0] = ldg_u32(w + w_lane);
            slot.s[q] = ldg_u16(reinterpret_cast<const uint8_t*>(a.s) + (first * groups * 2 + g) + g_lane);
            slot.b[q] = ldg_u16(reinterpret_cast<const uint8_t*>(a.b) + (first * groups * 2 + g) + g_lane);
        }
        if (++step == steps) { step = 0; if (tile + 1 < end) { ++tile; aim(); } }
    }
};
// Codes as f16 bit patterns, two in a word: the pattern of an integer n < 1024 is the number n * 2^-24, which the mixed
// multiply-add (v_fma_mix_f32) takes as it is, so a code costs its place in a half word and no conversion.  Word k of eight
// nibbles: nibbles k and k + 4; word k of four bytes: bytes k and k + 2.
template <int BITS, int WIDTH>
__device__ __forceinline__ void affine_halves(const uint32_t* words, uint32_t* half) {
    constexpr int PER = 32 / BITS / 2;   // half-word pairs of a word of codes
#pragma unroll
    for (int i = 0; i < WIDTH / 2; ++i) half[i] = (words[i / PER] >> (BITS * (i % PER))) & (BITS == 4 ? 0x000f000fu : 0x00ff00ffu);
}
// x * code i * 2^-24 + c, rounded once.  (In assembly: from the source form the compiler converts the codes once for all tokens
// instead, one instruction per code and twice the registers.)
template <int BITS>
__device__ __forceinline__ float affine_mad(float x, const uint32_t* half, int i, float c) {
    constexpr int PER = 32 / BITS / 2;
    const uint32_t h = half[i / (2 * PER) * PER + i % PER];
    float d;
    if ((i / PER) % 2) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(d) : "v"(x), "v"(h), "v"(c));
    else asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,1,0]" : "=v"(d) : "v"(x), "v"(h), "v"(c));
    return d;
}
template <int BITS>
__device__ __forceinline__ float affine_mul(float x, const uint32_t* half, int i) {
    constexpr int PER = 32 / BITS / 2;
    const uint32_t h = half[i / (2 * PER) * PER + i % PER];
    float d;
    if ((i / PER) % 2) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(d) : "v"(x), "v"(h));
    else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(d) : "v"(x), "v"(h));
    return d;
}
// sum of x * code over a block in the reference's order.  (A first quad or product is added to nothing: the reference adds it to
// +0, which can only turn a -0 into +0, and the row's sum starts from +0.)
template <int BITS, int WIDTH>
__device__ __forceinline__ float affine_dot_exact(const uint32_t* half, const float* x) {
    float dot = 0;
    if constexpr (BITS == 4) {
#pragma unroll
        for (int i = 0; i < WIDTH; i += 4) {
            float quad = affine_mul<BITS>(x[i], half, i);
#pragma unroll
            for (int k = 1; k < 4; ++k) quad = affine_mad<BITS>(x[i + k], half, i + k, quad);
            dot = i == 0 ? quad : dot + quad;
        }
    } else {
        dot = affine_mul<BITS>(x[0], half, 0);
#pragma unroll
        for (int i = 1; i < WIDTH; ++i) dot = affine_mad<BITS>(x[i], half, i, dot);
    }
    return dot * 0x1p24f;
}
template <int BITS, int WIDTH>
__device__ __forceinline__ float affine_dot_any(const uint32_t* codes, const float* x) {
    uint32_t words[WIDTH * BITS / 32];   // (a copy the compiler cannot see through: it would keep the conversions of both rows for all tokens)
#pragma unroll
    for (int i = 0; i < WIDTH * BITS / 32; ++i) asm("" : "=v"(words[i]) : "0"(codes[i]));
    auto code = [&](int i) { return float((words[i * BITS / 32] >> (i * BITS % 32)) & (BITS == 4 ? 15u : 255u)); };
    float dot = 0;
    if constexpr (BITS == 4) {
#pragma unroll
        for (int i = 0; i < WIDTH; i += 4) dot += x[i] * code(i) + x[i + 1] * code(i + 1) + x[i + 2] * code(i + 2) + x[i + 3] * code(i + 3);
    } else {
#pragma unroll
        for (int i = 0; i < WIDTH; ++i) dot += x[i] * code(i);
    }
    return dot;
}
// The bias half's input sum of one block.
template <int BITS, int WIDTH>
__device__ __forceinline__ float affine_sum(const float* x) {
    float sum = 0;
    if constexpr (BITS == 4) {
#pragma unroll
        for (int i = 0; i < WIDTH; i += 4) sum += bf(bf(bf(x[i] + x[i + 1]) + x[i + 2]) + x[i + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < WIDTH; ++i) sum += x[i];
    }
    return sum;
}

// The walk for nt staged tokens; out_at: where the output row of token (lane % TOKENS) begins; put(out_at, row, y) stores.
// (nt and exact are the same in every lane.  As template parameters they made eight walks, whose common first steps the
// compiler moved in front of the choice between them: 200 registers.)
template <int BITS, int WIDTH, bool GATED, uint32_t TOKENS, class Put>
__device__ __forceinline__ void affine_walk(AffineStream<BITS, WIDTH, GATED, TOKENS>& st,
                                            typename AffineStream<BITS, WIDTH, GATED, TOKENS>::Slot (&ring)[AffineStream<BITS, WIDTH, GATED, TOKENS>::kAhead],
                                            const uint8_t* lds, uint64_t out_at, uint32_t tile, bool float_output, uint32_t nt, bool exact, Put put) {
    using Stream = AffineStream<BITS, WIDTH, GATED, TOKENS>;
    constexpr int S = Stream::kStreams;
    const uint32_t blocks = st.blocks, token = affine_token_bytes<WIDTH>(st.K), lane = st.lane;
    const uint32_t total = (st.end - tile) * st.steps;
    float r[TOKENS][S];
#pragma unroll
    for (uint32_t t = 0; t < TOKENS; ++t)
#pragma unroll
        for (int q = 0; q < S; ++q) r[t][q] = 0;
    uint32_t step = 0;
    for (uint32_t i0 = 0; i0 < total; i0 += Stream::kAhead) {
#pragma unroll
        for (uint32_t d = 0; d < Stream::kAhead; ++d) {
            if (i0 + d >= total) break;
            float scale[S], bias[S];
            uint32_t words[S][Stream::DW];
#pragma unroll
            for (int q = 0; q < S; ++q) {
#pragma unroll
                for (uint32_t i = 0; i < Stream::DW; ++i) words[q][i] = ring[d].q[q][i];
                scale[q] = b16(uint16_t(ring[d].s[q])); bias[q] = b16(uint16_t(ring[d].b[q]));
            }
            st.fetch(ring[d]);
            const uint32_t b = step * 32 + lane;
            const uint8_t* block = lds + (Stream::kWide ? b : min(b, blocks - 1)) * AffineBlock<WIDTH>::kBytes;
            auto tokens = [&](auto dot_of) {
#pragma unroll
                for (uint32_t t = 0; t < TOKENS; ++t) {
                    if (t >= nt) break;
                    asm volatile("");   // (else the compiler moves every token's products in front of the question)
                    float x[WIDTH], sum;
                    affine_inputs<WIDTH>(block + t * token, x, sum);
#pragma unroll
                    for (int q = 0; q < S; ++q) {
                        const float more = r[t][q] + (scale[q] * dot_of(q, x) + sum * bias[q]);
                        r[t][q] = Stream::kWide || b < blocks ? more : r[t][q];
                    }
                }
            };
            if (exact) {
                uint32_t half[S][WIDTH / 2];
#pragma unroll
                for (int q = 0; q < S; ++q) affine_halves<BITS, WIDTH>(words[q], half[q]);
                tokens([&](int q, const float* x) { return affine_dot_exact<BITS, WIDTH>(half[q], x); });
            } else tokens([&](int q, const float* x) { return affine_dot_any<BITS, WIDTH>(words[q], x); });
            if (++step < st.steps) continue;
            step = 0;
            // every lane has all the sums: lane i * TOKENS + t finishes output row i of token t
            float v[2] = {0, 0};
#pragma unroll
            for (uint32_t t = 0; t < TOKENS; ++t) {
                if (t >= nt) break;
#pragma unroll
                for (int i = 0; i < Stream::kRows; ++i) {
                    const float first = lane_sum32(r[t][GATED ? 2 * i : i]), second = GATED ? lane_sum32(r[t][GATED ? 2 * i + 1 : i]) : 0.0f;
                    if (lane == uint32_t(i) * TOKENS + t) { v[0] = first; v[1] = second; }
                }
            }
            const uint32_t row = st.row(tile, lane / TOKENS);
            const float y = GATED ? swiglu_bf(v[0], v[1]) : float_output ? v[0] : bf(v[0]);
            if (lane < Stream::kRows * TOKENS && lane % TOKENS < nt && row < st.N) put(out_at, row, y);
#pragma unroll
            for (uint32_t t = 0; t < TOKENS; ++t)
#pragma unroll
                for (int q = 0; q < S; ++q) r[t][q] = 0;
            ++tile;
        }
    }
}

// Rows tile0 .. end - 1 (tiles) of the matrices for nt <= TOKENS tokens, by 256 threads: input row in_row(t), output row out_row(t).
// load(row, i): the four elements from 4 i on of an input row; put(at, row, y): stores y as element `row` of the output row that begins at `at`.
// choice, optional: what the matrices depend on is found while the input rows are staged.  choice.find() runs in front of the staging
// and choice.take(matrices) behind the workgroup's barrier; false: there is nothing to do.
struct AffineKnown {};
template <int BITS, int WIDTH, bool GATED, uint32_t TOKENS, class Load, class Put, class InRow, class OutRow, class Choice = AffineKnown>
__device__ __forceinline__ void affine_rows_by(const AffineMatrix (&m)[2], uint32_t K, uint32_t N, uint32_t group, Load load, Put put, uint32_t nt,
                                               InRow in_row, OutRow out_row, uint32_t tile0, uint32_t end, bool float_output, uint8_t* lds, uint32_t tid, Choice choice = {}) {
    constexpr bool kKnown = std::is_same_v<Choice, AffineKnown>;
    using Stream = AffineStream<BITS, WIDTH, GATED, TOKENS>;
    Stream st;
    st.K = K; st.N = N; st.blocks = K / WIDTH; st.shift = group == 64 ? 6 : 5; st.groups = K >> st.shift; st.steps = (st.blocks + 31) / 32;
    st.lane = tid & 31u; st.half = tid >> 5; st.tile = tile0; st.end = end; st.step = 0;
    st.m[0] = m[0]; st.m[1] = m[1];
    const uint32_t from = st.lane < nt ? in_row(st.lane) : 0u;   // lane t: token t's input row
    const uint64_t out_at = uint64_t(out_row(min(st.lane % TOKENS, nt - 1))) * N;
    typename Stream::Slot ring[Stream::kAhead];
    auto begin = [&] {
        st.aim();
#pragma unroll
        for (uint32_t d = 0; d < Stream::kAhead; ++d) st.fetch(ring[d]);
    };
    if constexpr (kKnown) begin();
    else choice.find();
    constexpr uint32_t kPieces = WIDTH / 4, P = AffineBlock<WIDTH>::kPiece;
    const uint32_t blocks = st.blocks, token = affine_token_bytes<WIDTH>(K);
    bool strange = false;
#pragma unroll 1
    for (uint32_t t = 0; t < nt; ++t) {
        const uint32_t src = uint32_t(__builtin_amdgcn_readlane(int(from), int(t)));
#pragma unroll 2
        for (uint32_t i = tid; i < K / 4; i += 256) {
            const uint4 q = load(src, i);
            const uint32_t v[4] = {q.x, q.y, q.z, q.w};
            uint32_t* to = reinterpret_cast<uint32_t*>(lds + t * token + i / kPieces * AffineBlock<WIDTH>::kBytes + i % kPieces * 16);
#pragma unroll
            for (int k = 0; k < 4; ++k) {   // (as a magnitude from 2^-100 on: one comparison)
                const uint32_t a = v[k] & 0x7fffffffu;
                strange |= (v[k] & 0xffffu) != 0 || (a - 0x0d800000u >= 0x71800000u - 0x0d800000u && a != 0);
            }
            typedef uint32_t piece __attribute__((ext_vector_type(P)));
#pragma unroll
            for (uint32_t k = 0; k < 4; k += P) {
                if constexpr (P == 4) *reinterpret_cast<piece*>(to) = piece{v[0], v[1], v[2], v[3]};
                else if constexpr (P == 2) *reinterpret_cast<piece*>(to + k) = piece{v[k], v[k + 1]};
                else to[k] = v[k];
            }
        }
    }
    // Each wave's finding crosses in block w of the first token, wave w's: in the padding behind the bias sum, or, where blocks
    // have none, in the sum's own place, read before the sums are written.  (An array of its own beside the rows would keep out
    // the longest rows, of 32768 elements, which fill a compute unit's LDS to the last byte.)
    constexpr bool kPadded = WIDTH >= 8;
    auto finding = [&](uint32_t w) { return reinterpret_cast<uint32_t*>(lds + w * AffineBlock<WIDTH>::kBytes + 4 * WIDTH + (kPadded ? 4 : 0)); };
    const bool any = __ballot(strange) != 0;
    if ((tid & 63u) == 0) *finding(tid >> 6) = any;
    lds_barrier();
    if constexpr (!kKnown) {
        if (!choice.take(st.m)) return;
        begin();
    }
    uint32_t found = 0;
    if constexpr (!kPadded) {
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) found |= *finding(w);
        lds_barrier();
    }
#pragma unroll 1
    for (uint32_t t = 0; t < nt; ++t)
#pragma unroll 1
        for (uint32_t b = tid; b < blocks; b += 256) {
            float xb[WIDTH], unset;
            uint8_t* block = lds + t * token + b * AffineBlock<WIDTH>::kBytes;
            affine_inputs<WIDTH>(block, xb, unset);
            *reinterpret_cast<float*>(block + 4 * WIDTH) = affine_sum<BITS, WIDTH>(xb);
        }
    lds_barrier();
    if constexpr (kPadded) {
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) found |= *finding(w);
    }
    const bool exact = __builtin_amdgcn_readfirstlane(int(found)) == 0;
    affine_walk<BITS, WIDTH, GATED, TOKENS>(st, ring, lds, out_at, tile0, float_output, nt, exact, put);
}
// The same for fp32 rows of x and out.
template <int BITS, int WIDTH, bool GATED, uint32_t TOKENS, class InRow, class OutRow, class Choice = AffineKnown>
__device__ __forceinline__ void affine_rows(const AffineMatrix (&m)[2], uint32_t K, uint32_t N, uint32_t group, const float* x, float* out, uint32_t nt,
                                            InRow in_row, OutRow out_row, uint32_t tile0, uint32_t end, bool float_output, uint8_t* lds, Choice choice = {}) {
    affine_rows_by<BITS, WIDTH, GATED, TOKENS>(m, K, N, group, [=](uint32_t row, uint32_t i) { return ldg_u4(x + uint64_t(row) * K, i); },
                                               [=](uint64_t at, uint32_t row, float y) { out[at + row] = y; }, nt, in_row, out_row, tile0, end, float_output, lds, threadIdx.x, choice);
}
}  // namespace zc
