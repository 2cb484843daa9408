// Affine rows for several tokens on the matrix cores, bit for bit the reference's lanes (qwen.metal:46-81, 112-144).
//
// The reference evaluates a block of sixteen (or eight) weights as quads: dot = ((q0 + q1) + q2) + q3, a quad being the fp32
// chain of four products.  The products are exact, and where a quad's inputs lie within 2^20 units of the smallest of them (its
// lowest significand bit) the chain is exact too, in any order: one v_mfma_f32_4x4x4_16b_bf16 then gives that quad's sums for sixteen blocks, four
// tokens and four weight rows.  The other quads run the chain itself, on four v_mfma_f32_4x4x1_16b_f32, each of which is one
// fused multiply-add per result, rounded to nearest (compared with fmaf over the whole range, subnormal results included).
// Which way a quad goes depends on the inputs alone, so it is found once, when the rows' images are made: about 0.1 % of the
// quads of normally distributed inputs and 1 % of SwiGLU activations run their chain.
// Byte codes (Q8) have one chain of eight per block and leave four bits of room only: they always run the chain.
//
// Lane (b, j) = 4 b + j holds the blocks 2 b and 2 b + 1 of a step's 32 for weight row j of the wave's four, half a step being one of them:
// sixteen bytes of codes a load, converted once for all tokens.  The instruction hands it the sums of four tokens in four
// registers, so no lane idles whatever the number of tokens, and nothing crosses lanes before a row is finished: a lane holds two
// reference lanes' sums per token.
//
// What bounds it: the vector unit.  Per half step and four weight rows a wave has about 15 vector instructions for the codes, 24 to add and fold four
// tokens, 5 matrix instructions, and as many again of addresses, waits and branches (ns on a SIMD with two waves or more: two-operand
// vector instructions 1.0, all others 1.8, the bf16 instruction 3.9 mostly beside them, the fp32 one 3.9 on the same unit).  Memory
// instructions came first until they were cut from twelve to four a step: a lane's two blocks in one load of sixteen bytes instead of two of
// eight, scale and bias in one load (lanes of b and b + 1 share a group: one takes the scale, the other the bias); 32 tokens of
// hidden 2048, 512 experts: gate/up 96 -> 62 us, down 53 -> 47.  Workgroups that take a contiguous share of the work list instead of a grid over
// all jobs there could be: 64 tokens of hidden 3072 that agree on eleven experts 157 -> 125 us.
// Two tokens a workgroup on the lanes of zc_affine.hpp -> this, gate/up and down, us: hidden 2560, 40 tokens 144 and 116 -> 105 and 105; hidden 2048, 32 tokens
// 81 and 52 -> 67 and 47; hidden 3072, average of six layers, 64 tokens 291 and 162 -> 138 and 87.  Eight tokens a workgroup (half the conversions, twice the
// accumulators: two waves a SIMD) took 121 and 75 where four took 136 and 74 (64 tokens of hidden 3072 that agree), but 83 and 78 where four took 62 and
// 46 (32 tokens of hidden 2048, most of whose experts have one token or two).
#pragma once
#include "zc_affine.hpp"

namespace zc {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kMatrixTokens = 4, kMatrixSteps = 64;                  // of a workgroup, at most: tokens and steps of a row (a lane each; the LDS rule ends at 31)
constexpr uint32_t kMatrixWaves = 4, kMatrixThreads = 64 * kMatrixWaves;

template <int BITS, int WIDTH>
struct MatrixForm {
    static constexpr uint32_t kStep = 32 * WIDTH, kQuads = WIDTH / 4, DW = WIDTH * BITS / 32;   // elements of a step, quads of a block, code words of a block
    static constexpr bool kWhole = WIDTH * BITS == 64;      // rows are whole steps (else the last one may be half a step)
    static constexpr uint32_t kHalfBytes = 128 * WIDTH;     // of four tokens' rows, per half step
    __host__ __device__ static constexpr uint32_t steps(uint32_t K) { return (K + kStep - 1) / kStep; }
    // LDS: the four tokens' rows, their bias sums, a byte of quad bits per token and step, what each wave has found
    __host__ __device__ static constexpr uint32_t sums_at(uint32_t K) { return steps(K) * 2 * kHalfBytes; }
    __host__ __device__ static constexpr uint32_t bits_at(uint32_t K) { return steps(K) * 2 * (kHalfBytes + 256); }
    __host__ __device__ static constexpr uint32_t found_at(uint32_t K) { return bits_at(K) + kMatrixTokens * kMatrixSteps; }
};
template <int BITS, int WIDTH> __host__ __device__ constexpr uint32_t matrix_staged_bytes(uint32_t K) { return MatrixForm<BITS, WIDTH>::found_at(K) + 4 * kMatrixWaves; }
// Workgroups of a compute unit: by LDS, and four waves a SIMD by registers.
__host__ __device__ constexpr uint32_t matrix_per_cu(uint32_t lds) { return 160 * 1024 / lds < 4 ? 160 * 1024 / lds : 4; }
// The rows whose products may round take turns in the same memory as the lanes stage them: two tokens at a time where room for them (a ninth
// more) costs no workgroup of a compute unit, else one.
template <int BITS, int WIDTH>
__host__ __device__ constexpr uint32_t matrix_lds_bytes(uint32_t K) {
    const uint32_t staged = matrix_staged_bytes<BITS, WIDTH>(K), two = 2 * affine_token_bytes<WIDTH>(K);
    return two > staged && two <= 160 * 1024 && matrix_per_cu(two) == matrix_per_cu(staged) ? two : staged;
}

// Where token i's piece of block b stands among a half step's 64 sixteen-byte pieces: reads take blocks of all four tokens side by side, writes
// sixteen blocks of one token, and both meet all banks.
__device__ __forceinline__ uint32_t matrix_piece(uint32_t b, uint32_t i) { return i * 16 + (b ^ (i * 4)); }
// The thread's index, a new value to the compiler each time: what is formed from it is formed where it is used, and not kept in registers
// around the loop over jobs.
__device__ __forceinline__ uint32_t matrix_thread() {
    uint32_t tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    return tid;
}

// What a quad of inputs is to the matrix cores: its bf16 values, elements in the order 0 2 1 3, and an information word: the
// BF16-rounded chain sum of the bias half (upper half), bit 0: the products' chain has to be run, bit 1: a value is not BF16 or lies
// outside [2^-100, 2^100] (zeros apart), so that products may round.
struct MatrixQuad { uint2 pairs; uint32_t info; };
__device__ __forceinline__ MatrixQuad matrix_quad(const uint32_t (&v)[4]) {
    uint32_t unit = 250, strange = 0;
    float above = 0, below = 0, f[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t a = v[k] & 0x7fffffffu;
        strange |= (v[k] & 0xffffu) != 0 || (a - 0x0d800000u >= 0x71800000u - 0x0d800000u && a != 0) ? 2u : 0u;
        f[k] = __uint_as_float(v[k]);
        const uint32_t lowest = (a >> 23) + uint32_t(__builtin_ctz(a | 0x00800000u));   // the exponent of the significand's lowest set bit, plus 150
        unit = min(unit, a ? lowest : 250u);
        above += fmaxf(f[k], 0.0f); below += fmaxf(-f[k], 0.0f);
    }
    // every partial sum of the quad lies below 15 max(above, below); up to 2^24 units it is exact (16 for 15: above and below are themselves rounded)
    const uint32_t chain = fmaxf(above, below) > __uint_as_float((unit - 3) << 23) ? 1u : 0u;
    return {make_uint2(__builtin_amdgcn_perm(v[2], v[0], 0x07060302u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)),
            __float_as_uint(bf(bf(bf(f[0] + f[1]) + f[2]) + f[3])) | strange | chain};
}

// A row's image: its quads' pairs, then their information words, in the place of the K floats of the row (three quarters of them).
__device__ __forceinline__ void matrix_image_put(float* row, uint32_t K, uint32_t quad, const MatrixQuad& q) {
    *reinterpret_cast<uint2*>(row + 2 * quad) = q.pairs;
    reinterpret_cast<uint32_t*>(row)[K / 2 + quad] = q.info;
}
// The image of row `row` of x, by a whole workgroup.
__device__ __forceinline__ void matrix_image_row(const float* x, float* image, uint32_t row, uint32_t K) {
    for (uint32_t quad = threadIdx.x; quad < K / 4; quad += blockDim.x) {
        const uint4 q = ldg_u4(x + uint64_t(row) * K, quad);
        const uint32_t v[4] = {q.x, q.y, q.z, q.w};
        matrix_image_put(image + uint64_t(row) * K, K, quad, matrix_quad(v));
    }
}

// The rows of nt tokens (lane t < nt of every wave holds token t's row index in `from`) into LDS.  IMAGE: x holds row images, else fp32
// rows.  Returns whether this thread met a strange value.  (What stands in the place of tokens that are not there is not used.)
template <int BITS, int WIDTH, bool IMAGE>
__device__ __forceinline__ bool matrix_stage(const float* x, uint32_t K, uint32_t nt, uint32_t from, uint8_t* lds) {
    using Form = MatrixForm<BITS, WIDTH>;
    const uint32_t tid = matrix_thread(), lane = tid & 63u, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t padded = Form::steps(K) * Form::kStep, chunks = (padded + 511) / 512, units = nt * chunks;   // a unit: 512 elements of one token, eight a lane
    uint32_t strange = 0;
    constexpr uint32_t kBatch = IMAGE ? 4 : 2;
    uint32_t t = 0, c = wave;
    while (c >= chunks) { c -= chunks; ++t; }
#pragma unroll 1
    for (uint32_t u0 = wave; u0 < units; u0 += kMatrixWaves * kBatch) {
        uint4 first[kBatch], second[kBatch];   // IMAGE: pairs and, in two words, information
        uint32_t at_t[kBatch], at_c[kBatch];
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) {
            at_t[i] = min(t, nt - 1); at_c[i] = c;   // (past the end: some unit again, not used)
            const uint32_t row = uint32_t(__builtin_amdgcn_readlane(int(from), int(at_t[i]))), e = c * 512 + lane * 8, piece = e < K ? e / 8 : 0u;
            const float* src = x + uint64_t(row) * K;
            if constexpr (IMAGE) {
                first[i] = ldg_u4(src, piece);
                const uint2 info = ldg_u2(src + K / 2, piece);
                second[i] = make_uint4(info.x, info.y, 0, 0);
            } else { first[i] = ldg_u4(src, 2 * piece); second[i] = ldg_u4(src, 2 * piece + 1); }
            c += kMatrixWaves;
            while (c >= chunks) { c -= chunks; ++t; }
        }
#pragma unroll
        for (uint32_t i = 0; i < kBatch; ++i) {
            if (u0 + kMatrixWaves * i >= units) break;
            MatrixQuad q[2];
            if constexpr (IMAGE) {
                q[0] = {make_uint2(first[i].x, first[i].y), second[i].x}; q[1] = {make_uint2(first[i].z, first[i].w), second[i].y};
            } else {
                const uint32_t v[2][4] = {{first[i].x, first[i].y, first[i].z, first[i].w}, {second[i].x, second[i].y, second[i].z, second[i].w}};
                q[0] = matrix_quad(v[0]); q[1] = matrix_quad(v[1]);
            }
            const uint32_t e = at_c[i] * 512 + lane * 8;
            const bool active = e < padded;
            if (!Form::kWhole && e >= K) { q[0] = MatrixQuad{}; q[1] = MatrixQuad{}; }   // the last step's missing half: zeros
            const uint32_t step = e / Form::kStep, block = WIDTH == 16 ? lane >> 1 : lane & 31u, half = block & 1u, b = block >> 1, piece = WIDTH == 16 ? lane & 1u : 0u;
            strange |= active ? q[0].info | q[1].info : 0u;
            const float s0 = __uint_as_float(q[0].info & 0xffff0000u), s1 = __uint_as_float(q[1].info & 0xffff0000u);
            float sum;
            if constexpr (BITS == 8) {
                auto low = [](uint32_t pair) { return __uint_as_float(pair << 16); };
                auto high = [](uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); };
                sum = (((((((low(q[0].pairs.x) + low(q[0].pairs.y)) + high(q[0].pairs.x)) + high(q[0].pairs.y)) + low(q[1].pairs.x)) + low(q[1].pairs.y)) + high(q[1].pairs.x)) + high(q[1].pairs.y));
            } else if constexpr (WIDTH == 16) sum = (dpp_f32<0xa0>(s0 + s1) + s0) + s1;   // in the odd lane: quads 0 and 1 of the even one (quad_perm [0,0,2,2]) before its own
            else sum = s0 + s1;
            if (active) {
                *reinterpret_cast<uint4*>(lds + (2 * step + half) * Form::kHalfBytes + piece * 1024 + matrix_piece(b, at_t[i]) * 16) = make_uint4(q[0].pairs.x, q[0].pairs.y, q[1].pairs.x, q[1].pairs.y);
                if (WIDTH == 8 || piece == 1) *reinterpret_cast<float*>(lds + Form::sums_at(K) + (2 * step + half) * 256 + b * 16 + at_t[i] * 4) = sum;
            }
            if constexpr (BITS == 4) {   // bit 4 h + k: quad k of a block of half h
                const uint64_t m0 = __ballot(q[0].info & 1u), m1 = __ballot(q[1].info & 1u);
                uint32_t bits = 0;
                if constexpr (WIDTH == 16) {
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) bits |= (m0 & (0x1111111111111111ull << j) ? 1u << 2 * j : 0u) | (m1 & (0x1111111111111111ull << j) ? 2u << 2 * j : 0u);
                } else {
                    const uint32_t mine0 = uint32_t(m0 >> (lane & 32u)), mine1 = uint32_t(m1 >> (lane & 32u));
#pragma unroll
                    for (uint32_t j = 0; j < 2; ++j) bits |= (mine0 & (0x55555555u << j) ? 1u << 4 * j : 0u) | (mine1 & (0x55555555u << j) ? 2u << 4 * j : 0u);
                }
                if (active && (lane & (4 * WIDTH - 1)) == 0) lds[Form::bits_at(K) + at_t[i] * kMatrixSteps + step] = uint8_t(bits);
            }
        }
    }
    return (strange & 2u) != 0;
}

// Two streams of four weight rows a wave: gate and up of the same four outputs, or two runs of four outputs.  The waves of a workgroup take
// its range of such tiles in turn.
template <int BITS, int WIDTH, bool GATED>
struct MatrixStream {
    using Form = MatrixForm<BITS, WIDTH>;
    static constexpr uint32_t kTileRows = GATED ? 4 : 8, kRows = GATED ? 1 : 2, DW = Form::DW;   // output rows of a tile, rows of a lane
    struct Slot { uint32_t q[2][2 * DW]; uint16_t g[2]; };   // of each stream: two neighbouring blocks' codes, and their group's scale (even b) or bias (odd b)
    uint32_t K, N, steps, lane, tile, end, step;             // tile, step: the next one to request
    AffineMatrix m[2];
    const uint8_t* meta[GATED ? 2 : 1];                      // this lane's array: scales or biases
    // Byte offsets of this lane's blocks in the next step (a matrix has less than 4 GiB).  They move by one addition a step, the same in every lane.
    // Rows of half a step more stop at the matrix's last load: past it are rows behind the last one, which are not stored, and the missing half
    // of its last step; the missing halves of other rows read the row behind.  (Whole rows come eight at a time and never end inside a tile.)
    uint32_t w_at[kRows], g_at[kRows];
    __device__ __forceinline__ void move(uint32_t w, uint32_t g) {
#pragma unroll
        for (uint32_t i = 0; i < kRows; ++i) {
            w_at[i] += w; g_at[i] += g;
            if constexpr (!Form::kWhole) { w_at[i] = min(w_at[i], N * (K / 8 * BITS) - DW * 8); g_at[i] = min(g_at[i], N * (K / 64) * 2 - 2); }
        }
    }
    __device__ __forceinline__ void aim() {
#pragma unroll
        for (uint32_t i = 0; i < kRows; ++i) {
            const uint32_t r = min(tile * kTileRows + i * 4 + (lane & 3u), N - 1);
            w_at[i] = r * (K / 8 * BITS) + (lane >> 2) * (DW * 8);
            g_at[i] = (r * (K / 64) + (lane >> 2) * 2 * WIDTH / 64) * 2;
        }
        move(0, 0);
    }
    __device__ __forceinline__ void fetch(Slot& slot) {      // past the end: the matrix's first row, the same bytes in every lane, not used
#pragma unroll
        for (uint32_t i = 0; i < kRows; ++i) asm volatile("" : "+v"(w_at[i]), "+v"(g_at[i]));   // (else a step that is requested again is copied, which waits for it)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const AffineMatrix& a = m[GATED ? q : 0];
            const uint32_t i = GATED ? 0 : q;
            if constexpr (DW == 2) {
                const uint4 v = ldg_u4_by_words(a.w + w_at[i]);
                slot.q[q][0] = v.x; slot.q[q][1] = v.y; slot.q[q][2 * DW - 2] = v.z; slot.q[q][2 * DW - 1] = v.w;
            } else { const uint2 v = ldg_u2_by_words(a.w + w_at[i]); slot.q[q][0] = v.x; slot.q[q][1] = v.y; }
            slot.g[q] = ldg_u16(meta[GATED ? q : 0] + g_at[i]);
        }
        constexpr uint32_t kW = 32 * DW * 4, kG = Form::kStep / 64 * 2;
        if (++step < steps) { move(kW, kG); return; }
        step = 0;
        if (tile + kMatrixWaves < end) {
            tile += kMatrixWaves;
            move(kMatrixWaves * kTileRows * (K / 8 * BITS) - (steps - 1) * kW, kMatrixWaves * kTileRows * (K / 64) * 2 - (steps - 1) * kG);
            return;
        }
#pragma unroll
        for (uint32_t i = 0; i < kRows; ++i) w_at[i] = g_at[i] = 0;
    }
};

__device__ __forceinline__ f32x4 matrix_chain_step(float x, float code, f32x4 c) { return __builtin_amdgcn_mfma_f32_4x4x1f32(x, code, c, 0, 0, 0); }
__device__ __forceinline__ float low_bf16(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float high_bf16(uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); }

// Four tokens' partial sums (register r: token r) over the lanes of equal (lane % 4), strides 16, 8, 4, 2 of the reference's lanes: every lane
// ends with the sum of row lane % 4 for token {0, 2, 1, 3}[lane / 16].
__device__ __forceinline__ float matrix_add_rows(float a, float b) {   // rows of sixteen lanes 0 and 2: a's rows 0 + 1, 2 + 3; rows 1 and 3: b's
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
}
__device__ __forceinline__ float matrix_reduce(f32x4 v) {
    auto swap_sum = [](auto rows) { return __uint_as_float(rows[0]) + __uint_as_float(rows[1]); };
    const float a = swap_sum(__builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[1]), false, false));
    const float b = swap_sum(__builtin_amdgcn_permlane32_swap(__float_as_uint(v[2]), __float_as_uint(v[3]), false, false));
    float s = matrix_add_rows(a, b);
    s = s + dpp_f32<0x128>(s);   // row_ror:8
    return s + dpp_f32<0x124>(s);   // row_ror:4
}

// The priority of a wave among those of its SIMD, by what is left of its workgroup's share (in steps): the top one at first, one less at
// a half, a quarter and an eighth.  A SIMD issues its oldest wave first among equals, so that of four workgroups on a compute unit, with shares
// alike, the first ended at 55 us and the last at 130, the end of it alone (64 tokens of hidden 3072 that agree, gate/up); this way those ahead
// give way to those behind.
struct MatrixPace {
    uint32_t next, level;
    __device__ __forceinline__ explicit MatrixPace(uint32_t all) : next(all / 2), level(3) { __builtin_amdgcn_s_setprio(3); }
    __device__ __forceinline__ void left(uint32_t steps) {
        if (steps > next || level == 0) return;
        next /= 2; --level;
        if (level == 2) __builtin_amdgcn_s_setprio(2);
        else if (level == 1) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
    }
};

// The walk over tiles for nt <= TOKENS staged tokens (1, 2 or 4); out_at: where the output row of this lane's token begins; chains: lane s holds
// step s's quad bits.  IMAGE (gate/up): output rows are images of the activations.
template <int BITS, int WIDTH, bool GATED, uint32_t TOKENS, bool IMAGE>
__device__ __forceinline__ void matrix_walk(MatrixStream<BITS, WIDTH, GATED>& st, const typename MatrixStream<BITS, WIDTH, GATED>::Slot& next, const uint8_t* lds, uint32_t chains,
                                            float* out, uint64_t out_at, uint32_t tile, bool float_output, uint32_t nt, uint32_t token, MatrixPace& pace, uint32_t after) {
    using Stream = MatrixStream<BITS, WIDTH, GATED>;
    using Slot = typename Stream::Slot;
    using Form = MatrixForm<BITS, WIDTH>;
    const uint32_t lane = st.lane, total = tile < st.end ? (st.end - tile + kMatrixWaves - 1) / kMatrixWaves * st.steps : 0u;
    const uint32_t rows_at = matrix_piece(lane >> 2, lane & 3u) * 16, sums_at = Form::sums_at(st.K) + lane * 4;
    const f32x4 zero = {0, 0, 0, 0};
    float acc[2][2][TOKENS];   // [stream][half][token]
    auto clear = [&] {
#pragma unroll
        for (uint32_t i = 0; i < 4 * TOKENS; ++i) (&acc[0][0][0])[i] = 0;
    };
    clear();
    Slot ring[2] = {next, {}};
    st.fetch(ring[1]);
    uint32_t step = 0;
    auto one = [&](const Slot& now) {
        asm volatile("; %0 tokens" : : "n"(TOKENS));   // (else the walks' first steps move in front of the choice between the walks)
        const uint32_t chained = BITS == 4 ? uint32_t(__builtin_amdgcn_readlane(int(chains), int(step))) : 0u;
        float scale[2], bias[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {   // (a bank of four lanes is one b: odd banks take the scale from the bank before, even ones the bias from the one behind)
            const int mine = int(uint32_t(now.g[q]) << 16);
            scale[q] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(mine, mine, 0x114, 0xf, 0xa, false));
            bias[q] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(mine, mine, 0x104, 0xf, 0x5, false));
        }
        if constexpr (!Form::kWhole) {   // (past the row's end: nothing, whatever the last pair's scale and bias are)
            const bool inside = step * 32 + (lane >> 2) * 2 < st.K / WIDTH;
#pragma unroll
            for (int q = 0; q < 2; ++q) { scale[q] = inside ? scale[q] : 0.0f; bias[q] = inside ? bias[q] : 0.0f; }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 rows[WIDTH / 8];
#pragma unroll
            for (int i = 0; i < WIDTH / 8; ++i) rows[i] = *reinterpret_cast<const u32x4*>(lds + (2 * step + h) * Form::kHalfBytes + i * 1024 + rows_at);
            const float sum = *reinterpret_cast<const float*>(lds + sums_at + (2 * step + h) * 256);
            auto fold = [&](int q, const f32x4 dot) {
                const f32x4 shift = matrix_chain_step(sum, bias[q], zero);   // bias * sum (a product added to zero)
#pragma unroll
                for (uint32_t r = 0; r < TOKENS; ++r) acc[q][h][r] = acc[q][h][r] + (scale[q] * dot[r] + shift[r]);
            };
            auto multiply = [&]<bool CHAINS>(uint32_t bits) {   // bits: the quads whose chain has to be run
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    if constexpr (BITS == 4) {
                        s16x4 code[Form::kQuads];   // bf16 codes, a quad's elements in the order 0 2 1 3 (a nibble read as an 8-bit float of four exponent bits is code * 2^-9)
#pragma unroll
                        for (uint32_t i = 0; i < Form::DW; ++i) {
                            uint32_t word = now.q[q][h * Form::DW + i];
                            asm volatile("" : "+v"(word));   // (else both streams' codes are converted before the first products)
                            const uint32_t even = word & 0x0f0f0f0fu, odd = (word >> 4) & 0x0f0f0f0fu;
                            auto two = [](bf16x2 v) { return __builtin_bit_cast(uint32_t, v); };
                            code[2 * i] = __builtin_bit_cast(s16x4, make_uint2(two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 512.0f, false)), two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 512.0f, false))));
                            code[2 * i + 1] = __builtin_bit_cast(s16x4, make_uint2(two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 512.0f, true)), two(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 512.0f, true))));
                        }
                        auto pair = [&](uint32_t k, int which) { return rows[k / 2][2 * (k % 2) + which]; };
                        f32x4 quad[Form::kQuads], dot;
#pragma unroll
                        for (uint32_t k = 0; k < Form::kQuads; ++k) {
                            quad[k] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, make_uint2(pair(k, 0), pair(k, 1))), code[k], zero, 0, 0, 0);
                            if constexpr (CHAINS) {
                                if (bits >> k & 1u) {
                                    uint2 c = __builtin_bit_cast(uint2, code[k]);
                                    asm volatile("" : "+v"(c.x), "+v"(c.y));
                                    quad[k] = matrix_chain_step(low_bf16(pair(k, 0)), low_bf16(c.x), zero);
                                    quad[k] = matrix_chain_step(low_bf16(pair(k, 1)), low_bf16(c.y), quad[k]);
                                    quad[k] = matrix_chain_step(high_bf16(pair(k, 0)), high_bf16(c.x), quad[k]);
                                    quad[k] = matrix_chain_step(high_bf16(pair(k, 1)), high_bf16(c.y), quad[k]);
                                }
                                dot = k == 0 ? quad[0] : dot + quad[k];
                                asm volatile("" : "+v"(dot));   // (else the sums wait until all four quads are there)
                            }
                        }
                        if constexpr (!CHAINS) {
                            dot = quad[0];
#pragma unroll
                            for (uint32_t k = 1; k < Form::kQuads; ++k) dot = dot + quad[k];
                        }
                        fold(q, dot);
                    } else {
                        float byte[8];
#pragma unroll
                        for (int k = 0; k < 8; ++k) byte[k] = float((now.q[q][h * Form::DW + k / 4] >> (8 * (k % 4))) & 255u);
                        f32x4 dot = zero;
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            const uint32_t pair = rows[0][2 * (k / 4) + k % 2];
                            dot = matrix_chain_step(k % 4 < 2 ? low_bf16(pair) : high_bf16(pair), byte[k], dot);
                        }
                        fold(q, dot);
                    }
                }
            };
            if constexpr (BITS == 4) {
                const uint32_t bits = chained >> (4 * h) & 15u;
                if (__builtin_expect(bits == 0, 1)) multiply.template operator()<false>(0);
                else { multiply.template operator()<true>(bits); asm volatile("; chains run"); }   // (an end of its own: else the last sums of both ways are joined behind them)
            } else multiply.template operator()<false>(0);
        }
        if (++step < st.steps) return;
        step = 0;
        float v[2];
        uint32_t in_tile;                                  // lane 4 b + j: row j of the tile, or of its second four
        bool mine = token < nt;                            // (one lane of each result)
        if constexpr (TOKENS <= 2) {                       // halves and streams take the places of four tokens in the sums (rows of a step or two are mostly their end: with
                                                           // this and offsets that move by an addition 40 tokens' down of 640 inputs 111 -> 104 us, 32 tokens' of 512 47 -> 45)
            float s[TOKENS];
#pragma unroll
            for (uint32_t t = 0; t < TOKENS; ++t) s[t] = matrix_reduce(f32x4{acc[0][0][t], acc[1][0][t], acc[0][1][t], acc[1][1][t]});
            v[0] = v[1] = matrix_add_rows(s[0], s[TOKENS - 1]);   // lanes from 32 on: the second stream's; odd rows of lanes: token 1's
            in_tile = (lane & 3u) + (GATED ? 0u : lane >> 5 << 2);
            mine = mine && !(lane & (GATED ? 44u : 12u));
            if constexpr (GATED) {
                const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[0]), false, false);
                v[0] = __uint_as_float(both[0]); v[1] = __uint_as_float(both[1]);
            }
        } else {                                           // the second four where b is odd; b / 4 the token
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                f32x4 first, second;
#pragma unroll
                for (uint32_t r = 0; r < TOKENS; ++r) { first[r] = acc[q][0][r]; second[r] = acc[q][1][r]; }
                v[q] = matrix_reduce(first) + matrix_reduce(second);
            }
            in_tile = lane & (GATED ? 3u : 7u);
            mine = mine && !(lane & (GATED ? 12u : 8u));
            if (!GATED && (lane & 4u)) v[0] = v[1];
        }
        clear();
        const float y = GATED ? swiglu_bf(v[0], v[1]) : float_output ? v[0] : bf(v[0]);
        const uint32_t row = tile * Stream::kTileRows + in_tile;
        mine = mine && row < st.N;
        if constexpr (IMAGE) {   // the wave's four outputs of a token are a quad
            const uint32_t quad[4] = {__float_as_uint(dpp_f32<0x00>(y)), __float_as_uint(dpp_f32<0x55>(y)), __float_as_uint(dpp_f32<0xaa>(y)), __float_as_uint(dpp_f32<0xff>(y))};
            const MatrixQuad put = matrix_quad(quad);
            if (mine && (lane & 3u) == 0) matrix_image_put(out + out_at, st.N, row / 4, put);
        } else if (mine) out[out_at + row] = y;
        tile += kMatrixWaves;
    };
    // A slot is requested again, in place, as soon as its step is done.  (With a copy of the slot in use the compiler waited at the loop's end for all
    // loads in flight; so it did where the loop could be left in its middle, hence the question in front of a step past the end.  Three slots: 3 to 8 % longer.)
#pragma unroll 1
    for (uint32_t i = 0; i < total; i += 2) {
        pace.left(after + total - i);
#pragma unroll
        for (uint32_t k = 0; k < 2; ++k) {
            if (i + k < total) one(ring[k]);
            __builtin_amdgcn_sched_barrier(0);
            st.fetch(ring[k]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Output rows first .. last - 1 of a job where a token's products may round: on the lanes (zc_affine.hpp), two tokens at a time.  Inputs are BF16 by
// contract; rows that are not cost more here than by the lanes' own kernels, since the work list is cut as if all jobs took the same time, and a job
// of four tokens is two turns.  us, a row at a time with nothing requested ahead -> this (the lanes' kernels): layers whose rows are all fp32, 8 tokens of
// hidden 2048 145 -> 93 (69), 64 of 2048 656 -> 361 (273), 64 of 3072 2089 -> 965 (668); gate/up 3072 x 1024 at 128 and 512 rows 163 -> 104 (82) and
// 599 -> 328 (291), with one such row among them 97 -> 46 (58) and 356 -> 146 (201).
template <int BITS, int WIDTH, bool GATED, class Load, class Put, class InRow, class OutRow>
__device__ __forceinline__ void matrix_strange_rows(const AffineMatrix (&m)[2], uint32_t K, uint32_t N, Load load, Put put, uint32_t nt, InRow in_row, OutRow out_row,
                                                    uint32_t first, uint32_t last, bool float_output, uint8_t* lds) {
    constexpr uint32_t kRows = AffineStream<BITS, WIDTH, GATED, kAffineTokens>::kTileRows;
    static_assert(kMatrixWaves * MatrixStream<BITS, WIDTH, GATED>::kTileRows % kRows == 0);   // a workgroup's range is whole tiles of either form
    asm volatile("" : "+s"(K), "+s"(N), "+s"(first), "+s"(last));   // (else what is formed from them is formed in front of the loop over jobs, for every job)
    const uint32_t most = kAffineTokens * affine_token_bytes<WIDTH>(K) <= matrix_lds_bytes<BITS, WIDTH>(K) ? kAffineTokens : 1u;
#pragma unroll 1
    for (uint32_t t0 = 0; t0 < nt; t0 += most) {
        lds_barrier();   // what was staged before has been read
        affine_rows_by<BITS, WIDTH, GATED, kAffineTokens>(m, K, N, 64, load, put, min(most, nt - t0), [&](uint32_t t) { return in_row(t0 + t); },
                                                          [&](uint32_t t) { return out_row(t0 + t); }, first / kRows, (last + kRows - 1) / kRows, float_output, lds, matrix_thread());
    }
}

// Tiles tile0 .. end - 1 (of MatrixStream) for nt <= 4 tokens: input row in_row(t), output row out_row(t); after: rounds that the workgroup has left then.
// IN: input rows are images (gate/up: made of the rows `fp32`; else written as images); OUT: output rows are to be.
// (A workgroup that runs several of them waits in front of each: what the one before staged has then been read.)
template <int BITS, int WIDTH, bool GATED, bool IN, bool OUT, class InRow, class OutRow>
__device__ __forceinline__ void matrix_rows(const AffineMatrix (&m)[2], uint32_t K, uint32_t N, const float* x, const float* fp32, float* out, uint32_t nt,
                                            InRow in_row, OutRow out_row, uint32_t tile0, uint32_t end, bool float_output, uint8_t* lds, MatrixPace& pace, uint32_t after) {
    using Stream = MatrixStream<BITS, WIDTH, GATED>;
    using Form = MatrixForm<BITS, WIDTH>;
    Stream st;
    const uint32_t tid = matrix_thread(), wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6))), first_tile = tile0 + wave;
    st.K = K; st.N = N; st.steps = Form::steps(K); st.lane = tid & 63u; st.tile = min(first_tile, end - 1); st.end = end; st.step = 0;
    st.m[0] = m[0]; st.m[1] = m[1];
#pragma unroll
    for (int q = 0; q < (GATED ? 2 : 1); ++q) st.meta[q] = reinterpret_cast<const uint8_t*>(st.lane & 4u ? m[q].b : m[q].s);
    const uint32_t from = st.lane < nt ? in_row(st.lane) : 0u;
    typename Stream::Slot next;
    st.aim();
    st.fetch(next);
    const uint32_t row16 = st.lane >> 4, token = nt <= 2 ? row16 & 1u : row16 == 1 ? 2u : row16 == 2 ? 1u : row16;   // as the sums are left
    const uint64_t out_at = uint64_t(out_row(min(token, nt - 1))) * N;
    uint32_t* found = reinterpret_cast<uint32_t*>(lds + Form::found_at(K));
    const bool any = __ballot(matrix_stage<BITS, WIDTH, IN>(x, K, nt, from, lds)) != 0;
    if (st.lane == 0) found[wave] = any;
    lds_barrier();
    const bool strange = __ballot(found[st.lane % kMatrixWaves] != 0) != 0;
    if (__builtin_expect(!strange, 1)) {
        uint32_t chains = 0;
        if constexpr (BITS == 4) {
            for (uint32_t t = 0; t < nt; ++t) chains |= lds[Form::bits_at(K) + t * kMatrixSteps + min(st.lane, st.steps - 1)];
        }
        auto walk = [&]<uint32_t TOKENS>() { matrix_walk<BITS, WIDTH, GATED, TOKENS, OUT>(st, next, lds, chains, out, out_at, first_tile, float_output, nt, token, pace, after * st.steps); };
        if (nt == 1) walk.template operator()<1>();
        else if (nt == 2) walk.template operator()<2>();
        else walk.template operator()<4>();
        return;
    }
    matrix_strange_rows<BITS, WIDTH, GATED>(m, K, N, [&](uint32_t row, uint32_t i) {
        if constexpr (!IN) return ldg_u4(x + uint64_t(row) * K, i);
        else if constexpr (GATED) return ldg_u4(fp32 + uint64_t(row) * K, i);
        else {   // (rows that were made as images are BF16)
            const uint2 pairs = ldg_u2(x + uint64_t(row) * K, i);
            return make_uint4(pairs.x << 16, pairs.y << 16, pairs.x & 0xffff0000u, pairs.y & 0xffff0000u);
        }
    }, [&](uint64_t at, uint32_t row, float y) {
        if constexpr (OUT) reinterpret_cast<uint16_t*>(out + at)[row / 4 * 4 + (row & 1u) * 2 + (row >> 1 & 1u)] = uint16_t(__float_as_uint(y) >> 16);
        else out[at + row] = y;
    }, nt, in_row, out_row, tile0 * Stream::kTileRows, min(end * Stream::kTileRows, N), float_output, lds);
    if constexpr (OUT) {   // the information words, from the pairs that the workgroup has just stored
        __syncthreads();
        const uint32_t first = tile0 * Stream::kTileRows / 4, quads = min(end * Stream::kTileRows, N) / 4 - first;
        for (uint32_t i = matrix_thread(); i < nt * quads; i += kMatrixThreads) {
            float* row = out + uint64_t(out_row(i / quads)) * N;
            const uint32_t quad = first + i % quads;
            const uint2 pairs = reinterpret_cast<const uint2*>(row)[quad];
            const uint32_t v[4] = {pairs.x << 16, pairs.y << 16, pairs.x & 0xffff0000u, pairs.y & 0xffff0000u};
            matrix_image_put(row, N, quad, matrix_quad(v));
        }
    }
}

// How the work of a launch, `jobs` jobs of `rounds` rounds (a tile per wave), is cut: workgroup w of n takes a contiguous piece, so that it stages a
// job's rows once and all pieces are alike to a round; workgroups of one XCD (every eighth) take neighbouring pieces, so that the jobs of
// one expert read its weights through one L2.  run(job, first round, end round, pace, rounds left then).
template <class Run>
__device__ __forceinline__ void matrix_piece_of_work(uint32_t jobs, uint32_t rounds, uint32_t steps, Run run) {
    const uint32_t n = gridDim.x, w = n % 8 == 0 ? blockIdx.x % 8 * (n / 8) + blockIdx.x / 8 : blockIdx.x;
    const uint64_t work = uint64_t(jobs) * rounds;
    const uint64_t first = work * w / n, end = work * (w + 1) / n;
    uint32_t job = uint32_t(first / rounds), round = uint32_t(first - uint64_t(job) * rounds);
    uint64_t left = end - first;
    MatrixPace pace(uint32_t(left) * steps);
#pragma unroll 1
    while (left) {
        const uint32_t take = uint32_t(min(left, uint64_t(rounds - round)));
        run(job, round, round + take, pace, uint32_t(left - take));
        left -= take; round = 0; ++job;
        if (left) lds_barrier();
    }
}

}  // namespace zc
