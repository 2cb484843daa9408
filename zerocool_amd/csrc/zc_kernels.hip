// Operator kernels of the MoE path with the reference's arithmetic kept to the bit:
// the 32-lane partition of every affine dot, the scalar order inside a lane, every
// BF16 rounding boundary.  On the lanes (zc_affine.hpp) one GPU lane plays one reference
// lane; on the matrix cores (zc_affine_matrix.hpp) sums that are exact in any order are
// formed together.  Results are bit-identical to the CPU statement of the same
// arithmetic for any input.
#include "zc_kernels.hpp"
#include <algorithm>
#include <type_traits>
#include "zc_device.hpp"
#include "zc_affine_matrix.hpp"
#include "zc_decode_common.hpp"   // lds_barrier; route_token: top-k + softmax of one token by one wavefront

namespace zc {

struct AffineJob {
    AffineMatrix m[2];               // gate (or the only matrix), up
    const float* x;                  // input rows, K floats each
    const int32_t* in_rows;          // gather of input rows, or null
    const int32_t* out_rows;         // scatter of output rows, or null
    float* out;                      // output rows, N floats each
    uint32_t K, N, group, tokens, chunk, float_output;   // chunk: tokens of a workgroup
    uint32_t tiles, share;           // row tiles, and how many of them a workgroup takes
    GatherCheck check;
};
// Whether the gather's list, of n rows, holds one outside the input; the launch's first wave answers the host.  Every wave looks at the whole
// list, so that no workgroup reads or writes anything of a refused call, and none waits for another: the list's words arrive with the
// workgroup's own.  (Where the host copies the list and looks at it before it enqueues the product, the GPU idles: eight
// experts of 21 rows each, hidden 2560 and intermediate 640, gate/up, down and scatter 337 us -> 186 this way.)
__device__ __forceinline__ bool gather_outside(const int32_t* rows, uint32_t n, uint32_t x_rows) {
    bool outside = false;
#pragma unroll
    for (uint32_t i = 0; i < kGatherInKernel; i += 64) outside |= ldg_u32(rows, min(i + (threadIdx.x & 63u), n - 1)) >= x_rows;
    return __ballot(outside) != 0;
}
__device__ __forceinline__ void gather_answer(const GatherCheck& c, bool outside) {
    __hip_atomic_store(c.slot, c.answer + (outside ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);   // (the word is all that the host waits for)
}
__device__ __forceinline__ bool gather_refused(const AffineJob& j) {
    if (!j.check.slot) return false;
    const bool outside = gather_outside(j.in_rows, j.tokens, j.check.x_rows);
    if (threadIdx.x == 0 && blockIdx.x + blockIdx.y + blockIdx.z == 0) gather_answer(j.check, outside);
    return outside;
}
__global__ __launch_bounds__(1024) void gather_check_kernel(const int32_t* rows, uint32_t n, GatherCheck check) {
    int outside = 0;
    for (uint32_t i = threadIdx.x; i < n; i += 1024) outside |= uint32_t(rows[i]) >= check.x_rows;
    outside = __syncthreads_or(outside);
    if (threadIdx.x == 0) gather_answer(check, outside != 0);
}
void launch_gather_check(hipStream_t s, const int32_t* rows, uint32_t n, const GatherCheck& check) {
    hipLaunchKernelGGL(gather_check_kernel, dim3(1), dim3(1024), 0, s, rows, n, check);
}
template <int BITS, int WIDTH, bool GATED, uint32_t TOKENS>
__global__ __launch_bounds__(256, TOKENS == 1 ? 4 : 3) void affine_op_kernel(AffineJob j) {
    extern __shared__ __align__(16) uint8_t affine_lds[];
    const uint32_t tile0 = blockIdx.x * j.share, end = min(tile0 + j.share, j.tiles);
    const uint64_t t0 = (uint64_t(blockIdx.z) * gridDim.y + blockIdx.y) * j.chunk;
    if (t0 >= j.tokens) return;
    if constexpr (GATED) { if (gather_refused(j)) return; }
    affine_rows<BITS, WIDTH, GATED, TOKENS>(j.m, j.K, j.N, j.group, j.x, j.out, min(j.chunk, j.tokens - uint32_t(t0)),
                                            [&](uint32_t t) { return j.in_rows ? uint32_t(j.in_rows[t0 + t]) : uint32_t(t0) + t; },
                                            [&](uint32_t t) { return j.out_rows ? uint32_t(j.out_rows[t0 + t]) : uint32_t(t0) + t; }, tile0, end, j.float_output != 0, affine_lds);
}

template <int BITS, int WIDTH, bool GATED>
__global__ __launch_bounds__(kMatrixThreads, 4) void affine_matrix_kernel(AffineJob j) {
    extern __shared__ __align__(16) uint8_t affine_lds[];
    if constexpr (GATED) { if (gather_refused(j)) return; }
    matrix_piece_of_work((j.tokens - 1) / kMatrixTokens + 1, (j.tiles + kMatrixWaves - 1) / kMatrixWaves, MatrixForm<BITS, WIDTH>::steps(j.K), [&](uint32_t job, uint32_t round, uint32_t rounds, MatrixPace& pace, uint32_t after) {
        const uint64_t t0 = uint64_t(job) * j.chunk;
        matrix_rows<BITS, WIDTH, GATED, false, false>(j.m, j.K, j.N, j.x, nullptr, j.out, min(j.chunk, j.tokens - uint32_t(t0)),
                                                              [&](uint32_t t) { return j.in_rows ? uint32_t(j.in_rows[t0 + t]) : uint32_t(t0) + t; },
                                                              [&](uint32_t t) { return j.out_rows ? uint32_t(j.out_rows[t0 + t]) : uint32_t(t0) + t; },
                                                              round * kMatrixWaves, min(rounds * kMatrixWaves, j.tiles), j.float_output != 0, affine_lds, pace, after);
    });
}

// The routed experts of one layer and the shared expert (the lanes' lists: where its format is theirs): blockIdx.y walks the shared expert's
// tokens, chunk by chunk, then the list of (expert, sorted positions) that the dispatch left; jobs past the device-side count exit.
struct ExpertPhase {
    const uint8_t* records; uint64_t stride; uint64_t off[6];          // byte offsets inside a record: codes, scales, biases of the (gate | down) projection, of up
    const uint8_t* shared_record; uint64_t shared_off[6];
    const uint32_t *jobs; const int32_t *count, *slots;
    const float *x, *shared_x; float *out, *shared_out;                // x: layer input (gate/up) or sorted activations (down); on the matrix cores both as row images
    const float* fp32;                                                 // matrix cores, gate/up: the rows that the images x and shared_x were made of
    const float* logits; int32_t *ids, *status; float* weights; uint32_t E;   // of one token alone: job j of the routed ones is its pick j
    uint32_t K, N, group, topk, tokens, chunk, shared_jobs, max_jobs, tiles, share;   // chunk: tokens of a job (a shared job too)
};
// Elements of a block of the shared expert's rows, of SHARED bits, where the routed experts have BITS and WIDTH: the row lengths are the same.
constexpr int shared_width(int BITS, int WIDTH, int SHARED) { return SHARED == BITS ? WIDTH : SHARED == 4 ? 2 * WIDTH : WIDTH / 2; }
__device__ __forceinline__ void expert_matrices(const ExpertPhase& p, bool shared, uint32_t expert, AffineMatrix (&m)[2]) {
    const uint8_t* r = shared ? p.shared_record : p.records + uint64_t(expert) * p.stride;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        auto at = [&](int i) { return r + (shared ? p.shared_off[3 * q + i] : p.off[3 * q + i]); };
        m[q] = AffineMatrix{at(0), reinterpret_cast<const uint16_t*>(at(1)), reinterpret_cast<const uint16_t*>(at(2))};
    }
}
// A job, if there is one of that number: its matrices, tokens and rows go to `run`.
template <bool GATED, class Run>
__device__ __forceinline__ void expert_job(const ExpertPhase& p, uint32_t job, Run run) {
    const bool shared = job < p.shared_jobs;
    uint32_t first = job * p.chunk, expert = 0, nt = min(p.chunk, p.tokens - first);
    if (!shared) {   // (the list has room for every job of the grid; what lies past the count is not used)
        const uint32_t count = uint32_t(uniform(*p.count)), packed = uint32_t(uniform(int32_t(p.jobs[min(job - p.shared_jobs, p.max_jobs - 1)])));
        if (job - p.shared_jobs >= count) return;
        first = packed & 0xfffffu; expert = (packed >> 20) & 1023u; nt = (packed >> 30) + 1u;
    }
    AffineMatrix m[2];
    expert_matrices(p, shared, expert, m);
    run(m, shared ? p.shared_x : p.x, shared ? p.shared_out : p.out, nt,
        [&, first](uint32_t t) { return GATED && !shared ? uint32_t(p.slots[first + t]) / p.topk : first + t; },
        [&, first](uint32_t t) { return GATED || shared ? first + t : uint32_t(p.slots[first + t]); });
}
template <int BITS, int WIDTH, bool GATED, uint32_t TOKENS>
__global__ __launch_bounds__(256, TOKENS == 1 ? 4 : 3) void expert_phase_kernel(ExpertPhase p) {
    extern __shared__ __align__(16) uint8_t affine_lds[];
    const uint32_t tile0 = blockIdx.x * p.share, end = min(tile0 + p.share, p.tiles);
    expert_job<GATED>(p, blockIdx.z * gridDim.y + blockIdx.y, [&](const AffineMatrix (&m)[2], const float* x, float* out, uint32_t nt, auto in_row, auto out_row) {
        affine_rows<BITS, WIDTH, GATED, TOKENS>(m, p.K, p.N, p.group, x, out, nt, in_row, out_row, tile0, end, false, affine_lds);
    });
}
// One token alone: there is nothing to sort, pick j's rows are row j.  The gate/up kernel makes the picks too (PER: candidates a lane, 0
// where `ids` holds the picks): the first wave of every workgroup selects them from the logits, all of them, while the others
// stage the input row.  Bound by the chain of latencies: logits -> picks -> codes, 2 to 2.5 us longer than a list's job -> codes, in
// place of a launch of 6 us and the gap behind it.  Hidden 2048, intermediate 512: picks, gate/up, down 5.9 + 9.0 + 5.6 -> 11.4 + 5.8 us, a
// layer 28.8 -> 23.6; hidden 2560, intermediate 640: 5.8 + 12.0 + 8.2 -> 13.0 + 7.0, a layer of a stack 37.7 -> 31.7.
template <int BITS, int WIDTH, bool GATED, int PER, int SHARED>
__global__ __launch_bounds__(256, 4) void expert_token_kernel(ExpertPhase p) {
    extern __shared__ __align__(16) uint8_t affine_lds[];
    const uint32_t tile0 = blockIdx.x * p.share, end = min(tile0 + p.share, p.tiles), tid = threadIdx.x;
    const bool shared = blockIdx.y < p.shared_jobs;
    const uint32_t row = shared ? 0u : blockIdx.y - p.shared_jobs;
    auto valid = [&](int32_t id) {
        if (uint32_t(id) < p.E) return true;
        if (tid == 0) atomicOr(p.status, 1);
        return false;
    };
    const float* x = shared ? p.shared_x : p.x;
    float* out = shared ? p.shared_out : p.out;
    auto in_row = [&](uint32_t) { return GATED ? 0u : row; };
    auto out_row = [&](uint32_t) { return row; };
    AffineMatrix m[2];
    if constexpr (SHARED != BITS) {
        if (shared) {
            expert_matrices(p, true, 0, m);
            affine_rows<SHARED, shared_width(BITS, WIDTH, SHARED), GATED, 1>(m, p.K, p.N, p.group, x, out, 1, in_row, out_row, tile0, end, false, affine_lds);
            return;
        }
    }
    if constexpr (PER == 0) {
        const int32_t id = shared ? 0 : uniform(p.ids[row]);
        if (!shared && !valid(id)) return;
        expert_matrices(p, shared, uint32_t(id), m);
        affine_rows<BITS, WIDTH, GATED, 1>(m, p.K, p.N, p.group, x, out, 1, in_row, out_row, tile0, end, false, affine_lds);
    } else {
        __shared__ int32_t ids_s[64];
        __shared__ float weights_s[64];
        __shared__ uint32_t pick[128];
        struct Picks {
            const ExpertPhase& p; const bool shared; const uint32_t row, tid; decltype(valid)& check;
            int32_t* ids; float* weights; uint32_t* pick;
            __device__ __forceinline__ void find() const {
                if (shared || tid >= 64) return;
                route_token<PER>([&](float (&cand)[PER], uint32_t per) {
#pragma unroll
                    for (int i = 0; i < PER; ++i) { const uint32_t e = tid * per + uint32_t(i); cand[i] = (uint32_t(i) < per && e < p.E) ? p.logits[e] : __uint_as_float(0xff800000u); }
                }, p.E, p.topk, tid, ids, weights, pick, [] {}, [] {});
            }
            __device__ __forceinline__ bool take(AffineMatrix (&m)[2]) const {
                int32_t id = 0;
                if (!shared) {
                    if (row == 0 && blockIdx.x == 0 && tid < p.topk) { p.ids[tid] = ids[tid]; p.weights[tid] = weights[tid]; }
                    id = uniform(ids[row]);
                    if (!check(id)) return false;
                }
                expert_matrices(p, shared, uint32_t(id), m);
                return true;
            }
        };
        affine_rows<BITS, WIDTH, GATED, 1>(m, p.K, p.N, p.group, x, out, 1, in_row, out_row, tile0, end, false, affine_lds,
                                           Picks{p, shared, row, tid, valid, ids_s, weights_s, pick});
    }
}
// SHARED: the bits of the shared expert's rows.  Where they are not BITS its jobs could have a launch of their own, 9.7 us for the Q8 gate/up of
// five tokens (hidden 2048, intermediate 512) in front of the routed Q4 jobs' 20 us; in one launch they take 26 us, a layer 63 -> 56.
template <int BITS, int WIDTH, bool GATED, int SHARED>
__global__ __launch_bounds__(kMatrixThreads, 4) void expert_matrix_kernel(ExpertPhase p) {
    extern __shared__ __align__(16) uint8_t affine_lds[];
    const uint32_t jobs = p.shared_jobs + uint32_t(uniform(*p.count));
    matrix_piece_of_work(jobs, (p.tiles + kMatrixWaves - 1) / kMatrixWaves, MatrixForm<BITS, WIDTH>::steps(p.K), [&](uint32_t job, uint32_t round, uint32_t rounds, MatrixPace& pace, uint32_t after) {
        expert_job<GATED>(p, job, [&](const AffineMatrix (&m)[2], const float* x, float* out, uint32_t nt, auto in_row, auto out_row) {
            if constexpr (SHARED != BITS) {
                if (job < p.shared_jobs) {
                    matrix_rows<SHARED, shared_width(BITS, WIDTH, SHARED), GATED, true, GATED>(m, p.K, p.N, x, p.fp32, out, nt, in_row, out_row, round * kMatrixWaves,
                                                                                               min(rounds * kMatrixWaves, p.tiles), false, affine_lds, pace, after);
                    return;
                }
            }
            matrix_rows<BITS, WIDTH, GATED, true, GATED>(m, p.K, p.N, x, p.fp32, out, nt, in_row, out_row, round * kMatrixWaves,
                                                                 min(rounds * kMatrixWaves, p.tiles), false, affine_lds, pace, after);
        });
    });
}

static bool wide(uint32_t K, uint32_t N) { return K % 512 == 0 && N % 8 == 0; }

template <bool GATED, typename Launch>
static void by_format(uint32_t bits, bool w, Launch&& launch) {
    if (bits == 4) { if (w) launch.template operator()<4, 16, GATED>(); else launch.template operator()<4, 8, GATED>(); }
    else           { if (w) launch.template operator()<8, 8, GATED>();  else launch.template operator()<8, 4, GATED>(); }
}
// Row tiles per workgroup: staging the input rows is paid once per workgroup, so as many as leave the chip a few thousand
// workgroups (256 compute units, up to five workgroups each).  (Eight tiles: 64 tokens of unshared experts 3 % faster, 16 to 32 tokens 3 to 5 % slower.)
static uint32_t affine_share(uint32_t tiles, uint64_t jobs) {
    uint32_t share = 4;
    while (share > 1 && uint64_t((tiles + share - 1) / share) * jobs < 2048) share /= 2;
    return share;
}
// Tokens per workgroup: two where their rows leave room for three workgroups in a compute unit's LDS.
template <int WIDTH> static uint32_t affine_chunk(uint32_t K) {
    uint32_t chunk = kAffineTokens;
    while (chunk > 1 && chunk * affine_token_bytes<WIDTH>(K) > 53 * 1024) chunk /= 2;
    return chunk;
}
// Whether the matrix cores take rows of this format: whole half steps, affine groups of 64, Q8 only where its blocks have eight elements, and
// four tokens' rows that leave room for two workgroups on a compute unit, and offsets in the codes of 32 bits.
template <int BITS, int WIDTH> static bool matrix_fits(uint32_t K, uint32_t N, uint32_t group) {
    if constexpr (BITS == 8 && WIDTH == 4) return false;
    else return group == 64 && uint64_t(K) * N / 8 * BITS < 1ull << 32 && K % (16 * WIDTH) == 0 && MatrixForm<BITS, WIDTH>::steps(K) <= kMatrixSteps && matrix_staged_bytes<BITS, WIDTH>(K) <= 80 * 1024;
}
// Workgroups of a launch: as many as fit the chip at once (LDS, and four waves a SIMD by registers), not more than there can be rounds.
static uint32_t matrix_grid(uint32_t lds, uint32_t tiles, uint64_t jobs) {
    return uint32_t(std::min<uint64_t>(256 * matrix_per_cu(lds), (tiles + kMatrixWaves - 1) / kMatrixWaves * jobs));
}
uint32_t affine_job_tokens(uint32_t K, uint32_t N, uint32_t group, uint32_t bits, bool matrix) {
    uint32_t chunk = 1;
    by_format<false>(bits, wide(K, N), [&]<int BITS, int WIDTH, bool GATED>() { chunk = matrix && matrix_fits<BITS, WIDTH>(K, N, group) ? kMatrixTokens : affine_chunk<WIDTH>(K); });
    return chunk;
}
bool affine_job_images(uint32_t chunk) { return chunk > kAffineTokens; }
// (A grid's y holds fewer than 2^16 workgroups: the rest of a longer list goes to z.)
static dim3 affine_grid(uint32_t x, uint32_t jobs) { const uint32_t y = std::min(jobs, 32768u); return dim3(x, y, (jobs + y - 1) / y); }

// Tokens from which the operators' products go to the matrix cores: a call of few tokens is a chain of latencies, longer there by the images' making
// and a barrier.  us a call, lanes -> matrix cores: gate/up at 16, 32, 48 and 128 rows, hidden 2048 7.5 -> 9.1, 9.9 -> 9.2, 13.2 -> 11.2, 24 -> 17;
// 2560 9.7 -> 10.4, 12.5 -> 13.2, 18 -> 13, 34 -> 27; 3072 12.7 -> 12.1, 21 -> 15, 28 -> 20, 57 -> 31.  Down at 32, 48, 96 and 128: 8.6 -> 6.7, 11.1 -> 7.6,
// 14.4 -> 12.1, 15.5 -> 12.0; 10.9 -> 10.4, 14.9 -> 12.4, 22 -> 18, 27 -> 22; 13.7 -> 11.9, 15.7 -> 20.2, 25.2 -> 26.2, 32 -> 26.
// Q8: gate/up at 48, 64 and 128, 2048 x 512 14.7 -> 13.9, 18.9 -> 14.2, 30 -> 23; 3072 x 1024 at 48 and 128 33 -> 24, 71 -> 53; down at 128
// and 192, 512 x 2048 16.8 -> 12.4, 22.6 -> 18.3; 1024 x 3072 37 -> 26, 52 -> 39.  Q4 rows of half steps: gate/up at 48 and 128, 640 x 2560 25.6 -> 15.2, 56 -> 27;
// 1920 x 640 18.4 -> 12.6, 36 -> 28; down at 128, 640 x 2560 26.8 -> 17.5, 1920 x 2560 59 -> 37.
// (All of it, and the figures below, with the matrix cores' side as it was before MatrixPace and the slots in place, which took up to a sixth off
// an expert phase of 32 to 64 tokens: the lines may lie a little high.)
constexpr uint32_t kMatrixFrom[2] = {128, 48};   // plain, gate/up
// And from a wave a SIMD on (two where a matrix has less than a workgroup's tiles), since with fewer the call lasts as long as one workgroup's chain,
// which is longer there.  Gate/up with 512, 768, 1024 and 2048 waves: 2048 x 64 7.6 -> 10.0, 9.0 -> 9.9, 10.4 -> 10.1, 17.4 -> 12.8; down 2048 x 128 7.2 -> 9.6, 8.5 ->
// 9.6, 9.7 -> 9.8, 16.4 -> 12.3; gate/up 4096 x 8 11.2 -> 15.7 at 512 and 16.4 -> 20.6 at 1024.
constexpr uint64_t kMatrixWavesFrom = 1024;
void launch_affine(hipStream_t s, const AffineDesc& a) {
    AffineJob j{};
    auto matrix = [](const zc_linear& l) { return AffineMatrix{(const uint8_t*)l.weight, (const uint16_t*)l.scales, (const uint16_t*)l.biases}; };
    j.m[0] = matrix(a.gate);
    if (a.gated) j.m[1] = matrix(a.up);
    j.x = a.x; j.in_rows = a.in_rows; j.out_rows = a.out_rows; j.out = a.out;
    j.K = a.gate.input; j.N = a.gate.output; j.group = a.gate.group; j.tokens = a.tokens; j.float_output = a.float_output; j.check = a.check;
    auto go = [&]<int BITS, int WIDTH, bool GATED>() {
        if constexpr (BITS == 4 || WIDTH == 8) {
            using Stream = MatrixStream<BITS, WIDTH, GATED>;
            j.tiles = (j.N + Stream::kTileRows - 1) / Stream::kTileRows;
            const uint64_t jobs = (uint64_t(j.tokens) + kMatrixTokens - 1) / kMatrixTokens;
            if (j.tokens >= kMatrixFrom[GATED] && jobs * j.tiles >= kMatrixWavesFrom * (j.tiles < kMatrixWaves ? 2 : 1) && matrix_fits<BITS, WIDTH>(j.K, j.N, j.group)) {
                j.chunk = kMatrixTokens;
                const uint32_t lds = matrix_lds_bytes<BITS, WIDTH>(j.K), grid = matrix_grid(lds, j.tiles, jobs);
                hipLaunchKernelGGL((affine_matrix_kernel<BITS, WIDTH, GATED>), dim3(grid), dim3(kMatrixThreads), lds, s, j);
                return;
            }
        }
        j.chunk = std::min(affine_chunk<WIDTH>(j.K), j.tokens);
        const uint32_t rows = j.chunk == 1 ? AffineStream<BITS, WIDTH, GATED, 1>::kTileRows : AffineStream<BITS, WIDTH, GATED, kAffineTokens>::kTileRows;
        const uint32_t chunks = (j.tokens + j.chunk - 1) / j.chunk;
        j.tiles = (j.N + rows - 1) / rows; j.share = affine_share(j.tiles, chunks);
        const dim3 grid = affine_grid((j.tiles + j.share - 1) / j.share, chunks);
        const uint32_t lds = j.chunk * affine_token_bytes<WIDTH>(j.K);
        if (j.chunk == 1) hipLaunchKernelGGL((affine_op_kernel<BITS, WIDTH, GATED, 1>), grid, dim3(256), lds, s, j);
        else hipLaunchKernelGGL((affine_op_kernel<BITS, WIDTH, GATED, kAffineTokens>), grid, dim3(256), lds, s, j);
    };
    if (a.gated) by_format<true>(a.gate.bits, wide(j.K, j.N), go);
    else by_format<false>(a.gate.bits, wide(j.K, j.N), go);
}

// Whether one token's gate/up launch makes the picks: every workgroup waits for them, so only while they take less than the launch they replace and
// the gap behind it.  Where there are as many lanes with candidates (eight a lane, up to 512 experts) as picks, they are found together, else
// one by one.  us a layer, a launch of their own -> inside, hidden 2048 and 3072:
//   together: 512 experts, 10, 20, 28 and 48 picks 24 -> 22, 37 -> 36, 45 -> 47, 73 -> 95 and 35 -> 34, 56 -> 56, 68 -> 70, 105 -> 124;
//             256 experts, 16, 20 and 24 picks 33 -> 31, 36 -> 36, 42 -> 42 and 49 -> 49, 56 -> 56, 61 -> 63
//   one by one: 64 experts, 10, 12, 16 and 28 picks 25 -> 24, 31 -> 30, 36 -> 34, 51 -> 58 and 35 -> 34, 42 -> 42, 49 -> 53, 70 -> 86; 1024 experts, 10, 12,
//             16, 28 and 63 picks 28 -> 27, 35 -> 34, 40 -> 40, 60 -> 79, 102 -> 143 and 40 -> 41, 49 -> 50, 57 -> 69, 81 -> 118, 144 -> 180
// (And the selection's words have to fit beside the longest rows, which fill a compute unit's LDS.)
bool expert_phase_routes(uint32_t K, uint32_t E, uint32_t topk) {
    const bool together = E <= 512 && topk <= (E + 7) / 8;
    return topk <= (together ? 20 : 12) && affine_token_bytes<16>(K) + 1024 <= 160 * 1024;
}
void launch_expert_phase(hipStream_t s, const ExpertPhaseDesc& d) {
    ExpertPhase p{};
    p.logits = d.logits; p.ids = d.ids; p.weights = d.weights; p.status = d.status; p.E = d.E;
    p.records = (const uint8_t*)d.records; p.stride = d.stride; p.shared_record = (const uint8_t*)d.shared_record;
    for (int i = 0; i < 6; ++i) { p.off[i] = d.off[i]; p.shared_off[i] = d.shared_off[i]; }
    p.jobs = d.jobs; p.count = d.count; p.slots = d.slots; p.max_jobs = d.max_jobs;
    p.x = d.x; p.out = d.out; p.shared_x = d.shared_x; p.shared_out = d.shared_out; p.fp32 = d.fp32;
    p.K = d.K; p.N = d.N; p.group = d.group; p.topk = d.topk; p.tokens = d.tokens; p.chunk = d.chunk;
    p.shared_jobs = (d.tokens + d.chunk - 1) / d.chunk;
    auto with_shared = [&](auto bits, auto launch) {   // the shared expert's bits as a constant
        if (d.shared_bits == d.bits) launch(bits);
        else launch(std::integral_constant<int, 12 - decltype(bits)::value>{});
    };
    auto go = [&]<int BITS, int WIDTH, bool GATED>() {
        const std::integral_constant<int, BITS> bits;
        if constexpr (BITS == 4 || WIDTH == 8) {
            if (d.chunk > kAffineTokens) {
                with_shared(bits, [&](auto other) {
                    constexpr int SHARED = decltype(other)::value, OTHER = shared_width(BITS, WIDTH, SHARED);
                    if constexpr (SHARED == 4 || OTHER == 8) {   // (the other formats have jobs of fewer tokens)
                        using Stream = MatrixStream<BITS, WIDTH, GATED>;
                        static_assert(Stream::kTileRows == MatrixStream<SHARED, OTHER, GATED>::kTileRows);
                        p.tiles = (p.N + Stream::kTileRows - 1) / Stream::kTileRows;
                        const uint32_t lds = std::max(matrix_lds_bytes<BITS, WIDTH>(d.K), matrix_lds_bytes<SHARED, OTHER>(d.K)), grid = matrix_grid(lds, p.tiles, d.max_jobs + p.shared_jobs);
                        hipLaunchKernelGGL((expert_matrix_kernel<BITS, WIDTH, GATED, SHARED>), dim3(grid), dim3(kMatrixThreads), lds, s, p);
                    }
                });
                return;
            }
        }
        if (d.ids) {
            with_shared(bits, [&](auto other) {
                constexpr int SHARED = decltype(other)::value, OTHER = shared_width(BITS, WIDTH, SHARED);
                constexpr uint32_t rows = AffineStream<BITS, WIDTH, GATED, 1>::kTileRows;
                static_assert(rows == AffineStream<SHARED, OTHER, GATED, 1>::kTileRows);
                p.tiles = (p.N + rows - 1) / rows; p.share = affine_share(p.tiles, d.max_jobs + p.shared_jobs);
                const dim3 grid((p.tiles + p.share - 1) / p.share, d.max_jobs + p.shared_jobs);
                const uint32_t lds = affine_token_bytes<WIDTH>(d.K);
                if constexpr (GATED) {
                    if (expert_phase_routes(d.K, d.E, d.topk)) {
                        if (d.E <= 512) hipLaunchKernelGGL((expert_token_kernel<BITS, WIDTH, true, 8, SHARED>), grid, dim3(256), lds, s, p);
                        else hipLaunchKernelGGL((expert_token_kernel<BITS, WIDTH, true, 16, SHARED>), grid, dim3(256), lds, s, p);
                        return;
                    }
                }
                hipLaunchKernelGGL((expert_token_kernel<BITS, WIDTH, GATED, 0, SHARED>), grid, dim3(256), lds, s, p);
            });
            return;
        }
        const uint32_t most = std::min(d.chunk, d.tokens), lds = most * affine_token_bytes<WIDTH>(d.K);
        const uint32_t rows = most == 1 ? AffineStream<BITS, WIDTH, GATED, 1>::kTileRows : AffineStream<BITS, WIDTH, GATED, kAffineTokens>::kTileRows;
        p.tiles = (p.N + rows - 1) / rows; p.share = affine_share(p.tiles, p.max_jobs + p.shared_jobs);
        const dim3 grid = affine_grid((p.tiles + p.share - 1) / p.share, p.max_jobs + p.shared_jobs);
        if (most == 1) hipLaunchKernelGGL((expert_phase_kernel<BITS, WIDTH, GATED, 1>), grid, dim3(256), lds, s, p);
        else hipLaunchKernelGGL((expert_phase_kernel<BITS, WIDTH, GATED, kAffineTokens>), grid, dim3(256), lds, s, p);
    };
    auto launch = [&](uint32_t bits) {
        if (d.gated) by_format<true>(bits, wide(d.K, d.N), go);
        else by_format<false>(bits, wide(d.K, d.N), go);
    };
    // The lists of the lanes' kernels: a shared expert of the other format has a launch of its own, without routed jobs.
    if (d.shared_bits != d.bits && !d.ids && d.chunk <= kAffineTokens) {
        p.max_jobs = 0;
        launch(d.shared_bits);
        p.max_jobs = d.max_jobs; p.shared_jobs = 0;
    }
    launch(d.bits);
}

// ---------------------------------------------------------------------------
// Plain (unquantised) rows: lane chain k = lane + 32 j (reference: qwen.metal:499-506)
// ---------------------------------------------------------------------------
// Row `row` of w [N][K] times the input row xr, by a group of 32 lanes; the result is in every lane.
__device__ __forceinline__ float plain_dot(const void* __restrict__ w, uint32_t dtype, const float* __restrict__ xr, uint32_t K, uint32_t N, uint32_t row, uint32_t lane) {
    float sum = 0;
    uint32_t k = lane;
    // every element's 32-bit word is aligned and inside the array: a four-byte aligned array with an even number of elements
    const bool even_rows = (reinterpret_cast<uintptr_t>(w) & 3u) == 0 && ((uint64_t(N) * K) & 1u) == 0;
    // `count` loads of each operand in flight; the additions stay in k order.  The weight's type is chosen outside the
    // batch: loads on either side of a branch would each be waited for where the sides join.
    auto batch = [&](auto count, auto kind) {
        constexpr int kLoads = decltype(count)::value, kKind = decltype(kind)::value;
        float xv[kLoads], wv[kLoads];
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            xv[j] = xr[k + 32 * j];
            const uint64_t at = uint64_t(row) * K + k + 32 * j;
            if constexpr (kKind == 0) wv[j] = reinterpret_cast<const float*>(w)[at];
            else if constexpr (kKind == 1) {   // a BF16 weight from the aligned 32-bit word that holds it
                const uint32_t word = reinterpret_cast<const uint32_t*>(w)[at >> 1];
                wv[j] = __uint_as_float((at & 1) ? (word & 0xffff0000u) : (word << 16));
            } else wv[j] = b16(reinterpret_cast<const uint16_t*>(w)[at]);
        }
#pragma unroll
        for (int j = 0; j < kLoads; ++j) sum += xv[j] * wv[j];
        k += kLoads * 32;
    };
    auto batches = [&](auto kind) {   // a row is one memory latency per batch: long rows take thirty-two loads at a time
        while (k + 31 * 32 < K) batch(std::integral_constant<int, 32>{}, kind);
        while (k + 15 * 32 < K) batch(std::integral_constant<int, 16>{}, kind);
        while (k + 7 * 32 < K) batch(std::integral_constant<int, 8>{}, kind);
    };
    if (dtype == 1) batches(std::integral_constant<int, 0>{});
    else if (even_rows) batches(std::integral_constant<int, 1>{});
    else batches(std::integral_constant<int, 2>{});
    for (; k < K; k += 32) {
        const float wv = dtype == 1 ? reinterpret_cast<const float*>(w)[uint64_t(row) * K + k]
                                    : b16(reinterpret_cast<const uint16_t*>(w)[uint64_t(row) * K + k]);
        sum += xr[k] * wv;
    }
    return lane_sum32(sum);
}
__global__ __launch_bounds__(256) void plain_kernel(const void* __restrict__ w, uint32_t dtype, const float* __restrict__ x, uint32_t K,
                                                    uint32_t N, uint32_t tokens, float* __restrict__ out, uint32_t float_output) {
    // one 32-lane group per (token, row) pair, eight pairs per workgroup whatever N is (a single row keeps all groups busy)
    const uint32_t lane = threadIdx.x & 31u;
    const uint64_t pair = uint64_t(blockIdx.x) * 8 + (threadIdx.x >> 5);
    if (pair >= uint64_t(N) * tokens) return;
    const uint32_t row = uint32_t(pair % N), t = uint32_t(pair / N);
    const float sum = plain_dot(w, dtype, x + uint64_t(t) * K, K, N, row, lane);
    if (lane == 0) out[uint64_t(t) * N + row] = float_output ? sum : bf(sum);
}
void launch_plain(hipStream_t s, const void* w, uint32_t dtype, const float* x, uint32_t K, uint32_t N,
                  uint32_t tokens, float* out, bool float_output) {
    const uint64_t pairs = uint64_t(N) * tokens;
    hipLaunchKernelGGL(plain_kernel, dim3(uint32_t((pairs + 7) / 8)), dim3(256), 0, s, w, dtype, x, K, N, tokens, out,
                       uint32_t(float_output));
}

// ---------------------------------------------------------------------------
// Router logits (reference: qwen.metal:512-534, metal.mm:818-822): sixteen contiguous
// K partitions, a k-ascending multiply-accumulate chain in each, partials added 0..15.
// One lane owns one (expert, partition) chain for TT tokens.
// ---------------------------------------------------------------------------
template <int TT>
__global__ __launch_bounds__(256) void router_kernel(const uint16_t* w, const float* x, uint32_t T, uint32_t K,
                                                     uint32_t E, const float* offsets, float* out) {
    const uint32_t e = blockIdx.x * 16 + threadIdx.x / 16, split = threadIdx.x % 16, t0 = blockIdx.y * TT;
    const uint32_t P = K / 16;
    float c[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) c[t] = 0;
    if (e < E) {
        const uint16_t* wr = w + uint64_t(e) * K + split * P;
        if (P % 8 == 0) {
            for (uint32_t i = 0; i < P; i += 8) {
                const uint4 wv = *reinterpret_cast<const uint4*>(wr + i);
                const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const uint32_t tt = t0 + t < T ? t0 + t : T - 1;
                    const float* xr = x + uint64_t(tt) * K + split * P + i;
                    const float4 a = *reinterpret_cast<const float4*>(xr), b = *reinterpret_cast<const float4*>(xr + 4);
                    const float xv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        c[t] = __builtin_fmaf(xv[k], __uint_as_float((k & 1) ? (ww[k / 2] & 0xffff0000u) : (ww[k / 2] << 16)), c[t]);
                }
            }
        } else {
            for (uint32_t i = 0; i < P; ++i)
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const uint32_t tt = t0 + t < T ? t0 + t : T - 1;
                    c[t] = __builtin_fmaf(x[uint64_t(tt) * K + split * P + i], b16(wr[i]), c[t]);
                }
        }
    }
    const uint32_t base = (threadIdx.x & 63u) & ~15u;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        float sum = 0;
        for (uint32_t sidx = 0; sidx < 16; ++sidx) sum += __shfl(c[t], base + sidx);
        if (split == 0 && e < E && t0 + t < T) out[uint64_t(t0 + t) * E + e] = offsets ? sum + offsets[e] : sum;
    }
}
// The same chains for short batches of rows that are a multiple of 128 long.  A chain is P = K / 16 dependent multiply-adds
// and the rest is latency: a lane's next 64 weights are requested before the current ones are used, the first before the input
// rows are staged in LDS, twelve loads a thread in flight (one padded piece per partition, so that the partitions' reads meet different
// banks).  A workgroup has four experts per wave and up to four tokens.  The workgroups behind the last expert's, if gate_w is not null, form
// the shared gate's plain dots of their tokens: a launch less, and its latency beside the logits'.
// Several tokens go to the matrix cores: a v_mfma_f32_4x4x1_16b_f32 is one fused multiply-add for each of sixteen partitions, four
// tokens and four experts, rounded as the chains' own.  Lane (partition, j) brings one input of token j and one weight of
// expert j, a quarter of the reads of LDS that a lane with four tokens' chains needs, and half the time on the vector unit.
// 512 experts: one token of 2048 inputs 5.0 us, of 2560 6.5; on the vector unit, with the staging's loads waited for one by one, -> here:
// 5 tokens of 2048 8.4 -> 5.8, 8 of 3072 11.4 -> 7.4, 40 of 2560 15.3 -> 12.3, 64 of 3072 19.2 -> 15.9.
template <uint32_t TOKENS, uint32_t BATCH>   // BATCH: sixteen-byte pieces of a row that a thread requests at once
__global__ __launch_bounds__(256) void router_short_kernel(const uint16_t* __restrict__ w, const float* __restrict__ x, uint32_t T, uint32_t K, uint32_t E,
                                                            const float* __restrict__ offsets, float* __restrict__ out, const void* __restrict__ gate_w, float* __restrict__ gate,
                                                            int32_t* status, uint32_t rows) {   // rows: tokens of a workgroup, at most TOKENS
    extern __shared__ __align__(16) float router_x[];   // [rows][16][P + 4], then the waves' partial sums: [4 * TOKENS][17]
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, j = lane & 3u, split = lane >> 2, experts = blockDim.x / 16, t0 = blockIdx.y * rows, P = K / 16, pitch = P + 4;
    const uint32_t nt = min(T - t0, rows);
    if (blockIdx.x * experts >= E) {
        for (uint32_t t = tid >> 5; t < nt; t += blockDim.x >> 5) {
            const float sum = plain_dot(gate_w, 0, x + uint64_t(t0 + t) * K, K, 1, 0, tid & 31u);
            if ((tid & 31u) == 0) gate[t0 + t] = bf(sum);
        }
        return;
    }
    const uint32_t e0 = blockIdx.x * experts + wave * 4;
    const uint16_t* wr = w + uint64_t(min(e0 + j, E - 1)) * K + split * P;
    uint4 ahead[8];
    auto request = [&](uint32_t i0) {
#pragma unroll
        for (int q = 0; q < 8; ++q) ahead[q] = ldg_u4(wr + min(i0 + 8 * uint32_t(q), P - 8));
    };
    request(0);
    uint32_t low = 0;
    for (uint32_t i0 = tid; i0 < K / 4; i0 += BATCH * blockDim.x) {   // (past the end: the last piece again, not used)
        uint4 v[TOKENS][BATCH];
#pragma unroll
        for (uint32_t t = 0; t < TOKENS; ++t)
#pragma unroll
            for (uint32_t u = 0; u < BATCH; ++u) v[t][u] = ldg_u4(x + uint64_t(t0 + min(t, nt - 1)) * K, min(i0 + u * blockDim.x, K / 4 - 1));
#pragma unroll
        for (uint32_t u = 0; u < BATCH; ++u) {
            const uint32_t i = i0 + u * blockDim.x, part = i / (P / 4), at = part * pitch + (i - part * (P / 4)) * 4;
#pragma unroll
            for (uint32_t t = 0; t < TOKENS; ++t) {
                low |= v[t][u].x | v[t][u].y | v[t][u].z | v[t][u].w;
                if (t < nt && i < K / 4) *reinterpret_cast<uint4*>(router_x + t * 16 * pitch + at) = v[t][u];
            }
        }
    }
    if (status && blockIdx.x == 0 && (low & 0xffffu)) atomicOr(status, 4);
    lds_barrier();
    const float* xr = router_x + (min(j, nt - 1) * 16 + split) * pitch;   // (tokens that are not there: the last one again, not used)
    f32x4 c = {0, 0, 0, 0};
    for (uint32_t i0 = 0; i0 < P; i0 += 64) {
        uint4 piece[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) piece[q] = ahead[q];
        if (i0 + 64 < P) request(i0 + 64);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (i0 + 8 * uint32_t(q) >= P) break;
            const uint32_t ww[4] = {piece[q].x, piece[q].y, piece[q].z, piece[q].w};
            const float4 a = *reinterpret_cast<const float4*>(xr + i0 + 8 * q), b = *reinterpret_cast<const float4*>(xr + i0 + 8 * q + 4);
            const float xv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float weight = (k & 1) ? high_bf16(ww[k / 2]) : low_bf16(ww[k / 2]);
                if constexpr (TOKENS == 1) c[0] = __builtin_fmaf(xv[k], weight, c[0]);
                else c = matrix_chain_step(xv[k], weight, c);
            }
        }
    }
    // the partials added 0..15, by lane 4 t + j for token t and expert j
    float* partial = router_x + rows * 16 * pitch + wave * (4 * TOKENS * 17);
#pragma unroll
    for (uint32_t t = 0; t < TOKENS; ++t) partial[(t * 4 + j) * 17 + split] = c[t];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) sum += partial[min(lane, 4 * TOKENS - 1) * 17 + i];
    const uint32_t e = e0 + j;
    if (split < nt && e < E) out[uint64_t(t0 + split) * E + e] = offsets ? sum + offsets[e] : sum;
}
void launch_router(hipStream_t s, const void* w, const float* x, uint32_t T, uint32_t K, uint32_t E,
                   const float* offsets, float* out, const void* gate_w, float* gate, int32_t* status) {
    const auto row_bytes = [&](uint32_t rows) { return size_t(rows) * (K + 64) * 4; };
    const uint32_t rows = T >= 4 ? 4 : T == 3 && row_bytes(3) > kRouterShortLds ? 2 : T;
    static_assert(4 * (kRouterStatusK + 64) * 4 <= kRouterShortLds && kRouterStatusK % 128 == 0);
    if (T <= 64 && K % 128 == 0 && row_bytes(rows) <= kRouterShortLds) {   // (two of its workgroups fit a compute unit's LDS)
        auto grid_of = [&](uint32_t waves) { return dim3((E + 4 * waves - 1) / (4 * waves) + (gate_w ? 1 : 0), (T + rows - 1) / rows); };
        auto lds_of = [&](uint32_t waves) { return row_bytes(rows) + waves * 4 * (T == 1 ? 1 : 4) * 17 * 4; };
        // Two waves spread the experts over more compute units, and stage the tokens' rows twice as often as four: while all workgroups
        // are on the chip at once, by LDS and, at three waves a SIMD, by registers (512 experts, us with one, two and four waves: 8 tokens of 3072 inputs 9.3, 7.4, 9.0, 32 of 2048
        // 12.7, 8.8, 10.6, 40 of 2560 21.4, 12.3, 13.7; 64 of 3072 24.7, 18.2, 15.9).
        const dim3 two = grid_of(2);
        const uint32_t waves = T == 1 ? 1 : two.x * two.y <= 256 * std::min<size_t>(160 * 1024 / lds_of(2), 6) ? 2 : 4;
        const dim3 grid = grid_of(waves);
        const size_t lds = lds_of(waves);
        // (Rows of one piece a thread request no more.  Both: 1024 experts, 64 tokens of 256 and 1024 inputs 8.1 -> 6.3 and 10.2 -> 7.7 us.)
#define ZC_ROUTER(...) hipLaunchKernelGGL((router_short_kernel<__VA_ARGS__>), grid, dim3(64 * waves), lds, s, (const uint16_t*)w, x, T, K, E, offsets, out, gate_w, gate, status, rows)
        if (T == 1) ZC_ROUTER(1, 12);
        else if (K <= 256 * waves) ZC_ROUTER(4, 1);
        else ZC_ROUTER(4, 3);
#undef ZC_ROUTER
        return;
    }
    if (gate_w) launch_plain(s, gate_w, 0, x, K, 1, T, gate, false);
    if (T >= 64 && K % 128 == 0) {
        launch_router_batch(s, w, x, T, K, E, offsets, out);
        return;
    }
    const uint32_t gx = (E + 15) / 16;
    if (T >= 4) hipLaunchKernelGGL(router_kernel<4>, dim3(gx, (T + 3) / 4), dim3(256), 0, s, (const uint16_t*)w, x, T, K, E, offsets, out);
    else hipLaunchKernelGGL(router_kernel<1>, dim3(gx, T), dim3(256), 0, s, (const uint16_t*)w, x, T, K, E, offsets, out);
}

// ---------------------------------------------------------------------------
// Route: top-k by descending value, lowest id on ties, nothing at or below -inf;
// softmax over the selected (reference: qwen.metal:742-795).  One wavefront per token.
// ---------------------------------------------------------------------------
constexpr int kRouteMaxPerLane = 16;   // experts <= 1024
constexpr int kRouteMaxTopK = 128;
__global__ __launch_bounds__(64) void route_kernel(const float* logits, uint32_t T, uint32_t E, uint32_t topk,
                                                   int32_t* ids, float* weights) {
    const uint32_t t = blockIdx.x, lane = threadIdx.x;
    __shared__ float scores[kRouteMaxTopK];
    __shared__ int32_t selected[kRouteMaxTopK];
    const float ninf = __uint_as_float(0xff800000u);
    const float* v = logits + uint64_t(t) * E;
    float cand[kRouteMaxPerLane];
#pragma unroll
    for (int i = 0; i < kRouteMaxPerLane; ++i) {
        const uint32_t e = lane + 64u * i;
        float c = e < E ? v[e] : ninf;
        cand[i] = c > ninf ? c : ninf;   // NaN and -inf never win
    }
    for (uint32_t j = 0; j < topk; ++j) {
        float best = ninf; uint32_t index = 0x7fffffffu;
#pragma unroll
        for (int i = 0; i < kRouteMaxPerLane; ++i) if (cand[i] > best) { best = cand[i]; index = lane + 64u * i; }
        float m = best;
#pragma unroll
        for (int o = 32; o; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        uint32_t winner = (best == m && best > ninf) ? index : 0x7fffffffu;
#pragma unroll
        for (int o = 32; o; o >>= 1) winner = min(winner, uint32_t(__shfl_xor(int(winner), o)));
        if (lane == 0) {
            selected[j] = winner < E ? int32_t(winner) : -1;
            scores[j] = winner < E ? v[winner] : ninf;   // reload keeps signed zero
        }
#pragma unroll
        for (int i = 0; i < kRouteMaxPerLane; ++i) if (lane + 64u * i == winner) cand[i] = ninf;
    }
    __syncthreads();
    // Four values per reference lane, lane sum, one reciprocal.
    float values[4], sum = 0;
    const float top = scores[0];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t j = lane * 4 + i;
        values[i] = (lane < 32 && j < topk) ? exp32(scores[j] - top) : 0.0f;
        sum += values[i];
    }
    const float inverse = 1.0f / lane_sum32(sum);
    if (lane < 32)
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t j = lane * 4 + i;
            if (j < topk) { ids[uint64_t(t) * topk + j] = selected[j]; weights[uint64_t(t) * topk + j] = values[i] * inverse; }
        }
}
// The same by route_token (at most 64 picks): candidates by a binary search over the lanes' maxima instead of one reduction
// through LDS per pick.  512 experts, top-10: 10.4 -> 4.7 us.
template <int PER>
__global__ __launch_bounds__(64) void route_fast_kernel(const float* __restrict__ logits, uint32_t E, uint32_t topk, int32_t* __restrict__ ids, float* __restrict__ weights) {
    __shared__ int32_t ids_s[64];
    __shared__ float weights_s[64];
    __shared__ uint32_t pick[128];
    const uint32_t t = blockIdx.x, lane = threadIdx.x;
    const float* row = logits + uint64_t(t) * E;
    route_token<PER>([&](float (&cand)[PER], uint32_t per) {
#pragma unroll
        for (int i = 0; i < PER; ++i) { const uint32_t e = lane * per + uint32_t(i); cand[i] = (uint32_t(i) < per && e < E) ? row[e] : __uint_as_float(0xff800000u); }
    }, E, topk, lane, ids_s, weights_s, pick, [] {}, [] {});
    __syncthreads();
    if (lane < topk) { ids[uint64_t(t) * topk + lane] = ids_s[lane]; weights[uint64_t(t) * topk + lane] = weights_s[lane]; }
}
void launch_route(hipStream_t s, const float* logits, uint32_t T, uint32_t E, uint32_t topk, int32_t* ids, float* weights) {
    if (topk <= 64) {
        if (E <= 512) hipLaunchKernelGGL(route_fast_kernel<8>, dim3(T), dim3(64), 0, s, logits, E, topk, ids, weights);
        else hipLaunchKernelGGL(route_fast_kernel<16>, dim3(T), dim3(64), 0, s, logits, E, topk, ids, weights);
        return;
    }
    hipLaunchKernelGGL(route_kernel, dim3(T), dim3(64), 0, s, logits, T, E, topk, ids, weights);
}

// ---------------------------------------------------------------------------
// Dispatch: stable counting sort of the flat slots p = t*topk + k by expert id
// (reference: model.cpp:449-479).  Up to 1024 slots and experts: one workgroup, thread p owns slot p and then expert p.  A
// slot's place among its wave's slots of the same expert comes from ten ballots over the id's bits, the waves' counts of
// every expert from a table in LDS, without any atomics; two scans over the experts give the rest.  (A wavefront per
// expert that scanned the whole id array took 14.4 us for 10 slots and 66 us for 400; this takes 5.8 us, the selection
// included, and 4.8 us.)
//
// jobs, optional: the list of (expert, sorted positions) that the expert kernels walk, at most `chunk` (up to four) positions of one
// expert each: first position | expert << 20 | (positions - 1) << 30 (a call has at most 2^20 slots).  `count` then is its
// length; else `selected` lists the experts that have slots and `count` is their number.
//
// ROUTE: tokens <= 16, and wave t first selects token t's experts (route_token) instead of reading `ids`: one launch less.
// ---------------------------------------------------------------------------
struct Dispatch {
    int32_t *offsets, *slots, *rows, *selected; uint32_t* jobs; int32_t *count, *status;
    uint32_t topk, E, chunk;
};
__device__ __forceinline__ uint32_t dispatch_job(uint32_t first, uint32_t expert, uint32_t positions) { return first | expert << 20 | (positions - 1) << 30; }
// The rows whose images the same launch leaves for the matrix cores, a workgroup a row (rows: 0 if none are wanted).
struct RowImages { const float* x; float* out; uint32_t rows, K; };
__global__ __launch_bounds__(256) void row_images_kernel(RowImages images) { matrix_image_row(images.x, images.out, blockIdx.x, images.K); }
constexpr uint32_t kDispatchSlots = 1024, kRouteTokens = 16;
template <bool ROUTE, int PER>
__global__ __launch_bounds__(1024) void dispatch_short_kernel(const float* __restrict__ logits, int32_t* __restrict__ ids, float* __restrict__ weights, uint32_t n, Dispatch d, RowImages images) {
    if (blockIdx.x) { matrix_image_row(images.x, images.out, blockIdx.x - 1, images.K); return; }
    __shared__ uint32_t table[16 * 512];           // [wave][expert] counts, two experts a word
    __shared__ uint32_t start[1024], wave_total[2][16];
    __shared__ uint16_t held[1024];
    __shared__ int32_t ids_s[ROUTE ? 1024 : 1];
    __shared__ float weights_s[ROUTE ? 1024 : 1];
    __shared__ uint32_t pick[ROUTE ? kRouteTokens * 128 : 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, waves = (n + 63) / 64, E = d.E;
    uint16_t* counts = reinterpret_cast<uint16_t*>(table);
    for (uint32_t i = tid; i < waves * 512; i += 1024) table[i] = 0;
    int32_t id = -1;
    if constexpr (ROUTE) {
        if (wave < n / d.topk) {
            const float* row = logits + uint64_t(wave) * E;
            route_token<PER>([&](float (&cand)[PER], uint32_t per) {
#pragma unroll
                for (int i = 0; i < PER; ++i) { const uint32_t e = lane * per + uint32_t(i); cand[i] = (uint32_t(i) < per && e < E) ? row[e] : __uint_as_float(0xff800000u); }
            }, E, d.topk, lane, ids_s + wave * d.topk, weights_s + wave * d.topk, pick + wave * 128, [] {}, [] {});
        }
        __syncthreads();
        if (tid < n) { id = ids_s[tid]; ids[tid] = id; weights[tid] = weights_s[tid]; }
    } else {
        if (tid < n) id = ids[tid];
        __syncthreads();
    }
    if (tid < n && (id < 0 || id >= int32_t(E))) { atomicOr(d.status, 1); id = -1; }
    // the wave's lanes with this lane's id
    uint64_t same = __ballot(id >= 0);
#pragma unroll
    for (int b = 0; b < 10; ++b) { const uint64_t m = __ballot((id >> b) & 1); same &= ((id >> b) & 1) ? m : ~m; }
    uint32_t rank = uint32_t(__popcll(same & ((1ull << lane) - 1)));
    if (id >= 0 && rank == 0) counts[wave * 1024 + uint32_t(id)] = uint16_t(__popcll(same));
    __syncthreads();
    // thread e: expert e's slots of earlier waves, their sum, and the scans over the experts (sums of at most 1024 each: two in a word)
    uint32_t total = 0;
    if (tid < E)
        for (uint32_t w = 0; w < waves; ++w) { const uint32_t c = counts[w * 1024 + tid]; counts[w * 1024 + tid] = uint16_t(total); total += c; }
    const uint32_t mine[2] = {total | (d.jobs ? (total + d.chunk - 1) / d.chunk : 0u) << 16, total ? 1u : 0u};
    uint32_t incl[2] = {mine[0], mine[1]};
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
        for (int v = 0; v < 2; ++v) { const uint32_t up = __shfl_up(incl[v], o); if (int(lane) >= o) incl[v] += up; }
    if (lane == 63) { wave_total[0][wave] = incl[0]; wave_total[1][wave] = incl[1]; }
    __syncthreads();
    uint32_t before[2] = {incl[0] - mine[0], incl[1] - mine[1]};
    for (uint32_t w = 0; w < wave; ++w) { before[0] += wave_total[0][w]; before[1] += wave_total[1][w]; }
    start[tid] = before[0]; held[tid] = uint16_t(total);
    if (tid < E) d.offsets[tid] = int32_t(before[0] & 0xffffu);
    if (tid < E && total && d.selected) d.selected[before[1]] = int32_t(tid);
    if (tid == 1023) { d.offsets[E] = int32_t((before[0] + mine[0]) & 0xffffu); *d.count = int32_t(d.jobs ? (before[0] + mine[0]) >> 16 : before[1] + mine[1]); }
    __syncthreads();
    if (id < 0) return;
    rank += counts[wave * 1024 + uint32_t(id)];
    const uint32_t first = start[id], at = (first & 0xffffu) + rank;
    d.slots[at] = int32_t(tid);
    if (d.rows) d.rows[at] = int32_t(tid / d.topk);
    if (d.jobs && rank % d.chunk == 0) d.jobs[(first >> 16) + rank / d.chunk] = dispatch_job(at, uint32_t(id), min(d.chunk, uint32_t(held[id]) - rank));
}
// More than 1024 experts (up to 8192): each wavefront owns experts e = wave, wave+16, ... and scans the id array in order.
__global__ __launch_bounds__(1024) void dispatch_kernel(const int32_t* ids, uint32_t n, uint32_t topk, uint32_t E,
                                                        int32_t* offsets, int32_t* slots, int32_t* rows,
                                                        int32_t* selected, int32_t* count, int32_t* status) {
    extern __shared__ int32_t cnt[];   // E + 1
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, waves = blockDim.x >> 6;
    int bad = 0;
    for (uint32_t p = tid; p < n; p += blockDim.x) bad |= (ids[p] < 0 || ids[p] >= int32_t(E));
    bad = __syncthreads_or(bad);
    if (tid == 0 && bad) atomicOr(status, 1);
    for (uint32_t e = wave; e < E; e += waves) {
        int32_t c = 0;
        for (uint32_t p0 = 0; p0 < n; p0 += 64) {
            const uint32_t p = p0 + lane;
            c += __popcll(__ballot(p < n && ids[p] == int32_t(e)));
        }
        if (lane == 0) cnt[e] = c;
    }
    __syncthreads();
    if (wave == 0) {
        int32_t running = 0, picked = 0;
        if (lane == 0) offsets[0] = 0;
        for (uint32_t base = 0; base < E; base += 64) {
            const uint32_t e = base + lane;
            const int32_t c = e < E ? cnt[e] : 0;
            int32_t incl = c;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) { const int32_t up = __shfl_up(incl, o); if (int(lane) >= o) incl += up; }
            if (e < E) offsets[e + 1] = running + incl;
            const uint64_t mask = __ballot(c > 0);
            if (c > 0) selected[picked + __popcll(mask & ((1ull << lane) - 1))] = int32_t(e);
            picked += __popcll(mask);
            running += __shfl(incl, 63);
        }
        if (lane == 0) *count = picked;
    }
    __syncthreads();
    __threadfence_block();
    for (uint32_t e = wave; e < E; e += waves) {
        int32_t pos = offsets[e];
        if (cnt[e] == 0) continue;
        for (uint32_t p0 = 0; p0 < n; p0 += 64) {
            const uint32_t p = p0 + lane;
            const bool m = p < n && ids[p] == int32_t(e);
            const uint64_t mask = __ballot(m);
            if (m) { const int32_t at = pos + __popcll(mask & ((1ull << lane) - 1)); slots[at] = int32_t(p); if (rows) rows[at] = int32_t(p / topk); }
            pos += __popcll(mask);
        }
    }
}
// The same sort for many slots (prefill), spread over the device: one wavefront per expert counts, one workgroup
// scans, one wavefront per expert places.  offsets[1 + e] doubles as the count array between the first two steps.
__global__ __launch_bounds__(256) void dispatch_count_kernel(const int32_t* __restrict__ ids, uint32_t n, uint32_t E, int32_t* __restrict__ offsets, int32_t* status, bool aligned) {
    const uint32_t lane = threadIdx.x & 63u, e = blockIdx.x * 4 + (threadIdx.x >> 6);
    {   // every workgroup checks its share of the ids (one workgroup doing all of them was the longest-running one)
        int bad = 0;
        for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) { const int32_t id = ids[p]; bad |= (id < 0 || id >= int32_t(E)); }
        if (bad) atomicOr(status, 1);
    }
    if (e >= E) return;
    int32_t c = 0;
    uint32_t p0 = 0;
    if (aligned && n >= 8 * 256) {   // eight steps' loads in flight, the next eight requested before these are counted
        int4 v[8], w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const int4*>(ids + j * 256 + 4 * lane);
        for (; p0 + 8 * 256 <= n; p0 += 8 * 256) {
            const uint32_t following = p0 + 16 * 256 <= n ? p0 + 8 * 256 : p0;   // none left: the same batch again, not counted
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = *reinterpret_cast<const int4*>(ids + following + j * 256 + 4 * lane);
#pragma unroll
            for (int j = 0; j < 8; ++j) c += (v[j].x == int32_t(e)) + (v[j].y == int32_t(e)) + (v[j].z == int32_t(e)) + (v[j].w == int32_t(e));
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = w[j];
        }
    }
    for (; p0 < n; p0 += 256) {   // a lane looks at four neighbouring slots per step
        const uint32_t p = p0 + 4 * lane;
        int4 v = make_int4(-1, -1, -1, -1);
        if (aligned && p + 3 < n) v = *reinterpret_cast<const int4*>(ids + p);   // sixteen-byte loads only from a sixteen-byte aligned array
        else { if (p < n) v.x = ids[p]; if (p + 1 < n) v.y = ids[p + 1]; if (p + 2 < n) v.z = ids[p + 2]; if (p + 3 < n) v.w = ids[p + 3]; }
        c += (v.x == int32_t(e)) + (v.y == int32_t(e)) + (v.z == int32_t(e)) + (v.w == int32_t(e));
    }
#pragma unroll
    for (int o = 32; o; o >>= 1) c += __shfl_xor(c, o);
    if (lane == 0) offsets[1 + e] = c;
}
// chunk: 0, or the jobs' positions; `selected` then receives every expert's first job, count the number of jobs.
__global__ __launch_bounds__(64) void dispatch_scan_kernel(uint32_t E, uint32_t chunk, int32_t* offsets, int32_t* selected, int32_t* count) {
    const uint32_t lane = threadIdx.x;
    int32_t running = 0, picked = 0;
    if (lane == 0) offsets[0] = 0;
    for (uint32_t base = 0; base < E; base += 64) {
        const uint32_t e = base + lane;
        const int32_t c = e < E ? offsets[1 + e] : 0;
        int32_t incl = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const int32_t up = __shfl_up(incl, o); if (int(lane) >= o) incl += up; }
        if (e < E) offsets[e + 1] = running + incl;
        if (chunk) {
            const int32_t jobs = (c + int32_t(chunk) - 1) / int32_t(chunk);
            int32_t before = jobs;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) { const int32_t up = __shfl_up(before, o); if (int(lane) >= o) before += up; }
            if (e < E) selected[e] = picked + before - jobs;
            picked += __shfl(before, 63);
            running += __shfl(incl, 63);
            continue;
        }
        const uint64_t mask = __ballot(c > 0);
        if (c > 0) selected[picked + __popcll(mask & ((1ull << lane) - 1))] = int32_t(e);
        picked += __popcll(mask);
        running += __shfl(incl, 63);
    }
    if (lane == 0) *count = picked;
}
__global__ __launch_bounds__(256) void dispatch_place_kernel(const int32_t* __restrict__ ids, uint32_t n, uint32_t topk, uint32_t E, const int32_t* __restrict__ offsets,
                                                             int32_t* __restrict__ slots, int32_t* __restrict__ rows, bool aligned,
                                                             uint32_t chunk, const int32_t* __restrict__ first_job, uint32_t* __restrict__ jobs) {
    const uint32_t lane = threadIdx.x & 63u, e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= E) return;
    int32_t pos = offsets[e];
    if (offsets[e + 1] == pos) return;
    if (jobs)
        for (uint32_t at = lane * chunk, held = uint32_t(offsets[e + 1] - pos); at < held; at += 64 * chunk)
            jobs[uint32_t(first_job[e]) + at / chunk] = dispatch_job(uint32_t(pos) + at, e, min(chunk, held - at));
    const uint64_t below = (1ull << lane) - 1;
    // eight steps of 256 slots, in order: four neighbouring slots per lane, slots of lower lanes first, then the lane's own
    auto place = [&](const int4 (&batch)[8], uint32_t q0) {
#pragma unroll
        for (int step = 0; step < 8; ++step) {
            if (q0 + step * 256 >= n) break;
            const uint32_t p = q0 + step * 256 + 4 * lane;
            const int4 v = batch[step];
            const bool m[4] = {v.x == int32_t(e), v.y == int32_t(e), v.z == int32_t(e), v.w == int32_t(e)};
            const uint64_t mask[4] = {__ballot(m[0]), __ballot(m[1]), __ballot(m[2]), __ballot(m[3])};
            if ((mask[0] | mask[1] | mask[2] | mask[3]) == 0) continue;   // uniform: none of these 256 slots is the expert's
            int32_t at = pos + __popcll(mask[0] & below) + __popcll(mask[1] & below) + __popcll(mask[2] & below) + __popcll(mask[3] & below);
            uint32_t token = p / topk, rest = p % topk;   // one division per step, not one per slot
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (m[j]) { slots[at] = int32_t(p + j); if (rows) rows[at] = int32_t(token); ++at; }
                if (++rest == topk) { rest = 0; ++token; }
            }
            pos += __popcll(mask[0]) + __popcll(mask[1]) + __popcll(mask[2]) + __popcll(mask[3]);
        }
    };
    uint32_t q0 = 0;
    if (aligned && n >= 8 * 256) {   // whole batches: the next batch is requested before this one is placed
        int4 ahead[8], next[8];
#pragma unroll
        for (int step = 0; step < 8; ++step) ahead[step] = *reinterpret_cast<const int4*>(ids + step * 256 + 4 * lane);
        for (; q0 + 8 * 256 <= n; q0 += 8 * 256) {
            const uint32_t following = q0 + 16 * 256 <= n ? q0 + 8 * 256 : q0;   // none left: the same batch again, not placed
#pragma unroll
            for (int step = 0; step < 8; ++step) next[step] = *reinterpret_cast<const int4*>(ids + following + step * 256 + 4 * lane);
            place(ahead, q0);
#pragma unroll
            for (int step = 0; step < 8; ++step) ahead[step] = next[step];
        }
    }
    for (; q0 < n; q0 += 8 * 256) {   // the ragged end, or an array that is not sixteen-byte aligned
        int4 ahead[8];
#pragma unroll
        for (int step = 0; step < 8; ++step) {
            const uint32_t p = q0 + step * 256 + 4 * lane;
            int4 v = make_int4(-1, -1, -1, -1);
            if (aligned && p + 3 < n) v = *reinterpret_cast<const int4*>(ids + p);   // sixteen-byte loads only from a sixteen-byte aligned array
            else { if (p < n) v.x = ids[p]; if (p + 1 < n) v.y = ids[p + 1]; if (p + 2 < n) v.z = ids[p + 2]; if (p + 3 < n) v.w = ids[p + 3]; }
            ahead[step] = v;
        }
        place(ahead, q0);
    }
}
static void launch_dispatch_any(hipStream_t s, const int32_t* ids, uint32_t n, const Dispatch& d, const RowImages& images) {
    if (n <= kDispatchSlots && d.E <= 1024) {
        hipLaunchKernelGGL((dispatch_short_kernel<false, 8>), dim3(1 + images.rows), dim3(1024), 0, s, nullptr, const_cast<int32_t*>(ids), nullptr, n, d, images);
        return;
    }
    if (images.rows) hipLaunchKernelGGL(row_images_kernel, dim3(images.rows), dim3(256), 0, s, images);
    if (n <= kDispatchSlots && !d.jobs) {
        hipLaunchKernelGGL(dispatch_kernel, dim3(1), dim3(1024), size_t(d.E + 1) * 4, s, ids, n, d.topk, d.E, d.offsets, d.slots, d.rows, d.selected, d.count, d.status);
        return;
    }
    const bool aligned = reinterpret_cast<uintptr_t>(ids) % 16 == 0;
    const uint32_t chunk = d.jobs ? d.chunk : 0;
    hipLaunchKernelGGL(dispatch_count_kernel, dim3((d.E + 3) / 4), dim3(256), 0, s, ids, n, d.E, d.offsets, d.status, aligned);
    hipLaunchKernelGGL(dispatch_scan_kernel, dim3(1), dim3(64), 0, s, d.E, chunk, d.offsets, d.selected, d.count);
    hipLaunchKernelGGL(dispatch_place_kernel, dim3((d.E + 3) / 4), dim3(256), 0, s, ids, n, d.topk, d.E, d.offsets, d.slots, d.rows, aligned, chunk, d.selected, d.jobs);
}
void launch_dispatch(hipStream_t s, const int32_t* ids, uint32_t tokens, uint32_t topk, uint32_t E, int32_t* offsets,
                     int32_t* slots, int32_t* rows, int32_t* selected, int32_t* count, int32_t* status) {
    launch_dispatch_any(s, ids, tokens * topk, Dispatch{offsets, slots, rows, selected, nullptr, count, status, topk, E, 0}, RowImages{});
}
// Routes, dispatch sort and the expert kernels' job list (E <= 1024; scratch: E words).
void launch_route_jobs(hipStream_t s, const float* logits, uint32_t tokens, uint32_t E, uint32_t topk, int32_t* ids, float* weights,
                       int32_t* offsets, int32_t* slots, uint32_t chunk, uint32_t* jobs, int32_t* count, int32_t* scratch, int32_t* status,
                       const float* x, uint32_t K, float* row_images) {
    const uint32_t n = tokens * topk;
    const RowImages images{x, row_images, row_images ? tokens : 0, K};
    Dispatch d{offsets, slots, nullptr, scratch, jobs, count, status, topk, E, chunk};
    if (n <= kDispatchSlots) d.selected = nullptr;
    if (tokens <= kRouteTokens && topk <= 64) {   // (n <= 1024)
        if (E <= 512) hipLaunchKernelGGL((dispatch_short_kernel<true, 8>), dim3(1 + images.rows), dim3(1024), 0, s, logits, ids, weights, n, d, images);
        else hipLaunchKernelGGL((dispatch_short_kernel<true, 16>), dim3(1 + images.rows), dim3(1024), 0, s, logits, ids, weights, n, d, images);
        return;
    }
    launch_route(s, logits, tokens, E, topk, ids, weights);
    launch_dispatch_any(s, ids, n, d, images);
}

// ---------------------------------------------------------------------------
// scatter_experts, moe_sum (reference: qwen.metal:800-816), inter-layer RMS glue
// ---------------------------------------------------------------------------
__global__ void scatter_kernel(const float* x, const int32_t* positions, uint32_t n, uint32_t H, float* out) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
    if (c < H && r < n) out[uint64_t(uint32_t(positions[r])) * H + c] = x[uint64_t(r) * H + c];
}
void launch_scatter(hipStream_t s, const float* x, const int32_t* positions, uint32_t n, uint32_t H, float* out) {
    hipLaunchKernelGGL(scatter_kernel, dim3((H + 255) / 256, n), dim3(256), 0, s, x, positions, n, H, out);
}
// General top-k keeps the reference's eight strided partials: partial j takes
// k = j, j+8, ...; partials are then added 0..7.  top-k 10 is the reference expression.
// V neighbouring columns from column c of token t (one 16-byte load per slot when V is 4); every column keeps the scalar arithmetic.
// HALF: the expert outputs are stored as bf16 (they are BF16 values: the same numbers, half the bytes; V is 4 then).
template <int V, bool HALF>
__device__ __forceinline__ void moe_sum_columns(const void* __restrict__ experts_in, const float* __restrict__ weights, const float* __restrict__ shared,
                                                const float* __restrict__ gate, uint32_t t, uint32_t c, uint32_t H, uint32_t topk, float* y) {
    typedef float row_t __attribute__((ext_vector_type(V)));
    auto row_of = [&](uint64_t slot) {
        if constexpr (HALF) {
            const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(experts_in) + slot * H + c);
            return row_t{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
        } else return *reinterpret_cast<const row_t*>(static_cast<const float*>(experts_in) + slot * H + c);
    };
    row_t partial[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) partial[k] = row_t(0);
    if (topk == 10) {   // the reference's shape: all ten rows requested before the first is used
        row_t value[10]; float weight[10];
#pragma unroll
        for (int k = 0; k < 10; ++k) { value[k] = row_of(uint64_t(t) * 10 + k); weight[k] = weights[uint64_t(t) * 10 + k]; }
#pragma unroll
        for (int k = 0; k < 10; ++k) {
            const row_t product = value[k] * weight[k];
            if (k < 8) partial[k] = product; else partial[k % 8] = partial[k % 8] + product;
        }
    } else
    for (uint32_t k = 0; k < topk; ++k) {
        const row_t product = row_of(uint64_t(t) * topk + k) * weights[uint64_t(t) * topk + k];
        if (k < 8) partial[k] = product; else partial[k % 8] = partial[k % 8] + product;
    }
    row_t sum = partial[0];
    for (uint32_t k = 1; k < 8 && k < topk; ++k) sum += partial[k];
    const float g = bf(sigmoid_bf(gate[t]));
    const row_t sh = *reinterpret_cast<const row_t*>(shared + uint64_t(t) * H + c);
    if constexpr (V == 1) y[0] = bf(bf(sum[0]) + bf(g * sh[0]));
    else {
#pragma unroll
        for (int i = 0; i < V; ++i) y[i] = bf(bf(sum[i]) + bf(g * sh[i]));
    }
}
template <int V, bool HALF = false>
__global__ __launch_bounds__(256) void moe_sum_kernel(const void* __restrict__ experts_in, const float* __restrict__ weights, const float* __restrict__ shared,
                                                      const float* __restrict__ gate, uint32_t T, uint32_t H, uint32_t topk, float* __restrict__ out) {
    const uint32_t c = (blockIdx.x * blockDim.x + threadIdx.x) * V, t = blockIdx.y;
    if (c >= H || t >= T) return;
    typedef float row_t __attribute__((ext_vector_type(V)));
    float y[V];
    moe_sum_columns<V, HALF>(experts_in, weights, shared, gate, t, c, H, topk, y);
    row_t row;
#pragma unroll
    for (int i = 0; i < V; ++i) row[i] = y[i];
    *reinterpret_cast<row_t*>(out + uint64_t(t) * H + c) = row;
}
void launch_moe_sum(hipStream_t s, const float* experts, const float* weights, const float* shared, const float* gate,
                    uint32_t T, uint32_t H, uint32_t topk, float* out) {
    const bool wide = H % 4 == 0 && ((reinterpret_cast<uintptr_t>(experts) | reinterpret_cast<uintptr_t>(shared) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
    if (wide) hipLaunchKernelGGL((moe_sum_kernel<4>), dim3((H / 4 + 255) / 256, T), dim3(256), 0, s, experts, weights, shared, gate, T, H, topk, out);
    else hipLaunchKernelGGL((moe_sum_kernel<1>), dim3((H + 255) / 256, T), dim3(256), 0, s, experts, weights, shared, gate, T, H, topk, out);
}
// The same with the expert outputs as bf16 rows (H a multiple of four, every array sixteen-byte aligned).
void launch_moe_sum_half(hipStream_t s, const uint16_t* experts, const float* weights, const float* shared, const float* gate,
                         uint32_t T, uint32_t H, uint32_t topk, float* out) {
    hipLaunchKernelGGL((moe_sum_kernel<4, true>), dim3((H / 4 + 255) / 256, T), dim3(256), 0, s, experts, weights, shared, gate, T, H, topk, out);
}
// Stand-in glue between stacked layers: x_next = bf(y * (1 / max|y|)) per token.
__device__ __forceinline__ uint32_t glue_magnitude(float y) { const uint32_t a = __float_as_uint(y) & 0x7fffffffu; return a <= 0x7f800000u ? a : 0u; }   // NaN does not take part
template <int WAVES>
__device__ __forceinline__ float glue_factor(uint32_t m, uint32_t* wave_max) {   // m: the largest magnitude of this thread's values
#pragma unroll
    for (int o = 32; o; o >>= 1) m = max(m, uint32_t(__shfl_xor(int(m), o)));
    if ((threadIdx.x & 63u) == 0) wave_max[threadIdx.x >> 6] = m;
    __syncthreads();
    m = wave_max[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) m = max(m, wave_max[w]);
    const float top = __uint_as_float(m);
    return (top > 0.0f && top < __uint_as_float(0x7f800000u)) ? 1.0f / top : 1.0f;
}
__global__ __launch_bounds__(256) void stack_glue_kernel(const float* y, uint32_t H, float* out) {
    __shared__ uint32_t wave_max[4];
    const float* row = y + uint64_t(blockIdx.x) * H;
    uint32_t m = 0;
    for (uint32_t k = threadIdx.x; k < H; k += blockDim.x) m = max(m, glue_magnitude(row[k]));
    const float inv = glue_factor<4>(m, wave_max);
    for (uint32_t k = threadIdx.x; k < H; k += blockDim.x) out[uint64_t(blockIdx.x) * H + k] = bf(row[k] * inv);
}
void launch_stack_glue(hipStream_t s, const float* y, uint32_t T, uint32_t H, float* out) {
    hipLaunchKernelGGL(stack_glue_kernel, dim3(T), dim3(256), 0, s, y, H, out);
}
// The combine and the glue in one launch, a workgroup per token that keeps its row in registers (H a multiple of four up to 4096,
// sixteen-byte aligned arrays); the layer's output itself is written only where `out` is not null.
// One token, hidden 2560: a launch and 2.9 us per layer less than the two kernels one after the other (3.3 and 5.3 us).
__global__ __launch_bounds__(1024) void moe_sum_glue_kernel(const float* __restrict__ experts, const float* __restrict__ weights, const float* __restrict__ shared,
                                                            const float* __restrict__ gate, uint32_t H, uint32_t topk, float* __restrict__ out, float* __restrict__ next) {
    __shared__ uint32_t wave_max[16];
    const uint32_t t = blockIdx.x, c = threadIdx.x * 4;
    float y[4] = {0, 0, 0, 0};
    if (c < H) moe_sum_columns<4, false>(experts, weights, shared, gate, t, c, H, topk, y);
    const float inv = glue_factor<16>(max(max(glue_magnitude(y[0]), glue_magnitude(y[1])), max(glue_magnitude(y[2]), glue_magnitude(y[3]))), wave_max);
    if (c >= H) return;
    if (out) *reinterpret_cast<float4*>(out + uint64_t(t) * H + c) = make_float4(y[0], y[1], y[2], y[3]);
    *reinterpret_cast<float4*>(next + uint64_t(t) * H + c) = make_float4(bf(y[0] * inv), bf(y[1] * inv), bf(y[2] * inv), bf(y[3] * inv));
}
void launch_moe_sum_glue(hipStream_t s, const float* experts, const float* weights, const float* shared, const float* gate,
                         uint32_t T, uint32_t H, uint32_t topk, float* out, float* next) {
    hipLaunchKernelGGL(moe_sum_glue_kernel, dim3(T), dim3(1024), 0, s, experts, weights, shared, gate, H, topk, out, next);
}
bool moe_sum_glue_fits(uint32_t H) { return H % 4 == 0 && H <= 4096; }

// ---------------------------------------------------------------------------
// Counter-based synthetic tensors
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t synth_word(uint64_t seed, uint64_t i) {
    const uint64_t h = hash64(seed, i >> 1);
    return (i & 1) ? uint32_t(h >> 32) : uint32_t(h);
}
__device__ __forceinline__ float synth_scale(uint64_t seed, uint64_t i, float lo, float span) {
    const float u = float(uint32_t(hash64(seed, i) >> 40)) * 5.9604644775390625e-08f;   // 24 bits * 2^-24
    return bf(lo + span * u);
}
// Irwin-Hall(12) on 16-bit fields of three hashes: integer arithmetic, so host and
// device agree exactly; variance (2^32-1)/2^32 of a unit normal, tails cut at 6.
__device__ __forceinline__ float synth_normal(uint64_t seed, uint64_t i, float sigma) {
    int32_t sum = 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const uint64_t h = hash64(seed, 3 * i + j);
        sum += int32_t(h & 0xffff) + int32_t((h >> 16) & 0xffff) + int32_t((h >> 32) & 0xffff) + int32_t(h >> 48);
    }
    return bf(float(2 * sum - 12 * 65535) * 7.62939453125e-06f * sigma);   // * 2^-17
}
__global__ void synth_words_kernel(uint32_t* dst, uint64_t count, uint64_t seed) {
    for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < count; i += uint64_t(gridDim.x) * blockDim.x)
        dst[i] = synth_word(seed, i);
}
__global__ void synth_scales_kernel(uint16_t* scales, uint16_t* biases, uint64_t count, uint64_t seed, float lo, float span, float factor) {
    for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < count; i += uint64_t(gridDim.x) * blockDim.x) {
        const float sc = synth_scale(seed, i, lo, span);
        scales[i] = uint16_t(__float_as_uint(sc) >> 16);
        biases[i] = uint16_t(__float_as_uint(bf(sc * factor)) >> 16);
    }
}
template <bool HALF>
__global__ void synth_normal_kernel(void* dst, uint64_t count, uint64_t seed, float sigma) {
    for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < count; i += uint64_t(gridDim.x) * blockDim.x) {
        const float v = synth_normal(seed, i, sigma);
        if constexpr (HALF) reinterpret_cast<uint16_t*>(dst)[i] = uint16_t(__float_as_uint(v) >> 16);
        else reinterpret_cast<float*>(dst)[i] = v;
    }
}
static dim3 flat_grid(uint64_t count) { return dim3(uint32_t(count / 256 + 1 < 65536 ? count / 256 + 1 : 65536)); }
void launch_synth_words(hipStream_t s, uint32_t* dst, uint64_t count, uint64_t seed) {
    hipLaunchKernelGGL(synth_words_kernel, flat_grid(count), dim3(256), 0, s, dst, count, seed);
}
void launch_synth_scales(hipStream_t s, uint16_t* sc, uint16_t* bi, uint64_t count, uint64_t seed, float lo, float span, float factor) {
    hipLaunchKernelGGL(synth_scales_kernel, flat_grid(count), dim3(256), 0, s, sc, bi, count, seed, lo, span, factor);
}
void launch_synth_normal(hipStream_t s, void* dst, uint64_t count, uint64_t seed, float sigma, bool half) {
    if (half) hipLaunchKernelGGL(synth_normal_kernel<true>, flat_grid(count), dim3(256), 0, s, dst, count, seed, sigma);
    else hipLaunchKernelGGL(synth_normal_kernel<false>, flat_grid(count), dim3(256), 0, s, dst, count, seed, sigma);
}
// Whole records: blockIdx.y = record, grid-stride over the record's dwords.
struct RecordLayout { uint64_t w[3], s[3], words[3], meta[3]; float lo[3], span[3], factor[3]; uint64_t bytes; };
__global__ void synth_records_kernel(uint8_t* records, uint64_t stride, RecordLayout l, uint64_t seed) {
    uint8_t* r = records + uint64_t(blockIdx.y) * stride;
    for (int p = 0; p < 3; ++p) {
        const uint64_t ps = seed + uint64_t(blockIdx.y) * 3 + p;
        uint32_t* w = reinterpret_cast<uint32_t*>(r + l.w[p]);
        for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < l.words[p]; i += uint64_t(gridDim.x) * blockDim.x)
            w[i] = synth_word(ps, i);
        uint16_t* sc = reinterpret_cast<uint16_t*>(r + l.s[p]);
        uint16_t* bi = sc + l.meta[p];
        for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < l.meta[p]; i += uint64_t(gridDim.x) * blockDim.x) {
            const float v = synth_scale(ps ^ 0x5CA1E5CA1Eull, i, l.lo[p], l.span[p]);
            sc[i] = uint16_t(__float_as_uint(v) >> 16);
            bi[i] = uint16_t(__float_as_uint(bf(v * l.factor[p])) >> 16);
        }
    }
}
void launch_synth_records(hipStream_t s, void* records, uint64_t stride, uint32_t count, const uint64_t* w_off,
                          const uint64_t* s_off, const uint64_t* words, const uint64_t* meta, const uint32_t* bits, uint64_t seed) {
    RecordLayout l{};
    for (int p = 0; p < 3; ++p) {
        l.w[p] = w_off[p]; l.s[p] = s_off[p]; l.words[p] = words[p]; l.meta[p] = meta[p];
        l.lo[p] = bits[p] == 8 ? 0.0002f : 0.002f; l.span[p] = bits[p] == 8 ? 0.0018f : 0.018f;
        l.factor[p] = bits[p] == 8 ? -128.0f : -8.0f;
    }
    hipLaunchKernelGGL(synth_records_kernel, dim3(64, count), dim3(256), 0, s, (uint8_t*)records, stride, l, seed);
}

}  // namespace zc
