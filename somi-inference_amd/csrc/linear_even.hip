// The product of some tens of rows (17 to 192) with its columns dealt out evenly over the compute units: bfloat16 in, float32 sums on
// the matrix cores.
//
// Reference: the same nn.Linear products as linear_plain.hip (somi_inference/models/qwen2.py:221-222, 268-271;
// qwen2_adapter.py:60-62), with the norm's row scale and the gate as in linear_fused.hip.
//
// Such a product is bound by reading w once, and a compute unit takes no more than its share of the memory's rate: what counts
// is that every unit has the same number of columns.  linear_mid.hip's 64- and 128-column workgroups leave 2 or 3 of them on a unit (7B
// gate_up, 37,888 x 3,584, at 64 rows: 592 workgroups on 256 units, 57 us and a reduce of 8, where the weight alone takes 41); 256-column
// tiles of the many-rows kernel leave 108 of 256 units without one (71 us at 128 rows).  Here a workgroup has a compute unit
// to itself and owns NS strips of 16 columns over all of K.  Measured, the launches that it replaces / here, us at 17, 64 and 128 rows:
//   gate_up of 37,888 x 3,584: 55 / 45, 63 / 51, 68 / 63 (at 192 rows 86 / 77);  of 27,648 x 5,120: 57 / 49, 65 / 56, 90 / 69;
//   of 28,672 x 4,096: 62 / 37, 61 / 40, 72 / 50 (see the start of a workgroup's K below);
//   down of 3,584 x 18,944: 27 / 28, 35 / 32, 50 / 39;  of 5,120 x 13,824: 28 / 30, 34 / 33, 50 / 40.
// What is left above the weight's time is x, which every workgroup reads: 7 TB/s of w and x together.
//
// Eight wavefronts share a stage (64 values of K: one 128-byte line of each of the workgroup's rows of w and of x) through LDS,
// held twice; the next DEPTH stages are on their way in registers.  Wavefront v owns row tiles v % 4 (v % 4 + 4, v % 4 + 8) and a share
// of the strips, by pairs (a gate strip and its up strip).  w is the A operand, so a lane has four neighbouring columns of a row.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

#define EVEN_WORD3 0x00020000u                    // raw buffer, 32-bit elements, no swizzle
#define EVEN_OUT_OF_RANGE 0x80000000u
#define EVEN_THREADS 512
#define EVEN_CK 64                                // values of K of a stage
#define EVEN_DEPTH 4
#define EVEN_MOST_ROWS 192

enum EvenForm { EVEN_GATED = 0, EVEN_PLANES = 1 };

struct EvenArgs {
    const bf16* x;                                // [M, K]
    const bf16* w;                                // [N, K]; gated: gate and up rows interleaved in blocks of 16
    int M, N, K;
    void* out;                                    // gated: [M, N / 2] bfloat16; planes: [splits][M, N] float32
    const float* stats;                           // gated: [stats_blocks][stats_stride] sums of squares of the rows
    int stats_blocks, stats_stride;
    float eps;
    int act, splits;
};

// LDS rows of 128 bytes hold their 16-byte pieces permuted by the row: 16 lanes that read one piece of 16 rows touch all banks once.
__device__ __forceinline__ int even_swizzle(int row) { return (row >> 1) & 7; }

template <int RT, int NS, int FORM>
__global__ void __launch_bounds__(EVEN_THREADS)
linear_even_kernel(const EvenArgs p) {
    constexpr int ROWS = 16 * RT, COLUMNS = 16 * NS, STAGE = (ROWS + COLUMNS) * 128;
    constexpr int PIECES = (ROWS + COLUMNS) * 8, LOADS = (PIECES + EVEN_THREADS - 1) / EVEN_THREADS;
    constexpr int RPW = RT > 4 ? RT / 4 : 1;              // row tiles of a wavefront
    constexpr int ROW_GROUPS = RT > 4 ? 4 : RT, STRIP_GROUPS = 8 / ROW_GROUPS, PAIRS = NS / 2;
    constexpr int MOST = 2 * ((PAIRS + STRIP_GROUPS - 1) / STRIP_GROUPS);      // strips of a wavefront at most
    static_assert(NS % 2 == 0 && (RT == 2 || RT == 4 || RT == 8 || RT == 12), "pairs of strips, 32, 64, 128 or 192 rows");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    float* part = reinterpret_cast<float*>(lds + 2 * STAGE);     // [EVEN_THREADS] parts of the rows' sums of squares
    float* scale = part + EVEN_THREADS;                          // [ROWS]

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int row_group = wave % ROW_GROUPS, strip_group = wave / ROW_GROUPS;
    const int first_strip = 2 * (strip_group * PAIRS / STRIP_GROUPS), strips = 2 * ((strip_group + 1) * PAIRS / STRIP_GROUPS) - first_strip;
    const int split = FORM == EVEN_PLANES ? blockIdx.x % p.splits : 0;
    const int n0 = (int)(FORM == EVEN_PLANES ? blockIdx.x / p.splits : blockIdx.x) * COLUMNS;
    const int K = p.K, M = p.M, N = p.N;
    const int stages = (K + EVEN_CK - 1) / EVEN_CK, each = (stages + p.splits - 1) / p.splits, first = split * each;
    const int mine = min(each, stages - first);          // (at least one: the host takes ceil(stages / each) splits)
    // Rows a multiple of 4 KB apart put a line of every row on the same memory channels, and workgroups that march through K together
    // all ask them at once: there each starts at another stage and goes round (28,672 x 4,096 at 17 and 64 rows: 55 and 57 us from the
    // same stage, 40 and 44 so; 37,888 x 3,584: 45 and 53 from the same stage, 46 and 54 so, x's lines being less often in the cache).
    const int start = FORM == EVEN_GATED && K % 2048 == 0 ? (int)((blockIdx.x >> 3) * 5u % (unsigned)mine) : 0;

    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, (int)((int64_t)M * K * 2), EVEN_WORD3);
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w + (int64_t)n0 * K), 0,
                                                                          (int)((int64_t)min(COLUMNS, N - n0) * K * 2), EVEN_WORD3);
    // rows 0 .. ROWS - 1 of a stage are x's, the others w's; eight lanes read a row's line.  Rows past M or N read as zeros.
    const int lrow = tid >> 3, lpiece = tid & 7;
    constexpr int ROWS_A_LOAD = EVEN_THREADS / 8;
    auto issue = [&](u32x4 (&st)[LOADS], int turn) {
        const int at = turn + start < mine ? turn + start : turn + start - mine;
        const int k0 = (first + at) * EVEN_CK + lpiece * 8;
        const bool inside = turn < mine && k0 < K;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int row = i * ROWS_A_LOAD + lrow;
            const bool is_x = ROWS % ROWS_A_LOAD == 0 ? i * ROWS_A_LOAD < ROWS : row < ROWS;
            const unsigned off = ((unsigned)(is_x ? row : row - ROWS) * (unsigned)K + (unsigned)k0) * 2u;
            const bool there = inside && row < ROWS + COLUMNS;
            if (is_x) st[i] = __builtin_amdgcn_raw_buffer_load_b128(xres, there ? off : EVEN_OUT_OF_RANGE, 0, 0);
            else st[i] = __builtin_amdgcn_raw_buffer_load_b128(wres, there ? off : EVEN_OUT_OF_RANGE, 0, SOMI_LOAD_ONCE);
        }
    };
    auto stash = [&](const u32x4 (&st)[LOADS], int buffer) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int row = i * ROWS_A_LOAD + lrow;
            if (PIECES % EVEN_THREADS == 0 || row < ROWS + COLUMNS)
                *reinterpret_cast<u32x4*>(lds + buffer * STAGE + row * 128 + ((lpiece ^ even_swizzle(row)) << 4)) = st[i];
        }
    };

    f32x4 acc[RPW][MOST];
#pragma unroll
    for (int a = 0; a < RPW; ++a)
#pragma unroll
        for (int s = 0; s < MOST; ++s) acc[a][s] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int buffer) {
        const char* stage = lds + buffer * STAGE;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int piece = ((half * 4 + g) ^ even_swizzle(r)) << 4;
            bf16x8 xv[RPW];
#pragma unroll
            for (int a = 0; a < RPW; ++a)
                xv[a] = *reinterpret_cast<const bf16x8*>(stage + ((row_group + 4 * a) * 16 + r) * 128 + piece);
#pragma unroll
            for (int s = 0; s < MOST; ++s) {
                if (s >= strips) continue;                // (the same for the whole wavefront)
                const bf16x8 wv = *reinterpret_cast<const bf16x8*>(stage + (ROWS + (first_strip + s) * 16 + r) * 128 + piece);
#pragma unroll
                for (int a = 0; a < RPW; ++a) acc[a][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv[a], acc[a][s], 0, 0, 0);
            }
        }
    };

    // stage `turn` is in LDS buffer turn & 1, register set d holds turn + 1 + d; a pass is DEPTH stages, so that sets and buffers are
    // named at compile time.  Stages past the end are zeros.
    static_assert(EVEN_DEPTH == 4, "a pass of four stages");
    u32x4 st[EVEN_DEPTH][LOADS];
#pragma unroll
    for (int d = 0; d < EVEN_DEPTH; ++d) issue(st[d], d);
    if (FORM == EVEN_GATED) {
        // the rows' sums of squares: thread (row, e) adds the blocks e, e + E, ... in order, then a row's E sums are added in order
        constexpr int E = EVEN_THREADS / ROWS;
        const int row = tid % ROWS, e = tid / ROWS;
        float sum = 0.f;
        if (row < M && e < E)
            for (int b = e; b < p.stats_blocks; b += E) sum += p.stats[(int64_t)b * p.stats_stride + row];
        part[tid] = sum;
        __syncthreads();
        if (tid < ROWS) {
            float whole = 0.f;
#pragma unroll
            for (int i = 0; i < E; ++i) whole += part[i * ROWS + tid];
            scale[tid] = 1.0f / sqrtf(whole / (float)K + p.eps);
        }
    }
    stash(st[0], 0);
    issue(st[0], EVEN_DEPTH);
    __syncthreads();
    for (int turn = 0; turn < mine; turn += EVEN_DEPTH) {
#pragma unroll
        for (int d = 0; d < EVEN_DEPTH; ++d) {
            constexpr int SETS = EVEN_DEPTH;
            stash(st[(d + 1) % SETS], (d + 1) & 1);
            issue(st[(d + 1) % SETS], turn + d + 1 + SETS);
            compute(d & 1);
            __syncthreads();
        }
    }

    // D[n][m]: lane (r, g) of strip s holds the columns 4 g .. 4 g + 3 of row r of its row tile
#pragma unroll
    for (int a = 0; a < RPW; ++a) {
        const int m = (row_group + 4 * a) * 16 + r;
        if (m >= M) continue;
        if (FORM == EVEN_GATED) {
            const float s = scale[m];
            const int inter = N / 2;
#pragma unroll
            for (int pair = 0; pair < MOST / 2; ++pair) {
                const int n = n0 / 2 + (first_strip / 2 + pair) * 16 + g * 4;
                if (2 * pair >= strips || n >= inter) continue;
                bf16x4 v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = (bf16)somi_gated(s * acc[a][2 * pair][i], s * acc[a][2 * pair + 1][i], p.act);
                *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(p.out) + (int64_t)m * inter + n) = v;
            }
        } else {
            float* to = reinterpret_cast<float*>(p.out) + ((int64_t)split * M + m) * N;
#pragma unroll
            for (int s = 0; s < MOST; ++s) {
                const int n = n0 + (first_strip + s) * 16 + g * 4;
                if (s >= strips || n >= N) continue;
                const f32x4 v = acc[a][s];
                if ((N & 3) == 0) *reinterpret_cast<f32x4*>(to + n) = v;
                else
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < N) to[n + i] = v[i];
            }
        }
    }
}

// h += the planes in order (+ bias), the next norm's weighted rows and the rows' sums of squares over 64 columns each: a workgroup
// takes 16 rows x 64 columns, the 16 lanes of a row read 256 consecutive bytes of a plane.
__global__ void __launch_bounds__(256)
linear_even_stream_kernel(const float* __restrict__ planes, int splits, const float* __restrict__ bias, float* __restrict__ h,
                          const float* __restrict__ norm_w, bf16* __restrict__ weighted, float* __restrict__ stats, int stats_stride, int M,
                          int N) {
    const int row = threadIdx.x >> 4, m = blockIdx.y * 16 + row, n = blockIdx.x * 64 + (threadIdx.x & 15) * 4;
    const int64_t plane = (int64_t)M * N;
    float square = 0.f;
    if (m < M && n < N) {
        const int64_t at = (int64_t)m * N + n;
        const bool four = (N & 3) == 0;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if (four) {
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
            for (int s = 0; s < splits; ++s) sum += *reinterpret_cast<const f32x4*>(planes + s * plane + at);
            const f32x4 before = *reinterpret_cast<const f32x4*>(h + at);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = before[i] + (sum[i] + (bias ? bias[n + i] : 0.f));
            *reinterpret_cast<f32x4*>(h + at) = f32x4{v[0], v[1], v[2], v[3]};
        } else {
            for (int i = 0; i < 4 && n + i < N; ++i) {
                float sum = 0.f;
                for (int s = 0; s < splits; ++s) sum += planes[s * plane + at + i];
                v[i] = h[at + i] + (sum + (bias ? bias[n + i] : 0.f));
                h[at + i] = v[i];
            }
        }
        if (weighted) {
            if (four) {
                bf16x4 next;
#pragma unroll
                for (int i = 0; i < 4; ++i) next[i] = (bf16)(norm_w[n + i] * v[i]);
                *reinterpret_cast<bf16x4*>(weighted + at) = next;
            } else {
                for (int i = 0; i < 4 && n + i < N; ++i) weighted[at + i] = (bf16)(norm_w[n + i] * v[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) square += v[i] * v[i];
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) square += __shfl_xor(square, off, 64);
    if ((threadIdx.x & 15) == 0 && m < stats_stride) stats[(int64_t)blockIdx.x * stats_stride + m] = m < M ? square : 0.f;
}

// ---------------------------------------------------------------------------------------------------------- host side
// Strips of a workgroup of the gated form, 6, 8, 10 or 12: the number that takes the least time, a round of workgroups (one a unit)
// the time of the lines that each reads, and no less than what four fifths of the units read at the memory's rate (37,888 x 3,584: at 64 rows 8 / 10 / 12
// strips 71 / 53 / 50 to 55 us, at 128 88 / 66 / 62; 27,648 x 5,120 at 64 rows 57 / 75 / 67).
static int even_strips(int M, int N, int units) {
    const int strips = ceil_div(N, 16), rows = ceil_div(M, 16) * 16;
    int64_t best = -1;
    int chosen = 0;
    for (int ns = 6; ns <= 12; ns += 2) {
        const int tiles = ceil_div(strips, ns), rounds = ceil_div(tiles, units), full = rounds * units * 4 / 5;
        const int64_t lines = (int64_t)(16 * ns + rows) * (tiles > full ? tiles : full);
        if (best < 0 || lines < best) best = lines, chosen = ns;
    }
    return chosen;
}

// Splits of K of the form that goes into the stream, by workgroups of eight strips: as many as fill the units, with four stages each at
// least.  (3,584 x 18,944, 9 splits of 28 tiles, at 17 / 64 / 128 rows 28 / 33 / 40 us; with six strips 29 / 38 / 48, ten 30 / 36 / 45,
// twelve, which need 13 planes, 30 / 34 / 42.  Portions of neighbouring stages: 5,120 x 13,824 at 64 rows with ten strips 38 us, 44 with the
// stages dealt out in turns.)
#define EVEN_STREAM_STRIPS 8
static int even_splits(int N, int K, int units) {
    const int tiles = ceil_div(N, 16 * EVEN_STREAM_STRIPS), stages = ceil_div(K, EVEN_CK);
    int splits = units / tiles < stages / 4 ? units / tiles : stages / 4;
    if (splits < 1) splits = 1;
    return ceil_div(stages, ceil_div(stages, splits));
}

// The launch shapes for these sizes on a device of so many compute units (0: this one).
extern "C" int somi_linear_even_choice(int M, int N, int K, int units, int* strips, int* splits) {
    SOMI_REQUIRE(N > 0 && K > 0 && units >= 0, "linear_even: bad sizes N=%d K=%d", N, K);
    if (units == 0) units = somi_units();
    *strips = even_strips(M, N, units);
    *splits = even_splits(N, K, units);
    return 0;
}

static int even_check(const void* x, const void* w, int M, int N, int K) {
    SOMI_REQUIRE(M >= 0 && N > 0 && K > 0, "linear_even: bad sizes M=%d N=%d K=%d", M, N, K);
    SOMI_REQUIRE(M <= EVEN_MOST_ROWS, "linear_even: at most %d rows, got %d", EVEN_MOST_ROWS, M);
    SOMI_REQUIRE(K % 8 == 0, "linear_even: K (%d) must be a multiple of 8", K);
    SOMI_REQUIRE((int64_t)K * 2 * 192 < (int64_t)1 << 31, "linear_even: K (%d) is too large", K);
    SOMI_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "linear_even: x and w must be 16-byte aligned");
    return 0;
}

template <int RT, int NS, int FORM>
static int even_launch(const EvenArgs& a, hipStream_t stream) {
    // more than half of a compute unit's LDS, so that a unit holds one workgroup
    const size_t needed = (size_t)2 * 16 * (RT + NS) * 128 + (EVEN_THREADS + 16 * RT) * sizeof(float);
    const size_t smem = needed > 82 * 1024 ? needed : 82 * 1024;
    (void)hipFuncSetAttribute((const void*)linear_even_kernel<RT, NS, FORM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipLaunchKernelGGL((linear_even_kernel<RT, NS, FORM>), dim3(ceil_div(a.N, 16 * NS) * a.splits), dim3(EVEN_THREADS), smem, stream, a);
    SOMI_LAUNCH_CHECK("linear_even");
    return 0;
}

// out[m, i] = act(s g) * (s u) -> bfloat16 [M, N / 2] for the products g, u of x's rows with w's gate and up rows (interleaved in
// blocks of 16); s[m] = 1 / sqrt(sum of stats[:, m] / K + eps) with stats [stats_blocks][stats_stride >= M] partial sums of squares.
// act 1: SiLU, 2: the tanh form of GELU.  M <= 192, N a multiple of 32, out 8-byte aligned.
extern "C" int somi_linear_even_gated(const void* x, float eps, const float* stats, int stats_blocks, int stats_stride, const void* w,
                                      void* out, int M, int N, int K, int act, hipStream_t stream) {
    if (even_check(x, w, M, N, K)) return 1;
    SOMI_REQUIRE(N % 32 == 0 && (uintptr_t)out % 8 == 0, "linear_even: the gated form needs whole pairs of strips, got N = %d", N);
    SOMI_REQUIRE(stats && stats_blocks > 0 && stats_stride >= M, "linear_even: bad row statistics");
    SOMI_REQUIRE(act == 1 || act == 2, "linear_even: activation %d (1: SiLU, 2: the tanh form of GELU)", act);
    if (M == 0) return 0;
    EvenArgs a = {};
    a.x = (const bf16*)x; a.w = (const bf16*)w; a.M = M; a.N = N; a.K = K; a.out = out; a.splits = 1;
    a.stats = stats; a.stats_blocks = stats_blocks; a.stats_stride = stats_stride; a.eps = eps; a.act = act;
    const int strips = even_strips(M, N, somi_units());
#define SOMI_EVEN(RT)                                                       \
    return strips == 6    ? even_launch<RT, 6, EVEN_GATED>(a, stream)       \
           : strips == 8  ? even_launch<RT, 8, EVEN_GATED>(a, stream)       \
           : strips == 10 ? even_launch<RT, 10, EVEN_GATED>(a, stream)      \
                          : even_launch<RT, 12, EVEN_GATED>(a, stream)
    if (M <= 32) SOMI_EVEN(2);
    if (M <= 64) SOMI_EVEN(4);
    if (M <= 128) SOMI_EVEN(8);
    SOMI_EVEN(12);
#undef SOMI_EVEN
}

// Planes of [M, N] float32 that somi_linear_even_residual needs.
extern "C" int somi_linear_even_planes(int N, int K) { return N > 0 && K > 0 ? even_splits(N, K, somi_units()) : 1; }

// h[m, n] += x[m, :] . w[n, :] (+ bias[n]), float32 in place; planes: somi_linear_even_planes(N, K) planes of [M, N] float32; stats:
// [ceil(N / 64)][stats_stride >= M], out, sums of squares of the new h over 64 columns each (0 from M on); weighted: [M, N] bfloat16 =
// norm_w * h, or null.  M <= 128 rows; planes and h 16-byte, weighted 8-byte aligned.
extern "C" int somi_linear_even_residual(const void* x, const void* w, const float* bias, float* h, float* stats, int stats_stride,
                                         const float* norm_w, void* weighted, float* planes, int M, int N, int K, hipStream_t stream) {
    if (even_check(x, w, M, N, K)) return 1;
    SOMI_REQUIRE(M <= 128, "linear_even: at most 128 rows into the stream, got %d", M);
    SOMI_REQUIRE(h && stats && planes && stats_stride >= M, "linear_even: h, stats and the planes are needed");
    SOMI_REQUIRE(!weighted || norm_w, "linear_even: the next rows need the norm's weight");
    SOMI_REQUIRE((((uintptr_t)h | (uintptr_t)planes) & 15) == 0 && (uintptr_t)weighted % 8 == 0, "linear_even: h and the planes must be aligned");
    if (M == 0) return 0;
    EvenArgs a = {};
    a.x = (const bf16*)x; a.w = (const bf16*)w; a.M = M; a.N = N; a.K = K; a.out = planes;
    a.splits = even_splits(N, K, somi_units());
    if (M <= 64 ? even_launch<4, EVEN_STREAM_STRIPS, EVEN_PLANES>(a, stream) : even_launch<8, EVEN_STREAM_STRIPS, EVEN_PLANES>(a, stream)) return 1;
    hipLaunchKernelGGL(linear_even_stream_kernel, dim3(ceil_div(N, 64), ceil_div(stats_stride, 16)), dim3(256), 0, stream, planes, a.splits,
                       bias, h, norm_w, (bf16*)weighted, stats, stats_stride, M, N);
    SOMI_LAUNCH_CHECK("linear_even_stream");
    return 0;
}
