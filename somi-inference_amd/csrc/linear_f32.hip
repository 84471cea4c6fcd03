// Linear layer in float32 on the matrix cores: out[m, n] = sum_k x[m, k] * w[n, k] (+ bias[n]), every operand, product and sum
// float32 (v_mfma_f32_16x16x4_f32; no reduced-precision mode), for any number of rows.
//
// Reference: nn.Linear / F.linear as used for q/k/v/o, the merged gate_up, down and the LM head
// (somi_inference/models/qwen2.py:221-222, 268-271, 296-298; qwen2_adapter.py:60-62).
//
// An element's sum has ONE order, whatever launch it is in: K in units of 32 is cut into F32_CHAINS contiguous chains of equal
// length (to a unit); a chain is summed by the matrix core in order of k; four neighbouring chains are added in order to a
// group, the groups in order to the total.  The order depends on K alone, so a row's result is the same bits in a step of one
// token and in a prompt of thousands, and the two kernels below may share K out as their shape asks:
//   * up to 32 rows the product is bound by reading w once.  A workgroup owns 16 (or 32) columns, its wavefronts one (or two)
//     chains each, so even 896 columns keep 56 x 16 wavefronts reading.  Rows are read in whole 128-byte lines (8 lanes a
//     row), two or three units in flight a wavefront, and turned through a private, swizzled piece of LDS into the operand
//     layout, as linear_skinny.hip does.
//   * more rows are tiles through LDS.  A 128 x 128 tile moves 8 bytes a clock and compute unit at the matrix cores' rate
//     (64 x 64: 16, more than the L2 gives every unit at once), so it is taken where there are tiles for the device; with
//     fewer tiles 64 x 64, and where those are too few as well, a tile's four groups go to four workgroups, whose sums a second
//     kernel adds.
//
// The gated form ends a product over gate and up rows (gate rows first) with silu(gate) * up: a workgroup takes the gate rows and the
// up rows of the same columns, so the activation is no kernel of its own (4.7 us a decode layer of a 0.5B model, 7 of a prompt of 512).
//
// Measured on an MI355X against the kernel this replaces for float32 (linear_plain.hip, 64 x 64 tiles of scalar multiply-adds, one
// thread an element over all of K): 8 rows by 37,888 over K = 3,584 in 87 us (6.3 TB/s of w), 896 by 4,864 11 us where it took
// 700, 2,048 rows by 37,888 4.2 ms (131 TFLOP/s; a library's 8,192-cubed product 151).
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

#define F32_WORD3 0x00020000u                     // raw buffer, 32-bit elements, no swizzle
#define F32_OUT_OF_RANGE 0x80000000u
#define F32_UNIT 32                               // k-values of a unit: one 128-byte line of a row
#define F32_CHAINS 16
#define F32_GROUPS 4
#define F32_GROUP_CHAINS (F32_CHAINS / F32_GROUPS)
#define F32_ROW_BYTES (F32_UNIT * 4)

// First unit of a chain (chain == F32_CHAINS: the end).
__device__ __forceinline__ int f32_chain_begin(int chain, int units) { return (int)((int64_t)chain * units / F32_CHAINS); }

// LDS rows of 128 bytes hold their 16-byte pieces permuted by the row, so that 16 lanes reading one piece of 16 rows, and 16
// lanes writing two rows, touch all 64 banks once.
__device__ __forceinline__ int f32_swizzle(int row) { return (row >> 1) & 7; }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t f32_rows(const float* base, int64_t first_row, int rows, int K) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + first_row * K), 0, (int)((int64_t)rows * K * 4), F32_WORD3);
}

__device__ __forceinline__ float f32_gated(float gate, float up) { return gate / (1.0f + expf(-gate)) * up; }

// ------------------------------------------------------------------------------------------------------------ few rows
// WAVES wavefronts, F32_CHAINS / WAVES chains each; MT blocks of 16 rows, NS of 16 columns; DEPTH units in flight.  GATED: N output
// columns, w: [2 N, K], the first block of columns is of gate, the second of up.
template <int WAVES, int MT, int NS, int DEPTH, bool GATED>
__global__ void __launch_bounds__(WAVES * 64)
linear_f32_rows_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                       float* __restrict__ out, int M, int N, int K) {
    constexpr int CPW = F32_CHAINS / WAVES;               // chains of a wavefront, neighbouring ones
    static_assert(CPW == 1 || CPW == 2, "one chain or two a wavefront");
    static_assert(!GATED || NS == 2, "gate and up");
    constexpr int NL = 2 * (NS + MT);                     // loads of a lane and unit: 8 rows each, w's then x's
    constexpr int WAVE_BYTES = 16 * (NS + MT) * F32_ROW_BYTES;
    constexpr int TILES = NS * MT, SUMS_BYTES = F32_CHAINS * TILES * 1024;
    __shared__ __attribute__((aligned(16))) char lds[WAVES * WAVE_BYTES > SUMS_BYTES ? WAVES * WAVE_BYTES : SUMS_BYTES];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (GATED ? 16 : 16 * NS);
    const int units = (K + F32_UNIT - 1) / F32_UNIT;
    const int first = f32_chain_begin(wave * CPW, units), last = f32_chain_begin((wave + 1) * CPW, units);
    char* mine = lds + wave * WAVE_BYTES;

    const __amdgpu_buffer_rsrc_t wres = f32_rows(w, n0, GATED ? 2 * N - n0 : min(16 * NS, N - n0), K);
    const __amdgpu_buffer_rsrc_t xres = f32_rows(x, 0, M, K);
    const int lrow = lane >> 3, lpiece = lane & 7;
    unsigned goff[NL];
    int soff[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int row = i * 8 + lrow;                     // rows 0 .. 16 NS - 1 are w's, the rest x's
        const int from = row >= 16 * NS ? row - 16 * NS : GATED && row >= 16 ? N + row - 16 : row;
        goff[i] = ((unsigned)from * (unsigned)K + lpiece * 4) * 4u;
        soff[i] = row * F32_ROW_BYTES + ((lpiece ^ f32_swizzle(row)) << 4);
    }
    // units past the wavefront's, and the pieces of the last unit past K, read as zeros
    auto issue = [&](u32x4 (&st)[NL], int unit) {
        const bool inside = unit < last && unit * F32_UNIT + lpiece * 4 < K;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const unsigned off = inside ? goff[i] + (unsigned)unit * F32_ROW_BYTES : F32_OUT_OF_RANGE;
            st[i] = i < 2 * NS ? __builtin_amdgcn_raw_buffer_load_b128(wres, off, 0, SOMI_LOAD_ONCE)
                               : __builtin_amdgcn_raw_buffer_load_b128(xres, off, 0, 0);
        }
    };
    f32x4 acc[TILES], chain[CPW][TILES];                  // tile s * MT + mt
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto consume = [&](const u32x4 (&st)[NL]) {
#pragma unroll
        for (int i = 0; i < NL; ++i) *reinterpret_cast<u32x4*>(mine + soff[i]) = st[i];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int piece = (half * 4 + g) ^ f32_swizzle(r);          // the same key for rows 16 apart
            f32x4 xv[MT], wv[NS];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                xv[mt] = *reinterpret_cast<const f32x4*>(mine + (16 * (NS + mt) + r) * F32_ROW_BYTES + (piece << 4));
#pragma unroll
            for (int s = 0; s < NS; ++s)
                wv[s] = *reinterpret_cast<const f32x4*>(mine + (16 * s + r) * F32_ROW_BYTES + (piece << 4));
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < TILES; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t / MT][j], xv[t % MT][j], acc[t], 0, 0, 0);
        }
    };

    // The wavefront's units are one contiguous range; set d holds unit `at + d`.  Units past the range are zeros, which leave a sum
    // as it is.
    const int second = f32_chain_begin(wave * CPW + 1, units);
    u32x4 st[DEPTH][NL];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) issue(st[d], first + d);
    bool folded = CPW == 1;
    auto fold = [&]() {                                   // the first of two chains is complete
        folded = true;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            chain[0][t] = acc[t];
            acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    for (int at = first; at < last; at += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            if (CPW == 2 && at + d == second) fold();
            consume(st[d]);
            issue(st[d], at + DEPTH + d);
        }
    }
    if (!folded) fold();
#pragma unroll
    for (int t = 0; t < TILES; ++t) chain[CPW - 1][t] = acc[t];

    __syncthreads();                                      // every wavefront is done with its staging space
    float* sums = reinterpret_cast<float*>(lds);          // [F32_CHAINS][TILES][64 lanes][4]
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            *reinterpret_cast<f32x4*>(sums + (((wave * CPW + c) * TILES + t) * 64 + lane) * 4) = chain[c][t];
    __syncthreads();
    // element idx of a block: column (idx / 64) * 4 + idx % 4 of row (idx / 4) % 16
    auto whole = [&](int idx) {
        float total = 0.f;
#pragma unroll
        for (int group = 0; group < F32_GROUPS; ++group) {
            float sum = 0.f;
#pragma unroll
            for (int c = 0; c < F32_GROUP_CHAINS; ++c) sum += sums[(group * F32_GROUP_CHAINS + c) * TILES * 256 + idx];
            total += sum;
        }
        return total;
    };
    for (int idx = threadIdx.x; idx < (GATED ? MT : TILES) * 256; idx += WAVES * 64) {
        const int tile = idx >> 8, l = (idx >> 2) & 63, i = idx & 3;
        const int n = n0 + tile / MT * 16 + (l >> 4) * 4 + i, m = tile % MT * 16 + (l & 15);
        float v = whole(idx);
        if (GATED) v = f32_gated(v, whole(MT * 256 + idx));
        if (n < N && m < M) out[(int64_t)m * N + n] = bias ? v + bias[n] : v;
    }
}

// ------------------------------------------------------------------------------------------------------------ more rows
// A workgroup's WM x WN wavefronts own RM x RN blocks of 16 x 16 each: a tile of 16 WM RM rows by 16 WN RN columns.  A stage is
// one unit of K of the tile's rows of x and w, held twice in LDS; the stages behind it come through registers, DEPTH of them in
// flight.  With `planes` the workgroup sums group blockIdx.z alone and leaves it there.  GATED (without planes): N output columns,
// w: [2 N, K]; a wavefront's two blocks of columns are gate and up of the same 16.
template <int WM, int WN, int RM, int RN, int DEPTH, bool GATED>
__global__ void __launch_bounds__(WM * WN * 64)
linear_f32_tile_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                       float* __restrict__ out, float* __restrict__ planes, int M, int N, int K) {
    constexpr int THREADS = WM * WN * 64, TM = 16 * WM * RM, TN = 16 * WN * RN;
    constexpr int STAGE = (TM + TN) * F32_ROW_BYTES, LOADS = (TM + TN) * 8 / THREADS, LOADS_X = TM * 8 / THREADS;
    static_assert(TM * 8 % THREADS == 0 && TN * 8 % THREADS == 0, "whole loads of x and of w");
    static_assert(!GATED || RN == 2, "gate and up");
    __shared__ __attribute__((aligned(16))) char lds[2 * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int r = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.x * TM, n0 = blockIdx.y * (GATED ? TN / 2 : TN);
    const int units = (K + F32_UNIT - 1) / F32_UNIT;
    const int first_chain = planes ? blockIdx.z * F32_GROUP_CHAINS : 0;
    const int last_chain = planes ? first_chain + F32_GROUP_CHAINS : F32_CHAINS;
    const int first = f32_chain_begin(first_chain, units), last = f32_chain_begin(last_chain, units);

    const __amdgpu_buffer_rsrc_t xres = f32_rows(x, m0, min(TM, M - m0), K);
    const __amdgpu_buffer_rsrc_t wres = f32_rows(w, n0, GATED ? 2 * N - n0 : min(TN, N - n0), K);
    const int lrow = tid >> 3, lpiece = tid & 7;
    constexpr int ROWS_A_LOAD = THREADS / 8;              // a multiple of 16, so a thread's loads share their swizzle
    static_assert(ROWS_A_LOAD % 16 == 0, "rows of one load");
    unsigned goff[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        int row = (i < LOADS_X ? i : i - LOADS_X) * ROWS_A_LOAD + lrow;
        if (GATED && i >= LOADS_X) row = ((row >> 4) & 1) * N + (row >> 5) * 16 + (row & 15);
        goff[i] = ((unsigned)row * (unsigned)K + lpiece * 4) * 4u;
    }
    const int soff = lrow * F32_ROW_BYTES + ((lpiece ^ f32_swizzle(lrow)) << 4);

    auto issue = [&](u32x4 (&st)[LOADS], int unit) {
        const bool inside = unit < last && unit * F32_UNIT + lpiece * 4 < K;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const unsigned off = inside ? goff[i] + (unsigned)unit * F32_ROW_BYTES : F32_OUT_OF_RANGE;
            st[i] = __builtin_amdgcn_raw_buffer_load_b128(i < LOADS_X ? xres : wres, off, 0, 0);
        }
    };
    auto stash = [&](const u32x4 (&st)[LOADS], int buffer) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            *reinterpret_cast<u32x4*>(lds + buffer * STAGE + soff + i * ROWS_A_LOAD * F32_ROW_BYTES) = st[i];
    };

    f32x4 acc[RM][RN], sum[RM][RN], total[RM][RN];        // of the chain, the group, the element
#pragma unroll
    for (int a = 0; a < RM; ++a)
#pragma unroll
        for (int b = 0; b < RN; ++b) acc[a][b] = sum[a][b] = total[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    int chain = first_chain, chain_end = f32_chain_begin(first_chain + 1, units);
    auto end_chains = [&](int unit) {                     // the chains that end in front of `unit` join their groups
        while (chain < last_chain && chain_end <= unit) {
            ++chain;
            const bool group_ends = chain % F32_GROUP_CHAINS == 0;
#pragma unroll
            for (int a = 0; a < RM; ++a)
#pragma unroll
                for (int b = 0; b < RN; ++b) {
                    sum[a][b] += acc[a][b];
                    acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (group_ends) {
                        total[a][b] += sum[a][b];
                        sum[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                }
            chain_end = f32_chain_begin(chain + 1, units);
        }
    };
    auto compute = [&](int buffer) {
        const char* stage = lds + buffer * STAGE;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int piece = ((half * 4 + g) ^ f32_swizzle(r)) << 4;
            f32x4 xv[RM], wv[RN];
#pragma unroll
            for (int a = 0; a < RM; ++a)
                xv[a] = *reinterpret_cast<const f32x4*>(stage + ((wm * RM + a) * 16 + r) * F32_ROW_BYTES + piece);
#pragma unroll
            for (int b = 0; b < RN; ++b)
                wv[b] = *reinterpret_cast<const f32x4*>(stage + (TM + (wn * RN + b) * 16 + r) * F32_ROW_BYTES + piece);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int a = 0; a < RM; ++a)
#pragma unroll
                    for (int b = 0; b < RN; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[b][j], xv[a][j], acc[a][b], 0, 0, 0);
        }
    };

    // stage `unit` is in LDS buffer (unit - first) & 1; register set d holds unit + 1 + d.  A pass of the loop is DEPTH units (an
    // even number of buffers' turns), so that sets and buffers are named at compile time.
    static_assert(DEPTH == 2, "a pass of two units");
    u32x4 st[DEPTH][LOADS];
    issue(st[0], first);
    issue(st[1], first + 1);
    stash(st[0], 0);
    issue(st[0], first + 2);
    __syncthreads();
    for (int unit = first; unit < last; unit += 2) {
        end_chains(unit);
        stash(st[1], 1);                                  // unit + 1
        issue(st[1], unit + 3);
        compute(0);
        __syncthreads();
        if (unit + 1 < last) {
            end_chains(unit + 1);
            stash(st[0], 0);                              // unit + 2
            issue(st[0], unit + 4);
            compute(1);
            __syncthreads();
        }
    }
    end_chains(last);

    float* to = planes ? planes + (int64_t)blockIdx.z * M * N : out;
    const bool wide = N % 4 == 0;                         // (out and the planes are 16-byte aligned)
#pragma unroll
    for (int a = 0; a < RM; ++a)
#pragma unroll
        for (int b = 0; b < (GATED ? 1 : RN); ++b) {
            const int m = m0 + (wm * RM + a) * 16 + r, n = n0 + (GATED ? wn : wn * RN + b) * 16 + g * 4;
            if (m >= M || n >= N) continue;
            f32x4 v = total[a][b];
            if (GATED) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = f32_gated(v[i], total[a][RN - 1][i]);
            }
            float* at = to + (int64_t)m * N + n;
            if (bias && !planes) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] += n + i < N ? bias[n + i] : 0.f;
            }
            if (wide) {
                *reinterpret_cast<f32x4*>(at) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) at[i] = v[i];
            }
        }
}

// The groups' sums added in order.  planes: [F32_GROUPS][M * N].
__global__ void __launch_bounds__(256)
linear_f32_join_kernel(const float* __restrict__ planes, const float* __restrict__ bias, float* __restrict__ out, int64_t count,
                       int N) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    if (N % 4 == 0) {
        for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < count / 4; i += stride) {
            f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < F32_GROUPS; ++p) v += reinterpret_cast<const f32x4*>(planes + p * count)[i];
            if (bias) v += *reinterpret_cast<const f32x4*>(bias + i * 4 % N);
            reinterpret_cast<f32x4*>(out)[i] = v;
        }
        return;
    }
    for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += stride) {
        float v = 0.f;
#pragma unroll
        for (int p = 0; p < F32_GROUPS; ++p) v += planes[p * count + i];
        out[i] = bias ? v + bias[i % N] : v;
    }
}

// The same of a gated product: planes: [F32_GROUPS][M, 2 N], out: [M, N].
__global__ void __launch_bounds__(256)
linear_f32_join_gated_kernel(const float* __restrict__ planes, float* __restrict__ out, int64_t count, int N) {
    const int64_t stride = (int64_t)gridDim.x * 256, plane = 2 * count;
    for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += stride) {
        const float* at = planes + i / N * 2 * N + i % N;
        float gate = 0.f, up = 0.f;
#pragma unroll
        for (int p = 0; p < F32_GROUPS; ++p) {
            gate += at[p * plane];
            up += at[p * plane + N];
        }
        out[i] = f32_gated(gate, up);
    }
}

// Which kernel a product of M rows and N columns takes on `units` compute units: 0 the few-rows kernel, else a tile of 64 x 64 (1)
// or 128 x 128 (2), plus 8 where its groups go to workgroups of their own.
//
// A compute unit's share of a product is counted in tiles of 128 x 128, whole tiles a unit; tiles of 64 x 64 are a quarter of one
// and reach 0.87 of its rate (their operands come from L2 at 9 TB/s).  512 x 9,728 over K = 896: 304 large tiles are two rounds of
// 256 units, 128 us; 1,216 small ones 5 quarter
// rounds, 89 us.  Fewer than two small tiles a unit leave matrix cores idle: their groups are
// shared out, which costs four planes written and read.
static int f32_choice(int M, int N, int units) {
    if (M <= 32) return 0;
    const int64_t small = (int64_t)ceil_div(M, 64) * ceil_div(N, 64), large = (int64_t)ceil_div(M, 128) * ceil_div(N, 128);
    if (small < 2 * (int64_t)units) return 1 + 8;
    const double small_cost = 0.25 / 0.87 * (double)((small + units - 1) / units);
    return M > 64 && (double)((large + units - 1) / units) <= small_cost ? 2 : 1;
}

// Planes of [M, N] floats that a product needs as its workspace (0: none).
extern "C" int somi_linear_f32_planes(int M, int N) { return M > 0 && N > 0 && (f32_choice(M, N, somi_units()) & 8) ? F32_GROUPS : 0; }

extern "C" int somi_linear_f32_choice(int M, int N, int units) { return f32_choice(M, N, units); }

template <int WM, int WN, int RM, int RN, bool GATED>
static void f32_launch_tile(const float* x, const float* w, const float* bias, float* out, float* planes, int M, int N, int K,
                            hipStream_t stream) {
    const dim3 grid(ceil_div(M, 16 * WM * RM), ceil_div(N, GATED ? 8 * WN * RN : 16 * WN * RN), planes ? F32_GROUPS : 1);
    hipLaunchKernelGGL((linear_f32_tile_kernel<WM, WN, RM, RN, 2, GATED>), grid, dim3(WM * WN * 64), 0, stream, x, w, bias, out, planes,
                       M, N, K);
}

static int f32_check(const float* x, const float* w, const float* bias, const float* out, const float* workspace, int M, int N, int K) {
    SOMI_REQUIRE(M >= 0 && N > 0 && K > 0, "linear_f32: bad sizes M=%d N=%d K=%d", M, N, K);
    SOMI_REQUIRE(K % 4 == 0, "linear_f32: K (%d) must be a multiple of 4", K);
    SOMI_REQUIRE((int64_t)K * 4 * 128 < (int64_t)1 << 31, "linear_f32: K (%d) is too large", K);
    SOMI_REQUIRE(ceil_div(N, 64) <= 65535, "linear_f32: too many columns for one launch (N=%d)", N);
    SOMI_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)bias | (uintptr_t)workspace) & 15) == 0,
                 "linear_f32: x, w, bias, out and the workspace must be 16-byte aligned");
    SOMI_REQUIRE(M == 0 || somi_linear_f32_planes(M, N) == 0 || workspace != nullptr, "linear_f32: %d rows by %d columns need a workspace", M,
                 N);
    return 0;
}

static int f32_join_blocks(int64_t items) {
    const int64_t blocks = (items + 255) / 256, most = 8 * (int64_t)somi_units();
    return (int)(blocks < 1 ? 1 : blocks < most ? blocks : most);
}

// x: [M, K], w: [N, K], bias: [N] or null, out: [M, N], all float32 and 16-byte aligned, K a multiple of 4; workspace:
// somi_linear_f32_planes(M, N) planes of [M, N] floats, 16-byte aligned, or null where that is 0.
extern "C" int somi_linear_f32(const float* x, const float* w, const float* bias, float* out, float* workspace, int M, int N, int K,
                               hipStream_t stream) {
    if (f32_check(x, w, bias, out, workspace, M, N, K)) return 1;
    if (M == 0) return 0;
    const int units = somi_units(), choice = f32_choice(M, N, units);
    if (choice == 0) {
        // One strip a workgroup until the strips fill the device twice, then two, which read x half as often; sixteen wavefronts
        // (one chain each) where strips are few and 64 KB hold their rows.
        const int strips = ceil_div(N, 16);
        const bool wide = strips >= 2 * units;
#define SOMI_F32_ROWS(W, MT, NS)                                                                                                    \
    hipLaunchKernelGGL((linear_f32_rows_kernel<W, MT, NS, 2, false>), dim3(ceil_div(strips, NS)), dim3(W * 64), 0, stream, x, w, bias, \
                       out, M, N, K)
        if (M <= 16 && !wide) SOMI_F32_ROWS(16, 1, 1);
        else if (M <= 16) SOMI_F32_ROWS(8, 1, 2);
        else if (!wide) SOMI_F32_ROWS(8, 2, 1);
        else SOMI_F32_ROWS(8, 2, 2);
#undef SOMI_F32_ROWS
        SOMI_LAUNCH_CHECK("linear_f32_rows");
        return 0;
    }
    float* planes = choice & 8 ? workspace : nullptr;
    if ((choice & 7) == 1) f32_launch_tile<2, 2, 2, 2, false>(x, w, bias, out, planes, M, N, K, stream);
    else f32_launch_tile<2, 4, 4, 2, false>(x, w, bias, out, planes, M, N, K, stream);
    SOMI_LAUNCH_CHECK("linear_f32_tile");
    if (planes != nullptr) {
        const int64_t count = (int64_t)M * N;
        hipLaunchKernelGGL(linear_f32_join_kernel, dim3(f32_join_blocks(count / 4)), dim3(256), 0, stream, planes, bias, out, count, N);
        SOMI_LAUNCH_CHECK("linear_f32_join");
    }
    return 0;
}

// out[m, n] = silu(x[m] . w[n]) * (x[m] . w[N + n]): w: [2 N, K] with the gate rows first, out: [M, N]; the rest as above, with a
// workspace for 2 N columns.  A row has the same bits as in somi_linear_f32 followed by the activation.
extern "C" int somi_linear_f32_gated(const float* x, const float* w, float* out, float* workspace, int M, int N, int K,
                                     hipStream_t stream) {
    SOMI_REQUIRE(N > 0 && N < (1 << 30), "linear_f32_gated: bad sizes M=%d N=%d K=%d", M, N, K);
    if (f32_check(x, w, nullptr, out, workspace, M, 2 * N, K)) return 1;
    SOMI_REQUIRE((int64_t)2 * N * K * 4 < (int64_t)1 << 31, "linear_f32_gated: the weight is too large (N=%d K=%d)", N, K);
    if (M == 0) return 0;
    const int choice = f32_choice(M, 2 * N, somi_units());
    if (choice == 0) {
        const dim3 grid(ceil_div(N, 16));
        if (M <= 16) hipLaunchKernelGGL((linear_f32_rows_kernel<8, 1, 2, 2, true>), grid, dim3(512), 0, stream, x, w, nullptr, out, M, N, K);
        else hipLaunchKernelGGL((linear_f32_rows_kernel<8, 2, 2, 2, true>), grid, dim3(512), 0, stream, x, w, nullptr, out, M, N, K);
        SOMI_LAUNCH_CHECK("linear_f32_rows");
        return 0;
    }
    if (choice & 8) {
        f32_launch_tile<2, 2, 2, 2, false>(x, w, nullptr, out, workspace, M, 2 * N, K, stream);
        const int64_t count = (int64_t)M * N;
        hipLaunchKernelGGL(linear_f32_join_gated_kernel, dim3(f32_join_blocks(count)), dim3(256), 0, stream, workspace, out, count, N);
    } else if (choice == 1) {
        f32_launch_tile<2, 2, 2, 2, true>(x, w, nullptr, out, nullptr, M, N, K, stream);
    } else {
        f32_launch_tile<2, 4, 4, 2, true>(x, w, nullptr, out, nullptr, M, N, K, stream);
    }
    SOMI_LAUNCH_CHECK("linear_f32_gated");
    return 0;
}
