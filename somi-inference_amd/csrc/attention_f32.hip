// Causal attention over cache pages in float32 on the matrix cores (v_mfma_f32_16x16x4_f32), for any mix of prompt portions and
// decoded tokens.
//
// Reference formulas: somi_inference/models/qwen2.py:158-186 (scores = q.k * D^-0.5, causal mask, float32 softmax,
// weights . v; query head h uses key/value head h // (nq / nkv)) and somi_inference/core/paged_attention.py:352-413.
//
// A query's result is the same bits whatever portion or batch its token arrives in.  Its keys lie in tiles of 32 (head sizes up to
// 64; 64 for larger ones) aligned to absolute positions.  A tile gives a maximum, a sum of weights relative to it and a weighted sum
// of values, each in one order; the tiles whose index is w modulo W = 16 (8) are joined in order, and so are the W results, w = 0
// first.  Every row of a matrix product is its own sum, so which queries share a tile's products does not matter.
//
// A workgroup of W wavefronts takes 16 (or 32) queries of one request and one key/value head: neighbouring tokens' heads
// of that group, so that a decoded token's heads and a prompt's tokens both fill rows.  Wavefront w walks the tiles w, w + W, ...;
// the W results meet in LDS.  (A tile is a chain of matrix instructions of one wavefront, so a request of some hundred
// keys takes as long as its tiles are wide: 4 requests of 512 keys, 14 heads of 64: 13.2 us, and about 16 with 64 keys and 8
// wavefronts; a prompt of 512 tokens 21.6 us, 2,048 144 us, 52 TFLOP/s; 28 heads of 128 471 us, 64 TFLOP/s.)  Keys are the A operand of the scores, so that a lane ends up with four neighbouring keys of one
// query, which is what the product with the values (stored by channel) takes as its B operand: weights never leave their registers.
// K and V come straight from memory in operand layout, 16 bytes a lane; workgroups share them through the caches.
//
// Few requests with long contexts leave compute units idle: their tiles are dealt out to `splits` workgroups by rounds of W,
// every tile's result goes to a workspace, and a second kernel joins them in the same order.
#include "attention_score.h"
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

// Keys of a tile, and wavefronts of a workgroup, for heads of D channels: more wavefronts have 128 registers each, which heads
// of more than 64 channels do not fit.
__host__ __device__ constexpr int af_tile(int D) { return D <= 64 ? 32 : 64; }
__host__ __device__ constexpr int af_waves(int D) { return D <= 64 ? 16 : 8; }
#define AF_MOST_WAVES 16
#define AF_MAX_TILES 2048                         // tiles of a request that the joining kernel holds

// Joins (mt, lt, ot) to (m, l, o): o = o a + ot b, l likewise.  A side without a key (-inf) gets the factor 0.
__device__ __forceinline__ void af_factors(float& m, float mt, float& a, float& b) {
    const float top = fmaxf(m, mt);
    a = m == -INFINITY ? 0.f : expf(m - top);
    b = mt == -INFINITY ? 0.f : expf(mt - top);
    m = top;
}
__device__ __forceinline__ float af_join(float o, float a, float ot, float b) { return __builtin_fmaf(ot, b, o * a); }

struct AfArgs {
    const float* q;
    int64_t q_stride;
    const float* kc;                              // [pages, nkv, page_size, D]
    const float* vc;                              // [pages, nkv, D, page_size]
    const int* table;
    int max_blocks;
    const int* entry_start;                       // [E + 1]
    const int* entry_first;                       // [E]
    int nq, nkv, page_size, page_shift;           // page_shift: log2 of the page size, or -1
    int window;
    float scale;
    float* out;
    float* part_o;                                // [queries, tiles, D] (queries: token * nq + head) or null
    float* part_ml;                               // [queries, tiles, 2]
    int splits, tiles;                            // tiles: the workspace's tiles a query
};

// NW: wavefronts of the workgroup, W or half of it; half of it takes the tiles of w and then those of w + W / 2.
template <int DT, int QB, int NW>
__global__ void __launch_bounds__(NW * 64)
attention_f32_kernel(const AfArgs p) {
    constexpr int D = DT * 16, AF_TILE = af_tile(D), AF_WAVES = af_waves(D), KB = AF_TILE / 16;
    static_assert(NW == AF_WAVES || (NW * 2 == AF_WAVES && QB == 1), "results of one block of queries in LDS at a time");
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int split = blockIdx.x % p.splits, block = blockIdx.x / p.splits;
    const int kvh = blockIdx.y, e = blockIdx.z;
    const int start = p.entry_start[e], G = p.nq / p.nkv;
    const int queries = (p.entry_start[e + 1] - start) * G;
    const int q0 = block * 16 * QB;
    if (q0 >= queries) return;
    const int first = p.entry_first[e];
    const int* table = p.table + (int64_t)e * p.max_blocks;

    // positions that the workgroup's queries see
    const int q_last = min(q0 + 16 * QB, queries) - 1;
    const int p_min = first + q0 / G, p_max = first + q_last / G;
    const int lo_min = score_first_key(p_min, p.window, 0), lo_max = score_first_key(p_max, p.window, 0);
    int64_t row[QB];                              // token * nq + head
    int pos[QB], lo[QB];
    f32x4 qf[QB][DT];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        const int flat = min(q0 + b * 16 + r, q_last);
        const int token = start + flat / G, head = kvh * G + flat % G;
        row[b] = (int64_t)token * p.nq + head;
        pos[b] = first + flat / G;
        lo[b] = score_first_key(pos[b], p.window, 0);
        const float* src = p.q + (int64_t)token * p.q_stride + (int64_t)head * D;
#pragma unroll
        for (int c = 0; c < DT; ++c) qf[b][c] = *reinterpret_cast<const f32x4*>(src + c * 16 + g * 4);
    }

    auto page_of = [&](int key) { return p.page_shift >= 0 ? key >> p.page_shift : key / p.page_size; };
    const int last_tile = p_max / AF_TILE, first_tile = lo_min / AF_TILE;
    int round = 0, round_end = last_tile / AF_WAVES + 1;
    if (p.splits > 1) {
        const int rounds = round_end;
        round = (int)((int64_t)split * rounds / p.splits);
        round_end = (int)((int64_t)(split + 1) * rounds / p.splits);
    }
    // [W][16][D + 4] sums of 16 queries at a time (rows padded against bank conflicts), and for every (w, query) its maximum, its sum of
    // weights and the two factors of its join
    float* so = lds;
    float* sm = lds + AF_WAVES * 16 * (D + 4);    // [W][16] maxima
    float* sl = sm + AF_WAVES * 16;               // [W][16] sums of weights
    float* sb = sl + AF_WAVES * 16;               // [W][16] factors of what came before
    float* sf = sb + AF_WAVES * 16;               // [W][16] factors of its own
    float* st = sf + AF_WAVES * 16;               // [16] the whole sums of weights
    float m[QB], l[QB];
    f32x4 o[QB][DT];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        m[b] = -INFINITY;
        l[b] = 0.f;
#pragma unroll
        for (int c = 0; c < DT; ++c) o[b][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto to_lds = [&](int b, int w) {
#pragma unroll
        for (int c = 0; c < DT; ++c) *reinterpret_cast<f32x4*>(so + (w * 16 + r) * (D + 4) + c * 16 + g * 4) = o[b][c];
        if (g == 0) {
            sm[w * 16 + r] = m[b];
            sl[w * 16 + r] = l[b];
        }
    };
    const int round_begin = round;
#pragma unroll 1
    for (int w = wave; w < AF_WAVES; w += NW) {
        if (w != wave) {                              // the second half: the first one's results go to their place
            to_lds(0, wave);
            m[0] = -INFINITY;
            l[0] = 0.f;
#pragma unroll
            for (int c = 0; c < DT; ++c) o[0][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (round = round_begin; round < round_end; ++round) {
            const int tile = round * AF_WAVES + w, k0 = tile * AF_TILE;
            if (tile < first_tile || tile > last_tile) continue;
            const bool inner = k0 >= lo_max && k0 + AF_TILE - 1 <= p_min;      // every query sees every key
            f32x4 s[QB][KB];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const int key = min(max(k0 + kb * 16 + r, lo_min), p_max);    // keys past either end: some key that is there
                const int page = page_of(key);
                const float* kr = p.kc + (((int64_t)table[page] * p.nkv + kvh) * p.page_size + (key - page * p.page_size)) * D + g * 4;
                f32x4 kf[DT];
#pragma unroll
                for (int c = 0; c < DT; ++c) kf[c] = *reinterpret_cast<const f32x4*>(kr + c * 16);
#pragma unroll
                for (int b = 0; b < QB; ++b) s[b][kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < DT; ++c)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int b = 0; b < QB; ++b)
                            s[b][kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][j], qf[b][c][j], s[b][kb], 0, 0, 0);
            }
            // where the values are: lane (r, g) takes channel c * 16 + r of keys 4 g .. 4 g + 3, 16 channels at a time; the first of them are
            // under way while the weights are made
            const float* vr[KB];
            bool there[KB][4];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const int want = k0 + kb * 16 + g * 4;
                const int key = min(max(want, lo_min & ~3), p_max & ~3), page = page_of(key);
                vr[kb] = p.vc + (((int64_t)table[page] * p.nkv + kvh) * D + r) * p.page_size + (key - page * p.page_size);
#pragma unroll
                for (int i = 0; i < 4; ++i) there[kb][i] = want + i >= lo_min && want + i <= p_max;
            }
            constexpr int AHEAD = QB == 2 ? 0 : DT > 12 ? 2 : DT < 4 ? DT : 4;
            f32x4 va[AHEAD > 0 ? AHEAD : 1][KB];
#pragma unroll
            for (int c = 0; c < AHEAD; ++c)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) va[c][kb] = *reinterpret_cast<const f32x4*>(vr[kb] + (int64_t)c * 16 * p.page_size);
            float mt[QB], lt[QB];
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                float top = -INFINITY;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = k0 + kb * 16 + g * 4 + i;
                        float v = s[b][kb][i] * p.scale;
                        if (!inner && (key < lo[b] || key > pos[b])) v = -INFINITY;
                        s[b][kb][i] = v;
                        top = fmaxf(top, v);
                    }
                top = fmaxf(top, __shfl_xor(top, 16, 64));
                top = fmaxf(top, __shfl_xor(top, 32, 64));
                float sum = 0.f;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float wgt = top == -INFINITY ? 0.f : expf(s[b][kb][i] - top);
                        s[b][kb][i] = wgt;
                        sum += wgt;
                    }
                sum += __shfl_xor(sum, 16, 64);
                sum += __shfl_xor(sum, 32, 64);
                mt[b] = top;
                lt[b] = sum;
            }
            float a[QB], f[QB];
#pragma unroll
            for (int b = 0; b < QB; ++b) {
                if (p.splits == 1) {
                    af_factors(m[b], mt[b], a[b], f[b]);
                    l[b] = af_join(l[b], a[b], lt[b], f[b]);
                } else {
                    m[b] = mt[b];
                    l[b] = lt[b];
                }
            }
#pragma unroll
            for (int c = 0; c < DT; ++c) {
                f32x4 vf[KB];
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
                    vf[kb] = c < AHEAD ? va[c < AHEAD ? c : 0][kb] : *reinterpret_cast<const f32x4*>(vr[kb] + (int64_t)c * 16 * p.page_size);
                if (!inner) {                         // a key that is not there has weight 0, but its place may hold anything
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                        for (int i = 0; i < 4; ++i) vf[kb][i] = there[kb][i] ? vf[kb][i] : 0.f;
                }
                f32x4 ot[QB];
#pragma unroll
                for (int b = 0; b < QB; ++b) ot[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int b = 0; b < QB; ++b)
                            ot[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[kb][i], s[b][kb][i], ot[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < QB; ++b) {
                    if (p.splits == 1) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) o[b][c][i] = af_join(o[b][c][i], a[b], ot[b][i], f[b]);
                    } else if (q0 + b * 16 + r < queries) {
                        *reinterpret_cast<f32x4*>(p.part_o + (row[b] * p.tiles + tile) * D + c * 16 + g * 4) = ot[b];
                    }
                }
            }
            if (p.splits > 1) {
#pragma unroll
                for (int b = 0; b < QB; ++b)
                    if (g == 0 && q0 + b * 16 + r < queries) {
                        p.part_ml[(row[b] * p.tiles + tile) * 2] = m[b];
                        p.part_ml[(row[b] * p.tiles + tile) * 2 + 1] = l[b];
                    }
            }
        }
    }
    if (p.splits > 1) return;

    // the W results in order
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        if (b > 0) __syncthreads();
        to_lds(b, NW == AF_WAVES ? wave : wave + NW);
        __syncthreads();
        for (int item = threadIdx.x; item < AF_WAVES * 16; item += NW * 64) {
            // the factors of every (w, query) side by side: what came before has the largest maximum before it
            float before = -INFINITY, a, f;
            for (int w = 0; w < item >> 4; ++w) before = fmaxf(before, sm[w * 16 + (item & 15)]);
            af_factors(before, sm[item], a, f);
            sb[item] = a;
            sf[item] = f;
        }
        __syncthreads();
        if (threadIdx.x < 16) {
            float whole = 0.f;
#pragma unroll
            for (int w = 0; w < AF_WAVES; ++w)
                whole = af_join(whole, sb[w * 16 + threadIdx.x], sl[w * 16 + threadIdx.x], sf[w * 16 + threadIdx.x]);
            st[threadIdx.x] = whole;
        }
        __syncthreads();
        for (int idx = threadIdx.x; idx < 16 * D; idx += NW * 64) {
            const int query = idx / D, d = idx % D, flat = q0 + b * 16 + query;
            if (flat >= queries) continue;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < AF_WAVES; ++w)
                v = af_join(v, sb[w * 16 + query], so[(w * 16 + query) * (D + 4) + d], sf[w * 16 + query]);
            p.out[((int64_t)(start + flat / G) * p.nq + kvh * G + flat % G) * D + d] = v / st[query];
        }
    }
}

// One workgroup a (token, head): the tiles' results of the workspace in the order of the kernel above.  positions: [tokens].
__global__ void __launch_bounds__(256)
attention_f32_join_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ positions,
                          int nq, int D, int tiles, int window, float* __restrict__ out) {
    __shared__ float before[AF_MAX_TILES], own[AF_MAX_TILES];
    __shared__ float wm[AF_MOST_WAVES], wl[AF_MOST_WAVES], wbefore[AF_MOST_WAVES], wown[AF_MOST_WAVES], whole;
    const int AF_TILE = af_tile(D), AF_WAVES = af_waves(D);
    const int token = blockIdx.x, tid = threadIdx.x;
    const int64_t row = (int64_t)token * nq + blockIdx.y;
    const int p = positions[token], n = p / AF_TILE + 1, first = score_first_key(p, window, 0) / AF_TILE;
    const float* ml = part_ml + row * tiles * 2;
    if (tid < AF_WAVES) {
        float m = -INFINITY, l = 0.f;
        for (int t = tid; t < n; t += AF_WAVES) {
            if (t < first) continue;
            float a, b;
            af_factors(m, ml[t * 2], a, b);
            l = af_join(l, a, ml[t * 2 + 1], b);
            before[t] = a;
            own[t] = b;
        }
        wm[tid] = m;
        wl[tid] = l;
    }
    __syncthreads();
    if (tid == 0) {
        float m = -INFINITY, l = 0.f;
        for (int w = 0; w < AF_WAVES; ++w) {
            af_factors(m, wm[w], wbefore[w], wown[w]);
            l = af_join(l, wbefore[w], wl[w], wown[w]);
        }
        whole = l;
    }
    __syncthreads();
    for (int d = tid; d < D; d += 256) {
        const float* src = part_o + row * tiles * D + d;
        float v = 0.f;
        for (int w = 0; w < AF_WAVES; ++w) {
            float o = 0.f;
            for (int t = w; t < n; t += AF_WAVES)
                if (t >= first) o = af_join(o, before[t], src[(int64_t)t * D], own[t]);
            v = af_join(v, wbefore[w], o, wown[w]);
        }
        out[row * D + d] = v / whole;
    }
}

extern "C" int somi_attention_f32_supported(int D, int page_size) {
    const bool sizes = D % 16 == 0 && D > 0 && (D <= 96 || D == 128 || D == 160 || D == 192 || D == 256);
    return sizes && page_size > 0 && page_size % 4 == 0;
}

extern "C" int somi_attention_f32_tile(int D) { return af_tile(D); }

// How many workgroups share a query's tiles when `blocks` workgroups would run on `units` compute units and a request has up to
// `max_context` keys: as many as fill the device, but two rounds of tiles (512 keys each) at least.  A joining kernel costs about 4 us,
// a round of tiles 2 to 4.
extern "C" int somi_attention_f32_splits(int blocks, int max_context, int D, int units) {
    const int tiles = ceil_div(max_context, af_tile(D)), rounds = ceil_div(tiles, af_waves(D));
    if (blocks <= 0 || tiles > AF_MAX_TILES || rounds < 4) return 1;
    const int splits = units / blocks < rounds / 2 ? units / blocks : rounds / 2;
    return splits > 1 ? splits : 1;
}

template <int DT, int QB, int NW>
static int af_launch(const AfArgs& a, int blocks, int n_entries, hipStream_t stream) {
    constexpr int waves = af_waves(DT * 16);
    const size_t smem = (size_t)(waves * 16 * (DT * 16 + 4) + 4 * waves * 16 + 16) * sizeof(float);
    if (smem > 64 * 1024)
        (void)hipFuncSetAttribute((const void*)attention_f32_kernel<DT, QB, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipLaunchKernelGGL((attention_f32_kernel<DT, QB, NW>), dim3(blocks * a.splits, a.nkv, n_entries), dim3(NW * 64), smem, stream, a);
    SOMI_LAUNCH_CHECK("attention_f32");
    return 0;
}

// D up to 64: W wavefronts a workgroup while a compute unit has one workgroup, half of them (two workgroups a unit) beyond.  Larger
// heads: 32 queries a workgroup where 16 would give every unit four workgroups, so keys and values are read half as often.
template <int DT>
static int af_dispatch(const AfArgs& a, int64_t queries, int n_entries, hipStream_t stream) {
    const int blocks = (int)((queries + 15) / 16);
    const int64_t workgroups = (int64_t)blocks * a.splits * a.nkv * n_entries;
    constexpr int W = af_waves(DT * 16);
    if constexpr (W == 16) {
        if (workgroups > somi_units()) return af_launch<DT, 1, W / 2>(a, blocks, n_entries, stream);
    } else if constexpr (DT <= 8) {
        if (a.splits == 1 && workgroups >= 4 * (int64_t)somi_units()) return af_launch<DT, 2, W>(a, (int)((queries + 31) / 32), n_entries, stream);
    }
    return af_launch<DT, 1, W>(a, blocks, n_entries, stream);
}

// q: token t's head h starts at q + t * q_stride + h * D.  k_cache: [pages, nkv, page_size, D]; v_cache: [pages, nkv, D, page_size];
// block_table: [n_entries, max_blocks]; entry_start: [n_entries + 1] offsets of the entries' tokens, entry_first: [n_entries] the
// position of each one's first token, positions: [n_tokens]; max_entry_len: the longest entry; max_context: keys that a request has
// at most.  All float32, q, k and v 16-byte aligned, q_stride a multiple of 4.  With splits > 1 (somi_attention_f32_splits, or fewer)
// part_o holds n_tokens * nq * tiles * D floats and part_ml n_tokens * nq * tiles * 2, tiles = ceil(max_context /
// somi_attention_f32_tile(D)).
extern "C" int somi_attention_f32(const float* q, int64_t q_stride, const float* k_cache, const float* v_cache, const int* block_table,
                                  int max_blocks, const int* entry_start, const int* entry_first, const int* positions, int n_tokens,
                                  int n_entries, int max_entry_len, int max_context, int nq, int nkv, int D, int page_size, int window,
                                  float scale, int splits, float* part_o, float* part_ml, float* out, hipStream_t stream) {
    SOMI_REQUIRE(n_tokens >= 0 && n_entries >= 0 && max_entry_len >= 0 && nq > 0 && nkv > 0 && max_blocks > 0 && max_context >= 0,
                 "attention_f32: bad sizes");
    SOMI_REQUIRE(nq % nkv == 0, "attention_f32: num_q_heads (%d) must be divisible by num_kv_heads (%d)", nq, nkv);
    SOMI_REQUIRE(somi_attention_f32_supported(D, page_size), "attention_f32: head size %d, pages of %d", D, page_size);
    SOMI_REQUIRE(window >= 0, "attention_f32: window must be >= 0");
    SOMI_REQUIRE((((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15) == 0 && q_stride % 4 == 0,
                 "attention_f32: q, k, v and out must be 16-byte aligned");
    const int tiles = ceil_div(max_context, af_tile(D));
    SOMI_REQUIRE(splits == 1 || (splits > 1 && part_o && part_ml && tiles <= AF_MAX_TILES), "attention_f32: %d splits of %d keys", splits,
                 max_context);
    if (n_tokens == 0 || n_entries == 0 || max_entry_len == 0) return 0;
    const int G = nq / nkv;
    const int64_t queries = (int64_t)max_entry_len * G;
    SOMI_REQUIRE(queries <= (1 << 30) && nkv <= 65535 && n_entries <= 65535, "attention_f32: too many queries, heads or entries");
    int shift = -1;
    for (int b = 0; b < 30; ++b)
        if (page_size == 1 << b) shift = b;
    const AfArgs a{q, q_stride, k_cache, v_cache, block_table, max_blocks, entry_start, entry_first, nq, nkv, page_size, shift, window,
                   scale, out, part_o, part_ml, splits, tiles};
    int rc = 1;
#define SOMI_AF(DT)                                              \
    case DT:                                                     \
        rc = af_dispatch<DT>(a, queries, n_entries, stream);     \
        break
    switch (D / 16) {
        SOMI_AF(1); SOMI_AF(2); SOMI_AF(3); SOMI_AF(4); SOMI_AF(5); SOMI_AF(6); SOMI_AF(8); SOMI_AF(10); SOMI_AF(12); SOMI_AF(16);
        default: return somi_fail("attention_f32: head size %d", D);
    }
#undef SOMI_AF
    if (rc != 0 || splits == 1) return rc;
    hipLaunchKernelGGL(attention_f32_join_kernel, dim3(n_tokens, nq), dim3(256), 0, stream, part_o, part_ml, positions, nq, D, tiles,
                       window, out);
    SOMI_LAUNCH_CHECK("attention_f32_join");
    return 0;
}
