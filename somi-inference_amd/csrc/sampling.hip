// Token choice from float32 logits: greedy argmax, or a draw from softmax(logits / T).
//
// Reference: somi_inference/core/sampler.py:104-114 (logits /= T when T > 0), :159-176 (T == 0: argmax,
// else float32 softmax and one multinomial draw) and :80-102 (repetition penalty: a positive logit is
// divided by the penalty, a non-positive one multiplied).  The draw here is by inverse CDF from a uniform
// number that the host derives from the request's own seed and token count, so a request's tokens do not
// depend on what else is in the batch.
#include "common.h"
#include "no_alloc.h"

#include <mutex>

// The vocabulary is cut into chunks of SAMPLE_CHUNK entries; one workgroup per (row, chunk) finds the
// chunk's maximum, its first index and (for a draw) the chunk's softmax mass relative to that maximum.  A
// second kernel, one workgroup per row, merges the chunks in index order, locates the chunk that holds the
// target mass u * total, and walks that chunk once more to pick the entry.  Chunk boundaries depend on the
// vocabulary only, so a row's token does not depend on the batch.
#define SAMPLE_NT 256
#define SAMPLE_PER_THREAD 8
#define SAMPLE_CHUNK (SAMPLE_NT * SAMPLE_PER_THREAD)

// What a row's top-k and top-p rules leave, as a place in its descending order: entries with a larger key than `key` and, of those
// with that key, the ones up to index `last`.  (The sampling kernels read the row through it, so nothing is written to the row.)
struct SampleCut {
    unsigned key;
    int last;
};
#define SAMPLE_KEEP_ALL SampleCut{0u, 0x7fffffff}

// value order == unsigned order of the key
__device__ __forceinline__ unsigned filter_key(float v) {
    const unsigned bits = __float_as_uint(v);
    return (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
}
__device__ __forceinline__ float filter_value(unsigned key) {
    return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}
__device__ __forceinline__ bool cut_keeps(const SampleCut& cut, unsigned key, int i) {
    return key > cut.key || (key == cut.key && i <= cut.last);
}

// Entries begin .. begin + SAMPLE_PER_THREAD - 1 of a row, -inf where the row ends or its cut took them.  `quads`: rows begin
// on 16 bytes and are a multiple of four entries (sample_quads), so they are read four at a time.
__device__ __forceinline__ void sample_read(const float* __restrict__ z, int vocab, int begin, const SampleCut& cut, bool quads,
                                            float (&v)[SAMPLE_PER_THREAD]) {
    if (quads) {
#pragma unroll
        for (int j = 0; j < SAMPLE_PER_THREAD; j += 4) {
            float4 four = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
            if (begin + j < vocab) four = *reinterpret_cast<const float4*>(z + begin + j);
            v[j] = four.x;
            v[j + 1] = four.y;
            v[j + 2] = four.z;
            v[j + 3] = four.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < SAMPLE_PER_THREAD; ++j) v[j] = begin + j < vocab ? z[begin + j] : -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < SAMPLE_PER_THREAD; ++j)
        if (!cut_keeps(cut, filter_key(v[j]), begin + j)) v[j] = -INFINITY;
}

__global__ void __launch_bounds__(SAMPLE_NT)
sample_chunks_kernel(const float* __restrict__ logits, int vocab, int chunks, const float* __restrict__ temperature,
                     const SampleCut* __restrict__ cuts, bool quads, float* __restrict__ part /*[rows, chunks, 3]: max, first index (as int bits), mass*/) {
    __shared__ float red[16];
    __shared__ float vals[SAMPLE_NT];
    __shared__ int idxs[SAMPLE_NT];
    const int row = blockIdx.y, chunk = blockIdx.x, tid = threadIdx.x;
    const float* z = logits + (int64_t)row * vocab;
    const float temp = temperature[row];
    const float inv_unit = temp > 0.f ? temp : 1.f;        // greedy compares the logits themselves
    const int begin = chunk * SAMPLE_CHUNK + tid * SAMPLE_PER_THREAD;
    float v[SAMPLE_PER_THREAD];
    sample_read(z, vocab, begin, cuts ? cuts[row] : SAMPLE_KEEP_ALL, quads, v);
    float best = -INFINITY;
    int best_i = vocab;
#pragma unroll
    for (int j = 0; j < SAMPLE_PER_THREAD; ++j) {
        const int i = begin + j;
        v[j] = i < vocab ? v[j] / inv_unit : -INFINITY;
        if (i < vocab && (v[j] > best || best_i == vocab)) { best = v[j]; best_i = i; }
    }
    vals[tid] = best;
    idxs[tid] = best_i;
    __syncthreads();
    for (int step = SAMPLE_NT / 2; step > 0; step >>= 1) {
        if (tid < step) {
            const float ov = vals[tid + step];
            const int oi = idxs[tid + step];
            const bool take = oi < vocab && (idxs[tid] == vocab || ov > vals[tid] || (ov == vals[tid] && oi < idxs[tid]));
            if (take) { vals[tid] = ov; idxs[tid] = oi; }
        }
        __syncthreads();
    }
    const float chunk_max = vals[0];
    float mass = 0.f;
    if (temp > 0.f) {
#pragma unroll
        for (int j = 0; j < SAMPLE_PER_THREAD; ++j)
            if (begin + j < vocab) mass += expf(v[j] - chunk_max);
        mass = block_sum<SAMPLE_NT>(mass, red);
    }
    if (tid == 0) {
        float* p = part + ((int64_t)row * chunks + chunk) * 3;
        p[0] = chunk_max;
        p[1] = __int_as_float(idxs[0]);
        p[2] = mass;
    }
}

__global__ void __launch_bounds__(SAMPLE_NT)
sample_pick_kernel(const float* __restrict__ logits, int vocab, int chunks, const float* __restrict__ temperature,
                   const float* __restrict__ uniform, const SampleCut* __restrict__ cuts, bool quads, const float* __restrict__ part,
                   int* __restrict__ out) {
    __shared__ float sums[SAMPLE_NT];
    __shared__ float s_before, s_target, s_max;
    __shared__ int s_chunk, s_owner;
    // a piece of the chunks' results at a time: the additions over the chunks are one thread's, in order, but reading them and
    // their exponentials is everybody's (one thread alone took 38 us for 75 chunks)
    __shared__ float c_mass[SAMPLE_NT], c_scale[SAMPLE_NT];
    __shared__ float red[16];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float* z = logits + (int64_t)row * vocab;
    const float* p = part + (int64_t)row * chunks * 3;
    const float temp = temperature[row];
    float mx = -INFINITY;
    for (int c = tid; c < chunks; c += SAMPLE_NT) mx = fmaxf(mx, p[c * 3]);
    mx = block_max<SAMPLE_NT>(mx, red);
    if (p[0] != p[0]) mx = p[0];                            // a first chunk whose maximum is NaN stays the maximum
    if (temp == 0.f) {
        // the first maximum in index order; where none compares equal (NaN) the first chunk's
        int first = chunks;
        for (int c = tid; c < chunks; c += SAMPLE_NT)
            if (p[c * 3] == mx && c < first) first = c;
        const float least = -block_max<SAMPLE_NT>(-(float)first, red);
        if (tid == 0) out[row] = __float_as_int(p[(least < (float)chunks ? (int)least : 0) * 3 + 1]);
        return;
    }
    float total = 0.f, run = 0.f, target = 0.f;
    int owner = -1, last_nonzero = 0;
    for (int pass = 0; pass < 2; ++pass) {
        for (int base = 0; base < chunks; base += SAMPLE_NT) {
            const int here = min(SAMPLE_NT, chunks - base);
            __syncthreads();
            if (tid < here) {
                c_mass[tid] = p[(base + tid) * 3 + 2];
                c_scale[tid] = expf(p[(base + tid) * 3] - mx);
            }
            __syncthreads();
            if (tid != 0) continue;
            if (pass == 0) {
#pragma unroll 8
                for (int c = 0; c < here; ++c) total += c_mass[c] * c_scale[c];
            } else {
                for (int c = 0; c < here; ++c) {
                    const float mass = c_mass[c] * c_scale[c];
                    if (mass > 0.f) last_nonzero = base + c;
                    if (owner < 0 && target < run + mass) { owner = base + c; s_before = run; }
                    run += mass;
                }
            }
        }
        target = uniform[row] * total;
    }
    if (tid == 0) {
        if (owner < 0) {                                    // rounding pushed the target past the total
            owner = last_nonzero;
            s_before = -INFINITY;                           // take the chunk's last entry with mass
        }
        s_chunk = owner;
        s_target = target;
        s_max = mx;
    }
    __syncthreads();
    const int begin = s_chunk * SAMPLE_CHUNK + tid * SAMPLE_PER_THREAD;
    float w[SAMPLE_PER_THREAD];
    float mine = 0.f;
    sample_read(z, vocab, begin, cuts ? cuts[row] : SAMPLE_KEEP_ALL, quads, w);
#pragma unroll
    for (int j = 0; j < SAMPLE_PER_THREAD; ++j) {
        w[j] = begin + j < vocab ? expf(w[j] / temp - s_max) : 0.f;
        mine += w[j];
    }
    sums[tid] = mine;
    __syncthreads();
    if (tid == 0) {
        const bool overshoot = s_before == -INFINITY;
        float run = overshoot ? 0.f : s_before;
        int owner = -1, last_nonzero = 0;
#pragma unroll 16
        for (int k = 0; k < SAMPLE_NT; ++k) {
            const float mass = sums[k];
            sums[k] = run;
            if (mass > 0.f) last_nonzero = k;
            if (!overshoot && owner < 0 && s_target < run + mass) owner = k;
            run += mass;
        }
        s_owner = owner < 0 ? last_nonzero : owner;
    }
    __syncthreads();
    if (tid == s_owner) {
        float run = sums[tid];
        int pick = -1, last = begin;
#pragma unroll
        for (int j = 0; j < SAMPLE_PER_THREAD; ++j) {
            if (w[j] > 0.f) last = begin + j;
            run += w[j];
            if (pick < 0 && s_before != -INFINITY && run > s_target) pick = begin + j;
        }
        out[row] = pick < 0 ? last : pick;
    }
}

static bool sample_quads(const void* logits, int vocab) { return vocab % 4 == 0 && (uintptr_t)logits % 16 == 0; }

extern "C" int somi_sample_workspace_floats(int rows, int vocab) {
    return rows * ceil_div(vocab, SAMPLE_CHUNK) * 3;
}

// logits: [rows, vocab] float32; temperature, uniform: [rows] float32 (uniform in [0, 1)); cuts: [rows] of what somi_sample_cuts
// found, or null; out: [rows] int32; workspace: somi_sample_workspace_floats(rows, vocab) floats.
extern "C" int somi_sample_through(const float* logits, int rows, int vocab, const float* temperature, const float* uniform,
                                   const void* cuts, int* out, float* workspace, hipStream_t stream) {
    SOMI_REQUIRE(rows >= 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", rows, vocab);
    SOMI_REQUIRE(rows <= 65535, "sample: too many rows");
    SOMI_REQUIRE(workspace != nullptr || rows == 0, "sample: a workspace is needed");
    if (rows == 0) return 0;
    const bool quads = sample_quads(logits, vocab);
    const int chunks = ceil_div(vocab, SAMPLE_CHUNK);
    hipLaunchKernelGGL(sample_chunks_kernel, dim3(chunks, rows), dim3(SAMPLE_NT), 0, stream, logits, vocab, chunks,
                       temperature, (const SampleCut*)cuts, quads, workspace);
    SOMI_LAUNCH_CHECK("sample_chunks");
    hipLaunchKernelGGL(sample_pick_kernel, dim3(rows), dim3(SAMPLE_NT), 0, stream, logits, vocab, chunks, temperature,
                       uniform, (const SampleCut*)cuts, quads, workspace, out);
    SOMI_LAUNCH_CHECK("sample_pick");
    return 0;
}

extern "C" int somi_sample(const float* logits, int rows, int vocab, const float* temperature,
                           const float* uniform, int* out, float* workspace, hipStream_t stream) {
    return somi_sample_through(logits, rows, vocab, temperature, uniform, nullptr, out, workspace, stream);
}

// The workspace of somi_sample_no_alloc: one array per GPU, held until the process ends.  In host code the
// array's name is only a handle for hipGetSymbolAddress; the address it yields differs from GPU to GPU and is
// what the kernels get.
static __device__ __align__(256) float scratch[SOMI_SAMPLE_SCRATCH_FLOATS];

#define SOMI_MAX_DEVICES 64
static float* g_scratch_ptr[SOMI_MAX_DEVICES];      // the array's address on each device, once asked for
static std::mutex g_scratch_mutex;

// The address of `scratch` on the current device (asked for once per device, with that device current).
static int scratch_on_current_device(float** ptr) {
    int device = -1;
    hipError_t err = hipGetDevice(&device);
    SOMI_REQUIRE(err == hipSuccess, "sample_no_alloc: hipGetDevice: %s", hipGetErrorString(err));
    SOMI_REQUIRE(device >= 0 && device < SOMI_MAX_DEVICES, "sample_no_alloc: device %d is beyond the %d this library "
                 "keeps a workspace for", device, SOMI_MAX_DEVICES);
    std::lock_guard<std::mutex> hold(g_scratch_mutex);
    if (g_scratch_ptr[device] == nullptr) {
        float* found = nullptr;
        err = hipGetSymbolAddress((void**)&found, HIP_SYMBOL(scratch));
        SOMI_REQUIRE(err == hipSuccess && found != nullptr, "sample_no_alloc: hipGetSymbolAddress on device %d: %s",
                     device, hipGetErrorString(err));
        g_scratch_ptr[device] = found;
    }
    *ptr = g_scratch_ptr[device];
    return 0;
}

extern "C" int somi_sample_no_alloc_capacity() { return SOMI_SAMPLE_SCRATCH_FLOATS; }

extern "C" int somi_sample_no_alloc(const float* logits, int rows, int vocab, const float* temperature,
                                    const float* uniform, int* out, hipStream_t stream) {
    SOMI_REQUIRE(rows >= 0 && vocab > 0, "sample_no_alloc: bad sizes rows=%d vocab=%d", rows, vocab);
    SOMI_REQUIRE(rows <= 65535, "sample_no_alloc: too many rows");
    if (rows == 0) return 0;
    SOMI_REQUIRE(logits && temperature && uniform && out, "sample_no_alloc: a null pointer among the arguments");
    const int64_t need = (int64_t)rows * ceil_div(vocab, SAMPLE_CHUNK) * 3;
    SOMI_REQUIRE(need <= SOMI_SAMPLE_SCRATCH_FLOATS,
                 "sample_no_alloc: %d rows of %d logits need %lld floats of workspace, the fixed one holds %d "
                 "(rows * ceil(vocab / %d) * 3 must not exceed it); use somi_sample with a workspace of your own",
                 rows, vocab, (long long)need, SOMI_SAMPLE_SCRATCH_FLOATS, SAMPLE_CHUNK);
    float* workspace = nullptr;
    if (scratch_on_current_device(&workspace) != 0) return 1;
    // every (row, chunk) triple that the second kernel reads is written by the first: nothing to clear
    return somi_sample(logits, rows, vocab, temperature, uniform, out, workspace, stream);
}

// logits[row, id] = logit > 0 ? logit / penalty : logit * penalty for each listed id (ids must be distinct).
__global__ void __launch_bounds__(256)
penalty_kernel(float* __restrict__ logits, int vocab, const int* __restrict__ ids, int n_ids, float penalty) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_ids) return;
    const int id = ids[i];
    if (id < 0 || id >= vocab) return;
    const float v = logits[id];
    logits[id] = v > 0.f ? v / penalty : v * penalty;
}

extern "C" int somi_repetition_penalty(float* logits_row, int vocab, const int* ids, int n_ids, float penalty,
                                       hipStream_t stream) {
    SOMI_REQUIRE(vocab > 0 && n_ids >= 0, "repetition_penalty: bad sizes");
    SOMI_REQUIRE(penalty > 0.f, "repetition_penalty: penalty must be > 0, got %g", (double)penalty);
    if (n_ids == 0) return 0;
    hipLaunchKernelGGL(penalty_kernel, dim3(ceil_div(n_ids, 256)), dim3(256), 0, stream, logits_row, vocab, ids,
                       n_ids, penalty);
    SOMI_LAUNCH_CHECK("repetition_penalty");
    return 0;
}

// The same rule for several rows at once, from one tensor into another (or in place): the ids of row r are
// ids[offsets[r] .. offsets[r + 1]), each counted once however often it is listed; a row with penalty 1 or no ids is copied.  A
// workgroup marks the ids of its piece of the row in LDS and passes the piece through once.
#define PENALTY_PIECE 4096
__global__ void __launch_bounds__(256)
penalty_rows_kernel(const float* logits, float* out, int vocab, bool quads, const int* __restrict__ offsets,
                    const int* __restrict__ ids, const float* __restrict__ penalties) {
    __shared__ unsigned marked[PENALTY_PIECE / 32];
    const int row = blockIdx.y, begin = blockIdx.x * PENALTY_PIECE, end = min(vocab, begin + PENALTY_PIECE), tid = threadIdx.x;
    const int first = offsets[row], last = offsets[row + 1];
    const float penalty = penalties[row];
    if (tid < PENALTY_PIECE / 32) marked[tid] = 0;
    __syncthreads();
    if (penalty != 1.0f)
        for (int i = first + tid; i < last; i += 256) {
            const int id = ids[i];
            if (id >= begin && id < end) atomicOr(&marked[(id - begin) >> 5], 1u << ((id - begin) & 31));
        }
    __syncthreads();
    const float* from = logits + (int64_t)row * vocab;
    float* to = out + (int64_t)row * vocab;
    auto passed = [&](float v, int i) {
        if (!((marked[(i - begin) >> 5] >> ((i - begin) & 31)) & 1u)) return v;
        return v > 0.f ? v / penalty : v * penalty;
    };
    if (quads) {
        for (int i = begin + tid * 4; i < end; i += 1024) {
            float4 v = *reinterpret_cast<const float4*>(from + i);
            v.x = passed(v.x, i);
            v.y = passed(v.y, i + 1);
            v.z = passed(v.z, i + 2);
            v.w = passed(v.w, i + 3);
            *reinterpret_cast<float4*>(to + i) = v;
        }
        return;
    }
    for (int i = begin + tid; i < end; i += 256) to[i] = passed(from[i], i);
}

// logits, out: [rows, vocab] float32 (the same tensor: in place); offsets: [rows + 1] int32 (ascending from 0); ids:
// [offsets[rows]] int32; penalties: [rows] float32, each > 0 (checked by the caller, who holds them on the host).
extern "C" int somi_repetition_penalty_rows(const float* logits, float* out, int rows, int vocab, const int* offsets,
                                            const int* ids, const float* penalties, hipStream_t stream) {
    SOMI_REQUIRE(rows >= 0 && vocab > 0, "repetition_penalty_rows: bad sizes");
    SOMI_REQUIRE(rows <= 65535, "repetition_penalty_rows: too many rows");
    if (rows == 0) return 0;
    hipLaunchKernelGGL(penalty_rows_kernel, dim3(ceil_div(vocab, PENALTY_PIECE), rows), dim3(256), 0, stream, logits, out, vocab,
                       sample_quads(logits, vocab) && sample_quads(out, vocab), offsets, ids, penalties);
    SOMI_LAUNCH_CHECK("repetition_penalty_rows");
    return 0;
}

// ---------------------------------------------------------------------------------------------------------
// Top-k and top-p masks (somi_inference/core/sampler.py:116-157), without sorting the row.
//
// Both rules keep a prefix of the row in descending order (equal entries in index order): top-k the first k entries; top-p, on
// softmax(z / T) of what top-k left, every entry whose predecessors hold a mass of at most p (so the entry that crosses p
// stays and the first entry is never removed, sampler.py:150-153).  Masses are integers (softmax mass in units of 2^-40 of the
// largest entry's), so sums do not depend on the order of additions and a row's result does not depend on timing or on the batch.
// One workgroup a row finds the last entry that stays; the kernels behind it read the row through that cut.
//
// Up to CUT_SORTED entries, the common top-k, take two passes over the row: every thread's (or four threads') largest entry, whose k-th largest bounds
// the row's k-th largest from below, then the few entries from that bound on into LDS, where they are put in order and top-p
// is a prefix sum.  (With equal or clustered entries more may pass the bound than LDS holds; then the search below.)  Everything
// else is a radix search for the entry at which the running weight (1, or mass) first exceeds a target, twelve bits
// of an order-preserving key at a time: a histogram of the weights, and the entries of the bin in which the running weight
// crosses go to LDS if they fit, so that the remaining bits need no further pass over the row.  64 rows of 152,064 logits, k = 50 and
// p = 0.95: 49 us; four passes of eight bits a rule, and one that wrote -inf over what the rule removed, took 375.
#define FILTER_NT 1024
#define FILTER_WAVES (FILTER_NT / 64)
#define CUT_SORTED 512                    // largest k of the sorted form
#define CUT_CANDIDATES 2048               // entries from the bound on that it holds
#define CUT_BINS 4096
#define CUT_LIST 7168                     // keys of the crossing bin that the search holds
typedef unsigned long long filter_u64;

__device__ __forceinline__ filter_u64 filter_mass(float v, float temp, float zmax) {
    return (filter_u64)(expf(v / temp - zmax) * 1099511627776.0f);           // 2^40; expf(-inf) = 0
}

struct CutShared {
    union {
        filter_u64 hist[CUT_BINS];
        unsigned largest[FILTER_NT];
        struct { unsigned key[CUT_SORTED]; int index[CUT_SORTED]; } sorted;
    };
    union {
        unsigned list[CUT_LIST];
        struct { unsigned key[CUT_CANDIDATES]; int index[CUT_CANDIDATES]; } candidate;
    };
    filter_u64 wave_sum[FILTER_WAVES];
    filter_u64 above, group;
    unsigned bound, count, wave_count[FILTER_WAVES];
    int bin, place;
};

// Calls f(value, index) for every entry of the row, several loads under way at a time.
struct CutRow {
    const float* at;
    int vocab;
    bool quads;
};
template <typename F>
__device__ __forceinline__ void cut_walk(const CutRow& r, F f) {
    constexpr int AHEAD = 8;
    const float* row = r.at;
    const int vocab = r.vocab;
    if (r.quads) {
        const int quads = vocab / 4;
        for (int base = 0; base < quads; base += AHEAD * FILTER_NT) {
            float4 v[AHEAD];
#pragma unroll
            for (int a = 0; a < AHEAD; ++a) {
                const int i = base + a * FILTER_NT + threadIdx.x;
                if (i < quads) v[a] = reinterpret_cast<const float4*>(row)[i];
            }
#pragma unroll
            for (int a = 0; a < AHEAD; ++a) {
                const int i = base + a * FILTER_NT + threadIdx.x;
                if (i < quads) {
                    f(v[a].x, i * 4);
                    f(v[a].y, i * 4 + 1);
                    f(v[a].z, i * 4 + 2);
                    f(v[a].w, i * 4 + 3);
                }
            }
        }
        return;
    }
    for (int base = 0; base < vocab; base += AHEAD * FILTER_NT) {
        float v[AHEAD];
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            const int i = base + a * FILTER_NT + threadIdx.x;
            if (i < vocab) v[a] = row[i];
        }
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            const int i = base + a * FILTER_NT + threadIdx.x;
            if (i < vocab) f(v[a], i);
        }
    }
}

// The sum of `mine` over the threads before this one; `total`: over all of them.  Two barriers.
__device__ __forceinline__ filter_u64 cut_before(filter_u64 mine, filter_u64& total, CutShared& sh) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    filter_u64 incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const filter_u64 other = __shfl_up(incl, off, 64);
        if (lane >= off) incl += other;
    }
    if (lane == 63) sh.wave_sum[wave] = incl;
    __syncthreads();
    filter_u64 before = 0;
    total = 0;
    for (int w = 0; w < FILTER_WAVES; ++w) {
        if (w < wave) before += sh.wave_sum[w];
        total += sh.wave_sum[w];
    }
    __syncthreads();
    return before + incl - mine;
}

// The index of the n-th (from 1) entry with this key that `limit` keeps, in index order; there are that many.  Every wavefront
// walks a contiguous piece of the row.
__device__ int cut_nth(const CutRow& row, unsigned key, const SampleCut& limit, unsigned n, CutShared& sh) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int piece = ((row.vocab + FILTER_WAVES - 1) / FILTER_WAVES + 63) / 64 * 64;
    const int begin = wave * piece, end = min(row.vocab, begin + piece);
    auto equal = [&](int i) { return i < end && filter_key(row.at[i]) == key && cut_keeps(limit, key, i); };
    unsigned mine = 0;
    for (int base = begin; base < end; base += 64) mine += __popcll(__ballot(equal(base + lane)));
    if (lane == 0) sh.wave_count[wave] = mine;
    __syncthreads();
    unsigned before = 0;
    for (int w = 0; w < wave; ++w) before += sh.wave_count[w];
    if (before < n && n <= before + mine)
        for (int base = begin; base < end; base += 64) {
            const bool is = equal(base + lane);
            const filter_u64 same = __ballot(is);
            if (is && before + __popcll(same & ((1ull << lane) - 1ull)) + 1 == n) sh.place = base + lane;
            before += __popcll(same);
        }
    __syncthreads();
    return sh.place;
}

// MASS: weights are softmax masses and the target is top_p times their total; else weights are 1 and the target is
// `target`.  Entries that `limit` does not keep are not there.  Called by the whole workgroup; every thread returns the same cut.
template <bool MASS>
__device__ SampleCut cut_search(const CutRow& row, const SampleCut& limit, float temp, float zmax,
                                filter_u64 target, float top_p, CutShared& sh) {
    const int tid = threadIdx.x;
    unsigned prefix = 0;
    filter_u64 above = 0;
    bool listed = false;
    unsigned count = 0;
    for (int level = 0; level < 3; ++level) {
        const int shift = level == 0 ? 20 : level == 1 ? 8 : 0, bins = level == 2 ? 256 : 4096;
        const unsigned known = level == 0 ? 0u : ~0u << (level == 1 ? 20 : 8);          // the bits found so far
        __syncthreads();
        for (int b = tid; b < bins; b += FILTER_NT) sh.hist[b] = 0;
        if (tid == 0) sh.bin = -1;
        __syncthreads();
        auto weigh = [&](unsigned key, float v) {
            if ((key & known) != prefix) return;
            const filter_u64 w = MASS ? filter_mass(v, temp, zmax) : 1ull;
            if (w != 0) atomicAdd(&sh.hist[(key >> shift) & (bins - 1)], w);
        };
        if (listed) {
            for (unsigned i = tid; i < count; i += FILTER_NT) weigh(sh.list[i], filter_value(sh.list[i]));
        } else {
            cut_walk(row, [&](float v, int i) {
                const unsigned key = filter_key(v);
                if (cut_keeps(limit, key, i)) weigh(key, v);
            });
        }
        __syncthreads();
        // thread t holds the bins from bins - 1 - 4 t down (one each at the last level): descending values in ascending threads
        const int per = bins >= FILTER_NT ? bins / FILTER_NT : 1, top = bins - 1 - tid * per;
        filter_u64 local[4], mine = 0, total;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            local[j] = j < per && top - j >= 0 ? sh.hist[top - j] : 0;
            mine += local[j];
        }
        filter_u64 run = above + cut_before(mine, total, sh);
        if (MASS && level == 0) target = (filter_u64)((double)top_p * (double)total);
        if (run <= target && run + mine > target) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (run <= target && run + local[j] > target) {
                    sh.bin = top - j;
                    sh.above = run;
                    sh.group = local[j];
                }
                run += local[j];
            }
        }
        if (tid == 0) sh.count = 0;
        __syncthreads();
        if (sh.bin < 0) return limit;                     // the target lies beyond the total: everything stays
        prefix |= (unsigned)sh.bin << shift;
        above = sh.above;
        if (!listed && level < 2) {
            const unsigned found = ~0u << shift;
            cut_walk(row, [&](float v, int i) {
                const unsigned key = filter_key(v);
                if ((key & found) != prefix || !cut_keeps(limit, key, i)) return;
                const unsigned at = atomicAdd(&sh.count, 1u);
                if (at < CUT_LIST) sh.list[at] = key;
            });
            __syncthreads();
            count = sh.count;
            listed = count <= CUT_LIST;
        }
    }
    filter_u64 each = MASS ? filter_mass(filter_value(prefix), temp, zmax) : 1ull;
    if (each == 0) each = 1;
    const filter_u64 members = sh.group / each, fit = (target - above) / each + 1;
    SampleCut cut{prefix, prefix == limit.key ? limit.last : 0x7fffffff};
    if (fit < members) cut.last = cut_nth(row, prefix, limit, (unsigned)fit, sh);
    return cut;
}

// The sorted form: the first k entries of the row in order (key descending, index ascending) in sh.sorted.  False if more entries
// than LDS holds reach the bound.
__device__ bool cut_sort(const CutRow& row, int k, CutShared& sh) {
    const int tid = threadIdx.x;
    unsigned mine = 0;
    cut_walk(row, [&](float v, int i) { mine = max(mine, filter_key(v)); });
    // A small k needs fewer of them: the largest of four threads each, so that ranking them is a sixteenth of the work (256
    // compared with 256 by a quarter of the threads; k of 64 then expects 74 entries from the bound on).
    const int together = k <= CUT_SORTED / 8 ? 4 : 1, groups = FILTER_NT / together;
    if (together == 4) {
        mine = max(mine, __shfl_xor(mine, 1, 64));
        mine = max(mine, __shfl_xor(mine, 2, 64));
    }
    __syncthreads();
    if (tid % together == 0) sh.largest[tid / together] = mine;
    if (tid == 0) sh.count = 0;
    __syncthreads();
    if (tid < groups) {
        const unsigned own = sh.largest[tid];
        int rank = 0;
        for (int t = 0; t < groups; t += 4) {
            const uint4 other = *reinterpret_cast<const uint4*>(&sh.largest[t]);
            rank += (other.x > own || (other.x == own && t < tid)) + (other.y > own || (other.y == own && t + 1 < tid)) +
                    (other.z > own || (other.z == own && t + 2 < tid)) + (other.w > own || (other.w == own && t + 3 < tid));
        }
        if (rank == k - 1) sh.bound = own;
    }
    __syncthreads();
    const unsigned bound = sh.bound;
    cut_walk(row, [&](float v, int i) {
        const unsigned key = filter_key(v);
        if (key < bound) return;
        const unsigned at = atomicAdd(&sh.count, 1u);
        if (at < CUT_CANDIDATES) {
            sh.candidate.key[at] = key;
            sh.candidate.index[at] = i;
        }
    });
    __syncthreads();
    const int n = sh.count;
    if (n > CUT_CANDIDATES) return false;
    for (int c = tid; c < n; c += FILTER_NT) {
        const unsigned key = sh.candidate.key[c];
        const int index = sh.candidate.index[c];
        int place = 0;
        for (int o = 0; o < n; ++o) {
            const unsigned other = sh.candidate.key[o];
            place += other > key || (other == key && sh.candidate.index[o] < index);
        }
        if (place < k) {
            sh.sorted.key[place] = key;
            sh.sorted.index[place] = index;
        }
    }
    __syncthreads();
    return true;
}

__device__ SampleCut cut_of_row(const CutRow& row, float temp, int k, float p, CutShared& sh) {
    SampleCut cut = SAMPLE_KEEP_ALL;
    if (!(temp > 0.f)) return cut;                          // greedy rows skip both rules (sampler.py:123, 142)
    const int tid = threadIdx.x;
    if (k > 0 && k < row.vocab) {
        if (k <= CUT_SORTED && cut_sort(row, k, sh)) {
            cut = SampleCut{sh.sorted.key[k - 1], sh.sorted.index[k - 1]};
            const float zmax = filter_value(sh.sorted.key[0]) / temp;
            if (!(p < 1.0f) || zmax == -INFINITY) return cut;
            const filter_u64 mass = tid < k ? filter_mass(filter_value(sh.sorted.key[tid]), temp, zmax) : 0;
            filter_u64 total;
            const filter_u64 before = cut_before(mass, total, sh);
            const filter_u64 target = (filter_u64)((double)p * (double)total);
            // the last entry whose predecessors hold at most the target
            if (tid < k && before <= target && (tid == k - 1 || before + mass > target)) sh.place = tid;
            __syncthreads();
            return SampleCut{sh.sorted.key[sh.place], sh.sorted.index[sh.place]};
        }
        __syncthreads();
        cut = cut_search<false>(row, cut, temp, 0.f, (filter_u64)(k - 1), 0.f, sh);
    }
    if (p < 1.0f) {
        float zmax = -INFINITY;
        cut_walk(row, [&](float v, int i) { zmax = fmaxf(zmax, v); });
        __syncthreads();
        zmax = block_max<FILTER_NT>(zmax, reinterpret_cast<float*>(sh.wave_count)) / temp;
        if (zmax == -INFINITY) return cut;
        cut = cut_search<true>(row, cut, temp, zmax, 0, p, sh);
    }
    return cut;
}

// WRITE: -inf over what the cut removes, in place; else the cut itself.
template <bool WRITE>
__global__ void __launch_bounds__(FILTER_NT)
sample_cut_kernel(const float* logits, float* masked, int vocab, bool quads, const float* __restrict__ temperature, const int* __restrict__ top_k,
                  const float* __restrict__ top_p, SampleCut* __restrict__ cuts) {
    __shared__ CutShared sh;
    const CutRow row{logits + (int64_t)blockIdx.x * vocab, vocab, quads};
    const SampleCut cut = cut_of_row(row, temperature[blockIdx.x], top_k[blockIdx.x], top_p[blockIdx.x], sh);
    if (WRITE) {
        float* to = masked + (int64_t)blockIdx.x * vocab;
        cut_walk(row, [&](float v, int i) {
            if (!cut_keeps(cut, filter_key(v), i)) to[i] = -INFINITY;
        });
    } else if (threadIdx.x == 0) {
        cuts[blockIdx.x] = cut;
    }
}

static int cut_check(const float* logits, int rows, int vocab) {
    SOMI_REQUIRE(rows >= 0 && vocab > 0, "sample_filter: bad sizes rows=%d vocab=%d", rows, vocab);
    SOMI_REQUIRE(vocab <= (1 << 22), "sample_filter: vocabulary of %d is beyond the 2^22 that the integer masses hold", vocab);
    return 0;
}

// logits: [rows, vocab] float32, in place; temperature, top_p: [rows] float32; top_k: [rows] int32 (-1 or >= vocab:
// off).  Rows with temperature 0 are left as they are.
extern "C" int somi_sample_filter(float* logits, int rows, int vocab, const float* temperature, const int* top_k,
                                  const float* top_p, hipStream_t stream) {
    if (cut_check(logits, rows, vocab)) return 1;
    if (rows == 0) return 0;
    hipLaunchKernelGGL((sample_cut_kernel<true>), dim3(rows), dim3(FILTER_NT), 0, stream, logits, logits, vocab,
                       sample_quads(logits, vocab), temperature, top_k, top_p, (SampleCut*)nullptr);
    SOMI_LAUNCH_CHECK("sample_filter");
    return 0;
}

// The same rules as cuts: [rows] pairs of 32-bit numbers for somi_sample_through; the logits stay as they are.
extern "C" int somi_sample_cuts(const float* logits, int rows, int vocab, const float* temperature, const int* top_k, const float* top_p,
                                void* cuts, hipStream_t stream) {
    if (cut_check(logits, rows, vocab)) return 1;
    if (rows == 0) return 0;
    hipLaunchKernelGGL((sample_cut_kernel<false>), dim3(rows), dim3(FILTER_NT), 0, stream, logits, (float*)nullptr, vocab,
                       sample_quads(logits, vocab), temperature, top_k, top_p, (SampleCut*)cuts);
    SOMI_LAUNCH_CHECK("sample_cuts");
    return 0;
}
