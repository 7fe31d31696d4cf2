// Mixture of gated experts over an fp32 stream (raven_moe_forward):
//     x += sum over the chosen experts of W_down ( silu(s W_gate h) * (s W_up h) )  +  sigmoid(g) W_down' ( silu(W_gate' h) * (W_up' h) )
// s = sigmoid(router logit): the factor of an expert's input is applied to the sums of its first two products, which is the same.
//
// One to a handful of rows (and fp32): moe_up_kernel forms the gated activations of a row's experts and of the shared one side by side, moe_down_kernel
// multiplies them by the down matrices and adds to the stream.  The first picks the row's experts itself from its logits -- a handful
// of wave reductions -- so no routing launch stands in between; for a single row it also takes the norm of the stream as a prologue.
// More bf16 rows: the rows are sorted by expert (moe_route_kernel, or moe_pick_kernel and moe_sort_kernel), or a few of them route themselves (pick_rows_kernel), and the experts run as one
// grouped product on the matrix cores (expert_rows_kernel, gemm_mid.hip, gemm_tiled.hip), rows gathered through the sorted list; every (token, expert) pair has a slot of
// its own, and moe_combine_kernel adds a token's slots and its shared expert to the stream in a fixed order.  So an expert's weights
// are read once and not once per row that picked it: 20 rows over 64 experts of 768 channels at width 2048, 6 each, read
// 55 experts instead of 120 (a layer of 16 rows: 168 us by row kernels, 109).

#include <algorithm>

#include "gemm_common.h"
#include "row_helpers.h"

namespace raven {

int ring_grouped(const void* x, int x_rows, const void* w, void* y, int rows, int N, int K, int swiglu, const RowGroups& g, hipStream_t s);

constexpr int kMaxExperts = 1024, kMaxTop = 32;
constexpr int kBigTileRows = 110;  // rows per expert from which the grouped products take 256-row tiles
constexpr int kPickRows = 32;  // tokens a workgroup of the two sorting kernels owns
constexpr int kRouteRows = 64, kRoutePairs = 2048;  // tokens and (token, expert) pairs up to which one workgroup picks and sorts

struct MoeArgs {
    const void *h, *up, *down, *shared_up, *shared_down;
    const float* logits;
    float* x;
    const float* factors;   // few rows: factors of the rows of h that are still to be applied (NormBehind), or null
    const float* norm;      // h null (one row): the norm of x that gives it, with its true width and eps
    int dim;
    float eps;
    void* act;              // few rows: [M, top * ff + shared_ff] of T
    int M, ld, ldl, experts, top, ff, sff;
    // chunks
    int* pick;              // [M, top]: expert
    float* pick_scale;      // [M, top]: its score
    int *slot_of;           // [M, top]: row of the grouped product
    int *slot_row;          // [M * top]: token of a slot
    float* slot_scale;      // [M * top]
    int *group_of, *group_row, *group_end, *used;
    int tile_rows;
    int* block_count;       // [ceil(M / kPickRows), experts]: pairs of a workgroup's tokens
    int fold;               // the shared expert is one more group (rows M * top ..+M - 1 of the product): extra group `experts`
    const void* y;          // [M * top, ld] of T, or float when fold
    const float* ys;        // [M, ld] or null
};

// a float as an integer of the same order; NaN below everything
__device__ __forceinline__ int ordered_key(float v) {
    const int b = __builtin_bit_cast(int, v + 0.0f);  // (the two zeros are equal)
    return v != v ? (int)0x80000000 : b < 0 ? b ^ 0x7fffffff : b;
}

// one wave: the `top` experts of largest logit (lower index first among equals); lane k holds the k-th one and its score.
// Up to 64 experts (a lane each) an expert's place is the number of experts before it, counted in one sweep over the others' logits
// through the lane-to-lane broadcast: 64 steps without a dependence, where `top` maxima over the wave, twelve exchanges each, took 3 us
// of every launch that picks six (routing of 20 rows 11.8 -> 8 us; a single row's products share the counting out over four waves).  One or two are found sooner by
// maxima (both launches of 8 rows of width 512, one of 8 experts of 512: 12.0 us, by counting 13.4).
// (U steps unrolled.  In a workgroup alone on its CU all 64 are 2.5 KB of code run once out of a cold instruction cache: routing of 20 rows 9.7 us, with 16
// 8.8.)
__host__ __device__ __forceinline__ bool picks_by_place(int experts, int top) { return experts <= 64 && top > 2; }
template <int U>
__device__ __forceinline__ void pick_by_place(float v, int experts, int& mine, float& score) {  // v: expert `lane`'s logit
    const int lane = threadIdx.x & 63;
    const int key = lane < experts ? ordered_key(v) : (int)0x80000000;
    int before = 0;
#pragma unroll U
    for (int j = 0; j < 64; ++j) {
        const int other = __builtin_amdgcn_readlane(key, j);
        before += other > key || (other == key && j < lane) ? 1 : 0;
    }
    // every lane has a place of its own (absent experts the last ones): lane l sends its number there
    mine = __builtin_amdgcn_ds_permute(before * 4, lane);
    const float s = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(before * 4, __builtin_bit_cast(int, v == v ? v : -INFINITY)));
    mine = min(mine, experts - 1);
    score = sigmoid_f32(s);
}
// The picks of a row are different experts whatever its logits are, as by place: where only minus infinity and NaN are left, the lowest numbers that have not been
// taken (the lists of picked_rows have room for one row of a token per expert).
__device__ __forceinline__ void pick_by_maxima(const float* logits, int experts, int top, int& mine, float& score) {
    const int lane = threadIdx.x & 63;
    float v[kMaxExperts / 64];
#pragma unroll
    for (int j = 0; j < kMaxExperts / 64; ++j) {
        v[j] = -INFINITY;
        if (64 * j < experts && lane + 64 * j < experts) v[j] = logits[lane + 64 * j];
    }
    mine = 0;
    float logit = 0.f;
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY;
        int at = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < kMaxExperts / 64; ++j)
            if (64 * j < experts && v[j] > best) {
                best = v[j];
                at = lane + 64 * j;
            }
        const float m = wave_max(best);
        int who = best == m ? at : 0x7fffffff;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) who = min(who, __shfl_xor(who, d, 64));
        if (lane == k) {
            mine = who;
            logit = m;
        }
#pragma unroll
        for (int j = 0; j < kMaxExperts / 64; ++j)
            if (lane + 64 * j == who) v[j] = -INFINITY;
    }
    if (const unsigned long long none = __ballot(lane < top && logit == -INFINITY))
        for (int k = __builtin_ctzll(none), e = 0; k < top; ++e) {  // (top <= experts)
            if (__any(lane < k && mine == e)) continue;
            if (lane == k) mine = e;
            ++k;
        }
    score = sigmoid_f32(logit);
}
__device__ __forceinline__ void pick_experts(const float* logits, int experts, int top, int& mine, float& score) {
    const int lane = threadIdx.x & 63;
    if (picks_by_place(experts, top)) pick_by_place<64>(lane < experts ? logits[lane] : 0.f, experts, mine, score);
    else pick_by_maxima(logits, experts, top, mine, score);
}

// ---- few rows --------------------------------------------------------------------------------------------
// A wave per (gate, up) row pair, over the concatenation of the row's experts and the shared one
template <typename T>
__global__ __launch_bounds__(256) void moe_up_kernel(MoeArgs a) {
    constexpr int E = Chunk<T>::N, U = 4;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* xs = reinterpret_cast<T*>(smem_raw);  // [ld]
    __shared__ int idx[kMaxTop];
    __shared__ float score[kMaxTop], red[4];
    const int m = blockIdx.y, nc = a.ld / E, total = a.top * a.ff + a.sff, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (a.h) {
        for (int i = threadIdx.x; i < nc; i += 256) store_chunk(xs + i * E, load_chunk(static_cast<const T*>(a.h) + (int64_t)m * a.ld + i * E));
    }
    if (wave == 0) {
        int e;
        float s;
        pick_by_maxima(a.logits + (int64_t)m * a.ldl, a.experts, a.top, e, s);
        if (lane < a.top) {
            idx[lane] = e;
            score[lane] = s;
            if (blockIdx.x == 0) a.pick[(int64_t)m * a.top + lane] = e;
        }
    }
    if (!a.h) {
        const float* x = a.x + (int64_t)m * a.ld;
        float ss = 0.f;
        for (int i = 4 * threadIdx.x; i < a.ld; i += 1024) {
            const f32x4 v = load4(x + i);
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        ss = wave_sum(ss);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)a.dim + a.eps);
        for (int i = 4 * threadIdx.x; i < a.ld; i += 1024) store4(xs + i, load4(x + i) * inv * load4(a.norm + i));
    }
    __syncthreads();
    const int p = blockIdx.x * 4 + wave;
    if (p >= total) return;
    const bool shared = p >= a.top * a.ff;
    const int slot = shared ? 0 : p / a.ff, r = shared ? p - a.top * a.ff : p - slot * a.ff;
    const T* g = shared ? static_cast<const T*>(a.shared_up) + (int64_t)r * a.ld
                        : static_cast<const T*>(a.up) + ((int64_t)idx[slot] * 2 * a.ff + r) * a.ld;
    const T* u = g + (int64_t)(shared ? a.sff : a.ff) * a.ld;
    float sg = 0.f, su = 0.f;
    for (int c0 = lane; c0 < nc; c0 += 64 * U) {
        Chunk<T> vg[U], vu[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int c = min(c0 + 64 * j, nc - 1);
            vg[j] = load_chunk_stream(g + c * E);
            vu[j] = load_chunk_stream(u + c * E);
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            if (c0 + 64 * j >= nc) break;
            const Chunk<T> x = load_chunk(xs + (c0 + 64 * j) * E);
            sg = dot_chunk(vg[j], x, sg);
            su = dot_chunk(vu[j], x, su);
        }
    }
    sg = wave_sum(sg);
    su = wave_sum(su);
    if (lane != 0) return;
    const float s = shared ? 1.f : score[slot];
    float v = silu_f32(s * sg) * (s * su);
    if (shared) v *= sigmoid_f32(a.logits[(int64_t)m * a.ldl + a.experts]);
    static_cast<T*>(a.act)[(int64_t)m * total + p] = from_f32<T>(v);
}

// The same where experts are picked by place, with nothing waited for twice: logits, row and norm weights are requested together, each wave counts a quarter of every
// expert's place (one wave counting all of it held up its SIMD, where the first waves of a CU's five workgroups meet), and a wave knows its own expert right behind the first
// barrier, so that its weights are on their way before the row is normed.  Bound by latencies in front of the weights: 44 MB (one row, 7 x 768 channels of width 2048)
// 13.4 -> 10.9 us, 6.9 of them at the rate of HBM.
template <typename T>
__global__ __launch_bounds__(256) void moe_up_place_kernel(MoeArgs a) {
    constexpr int E = Chunk<T>::N, U = 4, H = 2;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* xs = reinterpret_cast<T*>(smem_raw);  // [ld]
    __shared__ unsigned char place[4][64];  // (in bytes: beside the longest row, kMoeRowLds, there is 1 KB)
    __shared__ float red[4];
    const int m = blockIdx.y, nc = a.ld / E, total = a.top * a.ff + a.sff, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float* logits = a.logits + (int64_t)m * a.ldl;
    const float* x = a.x + (int64_t)m * a.ld;
    const float logit = logits[min(lane, a.experts - 1)];
    f32x4 xv[H], nv[H];
    if (a.h) {
        for (int i = tid; i < nc; i += 256) store_chunk(xs + i * E, load_chunk(static_cast<const T*>(a.h) + (int64_t)m * a.ld + i * E));
    } else {
#pragma unroll
        for (int j = 0; j < H; ++j) xv[j] = load4(x + min(4 * tid + 1024 * j, a.ld - 4));
#pragma unroll
        for (int j = 0; j < H; ++j) nv[j] = load4(a.norm + min(4 * tid + 1024 * j, a.ld - 4));
    }
    const int key = lane < a.experts ? ordered_key(logit) : (int)0x80000000;
    int before = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int at = 16 * wave + j, other = __builtin_amdgcn_readlane(key, at);
        before += other > key || (other == key && at < lane) ? 1 : 0;
    }
    place[wave][lane] = (unsigned char)before;
    if (!a.h) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < H; ++j)
            if (4 * tid + 1024 * j < a.ld) ss += xv[j][0] * xv[j][0] + xv[j][1] * xv[j][1] + xv[j][2] * xv[j][2] + xv[j][3] * xv[j][3];
        for (int i = 4 * tid + 1024 * H; i < a.ld; i += 1024) {
            const f32x4 v = load4(x + i);
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        ss = wave_sum(ss);
        if (lane == 0) red[wave] = ss;
    }
    __syncthreads();
    before = place[0][lane] + place[1][lane] + place[2][lane] + place[3][lane];
    if (blockIdx.x == 0 && wave == 0 && before < a.top) a.pick[(int64_t)m * a.top + before] = lane;
    const int own = blockIdx.x * 4 + wave, p = min(own, total - 1);
    const bool shared = p >= a.top * a.ff;
    const int slot = shared ? 0 : p / a.ff, r = shared ? p - a.top * a.ff : p - slot * a.ff;
    const int expert = __builtin_ctzll(__ballot(before == slot));  // (every lane has a place of its own)
    const T* g = shared ? static_cast<const T*>(a.shared_up) + (int64_t)r * a.ld : static_cast<const T*>(a.up) + ((int64_t)expert * 2 * a.ff + r) * a.ld;
    const T* u = g + (int64_t)(shared ? a.sff : a.ff) * a.ld;
    Chunk<T> vg[U], vu[U];
    auto request = [&](int c0) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int c = min(c0 + 64 * j, nc - 1);
            vg[j] = load_chunk_stream(g + c * E);
            vu[j] = load_chunk_stream(u + c * E);
        }
    };
    request(lane);
    const float gate = shared ? logits[a.experts] : __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, logit), expert));
    if (!a.h) {
        const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)a.dim + a.eps);
#pragma unroll
        for (int j = 0; j < H; ++j)
            if (4 * tid + 1024 * j < a.ld) store4(xs + 4 * tid + 1024 * j, xv[j] * inv * nv[j]);
        for (int i = 4 * tid + 1024 * H; i < a.ld; i += 1024) store4(xs + i, load4(x + i) * inv * load4(a.norm + i));
        __syncthreads();
    }
    float sg = 0.f, su = 0.f;
    for (int c0 = lane;;) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
            if (c0 + 64 * j >= nc) break;
            const Chunk<T> v = load_chunk(xs + (c0 + 64 * j) * E);
            sg = dot_chunk(vg[j], v, sg);
            su = dot_chunk(vu[j], v, su);
        }
        c0 += 64 * U;
        if (c0 - lane >= nc) break;
        request(c0);
    }
    sg = wave_sum(sg);
    su = wave_sum(su);
    if (lane != 0 || own >= total) return;
    const float s = shared ? 1.f : sigmoid_f32(gate == gate ? gate : -INFINITY);
    float v = silu_f32(s * sg) * (s * su);
    if (shared) v *= sigmoid_f32(gate);
    static_cast<T*>(a.act)[(int64_t)m * total + p] = from_f32<T>(v);
}

// a wave per output channel: its row of every chosen down matrix and of the shared one, as one long row, U pieces of 64 chunks at a time (up to 12: all at once).
// The picks are requested first and handed out by lane exchange, so that the weights wait for one round trip: 22 MB 7.4 -> 6.7 us (with six pieces at a time and a
// load of the pick in front of each).
template <typename T, int U>
__global__ __launch_bounds__(256) void moe_down_kernel(MoeArgs a) {
    constexpr int E = Chunk<T>::N;
    const int m = blockIdx.y, n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (n >= a.ld) return;
    const int pick = a.pick[(int64_t)m * a.top + min(lane, a.top - 1)];
    const float x = a.x[(int64_t)m * a.ld + n];
    const unsigned nf = a.ff / E, nr = a.top * nf, nc = nr + a.sff / E;
    const T* act = static_cast<const T*>(a.act) + (int64_t)m * nc * E;
    const T* down = static_cast<const T*>(a.down);
    const T* sdown = static_cast<const T*>(a.shared_down);
    float sum = 0.f;
    for (unsigned c0 = lane; c0 - lane < nc; c0 += 64 * U) {
        Chunk<T> w[U], v[U];
#pragma unroll
        for (int j = 0; j < U; ++j) v[j] = load_chunk(act + min(c0 + 64 * j, nc - 1) * E);
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const unsigned c = min(c0 + 64 * j, nc - 1), slot = c / nf;
            const int e = __shfl(pick, slot, 64);
            w[j] = load_chunk_stream(c < nr ? down + ((int64_t)e * a.ld + n) * a.ff + (c - slot * nf) * E : sdown + (int64_t)n * a.sff + (c - nr) * E);
        }
#pragma unroll
        for (int j = 0; j < U; ++j)
            if (c0 + 64 * j < nc) sum = dot_chunk(w[j], v[j], sum);
    }
    sum = wave_sum(sum);
    if (lane == 0) a.x[(int64_t)m * a.ld + n] = x + sum;
}

// ---- chunks ----------------------------------------------------------------------------------------------
// Both sorting kernels give kPickRows tokens to a workgroup.  The first picks their experts (a wave per token in turn) and counts
// its pairs per expert; the second adds the counts up -- every workgroup for itself: they are few --, so that it knows where each
// expert's rows start and which of them are its own, and puts its pairs there.  Inside a workgroup's share of an expert the order is
// whatever the counters give: no result depends on it.
__global__ __launch_bounds__(1024) void moe_pick_kernel(MoeArgs a) {
    __shared__ int count[kMaxExperts];
    const int m0 = blockIdx.x * kPickRows, wave = threadIdx.x >> 6;
    for (int e = threadIdx.x; e < a.experts; e += 1024) count[e] = 0;
    __syncthreads();
    for (int i = wave; i < kPickRows && m0 + i < a.M; i += 16) {
        const int64_t m = m0 + i;
        const int lane = threadIdx.x & 63;
        int e;
        float s;
        pick_experts(a.logits + m * a.ldl, a.experts, a.top, e, s);
        if (lane < a.top) {
            a.pick[m * a.top + lane] = e;
            a.pick_scale[m * a.top + lane] = s;
            atomicAdd(&count[e], 1);
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < a.experts; e += 1024) a.block_count[(int64_t)blockIdx.x * a.experts + e] = count[e];
}

__global__ __launch_bounds__(1024) void moe_sort_kernel(MoeArgs a) {
    __shared__ int before[kMaxExperts], total[kMaxExperts], wave_sums[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, blocks = gridDim.x, me = blockIdx.x;
    before[tid] = total[tid] = 0;
    __syncthreads();
    const int counts = blocks * a.experts;
    for (int i0 = tid; i0 < counts; i0 += 4096) {
        int v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = i0 + 1024 * j < counts ? a.block_count[i0 + 1024 * j] : 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (v[j] == 0) continue;
            const int i = i0 + 1024 * j, b = i / a.experts, e = i - b * a.experts;
            atomicAdd(&total[e], v[j]);
            if (b < me) atomicAdd(&before[e], v[j]);
        }
    }
    __syncthreads();
    // running sums over the experts of rows and of tile rows
    const int rows = total[tid], tiles = (rows + a.tile_rows - 1) / a.tile_rows;
    int r = rows, t = tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int pr = __shfl_up(r, d, 64), pt = __shfl_up(t, d, 64);
        if (lane >= d) {
            r += pr;
            t += pt;
        }
    }
    if (lane == 63) {
        wave_sums[0][wave] = r;
        wave_sums[1][wave] = t;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) {
        r += wave_sums[0][w];
        t += wave_sums[1][w];
    }
    const int first = r - rows, first_tile = t - tiles;
    before[tid] += first;  // where this workgroup's rows of expert tid start
    if (me == 0) {
        for (int i = 0; i < tiles; ++i) {
            a.group_of[first_tile + i] = tid;
            a.group_row[first_tile + i] = first + i * a.tile_rows;
            a.group_end[first_tile + i] = min(first + (i + 1) * a.tile_rows, first + rows);
        }
        int used = 0;
        for (int w = 0; w < 16; ++w) used += wave_sums[1][w];
        if (tid == 0) *a.used = used;
    }
    __syncthreads();
    const int lo = me * kPickRows * a.top, hi = min(a.M, (me + 1) * kPickRows) * a.top;
    for (int i = lo + tid; i < hi; i += 1024) {
        const int slot = atomicAdd(&before[a.pick[i]], 1);
        a.slot_of[i] = slot;
        a.slot_row[slot] = i / a.top;
        a.slot_scale[slot] = a.pick_scale[i];
    }
}

// Both of the above in one workgroup, for few rows; with fold the shared expert's rows follow as one more group of factor one
__global__ __launch_bounds__(1024) void moe_route_kernel(MoeArgs a) {
    __shared__ int count[kMaxExperts], start[kMaxExperts], pick[kRoutePairs], wave_sums[2][16];
    __shared__ float scale[kRoutePairs];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, pairs = a.M * a.top;
    count[tid] = 0;
    __syncthreads();
    auto keep = [&](int m, int e, float s) {
        if (lane < a.top) {
            pick[m * a.top + lane] = e;
            scale[m * a.top + lane] = s;
            atomicAdd(&count[e], 1);
        }
    };
    if (picks_by_place(a.experts, a.top)) {  // a wave's next row is requested before the one at hand is sorted (20 rows 8.8 -> 8.2 us)
        auto logit = [&](int m) { return a.logits[(int64_t)min(m, a.M - 1) * a.ldl + min(lane, a.experts - 1)]; };
        float next = logit(wave);
        for (int m = wave; m < a.M; m += 16) {
            const float v = lane < a.experts ? next : 0.f;
            next = logit(m + 16);
            int e;
            float s;
            pick_by_place<16>(v, a.experts, e, s);
            keep(m, e, s);
        }
    } else {
        for (int m = wave; m < a.M; m += 16) {
            int e;
            float s;
            pick_experts(a.logits + (int64_t)m * a.ldl, a.experts, a.top, e, s);
            keep(m, e, s);
        }
    }
    __syncthreads();
    const int rows = count[tid], tiles = (rows + a.tile_rows - 1) / a.tile_rows;
    int r = rows, t = tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int pr = __shfl_up(r, d, 64), pt = __shfl_up(t, d, 64);
        if (lane >= d) {
            r += pr;
            t += pt;
        }
    }
    if (lane == 63) {
        wave_sums[0][wave] = r;
        wave_sums[1][wave] = t;
    }
    __syncthreads();
    int used = 0;
    for (int w = 0; w < 16; ++w) {
        if (w < wave) {
            r += wave_sums[0][w];
            t += wave_sums[1][w];
        }
        used += wave_sums[1][w];
    }
    const int first = r - rows, first_tile = t - tiles;
    start[tid] = first;
    for (int i = 0; i < tiles; ++i) {
        a.group_of[first_tile + i] = tid;
        a.group_row[first_tile + i] = first + i * a.tile_rows;
        a.group_end[first_tile + i] = min(first + (i + 1) * a.tile_rows, first + rows);
    }
    const int shared_tiles = a.fold ? (a.M + a.tile_rows - 1) / a.tile_rows : 0;
    for (int i = tid; i < shared_tiles; i += 1024) {
        a.group_of[used + i] = a.experts;
        a.group_row[used + i] = pairs + i * a.tile_rows;
        a.group_end[used + i] = pairs + min((i + 1) * a.tile_rows, a.M);
    }
    if (tid == 0) *a.used = used + shared_tiles;
    __syncthreads();
    for (int i = tid; i < pairs; i += 1024) {
        const int slot = atomicAdd(&start[pick[i]], 1);
        a.slot_of[i] = slot;
        a.slot_row[slot] = i / a.top;
        a.slot_scale[slot] = a.factors ? scale[i] * a.factors[i / a.top] : scale[i];
    }
    if (a.fold)
        for (int m = tid; m < a.M; m += 1024) {
            a.slot_row[pairs + m] = m;
            a.slot_scale[pairs + m] = a.factors ? a.factors[m] : 1.f;
        }
}

// ---- few rows, no sorting ----------------------------------------------------------------------------------
// Up to 32 rows over up to 64 experts, behind a norm that is shared out between two products (NormBehind): logits and picks of a row in one launch, a workgroup per
// row and its waves the experts in turn.  A pair's row of the grouped products is its own number, and their units find the rows of their expert in the list of
// picks themselves (expert_rows_kernel, PICKED), so that nothing is sorted.  Bound by a workgroup's own read of the router (330 KB out of the L2 at width 2048); us at 20
// rows of width 2048, router product and sorting / this: 6.4 + 8.6 / 9.0; finding their rows costs the products 0.6 to 0.9 (59.0 -> 59.6, 28.1 -> 29.0).
template <int NC>
__global__ __launch_bounds__(1024) void pick_rows_kernel(MoeArgs a, const bf16* __restrict__ router, NormBehind b, float* __restrict__ logits, float* __restrict__ factors) {
    __shared__ float logit[80];
    const int m = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, pieces = a.ld / 8, rows = a.experts + (a.shared_up ? 1 : 0);
    float squares[kNormParts / 64];
#pragma unroll
    for (int i = 0; i < kNormParts / 64; ++i) squares[i] = b.squares[m * norm_pitch(b.parts) + min(lane + 64 * i, b.parts - 1)];
    Chunk<bf16> x[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c] = lane + 64 * c < pieces ? load_chunk(static_cast<const bf16*>(a.h) + (int64_t)m * a.ld + 8 * (lane + 64 * c)) : zero_chunk<bf16>();
    constexpr int R = 3;  // expert rows requested together
    float inv = 0.f;
#pragma unroll
    for (int e0 = 0; e0 < 5; e0 += R) {
        Chunk<bf16> w[R][NC];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < NC; ++c)
                w[r][c] = load_chunk(router + (int64_t)min(wave + 16 * (e0 + r), rows - 1) * a.ld + 8 * min(lane + 64 * c, pieces - 1));
        if (e0 == 0) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < kNormParts / 64; ++i) sum += lane + 64 * i < b.parts ? squares[i] : 0.f;
            inv = 1.0f / sqrtf(wave_sum(sum) / (float)b.dim + b.eps);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int e = wave + 16 * (e0 + r);
            if (e >= rows) continue;
            float s = 0.f;
#pragma unroll
            for (int c = 0; c < NC; ++c) s = dot_chunk(w[r][c], x[c], s);
            s = wave_sum(s) * inv;
            if (lane == 0) {
                logit[e] = s;
                logits[(int64_t)m * a.ldl + e] = s;
            }
        }
    }
    __syncthreads();
    if (wave != 0) return;
    int e;
    float s;
    pick_experts(logit, a.experts, a.top, e, s);
    if (lane < a.top) {
        a.pick[m * a.top + lane] = e;
        a.pick_scale[m * a.top + lane] = s * inv;
    }
    if (lane == 0) factors[m] = inv;
}

// ------------------------------------------------------------------------------------------------
// The grouped products of experts with at most 16 rows a tile: y[r] = x[x_row[r]] W_g^T.  One unit -- a tile's rows against 32 weight rows (up: 16 gate and 16 up
// rows) -- per workgroup of four waves that take the K steps in turn and never wait for each other; a wave's weight rows come as
// whole runs of 128 (down) or 256 bytes (up) into registers, go through its own LDS tile into operand layout and are multiplied on the
// matrix cores (the scheme of mfma_kernel in gemm_skinny.hip).  Bound by first reads of the weights: what the workgroups of a CU, three of up and five of down, keep
// in flight is some 80 to 100 KB, and some 50 units an expert, started as others end, leave no round half empty -- the units of 128 weight rows of
// gemm_mid.hip, two to a CU, made 1.3 rounds.  The K loop asks for nothing past its end and has no load under a branch, so that a wait counts only the step
// being parked.  us for a whole mixture (four launches, weights from HBM), 64 experts, 6 per row and a shared one, by gemm_mid.hip / now: width 2048, 4 rows
// 63 / 48, 8: 82 / 68, 20: 119 / 97, 40: 148 / 130; width 1024, 20 rows 44 / 38; 128 experts of 512, 8 per row, 20 rows 144 / 111.  Two register sets in
// flight were 5 % slower at 20 rows (fewer resident waves), three 27 %; 64 weight rows a unit 7 %.
// Weights that one tile alone reads are not kept in the caches.  An expert with several tiles keeps them, and its units of the same weight rows are numbered
// alike modulo 8, which puts them on one XCD: where all rows pick the same experts -- equal sequences side by side -- 40 rows of 64 experts of 864 at
// width 2304 took 76 us without either, 59 with both (61 by gemm_mid.hip).
// ------------------------------------------------------------------------------------------------
struct FewArgs {
    const bf16 *x, *w;
    void* y;               // [rows, N]
    int N, K, tiles_n, out_f32;
    RowGroups g;
    // PICKED: rows by their picks
    const int* pick;       // [M * top]
    const float* factors;  // UP: of the shared expert's rows
    int M, top, experts;
};
constexpr int kPickedRows = 32;  // tokens

// or of all lanes, by moves inside a row of 16 and four scalar reads (an exchange through the LDS costs 0.05 us a step)
__device__ __forceinline__ unsigned wave_or(unsigned v) {
    auto row = [](unsigned x, auto ctrl) { return x | (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xf, 0xf, true); };
    v = row(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
    v = row(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    v = row(v, std::integral_constant<int, 0x124>{});  // row_ror 4
    v = row(v, std::integral_constant<int, 0x128>{});  // row_ror 8
    return (unsigned)(__builtin_amdgcn_readlane((int)v, 0) | __builtin_amdgcn_readlane((int)v, 16) | __builtin_amdgcn_readlane((int)v, 32) | __builtin_amdgcn_readlane((int)v, 48));
}

// PICKED: the rows of unit group `which`, in LDS: row of x, row of the product and factor of each; the experts that rows pick come first, in their order, then tiles of
// 16 rows of the shared expert.  Returns their number, 0 behind the last group; *group: the expert, `experts` for the shared one
constexpr int kHeldPicks = 4;  // pieces of 64 picks that a lane keeps: all there are (moe_path: more than 8 rows go here with less than two picks per expert)
static_assert(64 * kHeldPicks >= 8 * kMaxTop && 64 * kHeldPicks >= 2 * 64, "every pick is held");
template <bool UP>
__device__ __forceinline__ int picked_rows(const FewArgs& a, int which, int* group, int* x_row, int* y_row, float* scale) {
    const int lane = threadIdx.x & 63, pairs = a.M * a.top;
    unsigned low = 0, high = 0;
    int held[kHeldPicks];
#pragma unroll
    for (int c = 0; c < kHeldPicks; ++c) held[c] = a.pick[min(64 * c + lane, pairs - 1)];
#pragma unroll
    for (int c = 0; c < kHeldPicks; ++c) {
        const unsigned bit = 1u << (held[c] & 31);
        if (held[c] < 32) low |= bit;
        else high |= bit;
    }
    const unsigned long long mask = ((unsigned long long)wave_or(high) << 32) | wave_or(low);
    const int touched = __popcll(mask);
    if (which >= touched) {
        const int first = (which - touched) * 16, n = a.g.extra_group < 0 ? 0 : min(a.M - first, 16);
        *group = a.experts;
        if (n > 0 && threadIdx.x < (unsigned)n) {
            x_row[threadIdx.x] = UP ? first + (int)threadIdx.x : pairs + first + (int)threadIdx.x;
            y_row[threadIdx.x] = pairs + first + threadIdx.x;
            if (UP) scale[threadIdx.x] = a.factors[first + threadIdx.x];
        }
        return max(n, 0);
    }
    const bool is_it = (mask >> lane) & 1 && __popcll(mask & ((1ull << lane) - 1)) == which;
    const int g = __builtin_ctzll(__ballot(is_it));
    *group = g;
    int n = 0;
    auto take = [&](int p0, int e) {
        const int p = p0 + lane;
        const bool own = p < pairs && e == g;
        const unsigned long long found = __ballot(own);
        const int at = n + __popcll(found & ((1ull << lane) - 1));
        if (own && threadIdx.x < 64 && at < kPickedRows) {  // (a token picks an expert once, so that there are no more)
            x_row[at] = UP ? p / a.top : p;
            y_row[at] = p;
            if (UP) scale[at] = a.g.x_scale[p];
        }
        n += __popcll(found);
    };
#pragma unroll
    for (int c = 0; c < kHeldPicks; ++c)
        if (64 * c < pairs) take(64 * c, held[c]);
    return min(n, kPickedRows);
}

constexpr int few_columns(bool up) { return up ? 16 : 32; }  // output columns of a unit

// PICKED: see picked_rows
template <bool UP, bool PICKED = false>
__global__ __launch_bounds__(256) void expert_rows_kernel(FewArgs a) {
    constexpr int KM = UP ? 128 : 64, NT = 2, COLS = few_columns(UP), NG = COLS / 16;  // a K step, tiles of 16 weight rows, of output columns
    constexpr int PITCH = KM + 8, LPR = KM / 8, RPI = 64 / LPR, IPT = 16 / RPI;   // lanes per row, rows per load, loads per tile
    __shared__ __align__(16) bf16 stage[4][16 * (NT + 1)][PITCH];
    static_assert(sizeof(stage) >= 3 * NT * 64 * 16, "the tiles double as the waves' sums");
    __shared__ int x_rows[PICKED ? kPickedRows : 1], y_rows[PICKED ? kPickedRows : 1];
    __shared__ float scales[PICKED && UP ? kPickedRows : 1];
    const int tile = (int)blockIdx.x / a.tiles_n, at = (int)blockIdx.x - tile * a.tiles_n;
    const int n0 = (at + (tile * a.tiles_n) % 8) % a.tiles_n * COLS;
    int g, row0 = 0, all, used = 0;
    if constexpr (PICKED) {
        all = picked_rows<UP>(a, tile, &g, x_rows, y_rows, scales);
        if (all == 0) return;
        __syncthreads();
    } else {
        used = *a.g.used;
        if (tile >= used) return;
        g = a.g.group_of[tile], row0 = a.g.group_row[tile], all = a.g.group_end[tile] - row0;
    }
    const bf16* W = g == a.g.extra_group ? a.g.w_extra : a.w + g * a.g.w_stride;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, ln = lane & 15, kq = lane >> 4;
    const int lr = lane / LPR, lc = (lane % LPR) * 8, K = a.K;
    bf16(*my)[PITCH] = stage[wave];
    const int n_steps = (K + KM - 1) / KM, mine = (n_steps - wave + 3) / 4;

    f32x4 acc[NT];
    // element offsets of this lane's rows: weight rows past N repeat the last one, token rows past the tile's likewise (neither is stored)
    unsigned wo[NT][IPT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < IPT; ++i) wo[t][i] = (unsigned)(min(n0 + (t % NG) * 16 + RPI * i + lr, a.N - 1) + (UP && t >= NG ? a.N : 0)) * (unsigned)K;
    // XI: load instructions that the token rows from `first` on need.  ONCE: no other tile reads these weights
    auto run = [&](int first, int rows, auto xi_tag, auto once_tag) __attribute__((always_inline)) {
        constexpr int XI = decltype(xi_tag)::value;
        constexpr bool ONCE = decltype(once_tag)::value;
        const bf16* xp[XI];
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int r = row0 + first + min(RPI * i + lr, rows - 1);
            xp[i] = a.x + (int64_t)(PICKED ? x_rows[r] : a.g.x_row ? a.g.x_row[r] : r) * K;
        }
        struct Staged {
            u32x4 w[NT][IPT], x[XI];
        } st;
        // step i of this wave
        auto fetch = [&](int i, Staged& s) __attribute__((always_inline)) {
            const int kc = min((wave + 4 * i) * KM + lc, K - 8);
#pragma unroll
            for (int t = 0; t < XI; ++t) s.x[t] = *reinterpret_cast<const u32x4*>(xp[t] + kc);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const u32x4* from = reinterpret_cast<const u32x4*>(W + wo[t][j] + kc);
                    s.w[t][j] = ONCE ? __builtin_nontemporal_load(from) : *from;
                }
        };
        auto park = [&](int i, Staged& s) __attribute__((always_inline)) {
            const bool past = (wave + 4 * i) * KM + lc >= K;  // columns past K are zeros
            const u32x4 z = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < IPT; ++j) *reinterpret_cast<u32x4*>(&my[t * 16 + RPI * j + lr][lc]) = past ? z : s.w[t][j];
#pragma unroll
            for (int t = 0; t < XI; ++t) *reinterpret_cast<u32x4*>(&my[NT * 16 + RPI * t + lr][lc]) = past ? z : s.x[t];
        };
        auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < KM / 32; ++j) {
                const bf16x8 xv = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&my[NT * 16 + ln][32 * j + 8 * kq]));
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const bf16x8 wv = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&my[t * 16 + ln][32 * j + 8 * kq]));
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv, acc[t], 0, 0, 0);
                }
            }
        };
        // lanes exchange data through the tile without a workgroup barrier: pin the order of the LDS accesses for the compiler
        auto wave_sync = []() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        if (mine <= 0) return;
        fetch(0, st);
#pragma unroll 1
        for (int i = 1; i < mine; ++i) {
            park(i - 1, st);
            wave_sync();
            fetch(i, st);
            multiply();
            wave_sync();
        }
        park(mine - 1, st);
        wave_sync();
        multiply();
    };
    bool alone;
    if constexpr (PICKED) {
        alone = all <= 16 && (g != a.experts || a.M <= 16);
    } else {
        const int before = a.g.group_of[max(tile - 1, 0)], after = a.g.group_of[min(tile + 1, used - 1)];
        alone = (tile == 0 || before != g) && (tile + 1 == used || after != g);
    }
    for (int first = 0; first < all; first += 16) {  // (a second round only of a picked expert with more than 16 rows)
        const int rows = min(16, all - first);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!alone) run(first, rows, std::integral_constant<int, IPT>{}, std::false_type{});
        else if (rows <= RPI) run(first, rows, std::integral_constant<int, 1>{}, std::true_type{});
        else run(first, rows, std::integral_constant<int, IPT>{}, std::true_type{});

        __syncthreads();
        f32x4(*sums)[NT][64] = reinterpret_cast<f32x4(*)[NT][64]>(&stage[0][0][0]);
        if (wave > 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t) sums[wave - 1][t][lane] = acc[t];
        }
        __syncthreads();
        if (wave == 0 && ln < rows) {
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] += sums[0][t][lane] + sums[1][t][lane] + sums[2][t][lane];
            // a lane holds columns 4 kq ..+3 of each tile for token row ln
            const int r = row0 + first + ln;
            const float xs = UP ? (PICKED ? scales[r] : a.g.x_scale[r]) : 1.f;
#pragma unroll
            for (int t = 0; t < NG; ++t) {
                const int n = n0 + 16 * t + 4 * kq;
                if (n >= a.N) continue;
                const int64_t to = (int64_t)(PICKED ? y_rows[r] : r) * a.N + n;
                f32x4 v = acc[t];
                if (UP) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = silu_f32(v[i] * xs) * (acc[UP ? t + 1 : t][i] * xs);
                }
                if (a.out_f32) {
                    store4(static_cast<float*>(a.y) + to, v);
                } else {
                    store4(static_cast<bf16*>(a.y) + to, v);
                }
            }
        }
        if (!PICKED || first + 16 >= all) return;
        __syncthreads();  // the sums have been read
    }
}

static int expert_rows(const void* x, const void* w, void* y, int N, int K, bool up, int out_f32, const RowGroups& g, hipStream_t s) {
    RAVEN_REQUIRE(g.n_tiles > 0 && N > 0 && N % 8 == 0 && K > 0 && K % 8 == 0 && (int64_t)2 * N * K < (1ll << 31) && (!up || g.x_scale), "moe: bad experts");
    FewArgs a{};
    a.x = static_cast<const bf16*>(x); a.w = static_cast<const bf16*>(w); a.y = y; a.N = N; a.K = K; a.out_f32 = out_f32; a.g = g;
    a.tiles_n = (N + few_columns(up) - 1) / few_columns(up);
    const int64_t units = (int64_t)a.tiles_n * g.n_tiles;
    RAVEN_REQUIRE(units < (1ll << 31), "moe: too many units");
    if (up) expert_rows_kernel<true><<<dim3((unsigned)units), dim3(256), 0, s>>>(a);
    else expert_rows_kernel<false><<<dim3((unsigned)units), dim3(256), 0, s>>>(a);
    return raven_host::check_launch("moe (rows of an expert)");
}

// The same over picks: g gives the matrices and, up, the factors of the pairs
static int picked_expert_rows(const void* x, const void* w, void* y, int N, int K, bool up, const RowGroups& g, const MoeArgs& m, hipStream_t s) {
    RAVEN_REQUIRE(m.M > 0 && m.M <= kPickedRows && m.M * m.top <= 64 * kHeldPicks && m.experts <= 64 && N > 0 && N % 8 == 0 && K > 0 && K % 8 == 0 && (int64_t)2 * N * K < (1ll << 31) && m.pick && m.factors &&
                      (!up || g.x_scale) && (g.extra_group < 0 || (g.extra_group == m.experts && g.w_extra)), "moe: bad picked experts");
    FewArgs a{};
    a.x = static_cast<const bf16*>(x); a.w = static_cast<const bf16*>(w); a.y = y; a.N = N; a.K = K; a.out_f32 = up ? 0 : 1; a.g = g;
    a.pick = m.pick; a.factors = m.factors; a.M = m.M; a.top = m.top; a.experts = m.experts;
    a.tiles_n = (N + few_columns(up) - 1) / few_columns(up);
    const int64_t groups = std::min(m.experts, m.M * m.top) + (g.extra_group >= 0 ? (m.M + 15) / 16 : 0);
    if (up) expert_rows_kernel<true, true><<<dim3((unsigned)(groups * a.tiles_n)), dim3(256), 0, s>>>(a);
    else expert_rows_kernel<false, true><<<dim3((unsigned)(groups * a.tiles_n)), dim3(256), 0, s>>>(a);
    return raven_host::check_launch("moe (rows of a picked expert)");
}

// Row of the products that a token's k-th pair has.  (Known at compile time which: decided per load, the loads of a token waited for each other, 32 of them 5.3 -> 11.9 us.)
template <bool PICKED>
__device__ __forceinline__ int64_t pair_row(const MoeArgs& a, int m, int k) {
    const int i = m * a.top + min(k, a.top - 1);
    return PICKED ? i : a.slot_of[i];
}
template <typename Y, bool PICKED>
__global__ __launch_bounds__(256) void moe_combine_kernel(MoeArgs a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int per = a.ld / 4;
    if (i >= (int64_t)a.M * per) return;
    const int m = (int)(i / per), c = 4 * (int)(i % per);
    const Y* y = static_cast<const Y*>(a.y);
    f32x4 x = load4(a.x + (int64_t)m * a.ld + c), shared = f32x4{0.f, 0.f, 0.f, 0.f};
    const float gate = a.ys ? sigmoid_f32(a.logits[(int64_t)m * a.ldl + a.experts]) : 0.f;
    if (a.ys) shared = load4(a.ys + (int64_t)m * a.ld + c);
    for (int k0 = 0; k0 < a.top; k0 += 8) {
        f32x4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = load4(y + pair_row<PICKED>(a, m, k0 + k) * a.ld + c);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (k0 + k < a.top) x += v[k];
    }
    if (a.ys) x += shared * gate;
    store4(a.x + (int64_t)m * a.ld + c, x);
}

// The same with the norm that the next layer begins with, h = T(x / rms(x) * w): a workgroup per row, whose pieces stay in registers.  The squares are added as
// norm_conv_kernel adds them, so that a layer gives the same bits whether it is called with the next one or by itself.  us at 20 rows of
// width 2048, sums and norm / this: 4.7 + 4.6 / 4.9; at 4096 rows 32 + 9.8 / 34.
constexpr int kCombineThreads = 512;
struct NextNorm {
    const float* w;  // [ld], zero past dim; null: none
    void* h;         // [M, ld] of bf16
    int dim;
    float eps;
};
template <typename Y, int P, bool PICKED>
__global__ __launch_bounds__(kCombineThreads) void moe_combine_norm_kernel(MoeArgs a, NextNorm next) {
    __shared__ float squares[kCombineThreads * P], red[4];
    const int m = blockIdx.x, tid = threadIdx.x, per = a.ld / 4;
    const Y* y = static_cast<const Y*>(a.y);
    const float gate = a.ys ? sigmoid_f32(a.logits[(int64_t)m * a.ldl + a.experts]) : 0.f;
    f32x4 x[P], w[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int c = 4 * min(tid + kCombineThreads * j, per - 1);
        w[j] = load4(next.w + c);
        x[j] = load4(a.x + (int64_t)m * a.ld + c);
        f32x4 shared = f32x4{0.f, 0.f, 0.f, 0.f};
        if (a.ys) shared = load4(a.ys + (int64_t)m * a.ld + c);
        for (int k0 = 0; k0 < a.top; k0 += 8) {
            f32x4 v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = load4(y + pair_row<PICKED>(a, m, k0 + k) * a.ld + c);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k0 + k < a.top) x[j] += v[k];
        }
        if (a.ys) x[j] += shared * gate;
        const bool own = tid + kCombineThreads * j < per;
        if (own) store4(a.x + (int64_t)m * a.ld + c, x[j]);
        squares[tid + kCombineThreads * j] = own ? x[j][0] * x[j][0] + x[j][1] * x[j][1] + x[j][2] * x[j][2] + x[j][3] * x[j][3] : 0.f;
    }
    __syncthreads();
    if (tid < 256) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < kCombineThreads / 256 * P; ++i) ss += squares[tid + 256 * i];
        ss = wave_sum(ss);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
    }
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)next.dim + next.eps);
#pragma unroll
    for (int j = 0; j < P; ++j)
        if (tid + kCombineThreads * j < per) store4(static_cast<bf16*>(next.h) + (int64_t)m * a.ld + 4 * (tid + kCombineThreads * j), x[j] * inv * w[j]);
}
template <typename Y, bool PICKED>
static int launch_combine_norm(const MoeArgs& a, const NextNorm& next, hipStream_t s) {
    const int p = (a.ld / 4 + kCombineThreads - 1) / kCombineThreads;
    if (p <= 1) moe_combine_norm_kernel<Y, 1, PICKED><<<dim3(a.M), dim3(kCombineThreads), 0, s>>>(a, next);
    else if (p <= 2) moe_combine_norm_kernel<Y, 2, PICKED><<<dim3(a.M), dim3(kCombineThreads), 0, s>>>(a, next);
    else moe_combine_norm_kernel<Y, 4, PICKED><<<dim3(a.M), dim3(kCombineThreads), 0, s>>>(a, next);
    return raven_host::check_launch("moe (combine, norm)");
}

// What runs the experts of M rows.  A chunk -- once its rows share weights (two per expert), or there are enough rows anyway -- keeps its slots in T
// and runs the shared expert as a product of its own.  Fewer rows keep slots and sums in float, as the row kernels do, and take the
// grouped products once reading each expert once saves more than their further launches cost.  us of a whole layer (a small recurrent unit in front), row kernels / grouped, means
// of four draws of picks: width 2048 (64 experts of 768 channels, 6 per row and a shared one) 2 rows 45 / 51, 3: 54 / 59, 4: 63 / 65, 6: 81 / 77, 8: 98 / 85, 16: 168 / 109; width
// 1024 (64 of 384) 4 rows 33 / 36, 6: 38 / 38, 8: 43 / 42, 12: 51 / 47; width 1024, one of 64 experts of 1024 and a shared one, 4 rows 31 / 34, 8: 38.5 / 37, 12: 45 / 41,
// 24: 68 / 51; width 4096, 2 of 8 experts of 4096, 2 rows 92 / 96, 3: 120 / 111, 8: 269 / 154.
enum MoePath { kMoeRows, kMoeFew, kMoeChunk };
constexpr size_t kMoeRowLds = 64 * 1024 - 1024;  // what a row may take of the row kernels' LDS; longer ones are refused for few rows
static bool few_rows_fit(const raven_moe* m, int M, int ld) {
    return (!m->shared_up || m->shared_ff == m->ff) && M >= 2 && M <= kRouteRows && M * m->top <= kRoutePairs && ld * sizeof(bf16) <= kMoeRowLds &&
           (int64_t)2 * m->ff * ld < (1ll << 31);
}
// Estimates in us, fitted to what 42 mixtures of 8 to 512 experts of 32 to 4096 channels at widths 256 to 7168 took with 2 to 32 rows, when the row kernels took 4 to 25 %
// longer and every batch was sorted.  Row kernels: weights as often as they are read, the shared expert's faster from the second row on, a share for
// each pick, and past 64 experts, where maxima pick, one for each workgroup that picks.  Grouped: four launches, and once the weights of the experts that rows
// pick on average, with a share for each.  Of two that are about the same, the row kernels.  With the present kernels the choice is 0.6 % slower than the better of the two on
// average, 13 % at most (layers of 16 mixtures of 8 to 300 experts at widths 256 to 4096, 111 calls; 40 experts of 384 at width 768, 4 per row, 12 rows: 39 / 34).
static bool grouping_pays(const raven_moe* m, int M, int ld) {
    const double pairs = (double)M * m->top, touched = m->experts * (1.0 - pow(1.0 - (double)m->top / m->experts, M)), shared = m->shared_up ? 1 : 0;
    const double expert = 6e-6 * ld * m->ff;  // MB
    const double rows = 7.4 + (pairs + shared) * expert / 6.1 + shared * (M - 1) * expert / 11 + pairs * (0.06 + (m->experts > 64 ? 0.57e-3 * m->ff : 0));
    const double grouped = 14.7 + (touched + shared) * (expert / 6.45 + 0.08);
    return grouped < 0.94 * rows;
}
// h: the rows, or null where only sizes are asked for.  The grouped kernels move whole 16-byte pieces into the LDS; operands that do not start
// on one stay with the row kernels, which take any address.
static MoePath moe_path(const raven_moe* m, const void* h, int M, int ld, int dtype) {
    if (dtype != RAVEN_BF16 || !raven_host::aligned16(h, m->up, m->down, m->shared_up, m->shared_down)) return kMoeRows;
    const double pairs = (double)M * m->top;
    if (M > 8 && (pairs >= 2.0 * m->experts || M > 128)) return kMoeChunk;
    if (!few_rows_fit(m, M, ld)) return kMoeRows;
    return grouping_pays(m, M, ld) ? kMoeFew : kMoeRows;
}

struct MoeChunk {
    int *pick, *slot_of, *slot_row, *group_of, *group_row, *group_end, *used, *block_count;
    void* y;
    float *pick_scale, *slot_scale, *ys;
    char *act, *sact, *lin;
    size_t lin_bytes;
    int n_tiles, tile_rows;
};
static size_t carve_moe(const raven_moe* m, int M, int ld, int dtype, MoePath path, char* base, MoeChunk* out) {
    const size_t es = raven_host::elt_size(dtype), pairs = (size_t)M * m->top;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char* p = base ? base + off : nullptr;
        off += raven_host::align_up(bytes);
        return p;
    };
    MoeChunk c{};
    if (path == kMoeRows) {
        c.act = take((size_t)M * (m->top * (size_t)m->ff + m->shared_ff) * es);
        c.pick = (int*)take(pairs * 4);
    } else {
        const bool fold = path == kMoeFew && m->shared_up;
        const size_t rows = pairs + (fold ? M : 0);
        // The smallest tile that most experts' rows fit into; 256 (by the ring kernel, twice the speed per row) from an average of 110 on, if
        // its units -- a tile by 128 channels of `up` or 256 of `down` -- fill the chip's 256 CUs over both products.  us for all launches of a mixture, width 2048, tiles of 16 / 32 / 64 / 256 rows: 100 tokens 169 / 163 / 167 / 218, 500:
        // 232 / 196 / 181 / 232 (16 rows as gemm_mid.hip took them), 1000: 344 / 255 / 218 / 249, 1500: 474 / 340 / 282 / 272, 4096: - / 695 / 518 / 394; width 1024, 500
        // tokens: 80 / 70 / 63 / 83, 1500: 144 / 109 / 94 / 96.  (128-row tiles of eight waves, as before: 230 at 500, 327 at 1500.)
        // Few units, tiles of 64 / 256: 12 experts of 136 at width 256, 2 per row, 1000 tokens 29 / 47; 16 of 768 at 1024, 1000 tokens 73 / 93, 4000
        // (400 units) 136 / 120; 8 of 2048 at 2048, 500 tokens (190) 105 / 116, 1000 (280) 134 / 122.
        // 16 rows by expert_rows_kernel against 32: 64 experts, 6 per row, 100 tokens (9 per expert) at widths 1024 / 1536 / 2048 / 2304 61 / 65, 90 / 104,
        // 136 / 157, 166 / 182; 150 (14) 65 / 66, 101 / 107, 154 / 161, 204 / 187; 200 (18) 72 / 67, 121 / 109, 178 / 168, 259 / 193.
        // Many experts so small that expert_rows_kernel's units are over before their loads overlap: 32 from three per expert on.  us by 16 / 32, 8 per row: 300 of 136
        // at width 264, 130 tokens 49 / 47.5, 300: 52 / 50; 256 of 64 at 256, 200: 38 / 36; 128 of 128 at 512, 130: 51 / 48; 300 of 256 at 256, 300: 60.5 / 58;
        // but 300 of 256 at 512, 300: 74 / 78; 200 of 384 at 384, 130: 64 / 67.5; 128 of 128 at 768, 130: 46.1 / 46.4; 64 of 128 at 256, 40: 25 / 27.
        const size_t mean = pairs / m->experts;
        const bool small = (ld < 320 || (size_t)ld * m->ff <= 80 * 1024) && (size_t)m->experts * ((m->ff + 15) / 16 + (ld + 31) / 32) >= 2500;
        const size_t big_tiles = pairs / 256 + m->experts / 2;  // an expert's last tile is half full on average
        const bool fills = big_tiles * ((m->ff + 127) / 128 + (ld + 255) / 256) > 256;
        c.tile_rows = path == kMoeFew || mean <= (small ? 2 : 10) ? 16 : mean <= 20 ? 32 : mean < kBigTileRows || !fills ? 64 : 256;
        auto tiles = [&](int height) { return (int)(pairs / height) + m->experts + (fold ? (M + height - 1) / height : 0); };
        c.n_tiles = tiles(c.tile_rows);
        const size_t table = (size_t)tiles(16) * 4;  // room for the lowest tiles whatever the height, so that more rows never need less
        c.pick = (int*)take(pairs * 4);
        c.pick_scale = (float*)take(pairs * 4);
        c.slot_of = (int*)take(pairs * 4);
        c.slot_row = (int*)take(rows * 4);
        c.slot_scale = (float*)take(rows * 4);
        c.group_of = (int*)take(table);
        c.group_row = (int*)take(table);
        c.group_end = (int*)take(table);
        c.used = (int*)take(4);
        c.block_count = (int*)take((size_t)((M + kPickRows - 1) / kPickRows) * m->experts * 4);
        c.act = take(rows * m->ff * es);
        c.y = take(rows * ld * (path == kMoeFew ? sizeof(float) : sizeof(bf16)));
        if (fold) {
            c.ys = static_cast<float*>(c.y) + pairs * ld;
        } else if (m->shared_up) {
            c.sact = take((size_t)M * m->shared_ff * es);
            c.ys = (float*)take((size_t)M * ld * sizeof(float));
            c.lin_bytes = raven_linear_workspace_bytes(M, ld > 2 * m->shared_ff ? ld : 2 * m->shared_ff);
            c.lin = take(c.lin_bytes);
        }
    }
    if (out) *out = c;
    return off;
}

// Room for M rows and for any smaller number: a grouped call over few rows keeps float slots and can need more than row kernels or a
// chunk over more rows do (64 experts, 8 per row, no shared one: 15 rows 1.17 MB, 16 rows 0.73)
static size_t moe_workspace(const raven_moe* m, int M, int ld, int dtype) {
    size_t need = carve_moe(m, M, ld, dtype, kMoeRows, nullptr, nullptr);
    if (dtype != RAVEN_BF16) return need;
    const int few = M < kRouteRows ? M : kRouteRows;
    if (few_rows_fit(m, few, ld)) need = std::max(need, carve_moe(m, few, ld, dtype, kMoeFew, nullptr, nullptr));
    if (moe_path(m, nullptr, M, ld, dtype) == kMoeChunk) need = std::max(need, carve_moe(m, M, ld, dtype, kMoeChunk, nullptr, nullptr));
    return need;
}

static int check_moe(const char* who, const raven_moe* m, int M, int ld, int dtype) {
    RAVEN_REQUIRE(dtype == RAVEN_F32 || dtype == RAVEN_BF16, "%s: unknown dtype %d", who, dtype);
    RAVEN_REQUIRE(m && m->experts > 0 && m->experts <= kMaxExperts && m->top > 0 && m->top <= m->experts && m->top <= kMaxTop, "%s: bad experts / top", who);
    RAVEN_REQUIRE(m->ff > 0 && m->ff % 8 == 0 && m->shared_ff >= 0 && m->shared_ff % 8 == 0 && ld > 0 && ld % 8 == 0 && M >= 0, "%s: bad sizes", who);
    RAVEN_REQUIRE(m->logit_ld >= m->experts + (m->shared_up ? 1 : 0), "%s: bad logit pitch %d", who, m->logit_ld);
    RAVEN_REQUIRE((m->shared_up == nullptr) == (m->shared_ff == 0) && (m->shared_up == nullptr) == (m->shared_down == nullptr), "%s: incomplete shared expert", who);
    return 0;
}

template <typename T>
static int run_moe_rows(const MoeArgs& a, hipStream_t s) {
    const size_t lds = (size_t)a.ld * sizeof(T);
    RAVEN_REQUIRE(lds <= kMoeRowLds, "moe: rows of %d channels do not fit the LDS", a.ld);
    const int total = a.top * a.ff + a.sff;
    const dim3 up((total + 3) / 4, a.M), down((a.ld + 3) / 4, a.M);
    if (picks_by_place(a.experts, a.top)) moe_up_place_kernel<T><<<up, dim3(256), lds, s>>>(a);
    else moe_up_kernel<T><<<up, dim3(256), lds, s>>>(a);
    // the fewest rounds of at most 12 pieces, of equal length
    const int pieces = (total / Chunk<T>::N + 63) / 64, rounds = (pieces + 11) / 12;
    switch (((pieces + rounds - 1) / rounds + 1) / 2) {
        case 1: moe_down_kernel<T, 2><<<down, dim3(256), 0, s>>>(a); break;
        case 2: moe_down_kernel<T, 4><<<down, dim3(256), 0, s>>>(a); break;
        case 3: moe_down_kernel<T, 6><<<down, dim3(256), 0, s>>>(a); break;
        case 4: moe_down_kernel<T, 8><<<down, dim3(256), 0, s>>>(a); break;
        case 5: moe_down_kernel<T, 10><<<down, dim3(256), 0, s>>>(a); break;
        default: moe_down_kernel<T, 12><<<down, dim3(256), 0, s>>>(a); break;
    }
    return raven_host::check_launch("moe (rows)");
}

}  // namespace raven

extern "C" size_t raven_moe_workspace_bytes(const raven_moe* m, int32_t M, int32_t ld, int32_t dtype) {
    if (raven::check_moe("moe_workspace_bytes", m, M, ld, dtype) || M == 0) return 0;
    return raven::moe_workspace(m, M, ld, dtype);
}

namespace raven {
// Rows behind a norm that is shared out between two products, which route themselves (moe_forward_picked)
bool moe_picks_itself(const raven_moe* m, const void* h, int M, int ld, int dtype) {
    return moe_path(m, h, M, ld, dtype) == kMoeFew && M <= kPickedRows && m->experts <= 64 && ld <= 16 * kNormParts && ld % 16 == 0 && raven_host::aligned16(m->router);
}
// Router, experts and sums of M rows: xw and behind as NormAhead left them; logits and factors are written.  next_norm, next_h: as for moe_forward
int moe_forward_picked(const raven_moe* m, const void* xw, const NormBehind& behind, float* factors, float* logits, float* x, int M, int ld, float eps, int dim, void* workspace,
                       size_t workspace_bytes, hipStream_t s, const float* next_norm, void* next_h) {
    if (const int rc = check_moe("moe", m, M, ld, RAVEN_BF16)) return rc;
    RAVEN_REQUIRE(m->up && m->down && m->router && xw && behind.squares && behind.parts > 0 && behind.parts <= kNormParts && factors && logits && x &&
                      moe_picks_itself(m, xw, M, ld, RAVEN_BF16), "moe: %d rows don't pick for themselves", M);
    RAVEN_REQUIRE(!next_norm || (next_h && dim > 0 && ld <= 16 * kCombineThreads), "moe: no norm behind %d rows", M);
    RAVEN_REQUIRE(workspace && ((uintptr_t)workspace & 255) == 0 && carve_moe(m, M, ld, RAVEN_BF16, kMoeFew, nullptr, nullptr) <= workspace_bytes,
                  "moe: workspace of %zu bytes is too small or unaligned", workspace_bytes);
    MoeChunk c;
    carve_moe(m, M, ld, RAVEN_BF16, kMoeFew, static_cast<char*>(workspace), &c);
    const bool fold = m->shared_up != nullptr;
    MoeArgs a{};
    a.h = xw; a.up = m->up; a.down = m->down; a.shared_up = m->shared_up; a.shared_down = m->shared_down;
    a.logits = logits; a.x = x; a.factors = factors; a.pick = c.pick; a.pick_scale = c.pick_scale;
    a.M = M; a.ld = ld; a.ldl = m->logit_ld; a.experts = m->experts; a.top = m->top; a.ff = m->ff; a.sff = m->shared_ff;
    a.y = c.y; a.ys = c.ys; a.fold = fold;
    const bf16* router = static_cast<const bf16*>(m->router);
    switch ((ld / 8 + 63) / 64) {
        case 1: pick_rows_kernel<1><<<dim3(M), dim3(1024), 0, s>>>(a, router, behind, logits, factors); break;
        case 2: pick_rows_kernel<2><<<dim3(M), dim3(1024), 0, s>>>(a, router, behind, logits, factors); break;
        case 3: pick_rows_kernel<3><<<dim3(M), dim3(1024), 0, s>>>(a, router, behind, logits, factors); break;
        case 4: pick_rows_kernel<4><<<dim3(M), dim3(1024), 0, s>>>(a, router, behind, logits, factors); break;
        case 5: pick_rows_kernel<5><<<dim3(M), dim3(1024), 0, s>>>(a, router, behind, logits, factors); break;
        default: pick_rows_kernel<6><<<dim3(M), dim3(1024), 0, s>>>(a, router, behind, logits, factors); break;
    }
    if (const int rc = raven_host::check_launch("moe (router, picks)")) return rc;
    RowGroups g{};
    g.x_scale = c.pick_scale; g.w_stride = (int64_t)2 * m->ff * ld; g.w_extra = static_cast<const bf16*>(m->shared_up); g.extra_group = fold ? m->experts : -1;
    if (const int rc = picked_expert_rows(xw, m->up, c.act, m->ff, ld, true, g, a, s)) return rc;
    g.w_stride = (int64_t)ld * m->ff; g.w_extra = static_cast<const bf16*>(m->shared_down);
    if (const int rc = picked_expert_rows(c.act, m->down, c.y, ld, m->ff, false, g, a, s)) return rc;
    if (next_norm) return launch_combine_norm<float, true>(a, NextNorm{next_norm, next_h, dim, eps}, s);
    moe_combine_kernel<float, true><<<dim3((unsigned)(((int64_t)M * (ld / 4) + 255) / 256)), dim3(256), 0, s>>>(a);
    return raven_host::check_launch("moe (combine)");
}
// Whether moe_forward applies rows' factors of its own for so many rows
bool moe_norms_behind(const raven_moe* m, const void* h, int M, int ld, int dtype) {  // ... and whether it can end with the norm that the next layer begins with
    return moe_path(m, h, M, ld, dtype) != kMoeRows && ld <= 16 * kCombineThreads;
}
bool moe_takes_factors(const raven_moe* m, const void* h, int M, int ld, int dtype) {
    return moe_path(m, h, M, ld, dtype) == kMoeFew && (!m->shared_up || m->shared_ff == m->ff);
}
// h null (one row): moe_up_kernel norms the row of x itself.  factors: the rows of the experts' inputs are these times h (moe_takes_factors).  next_norm, next_h (may be
// null): the norm of the rows that result, with dim and eps (moe_norms_behind)
int moe_forward(const raven_moe* m, const void* h, const float* factors, const float* norm, int dim, float eps, const float* logits, float* x, int M, int ld, int dtype,
                void* workspace, size_t workspace_bytes, hipStream_t s, const float* next_norm, void* next_h) {
    if (const int rc = check_moe("moe", m, M, ld, dtype)) return rc;
    if (M == 0) return 0;
    RAVEN_REQUIRE(m->up && m->down && (h || (norm && M == 1)) && logits && x, "moe: null pointer");
    const MoePath path = moe_path(m, h, M, ld, dtype);
    RAVEN_REQUIRE(!factors || path == kMoeFew, "moe: factors of %d rows", M);
    RAVEN_REQUIRE(!next_norm || (next_h && dim > 0 && dtype == RAVEN_BF16 && moe_norms_behind(m, h, M, ld, dtype)), "moe: no norm behind %d rows", M);
    RAVEN_REQUIRE(workspace && ((uintptr_t)workspace & 255) == 0 && carve_moe(m, M, ld, dtype, path, nullptr, nullptr) <= workspace_bytes,
                  "moe: workspace of %zu bytes is too small or unaligned", workspace_bytes);
    MoeChunk c;
    carve_moe(m, M, ld, dtype, path, static_cast<char*>(workspace), &c);
    MoeArgs a{};
    a.h = h; a.up = m->up; a.down = m->down; a.shared_up = m->shared_up; a.shared_down = m->shared_down;
    a.logits = logits; a.x = x; a.act = c.act; a.norm = norm; a.dim = dim; a.eps = eps; a.pick = c.pick;
    a.M = M; a.ld = ld; a.ldl = m->logit_ld; a.experts = m->experts; a.top = m->top; a.ff = m->ff; a.sff = m->shared_ff;
    if (path == kMoeRows) {
        RAVEN_REQUIRE(M <= 65535, "moe: %d rows in one call", M);
        return dtype == RAVEN_BF16 ? run_moe_rows<bf16>(a, s) : run_moe_rows<float>(a, s);
    }
    const int pairs = M * m->top, blocks = (M + kPickRows - 1) / kPickRows;
    const bool fold = path == kMoeFew && m->shared_up, few = path == kMoeFew;
    const int rows = pairs + (fold ? M : 0);
    a.pick_scale = c.pick_scale; a.slot_of = c.slot_of; a.slot_row = c.slot_row; a.slot_scale = c.slot_scale;
    a.group_of = c.group_of; a.group_row = c.group_row; a.group_end = c.group_end; a.used = c.used; a.tile_rows = c.tile_rows; a.block_count = c.block_count;
    a.y = c.y; a.ys = c.ys; a.fold = fold; a.factors = factors;
    // one workgroup picks for 16 rows at a time: from 33 rows on two launches of several are sooner done (64 rows, 2 of 12 experts of 136 at
    // width 256, the whole mixture 27.5 / 25.3 us; 4 of 32 of 96 43 / 39)
    if (few || (M <= kPickRows && pairs <= kRoutePairs)) {
        moe_route_kernel<<<dim3(1), dim3(1024), 0, s>>>(a);
    } else {
        moe_pick_kernel<<<dim3(blocks), dim3(1024), 0, s>>>(a);
        moe_sort_kernel<<<dim3(blocks), dim3(1024), 0, s>>>(a);
    }
    if (const int rc = raven_host::check_launch("moe (sort)")) return rc;
    const int64_t up_stride = (int64_t)2 * m->ff * ld, down_stride = (int64_t)ld * m->ff;
    RowGroups g{c.group_of, c.group_row, c.group_end, c.used, c.n_tiles, c.tile_rows, c.slot_row, c.slot_scale, up_stride,
                fold ? static_cast<const bf16*>(m->shared_up) : nullptr, fold ? m->experts : -1};
    const bool ring = c.tile_rows == 256, low = c.tile_rows == 16;
    int rc = ring ? ring_grouped(h, M, m->up, c.act, rows, m->ff, ld, 1, g, s)
             : low ? expert_rows(h, m->up, c.act, m->ff, ld, true, 0, g, s) : mid_grouped(h, M, m->up, c.act, rows, m->ff, ld, 1, 0, g, s);
    if (rc) return rc;
    g.x_row = nullptr; g.x_scale = nullptr; g.w_stride = down_stride;
    g.w_extra = fold ? static_cast<const bf16*>(m->shared_down) : nullptr;
    rc = ring ? ring_grouped(c.act, rows, m->down, c.y, rows, ld, m->ff, 0, g, s)
         : low ? expert_rows(c.act, m->down, c.y, ld, m->ff, false, few, g, s) : mid_grouped(c.act, rows, m->down, c.y, rows, ld, m->ff, 0, few, g, s);
    if (rc) return rc;
    if (m->shared_up && !fold) {
        raven_epilogue e{};
        e.scale = 1.f; e.out_f32 = 1;
        if (const int rc = raven_linear(h, nullptr, m->shared_up, nullptr, c.sact, M, m->shared_ff, ld, 0, 1, 0, dtype, c.lin, c.lin_bytes, s)) return rc;
        if (const int rc = raven_linear_epilogue(c.sact, nullptr, m->shared_down, c.ys, M, ld, m->shared_ff, 0, &e, dtype, c.lin, c.lin_bytes, s)) return rc;
    }
    if (next_norm) {
        const NextNorm next{next_norm, next_h, dim, eps};
        return few ? launch_combine_norm<float, false>(a, next, s) : launch_combine_norm<bf16, false>(a, next, s);
    }
    const dim3 grid((unsigned)(((int64_t)M * (ld / 4) + 255) / 256));
    if (few) moe_combine_kernel<float, false><<<grid, dim3(256), 0, s>>>(a);
    else moe_combine_kernel<bf16, false><<<grid, dim3(256), 0, s>>>(a);
    return raven_host::check_launch("moe (combine)");
}
}  // namespace raven

extern "C" int raven_moe_plan(const raven_moe* m, int32_t M, int32_t ld, int32_t dtype, int32_t* plan) {
    RAVEN_REQUIRE(plan, "moe_plan: null pointer");
    plan[0] = plan[1] = 0;
    if (const int rc = raven::check_moe("moe_plan", m, M, ld, dtype)) return rc;
    if (M == 0) return 0;
    plan[0] = raven::moe_path(m, nullptr, M, ld, dtype);
    plan[1] = raven::moe_picks_itself(m, nullptr, M, ld, dtype);
    return 0;
}

extern "C" int raven_moe_forward(const raven_moe* m, const void* h, const float* logits, float* x, int32_t M, int32_t ld, int32_t dtype,
                                 void* workspace, size_t workspace_bytes, void* stream) {
    RAVEN_REQUIRE(h || M == 0, "moe: null pointer");
    return raven::moe_forward(m, h, nullptr, nullptr, 0, 0.f, logits, x, M, ld, dtype, workspace, workspace_bytes, static_cast<hipStream_t>(stream), nullptr, nullptr);
}
