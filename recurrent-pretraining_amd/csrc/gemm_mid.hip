// Matrix-core products over a middling number of token rows (33 to a few thousand): Y[M,N] = concat(X0, X1)[M,K] W[N,K]^T in bf16 with fp32
// accumulation, with the epilogues of gemm_tiled.hip -- prompts of ordinary length, decode batches past 32 sequences, a serving engine's
// mixed steps, and long prompts against matrices too narrow to give every CU a 256 x 256 tile.
//
// What bounds these products is keeping weight bytes in flight (few rows) and the LDS (many), so
//   * operands go global -> LDS directly through a ring of NS stages, NS - 1 K steps of 64 ahead: 60 to 120 KB in flight on every CU, where
//     two stages behind staging registers left one step in flight (mlp.fc of the 3.5b shape at 93 rows: 3.2 TB/s);
//   * a unit owns `cols` output columns -- not whole tiles: as many as leave the chip ONE nearly full round of units (17920 gate columns =
//     249 x 72), the last 16-row tile partly filled; missing rows are clamped on the load side and not stored;
//   * where even the narrowest unit leaves CUs idle, K is cut into slices: fp32 sums in the workspace, added in slice order by a second
//     launch or by the norm that follows (splitk_sums_then_norm);
//   * 8 waves, two along the weight rows and four along the token rows, a wave NT x MT tiles of 16 x 16 (v_mfma_f32_16x16x32_bf16, W rows
//     as the A operand): two waves per SIMD hide each other's LDS reads; one barrier per K step.
// LDS rows are 128 bytes, 16-byte piece c of row r at position c ^ ((r >> 1) & 7) (applied on the global side), so that fragment reads are
// free of bank conflicts.  Unlike the tiles of gemm_tiled.hip a wave's partial sums over K slices are added after the fact, so results
// differ from those in the order of fp32 sums.
//
// us per launch at 93 rows of the 3.5b shape, weights from HBM (those of K = 5280 through their line-aligned copies), 128 x 128 tiles or passes of 32
// rows before / this kernel (both launches where K is split): Wqkv 68 / 52, attn.proj 62 / 26, mlp.fc 125 / 91, mlp.proj 112 / 55, adapter 78 / 38; at
// 195 rows 67 / 63, 59 / 35, 158 / 128, 188 / 83, 113 / 56; at 45 rows Wqkv 67 / 37, mlp.fc 110 / 74 (5.1 TB/s of weights), mlp.proj 72 / 43;
// 4096 x 2048 x 8192 with an fp32 residual 163 / 133.

#include "gemm_common.h"

namespace raven {

struct MidArgs {
    const bf16 *w, *x0, *x1, *residual;
    void* y;
    float* partial;        // [ks, M, N or 2N] when ks > 1
    int M, N, K0, K1, ldw, ldx;
    int out_f32;
    int cols, bm;          // output columns / token rows of a unit
    int wrows;             // LDS rows of a unit's weight tile (whole 16-row tiles)
    int tiles_m, tiles_n, ks;
    raven_epilogue epi;    // EPI_FREE only
    int rope_on;           // EPI_PLAIN: the rope epilogue instead of y
    RopeAppend rope;
    RowGroups groups;      // GROUPED only
};

__device__ __align__(16) unsigned int g_mid_zero[4];  // what a 16-byte piece past the end of K is loaded from

// Four neighbouring output columns n .. n + 3 of token row m; xs: the factor of a grouped SwiGLU row
template <int EPI, bool GROUPED = false>
__device__ __forceinline__ void mid_store(const MidArgs& a, int m, int n, f32x4 v, f32x4 up, float xs = 1.f) {
    const int64_t at = (int64_t)m * a.N + n;
    if constexpr (EPI == EPI_SWIGLU) {
        bf16 o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (GROUPED) {
                o[i] = from_f32<bf16>(silu_f32(v[i] * xs) * (up[i] * xs));
                continue;
            }
            const float g = round_to<bf16>(v[i]), u = round_to<bf16>(up[i]);
            o[i] = from_f32<bf16>(round_to<bf16>(silu_f32(g)) * u);
        }
        *reinterpret_cast<u32x2*>(static_cast<bf16*>(a.y) + at) = *reinterpret_cast<const u32x2*>(o);
    } else if constexpr (is_free(EPI)) {
        v *= a.epi.scale;
        if (a.epi.bias) v += *reinterpret_cast<const f32x4*>(a.epi.bias + n);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (EPI == EPI_FREE_GELU) v[i] = gelu_f32<bf16>(v[i]);
            if (EPI == EPI_FREE_TANH) v[i] = tanhf(v[i]);
        }
        if (a.epi.residual) v += *reinterpret_cast<const f32x4*>(a.epi.residual + at);
        if (a.out_f32) {
            *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + at) = v;
        } else {
            bf16 o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = from_f32<bf16>(v[i]);
            *reinterpret_cast<u32x2*>(static_cast<bf16*>(a.y) + at) = *reinterpret_cast<const u32x2*>(o);
        }
    } else {
        bf16 o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = from_f32<bf16>(v[i]);
        if (a.rope_on) {
            const RopeAppend& r = a.rope;
            const int h = r.nh * r.hd, sec = n >= 2 * h ? 2 : (n >= h ? 1 : 0);  // q, k or v columns; four of them lie in one head
            const int col = n - sec * h, head = col / r.hd, d = col - head * r.hd;
            const int b = m / r.S, sq = m - b * r.S, pos = (r.pos_dev ? *r.pos_dev : r.pos0) + sq;
            if (sec < 2) {
                if (r.qk_bias) {
                    bf16 bias[4];
                    *reinterpret_cast<u32x2*>(bias) = *reinterpret_cast<const u32x2*>(r.qk_bias + sec * h + col);
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = from_f32<bf16>(to_f32(o[i]) + to_f32(bias[i]));
                }
                const f32x4 f = *reinterpret_cast<const f32x4*>(r.freqs + (int64_t)pos * r.hd + d);  // (cos, sin) of two pairs
                rope_pair<bf16>(o[0], o[1], f[0], f[1]);
                rope_pair<bf16>(o[2], o[3], f[2], f[3]);
            }
            bf16* out = r.q_out + (int64_t)m * h + col;
            if (sec > 0) {
                if (pos >= r.t_max) return;
                out = (sec == 1 ? r.k : r.v) + r.slot_off + (((int64_t)b * r.nh + head) * r.t_max + pos) * r.hd + d;
            }
            *reinterpret_cast<u32x2*>(out) = *reinterpret_cast<const u32x2*>(o);
            return;
        }
        if (a.residual) {
            bf16 res[4];
            *reinterpret_cast<u32x2*>(res) = *reinterpret_cast<const u32x2*>(a.residual + at);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = from_f32<bf16>(to_f32(o[i]) + to_f32(res[i]));
        }
        if (a.out_f32) *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + at) = f32x4{to_f32(o[0]), to_f32(o[1]), to_f32(o[2]), to_f32(o[3])};
        else *reinterpret_cast<u32x2*>(static_cast<bf16*>(a.y) + at) = *reinterpret_cast<const u32x2*>(o);
    }
}

// GROUPED: row groups with a weight matrix each; a unit works on a copy of the arguments cut to its group's rows
template <int EPI, int WN, int WM, int NT, int MT, int NS, bool GROUPED = false>
__global__ __launch_bounds__(64 * WN * WM) void gemm_mid_kernel(MidArgs a) {
    constexpr bool SWIGLU = EPI == EPI_SWIGLU;
    constexpr int NW = WN * WM, XROWS = 16 * WM * MT, XP = XROWS / 8;
    // kilobyte pieces (8 rows x 128 bytes) a wave requests per step; with fewer token pieces than waves some are requested twice
    constexpr int WPW = 2 * NT / WM, XPW = XP >= NW ? XP / NW : 1, LPW = WPW + XPW;
    static_assert(NT % 2 == 0 && (2 * NT) % WM == 0 && (XP % NW == 0 || NW % XP == 0) && (NS - 1) * LPW < 64, "whole pieces; the wait counter holds 63 requests");
    extern __shared__ __align__(1024) unsigned char smem[];

    // which unit: K slices outermost, then bands of eight token tiles, so that the units of an XCD (ids congruent modulo 8) are neighbours
    if (GROUPED) a.tiles_m = *a.groups.used;
    const int mn = a.tiles_m * a.tiles_n, n_units = mn * a.ks;
    const int per_xcd = (n_units + 7) >> 3;
    const int logical = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
    if (logical >= n_units || ((int)blockIdx.x >> 3) >= per_xcd) return;
    const int slice = logical / mn, in_slice = logical - slice * mn;
    constexpr int GROUP = 8;
    const int band = in_slice / (GROUP * a.tiles_n), first_m = band * GROUP, gsz = min(a.tiles_m - first_m, GROUP);
    const int in_band = in_slice - band * GROUP * a.tiles_n, tile_n = in_band / gsz;
    int tile_m = first_m + (in_band - tile_n * gsz);
    const int* x_row = nullptr;
    if constexpr (GROUPED) {
        const int g = a.groups.group_of[tile_m], row = a.groups.group_row[tile_m];
        a.M = a.groups.group_end[tile_m] - row;
        a.w = g == a.groups.extra_group ? a.groups.w_extra : a.w + g * a.groups.w_stride;
        a.y = static_cast<char*>(a.y) + (int64_t)row * a.N * (a.out_f32 ? 4 : 2);
        if (a.groups.x_scale) a.groups.x_scale += row;
        if (a.groups.x_row) x_row = a.groups.x_row + row;
        else a.x0 += (int64_t)row * a.ldx;
        tile_m = 0;
    }

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, wm = wave / WN;
    const int K = a.K0 + a.K1, nk = (K + 63) >> 6;
    const int k0 = __builtin_amdgcn_readfirstlane((int)((int64_t)nk * slice / a.ks));
    const int n_steps = __builtin_amdgcn_readfirstlane((int)((int64_t)nk * (slice + 1) / a.ks)) - k0;
    const int n0 = tile_n * a.cols, ncols = min(a.cols, a.N - n0), m0 = tile_m * a.bm;
    const int wbytes = a.wrows * 128, stage = wbytes + XROWS * 128;
    const unsigned lds_base = (unsigned)(uintptr_t)(lds_byte*)smem;

    // ---- global side: request i of a wave is piece NW i + wave, rows 8 (NW i + wave) ..+7 of the weight tile (i < WPW) or of the token
    // rows; the lane that fills position s of row r fetches piece s ^ ((r >> 1) & 7) of the row's 128-byte step
    const int colp = ((lane & 7) ^ ((lane >> 4) | (4 * (wave & 1)))) * 8;
    unsigned goff[LPW];
    unsigned dst[LPW];  // offset inside a stage; weight pieces past the tile land behind the ring
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const bool is_w = i < WPW;
        const int piece = is_w ? NW * i + wave : (NW * (i - WPW) + wave) % XP, r = piece * 8 + (lane >> 3);
        if (is_w) {
            int row;
            if (SWIGLU) row = n0 + min((r >> 5) * 16 + (r & 15), ncols - 1) + ((r & 16) ? a.N : 0);
            else row = n0 + min(r, ncols - 1);
            goff[i] = (unsigned)row * (2u * a.ldw) + 2u * colp;
            dst[i] = piece * 1024;
        } else {
            int row = min(m0 + r, a.M - 1);
            if (GROUPED && x_row) row = x_row[row];
            goff[i] = (unsigned)row * (2u * a.ldx) + 2u * colp;
            dst[i] = wbytes + piece * 1024;
        }
    }
    const char* const zero = reinterpret_cast<const char*>(g_mid_zero);
    const char* const w0 = reinterpret_cast<const char*>(a.w);
    const char* const x0 = reinterpret_cast<const char*>(a.x0);
    const char* const x1 = reinterpret_cast<const char*>(a.x1) - 2 * (int64_t)a.K0;  // column c >= K0 of the token rows
    // requests FIRST .. LAST - 1 of step kk (columns 64 kk ..+63; zeros past K) into the stage at offset o
    auto issue = [&](int kk, int o, auto first_tag, auto last_tag) __attribute__((always_inline)) {
        const int c0 = kk << 6;
        const bool whole = c0 + 64 <= a.K0 || (c0 >= a.K0 && c0 + 64 <= K);  // the 64 columns lie in one segment and below K
#pragma unroll
        for (int i = decltype(first_tag)::value; i < decltype(last_tag)::value; ++i) {
            const bool is_w = i < WPW;
            const bool spare = is_w && (NW * i + wave) * 8 >= a.wrows;
            const unsigned to = __builtin_amdgcn_readfirstlane(lds_base + (spare ? NS * stage : o + (int)dst[i]));
            if (whole) {
                const char* base = (is_w ? w0 : (c0 < a.K0 ? x0 : x1)) + 2 * c0;
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(goff[i]), "s"(base), "s"(to) : "memory");
            } else {
                const int col = c0 + colp;
                const char* gp = col >= K ? zero : (is_w ? w0 : (col < a.K0 ? x0 : x1)) + 2 * c0 + goff[i];
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gp), "s"(to) : "memory");
            }
        }
    };

    // ---- LDS -> registers -> products
    const int l16 = lane & 15, q4 = lane >> 4;
    const unsigned pos0 = (q4 ^ ((l16 >> 1) & 7)) * 16;  // k-slice s of a step: pos0 ^ (64 s)
    const unsigned a_row = lds_base + (wn * NT * 16 + l16) * 128, b_row = lds_base + wbytes + (wm * MT * 16 + l16) * 128;
    const int used = min(max((a.wrows >> 4) - wn * NT, 0), NT);  // weight tiles of this wave that exist
    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 fa[2][NT], fb[2][MT];  // fragments of the two k-slices of a step
    auto fetch = [&](int o, auto sl_tag, auto full_tag) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full_tag)::value;
        constexpr int sl = decltype(sl_tag)::value;
        const unsigned ra = a_row + o + (pos0 ^ (64 * sl)), rb = b_row + o + (pos0 ^ (64 * sl));
        if (!FULL && used == 0) return;
#pragma unroll
        for (int j = 0; j < MT; ++j) fb[sl][j] = *reinterpret_cast<const lds_u32x4*>(rb + j * 2048);
#pragma unroll
        for (int t = 0; t < NT; ++t)  // (a tile that does not exist repeats the last one; its products are never stored)
            fa[sl][t] = *reinterpret_cast<const lds_u32x4*>(ra + (FULL ? t : min(t, used - 1)) * 2048);
    };
    auto multiply = [&](auto sl_tag, auto full_tag) __attribute__((always_inline)) {
        constexpr int sl = decltype(sl_tag)::value;
        if (!decltype(full_tag)::value && used == 0) return;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < MT; ++j)
                acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fa[sl][t]), __builtin_bit_cast(bf16x8, fb[sl][j]), acc[t][j], 0, 0, 0);
    };

    // ---- the ring: step i sits in stage i mod NS.  The barrier in the middle of step i says that every wave's requests of step i + 1 have
    // landed and that every wave has read out step i, whose stage step i + NS then takes.  The fragments of a slice are read under the
    // products of the slice before, the requests stand between the two slices' products: with reads, requests and products of all eight
    // waves one after the other behind the barrier a step took the sum of the three (Wqkv of the 3.5b shape at 93 rows 46 us).
    const int ring = NS * stage;
    using ic0 = std::integral_constant<int, 0>;
    using ic1 = std::integral_constant<int, 1>;
    using half = std::integral_constant<int, (LPW + 1) / 2>;
    using all = std::integral_constant<int, LPW>;
    auto arrive = [&](auto left_tag) __attribute__((always_inline)) {  // all but the requests of `left` steps have landed
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left_tag)::value * LPW) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    // lanes of a wave exchange data through LDS without a workgroup barrier: pin the order of the accesses for the compiler
    auto wave_sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto run = [&](auto full_tag) __attribute__((always_inline)) {
        int o = 0, i = 0;
        arrive(std::integral_constant<int, NS - 2>{});
        fetch(0, ic0{}, full_tag);
#pragma unroll 1
        for (; i + NS - 1 < n_steps; ++i) {
            const int free = o == 0 ? ring - stage : o - stage, next = o + stage == ring ? 0 : o + stage;
            fetch(o, ic1{}, full_tag);
            issue(k0 + i + NS - 1, free, ic0{}, half{});
            multiply(ic0{}, full_tag);
            issue(k0 + i + NS - 1, free, half{}, all{});
            arrive(std::integral_constant<int, NS - 2>{});
            fetch(next, ic0{}, full_tag);
            multiply(ic1{}, full_tag);
            o = next;
        }
        static_for<NS - 1>([&](auto j_tag) {  // nothing more to request
            constexpr int j = decltype(j_tag)::value;
            if (i < n_steps) {
                const int next = o + stage == ring ? 0 : o + stage;
                fetch(o, ic1{}, full_tag);
                multiply(ic0{}, full_tag);
                if constexpr (j < NS - 2) {
                    if (i + 1 < n_steps) {
                        arrive(std::integral_constant<int, NS - 3 - j>{});
                        fetch(next, ic0{}, full_tag);
                    }
                }
                multiply(ic1{}, full_tag);
                o = next;
                ++i;
            }
        });
    };
#pragma unroll 1
    for (int i = 0; i < NS - 1; ++i) issue(k0 + i, i * stage, ic0{}, all{});
    if (used == NT) run(std::true_type{});
    else run(std::false_type{});
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // requests past a short slice still write into the ring

    // ---- out: a lane holds columns 16 t + 4 q4 ..+3 of token row 16 j + l16.  A wave lays its sums down in LDS, rows of its columns,
    // and a rolled loop takes them from there: whole runs of columns per store, and little code -- unrolled over the accumulators
    // the epilogue ran once per unit out of a cold instruction cache (gelu outputs of 3000 x 4096 x 1024: 46 us, as a loop 36).
    __builtin_amdgcn_s_barrier();  // every wave has left the ring
    constexpr int JG = MT < 2 ? MT : 2, PITCH = NT * 64 + 16;   // row tiles at a time; bytes of an LDS row
    constexpr int UPR = SWIGLU ? NT * 2 : NT * 4;               // runs of four output columns per row
    const unsigned mine = lds_base + wave * (JG * 16 * PITCH);
    const int ntot = SWIGLU ? 2 * a.N : a.N;
    const int col0 = wn * (SWIGLU ? NT * 8 : NT * 16);          // this wave's first output column inside the unit
#pragma unroll 1
    for (int pass = 0; pass < MT / JG; ++pass) {
        static_for<MT / JG>([&](auto p_tag) {
            constexpr int ps = decltype(p_tag)::value;
            if (pass != ps) return;
#pragma unroll
            for (int j = 0; j < JG; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    *reinterpret_cast<__attribute__((address_space(3))) f32x4*>(mine + (j * 16 + l16) * PITCH + t * 64 + q4 * 16) = acc[t][ps * JG + j];
        });
        wave_sync();
#pragma unroll 2
        for (int it = 0; it < JG * 16 * UPR / 64; ++it) {
            const int idx = it * 64 + lane, row = idx / UPR, u = idx - row * UPR;
            const int col = col0 + 4 * u, mr = (wm * MT + pass * JG) * 16 + row, m = m0 + mr;
            if (col >= ncols || mr >= a.bm || m >= a.M) continue;
            const unsigned at = mine + row * PITCH + (SWIGLU ? (u >> 2) * 128 + (u & 3) * 16 : u * 16);
            const f32x4 v = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(at);
            const f32x4 up = SWIGLU ? *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(at + 64) : f32x4{0.f, 0.f, 0.f, 0.f};
            if (a.ks > 1) {
                float* p = a.partial + ((int64_t)slice * a.M + m) * ntot + n0 + col;
                *reinterpret_cast<f32x4*>(p) = v;
                if (SWIGLU) *reinterpret_cast<f32x4*>(p + a.N) = up;
            } else {
                const float xs = GROUPED && SWIGLU ? a.groups.x_scale[m] : 1.f;
                mid_store<EPI, GROUPED>(a, m, n0 + col, v, up, xs);
            }
        }
        wave_sync();
    }
}

// adds the K slices in slice order and applies the epilogue; a thread per four output columns, all its loads requested at once
template <int EPI, int KS>
__global__ __launch_bounds__(256) void gemm_mid_finish_kernel(MidArgs a) {
    constexpr bool SWIGLU = EPI == EPI_SWIGLU;
    const int per = a.N / 4;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)a.M * per) return;
    const int m = (int)(idx / per), n = 4 * (int)(idx - (int64_t)m * per), ntot = SWIGLU ? 2 * a.N : a.N;
    const float* p = a.partial + (int64_t)m * ntot + n;
    const int64_t next = (int64_t)a.M * ntot;
    f32x4 v[KS], u[SWIGLU ? KS : 1];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        v[s] = *reinterpret_cast<const f32x4*>(p + s * next);
        if (SWIGLU) u[SWIGLU ? s : 0] = *reinterpret_cast<const f32x4*>(p + s * next + a.N);
    }
#pragma unroll
    for (int s = 1; s < KS; ++s) {
        v[0] += v[s];
        if (SWIGLU) u[0] += u[SWIGLU ? s : 0];
    }
    mid_store<EPI>(a, m, n, v[0], u[0]);
}

// ------------------------------------------------------------------------------------------------
// host
// ------------------------------------------------------------------------------------------------
int g_mid = 1;                              // raven_set_tuning("gemm_mid"): 0 = never
int g_mid_nt = 0, g_mid_mt = 0, g_mid_ks = 0;  // raven_set_tuning("gemm_mid_nt" / "_mt" / "_ks"): 0 = by shape

constexpr int kMidMaxSlices = 8;
constexpr int kLds = 160 * 1024;

static int mid_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) cus = p.multiProcessorCount;
        if (cus <= 0) cus = 256;
    }
    return cus;
}

// stages of the ring of a variant (0: no such variant)
static constexpr int mid_stages(int nt, int mt) {
    return nt == 2 ? (mt == 1 ? 8 : mt == 2 ? 6 : 4) : nt == 4 ? (mt == 1 ? 6 : mt == 2 ? 5 : 3) : (mt == 1 ? 5 : mt == 2 ? 4 : 3);
}

// What a launch of a plan costs, in us, fitted to 1847 products of 33 to 4100 rows, 64 to 36000 columns and K of 64 to 18000 (standard deviation 8 %).
// The memory pipe delivers first reads of the weights at 9 TB/s and what comes out of L2 -- the token rows once per column of units, the
// weights again for further row tiles -- at 18; a K step takes the LDS the fragment reads of eight waves (8 clocks per kilobyte) and the
// requests' writes, at 2 clocks per ns; the largest units, with three or four stages in flight, fall short of that.  Every round of units fills its
// ring and drains its outputs anew: 3514 x 592 x 64 in three rounds takes 12.4 us, where a round's own work is 0.3 (128 x 128 tiles, one round: 5.2).
static double mid_estimate(const MidPlan& p, int M, int N, int K, int side, int cus) {
    const int64_t mn = (int64_t)p.tiles_n * p.tiles_m;
    const int nk = (K + 63) / 64, tiles_w = (p.cols * side + 15) / 16, wave_t = tiles_w < p.nt ? tiles_w : p.nt;
    const int rounds = (int)((mn * p.ks + cus - 1) / cus);
    const double weights = 2.0 * N * side * K, again = weights * (p.tiles_m - 1) + 2.0 * K * 64 * p.mt * mn;
    const double mem = weights / 9e6 + again / 18e6;
    const double lds = rounds * ((nk + p.ks - 1) / p.ks) * (128.0 * (wave_t + p.mt) + 16 * tiles_w + 64 * p.mt) / 2050.0;
    double us = (mem > lds ? mem : lds) * (1.0 + (p.mt == 4 && p.ks == 1 ? 0.23 : 0) + (p.nt == 6 ? 0.11 : 0)) + 3.8 * rounds + 6.2 * M * N / 6e6 / rounds;
    if (p.ks > 1) us += 1.2 + 15.0 * p.ks * M * N * side / 8e6;
    return us;
}

static MidPlan find_plan(int M, int N, int K, int swiglu, size_t room) {
    MidPlan best{};
    const int cus = mid_cus(), nk = (K + 63) / 64, side = swiglu ? 2 : 1;
    // the 128 x 128 tiles of gemm_tiled.hip: a K step takes 0.53 us on a CU with one of them and 0.34 more with each further one, and up to
    // 0.15 more per round the fuller the chip is
    const int64_t small = (int64_t)((M + 127) / 128) * ((N * side + 127) / 128);
    const double tiled = nk * (0.19 + 0.34 * (double)((small + cus - 1) / cus) + 0.154 * (double)small / cus) + 3.8 + 2.6 * M * N / 6e6;
    const bool forced = g_mid_nt || g_mid_mt || g_mid_ks;
    for (int nt = 2; nt <= 6; nt += 2)
        for (int mt = 1; mt <= 4; mt *= 2) {
            if ((g_mid_nt && nt != g_mid_nt) || (g_mid_mt && mt != g_mid_mt)) continue;
            const int ns = mid_stages(nt, mt);
            MidPlan p{};
            p.nt = nt;
            p.mt = mt;
            int cap = 32 * nt / side;                      // output columns of the largest unit
            // weight rows a stage has room for (the kilobyte behind the ring is needed where a tile has spare pieces)
            const int max_rows = ((kLds - 1024) / ns / 128 - 64 * mt) / 16 * 16;
            const bool whole_fits = ns * (32 * nt + 64 * mt) * 128 <= kLds;
            if (!whole_fits) cap = max_rows / side / 16 * 16;
            p.tiles_m = (M + 64 * mt - 1) / (64 * mt);
            p.rows = ((M + p.tiles_m - 1) / p.tiles_m + 15) / 16 * 16;
            // as few columns per unit as still run in the rounds that the largest unit needs
            const int64_t whole = (int64_t)((N + cap - 1) / cap) * p.tiles_m;
            int64_t tiles_n = (whole + cus - 1) / cus * cus / p.tiles_m;
            p.cols = (int)((N + tiles_n - 1) / tiles_n + 7) / 8 * 8;
            if (p.cols < 16 * nt / side) p.cols = 16 * nt / side;  // at least half of the variant's tiles
            if (p.cols > cap) p.cols = cap;
            if (whole_fits && (p.cols + 15) / 16 * 16 * side < 32 * nt && (p.cols + 15) / 16 * 16 * side > max_rows) p.cols = cap;
            p.tiles_n = (N + p.cols - 1) / p.cols;
            for (p.ks = 1; p.ks <= kMidMaxSlices; ++p.ks) {
                if (p.ks > 1 && (int64_t)p.tiles_n * p.tiles_m * p.ks > cus + cus / 32 && !g_mid_ks) break;
                if (p.ks > 1 && nk / p.ks < (g_mid_ks ? 1 : 6)) break;
                if (g_mid_ks && p.ks != g_mid_ks && p.ks < nk) continue;
                if (mid_workspace_bytes(M, N, p, swiglu) > room) break;
                p.us = (float)mid_estimate(p, M, N, K, side, cus);
                if ((forced || p.us < tiled) && (best.nt == 0 || p.us < best.us)) best = p;
            }
        }
    if (forced) best.us = 0.f;  // whatever else could run
    return best;
}

MidPlan mid_plan(int M, int N, int K0, int K1, int swiglu, size_t room) {
    if (!g_mid) return MidPlan{};
    // a product is planned several times on its way (does it fit, which row pitch, which launch): the last few shapes of this thread
    struct Known {
        int M, N, K, swiglu, knobs;
        size_t room;
        MidPlan plan;
    };
    static thread_local Known known[16];
    static thread_local int next = 0;
    const int K = K0 + K1, knobs = 1 + g_mid_nt + 10 * g_mid_mt + 100 * g_mid_ks;
    for (const Known& k : known)
        if (k.M == M && k.N == N && k.K == K && k.swiglu == swiglu && k.knobs == knobs && k.room == room) return k.plan;
    Known& k = known[next++ & 15];
    k = Known{M, N, K, swiglu, knobs, room, find_plan(M, N, K, swiglu, room)};
    return k.plan;
}

size_t mid_workspace_bytes(int M, int N, const MidPlan& p, int swiglu) {
    return p.ks > 1 ? (size_t)p.ks * M * N * (swiglu ? 2 : 1) * sizeof(float) : 0;
}

template <int EPI, int NT, int MT>
static int launch_mid_variant(const MidArgs& a, hipStream_t s) {
    constexpr int NS = mid_stages(NT, MT);
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_mid_kernel<EPI, 2, 4, NT, MT, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e != hipSuccess) {
            raven_host::set_error("gemm (mid): hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    const size_t lds = (size_t)NS * (a.wrows * 128 + MT * 8192) + (a.wrows < 32 * NT ? 1024 : 0);
    RAVEN_REQUIRE(lds <= (size_t)kLds && a.wrows <= 32 * NT && a.bm <= 64 * MT, "gemm (mid): a unit of %d x %d does not fit", a.cols, a.bm);
    const int64_t units = (int64_t)a.tiles_m * a.tiles_n * a.ks;
    gemm_mid_kernel<EPI, 2, 4, NT, MT, NS><<<dim3((unsigned)((units + 7) / 8 * 8)), dim3(512), lds, s>>>(a);
    return raven_host::check_launch("gemm (mid)");
}

template <int EPI>
static int launch_mid(const MidArgs& a, const MidPlan& p, hipStream_t s, bool finish) {
    int rc;
    switch (p.nt * 10 + p.mt) {
        case 21: rc = launch_mid_variant<EPI, 2, 1>(a, s); break;
        case 22: rc = launch_mid_variant<EPI, 2, 2>(a, s); break;
        case 24: rc = launch_mid_variant<EPI, 2, 4>(a, s); break;
        case 41: rc = launch_mid_variant<EPI, 4, 1>(a, s); break;
        case 42: rc = launch_mid_variant<EPI, 4, 2>(a, s); break;
        case 44: rc = launch_mid_variant<EPI, 4, 4>(a, s); break;
        case 61: rc = launch_mid_variant<EPI, 6, 1>(a, s); break;
        case 62: rc = launch_mid_variant<EPI, 6, 2>(a, s); break;
        case 64: rc = launch_mid_variant<EPI, 6, 4>(a, s); break;
        default: RAVEN_REQUIRE(false, "gemm (mid): no variant of %d x %d tiles", p.nt, p.mt);
    }
    if (rc || !finish) return rc;
    const dim3 grid((unsigned)(((int64_t)a.M * (a.N / 4) + 255) / 256));
#define RAVEN_MID_FINISH(KS_) case KS_: gemm_mid_finish_kernel<EPI, KS_><<<grid, dim3(256), 0, s>>>(a); break;
    switch (a.ks) {
        RAVEN_MID_FINISH(2) RAVEN_MID_FINISH(3) RAVEN_MID_FINISH(4) RAVEN_MID_FINISH(5) RAVEN_MID_FINISH(6) RAVEN_MID_FINISH(7) RAVEN_MID_FINISH(8)
        default: RAVEN_REQUIRE(false, "gemm (mid): %d slices", a.ks);
    }
#undef RAVEN_MID_FINISH
    return raven_host::check_launch("gemm (mid, sums)");
}

int mid_gemm(const ProductArgs& q, const MidPlan& p, void* workspace, hipStream_t s, int* ks_left) {
    MidArgs a{};
    a.w = q.w; a.x0 = q.x0; a.x1 = q.x1; a.residual = q.residual; a.y = q.y; a.partial = static_cast<float*>(workspace);
    a.M = q.M; a.N = q.N; a.K0 = q.K0; a.K1 = q.x1 ? q.K1 : 0; a.ldw = q.ldw; a.ldx = q.ldx; a.out_f32 = q.out_f32;
    a.cols = p.cols; a.bm = p.rows; a.wrows = (p.cols + 15) / 16 * 16 * (q.swiglu ? 2 : 1);
    a.tiles_m = p.tiles_m; a.tiles_n = p.tiles_n; a.ks = p.ks;
    if (q.epi) a.epi = *q.epi;
    if (q.rope) {
        a.rope = *q.rope;
        a.rope_on = 1;
    }
    RAVEN_REQUIRE(p.ks == 1 || (workspace && ((uintptr_t)workspace & 15) == 0), "gemm (mid): no workspace for the K slices");
    const bool finish = p.ks > 1 && !ks_left;
    if (ks_left) *ks_left = p.ks > 1 ? p.ks : 0;
    if (q.epi && q.epi->act == RAVEN_ACT_GELU) return launch_mid<EPI_FREE_GELU>(a, p, s, finish);
    if (q.epi && q.epi->act == RAVEN_ACT_TANH) return launch_mid<EPI_FREE_TANH>(a, p, s, finish);
    if (q.epi) return launch_mid<EPI_FREE>(a, p, s, finish);
    if (q.swiglu) return launch_mid<EPI_SWIGLU>(a, p, s, finish);
    return launch_mid<EPI_PLAIN>(a, p, s, finish);
}

template <int EPI, int WN, int WM, int NT, int MT, int NS>
static int launch_grouped(const MidArgs& a, hipStream_t s) {
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_mid_kernel<EPI, WN, WM, NT, MT, NS, true>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e != hipSuccess) {
            raven_host::set_error("gemm (grouped): hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    const size_t lds = (size_t)NS * (a.wrows + 16 * WM * MT) * 128 + (a.wrows < 16 * WN * NT ? 1024 : 0);
    RAVEN_REQUIRE(lds <= (size_t)kLds && a.wrows <= 16 * WN * NT, "gemm (grouped): a unit of %d columns does not fit", a.cols);
    const int64_t units = (int64_t)a.tiles_m * a.tiles_n;
    RAVEN_REQUIRE(units < (1 << 28), "gemm (grouped): too many units");
    gemm_mid_kernel<EPI, WN, WM, NT, MT, NS, true><<<dim3((unsigned)((units + 7) / 8 * 8)), dim3(64 * WN * WM), lds, s>>>(a);
    return raven_host::check_launch("gemm (grouped)");
}

// Tiles of 32 rows: four waves side by side along the weight rows -- with few token rows the eight waves of the larger tiles would
// read mostly rows that do not exist out of LDS --, four stages of 20 KB, two workgroups per CU, so that one streams while the
// other fills its ring or stores (a unit of an expert of 768 channels has 12 to 32 K steps).
template <int EPI>
static int launch_grouped_rows(const MidArgs& a, hipStream_t s) {
    switch (a.bm) {
        case 32: return launch_grouped<EPI, 4, 1, 2, 2, 4>(a, s);
        case 64: return launch_grouped<EPI, 2, 4, 4, 1, 3>(a, s);
        default: RAVEN_REQUIRE(false, "gemm (grouped): tiles of %d rows", a.bm);
    }
}

int mid_grouped(const void* x, int x_rows, const void* w, void* y, int rows, int N, int K, int swiglu, int out_f32, const RowGroups& g, hipStream_t s) {
    RAVEN_REQUIRE(x && w && y && g.group_of && g.group_row && g.group_end && g.used && g.n_tiles > 0 && N > 0 && N % 8 == 0 && K > 0 && K % 8 == 0 &&
                      (!swiglu || (g.x_scale && !out_f32)) && (g.extra_group < 0 || g.w_extra), "gemm (grouped): bad arguments");
    RAVEN_REQUIRE((int64_t)x_rows * K < (1ll << 31) && (int64_t)N * 2 * K < (1ll << 31) && (int64_t)rows * N < (1ll << 40), "gemm (grouped): too large");
    MidArgs a{};
    a.w = static_cast<const bf16*>(w);
    a.x0 = static_cast<const bf16*>(x);
    a.y = y;
    a.M = rows; a.N = N; a.K0 = K; a.ldw = K; a.ldx = K; a.out_f32 = out_f32;
    const int side = swiglu ? 2 : 1, cap = 128 / side;
    const int tiles_n = (N + cap - 1) / cap;
    a.cols = ((N + tiles_n - 1) / tiles_n + 7) / 8 * 8;
    if (a.cols < cap / 2) a.cols = cap / 2;
    a.wrows = (a.cols + 15) / 16 * 16 * side;
    a.tiles_n = (N + a.cols - 1) / a.cols;
    a.bm = g.tile_rows; a.tiles_m = g.n_tiles; a.ks = 1;
    a.epi.scale = 1.f;
    a.groups = g;
    return swiglu ? launch_grouped_rows<EPI_SWIGLU>(a, s) : launch_grouped_rows<EPI_FREE>(a, s);
}

}  // namespace raven
