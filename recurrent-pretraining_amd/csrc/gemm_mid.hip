// Matrix-core products over a middling number of token rows (33 to a few thousand; from 17 against long or large matrices): Y[M,N] = concat(X0, X1)[M,K] W[N,K]^T in bf16 with fp32
// accumulation, with the epilogues of gemm_tiled.hip -- prompts of ordinary length, decode batches past 32 sequences, a serving engine's
// mixed steps, and long prompts against matrices too narrow to give every CU a 256 x 256 tile, or the last round of a product of such tiles.
//
// What bounds these products is how a CU's loads queue: it has about 32 KB of lines on their way at a time, answered in order, so that the token rows,
// which hit the L2, wait as long as the weights from HBM in front of them (64 + 96 rows a step move at 53 bytes a ns on 30 CUs, 42 on all; the weights
// alone 51 and 22.5, the chip's 5.8 TB/s; the token rows alone 110).  A ring deeper than about 64 KB gives nothing; what counts is how few lines a
// unit asks for, and that products and LDS reads stay below that time.  So
//   * operands go global -> LDS directly through a ring of NS stages, NS - 1 K steps of 64 ahead;
//   * a unit owns `cols` output columns and `rows` token rows, not whole tiles: as many as leave the chip ONE nearly full round of units (17920 gate
//     columns = 249 x 72); the ring holds the 16-row tiles that exist and no others;
//   * where even the narrowest unit leaves CUs idle, K is cut into slices: fp32 sums in the workspace, added in slice order by a second
//     launch or by the norm that follows (splitk_sums_then_norm);
//   * 8 waves, two along the weight rows and four along the token rows (v_mfma_f32_16x16x32_bf16, W rows as the A operand); the unit's tiles are dealt
//     out evenly and a wave has a loop for each number of tiles it may get, NT or one less by MT or one less: with every wave multiplying NT x MT a
//     unit of 9 x 13 tiles made 192 products for 117;
//   * weight rows that one unit reads are loaded past the caches (`nt`): 5 to 9 % where HBM bounds the launch; those that two row tiles share are not (5 % slower).
// LDS rows are 128 bytes, 16-byte piece c of row r at position c ^ ((r >> 1) & 7) (applied on the global side), so that fragment reads are
// free of bank conflicts.  Unlike the tiles of gemm_tiled.hip a wave's partial sums over K slices are added after the fact, so results
// differ from those in the order of fp32 sums.
//
// us per launch, weights from HBM, rows of whole lines; whole 64 x 32-row tiles for every wave / these: 3.5b shape at 93 rows Wqkv 44.9 / 40, attn.proj 24.1 / 21.5,
// mlp.fc 78 / 68 (5.6 TB/s of weights), mlp.proj 56 / 44.5; at 195 rows 54.7 / 53.8, 32.3 / 26, 118 / 93, 82 / 56; width 2048 at 500 rows up 24.4 / 24.3, down
// 37 / 29.6; 1500 rows 63 / 59, 78 / 59; 4096 x 2048 x 8192 124 / 113; 260 x 3072 x 1536 10.5 / 9.5.

#include "gemm_common.h"

namespace raven {

struct MidArgs {
    const bf16 *w, *x0, *x1, *residual;
    void* y;
    float* partial;        // [ks, M, N or 2N] when ks > 1
    int M, N, K0, K1, ldw, ldx;
    int ldy, up_off;       // elements between two rows of y and of the residuals; weight rows from a gate row to its up row
    int out_f32;
    int kind;              // EPI_*
    int cols, bm;          // output columns / token rows of a unit
    int wtiles, xtiles;    // 16-row tiles of a unit's weight rows / token rows
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
    const int64_t at = (int64_t)m * a.ldy + n;
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
            const int h = r.nh * r.hd, nr = n + r.col0, sec = nr >= 2 * h ? 2 : (nr >= h ? 1 : 0);  // q, k or v columns; four of them lie in one head
            const int col = nr - sec * h, head = col / r.hd, d = col - head * r.hd;
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

// kilobyte pieces, two a tile, that a workgroup of so many waves asks for per step where its variant has room for so many tiles
__host__ __device__ constexpr int mid_requests(int tiles, int waves) { return (2 * tiles + waves - 1) / waves * waves; }

// GROUPED: row groups with a weight matrix each; a unit works on a copy of the arguments cut to its group's rows
// ONCE: every weight row is read by one unit
// HALF: rows of K = 64 n + 32 elements on a matrix that starts on a line (5280: 82.5 lines), so that odd rows start in the middle of one, and a step of 64 columns of such a
// row would be two half lines.  The unit's even rows are the first wave row's tiles and its odd rows the second's; odd rows are requested line by line too, 32 columns in
// front of the even ones, and their waves multiply each of the lines' halves with the token fragments of the half before: the same products in the same order.  Whole sums
// only: the odd rows' slices would begin and end 32 columns earlier, and a matrix give other bits than its copy with padded rows.  us per launch at 195 rows, weights from HBM,
// half lines / so: mlp.fc 110 / 99 (copies with padded rows 93), Wqkv 61 / 57; at 93 rows 90 / 74, 51 / 45 (there with token rows of half lines as well).
template <int WN, int WM, int NT, int MT, int NS, bool ONCE, bool GROUPED = false, bool HALF = false>
__global__ __launch_bounds__(64 * WN * WM) void gemm_mid_kernel(MidArgs a) {
    constexpr int NW = WN * WM, WPW = mid_requests(WN * NT, NW) / NW, XPW = mid_requests(WM * MT, NW) / NW, LPW = WPW + XPW;  // requests of a wave per step
    static_assert(NW % 2 == 0 && (NS - 1) * LPW < 64, "a wave's pieces have one parity; the wait counter holds 63 requests");
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

    const bool swiglu = a.kind == EPI_SWIGLU;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int K = a.K0 + a.K1, nk = (K + 63) >> 6;
    const int k0 = HALF ? 0 : __builtin_amdgcn_readfirstlane((int)((int64_t)nk * slice / a.ks));
    const int n_steps = HALF ? nk : __builtin_amdgcn_readfirstlane((int)((int64_t)nk * (slice + 1) / a.ks)) - k0;
    const int n0 = tile_n * a.cols, ncols = min(a.cols, a.N - n0), m0 = tile_m * a.bm, rows = min(a.bm, a.M - m0);
    // the wave's tiles, dealt out evenly; a SIMD's two waves (ids that differ by four) get a long and a short share of the token tiles
    const int wn = wave / WM, wm = (wn & 1) ? WM - 1 - wave % WM : wave % WM;
    static_assert(!HALF || (WN == 2 && !GROUPED), "a wave row for each parity");
    const int tw = __builtin_amdgcn_readfirstlane(((HALF == swiglu ? ncols : HALF ? ncols / 2 : 2 * ncols) + 15) >> 4), tx = __builtin_amdgcn_readfirstlane((rows + 15) >> 4);
    const int nw = HALF ? tw : tw / WN + (wn < tw % WN), tw0 = HALF ? wn * NT : wn * (tw / WN) + min(wn, tw % WN);
    const int nx = tx / WM + (wm < tx % WM), tx0 = wm * (tx / WM) + min(wm, tx % WM);
    const int wbytes = a.wtiles * 2048, stage = wbytes + a.xtiles * 2048, ring = NS * stage;
    const unsigned lds_base = (unsigned)(uintptr_t)(lds_byte*)smem;

    // ---- global side: request i of a wave is piece NW i + wave, eight rows of the weight tile (i < WPW) or of the token rows; the lane that
    // fills position s of row r fetches piece s ^ ((r >> 1) & 7) of the row's 128-byte step.  A SwiGLU tile is eight gate rows and their up
    // rows.  Requests past the unit's last piece fetch one line, of the last row, to behind the ring: the count of requests stays.
    const int colp = ((lane & 7) ^ ((lane >> 4) | (4 * (wave & 1)))) * 8;
    unsigned goff[LPW];
    unsigned dst[LPW];  // offset inside a stage
    bool spare[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const bool is_w = i < WPW;
        const int piece = is_w ? NW * i + wave : NW * (i - WPW) + wave, r = piece * 8 + (lane >> 3);
        spare[i] = (GROUPED || i == WPW - 1 || i == LPW - 1) && piece >= 2 * (is_w ? a.wtiles : a.xtiles);  // (of a plain unit only the last ones may be)
        if (is_w) {
            const int odd = HALF && r >= 16 * NT, rr = r - odd * 16 * NT, k = swiglu ? (rr >> 4) * 8 + (rr & 7) : rr;
            const int c = HALF ? (2 * k + odd < ncols ? 2 * k + odd : ncols - 2 + odd) : min(k, ncols - 1);
            goff[i] = (unsigned)(n0 + c + (swiglu && (rr & 8) ? a.up_off : 0)) * (2u * a.ldw) + 2u * colp - 64u * odd;
        } else {
            int row = m0 + min(r, rows - 1);
            if (GROUPED && x_row) row = x_row[row];
            goff[i] = (unsigned)row * (2u * a.ldx) + 2u * colp;
        }
        dst[i] = __builtin_amdgcn_readfirstlane(lds_base + (is_w ? 0 : wbytes) + piece * 1024);
    }
    const char* const zero = reinterpret_cast<const char*>(g_mid_zero);
    const char* const w0 = reinterpret_cast<const char*>(a.w);
    const char* const x0 = reinterpret_cast<const char*>(a.x0);
    const char* const x1 = reinterpret_cast<const char*>(a.x1) - 2 * (int64_t)a.K0;  // column c >= K0 of the token rows
    auto whole = [&](int kk) __attribute__((always_inline)) {  // the 64 columns of step kk lie in one segment and below K
        const int c0 = kk << 6;
        return c0 + 64 <= a.K0 || (c0 >= a.K0 && c0 + 64 <= K);
    };
    // requests FIRST .. LAST - 1 of step kk (columns 64 kk ..+63; zeros past K) into the stage at offset o; whole_tag: 1 whole, 0 not, 2 either
    auto issue = [&](int kk, int o, auto first_tag, auto last_tag, auto whole_tag) __attribute__((always_inline)) {
        const int c0 = kk << 6;
        if (decltype(whole_tag)::value == 1 || (decltype(whole_tag)::value == 2 && whole(kk))) {
            const char *wb = w0 + 2 * c0, *xb = (c0 < a.K0 ? x0 : x1) + 2 * c0;
#pragma unroll
            for (int i = decltype(first_tag)::value; i < decltype(last_tag)::value; ++i) {
                const unsigned to = __builtin_amdgcn_readfirstlane(spare[i] ? lds_base + ring : o + dst[i]);
                if (ONCE && i < WPW) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(goff[i]), "s"(wb), "s"(to) : "memory");
                else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(goff[i]), "s"(i < WPW ? wb : xb), "s"(to) : "memory");
            }
            return;
        }
        const int col = c0 + colp;
#pragma unroll
        for (int i = decltype(first_tag)::value; i < decltype(last_tag)::value; ++i) {
            const unsigned to = __builtin_amdgcn_readfirstlane(spare[i] ? lds_base + ring : o + dst[i]);
            unsigned off = goff[i];
            asm volatile("" : "+v"(off));  // (the address is not worth a register pair outside this step)
            const bool past = HALF && i < WPW && (NW * i + wave) * 8 >= 16 * NT ? false : col >= K;  // (odd rows: 32 columns less)
            const char* gp = past ? zero : (i < WPW ? w0 : (col < a.K0 ? x0 : x1)) + 2 * c0 + off;
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gp), "s"(to) : "memory");
        }
    };

    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // ---- the ring: step i sits in stage i mod NS.  The barrier in the middle of step i says that every wave's requests of step i + 1 have
    // landed and that every wave has read out step i, whose stage step i + NS then takes.  The fragments of a slice are read under the
    // products of the slice before, the requests stand between the two slices' products: with reads, requests and products of all eight
    // waves one after the other behind the barrier a step took the sum of the three (Wqkv of the 3.5b shape at 93 rows 46 us).
    const int l16 = lane & 15, q4 = lane >> 4;
    using ic0 = std::integral_constant<int, 0>;
    using ic1 = std::integral_constant<int, 1>;
    using ic2 = std::integral_constant<int, 2>;
    using half = std::integral_constant<int, (LPW + 1) / 2>;
    using all = std::integral_constant<int, LPW>;
    auto arrive = [&](auto left_tag) __attribute__((always_inline)) {  // all but the requests of `left` steps have landed
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left_tag)::value * LPW) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    auto arrive_left = [&](int left) __attribute__((always_inline)) {  // the same, NS - 2 at most
        static_for<NS - 1>([&](auto n_tag) {
            constexpr int n = decltype(n_tag)::value;
            if (n < NS - 2 ? left == n : left >= n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n * LPW) : "memory");
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    // NTW x MTW: tiles of this wave; a wave without any requests its share and multiplies nothing
    // LATE: the odd rows' waves of HALF, half a step behind
    auto run = [&](auto nt_tag, auto mt_tag, auto late_tag) __attribute__((always_inline)) {
        constexpr bool LATE = decltype(late_tag)::value;
        constexpr int NTW = decltype(nt_tag)::value, MTW = decltype(mt_tag)::value;
        const unsigned pos0 = (q4 ^ ((l16 >> 1) & 7)) * 16;  // k-slice s of a step: pos0 ^ (64 s)
        const unsigned a_row = lds_base + (tw0 * 16 + l16) * 128, b_row = lds_base + wbytes + (tx0 * 16 + l16) * 128;
        u32x4 fa[2][NTW ? NTW : 1], fb[2][MTW ? MTW : 1];  // fragments of the two k-slices of a step
        auto fetch = [&](int o, auto sl_tag) __attribute__((always_inline)) {
            constexpr int sl = decltype(sl_tag)::value;
            const unsigned ra = a_row + o + (pos0 ^ (64 * sl)), rb = b_row + o + (pos0 ^ (64 * sl));
#pragma unroll
            for (int j = 0; j < MTW; ++j) fb[sl][j] = *reinterpret_cast<const lds_u32x4*>(rb + j * 2048);
#pragma unroll
            for (int t = 0; t < NTW; ++t) fa[sl][t] = *reinterpret_cast<const lds_u32x4*>(ra + t * 2048);
        };
        auto multiply = [&](auto sl_tag) __attribute__((always_inline)) {
            constexpr int sl = decltype(sl_tag)::value;
#pragma unroll
            for (int t = 0; t < NTW; ++t)
#pragma unroll
                for (int j = 0; j < MTW; ++j)
                    acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fa[sl][t]), __builtin_bit_cast(bf16x8, fb[sl][j]), acc[t][j], 0, 0, 0);
        };
        // LATE: fragments of weight slice SL of the stage at o, of token slice SL into set DST; the products of set 0, whose fragments are followed by the next ones
        auto fetch_w = [&](int o, auto sl_tag) __attribute__((always_inline)) {
            constexpr int sl = decltype(sl_tag)::value;
#pragma unroll
            for (int t = 0; t < NTW; ++t) fa[sl][t] = *reinterpret_cast<const lds_u32x4*>(a_row + o + (pos0 ^ (64 * sl)) + t * 2048);
        };
        auto fetch_x = [&](int o, auto sl_tag, auto dst_tag) __attribute__((always_inline)) {
            constexpr int sl = decltype(sl_tag)::value, dst = decltype(dst_tag)::value;
#pragma unroll
            for (int j = 0; j < MTW; ++j) fb[dst][j] = *reinterpret_cast<const lds_u32x4*>(b_row + o + (pos0 ^ (64 * sl)) + j * 2048);
        };
        auto multiply_late = [&](int o) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < MTW; ++j) {
#pragma unroll
                for (int t = 0; t < NTW; ++t)
                    acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fa[0][t]), __builtin_bit_cast(bf16x8, fb[0][j]), acc[t][j], 0, 0, 0);
                fb[0][j] = *reinterpret_cast<const lds_u32x4*>(b_row + o + (pos0 ^ 64) + j * 2048);
            }
        };
        int o = 0, i = 0;
        arrive_left(n_steps - 1);
        if constexpr (LATE) {
            // the first line of an odd row begins with the end of the row before
#pragma unroll
            for (int t = 0; t < NTW; ++t) fa[0][t] = u32x4{0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < MTW; ++j) fb[0][j] = u32x4{0, 0, 0, 0};
        } else {
            fetch(0, ic0{});
        }
        // Small tiles: a loop without a branch for the steps whose requests are whole, another for the few that are not (uq of 1536 to 3072 columns at
        // 260 rows 10.7 -> 9.6 us).  Large ones: their products hide the branches, and registers are short.
        auto steps = [&](int end, auto whole_tag) __attribute__((always_inline)) {  // whose requests are of whole steps, or none of them
#pragma unroll 1
            for (; i < end; ++i) {
                const int free = o == 0 ? ring - stage : o - stage, next = o + stage == ring ? 0 : o + stage;
                if constexpr (LATE) {
                    fetch_w(o, ic1{});
                    fetch_x(o, ic0{}, ic1{});
                } else {
                    fetch(o, ic1{});
                }
                issue(k0 + i + NS - 1, free, ic0{}, half{}, whole_tag);
                if constexpr (LATE) multiply_late(o);
                else multiply(ic0{});
                issue(k0 + i + NS - 1, free, half{}, all{}, whole_tag);
                arrive(std::integral_constant<int, NS - 2>{});
                if constexpr (LATE) fetch_w(next, ic0{});
                else fetch(next, ic0{});
                multiply(ic1{});
                o = next;
            }
        };
        const int asked = n_steps - NS + 1;  // steps that still request
#pragma unroll 1
        while (i < asked) {
            const int kk = k0 + i + NS - 1;
            if constexpr (NT * MT > 6) steps(asked, ic2{});
            else if (whole(kk)) steps(min(asked, ((a.K0 & 63) && kk < (a.K0 >> 6) ? a.K0 >> 6 : K >> 6) - (k0 + NS - 1)), ic1{});
            else steps(i + 1, ic0{});
        }
        // nothing more to request: the last NS - 1 steps, or all of a shorter slice
        static_for<NS - 1>([&](auto j_tag) {
            constexpr int left = NS - 2 - decltype(j_tag)::value;  // steps behind this one
            if (n_steps <= left) return;
            const int next = o + stage == ring ? 0 : o + stage;
            if constexpr (LATE) {
                fetch_w(o, ic1{});
                fetch_x(o, ic0{}, ic1{});
                multiply_late(o);
            } else {
                fetch(o, ic1{});
                multiply(ic0{});
            }
            if constexpr (left > 0) {
                arrive(std::integral_constant<int, (left > 0 ? left - 1 : 0)>{});
                if constexpr (LATE) fetch_w(next, ic0{});
                else fetch(next, ic0{});
            }
            multiply(ic1{});
            o = next;
        });
    };
#pragma unroll 1
    for (int i = 0; i < NS - 1 && i < n_steps; ++i) issue(k0 + i, i * stage, ic0{}, all{}, ic2{});
    // (with fewer tiles than one less than the variant's the surplus fragments are whatever lies behind, and their products are not stored)
    using nt0 = std::integral_constant<int, NT>;
    using nt1 = std::integral_constant<int, NT - 1>;
    using mt0 = std::integral_constant<int, MT>;
    using mt1 = std::integral_constant<int, MT - 1>;
    auto run_tiles = [&](auto late_tag) __attribute__((always_inline)) {
        if (__builtin_expect(nw == NT && nx == MT, 1)) run(nt0{}, mt0{}, late_tag);
        else if (nw == 0 || nx == 0) run(ic0{}, ic0{}, std::false_type{});
        else if (nw == NT) { if constexpr (MT > 1) run(nt0{}, mt1{}, late_tag); }
        else if (nx == MT) { if constexpr (NT > 1) run(nt1{}, mt0{}, late_tag); }
        else { if constexpr (NT > 1 && MT > 1) run(nt1{}, mt1{}, late_tag); }
    };
    if constexpr (HALF) {
        if (wn == 1) run_tiles(std::true_type{});
        else run_tiles(std::false_type{});
    } else {
        run_tiles(std::false_type{});
    }

    // ---- out: a lane holds rows 4 q4 ..+3 of weight tile t for token row 16 j + l16.  A wave lays its sums down in LDS, rows of its columns,
    // and a rolled loop takes them from there: whole runs of columns per store, and little code -- unrolled over the accumulators
    // the epilogue ran once per unit out of a cold instruction cache (gelu outputs of 3000 x 4096 x 1024: 46 us, as a loop 36).
    // lanes of a wave exchange data through LDS without a workgroup barrier: pin the order of the accesses for the compiler
    auto wave_sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave has left the ring
    // HALF: the two waves of the same token rows lay their columns down side by side, and each stores every other run of them.
    constexpr int JG = MT % 2 ? 1 : 2, PITCH = (HALF ? 2 : 1) * NT * 64 + 16;    // row tiles at a time; bytes of an LDS row
    const unsigned mine = lds_base + (HALF ? wm : wave) * (JG * 16 * PITCH);
    const int ntot = swiglu ? 2 * a.N : a.N;
    const int col0 = HALF ? 0 : tw0 * (swiglu ? 8 : 16), col_end = HALF ? ncols : min(ncols, col0 + nw * (swiglu ? 8 : 16));  // this wave's output columns inside the unit
    auto out_sync = [&]() __attribute__((always_inline)) {
        if constexpr (HALF) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        } else {
            wave_sync();
        }
    };
    const int row_end = min(rows, (tx0 + nx) * 16);
#pragma unroll 1
    for (int pass = 0; pass < MT / JG; ++pass) {
        static_for<MT / JG>([&](auto p_tag) {
            constexpr int ps = decltype(p_tag)::value;
            if (pass != ps) return;
#pragma unroll
            for (int j = 0; j < JG; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const unsigned row = mine + (j * 16 + l16) * PITCH;
                    if constexpr (HALF) {  // column 2 k + wn, k = 16 t + 4 q4 + v; SwiGLU: gates, k = 8 t + 4 q4 + v, and behind them all the ups
                        const unsigned at = row + wn * 4 + (swiglu ? (q4 & 1) * 32 + t * 64 + (q4 >> 1) * (NT * 64) : t * 128 + q4 * 32);
#pragma unroll
                        for (int v = 0; v < 4; ++v) *reinterpret_cast<__attribute__((address_space(3))) float*>(at + 8 * v) = acc[t][ps * JG + j][v];
                    } else {
                        *reinterpret_cast<__attribute__((address_space(3))) f32x4*>(row + t * 64 + q4 * 16) = acc[t][ps * JG + j];
                    }
                }
        });
        out_sync();
        const int first = (tx0 + pass * JG) * 16;
        auto store = [&](auto kind_tag) __attribute__((always_inline)) {
            constexpr int EPI = decltype(kind_tag)::value;
            constexpr bool SWIGLU = EPI == EPI_SWIGLU;
            constexpr int UPR = (HALF ? 2 : 1) * (SWIGLU ? NT * 2 : NT * 4);  // runs of four output columns per row
#pragma unroll 2
            for (int idx = HALF ? 64 * wn + lane : lane; idx < JG * 16 * UPR; idx += HALF ? 128 : 64) {
                const int row = idx / UPR, u = idx - row * UPR, col = col0 + 4 * u, mr = first + row, m = m0 + mr;
                if (col >= col_end || mr >= row_end) continue;
                const unsigned at = mine + row * PITCH + (SWIGLU && !HALF ? (u >> 1) * 64 + (u & 1) * 16 : u * 16);
                const f32x4 v = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(at);
                const f32x4 up = SWIGLU ? *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(at + (HALF ? NT * 64 : 32)) : f32x4{0.f, 0.f, 0.f, 0.f};
                if (a.ks > 1) {
                    float* p = a.partial + ((int64_t)slice * a.M + m) * ntot + n0 + col;
                    *reinterpret_cast<f32x4*>(p) = v;
                    if (SWIGLU) *reinterpret_cast<f32x4*>(p + a.N) = up;
                } else {
                    const float xs = GROUPED && SWIGLU ? a.groups.x_scale[m] : 1.f;
                    mid_store<EPI, GROUPED>(a, m, n0 + col, v, up, xs);
                }
            }
        };
        if (swiglu) store(std::integral_constant<int, EPI_SWIGLU>{});
        else if (GROUPED || a.kind == EPI_FREE) store(std::integral_constant<int, EPI_FREE>{});
        else if (a.kind == EPI_PLAIN || a.ks > 1) store(std::integral_constant<int, EPI_PLAIN>{});
        else if (a.kind == EPI_FREE_GELU) store(std::integral_constant<int, EPI_FREE_GELU>{});
        else store(std::integral_constant<int, EPI_FREE_TANH>{});
        out_sync();
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
int g_mid_half = 1;                         // raven_set_tuning("gemm_mid_half"): 0 = rows that are no whole lines are read as they lie
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

// stages of the ring of a variant: as many as fit at its largest unit, 3 to 8 (nt 6, mt 4: three only up to 26 tiles in all)
static constexpr int mid_stages(int nt, int mt) {
    const int fit = (kLds - nt % 2 * 1024) / ((2 * nt + 4 * mt) * 2048);  // (odd nt: eight waves' requests are more than the unit's pieces)
    return fit > 8 ? 8 : fit < 3 ? 3 : fit;
}

// LDS of a unit of WN x WM waves: the ring and the kilobyte behind it, where more is asked for than the unit has pieces, or the sums on their way out
static size_t mid_lds_bytes(int wn, int wm, int nt, int mt, int ns, int wtiles, int xtiles) {
    const int waves = wn * wm;
    const bool spare = mid_requests(wn * nt, waves) > 2 * wtiles || mid_requests(wm * mt, waves) > 2 * xtiles;
    const size_t ring = (size_t)ns * (wtiles + xtiles) * 2048 + (spare ? 1024 : 0), sums = (size_t)waves * (mt % 2 ? 1 : 2) * 16 * (nt * 64 + 16);
    return ring > sums ? ring : sums;
}

// What a launch of a plan costs, in us, fitted to 3634 products of 33 to 4096 rows, 768 to 36000 columns and K of 768 to 18000 (standard deviation 9 %;
// the plans it picks for 317 shapes are 1.0 % slower than the best of each).  The terms are fitted together, their divisors are no rates (a launch reads weights
// at 5.8 TB/s at the most): bytes of weights by 8.8, bytes out of the caches -- the token rows once per column of units, the weights again for further
// row tiles -- by 60; a K step takes its fragment reads, products and requests; of the two the shorter one is hidden to two fifths.  Every round of units
// fills its ring and drains its outputs anew.
static double mid_estimate(const MidPlan& p, int M, int N, int K, int side, int cus) {
    const int64_t mn = (int64_t)p.tiles_n * p.tiles_m;
    const int nk = (K + 63) / 64, wtiles = (p.cols * side + 15) / 16;
    const int rounds = (int)((mn * p.ks + cus - 1) / cus);
    const double weights = 2.0 * N * side * K, again = weights * (p.tiles_m - 1) + 2.0 * K * p.rows * mn;
    const double mem = weights / 8.8e6 + again / 60e6;
    const double step = rounds * ((nk + p.ks - 1) / p.ks) * (37.0 * p.nt + 123 * p.mt + 21.5 * wtiles + 34) / 2050.0;
    double us = (mem > step ? mem + 0.6 * step : step + 0.6 * mem) + 2.1 * rounds + 6.7 * M * N / 6e6 / rounds + 1.3;
    if (p.ks > 1) us += 2.4 + 14.0 * p.ks * M * N * side / 8e6;
    return us;
}

// What the 128 x 128 tiles of gemm_tiled.hip take, in us: a K step takes 0.53 us on a CU with one of them and 0.34 more with each further one,
// and up to 0.15 more per round the fuller the chip is
static double tiled_estimate(int M, int N, int K, int side, int cus) {
    const int64_t small = (int64_t)((M + 127) / 128) * ((N * side + 127) / 128);
    return (K + 63) / 64 * (0.19 + 0.34 * (double)((small + cus - 1) / cus) + 0.154 * (double)small / cus) + 3.8 + 2.6 * M * N / 6e6;
}

static MidPlan find_plan(int M, int N, int K, int swiglu, size_t room, int ks_from) {
    MidPlan best{};
    const int cus = mid_cus(), nk = (K + 63) / 64, side = swiglu ? 2 : 1;
    const double tiled = tiled_estimate(M, N, K, side, cus);
    const bool forced = g_mid_nt || g_mid_mt || g_mid_ks;
    for (int mt = 1; mt <= 4; ++mt) {
        if (g_mid_mt && mt != g_mid_mt) continue;
        MidPlan p{};
        p.tiles_m = (M + 64 * mt - 1) / (64 * mt);
        p.rows = ((M + p.tiles_m - 1) / p.tiles_m + 15) / 16 * 16;
        if (g_mid_mt && p.rows < 64 * mt - 48) {  // the variant that was asked for, with tiles that have no rows
            p.rows = 64 * mt - 48;
            p.tiles_m = (M + p.rows - 1) / p.rows;
        }
        p.mt = (p.rows + 63) / 64;
        for (int nt = 1; nt <= 6; ++nt) {
            if (g_mid_nt && nt != g_mid_nt) continue;
            for (p.ks = ks_from; p.ks <= kMidMaxSlices; ++p.ks) {
                if (g_mid_ks && p.ks != (g_mid_ks < nk ? g_mid_ks : nk)) continue;
                const int cap = 32 * nt / side;  // output columns of the largest unit
                // as few columns per unit as still run in the rounds that the largest unit needs
                const int64_t whole = (int64_t)((N + cap - 1) / cap) * p.tiles_m * p.ks;
                const int64_t tiles_n = (whole + cus - 1) / cus * cus / (p.tiles_m * p.ks);
                p.cols = (int)((N + tiles_n - 1) / tiles_n + 7) / 8 * 8;
                if (g_mid_nt) {  // as few units as hold the columns, with the variant's number of tiles
                    const int fewest = (N + cap - 1) / cap, least = side == 2 ? 16 * nt - 8 : 32 * nt - 24;
                    p.cols = ((N + fewest - 1) / fewest + 7) / 8 * 8;
                    if (p.cols < least) p.cols = least;
                }
                if (p.cols > cap) p.cols = cap;
                p.tiles_n = (N + p.cols - 1) / p.cols;
                const int wtiles = (p.cols * side + 15) / 16;
                p.nt = (wtiles + 1) / 2;
                if (mid_lds_bytes(2, 4, p.nt, p.mt, mid_stages(p.nt, p.mt), wtiles, p.rows / 16) > (size_t)kLds) continue;
                if (p.ks > 1 && (int64_t)p.tiles_n * p.tiles_m * p.ks > cus + cus / 32 && !g_mid_ks) break;
                if (p.ks > 1 && nk / p.ks < (g_mid_ks ? 1 : 6)) break;
                if (mid_workspace_bytes(M, N, p, swiglu) > room) break;
                p.us = (float)mid_estimate(p, M, N, K, side, cus);
                if ((forced || ks_from > 1 || p.us < tiled) && (best.nt == 0 || p.us < best.us)) best = p;
            }
        }
    }
    if (forced) best.us = 0.f;  // whatever else could run
    return best;
}

MidPlan mid_plan(int M, int N, int K0, int K1, int swiglu, size_t room, int ks_from) {
    if (!g_mid) return MidPlan{};
    // a product is planned several times on its way (does it fit, which row pitch, which launch): the last few shapes of this thread
    struct Known {
        int M, N, K, swiglu, knobs;
        size_t room;
        MidPlan plan;
    };
    static thread_local Known known[16];
    static thread_local int next = 0;
    const int K = K0 + K1, knobs = 1 + g_mid_nt + 10 * g_mid_mt + 100 * g_mid_ks + 1000 * ks_from;
    for (const Known& k : known)
        if (k.M == M && k.N == N && k.K == K && k.swiglu == swiglu && k.knobs == knobs && k.room == room) return k.plan;
    Known& k = known[next++ & 15];
    k = Known{M, N, K, swiglu, knobs, room, find_plan(M, N, K, swiglu, room, ks_from)};
    return k.plan;
}

// The parts in which the sums of a product are added up belong to their accuracy where they leave unrounded, so they don't follow the estimate
// above, which drops slices as soon as a launch does without them: 2048 x 2048 at 33 to 165 rows in four slices 1.32e-7 from the
// exact sums, in one 2.70e-7.  They are those that units of whole groups of 64 rows by 32 columns are best cut into, which these
// sums have always had; a product takes that many or more.  0: 128 x 128 tiles.
static MidParts find_parts(int M, int N, int K, size_t room) {
    MidParts best{0, 0.f};
    const int cus = mid_cus(), nk = (K + 63) / 64;
    const double tiled = tiled_estimate(M, N, K, 1, cus);
    for (int nt = 2; nt <= 6; nt += 2)
        for (int mt = 1; mt <= 4; mt *= 2) {
            const int cap = nt * mt == 24 ? 160 : 32 * nt;
            const int64_t tiles_m = (M + 64 * mt - 1) / (64 * mt), whole = (N + cap - 1) / cap * tiles_m, across = (whole + cus - 1) / cus * cus / tiles_m;
            int cols = (int)((N + across - 1) / across + 7) / 8 * 8;
            cols = cols < 16 * nt ? 16 * nt : cols > cap ? cap : cols;
            const int64_t units = (N + cols - 1) / cols * tiles_m;
            const int tiles_w = (cols + 15) / 16, wave_t = tiles_w < nt ? tiles_w : nt;
            const double weights = 2.0 * N * K, again = weights * (tiles_m - 1) + 2.0 * K * 64 * mt * units, mem = weights / 9e6 + again / 18e6;
            for (int ks = 1; ks <= kMidMaxSlices; ++ks) {
                if (ks > 1 && (units * ks > cus + cus / 32 || nk / ks < 6 || (size_t)ks * M * N * sizeof(float) > room)) break;
                const int rounds = (int)((units * ks + cus - 1) / cus);
                const double lds = rounds * ((nk + ks - 1) / ks) * (128.0 * (wave_t + mt) + 16 * tiles_w + 64 * mt) / 2050.0;
                double us = (mem > lds ? mem : lds) * (1.0 + (mt == 4 && ks == 1 ? 0.23 : 0) + (nt == 6 ? 0.11 : 0)) + 3.8 * rounds + 6.2 * M * N / 6e6 / rounds;
                if (ks > 1) us += 1.2 + 15.0 * ks * M * N / 8e6;
                if ((float)us < tiled && (best.ks == 0 || (float)us < best.us)) best = MidParts{ks, (float)us};
            }
        }
    return best;
}

MidParts mid_float_parts(int M, int N, int K, size_t room) {
    if (!g_mid) return MidParts{0, 0.f};
    if (g_mid_nt || g_mid_mt || g_mid_ks) return MidParts{1, 0.f};  // a plan of the caller's own
    struct Known {
        int M, N, K;
        size_t room;
        MidParts parts;
    };
    static thread_local Known known[16];  // as in mid_plan
    static thread_local int next = 0;
    for (const Known& k : known)
        if (k.M == M && k.N == N && k.K == K && k.room == room) return k.parts;
    Known& k = known[next++ & 15];
    k = Known{M, N, K, room, find_parts(M, N, K, room)};
    return k.parts;
}

size_t mid_workspace_bytes(int M, int N, const MidPlan& p, int swiglu) {
    return p.ks > 1 ? (size_t)p.ks * M * N * (swiglu ? 2 : 1) * sizeof(float) : 0;
}

template <int NT, int MT, bool ONCE, bool HALF>
static int launch_mid_variant(const MidArgs& a, hipStream_t s) {
    constexpr int NS = mid_stages(NT, MT);
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_mid_kernel<2, 4, NT, MT, NS, ONCE, false, HALF>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e != hipSuccess) {
            raven_host::set_error("gemm (mid): hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    const size_t lds = mid_lds_bytes(2, 4, NT, MT, NS, a.wtiles, a.xtiles);
    RAVEN_REQUIRE(lds <= (size_t)kLds && a.wtiles <= 2 * NT && a.wtiles > 2 * (NT - 1) && a.xtiles <= 4 * MT && a.xtiles > 4 * (MT - 1), "gemm (mid): a unit of %d x %d does not fit", a.cols, a.bm);
    const int64_t units = (int64_t)a.tiles_m * a.tiles_n * a.ks;
    gemm_mid_kernel<2, 4, NT, MT, NS, ONCE, false, HALF><<<dim3((unsigned)((units + 7) / 8 * 8)), dim3(512), lds, s>>>(a);
    return raven_host::check_launch("gemm (mid)");
}

template <int EPI>
static int finish_slices(const MidArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)(((int64_t)a.M * (a.N / 4) + 255) / 256));
#define RAVEN_MID_FINISH(KS_) case KS_: gemm_mid_finish_kernel<EPI, KS_><<<grid, dim3(256), 0, s>>>(a); break;
    switch (a.ks) {
        RAVEN_MID_FINISH(2) RAVEN_MID_FINISH(3) RAVEN_MID_FINISH(4) RAVEN_MID_FINISH(5) RAVEN_MID_FINISH(6) RAVEN_MID_FINISH(7) RAVEN_MID_FINISH(8)
        default: RAVEN_REQUIRE(false, "gemm (mid): %d slices", a.ks);
    }
#undef RAVEN_MID_FINISH
    return raven_host::check_launch("gemm (mid, sums)");
}

// Rows that start on lines and in their middles by turns, in units whose tiles may be one more (HALF).  Not in slices: attn.proj at 195 rows takes 25.4 us
// where slices that begin 32 columns earlier took 24.5
static bool half_lines(const MidArgs& a, const MidPlan& p) {
    return g_mid_half && a.ks == 1 && a.K1 == 0 && a.ldw == a.K0 && a.K0 % 64 == 32 && a.K0 > 64 && ((uintptr_t)a.w & 127) == 0 && a.up_off % 2 == 0 &&
           mid_lds_bytes(2, 4, p.nt, p.mt, mid_stages(p.nt, p.mt), 2 * p.nt, a.xtiles) <= (size_t)kLds;
}

static int launch_mid(MidArgs a, const MidPlan& p, hipStream_t s, bool finish) {
    int rc;
    const bool half = half_lines(a, p);
    if (half) a.wtiles = 2 * p.nt;
#define RAVEN_MID_CASE(NT_, MT_)                                                                                                                    \
    case 10 * NT_ + MT_:                                                                                                                            \
        rc = a.tiles_m == 1 ? (half ? launch_mid_variant<NT_, MT_, true, true>(a, s) : launch_mid_variant<NT_, MT_, true, false>(a, s))             \
                            : (half ? launch_mid_variant<NT_, MT_, false, true>(a, s) : launch_mid_variant<NT_, MT_, false, false>(a, s));          \
        break;
#define RAVEN_MID_ROW(NT_) RAVEN_MID_CASE(NT_, 1) RAVEN_MID_CASE(NT_, 2) RAVEN_MID_CASE(NT_, 3) RAVEN_MID_CASE(NT_, 4)
    switch (p.nt * 10 + p.mt) {
        RAVEN_MID_ROW(1) RAVEN_MID_ROW(2) RAVEN_MID_ROW(3) RAVEN_MID_ROW(4) RAVEN_MID_ROW(5) RAVEN_MID_ROW(6)
        default: RAVEN_REQUIRE(false, "gemm (mid): no variant of %d x %d tiles", p.nt, p.mt);
    }
#undef RAVEN_MID_ROW
#undef RAVEN_MID_CASE
    if (rc || !finish) return rc;
    switch (a.kind) {
        case EPI_SWIGLU: return finish_slices<EPI_SWIGLU>(a, s);
        case EPI_FREE: return finish_slices<EPI_FREE>(a, s);
        case EPI_FREE_GELU: return finish_slices<EPI_FREE_GELU>(a, s);
        case EPI_FREE_TANH: return finish_slices<EPI_FREE_TANH>(a, s);
        default: return finish_slices<EPI_PLAIN>(a, s);
    }
}

int mid_gemm(const ProductArgs& q, const MidPlan& p, void* workspace, hipStream_t s, int* ks_left) {
    MidArgs a{};
    a.w = q.w; a.x0 = q.x0; a.x1 = q.x1; a.residual = q.residual; a.y = q.y; a.partial = static_cast<float*>(workspace);
    a.M = q.M; a.N = q.N; a.K0 = q.K0; a.K1 = q.x1 ? q.K1 : 0; a.ldw = q.ldw; a.ldx = q.ldx; a.ldy = q.ldy; a.up_off = q.up_off; a.out_f32 = q.out_f32;
    a.kind = !q.epi ? (q.swiglu ? EPI_SWIGLU : EPI_PLAIN) : q.epi->act == RAVEN_ACT_GELU ? EPI_FREE_GELU : q.epi->act == RAVEN_ACT_TANH ? EPI_FREE_TANH : EPI_FREE;
    a.cols = p.cols; a.bm = p.rows; a.wtiles = (p.cols * (q.swiglu ? 2 : 1) + 15) / 16; a.xtiles = p.rows / 16;
    a.tiles_m = p.tiles_m; a.tiles_n = p.tiles_n; a.ks = p.ks;
    if (q.epi) a.epi = *q.epi;
    if (q.rope) {
        a.rope = *q.rope;
        a.rope_on = 1;
    }
    RAVEN_REQUIRE(p.ks == 1 || (workspace && ((uintptr_t)workspace & 15) == 0), "gemm (mid): no workspace for the K slices");
    const bool finish = p.ks > 1 && !ks_left;
    if (ks_left) *ks_left = p.ks > 1 ? p.ks : 0;
    return launch_mid(a, p, s, finish);
}

// LDS of a unit of row groups
static size_t grouped_lds_bytes(int tile_rows, int wtiles, int xtiles) {
    return tile_rows == 32 ? mid_lds_bytes(4, 1, 2, 2, 4, wtiles, xtiles) : mid_lds_bytes(2, 4, 4, 1, 3, wtiles, xtiles);
}

template <int WN, int WM, int NT, int MT, int NS>
static int launch_grouped(const MidArgs& a, hipStream_t s) {
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_mid_kernel<WN, WM, NT, MT, NS, false, true>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e != hipSuccess) {
            raven_host::set_error("gemm (grouped): hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    const size_t lds = grouped_lds_bytes(a.bm, a.wtiles, a.xtiles);
    RAVEN_REQUIRE(lds <= (size_t)kLds && a.wtiles <= WN * NT && a.wtiles >= WN * NT / 2 && a.xtiles == WM * MT, "gemm (grouped): a unit of %d columns does not fit", a.cols);
    const int64_t units = (int64_t)a.tiles_m * a.tiles_n;
    RAVEN_REQUIRE(units < (1 << 28), "gemm (grouped): too many units");
    gemm_mid_kernel<WN, WM, NT, MT, NS, false, true><<<dim3((unsigned)((units + 7) / 8 * 8)), dim3(64 * WN * WM), lds, s>>>(a);
    return raven_host::check_launch("gemm (grouped)");
}

// Tiles of 32 rows: four waves side by side along the weight rows -- with few token rows the eight waves of the larger tiles would
// read mostly rows that do not exist out of LDS --, four stages of 20 KB, two workgroups per CU, so that one streams while the
// other fills its ring or stores (a unit of an expert of 768 channels has 12 to 32 K steps).
static int launch_grouped_rows(const MidArgs& a, hipStream_t s) {
    switch (a.bm) {
        case 32: return launch_grouped<4, 1, 2, 2, 4>(a, s);
        case 64: return launch_grouped<2, 4, 4, 1, 3>(a, s);
        default: RAVEN_REQUIRE(false, "gemm (grouped): tiles of %d rows", a.bm);
    }
}

// output columns of a unit, at least half of the variant's tiles
static int grouped_cols(int N, int swiglu) {
    const int cap = 128 / (swiglu ? 2 : 1), tiles_n = (N + cap - 1) / cap, cols = ((N + tiles_n - 1) / tiles_n + 7) / 8 * 8;
    return cols < cap / 2 ? cap / 2 : cols;
}

int mid_grouped(const void* x, int x_rows, const void* w, void* y, int rows, int N, int K, int swiglu, int out_f32, const RowGroups& g, hipStream_t s) {
    RAVEN_REQUIRE(x && w && y && g.group_of && g.group_row && g.group_end && g.used && g.n_tiles > 0 && N > 0 && N % 8 == 0 && K > 0 && K % 8 == 0 &&
                      (!swiglu || (g.x_scale && !out_f32)) && (g.extra_group < 0 || g.w_extra), "gemm (grouped): bad arguments");
    RAVEN_REQUIRE((int64_t)x_rows * K < (1ll << 31) && (int64_t)N * 2 * K < (1ll << 31) && (int64_t)rows * N < (1ll << 40), "gemm (grouped): too large");
    MidArgs a{};
    a.w = static_cast<const bf16*>(w);
    a.x0 = static_cast<const bf16*>(x);
    a.y = y;
    a.M = rows; a.N = N; a.K0 = K; a.ldw = K; a.ldx = K; a.ldy = N; a.up_off = N; a.out_f32 = out_f32;
    a.cols = grouped_cols(N, swiglu);
    a.kind = swiglu ? EPI_SWIGLU : EPI_FREE;
    a.wtiles = (a.cols * (swiglu ? 2 : 1) + 15) / 16;
    a.tiles_n = (N + a.cols - 1) / a.cols;
    a.bm = g.tile_rows; a.xtiles = (g.tile_rows + 15) / 16; a.tiles_m = g.n_tiles; a.ks = 1;
    a.epi.scale = 1.f;
    a.groups = g;
    return launch_grouped_rows(a, s);
}

}  // namespace raven

extern "C" int raven_middle_plan(int32_t M, int32_t N, int32_t K, int32_t swiglu, size_t workspace_bytes, int32_t* plan) {
    using namespace raven;
    RAVEN_REQUIRE(plan && M > 0 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0, "middle_plan: bad arguments");
    const MidPlan p = mid_plan(M, N, K, 0, swiglu, workspace_bytes);
    const int32_t out[6] = {p.nt, p.mt, p.cols, p.rows, p.ks, p.tiles_m * p.tiles_n * p.ks};
    for (int i = 0; i < 6; ++i) plan[i] = p.nt ? out[i] : 0;
    return 0;
}

extern "C" int raven_grouped_unit(int32_t N, int32_t swiglu, int32_t tile_rows, int32_t* unit) {
    using namespace raven;
    RAVEN_REQUIRE(unit && N > 0 && N % 8 == 0 && (tile_rows == 32 || tile_rows == 64), "grouped_unit: bad arguments");
    const int cols = grouped_cols(N, swiglu), wtiles = (cols * (swiglu ? 2 : 1) + 15) / 16;
    unit[0] = cols;
    unit[1] = wtiles;
    unit[2] = (int32_t)grouped_lds_bytes(tile_rows, wtiles, tile_rows / 16);
    return 0;
}
