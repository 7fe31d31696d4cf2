// Skinny GEMMs of the decode path: Y[M,N] = X[M,K] W[N,K]^T with M = a handful of token rows and
// W a weight matrix that is streamed from HBM exactly once per call (per 32 rows of X).
//
// Three kernels:
//   gemv_kernel  (any T, up to 8 rows of X per pass)  -- X lives in LDS, every wave owns whole rows
//                of W, reads them with 16-byte lane-contiguous loads and accumulates with
//                v_dot2_f32_bf16 / fp32 FMA; a DPP wave reduction finishes each row.
//   mfma_kernel  (bf16, up to 32 rows of X per pass)   -- 16-row tiles of W are the A operand of
//                v_mfma_f32_16x16x32_bf16, X is the B operand; the four or eight waves of a workgroup
//                split K and reduce through LDS.
//   rows_f32_kernel (float, 5 rows and more, fewer where K is short) -- 16 rows of W against 16 to 64 rows of X on v_mfma_f64_16x16x4_f64.
// Epilogues (all round the fp32 accumulator to T first, as an nn.Linear output would be stored):
//   plain (+ residual add in T, + optional float store)   RMM:493, 509, 711, 534-535
//   SwiGLU: T(T(silu(gate)) * up), gate row j, up row j+I  RMM:507-508
// The adapter's concat (RMM:776) is folded in by giving X as two pointers that cover K0 and K1.

#include <algorithm>
#include <string>
#include <type_traits>

#include "raven_common.h"
#include "row_helpers.h"

extern "C" int raven_gemv_fused(const void* x0, const void* x1, const void* norm_a, const void* norm_b, void* xa_out,
                                const void* w, const void* residual, void* y, int32_t N, int32_t K0, int32_t K1, float eps,
                                int32_t swiglu, int32_t out_f32, int32_t dtype, void* stream);

namespace raven {

extern int g_tiled_min_rows;
bool tiled_gemm_fits(int M, int N, int K0, int K1, int dtype, int swiglu, size_t workspace_bytes, bool aligned, int f32_sums = 0);
int tiled_gemm(const void* x0, int ldx, const void* x1, const void* w, const void* residual, void* y, int M, int N, int K0, int K1, int swiglu,
               int out_f32, void* workspace, size_t workspace_bytes, hipStream_t s, int* ks_left);

bool gemv1_fits(int K, int dtype);
int gemv1_free(const void* x0, const void* x1, const void* w, void* y, int N, int K0, int K1, const raven_epilogue& epi, int dtype,
               hipStream_t s);

constexpr int kNormNone = 0, kNormAhead = 1, kNormBehind = 2;

struct GemmArgs {
    const void* w;         // [N_total, K]
    const void* x0;        // [M, k0]
    const void* x1;        // [M, k1] or null
    const void* residual;  // [M, N] or null
    void* y;               // [M, N] (T, or float when out_f32)
    int M, N, K, k0, k1;   // N = number of output columns (I for SwiGLU)
    int out_f32;
    int units_per_wave;    // gemv: row pairs per wave
    int interleave;        // gemv: unit = u * total_waves + wave (1) or wave * units_per_wave + u (0)
    int row_stride;        // mfma: 1 = a tile is 16 neighbouring weight rows, 2 = every second row (see mfma_kernel)
    int line_aligned;      // mfma: the rows of a tile all start at the same offset inside a 128-byte line
    raven_epilogue epi;    // EPI_FREE only (residual and y already offset to the pass)
    int ldy;               // EPI_FREE only: elements between two rows of y and residual
    int rows_per_unit;     // mfma, ragged variants: weight rows (per side for SwiGLU) a workgroup owns; its last tile is partly empty
    int early;             // mfma, EPI_FREE: a residual whose pieces and those of y start on 16 bytes, requested in front of the weights
    NormAhead ahead;       // mfma, EPI_FREE only
    NormBehind behind;     // mfma, free epilogues only
};

// Launch-shape knobs (raven_set_tuning); 0 = automatic.
struct Tuning {
    int gemv_units_per_wave = 0;
    int gemv_interleave = 1;
    int gemv_nontemporal = 1;
    int gemv_wgs_per_cu = 4;
    int gemm_four_tiles = 1;
    int gemm_mfma_min_rows = 2;  // fewer rows go to the vector kernels (one row: the K-split GEMV)
    int gemm_one_round = 1;      // one workgroup of eight waves per CU: 0 never, 1 by rule, 2 wherever the matrix is narrow enough
    int gemm_ragged = 1;         // 0 never, 1 = one workgroup per resident slot with partly empty last tiles where the shape divides so
};
static Tuning g_tuning;
extern int g_f32_norm_rows;

int set_skinny_tuning(const char* key, int value) {
    const std::string k(key);
    if (k == "gemv_units_per_wave") g_tuning.gemv_units_per_wave = value;
    else if (k == "gemv_interleave") g_tuning.gemv_interleave = value;
    else if (k == "gemv_nontemporal") g_tuning.gemv_nontemporal = value;
    else if (k == "gemv_wgs_per_cu") g_tuning.gemv_wgs_per_cu = value;
    else if (k == "gemm_four_tiles") g_tuning.gemm_four_tiles = value;
    else if (k == "gemm_one_round") g_tuning.gemm_one_round = value;
    else if (k == "gemm_ragged") g_tuning.gemm_ragged = value;
    else if (k == "f32_norm_rows") g_f32_norm_rows = value;
    else if (k == "gemm_mfma_min_rows" && value >= 2) g_tuning.gemm_mfma_min_rows = value;
    else return -1;
    return 0;
}

// weight rows are read exactly once: stream them past the caches
template <bool NT, typename T>
__device__ __forceinline__ Chunk<T> load_weight(const T* p) {
    if (!NT) return load_chunk(p);
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    Chunk<T> c;
    *reinterpret_cast<u32x4*>(&c) = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return c;
}

template <typename T, int EPI = EPI_PLAIN>
__device__ __forceinline__ void store_out(const GemmArgs& a, int m, int n, float acc) {
    if (is_free(EPI)) {
        store_free<T, EPI>(a.epi, a.y, (int64_t)m * a.ldy + n, n, acc);
        return;
    }
    float r = round_to<T>(acc);
    if (a.residual) r = round_to<T>(r + to_f32(static_cast<const T*>(a.residual)[(int64_t)m * a.N + n]));
    if (a.out_f32)
        static_cast<float*>(a.y)[(int64_t)m * a.N + n] = r;
    else
        static_cast<T*>(a.y)[(int64_t)m * a.N + n] = from_f32<T>(r);
}

template <typename T>
__device__ __forceinline__ float swiglu(float gate_acc, float up_acc) {
    const float g = round_to<T>(gate_acc), u = round_to<T>(up_acc);
    return round_to<T>(round_to<T>(silu_f32(g)) * u);
}

// ------------------------------------------------------------------------------------------------
// gemv_kernel: 256 threads; dynamic LDS holds X as [MB][K] of T.  WIDE (float): products and sums in 64 bits, as in rows_f32_kernel.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ double dot_chunk(const Chunk<float>& a, const Chunk<float>& b, double acc) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_fma((double)a.v[e], (double)b.v[e], acc);
    return acc;
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) v += __shfl_xor(v, d, 64);
    return v;
}

template <typename T, int MB, int EPI, bool NT, bool WIDE = false>
__global__ __launch_bounds__(256) void gemv_kernel(GemmArgs a) {
    typedef std::conditional_t<WIDE, double, float> Sum;
    constexpr int E = Chunk<T>::N;
    constexpr int U = 4;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* xs = reinterpret_cast<T*>(smem_raw);

    const int K = a.K, n_chunks = K / E, c0 = a.k0 / E;
    // stage X: row m of LDS = concat(x0[m], x1[m]); rows >= M are zero
    for (int i = threadIdx.x; i < MB * n_chunks; i += 256) {
        const int m = i / n_chunks, c = i - m * n_chunks;
        Chunk<T> v = zero_chunk<T>();
        if (m < a.M) {
            v = (c < c0) ? load_chunk(static_cast<const T*>(a.x0) + (int64_t)m * a.k0 + c * E)
                         : load_chunk(static_cast<const T*>(a.x1) + (int64_t)m * a.k1 + (c - c0) * E);
        }
        store_chunk(xs + (int64_t)m * K + c * E, v);
    }
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int gwave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int total_waves = gridDim.x * 4;
    const int n_units = (EPI == EPI_SWIGLU) ? a.N : (a.N + 1) / 2;
    const T* W = static_cast<const T*>(a.w);

    for (int u = 0; u < a.units_per_wave; ++u) {
        // interleaved: at any moment the waves of the whole grid read neighbouring rows
        const int unit = a.interleave ? u * total_waves + gwave : gwave * a.units_per_wave + u;
        if (unit >= n_units) break;
        int r0, r1;
        bool r1_ok = true;
        if (EPI == EPI_SWIGLU) {
            r0 = unit;
            r1 = unit + a.N;
        } else {
            r0 = 2 * unit;
            r1 = r0 + 1;
            if (r1 >= a.N) { r1 = r0; r1_ok = false; }
        }
        const T* w0 = W + (int64_t)r0 * K;
        const T* w1 = W + (int64_t)r1 * K;
        Sum acc0[MB], acc1[MB];
#pragma unroll
        for (int m = 0; m < MB; ++m) acc0[m] = acc1[m] = 0;

        for (int c = lane; c < n_chunks; c += 64 * U) {
            Chunk<T> a0[U], a1[U];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int cc = c + 64 * j;
                if (cc < n_chunks) {
                    a0[j] = load_weight<NT>(w0 + cc * E);
                    a1[j] = load_weight<NT>(w1 + cc * E);
                } else {
                    a0[j] = zero_chunk<T>();
                    a1[j] = zero_chunk<T>();
                }
            }
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int cc = min(c + 64 * j, n_chunks - 1);
#pragma unroll
                for (int m = 0; m < MB; ++m) {
                    const Chunk<T> xv = load_chunk(xs + (int64_t)m * K + cc * E);
                    acc0[m] = dot_chunk(a0[j], xv, acc0[m]);
                    acc1[m] = dot_chunk(a1[j], xv, acc1[m]);
                }
            }
        }
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            acc0[m] = wave_sum(acc0[m]);
            acc1[m] = wave_sum(acc1[m]);
        }
        if (lane == 0) {
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                if (m < a.M) {
                    if (EPI == EPI_SWIGLU) {
                        static_cast<T*>(a.y)[(int64_t)m * a.N + unit] = from_f32<T>(swiglu<T>((float)acc0[m], (float)acc1[m]));
                    } else {
                        store_out<T, EPI>(a, m, r0, (float)acc0[m]);
                        if (r1_ok) store_out<T, EPI>(a, m, r1, (float)acc1[m]);
                    }
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// mfma_kernel: bf16, 4 waves (or 8) that split K; MT = ceil(M/16) batch tiles; NT weight
// tiles of 16 rows per workgroup.  D = A * B with A = W tile [16 n x 32 k], B = X^T [32 k x 16 m]:
// lane l supplies A[n = l%16][k = 8*(l/16) ..+8] and B[k = 8*(l/16) ..+8][m = l%16] and receives
// D[n = 4*(l/16) + v][m = l%16], v = 0..3.
//
// The MFMA operand layout puts 16 different matrix rows into 16 neighbouring lanes; loading it straight
// from global memory makes every quarter-wave touch 16 cache lines for 256 bytes, and the L1 address path
// (not HBM) then caps the kernel near 3 TB/s.  So K is walked in macro-steps of 128 elements: each wave
// loads its rows with row-contiguous 16-byte lanes (a quarter-wave reads 256 consecutive bytes of one
// row), parks them in a wave-private LDS tile with 272-byte row pitch, and reads the MFMA fragments from
// there (conflict-free: 16 rows x 16 bytes cover the 64 banks once).  The next macro-step's global loads
// are issued into registers as soon as the current one is parked, before it is multiplied.  No barrier inside the K loop: every
// wave only touches its own LDS tile.
//
// A quarter-wave's 256 bytes should also be two whole 128-byte lines: a row that starts 64 bytes into a line
// makes them three, and that alone costs 20 % of the bandwidth.  K = 5280 (10560 bytes per row) puts every
// second row there.  So with row_stride = 2 a tile is made of 16 rows of the SAME parity, all its rows are
// misaligned by the same amount, and the macro-steps of such a tile start `shift` elements into the row
// (at the next line boundary); the `shift` elements before them and whatever is left behind the last full
// macro-step are single 32-wide MFMA steps straight from global memory (first and last wave).
// ------------------------------------------------------------------------------------------------
// KM = k-values per macro-step: 128, or 64 for the variants with four weight tiles per workgroup (the same
// bytes per macro-step; a quarter-wave then reads two rows of 128 bytes).  LDS rows are KM + 8 elements long
// (272 or 144 bytes: both spread 16 rows over the 64 banks without conflicts for 16-byte reads).
//
// RAG: a workgroup owns a.rows_per_unit rows (per side for SwiGLU) instead of 16 per tile slot: its tile slots cover them
// 16 at a time and the last slot is partly empty (its missing rows are neither loaded nor stored).  This lets the host cut
// a matrix into exactly as many workgroups as the chip holds at once (17920 gate rows = 512 x 35), where whole tiles
// would leave a partly filled last round.
//
// WAVES = 8 with D register sets in flight: the variants of launch_one_round, one workgroup per CU.
// NORM: half of a norm that is shared out between two products (NormAhead, NormBehind); instantiations of their own, for with both behind run-time branches
// every launch of a free epilogue was 0.3 to 0.5 us longer.
template <int MT, int NT, int EPI, int KM = 128, bool RAG = false, int WAVES = 4, int D = 1, int NORM = kNormNone>
__global__ __launch_bounds__(64 * WAVES) void mfma_kernel(GemmArgs a) {
    constexpr int ROWS = 16 * (NT + MT);
    constexpr int kPitch = KM + 8;
    constexpr int LPR = KM / 8;        // lanes per row of a macro-step
    constexpr int RPI = 64 / LPR;      // rows per load instruction
    constexpr int IPT = 16 / RPI;      // load instructions per 16-row tile
    constexpr int NG = EPI == EPI_SWIGLU ? NT / 2 : NT;  // tiles side by side along N (SwiGLU: NG gate tiles + their NG up tiles)
    __shared__ __align__(16) bf16 stage[WAVES][ROWS][kPitch];
    static_assert(sizeof(bf16) * WAVES * ROWS * kPitch >= sizeof(float) * (WAVES - 1) * NT * MT * 64 * 4, "stage doubles as the reduction buffer");
    __shared__ float row_inv[NORM == kNormBehind ? 16 * MT : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ln = lane & 15, kq = lane >> 4;
    const int K = a.K;
    const int rs = a.row_stride;
    if constexpr (is_free(EPI)) {  // gemm_narrow_free: a grid row per 16 * MT rows of X
        const int64_t m0 = (int64_t)blockIdx.y * 16 * MT;
        a.M -= (int)m0;
        a.x0 = static_cast<const bf16*>(a.x0) + m0 * a.k0;
        a.y = static_cast<char*>(a.y) + m0 * a.ldy * (a.epi.out_f32 ? 4 : 2);
        if (a.epi.residual) a.epi.residual += m0 * a.ldy;
    }
    // a group is rs units: with rs = 2 the even unit takes the even rows of the group's tiles, the odd unit the odd rows
    const int group = rs == 2 ? blockIdx.x >> 1 : blockIdx.x;
    const int parity = rs == 2 ? blockIdx.x & 1 : 0;

    const bf16* W = static_cast<const bf16*>(a.w);
    int tile_row0[NT];  // first weight row of each tile; row i of the tile is tile_row0 + i * rs
    int tile_out0[NT];  // output column of that row
    bool tile_ok[NT];
    int tile_rows[NT];  // RAG: rows of the tile that exist (1..16 where tile_ok); 16 otherwise
    const int rpu = RAG ? a.rows_per_unit : 16 * NG;  // rows a unit owns per side
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int first = (group * rpu + (t % NG) * 16) * rs;   // SwiGLU: the first NG tiles are gate tiles, the others their up tiles
        tile_ok[t] = first < a.N && (!RAG || (t % NG) * 16 < rpu);
        tile_rows[t] = RAG ? min(16, rpu - (t % NG) * 16) : 16;
        tile_out0[t] = (tile_ok[t] ? first : group * rpu * rs) + parity;
        tile_row0[t] = tile_out0[t] + (EPI == EPI_SWIGLU ? (t / NG) * a.N : 0);
        if (RAG && !tile_ok[t]) tile_rows[t] = 1;  // reads row 0 of the unit's first tile, stores nothing
    }

    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    struct Staged {
        u32x4 w[NT][IPT];
        u32x4 x[MT][IPT];
    };
    bf16(*my)[kPitch] = stage[wave];
    const int lr = lane / LPR, lc = (lane % LPR) * 8;  // loader role: row within a group of RPI, first element of the chunk

    // What the ends of a shared norm read is requested in front of the weights, so that nothing waits for it: the sums of squares (16 lanes to a row, the
    // rows shared out over the waves), and the residuals and weights of wave 0, which stores.
    constexpr int RP = NORM == kNormBehind ? (16 * MT + 4 * WAVES - 1) / (4 * WAVES) : 1, SP = kNormParts / 64;
    f32x4 squares[RP][SP];
    const int pitch = norm_pitch(a.behind.parts);
    if constexpr (NORM == kNormBehind) {
#pragma unroll
        for (int j = 0; j < RP; ++j)
#pragma unroll
            for (int i = 0; i < SP; ++i)
                squares[j][i] = *reinterpret_cast<const f32x4*>(a.behind.squares + min(4 * (wave + WAVES * j) + kq, a.M - 1) * pitch + min(4 * (ln + 16 * i), pitch - 4));
    }
    constexpr bool EARLY = EPI == EPI_FREE && !RAG;  // (a residual requested behind the products: 2048 x 2048 at 20 rows 8.2 us, so 6.7)
    f32x4 res[EARLY ? NT : 1][MT], norm_w[NORM == kNormAhead ? NT : 1];
    if constexpr (EARLY) {
        auto four_of = [&](const float* p) { return rs == 1 ? *reinterpret_cast<const f32x4*>(p) : f32x4{p[0], p[2], p[4], p[6]}; };
        if (wave == 0 && a.early) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int n = tile_out0[t] + kq * 4 * rs;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) res[t][mt] = four_of(a.epi.residual + (int64_t)min(mt * 16 + ln, a.M - 1) * a.ldy + n);
                if constexpr (NORM == kNormAhead) norm_w[t] = four_of(a.ahead.weight + n);
            }
        }
    }
    // the rows' factors, formed while the first weights are on their way
    auto row_factors = [&]() __attribute__((always_inline)) {
        if constexpr (NORM == kNormBehind) {
            const NormBehind& b = a.behind;
#pragma unroll
            for (int j = 0; j < RP; ++j) {
                float sum = 0.f;
#pragma unroll
                for (int i = 0; i < SP; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum += 4 * (ln + 16 * i) + e < b.parts ? squares[j][i][e] : 0.f;
                const float inv = 1.0f / sqrtf(row16_sum(sum) / (float)b.dim + b.eps);
                const int m = 4 * (wave + WAVES * j) + kq;
                if (ln == 0 && m < a.M) {
                    row_inv[m] = inv;
                    if (b.factors && blockIdx.x == 0) b.factors[m] = inv;
                }
            }
        }
    };

    // X is given as up to two K segments (the adapter's concat); each is walked on its own
#pragma unroll 1
    for (int seg = 0; seg < 2; ++seg) {
        const int seg_len = seg == 0 ? a.k0 : a.k1;
        if (seg_len == 0) continue;
        const int wk0 = seg == 0 ? 0 : a.k0;  // column of W where this segment starts
        const bf16* X = static_cast<const bf16*>(seg == 0 ? a.x0 : a.x1);
        const int ldx = seg == 0 ? a.k0 : a.k1;
        // elements in front of the first 128-byte line boundary of this segment's weight rows (0 or 32, else not used)
        int shift = 0;
        if (a.line_aligned) {
            const int mis = (int)(reinterpret_cast<uintptr_t>(W + (int64_t)tile_row0[0] * K + wk0) & 127);
            shift = mis == 64 ? 32 : 0;
#pragma unroll
            for (int t = 1; t < NT; ++t)
                if ((int)(reinterpret_cast<uintptr_t>(W + (int64_t)tile_row0[t] * K + wk0) & 127) != mis) shift = 0;
            if (shift > seg_len) shift = 0;
        }
        const int n_macro = (seg_len - shift) / KM;
        // the waves take the macro-steps in turn, so that the workgroup as a whole walks its rows in pieces of
        // WAVES * KM contiguous elements (DRAM pages are then read in longer runs than one wave's 256 bytes)
        const int mb = wave, me = n_macro;

        auto fetch = [&](int mac, Staged& st) {  // global -> registers, row-contiguous lanes
            const int k = shift + mac * KM + lc;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < IPT; ++i) {
                    const int m = min(mt * 16 + RPI * i + lr, a.M - 1);  // rows past M repeat the last one; never stored
                    st.x[mt][i] = *reinterpret_cast<const u32x4*>(X + (int64_t)m * ldx + k);
                }
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < IPT; ++i) {
                    if (RAG && RPI * i + lr >= tile_rows[t]) continue;  // rows the tile does not have: their products are never stored
                    st.w[t][i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(W + (int64_t)(tile_row0[t] + (RPI * i + lr) * rs) * K + wk0 + k));
                }
        };
        auto park = [&](const Staged& st) {  // registers -> this wave's LDS tile
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < IPT; ++i) *reinterpret_cast<u32x4*>(&my[t * 16 + RPI * i + lr][lc]) = st.w[t][i];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < IPT; ++i) *reinterpret_cast<u32x4*>(&my[(NT + mt) * 16 + RPI * i + lr][lc]) = st.x[mt][i];
        };
        auto multiply = [&]() {  // LDS -> MFMA fragments
#pragma unroll
            for (int j = 0; j < KM / 32; ++j) {
                bf16x8 bv[MT];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)  // same access type as the stores in park(): the two must stay ordered
                    bv[mt] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&my[(NT + mt) * 16 + ln][32 * j + 8 * kq]));
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const bf16x8 av = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&my[t * 16 + ln][32 * j + 8 * kq]));
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv[mt], acc[t][mt], 0, 0, 0);
                }
            }
        };

        // lanes exchange data through the tile without a workgroup barrier: pin the order of the LDS
        // accesses for the compiler (the LDS itself executes one wave's accesses in order)
        auto wave_sync = []() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        if constexpr (D == 1) {
            // one register set: its loads for macro-step s+1 are in flight while step s is multiplied out of LDS
            Staged st{};
            if (mb < me) fetch(mb, st);
            if (seg == 0) row_factors();
            for (int mac = mb; mac < me; mac += WAVES) {
                park(st);
                wave_sync();
                if (mac + WAVES < me) fetch(mac + WAVES, st);
                multiply();
                wave_sync();
            }
        } else if (mb >= me) {
            if (seg == 0) row_factors();
        } else {
            // rounds of D steps, each requesting the next round's loads (none under a branch of its own, so that the waits count only the
            // set being parked); what lies past the end loads the wave's first step again and is not multiplied
            Staged st[D];
            const int steps = (me - mb + WAVES - 1) / WAVES;
            auto step_of = [&](int i) { return i < steps ? mb + i * WAVES : mb; };
#pragma unroll
            for (int d = 0; d < D; ++d) fetch(step_of(d), st[d]);
            if (seg == 0) row_factors();
            int done = 0;
#pragma unroll 1
            for (; done + D < steps; done += D) {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    park(st[d]);
                    wave_sync();
                    fetch(step_of(done + D + d), st[d]);
                    multiply();
                    wave_sync();
                }
            }
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (done + d >= steps) break;
                park(st[d]);
                wave_sync();
                multiply();
                wave_sync();
            }
        }
        // 32-element steps in front of the first and behind the last macro-step: first and last wave, straight from global memory
        if (wave == 0 || wave == WAVES - 1) {
            const int kb = wave == 0 ? 0 : shift + n_macro * KM, ke = wave == 0 ? shift : seg_len;
            for (int k = kb; k < ke; k += 32) {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int wr = RAG ? min(ln, tile_rows[t] - 1) : ln;  // a partly empty tile repeats its last row
                    const bf16x8 wv = *reinterpret_cast<const bf16x8*>(W + (int64_t)(tile_row0[t] + wr * rs) * K + wk0 + k + kq * 8);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        const int m = min(mt * 16 + ln, a.M - 1);
                        const bf16x8 xv = *reinterpret_cast<const bf16x8*>(X + (int64_t)m * ldx + k + kq * 8);
                        acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv, acc[t][mt], 0, 0, 0);
                    }
                }
            }
        }
    }

    // cross-wave reduction over the K split (the staging tiles are free now)
    __syncthreads();
    float(*red)[NT * MT][64][4] = reinterpret_cast<float(*)[NT * MT][64][4]>(&stage[0][0][0]);
    if (wave > 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[wave - 1][t * MT + mt][lane][v] = acc[t][mt][v];
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float others = red[0][t * MT + mt][lane][v];
#pragma unroll
                for (int r = 1; r < WAVES - 1; ++r) others += red[r][t * MT + mt][lane][v];
                acc[t][mt][v] += others;
            }

    if constexpr (NORM == kNormBehind) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const float inv = row_inv[min(mt * 16 + ln, a.M - 1)];
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t][mt] *= inv;
        }
    }
    if (EARLY && a.early) {  // (float outputs)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 16 + ln;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (!tile_ok[t]) continue;
                const int n = tile_out0[t] + kq * 4 * rs;
                const int64_t at = (int64_t)m * a.ldy + n;
                f32x4 f = acc[t][mt] * a.epi.scale;
                if (NORM == kNormNone && a.epi.bias) f += rs == 1 ? load4(a.epi.bias + n) : f32x4{a.epi.bias[n], a.epi.bias[n + 2], a.epi.bias[n + 4], a.epi.bias[n + 6]};
                f += res[t][mt];
                f32x4 g{};
                if constexpr (NORM == kNormAhead) g = f * norm_w[t];
                if (m < a.M) {
                    float* y = static_cast<float*>(a.y) + at;
                    if (rs == 1) {
                        store4(y, f);
                        if constexpr (NORM == kNormAhead) store4(a.ahead.xw + at, g);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            y[2 * v] = f[v];
                            if constexpr (NORM == kNormAhead) a.ahead.xw[at + 2 * v] = from_f32<bf16>(g[v]);
                        }
                    }
                }
                if constexpr (NORM == kNormAhead) {
                    float sq = f[0] * f[0] + f[1] * f[1] + f[2] * f[2] + f[3] * f[3];
                    sq += __shfl_xor(sq, 16, 64);
                    sq += __shfl_xor(sq, 32, 64);
                    // tiles in the order of their first columns; with rs = 2 the even and the odd columns of 32 are a tile each
                    if (kq == 0 && m < a.M) a.ahead.squares[m * norm_pitch(a.N / 16) + (tile_out0[t] - parity) / 16 + parity] = sq;
                }
            }
        }
        return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + ln;
        if (m >= a.M) continue;
        if (EPI == EPI_SWIGLU) {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                if (!tile_ok[g]) continue;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (RAG && kq * 4 + v >= tile_rows[g]) continue;
                    const int n = tile_out0[g] + (kq * 4 + v) * rs;
                    static_cast<bf16*>(a.y)[(int64_t)m * a.N + n] = from_f32<bf16>(swiglu<bf16>(acc[g][mt][v], acc[NG + g][mt][v]));
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (!tile_ok[t]) continue;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (!RAG || kq * 4 + v < tile_rows[t]) store_out<bf16, EPI>(a, m, tile_out0[t] + (kq * 4 + v) * rs, acc[t][mt][v]);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// rows_f32_kernel: a workgroup owns 16 weight rows (SwiGLU: 16 gate rows and their up rows) and 16 MT token rows, its four or eight waves split K
// and add up through LDS.  A lane loads 16 bytes of row l % 16 at columns 16 c + 4 (l / 16) ..+3 straight from memory -- of W and of X
// alike, so that product j of a chunk, which takes element j of every lane's load, multiplies the same columns on both sides.  Products
// and sums are in 64 bits (exact products; the fp32 instruction's one long chain of sums per element was 1.7 times further from the
// exact result than gemv_kernel's 64 short ones, and no faster here).
// What bounds it is a wave's walk over its share of K (small models) or the 64-byte row pieces (large matrices: about 3 TB/s), not the
// matrix cores.  It reads W once per 64 rows where gemv_kernel takes passes of 8, each a launch: a product of 17 rows, 256 x 704 to 1408 x 256, three
// launches of 4.5 to 8 us, now one of 5; 200 rows 25 launches.  With four waves the walk was longer than gemv_kernel's passes for few rows: us,
// passes / four waves / eight, 2048 x 2048 at 8 rows 11.7 / 12.1 / 9.8, 512 x 4096 at 9 rows 21.4 / 19.7 / 15.8, SwiGLU of 512 x 2048 at 9, 17 and 33 rows 13.5 / 19.4 / 14.9, 23.0 / 24.6 / 21.9, 42.3 / 42.6 / 39.1.
// ------------------------------------------------------------------------------------------------
// NORMED: the rows of x0 go through one or two RMSNorms first.  A workgroup norms its token rows itself, a wave per row in turn, and multiplies them out of
// the LDS: a small model's launch of its own for a norm takes 3.2 us, and 2.8 to enqueue, more than the repeated work of 16 to 90 workgroups.  Squares are added
// as rmsnorm_kernel adds them, rows of up to 1024 columns: the same bits.  Rotation and cache append of a chunk's q | k | v rows may ride in the epilogue.
struct NormedRows : GemmArgs {
    const float *norm_a, *norm_b;  // x0 <- norm_b(norm_a(x0)); norm_a may be null
    float* xa_out;                 // norm_a(x0), or null
    float eps;
    int rope_on;                   // EPI_PLAIN: the rows leave as RopeRows says instead of to y
    RopeRows rope;
};
constexpr int kNormedColumns = 1024;
__host__ __device__ constexpr int normed_pitch(int k0) { return k0 + 20; }  // floats: 16 rows' pieces of 16 bytes on all 64 banks

template <int EPI, int MT, int WAVES, bool NORMED = false>
__global__ __launch_bounds__(64 * WAVES) void rows_f32_kernel(std::conditional_t<NORMED, NormedRows, GemmArgs> a) {
    typedef __attribute__((ext_vector_type(4))) double f64x4;
    constexpr int NT = EPI == EPI_SWIGLU ? 2 : 1, U = 4;
    __shared__ __align__(16) f64x4 red[WAVES - 1][NT * MT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT, K = a.K;
    const float* w[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) w[t] = static_cast<const float*>(a.w) + (int64_t)(min(n0 + r, a.N - 1) + t * a.N) * K;
    int64_t row[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) row[j] = min(m0 + 16 * j + r, a.M - 1);
    const int chunks = (K + 15) / 16, c0 = chunks * wave / WAVES, c1 = chunks * (wave + 1) / WAVES;

    extern __shared__ __align__(16) float normed[];  // NORMED: [16 MT][normed_pitch(k0)]
    if constexpr (NORMED) {
        constexpr int RPW = 16 * MT / WAVES, NI = kNormedColumns / 256;
        const int pieces = a.k0 / 4, pitch = normed_pitch(a.k0);
        f32x4 v[RPW][NI];
#pragma unroll
        for (int i = 0; i < RPW; ++i)
#pragma unroll
            for (int n = 0; n < NI; ++n)
                if (256 * n < a.k0) v[i][n] = load4(static_cast<const float*>(a.x0) + (int64_t)min(m0 + wave + WAVES * i, a.M - 1) * a.k0 + 4 * min(lane + 64 * n, pieces - 1));
        auto norm = [&](f32x4 (&x)[NI], const float* weight) __attribute__((always_inline)) {
            float sums[NI];
#pragma unroll
            for (int n = 0; n < NI; ++n) {
                sums[n] = 0.f;
                if (256 * n >= a.k0) continue;
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) ss = __builtin_fmaf(x[n][e], x[n][e], ss);
                sums[n] = raven::wave_sum(lane + 64 * n < pieces ? ss : 0.f);
            }
            const float inv = rsqrtf((sums[0] + sums[1] + sums[2] + sums[3]) / (float)a.k0 + a.eps);
#pragma unroll
            for (int n = 0; n < NI; ++n)
                if (256 * n < a.k0) {
                    const f32x4 w = load4(weight + 4 * min(lane + 64 * n, pieces - 1));
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[n][e] = x[n][e] * inv * w[e];
                }
        };
        static_assert(NI == 4, "the sum above");
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            const int at = wave + WAVES * i;
            if (a.norm_a) {
                norm(v[i], a.norm_a);
#pragma unroll
                for (int n = 0; n < NI; ++n)
                    if (a.xa_out && blockIdx.x == 0 && m0 + at < a.M && lane + 64 * n < pieces) store4(a.xa_out + (int64_t)(m0 + at) * a.k0 + 4 * (lane + 64 * n), v[i][n]);
            }
            norm(v[i], a.norm_b);
#pragma unroll
            for (int n = 0; n < NI; ++n)
                if (lane + 64 * n < pieces) store4(normed + at * pitch + 4 * (lane + 64 * n), v[i][n]);
        }
        __syncthreads();
    }

    f64x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[t][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    auto load_x = [&](int j, int k) __attribute__((always_inline)) {
        const bool second = k >= a.k0;
        if constexpr (NORMED) {
            if (!second) return load4(normed + (16 * j + r) * normed_pitch(a.k0) + k);
        }
        const float* x = second ? static_cast<const float*>(a.x1) - a.k0 : static_cast<const float*>(a.x0);
        return *reinterpret_cast<const f32x4*>(x + row[j] * (second ? a.k1 : a.k0) + k);
    };
    auto multiply = [&](const f32x4 (&wv)[NT], const f32x4 (&xv)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)wv[t][i], (double)xv[j][i], acc[t][j], 0, 0, 0);
    };
    int c = c0;
    for (; c + U <= c1 && 16 * (c + U) <= K; c += U) {
        f32x4 wv[U][NT], xv[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = 16 * (c + u) + 4 * q;
#pragma unroll
            for (int t = 0; t < NT; ++t) wv[u][t] = *reinterpret_cast<const f32x4*>(w[t] + k);
#pragma unroll
            for (int j = 0; j < MT; ++j) xv[u][j] = load_x(j, k);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) multiply(wv[u], xv[u]);
    }
    for (; c < c1; ++c) {  // what is left, and a chunk that K ends inside
        const int k = 16 * c + 4 * q, kc = min(k, K - 4);
        f32x4 wv[NT], xv[MT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            wv[t] = *reinterpret_cast<const f32x4*>(w[t] + kc);
            if (k >= K) wv[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            xv[j] = load_x(j, kc);
            if (k >= K) xv[j] = f32x4{0.f, 0.f, 0.f, 0.f};  // (0 times an infinity that lies elsewhere is no zero)
        }
        multiply(wv, xv);
    }
    if (wave > 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < MT; ++j) red[wave - 1][t * MT + j][lane] = acc[t][j];
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int m = m0 + 16 * j + r;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int w = 0; w < WAVES - 1; ++w) acc[t][j] += red[w][t * MT + j][lane];
        if constexpr (NORMED && EPI == EPI_PLAIN) {
            if (a.rope_on) {  // as qkv_rope_append_tiled_kernel; a pair's halves lie in lanes 16 apart
                const RopeRows& p = a.rope;
                const int h = p.nh * p.hd, b = min(m, a.M - 1) / p.S, sq = min(m, a.M - 1) - b * p.S, pos = (p.pos_dev ? *p.pos_dev : p.pos0) + sq;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int n = min(n0 + 4 * v + q, a.N - 1), sec = n >= 2 * h ? 2 : n >= h ? 1 : 0, col = n - sec * h, head = col / p.hd, d = col - head * p.hd;
                    float x = (float)acc[0][j][v];
                    if (sec < 2 && p.qk_bias) x += p.qk_bias[n];
                    const float other = __shfl_xor(x, 16, 64);
                    if (sec < 2) {
                        const float* f = p.freqs + ((int64_t)pos * (p.hd / 2) + d / 2) * 2;
                        float first = q & 1 ? other : x, second = q & 1 ? x : other;
                        rope_pair<float>(first, second, f[0], f[1]);
                        x = q & 1 ? second : first;
                    }
                    if (m >= a.M || n0 + 4 * v + q >= a.N) continue;
                    if (sec == 0) p.q_out[(int64_t)m * h + col] = x;
                    else if (pos < p.t_max) (sec == 1 ? p.k : p.v)[(((int64_t)b * p.nh + head) * p.t_max + pos) * p.hd + d] = x;
                }
                continue;
            }
        }
        if (m >= a.M) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {  // a lane holds weight rows 4 v + q of token row r
            const int n = n0 + 4 * v + q;
            if (n >= a.N) continue;
            if constexpr (EPI == EPI_SWIGLU) static_cast<float*>(a.y)[(int64_t)m * a.N + n] = swiglu<float>((float)acc[0][j][v], (float)acc[NT - 1][j][v]);
            else store_out<float, EPI>(a, m, n, (float)acc[0][j][v]);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// host dispatch
// ------------------------------------------------------------------------------------------------
static int n_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) cus = p.multiProcessorCount;
        if (cus <= 0) cus = 256;
    }
    return cus;
}

template <typename T, int MB, int EPI, bool NT, bool WIDE = false>
static int launch_gemv_nt(GemmArgs a, hipStream_t s) {
    const size_t lds = (size_t)MB * a.K * sizeof(T);
    RAVEN_REQUIRE(lds <= 160 * 1024, "gemm: %d rows x K=%d does not fit the 160 KB LDS", MB, a.K);
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)gemv_kernel<T, MB, EPI, NT, WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) {
            raven_host::set_error("gemm: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    const int n_units = (EPI == EPI_SWIGLU) ? a.N : (a.N + 1) / 2;
    // as few units per wave as keeps every workgroup resident at once
    const int max_wgs = n_cus() * (g_tuning.gemv_wgs_per_cu > 0 ? g_tuning.gemv_wgs_per_cu : 4);
    int upw = g_tuning.gemv_units_per_wave;
    if (upw <= 0) {
        upw = 1;
        while ((n_units + 4 * upw - 1) / (4 * upw) > max_wgs) ++upw;
    }
    a.units_per_wave = upw;
    a.interleave = g_tuning.gemv_interleave;
    const int wgs = (n_units + 4 * upw - 1) / (4 * upw);
    gemv_kernel<T, MB, EPI, NT, WIDE><<<dim3(wgs), dim3(256), lds, s>>>(a);
    return raven_host::check_launch("gemv");
}

template <typename T, int MB, int EPI>
static int launch_gemv(GemmArgs a, hipStream_t s) {
    return g_tuning.gemv_nontemporal ? launch_gemv_nt<T, MB, EPI, true>(a, s) : launch_gemv_nt<T, MB, EPI, false>(a, s);
}

// Up to 8 float rows against a matrix that stays in the caches: once K is long, two rows of W per wave of the whole chip are read faster than 16 per
// workgroup, also with 64-bit sums.  us, rows_f32_kernel / this: 2 rows, 512 x 256 3.7 / 3.9, 512 x 1024 5.5 / 4.5, 512 x 4096 15.4 / 9.8; 4 rows,
// 512 x 1024 5.6 / 5.9, 512 x 4096 15.6 / 13.4; 8 rows, 512 x 4096 15.8 / 24.7.  SwiGLU: 2 rows, 512 x 128 4.0 / 3.8, 512 x 2048 15.2 / 6.8; 4 rows,
// 512 x 256 4.8 / 4.8, 512 x 2048 15.2 / 8.8; 8 rows, 512 x 704 7.1 / 8.1, 512 x 2048 14.9 / 13.3.  (32-bit sums: 512 x 4096 at 2 rows 8.6.)
// Of 8192 and more rows of W a wave takes several in turn: SwiGLU of 8192 x 512 at 2 and 4 rows 7.2 / 6.6 and 7.2 / 9.4, 16384 x 128 at 2 rows 5.5 / 9.0.
static bool gemv_wide_pays(int M, int N, int K, bool swiglu) {
    const int longest_rows = M <= 2 ? (swiglu ? 64 : 256) : M <= 4 ? (swiglu ? 256 : 1024) : swiglu ? 768 : 1 << 30;
    return K > longest_rows && N * (swiglu ? 2 : 1) < 8192 && (size_t)(M <= 2 ? 2 : M <= 4 ? 4 : 8) * K * sizeof(float) <= 160 * 1024;
}
template <int EPI>
static int dispatch_gemv_wide(GemmArgs a, hipStream_t s) {
    a.ldy = a.N;
    if (a.M <= 2) return launch_gemv_nt<float, 2, EPI, false, true>(a, s);
    if (a.M <= 4) return launch_gemv_nt<float, 4, EPI, false, true>(a, s);
    return launch_gemv_nt<float, 8, EPI, false, true>(a, s);
}

template <typename T, int EPI>
static int dispatch_gemv(GemmArgs a, hipStream_t s) {
    if (a.M <= 1) return launch_gemv<T, 1, EPI>(a, s);
    if (a.M <= 2) return launch_gemv<T, 2, EPI>(a, s);
    if (a.M <= 4) return launch_gemv<T, 4, EPI>(a, s);
    return launch_gemv<T, 8, EPI>(a, s);
}

// Whether a matrix of up to 1024 tiles of 16 rows (from 17 token rows on 768; SwiGLU: 256 pairs) goes in one round of the chip: the fewest tiles per
// workgroup that give every CU at most one workgroup, of eight waves.  Four waves a tile leave a CU with one or two short workgroups, or a second
// round of them; with eight, and the partial sums added through LDS, the K slices of gemm_splitk.hip and their second launch are not needed
// either, up to the length of K where the workgroups become too long (splits_k there).  But eight waves of short rows do little else than
// start and add up, and with few rows of X the shorter workgroups of four waves lose nothing.  Time of one round over that of four waves, from 2 x 3600 products:
//   one tile    K of 256 1.03 - 1.07, 512 1.02 - 1.04, 640 0.92, 2048 0.85 - 0.98, 8192 0.68 - 0.97 (SwiGLU up to 16 rows 512 1.03, 640 0.94, 4096 0.88 - 0.96;
//               17 rows 0.92 - 1.01, 32 rows 0.97 - 1.04, where rows alternate between whole and half lines 17 to 32 rows 1.01 - 1.07)
//   two tiles   up to 8 rows 0.95 - 1.18; 16 rows: K of 1536 1.05 - 1.08, 2048 0.92, 2560 1.02, 4096 0.95 - 1.03, 5120 0.92; 24 rows: 1536 1.05, 2048 0.90, 5120 0.87; with 257 tiles
//               for 256 CUs, half of them without a workgroup, 1.0 - 1.27 up to 16 rows, K of 2048 1.01, 0.98 and 0.95 at 17, 24 and 32, of 2560 1.10 - 1.05; from 509 tiles on (four tiles per four-wave workgroup past
//               16 rows) 0.7 - 0.88 at 24 rows, whatever K
//   three tiles 2 rows: 512 1.1 - 1.27, 1536 1.15, 2048 0.91 - 0.99, 2560 1.05 - 1.11, 3072 0.98 - 1.01, 5120 0.93 - 0.98, 8192 0.8; 24 rows 0.83 - 1.0
//   four tiles  2 rows 1.0 - 1.17, but 0.91 at 4096; 16 rows: 512 1.09, 2048 1.05, 2560 1.0, 4096 0.9, 5120 0.97, 6144 1.1
// Sets of two steps ahead (two and three tiles) throw away half of the last one when a wave's number of steps is odd, which a fifth step shows most;
// rows of a power of two bytes from 8 KB on put all rows of a tile on the same channels, which more and shorter workgroups than here suffer from
// with four tiles and less with two; tiles whose
// rows alternate between whole and half lines (no pairs of tiles to sort them into) take 1.1 - 1.27 with two tiles and more.
template <bool SWIGLU>
static bool one_round_pays(const GemmArgs& a, int tiles) {
    const int n = a.N / 16, cus = n_cus(), steps = (a.K / 64 + 7) / 8;  // steps: of 64 columns, per wave
    if (tiles == 1) return a.K > 512 && (!SWIGLU || a.M <= 16 || (a.M <= 24 && a.line_aligned));
    if (SWIGLU) return false;  // two gate tiles and their up tiles: no faster than the four-wave kernels (14.4 / 14.1 at 12288 x 2048)
    const int rs = a.row_stride;
    if (a.M > 16 && (n + 4 * rs - 1) / (4 * rs) * rs >= cus / 2) return true;  // (else dispatch_mfma takes four tiles per four-wave workgroup)
    if (!a.line_aligned || steps < 4) return false;
    const int pitch = 2 * a.K;
    const bool one_channel = pitch >= 8192 && (pitch & (pitch - 1)) == 0;
    if (tiles == 2) {
        if (a.M > 16) return n >= cus + cus / 8 || steps >= 6 || (steps == 4 && a.K >= 1792 && a.M > 24);
        if (n < cus + cus / 8 || steps == 5 || one_channel) return false;
        return a.M >= 16 || (n <= cus + cus / 2 && (a.M >= 12 || (rs == 2 && steps >= 6)));
    }
    if (tiles == 3) return a.M > 16 || steps == 4 || steps >= (a.M < 8 ? 8 : 6);
    return one_channel || (a.M > 12 && steps >= 6 && pitch % 4096 != 0);
}

// us per launch before / after: 2048 x 2048 at 8 rows 6.1 / 5.5, at 20 rows 9.3 / 7.0; 8192 x 2048 at 20 rows 15.3 / 10.9; 10304 x 2048 12.0 / 11.2 and
// 15.4 / 12.6; 15840 x 5280 at 16 rows 32.6 / 30.1.  More loads in flight than two sets of 64 columns per wave gain nothing: a CU's own rate of loads is
// the bound.
template <int EPI, int MT, int NORM>
static bool launch_one_round(const GemmArgs& a, hipStream_t s) {
    constexpr int side = EPI == EPI_SWIGLU ? 2 : 1;
    const int rs = a.row_stride, n_tiles16 = a.N / 16;
    auto groups = [&](int ng) { return (n_tiles16 + ng * rs - 1) / (ng * rs) * rs; };
    if (!g_tuning.gemm_one_round || g_tuning.gemm_four_tiles == 2) return false;
    int tiles = 1;
    while (tiles < 5 && groups(tiles) > n_cus()) ++tiles;
    // two token tiles against four weight tiles do not fit the registers
    if (tiles > (EPI == EPI_SWIGLU ? 1 : MT == 1 ? 4 : 3) || (g_tuning.gemm_one_round == 1 && !one_round_pays<EPI == EPI_SWIGLU>(a, tiles))) return false;
    if (tiles == 1) {
        mfma_kernel<MT, side, EPI, 128, false, 8, 1, NORM><<<dim3(groups(1)), dim3(512), 0, s>>>(a);
    } else if constexpr (EPI != EPI_SWIGLU) {
        if (tiles == 2) mfma_kernel<MT, 2, EPI, 64, false, 8, 2, NORM><<<dim3(groups(2)), dim3(512), 0, s>>>(a);
        else if (tiles == 3) mfma_kernel<MT, 3, EPI, 64, false, 8, 2, NORM><<<dim3(groups(3)), dim3(512), 0, s>>>(a);
        else if constexpr (MT == 1) mfma_kernel<1, 4, EPI, 64, false, 8, 1, NORM><<<dim3(groups(4)), dim3(512), 0, s>>>(a);
    }
    return true;
}

template <int EPI>
static int reads_residual_early(const GemmArgs& a) {
    return EPI == EPI_FREE && a.epi.residual && a.epi.out_f32 && a.ldy % 4 == 0 && raven_host::aligned16(a.y, a.epi.residual, a.epi.bias);
}

template <int EPI, int NORM = kNormNone>
static int dispatch_mfma(GemmArgs a, hipStream_t s) {
    const int n_tiles16 = a.N / 16;
    a.early = reads_residual_early<EPI>(a);
    // rows alternate between line-aligned and 64 bytes off when the row pitch is an odd multiple of 64 bytes:
    // tiles of equal parity then (needs whole pairs of tiles); any multiple of 128 bytes needs nothing special
    const int pitch = a.K * 2;
    a.row_stride = (pitch % 128 == 64 && a.N % 32 == 0) ? 2 : 1;
    a.line_aligned = (pitch * a.row_stride) % 128 == 0;
    const int rs = a.row_stride;
    if (a.M <= 16 ? launch_one_round<EPI, 1, NORM>(a, s) : launch_one_round<EPI, 2, NORM>(a, s)) return raven_host::check_launch("mfma gemm");
    // Four tiles per workgroup (64-wide K steps) halve the X re-reads per weight byte: 5.0 -> 5.7 TB/s in steady state
    // at 32 rows.  Their workgroups are twice as long, so the gain only survives where the grid is balanced: at most
    // one workgroup per CU (Wqkv: 248), or so many that the last round does not matter.  Tuning key gemm_four_tiles:
    // 0 never, 1 by this rule, 2 whenever the shape allows.
    const int groups4 = (n_tiles16 + 4 * rs - 1) / (4 * rs) * rs;       // plain epilogue: 4 tiles side by side
    const int groups2 = (n_tiles16 + 2 * rs - 1) / (2 * rs) * rs;       // SwiGLU with 4 tiles: 2 gate + 2 up
    const int g4 = EPI == EPI_SWIGLU ? groups2 : groups4;
    const bool four = g_tuning.gemm_four_tiles == 2 ||
                      (g_tuning.gemm_four_tiles == 1 && a.M > 16 && g4 >= n_cus() / 2 && (g4 <= n_cus() || g4 >= 8 * n_cus()));
    if constexpr (EPI == EPI_SWIGLU) {
        // A matrix that divides into one workgroup per resident slot (two per CU) of 33..48 gate rows: three tile slots
        // per side, the last one partly empty -- one full round instead of a partly filled last one, and the X tile is
        // fetched once per 70 weight rows instead of once per 32.  mlp.fc of the 3.5b shape (17920 = 512 x 35), us per
        // launch against the whole-tile variants: 32 rows 67.7 / 79.1, 16 rows 60.2 / 66.2, 8 rows 58.9 / 61.7
        int rpu = 0;
        if (g_tuning.gemm_ragged)
            for (int r = 33; r <= 48 && !rpu; ++r)
                if (a.N % (r * rs) == 0 && a.N / r <= 2 * n_cus() && a.N / r >= 2 * n_cus() - n_cus() / 4) rpu = r;
        if (rpu) {
            a.rows_per_unit = rpu;
            if (a.M <= 16) mfma_kernel<1, 6, EPI, 64, true><<<dim3(a.N / rpu), dim3(256), 0, s>>>(a);
            else           mfma_kernel<2, 6, EPI, 64, true><<<dim3(a.N / rpu), dim3(256), 0, s>>>(a);
        } else if (four) {
            if (a.M <= 16) mfma_kernel<1, 4, EPI, 64><<<dim3(groups2), dim3(256), 0, s>>>(a);
            else           mfma_kernel<2, 4, EPI, 64><<<dim3(groups2), dim3(256), 0, s>>>(a);
        } else if (a.M <= 16)
            mfma_kernel<1, 2, EPI><<<dim3(n_tiles16), dim3(256), 0, s>>>(a);
        else
            mfma_kernel<2, 2, EPI><<<dim3(n_tiles16), dim3(256), 0, s>>>(a);
    } else if (four) {
        if (a.M <= 16) mfma_kernel<1, 4, EPI, 64, false, 4, 1, NORM><<<dim3(groups4), dim3(256), 0, s>>>(a);
        else           mfma_kernel<2, 4, EPI, 64, false, 4, 1, NORM><<<dim3(groups4), dim3(256), 0, s>>>(a);
    } else {
        // two tiles per workgroup (X is then re-read from L2 once per two tiles) while that still leaves every
        // CU more than one workgroup; L2 -> L1 traffic, not HBM, is what limits this kernel
        const bool two = n_tiles16 / 2 >= n_cus() + n_cus() / 2;
        const int units = two ? groups2 : n_tiles16;
        if (a.M <= 16) {
            if (two) mfma_kernel<1, 2, EPI, 128, false, 4, 1, NORM><<<dim3(units), dim3(256), 0, s>>>(a);
            else     mfma_kernel<1, 1, EPI, 128, false, 4, 1, NORM><<<dim3(units), dim3(256), 0, s>>>(a);
        } else {
            if (two) mfma_kernel<2, 2, EPI, 128, false, 4, 1, NORM><<<dim3(units), dim3(256), 0, s>>>(a);
            else     mfma_kernel<2, 1, EPI, 128, false, 4, 1, NORM><<<dim3(units), dim3(256), 0, s>>>(a);
        }
    }
    return raven_host::check_launch("mfma gemm");
}

// Float rows: all of them in one launch (per 4 194 240, what a grid holds).  A few rows against a matrix that does not fit the caches stay with
// the vector kernel, whose whole-row loads stream twice as fast (5.5 TB/s): up to 8 rows from 32 MB on.
template <int EPI, int MT>
static void launch_rows_f32_tiles(const GemmArgs& a, dim3 grid, hipStream_t s) {
    // Up to 256 columns a wave of four has one round of loads to wait for (SwiGLU: two matrices' worth, eight waves are faster from there on).  Where the grid is several
    // rounds long, four waves leave more of it resident (16384 x 704 at 200 rows, SwiGLU, 113 / 141 us), but long rows of X are read sooner by eight:
    // us by four / eight, 16 token rows a workgroup, SwiGLU of 1408 x 512 at 50 rows 9.9 / 8.1, of 2816 x 1024 at 200 58.7 / 52.7; 32, 1536 x 512 at 400 18.7 / 16.9;
    // 64, 8192 x 2048 at 100 87 / 80, 1408 x 5632 at 500 173 / 158, but 1536 x 512 at 400 20.1 / 21.2.
    const int64_t units = (int64_t)grid.x * grid.y, cus = n_cus();
    const bool eight = EPI == EPI_SWIGLU ? (MT == 1 ? a.K >= 256 : a.K > 256 && units <= 2 * cus)
                                         : a.K > 256 && (MT == 1 ? units <= cus : MT == 2 || units <= 2 * cus || a.K >= 1024);
    if (eight) rows_f32_kernel<EPI, MT, 8><<<grid, dim3(512), 0, s>>>(a);
    else rows_f32_kernel<EPI, MT, 4><<<grid, dim3(256), 0, s>>>(a);
}
// Token rows of a workgroup, in tiles of 16: the fewest that take the fewest rounds of work.  The 64-bit matrix instruction is the slow part (64 cycles for 16 x 16 x 4), so a small
// model's product over 16 to 90 workgroups of 64 token rows leaves the chip idle.  us, 64 / 16 rows a workgroup: 256 x 704 at 17 rows (32 then) 6.7 / 4.8, at 100 11.6 / 5.0;
// 768 x 256 at 50 6.1 / 3.2; 512 x 1408 at 100 18.3 / 7.6.  Past one round 16 rows cost a quarter more for the same work (weights and token rows are
// read, and widened, for fewer products): 1536 x 512 at 400 20.1 / 20.4, with 32 rows 16.9; 2048 x 2048 at 500 88 / 115.  Matrices past 32 MB, which the caches between the XCDs
// and memory would hand out once per row tile, keep as many rows as there are (8192 x 2048 at 40 rows 40 / 43).
static int rows_f32_tiles(int M, int N, int K, bool swiglu) {
    const int most = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    if ((int64_t)N * K * (swiglu ? 8 : 4) > (32 << 20)) return most;
    int best = most;
    double least = 0;
    for (int mt = most; mt >= 1; mt /= 2) {
        const int64_t units = (int64_t)((N + 15) / 16) * ((M + 16 * mt - 1) / (16 * mt)), rounds = (units + n_cus() - 1) / n_cus();
        const double work = (double)rounds * mt * (mt == 1 && rounds > 1 ? 1.25 : 1.0);
        if (mt == most || work < least) {
            best = mt;
            least = work;
        }
    }
    return best;
}
template <int EPI>
static int launch_rows_f32(GemmArgs a, hipStream_t s) {
    a.ldy = a.N;
    const int M = a.M, mt = rows_f32_tiles(M, a.N, a.K, EPI == EPI_SWIGLU), most = 65535 * 16 * mt;
    for (int m0 = 0; m0 < M; m0 += most) {
        a.M = M - m0 < most ? M - m0 : most;
        const dim3 grid((a.N + 15) / 16, (a.M + 16 * mt - 1) / (16 * mt));
        if (mt == 1) launch_rows_f32_tiles<EPI, 1>(a, grid, s);
        else if (mt == 2) launch_rows_f32_tiles<EPI, 2>(a, grid, s);
        else launch_rows_f32_tiles<EPI, 4>(a, grid, s);
        if (const int rc = raven_host::check_launch("gemm (fp32 rows)")) return rc;
        a.x0 = static_cast<const float*>(a.x0) + (size_t)a.M * a.k0;
        if (a.x1) a.x1 = static_cast<const float*>(a.x1) + (size_t)a.M * a.k1;
        if (a.residual) a.residual = static_cast<const float*>(a.residual) + (size_t)a.M * a.N;
        if (a.epi.residual) a.epi.residual += (size_t)a.M * a.N;
        a.y = static_cast<float*>(a.y) + (size_t)a.M * a.N;
        if (m0 > M - most) break;  // (the next start may not fit an int)
    }
    return 0;
}

// ---- float rows behind norms ----
// What rows_f32_fused takes: rows of up to 1024 columns that go to rows_f32_kernel, few enough that norming them in every workgroup is cheaper than a launch.  us of a whole
// prompt (four recurrences of two blocks; passes queued one after the other), launches of their own / this: width 256, 5 to 64 tokens 392 to 425 / 306 to 331, 100: 391 / 389, 400: 628 / 785;
// width 384, 33: 424 / 375, 64: 442 / 461; width 512, 17: 423 / 407, 33: 447 / 505.
static bool rows_f32_takes(int M, int N, int K, bool swiglu) {
    return M >= 2 && (M > 8 || (size_t)N * K * (swiglu ? 8 : 4) < (32u << 20)) && !(M <= 8 && gemv_wide_pays(M, N, K, swiglu));
}
constexpr int kNormedValues = 16384;
int g_f32_norm_rows = 64;  // raven_set_tuning("f32_norm_rows"): up to so many rows
static size_t rows_f32_fused_lds(int mt, int K0) { return (size_t)16 * mt * normed_pitch(K0) * sizeof(float); }
static int rows_f32_fused_tiles(int M, int N, int K, bool swiglu) { return std::min(rows_f32_tiles(M, N, K, swiglu), 2); }
bool rows_f32_fused_fits(int M, int N, int K0, int K1, bool swiglu) {
    if (M < 2 || M > g_f32_norm_rows || (int64_t)M * K0 > kNormedValues || K0 > kNormedColumns || K0 % 4 != 0 || K1 % 4 != 0 || !rows_f32_takes(M, N, K0 + K1, swiglu)) return false;
    return rows_f32_fused_lds(rows_f32_fused_tiles(M, N, K0 + K1, swiglu), K0) <= 80 * 1024;  // (the waves' sums take up to 57 KB more)
}
template <int EPI, int MT, int WAVES>
static int launch_rows_f32_fused(const NormedRows& a, hipStream_t s) {
    static bool attr_set = false;
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute((const void*)rows_f32_kernel<EPI, MT, WAVES, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (e != hipSuccess) {
            raven_host::set_error("gemm (fp32 rows): hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return (int)e;
        }
        attr_set = true;
    }
    rows_f32_kernel<EPI, MT, WAVES, true><<<dim3((a.N + 15) / 16, (a.M + 16 * MT - 1) / (16 * MT)), dim3(64 * WAVES), rows_f32_fused_lds(MT, a.k0), s>>>(a);
    return raven_host::check_launch("gemm (fp32 rows, norms)");
}
// raven_gemv_fused for 2 and more float rows that rows_f32_fused_fits takes: y = concat(norm_b(norm_a(x0)), x1) W^T, or the gated half of it; xa_out = norm_a(x0).  With one
// norm it is norm_a that is given, as there.  rope (may be null): see RopeRows; y is then not written.
int rows_f32_fused(const void* x0, const void* x1, const void* norm_a, const void* norm_b, void* xa_out, const void* w, void* y, int M, int N, int K0, int K1, float eps,
                   int swiglu, const RopeRows* rope, hipStream_t s) {
    RAVEN_REQUIRE(rows_f32_fused_fits(M, N, K0, K1, swiglu != 0) && norm_a && raven_host::aligned16(x0, x1, norm_a, norm_b, xa_out, w), "gemm (fp32 rows, norms): unsupported shape or operands");
    NormedRows a{};
    a.w = w; a.x0 = x0; a.x1 = x1; a.y = y;
    a.M = M; a.N = N; a.K = K0 + K1; a.k0 = K0; a.k1 = K1; a.ldy = N; a.eps = eps;
    a.norm_a = norm_b ? static_cast<const float*>(norm_a) : nullptr;
    a.norm_b = static_cast<const float*>(norm_b ? norm_b : norm_a);
    a.xa_out = norm_b ? static_cast<float*>(xa_out) : nullptr;
    if (rope) {
        a.rope = *rope;
        a.rope_on = 1;
    }
    const bool one = rows_f32_fused_tiles(M, N, a.K, swiglu != 0) == 1;
    if (swiglu) return one ? launch_rows_f32_fused<EPI_SWIGLU, 1, 8>(a, s) : launch_rows_f32_fused<EPI_SWIGLU, 2, 8>(a, s);
    return one ? launch_rows_f32_fused<EPI_PLAIN, 1, 8>(a, s) : launch_rows_f32_fused<EPI_PLAIN, 2, 8>(a, s);
}

// Runs one GEMM over all M rows, in passes of at most 32 (MFMA) or 8 / 4 (vector) rows.
template <int EPI>
static int run_gemm(GemmArgs a, int dtype, hipStream_t s) {
    const size_t es = raven_host::elt_size(dtype);
    const bool mfma_ok = dtype == RAVEN_BF16 && a.K % 32 == 0 && a.k0 % 32 == 0 && a.N % 16 == 0;
    const int M = a.M;
    const size_t out_es = a.out_f32 ? 4 : es;
    RAVEN_REQUIRE(dtype != RAVEN_F32 || (size_t)a.K * es <= 160 * 1024, "gemm: one row of K=%d elements does not fit the 160 KB LDS", a.K);
    if (dtype == RAVEN_F32 && rows_f32_takes(M, a.N, a.K, EPI == EPI_SWIGLU)) return launch_rows_f32<EPI>(a, s);
    if (dtype == RAVEN_F32 && M >= 2 && M <= 8 && (size_t)a.N * a.K * (EPI == EPI_SWIGLU ? 8 : 4) < (32u << 20)) return dispatch_gemv_wide<EPI>(a, s);
    for (int m0 = 0; m0 < M;) {
        const int left = M - m0;
        int pass;
        if (left == 1 && gemv1_fits(a.K, dtype)) {  // a single row: the K-split one-row kernel
            const char* x0 = static_cast<const char*>(a.x0) + (size_t)m0 * a.k0 * es;
            const char* x1 = a.x1 ? static_cast<const char*>(a.x1) + (size_t)m0 * a.k1 * es : nullptr;
            const char* res = a.residual ? static_cast<const char*>(a.residual) + (size_t)m0 * a.N * es : nullptr;
            char* y = static_cast<char*>(a.y) + (size_t)m0 * a.N * out_es;
            if (is_free(EPI)) {
                raven_epilogue e = a.epi;
                if (e.residual) e.residual += (size_t)m0 * a.N;
                return gemv1_free(x0, x1, a.w, y, a.N, a.k0, a.k1, e, dtype, s);
            }
            return raven_gemv_fused(x0, x1, nullptr, nullptr, nullptr, a.w, res, y, a.N, a.k0, a.k1, 0.f, EPI == EPI_SWIGLU, a.out_f32,
                                    dtype, s);
        }
        const bool use_mfma = mfma_ok && left >= g_tuning.gemm_mfma_min_rows;
        if (use_mfma) pass = left < 32 ? left : 32;
        else {
            pass = dtype == RAVEN_BF16 ? (left < 4 ? left : 4) : (left < 8 ? left : 8);
            // the vector kernel keeps its X rows in LDS: as many rows per pass (1, 2, 4 or 8) as fit
            const size_t row_bytes = (size_t)a.K * es;
            RAVEN_REQUIRE(row_bytes <= 160 * 1024, "gemm: one row of K=%d elements does not fit the 160 KB LDS", a.K);
            while (pass > 1 && (size_t)(pass <= 2 ? 2 : pass <= 4 ? 4 : 8) * row_bytes > 160 * 1024) pass = pass > 4 ? 4 : pass > 2 ? 2 : 1;
        }
        GemmArgs p = a;
        p.M = pass;
        p.x0 = static_cast<const char*>(a.x0) + (size_t)m0 * a.k0 * es;
        if (a.x1) p.x1 = static_cast<const char*>(a.x1) + (size_t)m0 * a.k1 * es;
        if (a.residual) p.residual = static_cast<const char*>(a.residual) + (size_t)m0 * a.N * es;
        p.y = static_cast<char*>(a.y) + (size_t)m0 * a.N * out_es;
        if (a.epi.residual) p.epi.residual = a.epi.residual + (size_t)m0 * a.N;
        int rc;
        if (use_mfma) rc = dispatch_mfma<EPI>(p, s);
        else if (dtype == RAVEN_BF16) rc = dispatch_gemv<bf16, EPI>(p, s);
        else rc = dispatch_gemv<float, EPI>(p, s);
        if (rc != 0) return rc;
        m0 += pass;
    }
    return 0;
}

// The skinny kernels with the free epilogue (raven_linear_epilogue, which has checked the arguments)
int gemm_free(const void* x0, const void* x1, const void* w, void* y, int M, int N, int K0, int K1, const raven_epilogue& epi, int dtype,
              hipStream_t s) {
    GemmArgs a{};
    a.w = w; a.x0 = x0; a.x1 = x1; a.y = y;
    a.M = M; a.N = N; a.K = K0 + K1; a.k0 = K0; a.k1 = K1; a.out_f32 = epi.out_f32; a.epi = epi; a.ldy = N;
    switch (EPI_FREE + epi.act) {
        case EPI_FREE_GELU: return run_gemm<EPI_FREE_GELU>(a, dtype, s);
        case EPI_FREE_TANH: return run_gemm<EPI_FREE_TANH>(a, dtype, s);
        default: return run_gemm<EPI_FREE>(a, dtype, s);
    }
}

bool gemm_free_normed_fits(int M, int N, int K) { return M >= g_tuning.gemm_mfma_min_rows && M <= 32 && N % 16 == 0 && K % 32 == 0; }
// One of two products of 2 to 32 rows with an RMSNorm between them, both of which gemm_free takes in one launch (epilogue_in_one_launch): y = x W^T + residual in float and
// what the norm needs of it, or a product of such rows
int gemm_free_normed(const void* x, const void* w, void* y, int M, int N, int K, const raven_epilogue& epi, const NormAhead* ahead, const NormBehind* behind,
                     hipStream_t s) {
    RAVEN_REQUIRE(gemm_free_normed_fits(M, N, K) && (ahead != nullptr) != (behind != nullptr) && epi.act != RAVEN_ACT_TANH &&
                      !(ahead && (epi.act != RAVEN_ACT_NONE || !epi.out_f32 || !epi.residual || epi.bias || !raven_host::aligned16(y, epi.residual, ahead->weight, ahead->xw))) && !(behind && behind->parts > kNormParts),
                  "gemm (norm between): unsupported shape M=%d N=%d K=%d", M, N, K);
    GemmArgs a{};
    a.w = w; a.x0 = x; a.y = y;
    a.M = M; a.N = N; a.K = K; a.k0 = K; a.out_f32 = epi.out_f32; a.epi = epi; a.ldy = N;
    if (ahead) {
        a.ahead = *ahead;
        return dispatch_mfma<EPI_FREE, kNormAhead>(a, s);
    }
    a.behind = *behind;
    return epi.act == RAVEN_ACT_GELU ? dispatch_mfma<EPI_FREE_GELU, kNormBehind>(a, s) : dispatch_mfma<EPI_FREE, kNormBehind>(a, s);
}

// Many rows against a matrix of at most 128 rows, where 128 x 128 tiles would leave most of the chip idle: 32 x 32 pieces of the output,
// K split over a workgroup's waves.  ldy: row pitch of y and the residual.
bool gemm_narrow_fits(int M, int N, int K, int dtype) {
    return dtype == RAVEN_BF16 && M > 128 && M <= 8192 && N <= 128 && N % 16 == 0 && K % 32 == 0 && K >= 256;
}
template <int EPI>
static int launch_narrow(GemmArgs a, hipStream_t s) {
    a.early = reads_residual_early<EPI>(a);
    const int pitch = a.K * 2, n_tiles16 = a.N / 16;
    a.row_stride = (pitch % 128 == 64 && a.N % 32 == 0) ? 2 : 1;
    a.line_aligned = (pitch * a.row_stride) % 128 == 0;
    const int rs = a.row_stride, groups = (n_tiles16 + 2 * rs - 1) / (2 * rs) * rs;
    mfma_kernel<2, 2, EPI><<<dim3(groups, (a.M + 31) / 32), dim3(256), 0, s>>>(a);
    return raven_host::check_launch("mfma gemm (narrow)");
}
int gemm_narrow_free(const void* x, const void* w, void* y, int ldy, int M, int N, int K, const raven_epilogue& epi, hipStream_t s) {
    GemmArgs a{};
    a.w = w; a.x0 = x; a.y = y;
    a.M = M; a.N = N; a.K = K; a.k0 = K; a.out_f32 = epi.out_f32; a.epi = epi; a.ldy = ldy;
    switch (EPI_FREE + epi.act) {
        case EPI_FREE_GELU: return launch_narrow<EPI_FREE_GELU>(a, s);
        case EPI_FREE_TANH: return launch_narrow<EPI_FREE_TANH>(a, s);
        default: return launch_narrow<EPI_FREE>(a, s);
    }
}

static int check_common(const char* who, int M, int N, int K, int dtype) {
    RAVEN_REQUIRE(dtype == RAVEN_F32 || dtype == RAVEN_BF16, "%s: unknown dtype %d", who, dtype);
    RAVEN_REQUIRE(M >= 0 && N > 0 && K > 0, "%s: bad shape M=%d N=%d K=%d", who, M, N, K);
    const int elts = 16 / (int)raven_host::elt_size(dtype);
    RAVEN_REQUIRE(K % elts == 0, "%s: K=%d must be a multiple of %d", who, K, elts);
    return 0;
}

}  // namespace raven

extern "C" int raven_gemm(const void* x, const void* w, const void* residual, void* y, int32_t M, int32_t N, int32_t K,
                          int32_t dtype, int32_t out_f32, void* stream) {
    using namespace raven;
    if (int rc = check_common("gemm", M, N, K, dtype)) return rc;
    if (M == 0) return 0;
    RAVEN_REQUIRE(x && w && y, "gemm: null pointer");
    if (M >= g_tiled_min_rows && tiled_gemm_fits(M, N, K, 0, dtype, 0, 0, raven_host::aligned16(x, w, residual, y)))
        return tiled_gemm(x, 0, nullptr, w, residual, y, M, N, K, 0, 0, out_f32, nullptr, 0, static_cast<hipStream_t>(stream), nullptr);
    GemmArgs a{};
    a.w = w; a.x0 = x; a.x1 = nullptr; a.residual = residual; a.y = y;
    a.M = M; a.N = N; a.K = K; a.k0 = K; a.k1 = 0; a.out_f32 = out_f32;
    return run_gemm<EPI_PLAIN>(a, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int raven_adapter_gemm_concat(const void* x0, const void* x1, const void* w, void* y, int32_t M, int32_t N,
                                         int32_t K0, int32_t K1, int32_t dtype, void* stream) {
    using namespace raven;
    if (int rc = check_common("adapter", M, N, K0 + K1, dtype)) return rc;
    if (M == 0) return 0;
    RAVEN_REQUIRE(x0 && x1 && w && y, "adapter: null pointer");
    const int elts = 16 / (int)raven_host::elt_size(dtype);
    RAVEN_REQUIRE(K0 > 0 && K1 > 0 && K0 % elts == 0 && K1 % elts == 0, "adapter: K0=%d, K1=%d must be positive multiples of %d", K0, K1, elts);
    if (M >= g_tiled_min_rows && tiled_gemm_fits(M, N, K0, K1, dtype, 0, 0, raven_host::aligned16(x0, x1, w, y)))
        return tiled_gemm(x0, 0, x1, w, nullptr, y, M, N, K0, K1, 0, 0, nullptr, 0, static_cast<hipStream_t>(stream), nullptr);
    GemmArgs a{};
    a.w = w; a.x0 = x0; a.x1 = x1; a.residual = nullptr; a.y = y;
    a.M = M; a.N = N; a.K = K0 + K1; a.k0 = K0; a.k1 = K1; a.out_f32 = 0;
    return run_gemm<EPI_PLAIN>(a, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int raven_gemm_swiglu(const void* x, const void* fc, void* out, int32_t M, int32_t I, int32_t K, int32_t dtype,
                                 void* stream) {
    using namespace raven;
    if (int rc = check_common("gemm_swiglu", M, I, K, dtype)) return rc;
    if (M == 0) return 0;
    RAVEN_REQUIRE(x && fc && out, "gemm_swiglu: null pointer");
    if (M >= g_tiled_min_rows && tiled_gemm_fits(M, I, K, 0, dtype, 1, 0, raven_host::aligned16(x, fc, out)))
        return tiled_gemm(x, 0, nullptr, fc, nullptr, out, M, I, K, 0, 1, 0, nullptr, 0, static_cast<hipStream_t>(stream), nullptr);
    GemmArgs a{};
    a.w = fc; a.x0 = x; a.x1 = nullptr; a.residual = nullptr; a.y = out;
    a.M = M; a.N = I; a.K = K; a.k0 = K; a.k1 = 0; a.out_f32 = 0;
    return run_gemm<EPI_SWIGLU>(a, dtype, static_cast<hipStream_t>(stream));
}
