// What the matrix-core products over many token rows share (gemm_tiled.hip, gemm_mid.hip).
#pragma once

#include <type_traits>
#include <utility>

#include "raven_common.h"

namespace raven {

// A chunk's fused q | k | v product (3 * nh * hd columns) may leave through this epilogue instead of y: it adds the q / k bias, rotates
// q and k (RoPE on adjacent pairs) and writes q to q_out and k, v to their cache rows -- what qkv_rope_append_tiled_kernel
// (attention.hip) does to a stored product, with the same functions in the same order.
struct RopeAppend {
    const float* freqs;
    const bf16* qk_bias;   // [2, nh * hd] or null
    bf16* q_out;           // [M, nh * hd]
    bf16 *k, *v;           // cache tensors, [.., batch, nh, t_max, hd] from slot_off on
    int64_t slot_off;
    const int* pos_dev;    // position of a sequence's first row, on the device (or null: pos0)
    int nh, hd, t_max, S, pos0;
    int col0;              // column of the whole product that this launch's column 0 is
};

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, static_cast<F&&>(f));
}

// One product as the host side of both files passes it on
struct ProductArgs {
    const bf16* w;         // [N or 2N, K0 + K1], rows ldw apart
    const bf16* x0;        // [M, K0], rows ldx apart
    const bf16* x1;        // [M, K1] or null, rows ldx apart
    const bf16* residual;  // [M, N] or null, rows ldy apart
    void* y;               // [M, N] bf16, or float when out_f32, rows ldy apart
    int M, N, K0, K1, ldw, ldx;
    int ldy;               // elements between two rows of y and of the residuals
    int up_off;            // SwiGLU: weight rows from a gate row to its up row
    int swiglu, out_f32;
    const raven_epilogue* epi;   // free epilogue, or null
    const RopeAppend* rope;      // or null
};

// Products of row groups with a weight matrix each: tile row t multiplies rows group_row[t] .. group_end[t] - 1 (at most tile_rows of them)
// with the matrix of group group_of[t].  The first *used entries are tiles; a launch is sized for n_tiles, and its workgroups share the used
// ones out over the XCDs (shared out by n_tiles, a fifth of the chip idled behind the unused ones of a 4096-token chunk)
struct RowGroups {
    const int *group_of, *group_row, *group_end, *used;
    int n_tiles, tile_rows;
    const int* x_row;        // row of x behind a row of the product, or null: the same
    const float* x_scale;    // SwiGLU: factor of a row of x, applied to its sums
    int64_t w_stride;        // elements between two groups' matrices
    const bf16* w_extra;     // matrix of group extra_group (-1: none), which lies elsewhere
    int extra_group;
};

// gemm_mid.hip: how a product over a middling number of rows is cut (0 units: not one for that kernel)
struct MidPlan {
    int nt, mt;            // 16-row tiles of a wave along the weight rows / the token rows
    int cols;              // output columns of a unit
    int rows;              // token rows of a unit
    int tiles_m, tiles_n, ks;
    float us;              // the estimate it was chosen by
};
MidPlan mid_plan(int M, int N, int K0, int K1, int swiglu, size_t room, int ks_from = 1);  // room: bytes of workspace for K slices, ks_from of them or more
struct MidParts {
    int ks;                // 0: none
    float us;
};
MidParts mid_float_parts(int M, int N, int K, size_t room);  // the fewest slices of 33 and more rows of sums that leave unrounded
size_t mid_workspace_bytes(int M, int N, const MidPlan& p, int swiglu);  // 0 when K is not split
// ks_left (may be null): the K slices stay in the workspace ([slices, M, N] float) for the caller to add; receives their number, 0
// when the product was finished
int mid_gemm(const ProductArgs& a, const MidPlan& p, void* workspace, hipStream_t s, int* ks_left);
// y[r] = x[x_row[r]] W_g^T, W_g [N or 2N, K] the matrix of row r's group.  swiglu: y = T(silu(s gate) * (s up)) with s = x_scale[r]; else
// y = the sums, as T or (out_f32) as they are.  tile_rows 32 or 64; rows: rows of the product, x_rows: rows of x.
int mid_grouped(const void* x, int x_rows, const void* w, void* y, int rows, int N, int K, int swiglu, int out_f32, const RowGroups& g, hipStream_t s);

}  // namespace raven
