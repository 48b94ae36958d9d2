// Chunk tiles and MFMA operands as bf16 planes (tt_planes.h), for the tree
// gated-delta-rule kernels: v_mfma_f32_16x16x32_bf16, operands from LDS planes,
// from accumulators or from global rows.
#pragma once

#include "tt_gdn_common.h"
#include "tt_planes.h"

namespace {

// bf16 planes of a chunk's tiles in LDS, rows = tokens. A tile read by rows
// (16 rows x 16 bytes a pass) has rows of 272 bytes (A: 80), one read by
// columns through the transposing read (8 rows x 32 bytes) rows of 288 (96):
// both reach every bank once a pass.
constexpr int PR = GD + 8, PC = GD + 16;   // [token][state row] tiles
constexpr int AR = GC + 8, AC = GC + 16;   // [token][token]
// The same without padding: the 16-byte pieces of a row exchanged by its number
// (rows that one read covers, and the writes, still reach every bank once a
// pass). PRS for tiles read by rows, PCS by columns.
constexpr int PRS = GD, PCS = -GD;
constexpr int row_elems(int P) { return P < 0 ? -P : P; }
constexpr bool swapped(int P) { return P == PRS || P == PCS; }
// Element (row, d) of such a tile.
template <int P>
__device__ __forceinline__ int tile_at(int row, int d) {
    const int x = P == PRS ? row & 15 : (2 * (row & 7)) ^ (row & 1);
    return row * GD + (((d >> 3) ^ x) << 3) + (d & 7);
}
template <typename TIn>
constexpr int kInPlanes = sizeof(TIn) == 2 ? 1 : 3;

__device__ __forceinline__ f32x4 mfma16b(const bf16x8& a, const bf16x8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// An operand of N planes (h, m, l).
template <int N>
struct Op {
    bf16x8 p[N];
};
// acc + A B, the smallest terms first.
template <int NA, int NB>
__device__ __forceinline__ f32x4 mul_planes(const Op<NA>& a, const Op<NB>& b, f32x4 acc) {
    if constexpr (NA == 3) acc = mfma16b(a.p[2], b.p[0], acc);
    if constexpr (NB == 3) acc = mfma16b(a.p[0], b.p[2], acc);
    if constexpr (NA == 3 && NB == 3) acc = mfma16b(a.p[1], b.p[1], acc);
    if constexpr (NA == 3) acc = mfma16b(a.p[1], b.p[0], acc);
    if constexpr (NB == 3) acc = mfma16b(a.p[0], b.p[1], acc);
    return mfma16b(a.p[0], b.p[0], acc);
}
// The same over a longer contraction: h h in one sum and the smaller terms in
// another (added at the end), so that only the large ones round at the size of
// the result.
struct Sum2 {
    f32x4 big = {}, small = {};
    template <int NA, int NB>
    __device__ __forceinline__ void add(const Op<NA>& a, const Op<NB>& b) {
        if constexpr (NA == 3) small = mfma16b(a.p[2], b.p[0], small);
        big = mfma16b(a.p[0], b.p[0], big);
        if constexpr (NB == 3) small = mfma16b(a.p[0], b.p[2], small);
        if constexpr (NA == 3 && NB == 3) small = mfma16b(a.p[1], b.p[1], small);
        if constexpr (NA == 3) small = mfma16b(a.p[1], b.p[0], small);
        if constexpr (NB == 3) small = mfma16b(a.p[0], b.p[1], small);
    }
    __device__ __forceinline__ f32x4 sum() const { return big + small; }
};
// The bf16 MFMA aligns its 16 products to the largest and drops the bits below
// towards minus infinity: a bias of one sign, far below one rounding, but one
// that a sum over thousands of tokens (the conv's weight gradient) collects.
// Results whose rows are tokens are therefore formed negated in the odd rows
// (the A operand's rows times alt(row)) and taken back negated: the bias
// alternates from token to token and cancels in such sums.
__device__ __forceinline__ float alt(int row) { return row & 1 ? -1.0f : 1.0f; }
__device__ __forceinline__ void add_alt(f32x4& acc, const f32x4& x) {   // rows 4 (l >> 4) + v
    acc[0] += x[0];
    acc[1] -= x[1];
    acc[2] += x[2];
    acc[3] -= x[3];
}
// Two 16-row accumulator tiles (rows 4 (l >> 4) + v) as the operand of a
// 32-deep contraction: element e of lane l is row 4 (l >> 4) + (e & 3) of tile
// e / 4, the k order of every operand here.
__device__ __forceinline__ Op<3> op_acc(const f32x4& t0, const f32x4& t1) {
    Split8 w = split_begin(t0, t1);
    w.all();
    const Planes q = w.planes();
    return {{q.h, q.m, q.l}};
}
// Row operand X[row][k0 + k] of a tile with rows of P elements (N planes, each
// [GC][P]), g4 = 4 (l >> 4).
template <int N, int P>
__device__ __forceinline__ Op<N> op_rows(const __bf16* X, int row, int k0, int g4) {
    Op<N> o;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        if constexpr (swapped(P)) {
            const __bf16* x = X + n * GC * GD;
            o.p[n] = cat44(*(const bf16x4*)(x + tile_at<P>(row, k0 + g4)), *(const bf16x4*)(x + tile_at<P>(row, k0 + 16 + g4)));
        } else {
            const __bf16* x = X + n * GC * P + row * P + k0 + g4;
            o.p[n] = cat44(*(const bf16x4*)x, *(const bf16x4*)(x + 16));
        }
    }
    return o;
}
// Column operand X[k][c0 + (l & 15)], k over the tile's 32 tokens.
template <int N, int P>
__device__ __forceinline__ Op<N> op_cols(const __bf16* X, int c0, int lane) {
    const int j = lane & 15;
    Op<N> o;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        if constexpr (swapped(P)) {
            const __bf16* x = X + n * GC * GD + tile_at<P>(4 * (lane >> 4) + (j >> 2), c0 + 4 * (j & 3));
            o.p[n] = cat44(ds_read_tr(x), ds_read_tr(x + 16 * GD));
        } else {
            const __bf16* x = X + n * GC * P + (4 * (lane >> 4) + (j >> 2)) * P + c0 + 4 * (j & 3);
            o.p[n] = cat44(ds_read_tr(x), ds_read_tr(x + 16 * P));
        }
    }
    return o;
}

// 16 consecutive elements of row i at column d0 as planes of a tile with rows of P elements.
template <int P>
__device__ __forceinline__ void put16(__bf16* X, int i, int d0, const bf16x8 (&x)[2]) {
    *(bf16x8*)(X + i * P + d0) = x[0];
    *(bf16x8*)(X + i * P + d0 + 8) = x[1];
}
template <int P>
__device__ __forceinline__ void put16(__bf16* X, int i, int d0, const f32x4 (&x)[4]) {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        Split8 w = split_begin(x[2 * n], x[2 * n + 1]);
        w.all();
        const Planes q = w.planes();
        __bf16* d;
        if constexpr (swapped(P)) d = X + tile_at<P>(i, d0 + 8 * n);
        else d = X + i * P + d0 + 8 * n;
        *(bf16x8*)d = q.h;
        *(bf16x8*)(d + GC * row_elems(P)) = q.m;
        *(bf16x8*)(d + 2 * GC * row_elems(P)) = q.l;
    }
}
// 1 / sqrt(|row|^2 + eps) (1 without the l2 norm) of the row whose 128
// elements this thread and its seven neighbours hold.
template <int NV, typename Vec>
__device__ __forceinline__ float row_norm(const GdnDev& p, const Vec (&x)[NV]) {
    constexpr int EV = 16 / NV;
    float s = 0.0f;
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int e = 0; e < EV; ++e) s = fmaf((float)x[n][e], (float)x[n][e], s);
    s = row8_sum(s);
    return p.l2 ? 1.0f / sqrtf(s + 1e-6f) : 1.0f;
}

// Accumulator-layout values in the problem dtype (dO) as an operand: its bf16 values as they are, or three planes.
template <typename TIn>
__device__ __forceinline__ Op<kInPlanes<TIn>> op_in(const f32x4& t0, const f32x4& t1) {
    if constexpr (kInPlanes<TIn> == 1)
        return {{pack8(t0[0], t0[1], t0[2], t0[3], t1[0], t1[1], t1[2], t1[3])}};
    else
        return op_acc(t0, t1);
}

// A row of the problem dtype as an operand: columns k0 + g4 .. +3 and
// k0 + 16 + g4 .. +3 (zeros when the row does not exist).
template <typename TIn>
__device__ __forceinline__ Op<kInPlanes<TIn>> op_global(const TIn* row, bool in, int k0, int g4) {
    if constexpr (kInPlanes<TIn> == 1) {
        const bf16x4 z = {};
        return {{cat44(in ? *(const bf16x4*)(row + k0 + g4) : z, in ? *(const bf16x4*)(row + k0 + 16 + g4) : z)}};
    } else {
        const f32x4 z = {};
        return op_acc(in ? load4(row + k0 + g4) : z, in ? load4(row + k0 + 16 + g4) : z);
    }
}
// A [32 x 32] accumulator quadrant into planes with rows of P elements.
template <int P>
__device__ __forceinline__ void put_quadrant(__bf16* X, int row, int colj, const f32x4& x) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        float r = x[v];
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            const __bf16 b = (__bf16)r;
            X[n * GC * P + (row + v) * P + colj] = b;
            r -= (float)b;
        }
    }
}
__device__ __forceinline__ float sum16(float x) {   // over the 16 lanes of a row of accumulators
    x += __shfl_xor(x, 1);
    x += __shfl_xor(x, 2);
    x += __shfl_xor(x, 4);
    return x + __shfl_xor(x, 8);
}

}  // namespace
