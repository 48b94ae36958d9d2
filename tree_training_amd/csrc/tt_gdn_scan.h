// Level scans of the tree gated delta rule: the forward scan of the states and
// the reverse scan of their gradients, per (node, v head), one launch per tree
// level (tt_gdn.hip has the equations).
//
// The products run on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16) on
// operands split into bf16 planes (tt_planes.h): W, A, V', dV' and the states
// into three, q, k and dO as they come (one plane for bf16 problems, exact;
// three for fp32), with the l2 norms and decays as per-token factors on the
// other operand or on the result. A 16-column slice of a chunk takes a wave
// 108 MFMAs of 16 cycles forward and 102 reverse (bf16 problems) where
// v_mfma_f32_16x16x4_f32 took 208 and 200 of 32. On the 16K agent tree (32 v
// heads, bf16) the column-layout levels went 867 -> 600 us forward and 1098 ->
// 830 reverse, the row-layout ones 164 -> 140 and 256 -> 228. Neither the pipes
// nor memory are full now (column levels: MFMA 12 and 8 % busy, 4.0 and 2.6 TB/s
// of a copy's 6.2): a level is a chain of chunks, two barriers each, at two waves a
// SIMD.
//
// fp32 problems hold q and k as three planes too. The forward's tiles are packed
// for two workgroups a CU (kScanPacked), the reverse ones and the truncated
// rule's (88 to 104 KB) leave one. 16,318 tokens, 32 v heads, exact rule: forward
// 1,311 us on fp32 MFMAs, 1,419 on padded tiles, 1,247 packed; forward and
// backward 5.59 -> 5.25 ms. Trees of one or two chunks a node pay the splits once a
// launch (47 tokens: 22.2 -> 22.8 us forward, 66.6 -> 64.0 backward).
#pragma once

#include "tt_gdn_planes.h"

namespace {

// A chunk's scan inputs, held in registers one chunk ahead of their use (the
// loads of the next chunk are in flight while a chunk computes): this
// thread's share of the q and k rows (row t/8, dims 16 (t%8) .. +15, in the
// problem dtype) and of W's rows, four entries of A (row t/8, columns
// 4 (t%8) ..) and the decays, and this lane's 16 x 16 tiles of U (forward) or
// dO (reverse).
template <typename TIn>
struct ScanAhead {
    using Vec = typename std::conditional<sizeof(TIn) == 2, bf16x8, f32x4>::type;
    static constexpr int NV = 16 * (int)sizeof(TIn) / 16;   // vectors per 16 elements
    Vec q[NV], k[NV];
    f32x4 w[4];
    f32x4 a;
    float gi, gl, gil, gll;   // G_i, G_L; their low parts
    f32x4 x[2];
};

// Loads the parts of chunk (start, len) that do not depend on the state: q/k
// rows, W rows, A and the decays from its workspace slot cw.
template <typename TIn>
__device__ __forceinline__ void scan_fetch_rows(const GdnDev& p, const float* cw, int start, int len, int h,
                                                ScanAhead<TIn>& x) {
    using Vec = typename ScanAhead<TIn>::Vec;
    constexpr int NV = ScanAhead<TIn>::NV, EV = 16 / NV;
    const int t = threadIdx.x, i = t >> 3, d0 = 16 * (t & 7), hk = h / p.rep;
    if (i < len) {
        const int64_t tok = start + i;
        const TIn* qp = (const TIn*)p.q + tok * p.q_st + (int64_t)hk * p.q_sh + d0;
        const TIn* kp = (const TIn*)p.k + tok * p.k_st + (int64_t)hk * p.k_sh + d0;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            x.q[n] = *(const Vec*)(qp + EV * n);
            x.k[n] = *(const Vec*)(kp + EV * n);
        }
    } else {
#pragma unroll
        for (int n = 0; n < NV; ++n) {
#pragma unroll
            for (int e = 0; e < EV; ++e) x.q[n][e] = x.k[n][e] = (TIn)0.0f;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) x.w[e] = *(const f32x4*)(cw + kWsW + i * GD + d0 + 4 * e);
    x.a = *(const f32x4*)(cw + kWsA + i * GC + 4 * (t & 7));
    x.gi = cw[kWsG + i];
    x.gl = cw[kWsG + GC - 1];
    x.gil = cw[kWsGlo + i];
    x.gll = cw[kWsGlo + GC - 1];
}

// x times alt(i) (bf16 values: the sign bits).
__device__ __forceinline__ void alt_row(bf16x8 (&x)[2], int i) {
    const unsigned m = i & 1 ? 0x80008000u : 0u;
#pragma unroll
    for (int n = 0; n < 2; ++n) x[n] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, x[n]) ^ (u32x4){m, m, m, m});
}
__device__ __forceinline__ void alt_row(f32x4 (&x)[4], int i) {
#pragma unroll
    for (int n = 0; n < 4; ++n) x[n] *= alt(i);
}

// A fetched chunk in LDS: q, k, W and A as planes with rows of
// PQ, PK, PW and PA elements, and the per-token factors fq = scale e^{G_i} /
// |q_i| and fk = e^{G_L - G_i} / |k_i|. ALT (the reverse scan): rows i of k and
// columns i of A times alt(i), so that dV' comes out times alt of its token.
template <typename TIn, int PQ, int PK, int PW, int PA, bool ALT>
struct ScanTiles {
    static constexpr int NQ = kInPlanes<TIn>;
    __bf16 Q[NQ * GC * row_elems(PQ)];
    __bf16 K[NQ * GC * row_elems(PK)];
    __bf16 W[3 * GC * row_elems(PW)];
    __bf16 A[3 * GC * PA];
    float fq[GC], fk[GC];
    float el;   // e^{G_L}
    __device__ __forceinline__ void stage(const GdnDev& p, const ScanAhead<TIn>& x) {
        const int t = threadIdx.x, i = t >> 3, d0 = 16 * (t & 7);
        put16<PQ>(Q, i, d0, x.q);
        if constexpr (ALT) {
            typename ScanAhead<TIn>::Vec k[ScanAhead<TIn>::NV];
#pragma unroll
            for (int n = 0; n < ScanAhead<TIn>::NV; ++n) k[n] = x.k[n];
            alt_row(k, i);
            put16<PK>(K, i, d0, k);
        } else {
            put16<PK>(K, i, d0, x.k);
        }
        put16<PW>(W, i, d0, x.w);
        {
            float a0 = x.a[0], a1 = ALT ? -x.a[1] : x.a[1], a2 = x.a[2], a3 = ALT ? -x.a[3] : x.a[3];
            __bf16* d = A + i * PA + 4 * (t & 7);
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                const uint32_t u0 = pack_bf16(a0, a1), u1 = pack_bf16(a2, a3);
                *(u32x2*)(d + n * GC * PA) = (u32x2){u0, u1};
                sub_bf16(u0, a0, a1);
                sub_bf16(u1, a2, a3);
            }
        }
        const float nq = row_norm(p, x.q), nk = row_norm(p, x.k);
        if ((t & 7) == 0) {
            fq[i] = nq * p.scale * expf(x.gi);
            fk[i] = nk * expf(gdiff(x.gl, x.gll, x.gi, x.gil));
            if (t == 0) el = expf(x.gl);
        }
    }
};
// fp32, exact rule: the forward's tiles without padding, 82 KB a workgroup instead
// of 88 (rows: 104), so that two share a CU. The column layout takes them for
// levels of more than a workgroup a CU (launch_scan).
template <typename TIn, bool TRUNC>
constexpr bool kScanPacked = kInPlanes<TIn> == 3 && !TRUNC;
template <typename TIn, int P = PR, int C = PC>
using FwdTiles = ScanTiles<TIn, P, C, P, AR, false>;   // q, W and A by rows, k by columns
template <typename TIn>
using RevTiles = ScanTiles<TIn, PC, PR, PC, AC, true>;   // k by rows, q, W and A by columns

// S e + x: the products of an update are summed apart and join the state with
// one rounding.
__device__ __forceinline__ f32x4 fma_tile(const f32x4& S, float e, const f32x4& x) {
    f32x4 r;
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = fmaf(S[v], e, x[v]);
    return r;
}
// x times the factors of tokens tok0 .. tok0 + 3, rounded (never fused into a
// sum: both layouts must round alike).
__device__ __forceinline__ f32x4 scale_tok(const f32x4& x, const float* f, int tok0) {
#pragma clang fp contract(off)
    const f32x4 s = *(const f32x4*)(f + tok0);
    return x * s;
}
// O of the same tokens: fq (q S) + A V'.
__device__ __forceinline__ f32x4 out_tok(const f32x4& qs, const float* fq, int tok0, const f32x4& av) {
    const f32x4 s = *(const f32x4*)(fq + tok0);
    f32x4 o;
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = fmaf(qs[v], s[v], av[v]);
    return o;
}

// Column layout of the level scans. The value columns of the delta rule are
// independent (column j of V', O and S depends only on column j of U, S and
// V'); each wave owns 16 of them (16 x 16 accumulator tiles), and a (node,
// v head) takes two workgroups of four waves (64 columns each) on different
// CUs. A level with few nodes is a serial chain of chunks per node while most
// CUs idle, and each chunk then runs on twice the MFMA pipes of one
// workgroup. Workgroup x of a level launch takes a head and a column block;
// with Hv a multiple of 8 the two blocks of a head are 8 apart (same XCD and
// L2, dispatched together).
constexpr int SCAN_COLS = 64;
constexpr int kScanSplit = GD / SCAN_COLS;
__device__ __forceinline__ void scan_block(const GdnDev& p, int& h, int& c0) {
    const int bx = blockIdx.x;
    int cs;
    if ((p.hv & 7) == 0) {
        h = ((bx >> 4) << 3) | (bx & 7);
        cs = (bx >> 3) & 1;
    } else {
        h = bx >> 1;
        cs = bx & 1;
    }
    c0 = SCAN_COLS * cs;
}

// Start of a node's forward scan: its parent's final state (a root's: the
// initial state, or none).
struct ScanNode {
    int node, start, len, chunk0, n_ch;
    const float* s0;
    __device__ __forceinline__ bool init(const GdnDev& p, int lvl_begin) {
        node = p.level_nodes[lvl_begin + blockIdx.y];
        if (node < 0 || node >= p.n_nodes) return false;
        start = p.node_start[node];
        len = p.node_len[node];
        chunk0 = p.node_chunk0[node];
        if (start < 0 || len < 0 || start > p.n_tokens - len) return false;        // malformed node: skipped
        n_ch = tt_cdiv(len, GC);
        return chunk0 >= 0 && chunk0 <= p.n_chunks - n_ch;
    }
    __device__ __forceinline__ const float* state0(const GdnDev& p, const float* states, int h) const {
        int par = p.parent[node];
        if (par >= node || par < -1) par = -1;                                     // parents precede children
        return par >= 0 ? states + ((size_t)par * p.hv + h) * GD * GD
                        : (p.init ? p.init + (size_t)h * GD * GD : nullptr);
    }
};

// Wave w owns value columns c0 + 16w .. +15 of one (node, v head): its
// 128 x 16 state slice lives in eight 16 x 16 accumulator tiles (rows
// 16 rb + 4 (l >> 4) + v) for the whole node, split into planes once a chunk.
// Per chunk (two 16-token tiles):
//   V' = U - W S,  qS  (A = W / q rows from LDS, B = S from registers)
//   O = fq qS + A V'  (B = V' from registers)
//   S <- e^{G_L} S + k^T (fk V')  (A = k from LDS, B = fk V')
// out may be null (the backward's recompute); chunk_sin / chunk_vp, when
// given, receive each chunk's initial state and V' ([n_chunks, Hv, 128, 128]
// and [n_chunks, Hv, 32, 128] floats).
// TRUNC (the reference's per-node correction): V' = U - W S0 with S0 the
// node's initial state, whose planes stay in registers, for every chunk.
template <typename TIn, bool TRUNC, bool packed>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_scan_cols_kernel(GdnDev p, int lvl_begin, float* __restrict__ ws,
                                                      TIn* __restrict__ out, float* __restrict__ states,
                                                      float* __restrict__ chunk_sin, float* __restrict__ chunk_vp) {
    constexpr int NQ = kInPlanes<TIn>;
    constexpr int P = packed ? PRS : PR, C = packed ? PCS : PC;
    __shared__ __attribute__((aligned(16))) FwdTiles<TIn, P, C> L;
    ScanNode nd;
    if (!nd.init(p, lvl_begin)) return;
    int h, cb;
    scan_block(p, h, cb);
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, c16 = lane & 15, g4 = 4 * (lane >> 4);
    const int jt = cb + 16 * wave, j = jt + c16;                          // the wave's first and this lane's column
    const int start = nd.start, len = nd.len, chunk0 = nd.chunk0, n_ch = nd.n_ch;
    const float* s0 = nd.state0(p, states, h);
    f32x4 S[8];
    if (s0) {
#pragma unroll
        for (int rb = 0; rb < 8; ++rb) S[rb] = load_t16(s0 + jt + 16 * rb * GD, lane);
    } else {
#pragma unroll
        for (int rb = 0; rb < 8; ++rb) S[rb] = (f32x4){};
    }

    Op<3> s0p[4];   // TRUNC
    if constexpr (TRUNC) {
#pragma unroll
        for (int w4 = 0; w4 < 4; ++w4) s0p[w4] = op_acc(S[2 * w4], S[2 * w4 + 1]);
    }

    // U and the state-independent chunk terms, one chunk ahead.
    ScanAhead<TIn> nx;
    auto fetch = [&](int ci) {
        const float* cw = ws + ((size_t)(chunk0 + ci) * p.hv + h) * kWsChunk;
        scan_fetch_rows<TIn>(p, cw, start + GC * ci, min(GC, len - GC * ci), h, nx);
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) nx.x[tb] = load_t16(cw + kWsU + 16 * tb * GD + jt, lane);
    };
    if (n_ch > 0) fetch(0);
    for (int ci = 0; ci < n_ch; ++ci) {
        const int c0 = GC * ci, Lc = min(GC, len - c0);
        const size_t ch = (size_t)(chunk0 + ci) * p.hv + h;
        if (chunk_sin) {
            float* sp = chunk_sin + ch * GD * GD + jt;
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) store_t16(sp + 16 * rb * GD, lane, S[rb]);
        }
        lds_barrier();   // readers of the previous chunk's tiles are done
        L.stage(p, nx);
        f32x4 vp[2] = {nx.x[0], nx.x[1]}, qs[2] = {};
        if (ci + 1 < n_ch) fetch(ci + 1);
        lds_barrier();

        // packed: the operands' LDS offsets are formed once a chunk, and their
        // reads stay with their products (held across, they spill)
        int lo = lane;
        if constexpr (packed) asm volatile("" : "+v"(lo));
        const int lane = lo, c16 = lane & 15, g4 = 4 * (lane >> 4);

        // V' = U - W S and q S over the 128 state rows as four partial sums
        // added in order: the partition of the row layout's waves
        // (gdn_scan_rows_kernel), so both layouts give the same bits.
#pragma unroll
        for (int w4 = 0; w4 < 4; ++w4) {
            if constexpr (packed) __builtin_amdgcn_sched_barrier(0);
            const Op<3> sp = op_acc(S[2 * w4], S[2 * w4 + 1]);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                vp[tb] -= mul_planes(op_rows<3, P>(L.W, 16 * tb + c16, 32 * w4, g4), TRUNC ? s0p[w4] : sp, (f32x4){});
                qs[tb] += mul_planes(op_rows<NQ, P>(L.Q, 16 * tb + c16, 32 * w4, g4), sp, (f32x4){});
            }
        }
        if (chunk_vp) {
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) store_t16(chunk_vp + ch * GC * GD + 16 * tb * GD + jt, lane, vp[tb]);
        }
        // O = fq (q S) + A V', token tile by token tile.
        if (out) {
            const Op<3> vpl = op_acc(vp[0], vp[1]);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                const f32x4 av = mul_planes(op_rows<3, AR>(L.A, 16 * tb + c16, 0, g4), vpl, (f32x4){});
                const f32x4 o = out_tok(qs[tb], L.fq, 16 * tb + g4, av);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * tb + g4 + v;
                    if (i < Lc) out[((int64_t)(start + c0 + i) * p.hv + h) * GD + j] = (TIn)o[v];
                }
            }
        }
        // S <- e^{G_L} S + k^T (fk V')
        {
            const Op<3> vs = op_acc(scale_tok(vp[0], L.fk, g4), scale_tok(vp[1], L.fk, 16 + g4));
            const float el = L.el;
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) {
                if (packed && rb % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                S[rb] = fma_tile(S[rb], el, mul_planes(op_cols<NQ, C>(L.K, 16 * rb, lane), vs, (f32x4){}));
            }
        }
    }

    // Final state of the node (the initial state of its children).
    float* sp = states + ((size_t)nd.node * p.hv + h) * GD * GD + jt;
#pragma unroll
    for (int rb = 0; rb < 8; ++rb) store_t16(sp + 16 * rb * GD, lane, S[rb]);
}

// Row layout of the level scans, for levels of few nodes: a workgroup takes 16 value columns of one (node, v head), eight
// workgroups per pair, and its wave w the state rows 32w .. 32w+31 of them.
// The products over the state rows (W S and q^ S) are summed over the four
// waves through LDS, in wave order; every wave then updates its own rows. A
// chunk costs each wave about a quarter of the column layout's MFMAs, for
// four times the workgroups: a level with few nodes runs a serial chain of
// chunks on a mostly idle chip, and that chain gets shorter.
constexpr int ROWS_COLS = 16;
constexpr int kRowsSplit = GD / ROWS_COLS;
__device__ __forceinline__ void rows_block(const GdnDev& p, int& h, int& c0) {
    const int bx = blockIdx.x;
    int cs;
    if ((p.hv & 7) == 0) {   // the eight column blocks of a head on one XCD (same L2)
        h = ((bx >> 6) << 3) | (bx & 7);
        cs = (bx >> 3) & 7;
    } else {
        h = bx >> 3;
        cs = bx & 7;
    }
    c0 = ROWS_COLS * cs;
}

// A wave's partial products (W S and q S, both token tiles) lie lane-major in a
// buffer or, packed, over the wave's own columns of W's first two planes, which
// no other wave reads.
template <typename TIn, bool PACKED>
struct ScanRowsLds {
    FwdTiles<TIn> T;
    f32x4 P[4][4][64];
    __device__ __forceinline__ f32x4& part(int w, int n, int lane) { return P[w][n][lane]; }
};
typedef f32x4 __attribute__((may_alias)) f32x4_alias;
template <typename TIn>
struct ScanRowsLds<TIn, true> {
    FwdTiles<TIn, PRS, PCS> T;
    __device__ __forceinline__ f32x4_alias& part(int w, int n, int lane) {
        const int row = 16 * (n & 1) + (lane & 15);
        return *(f32x4_alias*)(T.W + (n >> 1) * GC * GD + tile_at<PRS>(row, 32 * w + 8 * (lane >> 4)));
    }
};

// As gdn_scan_cols_kernel, in the row layout: wave w holds the 32 x 16 slice
// S[32w .., c0 ..] in two 16 x 16 accumulator tiles.
template <typename TIn, bool TRUNC>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_scan_rows_kernel(GdnDev p, int lvl_begin, float* __restrict__ ws,
                                                      TIn* __restrict__ out, float* __restrict__ states,
                                                      float* __restrict__ chunk_sin, float* __restrict__ chunk_vp) {
    constexpr int NQ = kInPlanes<TIn>;
    constexpr bool packed = kScanPacked<TIn, TRUNC>;
    constexpr int P = packed ? PRS : PR, C = packed ? PCS : PC;
    __shared__ __attribute__((aligned(16))) ScanRowsLds<TIn, packed> L;
    ScanNode nd;
    if (!nd.init(p, lvl_begin)) return;
    int h, cb;
    rows_block(p, h, cb);
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, c16 = lane & 15, g4 = 4 * (lane >> 4);
    const int j = cb + c16;                                               // this lane's value column
    const int rb0 = 2 * wave;                                             // the wave's first row tile
    const int start = nd.start, len = nd.len, chunk0 = nd.chunk0, n_ch = nd.n_ch;
    const float* s0 = nd.state0(p, states, h);
    f32x4 S[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) S[r] = s0 ? load_t16(s0 + cb + 16 * (rb0 + r) * GD, lane) : (f32x4){};
    const Op<3> s0p = op_acc(S[0], S[1]);   // TRUNC

    ScanAhead<TIn> nx;
    auto fetch = [&](int ci) {
        const float* cw = ws + ((size_t)(chunk0 + ci) * p.hv + h) * kWsChunk;
        scan_fetch_rows<TIn>(p, cw, start + GC * ci, min(GC, len - GC * ci), h, nx);
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) nx.x[tb] = load_t16(cw + kWsU + 16 * tb * GD + cb, lane);
    };
    if (n_ch > 0) fetch(0);
    for (int ci = 0; ci < n_ch; ++ci) {
        const int c0 = GC * ci, Lc = min(GC, len - c0);
        const size_t ch = (size_t)(chunk0 + ci) * p.hv + h;
        if (chunk_sin) {
            float* sp = chunk_sin + ch * GD * GD + cb;
#pragma unroll
            for (int r = 0; r < 2; ++r) store_t16(sp + 16 * (rb0 + r) * GD, lane, S[r]);
        }
        lds_barrier();   // readers of the previous chunk's tiles and partials are done
        L.T.stage(p, nx);
        f32x4 vp[2] = {nx.x[0], nx.x[1]}, qs[2] = {};
        if (ci + 1 < n_ch) fetch(ci + 1);
        const Op<3> sp = op_acc(S[0], S[1]);
        lds_barrier();

        // this wave's rows of W S and q S (all of W's reads before the partials)
        f32x4 part[4];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            part[tb] = mul_planes(op_rows<3, P>(L.T.W, 16 * tb + c16, 32 * wave, g4), TRUNC ? s0p : sp, (f32x4){});
            part[2 + tb] = mul_planes(op_rows<NQ, P>(L.T.Q, 16 * tb + c16, 32 * wave, g4), sp, (f32x4){});
        }
#pragma unroll
        for (int n = 0; n < 4; ++n) L.part(wave, n, lane) = part[n];
        lds_barrier();
        // V' = U - W S and q S, the partials summed in wave order
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                vp[tb] -= L.part(w, tb, lane);
                qs[tb] += L.part(w, 2 + tb, lane);
            }
        }
        if (chunk_vp && wave == 0) {
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) store_t16(chunk_vp + ch * GC * GD + 16 * tb * GD + cb, lane, vp[tb]);
        }
        // S <- e^{G_L} S + k^T (fk V') on this wave's rows
        const Op<3> vs = op_acc(scale_tok(vp[0], L.T.fk, g4), scale_tok(vp[1], L.T.fk, 16 + g4));
        const float el = L.T.el;
#pragma unroll
        for (int r = 0; r < 2; ++r)
            S[r] = fma_tile(S[r], el, mul_planes(op_cols<NQ, C>(L.T.K, 16 * (rb0 + r), lane), vs, (f32x4){}));
        // O = fq (q S) + A V': waves 0 and 1 take one token tile each
        if (out && wave < 2) {
            const int tb = wave;
            const Op<3> vpl = op_acc(vp[0], vp[1]);
            const f32x4 av = mul_planes(op_rows<3, AR>(L.T.A, 16 * tb + c16, 0, g4), vpl, (f32x4){});
            const f32x4 o = out_tok(tb ? qs[1] : qs[0], L.T.fq, 16 * tb + g4, av);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = 16 * tb + g4 + v;
                if (i < Lc) out[((int64_t)(start + c0 + i) * p.hv + h) * GD + j] = (TIn)o[v];
            }
        }
    }

    float* sp = states + ((size_t)nd.node * p.hv + h) * GD * GD + cb;
#pragma unroll
    for (int r = 0; r < 2; ++r) store_t16(sp + 16 * (rb0 + r) * GD, lane, S[r]);
}

// ----------------------------------------------------------------------------
// reverse scan
// ----------------------------------------------------------------------------
// dS after a node, NT 16-row tiles from row tile rb0 at the columns of
// `col0`: its state's incoming gradient, if any, plus the sum over its
// children of their dS at entry.
template <int NT>
__device__ __forceinline__ void rscan_start(const GdnDev& p, int node, int h, int rb0, int col0, int lane,
                                            const float* node_dsin, f32x4 (&dS)[NT]) {
    if (p.d_states && (!p.d_states_last || node == p.n_nodes - 1)) {
        const float* sp = p.d_states + ((size_t)(p.d_states_last ? 0 : node) * p.hv + h) * GD * GD + col0;
#pragma unroll
        for (int r = 0; r < NT; ++r) dS[r] = load_t16(sp + 16 * (rb0 + r) * GD, lane);
    } else {
#pragma unroll
        for (int r = 0; r < NT; ++r) dS[r] = (f32x4){};
    }
    const int c_lo = max(p.child_off[node], 0), c_hi = min(p.child_off[node + 1], p.n_nodes);
    for (int ci = c_lo; ci < c_hi; ++ci) {
        const int child = p.child[ci];
        if (child <= node || child >= p.n_nodes) continue;              // children follow their parent
        const float* sp = node_dsin + ((size_t)child * p.hv + h) * GD * GD + col0;
#pragma unroll
        for (int r = 0; r < NT; ++r) dS[r] += load_t16(sp + 16 * (rb0 + r) * GD, lane);
    }
}
// The chunk terms and this lane's dO tiles (column j, zero past the chunk).
template <typename TIn>
__device__ __forceinline__ void rscan_fetch(const GdnDev& p, const ScanNode& nd, int ci, int h, int j, int g4,
                                            const float* ws, const TIn* d_o, int64_t do_st, int64_t do_sh,
                                            ScanAhead<TIn>& x) {
    const int c0 = GC * ci, Lc = min(GC, nd.len - c0);
    const float* cw = ws + ((size_t)(nd.chunk0 + ci) * p.hv + h) * kWsChunk;
    scan_fetch_rows<TIn>(p, cw, nd.start + c0, Lc, h, x);
    const TIn* base = d_o + (int64_t)(nd.start + c0) * do_st + (int64_t)h * do_sh + j;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * tb + g4 + v;
            x.x[tb][v] = i < Lc ? (float)base[(int64_t)i * do_st] : 0.0f;
        }
}
// Column layout as gdn_scan_cols_kernel (scan_block). Wave w owns value
// columns c0 + 16w .. +15: its 128 x 16 slice of dS lives in eight 16 x 16
// accumulator tiles, dO of the chunk is loaded in accumulator layout (rows =
// tokens, two 16-token tiles), and dV' is produced in it, so all three are
// MFMA B operands straight from registers:
//   dV' = A^T dO + fk (k dS),  dS <- e^{G_L} dS + q^T (fq dO) - W^T dV'.
// TRUNC (V' = U - W S0 with the node's initial state S0): the W terms of all
// chunks belong to the gradient at the node's entry; they are summed apart
// and join it there.
template <typename TIn, bool TRUNC>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_rscan_cols_kernel(
        GdnDev p, int lvl_begin, const float* __restrict__ ws, const TIn* __restrict__ d_o, int64_t do_st,
        int64_t do_sh, float* __restrict__ chunk_dso, float* __restrict__ chunk_dvp, float* __restrict__ node_dsin) {
    constexpr int NQ = kInPlanes<TIn>;
    __shared__ __attribute__((aligned(16))) RevTiles<TIn> L;
    ScanNode nd;
    if (!nd.init(p, lvl_begin) || nd.len < 1) return;
    int h, cb;
    scan_block(p, h, cb);
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, c16 = lane & 15, g4 = 4 * (lane >> 4);
    const int jt = cb + 16 * wave, j = jt + c16;
    f32x4 dS[8];
    rscan_start<8>(p, nd.node, h, 0, jt, lane, node_dsin, dS);

    f32x4 wsum[8] = {};   // TRUNC: - sum_c W_c^T dV'_c
    // one chunk ahead (the walk runs backwards)
    ScanAhead<TIn> nx;
    rscan_fetch<TIn>(p, nd, nd.n_ch - 1, h, j, g4, ws, d_o, do_st, do_sh, nx);
    for (int ci = nd.n_ch - 1; ci >= 0; --ci) {
        const size_t chn = (size_t)(nd.chunk0 + ci) * p.hv + h;
        {   // the gradient of this chunk's output state
            float* sp = chunk_dso + chn * GD * GD + jt;
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) store_t16(sp + 16 * rb * GD, lane, dS[rb]);
        }
        lds_barrier();   // readers of the previous chunk's tiles are done
        L.stage(p, nx);
        const f32x4 dov[2] = {nx.x[0], nx.x[1]};
        if (ci > 0) rscan_fetch<TIn>(p, nd, ci - 1, h, j, g4, ws, d_o, do_st, do_sh, nx);
        lds_barrier();

        // dV' as four partial sums added in order, partial w4 holding the
        // state rows 32 w4 .. +31 and (w4 < 2) the A^T dO term of token tile
        // w4: the partition of the row layout's waves (gdn_rscan_rows_kernel),
        // so both layouts give the same bits.
        const Op<NQ> dop = op_in<TIn>(dov[0], dov[1]);
        f32x4 dv[2] = {};
#pragma unroll
        for (int w4 = 0; w4 < 4; ++w4) {
            const Op<3> sp = op_acc(dS[2 * w4], dS[2 * w4 + 1]);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                f32x4 pd = scale_tok(
                    mul_planes(op_rows<NQ, PR>(L.K, 16 * tb + c16, 32 * w4, g4), sp, (f32x4){}), L.fk, 16 * tb + g4);
                if (tb == w4) pd = mul_planes(op_cols<3, AC>(L.A, 16 * tb, lane), dop, pd);
                add_alt(dv[tb], pd);
            }
        }
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) store_t16(chunk_dvp + chn * GC * GD + 16 * tb * GD + jt, lane, dv[tb]);

        // dS <- e^{G_L} dS + q^T (fq dO) - W^T dV'
        const Op<3> dos = op_acc(scale_tok(dov[0], L.fq, g4), scale_tok(dov[1], L.fq, 16 + g4));
        const Op<3> dvs = op_acc(-dv[0], -dv[1]);
        const float el = L.el;
#pragma unroll
        for (int rb = 0; rb < 8; ++rb) {
            f32x4 x = mul_planes(op_cols<NQ, PC>(L.Q, 16 * rb, lane), dos, (f32x4){});
            if constexpr (TRUNC) wsum[rb] += mul_planes(op_cols<3, PC>(L.W, 16 * rb, lane), dvs, (f32x4){});
            else x = mul_planes(op_cols<3, PC>(L.W, 16 * rb, lane), dvs, x);
            dS[rb] = fma_tile(dS[rb], el, x);
        }
    }
    if constexpr (TRUNC) {
#pragma unroll
        for (int rb = 0; rb < 8; ++rb) dS[rb] += wsum[rb];
    }
    // dS at the node's entry, summed into its parent by the next (shallower) level.
    float* sp = node_dsin + ((size_t)nd.node * p.hv + h) * GD * GD + jt;
#pragma unroll
    for (int rb = 0; rb < 8; ++rb) store_t16(sp + 16 * rb * GD, lane, dS[rb]);
}

template <typename TIn>
struct RscanRowsLds {
    RevTiles<TIn> T;
    f32x4 P[4][2][64];   // per wave: its partial dV', both token tiles, lane-major
};

// As gdn_rscan_cols_kernel, in the row layout of gdn_scan_rows_kernel: wave w holds dS[32w .., c0 ..]. dV' is summed over the
// waves' rows through LDS, in wave order (waves 0 and 1 also add the A^T dO
// term of token tiles 0 and 1); every wave then updates its rows of dS.
template <typename TIn, bool TRUNC>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_rscan_rows_kernel(
        GdnDev p, int lvl_begin, const float* __restrict__ ws, const TIn* __restrict__ d_o, int64_t do_st,
        int64_t do_sh, float* __restrict__ chunk_dso, float* __restrict__ chunk_dvp, float* __restrict__ node_dsin) {
    constexpr int NQ = kInPlanes<TIn>;
    __shared__ __attribute__((aligned(16))) RscanRowsLds<TIn> L;
    ScanNode nd;
    if (!nd.init(p, lvl_begin) || nd.len < 1) return;
    int h, cb;
    rows_block(p, h, cb);
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, c16 = lane & 15, g4 = 4 * (lane >> 4);
    const int j = cb + c16;
    const int rb0 = 2 * wave;
    f32x4 dS[2];
    rscan_start<2>(p, nd.node, h, rb0, cb, lane, node_dsin, dS);
    f32x4 wsum[2] = {};   // TRUNC: - sum_c W_c^T dV'_c

    ScanAhead<TIn> nx;
    rscan_fetch<TIn>(p, nd, nd.n_ch - 1, h, j, g4, ws, d_o, do_st, do_sh, nx);
    for (int ci = nd.n_ch - 1; ci >= 0; --ci) {
        const size_t chn = (size_t)(nd.chunk0 + ci) * p.hv + h;
        {
            float* sp = chunk_dso + chn * GD * GD + cb;
#pragma unroll
            for (int r = 0; r < 2; ++r) store_t16(sp + 16 * (rb0 + r) * GD, lane, dS[r]);
        }
        lds_barrier();   // readers of the previous chunk's tiles and partials are done
        L.T.stage(p, nx);
        const f32x4 dov[2] = {nx.x[0], nx.x[1]};
        if (ci > 0) rscan_fetch<TIn>(p, nd, ci - 1, h, j, g4, ws, d_o, do_st, do_sh, nx);
        const Op<3> sp = op_acc(dS[0], dS[1]);
        lds_barrier();

        const Op<NQ> dop = op_in<TIn>(dov[0], dov[1]);
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            f32x4 pd = scale_tok(mul_planes(op_rows<NQ, PR>(L.T.K, 16 * tb + c16, 32 * wave, g4), sp, (f32x4){}),
                                 L.T.fk, 16 * tb + g4);
            if (tb == wave) pd = mul_planes(op_cols<3, AC>(L.T.A, 16 * tb, lane), dop, pd);
            L.P[wave][tb][lane] = pd;
        }
        lds_barrier();
        f32x4 dv[2] = {};
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
#pragma unroll
            for (int w = 0; w < 4; ++w) add_alt(dv[tb], L.P[w][tb][lane]);
        }
        if (wave == 0) {
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) store_t16(chunk_dvp + chn * GC * GD + 16 * tb * GD + cb, lane, dv[tb]);
        }

        // dS <- e^{G_L} dS + q^T (fq dO) - W^T dV' on this wave's rows
        const Op<3> dos = op_acc(scale_tok(dov[0], L.T.fq, g4), scale_tok(dov[1], L.T.fq, 16 + g4));
        const Op<3> dvs = op_acc(-dv[0], -dv[1]);
        const float el = L.T.el;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            f32x4 x = mul_planes(op_cols<NQ, PC>(L.T.Q, 16 * (rb0 + r), lane), dos, (f32x4){});
            if constexpr (TRUNC) wsum[r] += mul_planes(op_cols<3, PC>(L.T.W, 16 * (rb0 + r), lane), dvs, (f32x4){});
            else x = mul_planes(op_cols<3, PC>(L.T.W, 16 * (rb0 + r), lane), dvs, x);
            dS[r] = fma_tile(dS[r], el, x);
        }
    }
    if constexpr (TRUNC) {
#pragma unroll
        for (int r = 0; r < 2; ++r) dS[r] += wsum[r];
    }
    float* sp = node_dsin + ((size_t)nd.node * p.hv + h) * GD * GD + cb;
#pragma unroll
    for (int r = 0; r < 2; ++r) store_t16(sp + 16 * (rb0 + r) * GD, lane, dS[r]);
}

}  // namespace
