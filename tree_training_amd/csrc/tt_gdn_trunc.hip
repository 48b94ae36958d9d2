// The reference's own within-node correction for the tree gated delta rule
// (tt_gdn_problem.reference_truncated = 1; tree_dfs_ssm.py:100-150): each whole
// node is one chunk and its correction is built from the uncorrected rows,
//   R = -strictly_lower(beta k^ k^T * D),  D[i][m] = exp(G_i - G_m),
//   [U | W] = (I + R + R^2) Y0,  Y0 = [beta v | beta e^G k^],
// with G the node's cumulative log decay (node-level, not chunk-level). The
// level scans then take V' = U - W S_parent for every chunk of the node.
//
// R is never stored: a node is cut into the same 32-row blocks the scans walk
// (one block = one chunk), and R applied to a block-row is a sum over the
// node's other blocks (earlier ones for R, later ones for R^T), each R block
// formed on the fly from k^ k^T and the decays (bf16 planes, tt_planes.h). The work is
// quadratic in the node length, like the reference's L x L matrices.
//
// Backward, given dF = [dV' | dW] of every chunk (level scans):
//   dF1 = R^T dF,  dY0 = dF + dF1 + R^T dF1,
//   E = strictly_lower(dF (Y0 + R Y0)^T + dF1 Y0^T)     (the gradient of R),
// and through R[i][m] = -beta_i (k^_i . k^_m) D[i][m], with M = E * D:
//   dbeta_i -= sum_m M[i][m] (k^_i . k^_m),  dG_i -= beta_i sum_m M[i][m] (k^_i . k^_m),
//   dk^_i  -= beta_i sum_m M[i][m] k^_m,     dk^_m -= sum_i M[i][m] beta_i k^_i,
//   dG_m  += sum_i beta_i M[i][m] (k^_i . k^_m),
// plus the Y0 terms (dv = beta dY0_v, dbeta, dk^ and dG from beta e^G k^). The
// node-level dG becomes dg by a suffix sum over the node; the chunk backward
// (tt_gdn.hip) adds dk^ and that suffix sum to its own terms.
#include "tt_gdn_planes.h"

namespace {

constexpr int GW = 2 * GD;        // width of [v | k] rows

// Node of chunk c and the chunk's block index within it; false for a malformed list.
__device__ __forceinline__ bool chunk_block(const GdnDev& p, int c, int& node, int& b, int& nb) {
    node = p.chunk_node[c];
    if (node < 0 || node >= p.n_nodes) return false;
    const int len = p.node_len[node], c0 = p.node_chunk0[node];
    nb = tt_cdiv(len, GC);
    b = c - c0;
    return len >= 1 && b >= 0 && b < nb && c0 >= 0 && c0 <= p.n_chunks - nb;
}

// Values of the chunk rows per (chunk, head): the node-level decay, and 1 / |k|
// (1 without the l2 norm) in the chunk terms' T slot, which this mode has no
// inverse for.
struct NodeRows {
    const float* gn;     // [chunk, hv, 32]
    const float* prep;   // the chunk terms
    __device__ __forceinline__ float fk(size_t ch, int row) const { return prep[ch * kWsChunk + kWsT + row]; }
};

// Workgroup -> (chunk, v head), heads fastest: with Hv a multiple of 8 a head
// stays on one XCD, whose L2 then holds the blocks that a node's workgroups
// share.
__device__ __forceinline__ void chunk_head(const GdnDev& p, int& c, int& h) {
    c = __builtin_amdgcn_readfirstlane(blockIdx.x / p.hv);
    h = __builtin_amdgcn_readfirstlane(blockIdx.x % p.hv);
}

// ----------------------------------------------------------------------------
// node-level decay: gn = the chunk cumulative sums (prep) plus the sum over the
// node's earlier chunks
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(64) void gdn_gnode_kernel(GdnDev p, const float* __restrict__ prep,
                                                       float* __restrict__ gn) {
    const int node = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int len = p.node_len[node], c0 = p.node_chunk0[node], nch = tt_cdiv(len, GC);
    if (len < 1 || c0 < 0 || c0 > p.n_chunks - nch) return;
    float carry = 0.0f;
    for (int b = 0; b < nch; ++b) {
        const size_t chn = (size_t)(c0 + b) * p.hv + h;
        const float gv = lane < GC ? prep[chn * kWsChunk + kWsG + lane] : 0.0f;
        const float last = __shfl(gv, GC - 1);
        if (lane < GC) gn[chn * GC + lane] = gv + carry;
        carry += last;
    }
}
// 1 / |k| (NodeRows::fk) and Y0 = [beta v | beta e^G k^] of every row, Y0 into
// the chunk terms' U and W slots.
template <typename TIn>
__global__ __launch_bounds__(GT) void gdn_y0_kernel(GdnDev p, float* __restrict__ prep, const float* __restrict__ gn) {
    int c, h, start, len;
    chunk_head(p, c, h);
    if (!chunk_span(p, c, start, len)) return;
    const int t = threadIdx.x, i = t >> 3, d0 = 16 * (t & 7);
    const size_t chn = (size_t)c * p.hv + h;
    const int64_t tok = start + i;
    float kv[16], vv[16], bt = 0.0f;
    if (i < len) {
        load16((const TIn*)p.k + tok * p.k_st + (int64_t)(h / p.rep) * p.k_sh + d0, kv);
        load16((const TIn*)p.v + tok * p.v_st + (int64_t)h * p.v_sh + d0, vv);
        bt = p.beta[tok * p.b_st + h];
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) kv[e] = vv[e] = 0.0f;
    }
    float sk = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) sk = fmaf(kv[e], kv[e], sk);
    sk = row8_sum(sk);
    const float f = p.l2 ? 1.0f / sqrtf(sk + 1e-6f) : 1.0f, bg = bt * expf(gn[chn * GC + i]);
    if ((t & 7) == 0) prep[chn * kWsChunk + kWsT + i] = f;
    float* u = prep + chn * kWsChunk + kWsU + i * GD + d0;
    float* w = prep + chn * kWsChunk + kWsW + i * GD + d0;
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
        *(f32x4*)(u + e) = (f32x4){bt * vv[e], bt * vv[e + 1], bt * vv[e + 2], bt * vv[e + 3]};
        *(f32x4*)(w + e) = (f32x4){bg * (f * kv[e]), bg * (f * kv[e + 1]), bg * (f * kv[e + 2]), bg * (f * kv[e + 3])};
    }
}

// A target block (chunk c, v head h) and where its node's blocks are; the
// wave's quadrant of a [32 target rows x 32 partner rows] matrix (rows
// 16 qi + g4 + v, column 16 qj + c16 of lane l).
struct BlockPair {
    int b, nb, start, len, nstart, nlen, chunk0, h, hk;
    int qi, qj, lane, c16, g4, qr, qc;
    size_t chn;
    __device__ __forceinline__ bool init(const GdnDev& p) {
        int c, node;
        chunk_head(p, c, h);
        if (!chunk_block(p, c, node, b, nb) || !chunk_span(p, c, start, len)) return false;
        hk = h / p.rep;
        nstart = p.node_start[node];
        nlen = p.node_len[node];
        chunk0 = p.node_chunk0[node];
        chn = (size_t)c * p.hv + h;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        qi = wave >> 1;
        qj = wave & 1;
        lane = threadIdx.x & 63;
        c16 = lane & 15;
        g4 = 4 * (lane >> 4);
        qr = 16 * qi + g4;
        qc = 16 * qj + c16;
        return true;
    }
    __device__ __forceinline__ size_t partner(const GdnDev& p, int bp, int& startp, int& lenp) const {
        startp = nstart + GC * bp;
        lenp = min(GC, nlen - GC * bp);
        return (size_t)(chunk0 + bp) * p.hv + h;
    }
    // k rows 16 tile + c16 of the block at `st` (of `n` rows) as four operands, as they come
    template <typename TIn>
    __device__ __forceinline__ void k_rows(const GdnDev& p, int st, int n, int tile, Op<kInPlanes<TIn>> (&x)[4]) const {
        const int r = 16 * tile + c16;
        const TIn* row = (const TIn*)p.k + (int64_t)(st + r) * p.k_st + (int64_t)hk * p.k_sh;
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m] = op_global<TIn>(row, r < n, 32 * m, g4);
    }
    // beta of row r of the block at `st` (zero past its n rows)
    __device__ __forceinline__ float beta(const GdnDev& p, int st, int n, int r) const {
        return r < n ? p.beta[(int64_t)(st + r) * p.b_st + h] : 0.0f;
    }
};
// k k^T of the quadrant (no norms).
template <int NQ>
__device__ __forceinline__ f32x4 kk_quadrant(const Op<NQ> (&a)[4], const Op<NQ> (&b)[4]) {
    Sum2 x;
#pragma unroll
    for (int m = 0; m < 4; ++m) x.add(a[m], b[m]);
    return x.sum();
}
// Column operand of a [GC][ld] fp32 matrix in global memory: rows k (n of
// them exist), column at `col`.
__device__ __forceinline__ Op<3> op_gcols(const float* col, int ld, int g4) {
    f32x4 a, b;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        a[v] = col[(g4 + v) * ld];
        b[v] = col[(16 + g4 + v) * ld];
    }
    return op_acc(a, b);
}

// ----------------------------------------------------------------------------
// out = R X over a node's blocks (lower: target block b, partners b' <= b) or
// out = R^T X (upper: partners b' >= b), [32 x 256] per (chunk, v head).
// ----------------------------------------------------------------------------
enum { TRI_Y1 = 0, TRI_UW = 1, TRI_DF1 = 2, TRI_DY0 = 3 };
struct TriArgs {
    NodeRows rows;
    const float* xa;      // TRI_UW: y1; TRI_DF1: dV'; TRI_DY0: dF1
    const float* xb;      // TRI_DF1: dW
    const float* fa;      // TRI_DY0: dV' and dW (the target's dF)
    const float* fb;
    float* out;           // TRI_Y1: y1; TRI_DF1: dF1; TRI_DY0: dY0 ([chunk, hv, 32, 256])
    float* prep;          // chunk terms: U and W slots hold Y0, and U, W after TRI_UW
};

// MODE: TRI_Y1   y1 = R Y0
//       TRI_UW   [U | W] = Y0 + y1 + R y1, into the chunk terms
//       TRI_DF1  dF1 = R^T [dV' | dW]
//       TRI_DY0  dY0 = dF + dF1 + R^T dF1
// Wave w forms its quadrant of each R block from k rows read straight into MFMA
// operands, shares it through LDS as planes (rows times alt; two buffers, one
// barrier a block) and owns output columns 64w .. 64w+63, whose X it reads as
// operands from global memory: 15 KB of LDS, so the chains of short blocks of
// many workgroups overlap on a CU. 4,096-token tree, 16 v heads, bf16:
// 281-403 -> 117-149 us a mode (fp32 MFMA before).
template <int MODE, typename TIn>
__global__ __launch_bounds__(GT) void gdn_tri_kernel(GdnDev p, TriArgs a) {
    constexpr bool UPPER = MODE >= TRI_DF1;
    constexpr int NQ = kInPlanes<TIn>;
    __shared__ __attribute__((aligned(16))) __bf16 R[2][3 * GC * AR];
    BlockPair q;
    if (!q.init(p)) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool vcols = wave < 2;   // the wave's columns: of v (0 .. 127) or of k (128 .. 255)
    const int cw = 64 * (wave & 1) + q.c16;
    Op<NQ> kt[4];
    q.k_rows<TIn>(p, q.start, q.len, q.qi, kt);
    f32x4 gt, ft;   // decay and -(beta, lower) / |k| of the quadrant's rows, times alt
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = q.qr + v;
        gt[v] = a.rows.gn[q.chn * GC + r];
        ft[v] = -a.rows.fk(q.chn, r) * alt(v) * (UPPER ? 1.0f : q.beta(p, q.start, q.len, r));
    }
    f32x4 acc[2][4] = {};
    const int bp0 = UPPER ? q.b : 0, bp1 = UPPER ? q.nb : q.b + 1;
    for (int bp = bp0; bp < bp1; ++bp) {
        int startp, lenp;
        const size_t chp = q.partner(p, bp, startp, lenp);
        __bf16* Rb = R[(bp - bp0) & 1];
        {
            f32x4 r = {};
            if (bp != q.b || (UPPER ? q.qj >= q.qi : q.qi >= q.qj)) {
                Op<NQ> kp[4];
                q.k_rows<TIn>(p, startp, lenp, q.qj, kp);
                const float gp = a.rows.gn[chp * GC + q.qc];
                const float fp = a.rows.fk(chp, q.qc) * (UPPER ? q.beta(p, startp, lenp, q.qc) : 1.0f);
                r = kk_quadrant<NQ>(kt, kp);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = q.qr + v;
                    const bool vis = i < q.len && q.qc < lenp && (bp != q.b || (UPPER ? q.qc > i : q.qc < i));
                    r[v] = vis ? ft[v] * (r[v] * fp) * expf(UPPER ? gp - gt[v] : gt[v] - gp) : 0.0f;
                }
            }
            put_quadrant<AR>(Rb, q.qr, q.qc, r);
        }
        // this wave's columns of the partner's X
        Op<3> x[4];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const int col = cw + 16 * cb;
            if constexpr (MODE == TRI_Y1) {
                x[cb] = op_gcols(a.prep + chp * kWsChunk + (vcols ? kWsU : kWsW) + col, GD, q.g4);
            } else if constexpr (MODE == TRI_DF1) {
                x[cb] = op_gcols((vcols ? a.xa : a.xb) + chp * GC * GD + col, GD, q.g4);
            } else {
                x[cb] = op_gcols(a.xa + chp * GC * GW + (vcols ? 0 : GD) + col, GW, q.g4);
            }
        }
        lds_barrier();   // the R block is complete
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const Op<3> r = op_rows<3, AR>(Rb, 16 * tb + q.c16, 0, q.g4);
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[tb][cb] += mul_planes(r, x[cb], (f32x4){});
        }
    }

    // Accumulator element v: row 16 tb + g4 + v (times alt), column 16 cb of the wave's.
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * tb + q.g4 + v;
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) {
                const int col = cw + 16 * cb, j = (vcols ? 0 : GD) + col;
                float val = v & 1 ? -acc[tb][cb][v] : acc[tb][cb][v];
                if constexpr (MODE == TRI_UW) {
                    float* y0 = a.prep + q.chn * kWsChunk + (vcols ? kWsU : kWsW) + i * GD + col;
                    *y0 = val + (*y0 + a.xa[(q.chn * GC + i) * GW + j]);
                } else {
                    if constexpr (MODE == TRI_DY0)
                        val += (vcols ? a.fa : a.fb)[(q.chn * GC + i) * GD + col] + a.xa[(q.chn * GC + i) * GW + j];
                    a.out[(q.chn * GC + i) * GW + j] = val;
                }
            }
        }
}

// ----------------------------------------------------------------------------
// gradient of R: row side (per target block b over partners b' <= b) and
// column side (partners b' >= b: rows of R in the partner, columns in the target)
// ----------------------------------------------------------------------------
struct EArgs {
    NodeRows rows;
    const float* y1;      // R Y0
    const float* dvp;     // dV' ([chunk, hv, 32, 128])
    const float* dw;      // dW
    const float* df1;     // R^T dF ([chunk, hv, 32, 256])
    const float* dy0;     // dF + dF1 + R^T dF1
    float* dkr;           // dk^ from the correction, [chunk, hv, 32, 128]
    float* dgn;           // node-level dG, [chunk, hv, 32]
    void* dv;             // [T, Hv, 128] problem dtype (row side only)
    float* dbeta;         // [T, Hv] (row side only)
};

struct ELds {
    union {
        float E[4][GC * MS];    // the waves' slices of the 512-wide contraction
        float J[GC * RS];       // at the end: dk^ rows
    };
    __bf16 M[3 * GC * AR];
    float sum[2][GC];           // row sums over the column tiles
};

// Wave w's 128 columns of the 512-wide contraction E = [dF | dF1] [Y0 + y1 | Y0]^T:
//   w = 0: dV' . (beta v + y1_v)      w = 1: dW . (beta e^G k^ + y1_k)
//   w = 2: dF1_v . beta v             w = 3: dF1_k . beta e^G k^
// Row `row` of a block (chunk-head ch, tokens st .. st + n - 1) of [Y0 + y1 | Y0].
template <typename TIn>
__device__ __forceinline__ Op<3> e_op_y(const GdnDev& p, const EArgs& a, const BlockPair& q, int wave, size_t ch,
                                        int st, int n, int row, float f, int k0) {
    const int64_t tok = st + row;
    const TIn* x = (wave & 1) == 0 ? (const TIn*)p.v + tok * p.v_st + (int64_t)q.h * p.v_sh
                                   : (const TIn*)p.k + tok * p.k_st + (int64_t)q.hk * p.k_sh;
    f32x4 y[2] = {};
#pragma unroll
    for (int n2 = 0; n2 < 2; ++n2) {
        const int d = k0 + 16 * n2 + q.g4;
        if (row < n) y[n2] = load4(x + d) * f;
        if (wave < 2) y[n2] += *(const f32x4*)(a.y1 + (ch * GC + row) * GW + (wave ? GD : 0) + d);
    }
    return op_acc(y[0], y[1]);
}
// ... and of [dF | dF1].
__device__ __forceinline__ Op<3> e_op_f(const EArgs& a, const BlockPair& q, int wave, size_t ch, int row, int k0) {
    const float* x = wave == 0 ? a.dvp + (ch * GC + row) * GD
                   : wave == 1 ? a.dw + (ch * GC + row) * GD
                               : a.df1 + (ch * GC + row) * GW + (wave == 2 ? 0 : GD);
    return op_acc(*(const f32x4*)(x + k0 + q.g4), *(const f32x4*)(x + k0 + 16 + q.g4));
}

// ROW: M = E * D over partners b' <= b: dk^ rows of the target
// -= beta (M k^_p), dbeta, dG, and the Y0 terms (dv among them). Otherwise the
// column side: M^T over partners b' >= b, dk^ += M^T (beta k^)_p (negated), dG.
// The target's planes of F (ROW) or Y stay in registers (96); the partner's
// rows come straight into operands. 4,096-token tree, 16 v heads, bf16:
// rows 523 -> 405 us, columns 446 -> 283. Bound by the latency of those loads:
// the registers leave two waves a SIMD. fp32 problems, with three planes of k as
// well, spill 35 and 41 registers there (the same tree, the whole fp32 step: 3.94 ->
// 2.58 ms; 16,318 tokens, 32 v heads: 23.5 -> 16.9).
template <typename TIn, bool ROW>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_e_kernel(GdnDev p, EArgs a) {
    constexpr int NQ = kInPlanes<TIn>;
    __shared__ __attribute__((aligned(16))) ELds L;
    BlockPair q;
    if (!q.init(p)) return;
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int w0 = 32 * wave;   // this wave's columns of dk^

    // y's factor of a row: beta (times e^G / |k| in the k slices)
    auto y_factor = [&](size_t ch, int st, int n, int row) {
        float f = q.beta(p, st, n, row);
        if (wave & 1) f *= expf(a.rows.gn[ch * GC + row]) * a.rows.fk(ch, row);
        return f;
    };
    Op<3> at[2][4];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
        const int row = 16 * tb + q.c16;
        const float f = ROW ? 0.0f : y_factor(q.chn, q.start, q.len, row);
#pragma unroll
        for (int m = 0; m < 4; ++m)
            at[tb][m] = ROW ? e_op_f(a, q, wave, q.chn, row, 32 * m)
                            : e_op_y<TIn>(p, a, q, wave, q.chn, q.start, q.len, row, f, 32 * m);
    }
    Op<NQ> kt[4];
    q.k_rows<TIn>(p, q.start, q.len, q.qi, kt);
    f32x4 gt, ft;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        gt[v] = a.rows.gn[q.chn * GC + q.qr + v];
        ft[v] = a.rows.fk(q.chn, q.qr + v);
    }
    f32x4 dk[2][2] = {};   // row tile, column tile w0 + 16 cb
    f32x4 sums = {};       // sum over the partners of M (k^ . k^) (column side: times beta)
    const int bp0 = ROW ? 0 : q.b, bp1 = ROW ? q.b + 1 : q.nb;
    for (int bp = bp0; bp < bp1; ++bp) {
        int startp, lenp;
        const size_t chp = q.partner(p, bp, startp, lenp);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const int row = 16 * cb + q.c16;
            const float f = ROW ? y_factor(chp, startp, lenp, row) : 0.0f;
            Sum2 e[2];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const Op<3> x = ROW ? e_op_y<TIn>(p, a, q, wave, chp, startp, lenp, row, f, 32 * m)
                                    : e_op_f(a, q, wave, chp, row, 32 * m);
                e[0].add(at[0][m], x);
                e[1].add(at[1][m], x);
            }
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                const f32x4 r = e[tb].sum();
#pragma unroll
                for (int v = 0; v < 4; ++v) L.E[wave][(16 * tb + q.g4 + v) * MS + row] = r[v];
            }
        }
        const float gp = a.rows.gn[chp * GC + q.qc], fp = a.rows.fk(chp, q.qc);
        const float bm = ROW ? 1.0f : q.beta(p, startp, lenp, q.qc);
        f32x4 kk = {};
        const bool any = bp != q.b || (ROW ? q.qi >= q.qj : q.qj >= q.qi);
        if (any) {
            Op<NQ> kp[4];
            q.k_rows<TIn>(p, startp, lenp, q.qj, kp);
            kk = kk_quadrant<NQ>(kt, kp);
        }
        lds_barrier();   // the four slices of E are complete
        {
            f32x4 mv = {};
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = q.qr + v, idx = i * MS + q.qc;
                const bool vis = i < q.len && q.qc < lenp && (bp != q.b || (ROW ? q.qc < i : q.qc > i));
                if (vis)
                    mv[v] = bm * (((L.E[0][idx] + L.E[1][idx]) + (L.E[2][idx] + L.E[3][idx])) *
                                  expf(ROW ? gt[v] - gp : gp - gt[v]));
                sums[v] = fmaf(mv[v], kk[v] * (ft[v] * fp), sums[v]);
                mv[v] *= v & 1 ? -fp : fp;   // times alt; 1 / |k| of the partner's row
            }
            put_quadrant<AR>(L.M, q.qr, q.qc, mv);
        }
        lds_barrier();   // M is complete, E's readers are done
        // dk^ rows += M k_p over head dims w0 + 16 cb + c16
        const Op<3> m0 = op_rows<3, AR>(L.M, q.c16, 0, q.g4), m1 = op_rows<3, AR>(L.M, 16 + q.c16, 0, q.g4);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const TIn* kc = (const TIn*)p.k + (int64_t)startp * p.k_st + (int64_t)q.hk * p.k_sh + w0 + 16 * cb + q.c16;
            f32x4 x[2];
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int m = 16 * tb + q.g4 + v;
                    x[tb][v] = m < lenp ? (float)kc[(int64_t)m * p.k_st] : 0.0f;
                }
            const Op<NQ> kx = op_in<TIn>(x[0], x[1]);
            dk[0][cb] += mul_planes(m0, kx, (f32x4){});
            dk[1][cb] += mul_planes(m1, kx, (f32x4){});
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float r = sum16(sums[v]);
        if (q.c16 == 0) L.sum[q.qj][q.qr + v] = r;
    }
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int v = 0; v < 4; ++v)   // E's readers passed the last barrier
                L.J[(16 * tb + q.g4 + v) * RS + w0 + 16 * cb + q.c16] = v & 1 ? dk[tb][cb][v] : -dk[tb][cb][v];
    lds_barrier();
    // Per row: thread t owns row t/8, dims 16 (t % 8) .. +15 of v and of k.
    const int i = t >> 3, d0 = 16 * (t & 7);
    const bool in = i < q.len;
    const int64_t tok = q.start + i;
    const float s_row = L.sum[0][i] + L.sum[1][i];
    float* dst = a.dkr + (q.chn * GC + i) * GD + d0;
    if constexpr (ROW) {
        const float bt = q.beta(p, q.start, q.len, i), eg = expf(a.rows.gn[q.chn * GC + i]);
        const float fk = a.rows.fk(q.chn, i);
        const float* dyr = a.dy0 + (q.chn * GC + i) * GW;
        float vv[16], kv[16];
        if (in) {
            load16((const TIn*)p.v + tok * p.v_st + (int64_t)q.h * p.v_sh + d0, vv);
            load16((const TIn*)p.k + tok * p.k_st + (int64_t)q.hk * p.k_sh + d0, kv);
        } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) vv[e] = kv[e] = 0.0f;
        }
        float vdot = 0.0f, kdot = 0.0f;
        f32x4 dvo[4];
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            const f32x4 dyv = *(const f32x4*)(dyr + d0 + 4 * e4);
            const f32x4 dyk = *(const f32x4*)(dyr + GD + d0 + 4 * e4);
            f32x4 kr = *(const f32x4*)&L.J[i * RS + d0 + 4 * e4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                vdot = fmaf(dyv[e], vv[4 * e4 + e], vdot);
                kdot = fmaf(dyk[e], kv[4 * e4 + e] * fk, kdot);
                kr[e] = fmaf(bt * eg, dyk[e], bt * kr[e]);
                dvo[e4][e] = bt * dyv[e];
            }
            *(f32x4*)(dst + 4 * e4) = kr;
        }
        if (in)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) store4((TIn*)a.dv + tok * p.dv_st + q.h * GD + d0 + 4 * e4, dvo[e4]);
        vdot = row8_sum(vdot);
        kdot = row8_sum(kdot);
        if ((t & 7) == 0) {
            if (in) a.dbeta[tok * p.hv + q.h] = -s_row + vdot + eg * kdot;
            a.dgn[q.chn * GC + i] = in ? bt * (eg * kdot - s_row) : 0.0f;
        }
    } else {
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4)
            *(f32x4*)(dst + 4 * e4) = *(const f32x4*)(dst + 4 * e4) + *(const f32x4*)&L.J[i * RS + d0 + 4 * e4];
        if ((t & 7) == 0 && in) a.dgn[q.chn * GC + i] += s_row;
    }
}

// ----------------------------------------------------------------------------
// node-level dG -> its suffix sums over the node (in place): dg_i gets
// sum_{j >= i in the node} dG_j, G being the node's cumulative sum
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(64) void gdn_gsuffix_kernel(GdnDev p, float* __restrict__ dgn) {
    const int node = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int len = p.node_len[node], c0 = p.node_chunk0[node], nch = tt_cdiv(len, GC);
    if (len < 1 || c0 < 0 || c0 > p.n_chunks - nch) return;
    float carry = 0.0f;
    for (int b = nch - 1; b >= 0; --b) {
        const size_t chn = (size_t)(c0 + b) * p.hv + h;
        const int lenc = min(GC, len - GC * b);
        float v = lane < lenc ? dgn[chn * GC + lane] : 0.0f;
#pragma unroll
        for (int o = 1; o < GC; o <<= 1) {
            const float up = __shfl_down(v, o, GC);
            if ((lane & (GC - 1)) + o < GC) v += up;
        }
        const float total = __shfl(v, 0);
        if (lane < GC) dgn[chn * GC + lane] = lane < lenc ? v + carry : 0.0f;
        carry += total;
    }
}

template <typename TIn>
int trunc_fwd(const GdnDev& d, float* prep, float* gn, float* y1, hipStream_t s) {
    const NodeRows rows{gn, prep};
    const dim3 grid((unsigned)((size_t)d.n_chunks * d.hv));
    hipLaunchKernelGGL(gdn_gnode_kernel, dim3(d.n_nodes, d.hv), dim3(64), 0, s, d, prep, gn);
    hipLaunchKernelGGL((gdn_y0_kernel<TIn>), grid, dim3(GT), 0, s, d, prep, gn);
    TriArgs a{rows, nullptr, nullptr, nullptr, nullptr, y1, prep};
    hipLaunchKernelGGL((gdn_tri_kernel<TRI_Y1, TIn>), grid, dim3(GT), 0, s, d, a);
    a.xa = y1;
    a.out = nullptr;
    hipLaunchKernelGGL((gdn_tri_kernel<TRI_UW, TIn>), grid, dim3(GT), 0, s, d, a);
    return hipGetLastError() == hipSuccess ? TT_OK : TT_E_HIP;
}

template <typename TIn>
int trunc_bwd(const GdnDev& d, const GdnTruncBwd& w, void* dv, float* dbeta, hipStream_t s) {
    const NodeRows rows{w.gn, w.prep};
    const dim3 grid((unsigned)((size_t)d.n_chunks * d.hv));
    TriArgs t1{rows, w.dvp, w.dw, nullptr, nullptr, w.df1, nullptr};
    hipLaunchKernelGGL((gdn_tri_kernel<TRI_DF1, TIn>), grid, dim3(GT), 0, s, d, t1);
    TriArgs t2{rows, w.df1, nullptr, w.dvp, w.dw, w.dy0, nullptr};
    hipLaunchKernelGGL((gdn_tri_kernel<TRI_DY0, TIn>), grid, dim3(GT), 0, s, d, t2);
    EArgs e{rows, w.y1, w.dvp, w.dw, w.df1, w.dy0, w.dkr, w.dgn, dv, dbeta};
    hipLaunchKernelGGL((gdn_e_kernel<TIn, true>), grid, dim3(GT), 0, s, d, e);
    hipLaunchKernelGGL((gdn_e_kernel<TIn, false>), grid, dim3(GT), 0, s, d, e);
    hipLaunchKernelGGL(gdn_gsuffix_kernel, dim3(d.n_nodes, d.hv), dim3(64), 0, s, d, w.dgn);
    return hipGetLastError() == hipSuccess ? TT_OK : TT_E_HIP;
}

}  // namespace

int tt_gdn_trunc_fwd_launch(const GdnDev& d, float* prep, float* gn, float* y1, hipStream_t s) {
    return d.dtype == TT_DTYPE_BF16 ? trunc_fwd<__bf16>(d, prep, gn, y1, s) : trunc_fwd<float>(d, prep, gn, y1, s);
}

int tt_gdn_trunc_bwd_launch(const GdnDev& d, const GdnTruncBwd& w, void* dv, float* dbeta, hipStream_t s) {
    return d.dtype == TT_DTYPE_BF16 ? trunc_bwd<__bf16>(d, w, dv, dbeta, s) : trunc_bwd<float>(d, w, dv, dbeta, s);
}
