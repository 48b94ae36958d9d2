// Tree gated delta rule (the linear-attention layers of Qwen3.5-style models)
// over a DFS-packed tree: forward for gfx950.
//
// Semantics: the gated delta rule token by token along every root-to-leaf
// path — each node continues from its parent's final state (a root from the
// caller's initial state, or zero) — evaluated exactly in TT_GDN_CHUNK =
// 32-token chunks (a node is cut into consecutive chunks; its last chunk may
// be short):
//   G = cumsum(g), D[i][j] = exp(G_i - G_j) (j <= i),
//   N = -strictly_lower(beta k k^T * D),  T = (I - N)^-1,
//   U = T (beta v),  W = T (beta e^G k),  A = lower_incl(q k^T * D),
//   V' = U - W S,  O = e^G (q S) + A V',  S <- e^{G_last} S + (k e^{G_last - G})^T V'.
// q and k are l2-normalised in the kernels and q is scaled; v head h reads q/k
// head h / (Hv / Hk).
//
// Two kernels:
//  * gdn_prep_kernel — one workgroup per (chunk, v head), all chunks at once:
//    everything that does not depend on the state (A, T by a product of
//    (I + N^(2^r)) factors, U, W, G) into the workspace.
//  * gdn_scan_cols_kernel — per (node, v head) two workgroups of four waves,
//    one launch per tree level so a node's parent state (in the caller's
//    node_states buffer) is complete when it starts; each wave holds a
//    128 x 16 value slice of the state in MFMA accumulators (the delta rule is
//    independent per value column) and walks the node's chunks. Levels of
//    one or two nodes use gdn_scan_rows_kernel instead (eight workgroups per
//    pair, each wave a 32 x 16 slice), which gives the same bits.
// fp32 accuracy end to end: products on bf16 planes of fp32 operands
// (tt_gdn_planes.h), the inverse and element-wise work on the vector ALUs.
#include "tt_gdn_common.h"
#include "tt_gdn_scan.h"

namespace {


// ----------------------------------------------------------------------------
// prep: per (chunk, v head) A, T, U, W, G
// ----------------------------------------------------------------------------
// bf16 problems move q and v through LDS too (coalesced rows, and 37 KB still let
// four workgroups share a CU: 268 us against 358 for operands straight from
// memory); in fp32 their planes would leave two (32 us against 23).
template <typename TIn>
constexpr bool kPrepTiles = sizeof(TIn) == 2;

template <typename TIn>
struct PrepLds {
    __bf16 K[kInPlanes<TIn> * GC * PC];           // k as it comes
    __bf16 Q[kPrepTiles<TIn> ? GC * PC : 8];      // q as it comes; v once the products with q are done
    float R[8 * 16 * 17];     // the 16 x 16 blocks of the inverse
    float N[GC * MS];         // N = -strictly_lower(beta k^ k^T * D)
    float Tm[GC * MS];        // T = (I - N)^-1
    float G[GC], Glo[GC], beta[GC];
    float bg[GC];             // beta e^G / |k|
    float fq[GC], fk[GC];     // scale / |q|, 1 / |k|
};

// q k^T and k k^T (a 16 x 16 quadrant a wave, the upper one not read), U and W
// (32 columns a wave) on planes, the norms and decays as factors of rows and
// columns; the inverse T on the vector ALUs. A chain of a dozen barriers, so
// latency bounds the kernel. 16K agent tree, 32 v heads, bf16: 384 us on fp32
// MFMAs (three workgroups a CU) -> 268; fp32, 2,111 tokens, 8 v heads: 23 us both.
// TRUNC (the reference's per-node correction): only A and G here; U and W
// come from the node-level kernels of tt_gdn_trunc.hip.
template <typename TIn, bool TRUNC>
__global__ __launch_bounds__(GT) void gdn_prep_kernel(GdnDev p, float* __restrict__ ws) {
    constexpr int NQ = kInPlanes<TIn>;
    __shared__ __attribute__((aligned(16))) PrepLds<TIn> L;
    const int c = blockIdx.x, h = blockIdx.y;
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int c16 = lane & 15, g4 = 4 * (lane >> 4);
    int start, len;
    if (!chunk_span(p, c, start, len)) return;
    float* out = ws + ((size_t)c * p.hv + h) * kWsChunk;

    const int qi = wave >> 1, qj = wave & 1;            // this wave's quadrant
    const int qr = 16 * qi + g4, qc = 16 * qj + c16;    // this lane's first row and its column there
    const int w0 = 32 * wave;                           // this wave's columns of U and W
    constexpr bool TILES = kPrepTiles<TIn>;
    using Vec = typename std::conditional<sizeof(TIn) == 2, bf16x8, f32x4>::type;
    constexpr int NV = (int)sizeof(TIn);
    const int i8 = t >> 3, d8 = 16 * (t & 7);           // this thread's row and its first dim there
    Vec vv[NV];        // TILES: that part of v
    Op<NQ> qop[4];     // else: q rows of the quadrant's row tile
    f32x4 vx[2][2];    // and v columns w0 + 16 cb + c16, rows 16 tb + g4 .. +3
    {
        const int hk = h / p.rep;
        const auto row16 = [&](const void* x, int64_t st, int64_t off, Vec (&r)[NV]) {
            const TIn* xp = (const TIn*)x + (int64_t)(start + i8) * st + off + d8;
#pragma unroll
            for (int n = 0; n < NV; ++n) {
                if (i8 < len) {
                    r[n] = *(const Vec*)(xp + 16 / NV * n);
                } else {
#pragma unroll
                    for (int e = 0; e < 16 / NV; ++e) r[n][e] = (TIn)0.0f;
                }
            }
        };
        Vec kv[NV], qv[NV];
        row16(p.k, p.k_st, hk * p.k_sh, kv);
        if constexpr (TILES) {
            row16(p.q, p.q_st, hk * p.q_sh, qv);
            if constexpr (!TRUNC) row16(p.v, p.v_st, h * p.v_sh, vv);
            put16<PC>(L.Q, i8, d8, qv);
            const float nq = row_norm(p, qv);
            if ((t & 7) == 0) L.fq[i8] = nq * p.scale;
        } else if (qi >= qj) {
            const int row = 16 * qi + c16;
            const TIn* qp = (const TIn*)p.q + (int64_t)(start + row) * p.q_st + (int64_t)hk * p.q_sh + g4;
            float ss = 0.0f;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const f32x4 x0 = row < len ? load4(qp + 32 * m) : (f32x4){};
                const f32x4 x1 = row < len ? load4(qp + 32 * m + 16) : (f32x4){};
                ss += dot4(x0, x0) + dot4(x1, x1);
                qop[m] = op_in<TIn>(x0, x1);
            }
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            if (qj == 0 && lane < 16) L.fq[row] = (p.l2 ? 1.0f / sqrtf(ss + 1e-6f) : 1.0f) * p.scale;
        }
        if constexpr (!TRUNC && !TILES) {
            const TIn* vp = (const TIn*)p.v + (int64_t)start * p.v_st + (int64_t)h * p.v_sh + w0 + c16;
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int m = 16 * tb + g4 + v;
                        vx[cb][tb][v] = m < len ? (float)vp[(int64_t)m * p.v_st + 16 * cb] : 0.0f;
                    }
        }
        put16<PC>(L.K, i8, d8, kv);
        const float nk = row_norm(p, kv);
        if ((t & 7) == 0) L.fk[i8] = nk;
    }
    if (wave == 0) {
        // cumulative decay over the chunk (lanes 0..31; padded rows add 0),
        // each step's rounding error (two-sum) carried in lo
        const bool valid = lane < len;
        const int64_t tok = start + lane;
        float gv = valid ? p.g[tok * p.g_st + h] : 0.0f, lo = 0.0f;
        const float bv = valid ? p.beta[tok * p.b_st + h] : 0.0f;
#pragma unroll
        for (int o = 1; o < GC; o <<= 1) {
            const float up = __shfl_up(gv, o, GC), up_lo = __shfl_up(lo, o, GC);
            if ((lane & (GC - 1)) >= o) {
                const float sum = gv + up, bp = sum - gv;
                lo += up_lo + ((gv - (sum - bp)) + (up - bp));
                gv = sum;
            }
        }
        if (lane < GC) {
            L.G[lane] = gv;
            L.Glo[lane] = lo;
            L.beta[lane] = bv;
            out[kWsG + lane] = gv;
            out[kWsGlo + lane] = lo;
        }
    }
    lds_barrier();

    // A = lower_incl(q^ k^T * D), N = -strictly_lower(beta k^ k^T * D); the
    // diagonal quadrants of N also start the inverse (below).
    constexpr int BS = 17;                                   // row stride of the 16 x 16 blocks
    constexpr int B16 = 16 * BS;
    float* sc = L.R;
    {
        f32x4 qk = {}, kk = {};
        if (qi >= qj) {
            Sum2 x, y;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const Op<NQ> kj = op_rows<NQ, PC>(L.K, 16 * qj + c16, 32 * m, g4);
                if constexpr (TILES) x.add(op_rows<NQ, PC>(L.Q, 16 * qi + c16, 32 * m, g4), kj);
                else x.add(qop[m], kj);
                if constexpr (!TRUNC) y.add(op_rows<NQ, PC>(L.K, 16 * qi + c16, 32 * m, g4), kj);
            }
            qk = x.sum();
            kk = y.sum();
        }
        const float gj = L.G[qc], glj = L.Glo[qc], fkj = L.fk[qc];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = qr + v;
            const float dec = qc <= i ? expf(gdiff(L.G[i], L.Glo[i], gj, glj)) : 0.0f;
            out[kWsA + i * GC + qc] = qc <= i ? qk[v] * (L.fq[i] * fkj) * dec : 0.0f;
            if constexpr (!TRUNC) {
                const float n = qc < i ? -L.beta[i] * (kk[v] * (L.fk[i] * fkj)) * dec : 0.0f;
                L.N[i * MS + qc] = n;
                if (qi == qj) {
                    float* b = sc + qi * 4 * B16 + (g4 + v) * BS + c16;
                    b[0] = n;
                    b[2 * B16] = n + (qc == i ? 1.0f : 0.0f);
                }
            }
        }
        if (!TRUNC && t < GC) L.bg[t] = L.beta[t] * expf(L.G[t] + L.Glo[t]) * L.fk[t];
    }
    if constexpr (TRUNC) return;
    lds_barrier();   // N complete, q's readers are done
    if constexpr (TILES) put16<PC>(L.Q, i8, d8, vv);

    // T = (I - N)^-1 by 16 x 16 blocks. With N = [[N11, 0], [N21, N22]],
    // T = [[T11, 0], [T22 N21 T11, T22]] and, each Nbb strictly lower
    // triangular (Nbb^16 = 0), Tbb = (I + Nbb)(I + Nbb^2)(I + Nbb^4)(I + Nbb^8):
    // from T = I + Nbb, P = Nbb, three rounds of P <- P P, then T <- T + T P.
    // Waves 0-1 take block 1, waves 2-3 block 2 (thread u: row u/8, columns
    // 2 (u%8), +1), with double-buffered P and T in the partial-product
    // buffer R (free again); then X = N21 T11 and T21 = T22 X, a thread an
    // entry. A quarter of the work of squaring the whole 32 x 32 matrix.
    {
        const int blk = t >> 7, u = t & 127, bi = u >> 3, bj = 2 * (u & 7), o = 16 * blk;
        // block blk: P buffers at pb, pb + B16; T buffers at pb + 2 B16, pb + 3 B16
        const int pb = blk * 4 * B16, tb = pb + 2 * B16;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const int pc = pb + (r & 1) * B16, pn = pb + ((r + 1) & 1) * B16;
            float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const float pim = sc[pc + bi * BS + m];
                a0 = fmaf(pim, sc[pc + m * BS + bj], a0);
                a1 = fmaf(pim, sc[pc + m * BS + bj + 1], a1);
            }
            sc[pn + bi * BS + bj] = a0;
            sc[pn + bi * BS + bj + 1] = a1;
            __syncthreads();
            const int tc0 = tb + (r & 1) * B16, tn = tb + ((r + 1) & 1) * B16;
            float t0 = sc[tc0 + bi * BS + bj], t1 = sc[tc0 + bi * BS + bj + 1];
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const float tim = sc[tc0 + bi * BS + m];
                t0 = fmaf(tim, sc[pn + m * BS + bj], t0);
                t1 = fmaf(tim, sc[pn + m * BS + bj + 1], t1);
            }
            sc[tn + bi * BS + bj] = t0;
            sc[tn + bi * BS + bj + 1] = t1;
            __syncthreads();
        }
        // Tbb is in the second T buffer of its block; X = N21 T11 goes to
        // block 1's first P buffer.
        constexpr int T11 = 3 * B16, T22 = 4 * B16 + 3 * B16, X = 0;
        const int xi = t >> 4, xj = t & 15;
        {
            float x = 0.0f;
#pragma unroll
            for (int m = 0; m < 16; ++m) x = fmaf(L.N[(16 + xi) * MS + m], sc[T11 + m * BS + xj], x);
            sc[X + xi * BS + xj] = x;
        }
        __syncthreads();
        float t21 = 0.0f;
#pragma unroll
        for (int m = 0; m < 16; ++m) t21 = fmaf(sc[T22 + xi * BS + m], sc[X + m * BS + xj], t21);
        L.Tm[(16 + xi) * MS + xj] = t21;
        L.Tm[xi * MS + 16 + xj] = 0.0f;
#pragma unroll
        for (int e = 0; e < 2; ++e) L.Tm[(o + bi) * MS + o + bj + e] = sc[tb + B16 + bi * BS + bj + e];
        __syncthreads();
        const int ti = t >> 3, tc = 4 * (t & 7);
        *(f32x4*)(out + kWsT + ti * GC + tc) = *(const f32x4*)&L.Tm[ti * MS + tc];
    }

    // U = T (beta v), W = T (beta e^G k^): wave w produces columns 32w .. 32w+31,
    // the odd rows formed negated (alt).
    {
        Op<3> tu[2], tw[2];   // rows of T, its columns times beta and beta e^G / |k|
        const f32x4 b0 = *(const f32x4*)&L.beta[g4], b1 = *(const f32x4*)&L.beta[16 + g4];
        const f32x4 e0 = *(const f32x4*)&L.bg[g4], e1 = *(const f32x4*)&L.bg[16 + g4];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const float* row = &L.Tm[(16 * tb + c16) * MS + g4];
            const f32x4 x0 = alt(c16) * *(const f32x4*)row, x1 = alt(c16) * *(const f32x4*)(row + 16);
            tu[tb] = op_acc(x0 * b0, x1 * b1);
            tw[tb] = op_acc(x0 * e0, x1 * e1);
        }
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const Op<NQ> kc = op_cols<NQ, PC>(L.K, w0 + 16 * cb, lane);
            Op<NQ> vc;
            if constexpr (TILES) vc = op_cols<NQ, PC>(L.Q, w0 + 16 * cb, lane);
            else vc = op_in<TIn>(vx[cb][0], vx[cb][1]);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                const f32x4 u = mul_planes(tu[tb], vc, (f32x4){}), w = mul_planes(tw[tb], kc, (f32x4){});
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int o = (16 * tb + g4 + v) * GD + w0 + 16 * cb + c16;
                    out[kWsU + o] = v & 1 ? -u[v] : u[v];
                    out[kWsW + o] = v & 1 ? -w[v] : w[v];
                }
            }
        }
    }
}

// ----------------------------------------------------------------------------
// backward
// ----------------------------------------------------------------------------
// The backward recomputes the forward (prep + level scans, keeping each
// chunk's initial state S and V'), then:
//  * gdn_rscan_cols_kernel — reverse level scan (deepest level first) of dS, the
//    gradient of the state after a chunk, per (node, v head):
//      dV' = A^T dO + (e^{G_L - G} k^) dS,
//      dS <- e^{G_L} dS + (e^G q^)^T dO - W^T dV'.
//    A node's last chunk starts from the incoming gradient of its final
//    state (if the caller gives one) plus the sum of its children's dS at
//    entry.
//  * gdn_init_grad_kernel — when the initial state's gradient is wanted: the
//    sum of the roots' dS at entry.
//  * gdn_bwd_state_kernel — per (chunk, v head), the products with the
//    128 x 128 states: X = dO S^T, dW = -dV' S^T, dK~ = V' dS^T, <S, dS>.
//  * gdn_bwd_chunk_kernel — per (chunk, q/k head, looping over its v heads),
//    everything else: the chunk's 32 x 32 algebra (A, T = (I - N)^-1, N),
//    dv, dbeta, dg (reverse cumulative sum of dG within the chunk), and
//    dq, dk summed over the v heads of the group, then through the l2 norm.

// Gradient of the initial state: the sum over the roots, in node order (the
// order in which a node's children's terms are summed), of their state
// gradient at entry. Thread: four consecutive floats of one v head's
// 128 x 128 block.
__global__ __launch_bounds__(GT) void gdn_init_grad_kernel(GdnDev p, const float* __restrict__ node_dsin) {
    const int h = blockIdx.y;
    const int e = 4 * (blockIdx.x * GT + threadIdx.x);
    f32x4 acc = {};
    for (int node = 0; node < p.n_nodes; ++node) {
        const int par = p.parent[node];
        if (par >= 0 && par < node) continue;   // roots only, by the forward scan's rule
        acc += *(const f32x4*)(node_dsin + ((size_t)node * p.hv + h) * GD * GD + e);
    }
    *(f32x4*)(p.d_init + (size_t)h * GD * GD + e) = acc;
}

// State products on fp32 MFMA. The contraction (value dimension, 128) runs in
// four 32-column chunks; per chunk the block stages, with coalesced loads,
// columns v0..v0+31 of all 128 rows of S and dS and of the 32 rows of dO, dV'
// and V' into LDS rows of SCS = 34 floats: the MFMA operand reads (lane =
// row, one float per lane, two adjacent columns per step) then reach all 64
// banks once. Wave w produces columns 32w .. 32w+31 of X, dW and dK~ (rows of
// S / dS 32w .. 32w+31) as accumulators.
constexpr int SCS = 34;
struct StateGradLds {     // gdn_dw_s0_kernel: one chunk of S0 and of dV'
    float S[GD * SCS];
    float A2[GC * SCS];
};

// One 32-column slice of the value dimension of both S and dS (all 128 rows)
// and the matching columns of dO, dV' and V', staged together: every input
// is read once.
struct StatePairLds {
    float S[GD * SCS];
    float dS[GD * SCS];
    float A1[GC * SCS];   // dO
    float A2[GC * SCS];   // dV'
    float A3[GC * SCS];   // V'
    float red[GT / 64];
};

// Registers of one slice: S and dS at the same positions (thread t: row
// t >> 1, columns 16 (t & 1) .. +15) and the 32-row tiles (row t >> 3,
// columns 4 (t & 7) .. +3).
template <typename TIn>
struct StateChunk {
    float s[16];
    float ds[16];
    f32x4 vp, dvp;
    u32x4 d;        // dO as loaded (bf16: two per word; converted when committed)
};

// X = dO S^T, dW = -dV' S^T, dK~ = V' dS^T ([GC x GD] each) and <S, dS>.
template <typename TIn>
__global__ __launch_bounds__(GT) void gdn_bwd_state_kernel(GdnDev p, const TIn* __restrict__ d_o, int64_t do_st,
                                                           int64_t do_sh, const float* __restrict__ chunk_sin,
                                                           const float* __restrict__ chunk_dso,
                                                           const float* __restrict__ chunk_vp,
                                                           const float* __restrict__ chunk_dvp,
                                                           float* __restrict__ xo, float* __restrict__ dwo,
                                                           float* __restrict__ dkto, float* __restrict__ sdot) {
    __shared__ __attribute__((aligned(16))) StatePairLds L;
    const int c = blockIdx.x, h = blockIdx.y, t = threadIdx.x;
    int start, len;
    if (!chunk_span(p, c, start, len)) return;
    const size_t chn = (size_t)c * p.hv + h;
    const int wave = t >> 6, lane = t & 63, col = lane & 31, half = lane >> 5;
    const float* Sin = chunk_sin + chn * GD * GD;
    const float* dSo = chunk_dso + chn * GD * GD;
    const float* dVp = chunk_dvp + chn * GC * GD;
    const float* Vp = chunk_vp + chn * GC * GD;
    const int sr = t >> 1, sc = 16 * (t & 1);      // S / dS staging: row, first column
    const int ar = t >> 3, ac = 4 * (t & 7);       // 32-row tiles: row, first column
    // rows past the chunk's length read its last row and are zeroed at commit
    const TIn* dor = d_o + (int64_t)(start + min(ar, len - 1)) * do_st + (int64_t)h * do_sh;
    const bool arow_in = ar < len;

    auto fetch = [&](int k, StateChunk<TIn>& r) {
        const int v0 = GC * k;
        const int so = sr * GD + v0 + sc;
#pragma unroll
        for (int e = 0; e < 16; e += 4) {
            const f32x4 x4 = *(const f32x4*)(Sin + so + e);
            const f32x4 y4 = *(const f32x4*)(dSo + so + e);
            r.s[e] = x4[0]; r.s[e + 1] = x4[1]; r.s[e + 2] = x4[2]; r.s[e + 3] = x4[3];
            r.ds[e] = y4[0]; r.ds[e + 1] = y4[1]; r.ds[e + 2] = y4[2]; r.ds[e + 3] = y4[3];
        }
        if constexpr (sizeof(TIn) == 2) {
            const u32x2 raw = *(const u32x2*)(dor + v0 + ac);
            r.d = (u32x4){raw[0], raw[1], 0u, 0u};
        } else {
            r.d = *(const u32x4*)(dor + v0 + ac);
        }
        r.dvp = *(const f32x4*)(dVp + ar * GD + v0 + ac);
        r.vp = *(const f32x4*)(Vp + ar * GD + v0 + ac);
    };
    auto commit = [&](const StateChunk<TIn>& r) {
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
            *(float2*)&L.S[sr * SCS + sc + e] = (float2){r.s[e], r.s[e + 1]};
            *(float2*)&L.dS[sr * SCS + sc + e] = (float2){r.ds[e], r.ds[e + 1]};
        }
        const float z = arow_in ? 1.0f : 0.0f;   // dO rows past the chunk are zero
        float dv4[4];
        if constexpr (sizeof(TIn) == 2) {   // bf16 -> fp32: the high half of a float
            dv4[0] = __uint_as_float(r.d[0] << 16);
            dv4[1] = __uint_as_float(r.d[0] & 0xffff0000u);
            dv4[2] = __uint_as_float(r.d[1] << 16);
            dv4[3] = __uint_as_float(r.d[1] & 0xffff0000u);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) dv4[e] = __uint_as_float(r.d[e]);
        }
        *(float2*)&L.A1[ar * SCS + ac] = (float2){z * dv4[0], z * dv4[1]};
        *(float2*)&L.A1[ar * SCS + ac + 2] = (float2){z * dv4[2], z * dv4[3]};
        *(float2*)&L.A2[ar * SCS + ac] = (float2){r.dvp[0], r.dvp[1]};
        *(float2*)&L.A2[ar * SCS + ac + 2] = (float2){r.dvp[2], r.dvp[3]};
        *(float2*)&L.A3[ar * SCS + ac] = (float2){r.vp[0], r.vp[1]};
        *(float2*)&L.A3[ar * SCS + ac + 2] = (float2){r.vp[2], r.vp[3]};
    };

    f32x16 x = (f32x16){}, w = (f32x16){}, kt = (f32x16){};
    float sd = 0.0f;
    const float* brow = &L.S[(32 * wave + col) * SCS + half];    // B: S row 32w + col, columns 2 step + half
    const float* dbrow = &L.dS[(32 * wave + col) * SCS + half];  // B: the same row of dS
    const float* arow1 = &L.A1[col * SCS + half];                // A: row col, columns 2 step + half
    const float* arow2 = &L.A2[col * SCS + half];
    const float* arow3 = &L.A3[col * SCS + half];
    StateChunk<TIn> cur, nxt;
    fetch(0, cur);
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        __syncthreads();   // the previous slice's readers are done
        commit(cur);
#pragma unroll
        for (int e = 0; e < 16; ++e) sd = fmaf(cur.s[e], cur.ds[e], sd);   // <S, dS>, this thread's share
        __syncthreads();
        if (k + 1 < 4) fetch(k + 1, nxt);
#pragma unroll
        for (int st = 0; st < GC / 2; ++st) {
            const float b = brow[2 * st];
            x = mfma_f32(arow1[2 * st], b, x);
            w = mfma_f32(arow2[2 * st], b, w);
            kt = mfma_f32(arow3[2 * st], dbrow[2 * st], kt);
        }
        cur = nxt;
    }
    // Accumulator element r: row acc_row(r, half) (token), column 32w + col.
    store_acc<0>(acc_mat(xo + chn * GC * GD, GC, half, 32 * wave + col), x);
    store_acc<0>(acc_mat(dwo + chn * GC * GD, GC, half, 32 * wave + col), -w);
    store_acc<0>(acc_mat(dkto + chn * GC * GD, GC, half, 32 * wave + col), kt);
    sd = wave_sum(sd);
    if (lane == 0) L.red[wave] = sd;
    __syncthreads();
    if (t == 0) {
        float tot = 0.0f;
#pragma unroll
        for (int w2 = 0; w2 < GT / 64; ++w2) tot += L.red[w2];
        sdot[chn] = tot;
    }
}

// The reference's per-node correction (V' = U - W S0 for every chunk of a
// node): dW = -dV' S0^T with S0 the node's initial state (its first chunk's
// S), per (chunk, v head); it replaces the dW of gdn_bwd_state_kernel, whose
// S is the chunk's own. Same staging as there: per 32-column chunk of the
// value dimension, all 128 rows of S0 and the 32 rows of dV' in LDS rows of
// SCS floats; wave w produces columns 32w .. 32w+31.
__global__ __launch_bounds__(GT) void gdn_dw_s0_kernel(GdnDev p, const float* __restrict__ chunk_sin,
                                                       const float* __restrict__ chunk_dvp,
                                                       float* __restrict__ dwo) {
    __shared__ __attribute__((aligned(16))) StateGradLds L;
    const int c = blockIdx.x, h = blockIdx.y, t = threadIdx.x;
    int start, len;
    if (!chunk_span(p, c, start, len)) return;
    const size_t chn = (size_t)c * p.hv + h;
    const int wave = t >> 6, lane = t & 63, col = lane & 31, half = lane >> 5;
    const float* S0 = chunk_sin + ((size_t)p.node_chunk0[p.chunk_node[c]] * p.hv + h) * GD * GD;
    const float* dVp = chunk_dvp + chn * GC * GD;
    const int sr = t >> 1, sc = 16 * (t & 1);      // S0 staging: row, first column
    const int ar = t >> 3, ac = 4 * (t & 7);       // dV' staging: row, first column
    f32x16 w = {};
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        const int v0 = GC * k;
        __syncthreads();   // the previous chunk's readers are done
#pragma unroll
        for (int e = 0; e < 16; e += 4) {   // rows of SCS floats: 8-byte aligned stores
            const f32x4 x4 = *(const f32x4*)(S0 + sr * GD + v0 + sc + e);
            *(float2*)&L.S[sr * SCS + sc + e] = (float2){x4[0], x4[1]};
            *(float2*)&L.S[sr * SCS + sc + e + 2] = (float2){x4[2], x4[3]};
        }
        const f32x4 a2 = *(const f32x4*)(dVp + ar * GD + v0 + ac);
        *(float2*)&L.A2[ar * SCS + ac] = (float2){a2[0], a2[1]};
        *(float2*)&L.A2[ar * SCS + ac + 2] = (float2){a2[2], a2[3]};
        __syncthreads();
#pragma unroll
        for (int st = 0; st < GC / 2; ++st)
            w = mfma_f32(L.A2[col * SCS + half + 2 * st], L.S[(32 * wave + col) * SCS + half + 2 * st], w);
    }
    store_acc<0>(acc_mat(dwo + chn * GC * GD, GC, half, 32 * wave + col), -w);
}

// One 16 x 16 quadrant a wave of a 32 x 32 product: rows 16 qi + g4 + v,
// column 16 qj + c16, in accumulator layout.
template <typename TIn>
struct ChunkGradLds {
    static constexpr int NQ = kInPlanes<TIn>;
    __bf16 Q[NQ * GC * PC];   // q and k as they come
    __bf16 K[NQ * GC * PC];
    union {
        __bf16 X[3 * GC * PR];   // V', then dV', then dW
        float J[GC * RS];        // the last join of product and element-wise terms
    };
    union {
        __bf16 P[2 * 3 * GC * AC];   // dP fk_j and dP fq_i
        float Y[GC * MS];            // Y = T^T dT
    };
    float T[GC * MS];
    float M[GC * MS];     // dT, then E
    float S[GC * MS];     // dA * A + dN * N (the pair terms of dG), then its row prefix sums
    float G[GC], Glo[GC], B[GC], Bg[GC], fq[GC], fk[GC];   // Bg: beta e^G
    float Grow[GC], Crow[GC];
    float bv[2][GC], bk[2][GC];   // column sums over the row tiles of T * (dV' v^T), T * (dW k^^T)
    float db[2][GC];              // row sums over the column tiles of the pair terms of dbeta
};

// Four fp32 values at columns c0 .. c0 + 3 of row i of a tile of planes.
template <int N, int P>
__device__ __forceinline__ f32x4 row4(const __bf16* X, int i, int c0) {
    f32x4 r = load4(X + i * P + c0);
    if constexpr (N == 3) {
        r += load4(X + GC * P + i * P + c0);
        r += load4(X + 2 * GC * P + i * P + c0);
    }
    return r;
}
// Column operand f X[k][c0 + c16] of a [GC][MS] fp32 matrix, k over its 32 rows.
__device__ __forceinline__ Op<3> op_fcols(const float* X, int c0, int c16, int g4, float f) {
    f32x4 a, b;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        a[v] = f * X[(g4 + v) * MS + c0 + c16];
        b[v] = f * X[(16 + g4 + v) * MS + c0 + c16];
    }
    return op_acc(a, b);
}
// The compiler moves no work across: overlapped, the phases of a head do not
// fit the registers.
__device__ __forceinline__ void phase() { __builtin_amdgcn_sched_barrier(0); }

// Products by tiles of v_mfma_f32_16x16x32_bf16 on planes: a [32 x 32] result
// is a quadrant a wave (the upper one holds nothing that is read and is left
// out), a [32 x 128] one 32 columns a wave. The three [32 x 128] inputs that
// need splitting (V', dV', dW) pass through one LDS tile in turn, each loaded a
// phase ahead; q, k, v and dO of bf16 problems are used as they come. A head
// is a chain of nine barriers, so latency bounds the kernel: 78 KB of LDS and
// 256 registers (bf16) let two workgroups share a CU, one working behind the
// other's barriers and loads. 16K agent tree, 16/32 heads, bf16: 1553 -> 1032
// us against one workgroup a CU on fp32 MFMAs (120 KB, sums of four partial
// products through LDS); fp32, 2,081 tokens, 4/8 heads: 84 -> 70 us.
// Element-wise work: thread t owns row i = t/8 and columns 32m + 4s + e
// (s = t%8; m, e < 4) of [32 x 128] rows; [32 x 32] results stay in the
// quadrant layout.
// TRUNC (the reference's per-node correction): U and W do not come from the
// chunk's T, so the T part is left out; dv and dbeta are complete already
// (tt_gdn_trunc.hip), and trk (dk^ of the correction, [chunk, Hv, 32, 128])
// and trg (the node-level suffix sums of its dG, [chunk, Hv, 32]) are added.
template <typename TIn, bool TRUNC>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(sizeof(TIn) == 2 ? 2 : 1, 2))) void gdn_bwd_chunk_kernel(
        GdnDev p, const TIn* __restrict__ d_o, int64_t do_st, int64_t do_sh, const float* __restrict__ ws,
        const float* __restrict__ chunk_vp, const float* __restrict__ chunk_dvp, const float* __restrict__ xo,
        const float* __restrict__ dwo, const float* __restrict__ dkto, const float* __restrict__ sdot,
        TIn* __restrict__ dq, TIn* __restrict__ dk, TIn* __restrict__ dv, float* __restrict__ dg,
        float* __restrict__ dbeta, const float* __restrict__ trk, const float* __restrict__ trg) {
    constexpr int NQ = kInPlanes<TIn>;
    __shared__ __attribute__((aligned(16))) ChunkGradLds<TIn> L;
    const int c = blockIdx.x, hk = blockIdx.y, t = threadIdx.x;
    int start, len;
    if (!chunk_span(p, c, start, len)) return;
    const int i = t >> 3, s = t & 7;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, c16 = lane & 15, g4 = 4 * (lane >> 4);
    const int qi = wave >> 1, qj = wave & 1;            // this wave's quadrant ...
    const bool lower = qi >= qj;                        // ... and whether it holds pairs j <= i
    const int qr = 16 * qi + g4, qc = 16 * qj + c16;    // this lane's first row and its column there
    const int w0 = 32 * wave;                           // this wave's columns of [32 x 128] results
    const bool valid = i < len;
    const int64_t tok = start + i;

    {   // q and k rows as they come, and their norms
        using Vec = typename std::conditional<sizeof(TIn) == 2, bf16x8, f32x4>::type;
        constexpr int NV = (int)sizeof(TIn), EV = 16 / NV;
        Vec qv[NV], kv[NV];
        const TIn* qp = (const TIn*)p.q + tok * p.q_st + (int64_t)hk * p.q_sh + 16 * s;
        const TIn* kp = (const TIn*)p.k + tok * p.k_st + (int64_t)hk * p.k_sh + 16 * s;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            if (valid) {
                qv[n] = *(const Vec*)(qp + EV * n);
                kv[n] = *(const Vec*)(kp + EV * n);
            } else {
#pragma unroll
                for (int e = 0; e < EV; ++e) qv[n][e] = kv[n][e] = (TIn)0.0f;
            }
        }
        put16<PC>(L.Q, i, 16 * s, qv);
        put16<PC>(L.K, i, 16 * s, kv);
        const float nq = row_norm(p, qv), nk = row_norm(p, kv);
        if (s == 0) {
            L.fq[i] = nq * p.scale;
            L.fk[i] = nk;
        }
    }
    // One of the [32 x 128] fp32 inputs of a head on its way to L.X: row i,
    // columns 16 s .. +15.
    f32x4 xr[4];
    auto fetch_x = [&](const float* src, size_t chn) {
#pragma unroll
        for (int e = 0; e < 4; ++e) xr[e] = *(const f32x4*)(src + (chn * GC + i) * GD + 16 * s + 4 * e);
    };
    const size_t chn0 = (size_t)c * p.hv + hk * p.rep;
    fetch_x(chunk_vp, chn0);
    lds_barrier();
    f32x4 kk = {};   // k^ k^T
    if (!TRUNC && lower) {
        Sum2 x;
#pragma unroll
        for (int m = 0; m < 4; ++m)
            x.add(op_rows<NQ, PC>(L.K, 16 * qi + c16, 32 * m, g4), op_rows<NQ, PC>(L.K, 16 * qj + c16, 32 * m, g4));
        kk = x.sum();
#pragma unroll
        for (int v = 0; v < 4; ++v) kk[v] *= L.fk[qr + v] * L.fk[qc];
    }
    float dqa[16], dka[16];   // element-wise terms (row layout)
#pragma unroll
    for (int e = 0; e < 16; ++e) dqa[e] = dka[e] = 0.0f;
    f32x4 dqm[2][2] = {}, dkm[2][2] = {};   // product terms: row tile, column tile w0 + 16 cb

#pragma unroll 1
    for (int hh = 0; hh < p.rep; ++hh) {
        const int h = hk * p.rep + hh;
        const size_t chn = chn0 + hh;
        // The thread's coordinates, made opaque to the compiler once a head and
        // again halfway: hoisted out of the loop, the LDS and global addresses
        // made of them spill 150 registers.
#define TT_CHUNK_COORDS()                                                                                \
    int to = threadIdx.x;                                                                                \
    asm volatile("" : "+v"(to));                                                                         \
    const int i = to >> 3, s = to & 7, lane = to & 63, c16 = lane & 15, g4 = 4 * (lane >> 4);            \
    const int qr = 16 * qi + g4, qc = 16 * qj + c16;                                                     \
    (void)i, (void)s, (void)lane, (void)c16, (void)g4, (void)qr, (void)qc
        TT_CHUNK_COORDS();
        const bool valid = i < len;
        const int64_t tok = start + i;
        const float* cw = ws + chn * kWsChunk;
        // e^{G_L} <S, dS> for dg, loaded here so its latency hides behind the head's work
        const float gsd = sdot[chn];
        f32x4 aq;   // this lane's entries of A
#pragma unroll
        for (int v = 0; v < 4; ++v) aq[v] = cw[kWsA + (qr + v) * GC + qc];
        Op<NQ> dop[4];   // dO rows of the quadrant's row tile
        {
            const TIn* row = d_o + (int64_t)(start + 16 * qi + c16) * do_st + (int64_t)h * do_sh;
#pragma unroll
            for (int m = 0; m < 4; ++m) dop[m] = op_global<TIn>(row, 16 * qi + c16 < len, 32 * m, g4);
        }
        // the previous head's last readers of X, T, G and B are two barriers back
        put16<PR>(L.X, i, 16 * s, xr);
        if constexpr (!TRUNC) *(f32x4*)&L.T[i * MS + 4 * s] = *(const f32x4*)(cw + kWsT + i * GC + 4 * s);
        if (t < GC) {
            const float gt = cw[kWsG + t], bt = t < len ? p.beta[(int64_t)(start + t) * p.b_st + h] : 0.0f;
            L.G[t] = gt;
            L.Glo[t] = cw[kWsGlo + t];
            L.B[t] = bt;
            L.Bg[t] = bt * expf(gt);
        }
        if constexpr (!TRUNC) fetch_x(chunk_dvp, chn);
        lds_barrier();
        const float gi = L.G[i], gl = L.G[GC - 1], egi = expf(gi);
        const float ed = expf(gdiff(gl, L.Glo[GC - 1], gi, L.Glo[i])), egl = expf(gl);
        const float bj = L.B[qc], ej = expf(L.G[qc] + L.Glo[qc]), fkj = L.fk[qc];

        // dA = dO V'^T; the pair terms dA * A of dG; dP = dA * D (j <= i), once
        // times fk_j (for dq^) and once times fq_i (for dk^).
        f32x4 pair = {};
        {
            f32x4 da = {};
            if (lower) {
                Sum2 x;
#pragma unroll
                for (int m = 0; m < 4; ++m) x.add(dop[m], op_rows<3, PR>(L.X, 16 * qj + c16, 32 * m, g4));
                da = x.sum();
            }
            f32x4 pk, pq;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = qr + v;
                const bool in = qc <= r;
                const float x = in ? da[v] : 0.0f;
                pair[v] = x * aq[v];
                const float dpv = in ? x * expf(gdiff(L.G[r], L.Glo[r], L.G[qc], L.Glo[qc])) : 0.0f;
                pk[v] = v & 1 ? -(dpv * fkj) : dpv * fkj;   // rows i of dP: alt(i)
                pq[v] = dpv * (L.fq[r] * alt(c16));         // rows j of dP^T: alt(j)
            }
            put_quadrant<AC>(L.P, qr, qc, pk);
            put_quadrant<AC>(L.P + 3 * GC * AC, qr, qc, pq);
        }
        phase();
        // O's state term e^G q^ S: dq^ += e^G X, dG += e^G q^ . X; the output
        // state's (e^{G_L - G} k^)^T V': dk^, and c_i = e^{G_L - G_i} k^_i . dK~_i.
        float dgp = 0.0f, cp = 0.0f;
        {
            const float* xp = xo + (chn * GC + i) * GD;
            const float* kp = dkto + (chn * GC + i) * GD;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const f32x4 x = *(const f32x4*)(xp + 32 * m + 4 * s), y = *(const f32x4*)(kp + 32 * m + 4 * s);
                dgp += dot4(row4<NQ, PC>(L.Q, i, 32 * m + 4 * s), x);
                cp += dot4(row4<NQ, PC>(L.K, i, 32 * m + 4 * s), y);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    dqa[4 * m + e] = fmaf(egi, x[e], dqa[4 * m + e]);
                    dka[4 * m + e] = fmaf(ed, y[e], dka[4 * m + e]);
                }
            }
            dgp = row8_sum(dgp) * (egi * L.fq[i]);
            cp = row8_sum(cp) * (ed * L.fk[i]);
        }
        if constexpr (TRUNC) {   // the correction's dk^ (its dv, dbeta are complete)
            const float* kr = trk + (chn * GC + i) * GD;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const f32x4 x = *(const f32x4*)(kr + 32 * m + 4 * s);
#pragma unroll
                for (int e = 0; e < 4; ++e) dka[4 * m + e] += x[e];
            }
        }
        phase();
        lds_barrier();   // dP complete, X's readers are done
        if constexpr (!TRUNC) {
            put16<PR>(L.X, i, 16 * s, xr);
            fetch_x(dwo, chn);
        } else if (hh + 1 < p.rep) {
            fetch_x(chunk_vp, chn + 1);
        }
        phase();
        // dq^ += dP k^, dk^ += dP^T q^ (contraction over the chunk's 32 tokens).
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            phase();
            const Op<NQ> kc = op_cols<NQ, PC>(L.K, w0 + 16 * cb, lane), qcv = op_cols<NQ, PC>(L.Q, w0 + 16 * cb, lane);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                add_alt(dqm[tb][cb], mul_planes(op_rows<3, AC>(L.P, 16 * tb + c16, 0, g4), kc, (f32x4){}));
                add_alt(dkm[tb][cb], mul_planes(op_cols<3, AC>(L.P + 3 * GC * AC, 16 * tb, lane), qcv, (f32x4){}));
            }
        }
        float dbp = 0.0f;
        if constexpr (!TRUNC) {
            TT_CHUNK_COORDS();
            const Op<3> tt[2] = {op_fcols(L.T, 0, c16, g4, alt(c16)), op_fcols(L.T, 16, c16, g4, alt(c16))};   // T^T by rows
            Op<NQ> vop[4];   // v rows of the quadrant's column tile
            {
                const TIn* row = (const TIn*)p.v + (int64_t)(start + 16 * qj + c16) * p.v_st + (int64_t)h * p.v_sh;
#pragma unroll
                for (int m = 0; m < 4; ++m) vop[m] = op_global<TIn>(row, 16 * qj + c16 < len, 32 * m, g4);
            }
            phase();
            lds_barrier();   // dV' in X; dP's readers are done
            // dT's part dV' v^T, and dBv = T^T dV': dv = beta dBv.
            TIn* const dvh = dv + (int64_t)start * p.dv_st + h * GD + w0;   // uniform; 32-bit offsets of its rows
            f32x4 tv = {};
            if (lower) {
                Sum2 x;
#pragma unroll
                for (int m = 0; m < 4; ++m) x.add(op_rows<3, PR>(L.X, 16 * qi + c16, 32 * m, g4), vop[m]);
                tv = x.sum();
            }
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) {
                phase();
                const Op<3> x = op_cols<3, PR>(L.X, w0 + 16 * cb, lane);
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) {
                    const f32x4 o = mul_planes(tt[tb], x, (f32x4){});
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int r = 16 * tb + g4 + v;
                        const float x = v & 1 ? -o[v] : o[v];
                        if (r < len) dvh[(unsigned)(r * p.dv_st + 16 * cb + c16)] = (TIn)(L.B[r] * x);
                    }
                }
            }
            phase();
            lds_barrier();   // X's readers are done
            put16<PR>(L.X, i, 16 * s, xr);
            if (hh + 1 < p.rep) fetch_x(chunk_vp, chn + 1);
            lds_barrier();
            // dT's part dW k^^T, and dBk = T^T dW: dk^ += beta e^G dBk.
            f32x4 tk = {};
            if (lower) {
                Sum2 x;
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    x.add(op_rows<3, PR>(L.X, 16 * qi + c16, 32 * m, g4),
                          op_rows<NQ, PC>(L.K, 16 * qj + c16, 32 * m, g4));
                tk = x.sum();
            }
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) {
                phase();
                const Op<3> x = op_cols<3, PR>(L.X, w0 + 16 * cb, lane);
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) {
                    const f32x4 o = mul_planes(tt[tb], x, (f32x4){});
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int r = 16 * tb + g4 + v;
                        dkm[tb][cb][v] = fmaf(L.Bg[r], v & 1 ? -o[v] : o[v], dkm[tb][cb][v]);
                    }
                }
            }
            phase();
            // dbeta and dG take sum_c v_ic dBv_ic = sum_m T_mi (dV' v^T)_mi and
            // the same of k^ and dW: column sums over the rows of T * (...).
            {
                float sv = 0.0f, sk = 0.0f;
                f32x4 dt;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float tm = L.T[(qr + v) * MS + qc], k1 = tk[v] * fkj;
                    sv = fmaf(tm, tv[v], sv);
                    sk = fmaf(tm, k1, sk);
                    dt[v] = bj * fmaf(ej, k1, tv[v]);   // dT = dV' (beta v)^T + dW (beta e^G k^)^T
                }
                sv += __shfl_xor(sv, 16);
                sk += __shfl_xor(sk, 16);
                sv += __shfl_xor(sv, 32);
                sk += __shfl_xor(sk, 32);
                if (g4 == 0) {
                    L.bv[qi][qc] = sv;
                    L.bk[qi][qc] = sk;
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) L.M[(qr + v) * MS + qc] = dt[v];
            }
            lds_barrier();   // dT complete
            phase();
            // Y = T^T dT (only m' <= i is read)
            if (lower) {
                const f32x4 y = mul_planes(qi ? tt[1] : tt[0], op_fcols(L.M, 16 * qj, c16, g4, 1.0f), (f32x4){});
#pragma unroll
                for (int v = 0; v < 4; ++v) L.Y[(qr + v) * MS + qc] = v & 1 ? -y[v] : y[v];
            }
            {
                const float vb = L.bv[0][i] + L.bv[1][i], kb = L.bk[0][i] + L.bk[1][i];
                dbp = fmaf(egi, kb, vb);
                dgp = fmaf(L.Bg[i], kb, dgp);
            }
            lds_barrier();   // Y complete, dT's readers are done
            // dN = Y T^T (strictly lower): dbeta, dG and E = dL/d(k^ k^T) from
            // N = -beta (k^ k^T) * D.
            {
                f32x4 dn = {};
                if (lower) {
                    const int yr = (16 * qi + c16) * MS + g4, tr = (16 * qj + c16) * MS + g4;
                    // m' <= j: the second half of Y's and T's rows is not read for the upper column tile
                    const f32x4 z = {};
                    dn = mul_planes(op_acc(*(const f32x4*)&L.Y[yr], qi && qj ? *(const f32x4*)&L.Y[yr + 16] : z),
                                    op_acc(*(const f32x4*)&L.T[tr], qj ? *(const f32x4*)&L.T[tr + 16] : z), (f32x4){});
                }
                f32x4 db;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = qr + v;
                    const bool in = qc < r;
                    const float dd = in ? expf(gdiff(L.G[r], L.Glo[r], L.G[qc], L.Glo[qc])) : 0.0f;
                    const float x = in ? -dn[v] * dd : 0.0f;   // dN D
                    db[v] = x * kk[v];
                    pair[v] = fmaf(L.B[r], db[v], pair[v]);
                    L.M[r * MS + qc] = x * L.B[r];
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float r = sum16(db[v]);
                    if (c16 == 0) L.db[qj][qr + v] = r;
                }
            }
        }
        phase();
        {
            TT_CHUNK_COORDS();
#pragma unroll
            for (int v = 0; v < 4; ++v) L.S[(qr + v) * MS + qc] = pair[v];
        }
        if (s == 0) {
            L.Grow[i] = dgp;
            L.Crow[i] = cp;
        }
        lds_barrier();
        if constexpr (!TRUNC) {
            // dk^ += (E + E^T) k^
            const f32x4 f0 = *(const f32x4*)(L.fk + g4) * alt(c16), f1 = *(const f32x4*)(L.fk + 16 + g4) * alt(c16);
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                const int r = 16 * tb + c16;
                f32x4 a = *(const f32x4*)&L.M[r * MS + g4], b = *(const f32x4*)&L.M[r * MS + 16 + g4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    a[v] = (a[v] + L.M[(g4 + v) * MS + r]) * f0[v];
                    b[v] = (b[v] + L.M[(16 + g4 + v) * MS + r]) * f1[v];
                }
                const Op<3> e = op_acc(a, b);
#pragma unroll
                for (int cb = 0; cb < 2; ++cb)
                    add_alt(dkm[tb][cb], mul_planes(e, op_cols<NQ, PC>(L.K, w0 + 16 * cb, lane), (f32x4){}));
            }
            if (s == 0 && valid) dbeta[tok * p.hv + h] = dbp + (L.db[0][i] + L.db[1][i]);
        }
        // S holds every pair term of dG: its rows become exclusive prefix sums,
        // S[i][c] = sum_{j < c} p_ij (thread (i, s): four columns, a scan over
        // the row's eight threads), for the dg sums below.
        {
            f32x4 v = *(const f32x4*)&L.S[i * MS + 4 * s];
            const float tot = v[0] + v[1] + v[2] + v[3];
            float pre = __shfl_up(tot, 1, 8);
            if (s == 0) pre = 0.0f;
#pragma unroll
            for (int o = 1; o < 8; o <<= 1) {
                const float up = __shfl_up(pre, o, 8);
                if (s >= o) pre += up;
            }
            f32x4 x;
            x[0] = pre;
            x[1] = pre + v[0];
            x[2] = x[1] + v[1];
            x[3] = x[2] + v[2];
            *(f32x4*)&L.S[i * MS + 4 * s] = x;
        }
        // dg_t = sum of dG_u over u >= t within the chunk (G is its cumulative
        // sum). A pair term p_ij (S, i > j: the factors e^{G_i - G_j} of A and
        // N) adds to dG_i and subtracts from dG_j, so it reaches dg_t exactly
        // when i >= t > j; a term c_i of the output state's e^{G_L - G_i}
        // (Crow) reaches it when i < t; e^{G_L} S's reaches every t. Summing
        // just those sets, rather than suffix sums of row minus column sums
        // in which the pairs inside [t, L] cancel only up to rounding, keeps
        // dg accurate relative to its own size: dg_t = sum_{i >= t} (S[i][t] +
        // the terms of e^{G_i} alone) + sum_{i < t} c_i + the e^{G_L} term.
        // Token t's eight threads take rows s, s + 8, s + 16 and s + 24.
        lds_barrier();
        {
            float x = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = s + 8 * e;
                x += r >= i ? L.S[r * MS + i] + L.Grow[r] : L.Crow[r];
            }
            x = row8_sum(x) + egl * gsd;
            if constexpr (TRUNC) x += trg[chn * GC + i];
            if (s == 0 && valid) dg[tok * p.hv + h] = x;
        }
    }

#undef TT_CHUNK_COORDS
    // The product terms join the element-wise ones through J, dq^ then dk^.
    auto join = [&](const f32x4 (&m)[2][2], float (&a)[16]) {
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int v = 0; v < 4; ++v) L.J[(16 * tb + g4 + v) * RS + w0 + 16 * cb + c16] = m[tb][cb][v];
        lds_barrier();
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const f32x4 x = *(const f32x4*)&L.J[i * RS + 32 * n + 4 * s];
#pragma unroll
            for (int e = 0; e < 4; ++e) a[4 * n + e] += x[e];
        }
        lds_barrier();
    };
    join(dqm, dqa);
    join(dkm, dka);

    // Through q^ = scale q / sqrt(|q|^2 + eps) and k^ = k / sqrt(|k|^2 + eps).
    if (valid) {
        const TIn* qr = (const TIn*)p.q + tok * p.q_st + (int64_t)hk * p.q_sh;
        const TIn* kr = (const TIn*)p.k + tok * p.k_st + (int64_t)hk * p.k_sh;
        f32x4 qv[4], kv[4];
        float sq = 0.0f, sk = 0.0f, dq_dot = 0.0f, dk_dot = 0.0f;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            qv[m] = load4(qr + 32 * m + 4 * s);
            kv[m] = load4(kr + 32 * m + 4 * s);
            sq += dot4(qv[m], qv[m]);
            sk += dot4(kv[m], kv[m]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dq_dot = fmaf(qv[m][e], dqa[4 * m + e], dq_dot);
                dk_dot = fmaf(kv[m][e], dka[4 * m + e], dk_dot);
            }
        }
        sq = row8_sum(sq);
        sk = row8_sum(sk);
        dq_dot = row8_sum(dq_dot);
        dk_dot = row8_sum(dk_dot);
        float aq = p.scale, bq = 0.0f, ak = 1.0f, bk = 0.0f;
        if (p.l2) {
            const float rq = 1.0f / sqrtf(sq + 1e-6f), rk = 1.0f / sqrtf(sk + 1e-6f);
            aq = p.scale * rq;
            bq = -p.scale * rq * rq * rq * dq_dot;
            ak = rk;
            bk = -rk * rk * rk * dk_dot;
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            f32x4 oq, ok;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                oq[e] = fmaf(aq, dqa[4 * m + e], bq * qv[m][e]);
                ok[e] = fmaf(ak, dka[4 * m + e], bk * kv[m][e]);
            }
            store4(dq + tok * p.dq_st + hk * GD + 32 * m + 4 * s, oq);
            store4(dk + tok * p.dk_st + hk * GD + 32 * m + 4 * s, ok);
        }
    }
}

}  // namespace

// Float counts per (chunk, v head) of the truncated mode's node-level terms:
// the node-level decay [32] and R (beta [v | e^G k]) rows [32 x 256].
constexpr size_t kTrGn = GC, kTrY1 = (size_t)GC * 2 * GD;

size_t tt_gdn_ws_bytes_impl(int n_chunks, int n_heads_v, bool trunc) {
    return (size_t)n_chunks * (size_t)n_heads_v * (kWsChunk + (trunc ? kTrGn + kTrY1 : 0)) * sizeof(float);
}

namespace {
constexpr int kMaxGridY = 65535;   // grid y limit: a level's nodes beyond it go to further launches


template <typename TIn, bool TRUNC>
void launch_prep(const GdnDev& d, float* prep, hipStream_t s) {
    hipLaunchKernelGGL((gdn_prep_kernel<TIn, TRUNC>), dim3(d.n_chunks, d.hv), dim3(GT), 0, s, d, prep);
}
// A level of n nodes runs in the row layout when the column
// layout would leave most of the chip idle: at most TT_GDN_ROWS_MAX_PAIRS
// (node, v head) pairs, two column workgroups each. On the 16K agent tree (32
// v heads) 64 pairs (levels of one or two nodes) timed best: 5.60 -> 5.40 ms
// per step, against 5.43 ms for 128 and for 256. The truncated rule on a
// 4,096-token tree (16 v heads): scans of both directions 863 -> 710 us with it.
#ifndef TT_GDN_ROWS_MAX_PAIRS
#define TT_GDN_ROWS_MAX_PAIRS 64
#endif
bool use_rows(const GdnDev& d, int n) { return (int64_t)n * d.hv <= TT_GDN_ROWS_MAX_PAIRS; }

template <typename TIn, bool TRUNC>
void launch_scan(const GdnDev& d, int b, int n, float* prep, TIn* out, float* states, float* sin, float* vp,
                 hipStream_t s) {
    // grid (v head x column block, node): all heads of a level's first
    // (longest) nodes are dispatched first. Packed tiles where a CU has more
    // than one workgroup to run; with one, padded ones are the faster (fp32,
    // 2,075 tokens, 8 v heads, up to 192 workgroups: 166 us against 168).
    constexpr bool can_pack = kScanPacked<TIn, TRUNC>;
    const bool pack = can_pack && (int64_t)n * d.hv * kScanSplit > 256;
    for (int b0 = 0; b0 < n; b0 += kMaxGridY) {
        const dim3 cols(d.hv * kScanSplit, min(kMaxGridY, n - b0));
        if (use_rows(d, n))
            hipLaunchKernelGGL((gdn_scan_rows_kernel<TIn, TRUNC>), dim3(d.hv * kRowsSplit, min(kMaxGridY, n - b0)),
                               dim3(GT), 0, s, d, b + b0, prep, out, states, sin, vp);
        else if (pack)
            hipLaunchKernelGGL((gdn_scan_cols_kernel<TIn, TRUNC, can_pack>), cols, dim3(GT), 0, s, d, b + b0, prep,
                               out, states, sin, vp);
        else
            hipLaunchKernelGGL((gdn_scan_cols_kernel<TIn, TRUNC, false>), cols, dim3(GT), 0, s, d, b + b0, prep, out,
                               states, sin, vp);
    }
}

// The forward: chunk terms (prep; TRUNC: plus the node-level U, W), then one
// scan launch per tree level. gn, y1: TRUNC scratch.
template <typename TIn, bool TRUNC>
int gdn_forward(const GdnDev& d, const int32_t* level_offsets, int n_levels, TIn* out, float* states, float* prep,
                float* sin, float* vp, float* gn, float* y1, hipStream_t s) {
    launch_prep<TIn, TRUNC>(d, prep, s);
    if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    if constexpr (TRUNC) {
        const int rc = tt_gdn_trunc_fwd_launch(d, prep, gn, y1, s);
        if (rc != TT_OK) return rc;
    }
    for (int l = 0; l < n_levels; ++l) {
        const int b = level_offsets[l], n = level_offsets[l + 1] - b;
        if (n <= 0) continue;
        launch_scan<TIn, TRUNC>(d, b, n, prep, out, states, sin, vp, s);
        if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    }
    return TT_OK;
}

template <typename TIn>
int gdn_forward_any(const GdnDev& d, const int32_t* level_offsets, int n_levels, TIn* out, float* states,
                    float* prep, float* sin, float* vp, float* gn, float* y1, hipStream_t s) {
    return d.trunc ? gdn_forward<TIn, true>(d, level_offsets, n_levels, out, states, prep, sin, vp, gn, y1, s)
                   : gdn_forward<TIn, false>(d, level_offsets, n_levels, out, states, prep, sin, vp, gn, y1, s);
}
}  // namespace

int tt_gdn_fwd_launch(const GdnDev& d, const int32_t* level_offsets, int n_levels, void* out, float* states,
                      float* ws, hipStream_t s) {
    const size_t ch = (size_t)d.n_chunks * d.hv;
    float* gn = ws + ch * kWsChunk;
    float* y1 = gn + ch * kTrGn;
    if (d.dtype == TT_DTYPE_BF16)
        return gdn_forward_any<__bf16>(d, level_offsets, n_levels, (__bf16*)out, states, ws, nullptr, nullptr, gn,
                                       y1, s);
    return gdn_forward_any<float>(d, level_offsets, n_levels, (float*)out, states, ws, nullptr, nullptr, gn, y1, s);
}

// The backward's float buffers. "Saved" (what the forward can keep for it):
// per (chunk, v head) the prep terms [kWsChunk], the chunk's initial state S
// [128 x 128] and V' [32 x 128]; TRUNC: also the node-level decay [32] and
// R-rows y1 [32 x 256]. Scratch: per (chunk, v head) dS [128 x 128], dV', X,
// dW, dK~ [32 x 128]; TRUNC: dF1, dY0 [32 x 256], the correction's dk^
// [32 x 128] and dG [32]; per (node, v head) dS at entry [128 x 128]; when the
// backward recomputes the forward, the node states [128 x 128]; <S, dS> per
// (chunk, v head) last (it breaks 16-byte alignment).
namespace {
struct GdnBwdWs {
    float *prep, *sin, *vp, *gn, *y1, *dso, *dvp, *x, *dw, *dkt, *df1, *dy0, *dkr, *dgn, *dsn, *nstate, *sdot;
};
size_t gdn_saved_floats(size_t ch, bool trunc) {
    return ch * (kWsChunk + GD * GD + GC * GD + (trunc ? kTrGn + kTrY1 : 0));
}
size_t gdn_scratch_floats(size_t ch, size_t nd, bool recompute, bool trunc) {
    return ch * (GD * GD + 4 * GC * GD + 1 + (trunc ? 2 * kTrY1 + GC * GD + GC : 0)) +
           nd * GD * GD * (recompute ? 2 : 1);
}
GdnBwdWs gdn_bwd_carve(float* saved, float* scratch, size_t n_chunks, size_t n_nodes, size_t hv, bool recompute,
                       bool trunc) {
    const size_t ch = n_chunks * hv, nd = n_nodes * hv;
    GdnBwdWs w = {};
    float* q = saved;
    w.prep = q; q += ch * kWsChunk;
    w.sin = q; q += ch * GD * GD;
    w.vp = q; q += ch * GC * GD;
    if (trunc) {
        w.gn = q; q += ch * kTrGn;
        w.y1 = q; q += ch * kTrY1;
    }
    q = scratch;
    if (!q) return w;
    w.dso = q; q += ch * GD * GD;
    w.dvp = q; q += ch * GC * GD;
    w.x = q; q += ch * GC * GD;
    w.dw = q; q += ch * GC * GD;
    w.dkt = q; q += ch * GC * GD;
    if (trunc) {
        w.df1 = q; q += ch * kTrY1;
        w.dy0 = q; q += ch * kTrY1;
        w.dkr = q; q += ch * GC * GD;
        w.dgn = q; q += ch * GC;
    }
    w.dsn = q; q += nd * GD * GD;
    w.nstate = nullptr;
    if (recompute) { w.nstate = q; q += nd * GD * GD; }
    w.sdot = q;
    return w;
}
}  // namespace

size_t tt_gdn_saved_bytes_impl(int n_chunks, int n_heads_v, bool trunc) {
    return gdn_saved_floats((size_t)n_chunks * n_heads_v, trunc) * sizeof(float);
}
size_t tt_gdn_bwd_ws_bytes_impl(int n_chunks, int n_nodes, int n_heads_v, bool recompute, bool trunc) {
    const size_t ch = (size_t)n_chunks * n_heads_v, nd = (size_t)n_nodes * n_heads_v;
    return ((recompute ? gdn_saved_floats(ch, trunc) : 0) + gdn_scratch_floats(ch, nd, recompute, trunc)) *
           sizeof(float);
}

int tt_gdn_fwd_save_launch(const GdnDev& d, const int32_t* level_offsets, int n_levels, void* out, float* states,
                           float* saved, hipStream_t s) {
    const GdnBwdWs w = gdn_bwd_carve(saved, nullptr, d.n_chunks, d.n_nodes, d.hv, false, d.trunc);
    if (d.dtype == TT_DTYPE_BF16)
        return gdn_forward_any<__bf16>(d, level_offsets, n_levels, (__bf16*)out, states, w.prep, w.sin, w.vp, w.gn,
                                       w.y1, s);
    return gdn_forward_any<float>(d, level_offsets, n_levels, (float*)out, states, w.prep, w.sin, w.vp, w.gn, w.y1,
                                  s);
}

// saved == nullptr: recompute the forward into the front of ws; otherwise
// saved holds what tt_gdn_fwd_save_launch wrote for the same problem.
template <typename TIn, bool TRUNC>
static int gdn_bwd_run(const GdnDev& d, const int32_t* level_offsets, int n_levels, const TIn* d_o, int64_t do_st,
                       int64_t do_sh, TIn* dq, TIn* dk, TIn* dv, float* dg, float* dbeta, const float* saved,
                       float* ws, hipStream_t s) {
    const bool recompute = saved == nullptr;
    float* sv = recompute ? ws : const_cast<float*>(saved);
    float* scratch = recompute ? ws + gdn_saved_floats((size_t)d.n_chunks * d.hv, TRUNC) : ws;
    const GdnBwdWs w = gdn_bwd_carve(sv, scratch, d.n_chunks, d.n_nodes, d.hv, recompute, TRUNC);
    if (recompute) {
        const int rc = gdn_forward<TIn, TRUNC>(d, level_offsets, n_levels, (TIn*)nullptr, w.nstate, w.prep, w.sin,
                                               w.vp, w.gn, w.y1, s);
        if (rc != TT_OK) return rc;
    }
    for (int l = n_levels - 1; l >= 0; --l) {
        const int b = level_offsets[l], n = level_offsets[l + 1] - b;
        if (n <= 0) continue;
        for (int b0 = 0; b0 < n; b0 += kMaxGridY) {
            if (use_rows(d, n))
                hipLaunchKernelGGL((gdn_rscan_rows_kernel<TIn, TRUNC>), dim3(d.hv * kRowsSplit, min(kMaxGridY, n - b0)),
                                   dim3(GT), 0, s, d, b + b0, w.prep, d_o, do_st, do_sh, w.dso, w.dvp, w.dsn);
            else
                hipLaunchKernelGGL((gdn_rscan_cols_kernel<TIn, TRUNC>),
                                   dim3(d.hv * kScanSplit, min(kMaxGridY, n - b0)), dim3(GT), 0, s, d, b + b0,
                                   w.prep, d_o, do_st, do_sh, w.dso, w.dvp, w.dsn);
        }
        if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    }
    if (d.d_init) {
        static_assert(GD * GD % (4 * GT) == 0, "one f32x4 per thread");
        hipLaunchKernelGGL(gdn_init_grad_kernel, dim3(GD * GD / (4 * GT), d.hv), dim3(GT), 0, s, d, w.dsn);
        if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    }
    hipLaunchKernelGGL(gdn_bwd_state_kernel<TIn>, dim3(d.n_chunks, d.hv), dim3(GT), 0, s, d, d_o, do_st, do_sh,
                       w.sin, w.dso, w.vp, w.dvp, w.x, w.dw, w.dkt, w.sdot);
    if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    if constexpr (TRUNC) {
        hipLaunchKernelGGL(gdn_dw_s0_kernel, dim3(d.n_chunks, d.hv), dim3(GT), 0, s, d, w.sin, w.dvp, w.dw);
        const GdnTruncBwd tb{w.prep, w.gn, w.y1, w.dvp, w.dw, w.df1, w.dy0, w.dkr, w.dgn};
        const int rc = tt_gdn_trunc_bwd_launch(d, tb, dv, dbeta, s);
        if (rc != TT_OK) return rc;
    }
    hipLaunchKernelGGL((gdn_bwd_chunk_kernel<TIn, TRUNC>), dim3(d.n_chunks, d.hk), dim3(GT), 0, s, d, d_o, do_st,
                       do_sh, w.prep, w.vp, w.dvp, w.x, w.dw, w.dkt, w.sdot, dq, dk, dv, dg, dbeta, w.dkr, w.dgn);
    if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    return TT_OK;
}

template <typename TIn>
static int gdn_bwd_any(const GdnDev& d, const int32_t* level_offsets, int n_levels, const TIn* d_o, int64_t do_st,
                       int64_t do_sh, TIn* dq, TIn* dk, TIn* dv, float* dg, float* dbeta, const float* saved,
                       float* ws, hipStream_t s) {
    return d.trunc ? gdn_bwd_run<TIn, true>(d, level_offsets, n_levels, d_o, do_st, do_sh, dq, dk, dv, dg, dbeta,
                                            saved, ws, s)
                   : gdn_bwd_run<TIn, false>(d, level_offsets, n_levels, d_o, do_st, do_sh, dq, dk, dv, dg, dbeta,
                                             saved, ws, s);
}

int tt_gdn_bwd_launch(const GdnDev& d, const int32_t* level_offsets, int n_levels, const void* d_o, int64_t do_st,
                      int64_t do_sh, void* dq, void* dk, void* dv, float* dg, float* dbeta, const float* saved,
                      float* ws, hipStream_t s) {
    if (d.dtype == TT_DTYPE_BF16)
        return gdn_bwd_any<__bf16>(d, level_offsets, n_levels, (const __bf16*)d_o, do_st, do_sh, (__bf16*)dq,
                                   (__bf16*)dk, (__bf16*)dv, dg, dbeta, saved, ws, s);
    return gdn_bwd_any<float>(d, level_offsets, n_levels, (const float*)d_o, do_st, do_sh, (float*)dq, (float*)dk,
                              (float*)dv, dg, dbeta, saved, ws, s);
}
