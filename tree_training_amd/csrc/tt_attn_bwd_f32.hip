// Tree-masked GQA attention backward for fp32 models (operands split into bf16
// planes; see tt_f32_tiles.h): delta, dQ (query-major) and dK/dV (key-major).
#include "tt_f32_tiles.h"

namespace {

// delta = rowsum(dO * O), one row per 16 threads (when TT_BWD_DELTA runs
// without TT_BWD_DQ; otherwise the dQ pass computes it).
__global__ __launch_bounds__(256) void bwd_delta_f32_kernel(AttnDev a, BwdDev b) {
    const int row = blockIdx.x * 16 + (threadIdx.x >> 4), sub = threadIdx.x & 15;
    const int total = a.n_q * a.hq;
    float acc = 0.0f;
    int i = 0, h = 0;
    if (row < total) {
        i = row / a.hq;
        h = row - i * a.hq;
        const float* op = (const float*)b.o + ((size_t)i * a.hq + h) * D + 8 * sub;
        const float* dp = (const float*)b.dout + i * b.do_st + h * b.do_sh + 8 * sub;
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const f32x4 ov = *(const f32x4*)(op + e), dv = *(const f32x4*)(dp + e);
            acc += ov[0] * dv[0] + ov[1] * dv[1] + ov[2] * dv[2] + ov[3] * dv[3];
        }
    }
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) acc += __shfl_xor(acc, o);
    if (row < total && sub == 0) b.delta[(size_t)h * a.n_q + i] = acc;
}

// dQ: per 32-key step, S^T and dP^T, dS^T = P^T (dP^T - delta), then
// dQ^T += K^T dS^T. Bound by the matrix cores (144 MFMAs, 4608 cycles, a wave
// and step); while S and dP of step s + 1 run, dS of step s is formed and
// split and step s + 2's keys and values are split. FUSE_DELTA: delta of the
// rows is computed here (and stored for the dK/dV pass) instead of read.
// 16,318-token agent tree, 32/8 heads: 5.95 -> 3.80 ms (1.09 PFLOP/s of plane
// products) against fp32 MFMAs; 4.16 before dS and the splits moved behind the
// MFMAs.
struct DqStageF {
    bf16 K[3][3 * PLANE];   // step s in K[s % 3]: read as rows in step s - 1, transposed in step s
    bf16 V[2][3 * PLANE];   // step s in V[s & 1], read in step s - 1
    Bounds32Ring bnd;
    bf16x8 dlow[4 * 8 * 64];   // dO's third plane, each lane's own (the registers it would take spill)
};

template <bool FUSE_DELTA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_dq_f32_kernel(AttnDev a,
                                                                                                   BwdDev bw) {
    __shared__ __attribute__((aligned(16))) DqStageF st;

    int qb, h;
    decode_qblock(a, qb, h);
    const int g = __builtin_amdgcn_readfirstlane(h / a.rep);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int col = lane & 31, half = lane >> 5;
    const int q0 = qb * TT_BQ + wave * 32, qi = q0 + col;
    const bool valid = qi < a.n_q;
    const int qr = min(qi, a.n_q - 1);
    const float c = a.scale * TT_LOG2E;
    const RowOffsG kro = row_offsg(col, half);
    const TrOffsG tro = tr_offsg(lane);

    Planes q[8], dov[8];
    load_row_planes((const float*)a.q + (int64_t)qr * a.q_st + h * a.q_sh, valid, half, q);
    const float* drow = (const float*)bw.dout + (int64_t)qr * bw.do_st + h * bw.do_sh;
    load_row_planes(drow, valid, half, dov);
    bf16x8* const dl = st.dlow + wave * 512 + lane;
#pragma unroll
    for (int t = 0; t < 8; ++t) dl[64 * t] = dov[t].l;
    float lse2 = INFINITY, dlt = 0.0f;
    if (valid) {
        lse2 = bw.lse[(size_t)h * a.n_q + qi] * TT_LOG2E;
        if constexpr (FUSE_DELTA) {
            const float* orow = (const float*)bw.o + ((size_t)qi * a.hq + h) * D;
            float acc = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int d = 16 * (i >> 1) + 8 * half + 4 * (i & 1);
                const f32x4 ov = *(const f32x4*)(orow + d), dv = *(const f32x4*)(drow + d);
                acc += ov[0] * dv[0] + ov[1] * dv[1] + ov[2] * dv[2] + ov[3] * dv[3];
            }
            dlt = acc;
        } else {
            dlt = bw.delta[(size_t)h * a.n_q + qi];
        }
    }
    if constexpr (FUSE_DELTA) {
        dlt = halves_sum(dlt);
        if (valid && half == 0) bw.delta[(size_t)h * a.n_q + qi] = dlt;
    }

    const KvWalkF w(a, qb);
    RowsF kr, vr;
    Bounds32 nb;
    f32x16 dq[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) dq[i] = (f32x16){};
    f32x16 sc = {}, dp = {};   // scores and dP of the running step
    bool vis = false;
    // S^T and dP^T of a step (planes K, V) with work(IntT<j>) behind its j-th MFMA, j < 96
    auto scores = [&](const bf16* K, const bf16* V, f32x16& s, f32x16& d, auto&& work) {
        Planes k[2], v[2];
        bf16x8 low[2];
        k[0] = read_row_planes<0>(K, kro);
        v[0] = read_row_planes<0>(V, kro);
        low[0] = dl[0];
        static_for<8>([&](auto tt) {
            constexpr int t = decltype(tt)::value;
            if constexpr (t + 1 < 8) {
                k[(t + 1) & 1] = read_row_planes<t + 1>(K, kro);
                v[(t + 1) & 1] = read_row_planes<t + 1>(V, kro);
                low[(t + 1) & 1] = dl[64 * (t + 1)];
            }
            mfma_split2(k[t & 1], q[t], s, v[t & 1], Planes{dov[t].h, dov[t].m, low[t & 1]}, d,
                        [&](auto ii) { work(IntT<12 * t + decltype(ii)::value>{}); });
        });
    };
    if (w.n > 0) {   // the walk has two steps per listed tile: w.n >= 2
        const int k0 = w.key0(0), k1 = w.key0(1), k2 = w.key0(min(2, w.n - 1));
        load_keys(a, k0, g, false, kr);
        load_keys(a, k0, g, true, vr);
        nb.load(a, k0);
        store_rows_f(kr, st.K[0]);
        store_rows_f(vr, st.V[0]);
        nb.store(st.bnd, 0);
        load_keys(a, k1, g, false, kr);
        load_keys(a, k1, g, true, vr);
        nb.load(a, k1);
        store_rows_f(kr, st.K[1]);
        store_rows_f(vr, st.V[1]);
        nb.store(st.bnd, 1);
        load_keys(a, k2, g, false, kr);
        load_keys(a, k2, g, true, vr);
        nb.load(a, k2);
        lds_barrier();
        vis = (w.entry(0) & 1) || step_visible(st.bnd, 0, q0, lane);
        if (vis) scores(st.K[0], st.V[0], sc, dp, NoWork{});
        lds_barrier();   // V[0] is written again in step 0
    }
    int b0 = 0;   // s % 3
    for (int s = 0; s < w.n; ++s) {
        const bool full = w.entry(s) & 1;
        const int s1 = min(s + 1, w.n - 1);
        const bool vis_next = s + 1 < w.n && ((w.entry(s1) & 1) || step_visible(st.bnd, s1, q0, lane));
        const int k3 = w.key0(min(s + 3, w.n - 1));
        const int b1 = b0 == 2 ? 0 : b0 + 1, b2 = b1 == 2 ? 0 : b1 + 1;
        if (vis && !full) mask_half(sc, st.bnd.lo[s & 3], st.bnd.hi[s & 3], qi, half);
        // Work slots: 0 .. 15 dS, 16 .. 31 its split, 32 .. 75 the split of step s + 2's keys and values.
        Split8 ds0, ds1;
        StoreRows k_lo(kr, 0, st.K[b2]), k_hi(kr, 1, st.K[b2]), v_lo(vr, 0, st.V[s & 1]), v_hi(vr, 1, st.V[s & 1]);
        auto slot = [&](auto jj) {
            constexpr int j = decltype(jj)::value;
            if constexpr (j < 16) sc[j] = fast_exp2(fmaf(sc[j], c, -lse2)) * (dp[j] - dlt);   // dS^T
            if constexpr (j == 16) ds0 = split_begin(sc, 0);
            if constexpr (j >= 16 && j < 24) ds0.slice<j - 16>();
            if constexpr (j == 24) ds1 = split_begin(sc, 8);
            if constexpr (j >= 24 && j < 32) ds1.slice<j - 24>();
            if constexpr (j >= 32 && j < 43) k_lo.slice<j - 32>();
            if constexpr (j >= 43 && j < 54) k_hi.slice<j - 43>();
            if constexpr (j >= 54 && j < 65) v_lo.slice<j - 54>();
            if constexpr (j >= 65 && j < 76) v_hi.slice<j - 65>();
        };
        f32x16 sn = {}, dn = {};
        if (vis_next)
            scores(st.K[b1], st.V[(s + 1) & 1], sn, dn, slot);
        else
            static_for<76>([&](auto jj) { slot(jj); });
        load_keys(a, k3, g, false, kr);
        load_keys(a, k3, g, true, vr);
        if (vis) {
            const bf16* K = st.K[b0];
            const Planes ds[2] = {ds0.planes(), ds1.planes()};
            Planes kt[4];
            kt[0] = read_tr_planes(K, tro, 0, 0);
            kt[1] = read_tr_planes(K, tro, 0, 1);
            static_for<4>([&](auto uu) {
                constexpr int u = decltype(uu)::value, d0 = 2 * (u & 1), n = u + 1, n0 = 2 * (n & 1);
                if constexpr (u < 3) {
                    kt[n0] = read_tr_planes(K, tro, 16 * (n >> 1), n0);
                    kt[n0 + 1] = read_tr_planes(K, tro, 16 * (n >> 1), n0 + 1);
                }
                mfma_split2(kt[d0], ds[u >> 1], dq[d0], kt[d0 + 1], ds[u >> 1], dq[d0 + 1]);
            });
        }
        nb.store(st.bnd, s + 2);
        nb.load(a, k3);
        sc = sn;
        dp = dn;
        vis = vis_next;
        b0 = b1;
        lds_barrier();
    }

    if (valid) {
        float* op = (float*)bw.dq + ((size_t)qi * a.hq + h) * D;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                f32x4 wv;
#pragma unroll
                for (int e = 0; e < 4; ++e) wv[e] = dq[db][4 * grp + e] * a.scale;
                *(f32x4*)(op + 32 * db + 8 * grp + 4 * half) = wv;
            }
    }
}

// ----------------------------------------------------------------------------
// dK, dV (key-major, persistent over the plan's work items). Bound by the
// matrix cores: 192 MFMAs (6144 cycles) a wave and 32-query step. Starting
// the next step's S and dP early, as the dQ pass does, would take 32 more
// registers than the wave has.
// 16,318-token agent tree, 32/8 heads: 9.24 -> 4.68 ms (1.18 PFLOP/s of plane
// products) against fp32 MFMAs.
// ----------------------------------------------------------------------------
struct QStageF {
    bf16 Q[3 * PLANE];
    bf16 Dn[3 * PLANE];
    float lse[TT_BQB];    // log2 units
    float ndlt[TT_BQB];   // -delta
};

// A 32-query block of head h: its Q and dO rows (rows past n_q alias the last
// query; their lse is +inf), its lse (wave 0) and delta (wave 1).
struct QBlockF {
    RowsF q, d;
    float sv;
    int q0;
    __device__ __forceinline__ void load(const AttnDev& a, const BwdDev& bw, int q0_, int h) {
        q0 = q0_;
        if (q0 + TT_BQB <= a.n_q) {
            q.load_buf((const float*)a.q + (int64_t)q0 * a.q_st + h * a.q_sh, 4u * (uint32_t)a.q_st);
            d.load_buf((const float*)bw.dout + (int64_t)q0 * bw.do_st + h * bw.do_sh, 4u * (uint32_t)bw.do_st);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int64_t qq = min(q0 + (int)(threadIdx.x >> 4) + 16 * i, a.n_q - 1);
                q.load_row(i, (const float*)a.q + qq * a.q_st + h * a.q_sh);
                d.load_row(i, (const float*)bw.dout + qq * bw.do_st + h * bw.do_sh);
            }
        }
        const int wave = threadIdx.x >> 6;
        if (wave < 2) {
            const float* src = (wave == 0 ? bw.lse : bw.delta) + (size_t)h * a.n_q;
            sv = src[min(q0 + (int)(threadIdx.x & 31), a.n_q - 1)];
        }
    }
    __device__ __forceinline__ void store_stats(const AttnDev& a, QStageF& S) const {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        if (wave < 2 && lane < TT_BQB) {
            const bool in = q0 + lane < a.n_q;
            if (wave == 0) S.lse[lane] = in ? sv * TT_LOG2E : INFINITY;
            else S.ndlt[lane] = in ? -sv : 0.0f;
        }
    }
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_dkdv_f32_kernel(AttnDev a,
                                                                                                     BwdDev bw) {
    __shared__ __attribute__((aligned(16))) QStageF St[2];
    __shared__ bf16x8 vlow[4 * 8 * 64];   // V's third plane, each lane's own (the registers it would take spill)

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int col = lane & 31, half = lane >> 5;
    const float c = a.scale * TT_LOG2E;
    const RowOffsG qro = row_offsg(col, half);
    const TrOffsG tro = tr_offsg(lane);
    const int n_work = (*a.n_items) * a.hkv;

    for (int w_id = blockIdx.x; w_id < n_work; w_id += gridDim.x) {
        const int g = __builtin_amdgcn_readfirstlane(w_id % a.hkv);
        const int item = __builtin_amdgcn_readfirstlane(w_id / a.hkv);
        const int2 rc = a.kb_item[item];           // (tile rank, chunk): the plan's item order
        const int lo_r = __builtin_amdgcn_readfirstlane(rc.x);
        const int chunk = __builtin_amdgcn_readfirstlane(rc.y);
        const int kb = __builtin_amdgcn_readfirstlane(a.kb_order[lo_r]);
        // a later item's slot: the tile's items before it that are not its
        // first, after those of the tiles ranked before it
        const int64_t slot = (int64_t)a.kb_base[lo_r] - lo_r + chunk - 1;
        const int qlo = __builtin_amdgcn_readfirstlane(a.kb_qlo[kb]);
        const int qhi = __builtin_amdgcn_readfirstlane(a.kb_qhi[kb]);
        const int qch = tt_qch(a.n_q);
        const bool split = tt_kb_items(qlo, qhi, qch) > 1;
        int q_start, q_stop;
        tt_kb_item_range(qlo, qhi, qch, chunk, q_start, q_stop);
        // a tile of gateway keys that no query sees adds nothing anywhere
        if (q_stop <= q_start && kb * TT_BKB + TT_BKB <= a.n_past) continue;

        const int kk = kb * TT_BKB + wave * 32 + col;   // this lane's key
        int lo = 0, hi = 0;
        Planes kr[8], vr[8];   // K and V of the lane's key
        load_row_planes(key_row_f(a, min(kk, a.n_keys - 1), g, false), kk < a.n_keys, half, kr);
        load_row_planes(key_row_f(a, min(kk, a.n_keys - 1), g, true), kk < a.n_keys, half, vr);
        bf16x8* const vl = vlow + wave * 512 + lane;
#pragma unroll
        for (int t = 0; t < 8; ++t) vl[64 * t] = vr[t].l;
        if (kk < a.n_keys) {
            lo = max(a.key_lo[kk], 0);
            hi = min(a.key_hi[kk], a.n_q);
        }
        if (lo >= hi) { lo = a.n_q; hi = 0; }
        const unsigned vis_w = (unsigned)(hi - lo);
        const int w_lo = wave_min_i(lo), w_hi = wave_max_i(hi);
        const int w_maxlo = wave_max_i(lo < hi ? lo : -1), w_minhi = wave_min_i(lo < hi ? hi : -1);
        const bool w_all_vis = wave_min_i((kk < a.n_keys && lo < hi) ? 1 : 0) == 1;

        f32x16 dk[4], dv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) { dk[i] = (f32x16){}; dv[i] = (f32x16){}; }

        const int q_top = (q_stop > q_start) ? ((q_stop - 1) / TT_BQB) * TT_BQB : 0;
        const int n_steps = (q_stop > q_start) ? ((q_top - q_start) / TT_BQB + 1) * a.rep : 0;
        // step s covers query block q0 of q head g * rep + hh; (qn, hn): the block loaded next
        QBlockF blk;
        int q0 = q_top, qn = q_top, hn = 0;
        auto advance = [&] {
            if (++hn == a.rep) {
                hn = 0;
                qn = max(qn - TT_BQB, 0);
            }
        };
        int hh = 0;
        if (n_steps > 0) {
            blk.load(a, bw, qn, g * a.rep);
            store_rows_f(blk.q, St[0].Q);
            store_rows_f(blk.d, St[0].Dn);
            blk.store_stats(a, St[0]);
            advance();
            blk.load(a, bw, qn, g * a.rep + hn);
            lds_barrier();
        }
        for (int s = 0; s < n_steps; ++s) {
            const QStageF& S = St[s & 1];
            QStageF& N = St[(s + 1) & 1];   // last read in step s - 1
            const int q0_cur = q0, q1 = min(q0_cur + TT_BQB, a.n_q);
            if (++hh == a.rep) {
                hh = 0;
                q0 -= TT_BQB;
            }
            blk.store_stats(a, N);
            advance();
            if (!((q0_cur < w_hi) && (q1 > w_lo))) {   // no key of this wave is seen here
                store_rows_f(blk.q, N.Q);
                store_rows_f(blk.d, N.Dn);
                blk.load(a, bw, qn, g * a.rep + hn);
                lds_barrier();
                continue;
            }
            const bool full = w_all_vis && (w_maxlo <= q0_cur) && (w_minhi >= q1);

            // S = Q K^T and dP = dO V^T: rows = queries, lane = key column.
            // Operands are read one group of twelve MFMAs ahead of their use;
            // the next block's rows are split behind the first 44 MFMAs.
            f32x16 sc = {}, dp = {};
            Planes qp[2], dn[2];
            bf16x8 low[2];
            StoreRows q_lo(blk.q, 0, N.Q), q_hi(blk.q, 1, N.Q), d_lo(blk.d, 0, N.Dn), d_hi(blk.d, 1, N.Dn);
            qp[0] = read_row_planes<0>(S.Q, qro);
            dn[0] = read_row_planes<0>(S.Dn, qro);
            low[0] = vl[0];
            static_for<8>([&](auto tt) {
                constexpr int t = decltype(tt)::value;
                if constexpr (t + 1 < 8) {
                    qp[(t + 1) & 1] = read_row_planes<t + 1>(S.Q, qro);
                    dn[(t + 1) & 1] = read_row_planes<t + 1>(S.Dn, qro);
                    low[(t + 1) & 1] = vl[64 * (t + 1)];
                }
                mfma_split2(qp[t & 1], kr[t], sc, dn[t & 1], Planes{vr[t].h, vr[t].m, low[t & 1]}, dp, [&](auto ii) {
                    constexpr int j = 12 * t + decltype(ii)::value;
                    if constexpr (j < 11) q_lo.slice<j>();
                    if constexpr (j >= 11 && j < 22) q_hi.slice<j - 11>();
                    if constexpr (j >= 22 && j < 33) d_lo.slice<j - 22>();
                    if constexpr (j >= 33 && j < 44) d_hi.slice<j - 33>();
                });
            });
            blk.load(a, bw, qn, g * a.rep + hn);
            unsigned seen = 0xffffu;   // bit r: accumulator row r's query sees the lane's key
            if (!full) {
                seen = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    seen |= (unsigned)(q0_cur + acc_row(r, half) - lo) < vis_w ? 1u << r : 0u;
            }
            // P and dS of row r; a mask over the bits, so that an overflowing
            // exp of an invisible score never propagates
            f32x4 l2[4], nd[4];
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                l2[grp] = *(const f32x4*)(S.lse + 8 * grp + 4 * half);
                nd[grp] = *(const f32x4*)(S.ndlt + 8 * grp + 4 * half);
            }
            auto row = [&](auto rr) {
                constexpr int r = decltype(rr)::value;
                const unsigned keep = (unsigned)__builtin_amdgcn_sbfe((int)seen, r, 1);
                const float p = fast_exp2(fmaf(sc[r], c, -l2[r >> 2][r & 3]));
                const float d = p * (dp[r] + nd[r >> 2][r & 3]);
                sc[r] = __uint_as_float(__float_as_uint(p) & keep);
                dp[r] = __uint_as_float(__float_as_uint(d) & keep);
            };
            static_for<8>([&](auto rr) { row(rr); });
            // dV += P^T dO, dK += dS^T Q: contraction over the 32 queries;
            // rows 8 .. 15 are formed behind the MFMAs of rows 0 .. 7.
            Planes pp[2], pd[2];
            dn[0] = read_tr_planes(S.Dn, tro, 0, 0);
            qp[0] = read_tr_planes(S.Q, tro, 0, 0);
            Split8 wp = split_begin(sc, 0), wd = split_begin(dp, 0);
            wp.all();
            wd.all();
            pp[0] = wp.planes();
            pd[0] = wd.planes();
            static_for<8>([&](auto uu) {
                constexpr int u = decltype(uu)::value, n = u + 1;
                if constexpr (n < 8) {
                    dn[n & 1] = read_tr_planes(S.Dn, tro, 16 * (n >> 2), n & 3);
                    qp[n & 1] = read_tr_planes(S.Q, tro, 16 * (n >> 2), n & 3);
                }
                mfma_split2(pp[u >> 2], dn[u & 1], dv[u & 3], pd[u >> 2], qp[u & 1], dk[u & 3], [&](auto ii) {
                    constexpr int j = 12 * u + decltype(ii)::value;
                    if constexpr (j < 8) row(IntT<8 + j>{});
                    if constexpr (j == 8) wp = split_begin(sc, 8);
                    if constexpr (j >= 8 && j < 16) wp.slice<j - 8>();
                    if constexpr (j == 16) wd = split_begin(dp, 8);
                    if constexpr (j >= 16 && j < 24) wd.slice<j - 16>();
                    if constexpr (j == 24) {
                        pp[1] = wp.planes();
                        pd[1] = wd.planes();
                    }
                });
            });
            lds_barrier();
        }

        // Epilogue: rows of dk/dv = this wave's keys, columns = d (as the bf16 pass).
        const bool det_split = split && bw.det;
        // a split tile's rows in the split sums (first items) and a later item's
        // slot: one that lies beyond the workspace writes nothing (the tile's
        // gradients become NaN in the finalize)
        const SplitRows sr = split ? split_rows(a, bw, kb) : SplitRows{0, false};
        const bool det_skip = det_split && (chunk > 0 ? slot >= bw.det_cap : !sr.ok);
        float* const sk = chunk == 0 ? bw.dk_ws : bw.dk_slot;
        float* const sv = chunk == 0 ? bw.dv_ws : bw.dv_slot;
        const int64_t srow = chunk == 0 ? sr.row0 : slot * TT_BKB - kb * TT_BKB;
        const int kbase = kb * TT_BKB + wave * 32;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = kbase + acc_row(r, half);
            if (key >= a.n_keys || det_skip) continue;
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const int d = 32 * db + col;
                const float gk = dk[db][r] * a.scale, gv = dv[db][r];
                const size_t widx = ((size_t)key * a.hkv + g) * D + d;
                if (det_split) {
                    const size_t sidx = ((size_t)(srow + key) * a.hkv + g) * D + d;
                    sk[sidx] = gk;
                    sv[sidx] = gv;
                } else if (key < a.n_past) {
                    if (bw.dk_acc) {
                        if (split) {
                            atomicAdd(bw.dk_acc + widx, gk);
                            atomicAdd(bw.dv_acc + widx, gv);
                        } else {
                            bw.dk_acc[widx] += gk;
                            bw.dv_acc[widx] += gv;
                        }
                    }
                } else if (split) {
                    if (sr.ok) {
                        const size_t cidx = ((size_t)(sr.row0 + key) * a.hkv + g) * D + d;
                        atomicAdd(bw.dk_ws + cidx, gk);
                        atomicAdd(bw.dv_ws + cidx, gv);
                    }
                } else {
                    const size_t idx = ((size_t)(key - a.n_past) * a.hkv + g) * D + d;
                    ((float*)bw.dk)[idx] = gk;
                    ((float*)bw.dv)[idx] = gv;
                }
            }
        }
        __syncthreads();   // the stages are reused by the next item
    }
}

}  // namespace

int tt_bwd_f32_launch(const AttnDev& a, const BwdDev& b, hipStream_t s) {
    const bool fuse = (b.parts & TT_BWD_DELTA) && (b.parts & TT_BWD_DQ);
    if ((b.parts & TT_BWD_DELTA) && !fuse) {
        hipLaunchKernelGGL(bwd_delta_f32_kernel, dim3(tt_cdiv(a.n_q * a.hq, 16)), dim3(256), 0, s, a, b);
        if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    }
    if (b.parts & TT_BWD_DQ) {
        if (fuse)
            hipLaunchKernelGGL(bwd_dq_f32_kernel<true>, dim3(a.n_qb * a.hq), dim3(256), 0, s, a, b);
        else
            hipLaunchKernelGGL(bwd_dq_f32_kernel<false>, dim3(a.n_qb * a.hq), dim3(256), 0, s, a, b);
        if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    }
    if (b.parts & TT_BWD_DKDV) {
        // one workgroup per CU (the kernel holds a SIMD's whole register file and 130 KB of LDS)
        const int grid = (1024 / a.hkv) * a.hkv > 0 ? (1024 / a.hkv) * a.hkv : a.hkv;
        if (b.det) {
            hipLaunchKernelGGL(bwd_dkdv_f32_kernel, dim3(grid), dim3(256), 0, s, a, b);
            hipLaunchKernelGGL(bwd_split_finalize_det_kernel<float>, dim3(a.n_kb, a.hkv), dim3(256), 0, s, a, b);
        } else {
            hipLaunchKernelGGL(bwd_split_zero_kernel, dim3(a.n_kb, a.hkv), dim3(256), 0, s, a, b);
            hipLaunchKernelGGL(bwd_dkdv_f32_kernel, dim3(grid), dim3(256), 0, s, a, b);
            hipLaunchKernelGGL(bwd_split_finalize_kernel<float>, dim3(a.n_kb, a.hkv, 4), dim3(256), 0, s, a, b);
        }
        if (hipGetLastError() != hipSuccess) return TT_E_HIP;
    }
    return TT_OK;
}
