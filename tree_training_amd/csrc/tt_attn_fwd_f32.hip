// Tree-masked GQA attention forward for fp32 models (operands split into bf16
// planes; see tt_f32_tiles.h).
#include "tt_f32_tiles.h"

namespace {

// Bound by the matrix cores: a 32-key step is 96 MFMAs (3072 cycles) a wave,
// and everything else is placed behind them: while the scores of step s + 1
// run, the exponentials and the split of step s's probabilities and the split
// of step s + 2's keys; while O += P V of step s runs, the split of step
// s + 1's values. Only the row max stands between them.
// 16,318-token agent tree, 32/8 heads: 4.64 -> 2.95 ms (148 useful TFLOP/s;
// the plane products run at 0.94 PFLOP/s, a large bf16 library GEMM on the same
// card at 1.23) against fp32 MFMAs.
struct FwdStageF {
    bf16 K[2][3 * PLANE];   // step s in K[s & 1]: read while step s - 1 runs
    bf16 V[2][3 * PLANE];   // step s in V[s & 1]
    Bounds32Ring bnd;
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void fwd_f32_kernel(
    AttnDev a, float* __restrict__ out, float* __restrict__ lse) {
    __shared__ __attribute__((aligned(16))) FwdStageF st;

    int qb, h;
    decode_qblock(a, qb, h);
    const int g = __builtin_amdgcn_readfirstlane(h / a.rep);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int col = lane & 31, half = lane >> 5;
    const int q0 = qb * TT_BQ + wave * 32, qi = q0 + col;
    const float c = a.scale * TT_LOG2E;
    const RowOffsG kro = row_offsg(col, half);
    const TrOffsG tro = tr_offsg(lane);

    const KvWalkF w(a, qb);
    RowsF kr, vr;
    Bounds32 nb;
    f32x16 o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (f32x16){};
    float m_run = -INFINITY, l_run = 0.0f;
    Planes q[8];
    f32x16 sc = {};   // scores of the running step
    bool vis = false;
    if (w.n > 0) {   // the walk has two steps per listed tile: w.n >= 2
        const int k0 = w.key0(0), k1 = w.key0(1), k2 = w.key0(min(2, w.n - 1));
        load_keys(a, k0, g, false, kr);
        load_keys(a, k0, g, true, vr);
        nb.load(a, k0);
        load_row_planes((const float*)a.q + (int64_t)min(qi, a.n_q - 1) * a.q_st + h * a.q_sh, qi < a.n_q, half, q);
        store_rows_f(kr, st.K[0]);
        store_rows_f(vr, st.V[0]);
        nb.store(st.bnd, 0);
        load_keys(a, k1, g, false, kr);
        load_keys(a, k1, g, true, vr);
        nb.load(a, k1);
        store_rows_f(kr, st.K[1]);
        nb.store(st.bnd, 1);
        load_keys(a, k2, g, false, kr);
        nb.load(a, k2);
        lds_barrier();
        vis = (w.entry(0) & 1) || step_visible(st.bnd, 0, q0, lane);
        if (vis) {
            f32x16 sc1 = {};
            static_for<4>([&](auto uu) {
                constexpr int u = decltype(uu)::value;
                mfma_split2(read_row_planes<2 * u>(st.K[0], kro), q[2 * u], sc,
                            read_row_planes<2 * u + 1>(st.K[0], kro), q[2 * u + 1], sc1);
            });
            sc += sc1;
        }
        lds_barrier();   // K[0] is written again in step 0
    }
    for (int s = 0; s < w.n; ++s) {
        const bool full = w.entry(s) & 1;
        const int s1 = min(s + 1, w.n - 1);
        const bool vis_next = s + 1 < w.n && ((w.entry(s1) & 1) || step_visible(st.bnd, s1, q0, lane));
        const int k3 = w.key0(min(s + 3, w.n - 1)), k2 = w.key0(min(s + 2, w.n - 1));
        float m_use = 0.0f;
        if (vis) {
            if (!full) mask_half(sc, st.bnd.lo[s & 3], st.bnd.hi[s & 3], qi, half);
            float mx0 = -INFINITY, mx1 = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                mx0 = fmaxf(mx0, sc[r]);
                mx1 = fmaxf(mx1, sc[r + 1]);
            }
            const float mxc = halves_max(fmaxf(mx0, mx1)) * c;
            const bool grow = mxc > m_run + TT_RESCALE_LOG2;
            if (__ballot(grow)) {
                const float alpha = grow ? fast_exp2(m_run - mxc) : 1.0f;
                m_run = grow ? mxc : m_run;
                l_run *= alpha;
#pragma unroll
                for (int db = 0; db < 4; ++db) o[db] *= alpha;
            }
            m_use = (m_run == -INFINITY) ? 0.0f : m_run;
        }
        // Work slots: 0 .. 15 the exponentials, 16 .. 31 the split of P, 26 .. 47 that of step s + 2's keys.
        float ps = 0.0f;
        Split8 p0, p1;
        StoreRows k_lo(kr, 0, st.K[s & 1]), k_hi(kr, 1, st.K[s & 1]);
        auto slot = [&](auto jj) {
            constexpr int j = decltype(jj)::value;
            if constexpr (j < 16) {
                sc[j] = fast_exp2(fmaf(sc[j], c, -m_use));
                ps += sc[j];
            }
            if constexpr (j == 16) p0 = split_begin(sc, 0);
            if constexpr (j >= 16 && j < 24) p0.slice<j - 16>();
            if constexpr (j == 24) p1 = split_begin(sc, 8);
            if constexpr (j >= 24 && j < 32) p1.slice<j - 24>();
            if constexpr (j >= 26 && j < 37) k_lo.slice<j - 26>();
            if constexpr (j >= 37) k_hi.slice<j - 37>();
        };
        f32x16 sn = {};   // scores of step s + 1
        if (vis_next) {
            // operands are read one group of twelve MFMAs ahead of their use;
            // even and odd 16-dim groups sum apart
            const bf16* K = st.K[(s + 1) & 1];
            f32x16 sn1 = {};
            Planes k[4];
            k[0] = read_row_planes<0>(K, kro);
            k[1] = read_row_planes<1>(K, kro);
            static_for<4>([&](auto uu) {
                constexpr int u = decltype(uu)::value, c0 = 2 * (u & 1), n0 = 2 - c0;
                if constexpr (u < 3) {
                    k[n0] = read_row_planes<(2 * u + 2) & 7>(K, kro);
                    k[n0 + 1] = read_row_planes<(2 * u + 3) & 7>(K, kro);
                }
                mfma_split2(k[c0], q[2 * u], sn, k[c0 + 1], q[2 * u + 1], sn1,
                            [&](auto ii) { slot(IntT<12 * u + decltype(ii)::value>{}); });
            });
            sn += sn1;
        } else {
            static_for<48>([&](auto jj) { slot(jj); });
        }
        if (vis) l_run += ps;
        load_keys(a, k3, g, false, kr);
        StoreRows v_lo(vr, 0, st.V[(s + 1) & 1]), v_hi(vr, 1, st.V[(s + 1) & 1]);
        auto vslot = [&](auto jj) {
            constexpr int j = decltype(jj)::value - 24;
            if constexpr (j >= 0 && j < 11) v_lo.slice<j>();
            if constexpr (j >= 11 && j < 22) v_hi.slice<j - 11>();
        };
        if (vis) {   // O^T += V^T P^T: keys 16 (u / 2) .. +15, d blocks 2 (u % 2), +1
            const bf16* V = st.V[s & 1];
            const Planes p[2] = {p0.planes(), p1.planes()};
            Planes v[4];
            v[0] = read_tr_planes(V, tro, 0, 0);
            v[1] = read_tr_planes(V, tro, 0, 1);
            static_for<4>([&](auto uu) {
                constexpr int u = decltype(uu)::value, d0 = 2 * (u & 1), n = u + 1, n0 = 2 * (n & 1);
                if constexpr (u < 3) {
                    v[n0] = read_tr_planes(V, tro, 16 * (n >> 1), n0);
                    v[n0 + 1] = read_tr_planes(V, tro, 16 * (n >> 1), n0 + 1);
                }
                mfma_split2(v[d0], p[u >> 1], o[d0], v[d0 + 1], p[u >> 1], o[d0 + 1],
                            [&](auto ii) { vslot(IntT<12 * u + decltype(ii)::value>{}); });
            });
        } else {
            static_for<48>([&](auto jj) { vslot(jj); });
        }
        load_keys(a, k2, g, true, vr);
        nb.store(st.bnd, s + 2);
        nb.load(a, k3);
        sc = sn;
        vis = vis_next;
        lds_barrier();
    }

    const float l_tot = halves_sum(l_run);
    if (qi < a.n_q) {
        const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        float* op = out + ((size_t)qi * a.hq + h) * D;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                f32x4 wv;
#pragma unroll
                for (int e = 0; e < 4; ++e) wv[e] = o[db][4 * grp + e] * inv;
                *(f32x4*)(op + 32 * db + 8 * grp + 4 * half) = wv;
            }
        if (half == 0) {
            const float m_fin = (m_run == -INFINITY) ? 0.0f : m_run;
            lse[(size_t)h * a.n_q + qi] = l_tot > 0.0f ? (m_fin + __log2f(l_tot)) * TT_LN2 : -INFINITY;
        }
    }
}

}  // namespace

int tt_fwd_f32_launch(const AttnDev& a, void* o, float* lse, hipStream_t s) {
    hipLaunchKernelGGL(fwd_f32_kernel, dim3(a.n_qb * a.hq), dim3(256), 0, s, a, (float*)o, lse);
    return hipGetLastError() == hipSuccess ? TT_OK : TT_E_HIP;
}
