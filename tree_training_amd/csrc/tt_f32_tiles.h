// Device code shared by the fp32 tree-attention kernels (forward in
// tt_attn_fwd_f32.hip, backward in tt_attn_bwd_f32.hip).
//
// fp32 products run on gfx950's bf16 matrix cores, on operands split into bf16
// planes (tt_planes.h).
//
// The tiling, plan walk, masks and dK/dV work items are the bf16 path's
// (tt_bf16_tiles.h) in steps of 32 keys (forward, dQ) or 32 queries (dK/dV).
// A step's fp32 rows are loaded into registers a step before they are split
// and stored as bf16 planes (the row-group layout, read as rows and
// transposed), which a step later are read; two LDS stages, one barrier a
// step. One wave per SIMD: the operand planes of the wave's own 32 rows stay
// in registers (96 per tensor). The wave issues in order, so the vector work
// (splits, softmax) is placed between the MFMAs in slices of a few
// instructions, one behind each MFMA (mfma_split2).
#pragma once

#include "tt_bf16_tiles.h"
#include "tt_planes.h"

namespace {

constexpr int PLANE = 8 * GPITCH;   // one bf16 plane of a 32-row tile (row groups)

struct NoWork {
    template <typename I>
    __device__ __forceinline__ void operator()(I) const {}
};
// x += a b and y += c d, the smallest terms first; the two sums alternate, so
// no MFMA waits for the one before it. work(IntT<i>) is issued behind the
// i-th of the twelve MFMAs.
template <typename F = NoWork>
__device__ __forceinline__ void mfma_split2(const Planes& a, const Planes& b, f32x16& x, const Planes& c,
                                            const Planes& d, f32x16& y, F&& work = F{}) {
#define TT_SLOT(I)               \
    work(IntT<I>{});             \
    __builtin_amdgcn_sched_barrier(0)
    __builtin_amdgcn_sched_barrier(0);
    x = mfma32(a.l, b.h, x);
    TT_SLOT(0);
    y = mfma32(c.l, d.h, y);
    TT_SLOT(1);
    x = mfma32(a.h, b.l, x);
    TT_SLOT(2);
    y = mfma32(c.h, d.l, y);
    TT_SLOT(3);
    x = mfma32(a.m, b.m, x);
    TT_SLOT(4);
    y = mfma32(c.m, d.m, y);
    TT_SLOT(5);
    x = mfma32(a.m, b.h, x);
    TT_SLOT(6);
    y = mfma32(c.m, d.h, y);
    TT_SLOT(7);
    x = mfma32(a.h, b.m, x);
    TT_SLOT(8);
    y = mfma32(c.h, d.m, y);
    TT_SLOT(9);
    x = mfma32(a.h, b.h, x);
    TT_SLOT(10);
    y = mfma32(c.h, d.h, y);
    TT_SLOT(11);
#undef TT_SLOT
}
template <int T>
__device__ __forceinline__ Planes read_row_planes(const bf16* X, const RowOffsG& ro) {
    return {read_rowg<T>(X, ro), read_rowg<T>(X + PLANE, ro), read_rowg<T>(X + 2 * PLANE, ro)};
}
__device__ __forceinline__ Planes read_tr_planes(const bf16* X, const TrOffsG& to, int r0, int db) {
    return {read_trg(X, to, r0, db), read_trg(X + PLANE, to, r0, db), read_trg(X + 2 * PLANE, to, r0, db)};
}

__device__ __forceinline__ const float* key_row_f(const AttnDev& a, int kk, int g, bool isv) {
    if (kk < a.n_past) {
        return isv ? (const float*)a.vp + kk * a.vp_st + g * a.vp_sh
                   : (const float*)a.kp + kk * a.kp_st + g * a.kp_sh;
    }
    const int64_t t = kk - a.n_past;
    return isv ? (const float*)a.v + t * a.v_st + g * a.v_sh : (const float*)a.k + t * a.k_st + g * a.k_sh;
}

// 32 fp32 rows on their way to three bf16 planes: thread t holds rows t / 16
// and t / 16 + 16, floats 8 (t % 16) .. +7.
struct RowsF {
    f32x4 x[4];
    // rows that all exist: row 0 at `base` (uniform), rows `stb` bytes apart
    __device__ __forceinline__ void load_buf(const float* base, uint32_t stb) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(base), (short)0, (int)(31u * stb + 4u * D), 0x00020000);
        const uint32_t vo = (threadIdx.x >> 4) * stb + 32u * (threadIdx.x & 15);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            x[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 rs, (int)(vo + 16u * (i & 1)), (int)(16u * (i >> 1) * stb), 0));
    }
    __device__ __forceinline__ void load_row(int i, const float* row) {
        const float* p = row + 8 * (threadIdx.x & 15);
        x[2 * i] = *(const f32x4*)p;
        x[2 * i + 1] = *(const f32x4*)(p + 4);
    }
};
// Splits and stores the i-th of the thread's two row pieces: eleven slices.
struct StoreRows {
    static constexpr int SLICES = Split8::SLICES + 3;
    Split8 w;
    bf16* d;
    __device__ __forceinline__ StoreRows(const RowsF& r, int i, bf16* X)
        : w(split_begin(r.x[2 * i], r.x[2 * i + 1])),
          d(X + tile_offg((threadIdx.x >> 4) + 16 * i, 8 * (threadIdx.x & 15))) {}
    template <int I>
    __device__ __forceinline__ void slice() {
        w.template slice<I>();
        if constexpr (I == Split8::SLICES) *(bf16x8*)d = Split8::vec(w.h);
        if constexpr (I == Split8::SLICES + 1) *(bf16x8*)(d + PLANE) = Split8::vec(w.m);
        if constexpr (I == Split8::SLICES + 2) *(bf16x8*)(d + 2 * PLANE) = Split8::vec(w.l);
    }
};
__device__ __forceinline__ void store_rows_f(const RowsF& r, bf16* X) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        StoreRows st(r, i, X);
        static_for<StoreRows::SLICES>([&](auto j) { st.slice<decltype(j)::value>(); });
    }
}

// The planes of the lane's own row in operand order: x[t] holds dims
// 16 t + 8 half .. +7 (zeros when the row does not exist).
__device__ __forceinline__ void load_row_planes(const float* row, bool valid, int half, Planes (&x)[8]) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const float* p = row + 16 * t + 8 * half;
        const f32x4 z = {};
        Split8 w = split_begin(valid ? *(const f32x4*)p : z, valid ? *(const f32x4*)(p + 4) : z);
        w.all();
        x[t] = w.planes();
    }
}

// ----------------------------------------------------------------------------
// forward and dQ: the plan's 64-key tiles in steps of 32 keys
// ----------------------------------------------------------------------------
// Visible query intervals of the 32 keys of a step: step s in slot s & 3.
struct Bounds32Ring {
    int lo[4][32];
    int hi[4][32];
};

// Step s of a query block's walk covers keys k0 .. k0 + 31, half s & 1 of the
// s / 2-th listed tile (rows past the last key alias it; their empty bounds
// mask them).
struct KvWalkF {
    const int* list;
    int n;   // steps
    __device__ __forceinline__ KvWalkF(const AttnDev& a, int qb)
        : list(a.row_list + (size_t)qb * a.n_kt), n(2 * __builtin_amdgcn_readfirstlane(a.row_cnt[qb])) {}
    __device__ __forceinline__ int entry(int s) const { return __builtin_amdgcn_readfirstlane(list[s >> 1]); }
    __device__ __forceinline__ int key0(int s) const { return (entry(s) >> 1) * TT_BK + 32 * (s & 1); }
};
__device__ __forceinline__ void load_keys(const AttnDev& a, int k0, int g, bool isv, RowsF& r) {
    if (k0 + 32 <= a.n_past) {
        r.load_buf(isv ? (const float*)a.vp + k0 * a.vp_st + g * a.vp_sh
                       : (const float*)a.kp + k0 * a.kp_st + g * a.kp_sh,
                   4u * (uint32_t)(isv ? a.vp_st : a.kp_st));
    } else if (k0 >= a.n_past && k0 + 32 <= a.n_keys) {
        const int64_t t0 = k0 - a.n_past;
        r.load_buf(isv ? (const float*)a.v + t0 * a.v_st + g * a.v_sh : (const float*)a.k + t0 * a.k_st + g * a.k_sh,
                   4u * (uint32_t)(isv ? a.v_st : a.k_st));
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            r.load_row(i, key_row_f(a, min(k0 + (int)(threadIdx.x >> 4) + 16 * i, a.n_keys - 1), g, isv));
    }
}
// ... on their way there (threads 0 .. 31).
struct Bounds32 {
    int lo, hi;
    __device__ __forceinline__ void load(const AttnDev& a, int k0) {
        if (threadIdx.x < 32) {
            const int kk = k0 + threadIdx.x;
            lo = kk < a.n_keys ? a.key_lo[kk] : 0;
            hi = kk < a.n_keys ? a.key_hi[kk] : 0;
        }
    }
    __device__ __forceinline__ void store(Bounds32Ring& b, int s) const {
        if (threadIdx.x < 32) {
            b.lo[s & 3][threadIdx.x] = lo;
            b.hi[s & 3][threadIdx.x] = hi;
        }
    }
};
// Whether any key of step s is seen by any of the wave's queries [q0, q0 + 32).
__device__ __forceinline__ bool step_visible(const Bounds32Ring& b, int s, int q0, int lane) {
    return __ballot(max(b.lo[s & 3][lane & 31], q0) < min(b.hi[s & 3][lane & 31], q0 + 32)) != 0ull;
}

}  // namespace
