// Row-wise softmax cross-entropy with its logit gradient, for gfx950: the
// leaf-loss step after the tree forward, applied to one chunk of lm_head
// logits at a time so the [T, V] logits never exist at once.
//
// Row r (label y, weight c): lse = log sum_j exp(x_j),
//   loss[r] = c (lse - x_y),   grad[r][j] = c (exp(x_j - lse) - [j == y]);
// a row whose label is ignore_index gets loss 0 and a zero gradient. grad may
// alias the logits (each element is read before the same thread writes it).
// One workgroup per row. Rows of 64 (fp32: 48) to 320 KB are held in registers
// (2 x row bytes of HBM traffic); others take an online max/sum pass, then the
// gradient pass (3 x row bytes). fp32 arithmetic.
#include "tt_common.h"
#include "tt_internal.h"

namespace {

constexpr int CE_T = 256;

template <typename T>
__device__ __forceinline__ void ce_ld8(const T* p, float (&x)[8]) {
    if constexpr (sizeof(T) == 2) {
        const bf16x8 a = *(const bf16x8*)p;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (float)a[e];
    } else {
        const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = a[e];
            x[4 + e] = b[e];
        }
    }
}

template <typename T>
__device__ __forceinline__ void ce_st8(T* p, const float (&x)[8]) {
    if constexpr (sizeof(T) == 2) {
        bf16x8 a;
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = (__bf16)x[e];
        *(bf16x8*)p = a;
    } else {
        *(f32x4*)p = (f32x4){x[0], x[1], x[2], x[3]};
        *(f32x4*)(p + 4) = (f32x4){x[4], x[5], x[6], x[7]};
    }
}

// (m, s) <- merge of two online-softmax partials (s relative to m). Without a
// logit above -inf on either side the sums are zero, or a NaN that must stay.
__device__ __forceinline__ void merge_ms(float& m, float& s, float m2, float s2) {
    const float mn = fmaxf(m, m2);
    if (mn == -INFINITY) {
        s += s2;
        return;
    }
    s = s * exp2f((m - mn) * TT_LOG2E) + s2 * exp2f((m2 - mn) * TT_LOG2E);
    m = mn;
}

template <typename T>
__global__ __launch_bounds__(CE_T) void ce_rows_kernel(const T* logits, int64_t ld, int V,
                                                       const int32_t* __restrict__ labels,
                                                       const float* __restrict__ row_scale, int ignore_index,
                                                       float* __restrict__ loss, T* grad, int64_t ldg) {
    __shared__ float red_m[CE_T / 64], red_s[CE_T / 64];
    __shared__ float row_lse;
    const int row = blockIdx.x, tid = threadIdx.x;
    const T* x = logits + (int64_t)row * ld;
    T* g = grad + (int64_t)row * ldg;
    const int lab = labels[row];
    const bool ignore = lab == ignore_index;
    const bool valid = !ignore && lab >= 0 && lab < V;
    const float sc = row_scale[row];
    const int v8 = V & ~7;

    float m = -INFINITY, s = 0.0f;
    for (int j = 8 * tid; j < v8; j += 8 * CE_T) {
        float v[8];
        ce_ld8(x + j, v);
        float m8 = v[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) m8 = fmaxf(m8, v[e]);
        // a group of nothing but -inf (a masked vocabulary) adds exp(-inf) = 0, not exp(-inf + inf)
        const float ms = m8 == -INFINITY ? 0.0f : m8;
        float s8 = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) s8 += exp2f((v[e] - ms) * TT_LOG2E);
        merge_ms(m, s, m8, s8);
    }
    for (int j = v8 + tid; j < V; j += CE_T) {
        const float vj = (float)x[j], mj = vj == -INFINITY ? 0.0f : vj;
        merge_ms(m, s, vj, exp2f((vj - mj) * TT_LOG2E));   // as a group of one
    }
    // wave, then workgroup
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float m2 = __shfl_xor(m, o), s2 = __shfl_xor(s, o);
        merge_ms(m, s, m2, s2);
    }
    if ((tid & 63) == 0) {
        red_m[tid >> 6] = m;
        red_s[tid >> 6] = s;
    }
    __syncthreads();
    if (tid == 0) {
        float mm = red_m[0], ss = red_s[0];
#pragma unroll
        for (int w = 1; w < CE_T / 64; ++w) merge_ms(mm, ss, red_m[w], red_s[w]);
        const float lse = mm + logf(ss);
        row_lse = lse;
        loss[row] = ignore ? 0.0f : (valid ? sc * (lse - (float)x[lab]) : __builtin_nanf(""));
    }
    __syncthreads();   // the label's logit is read before any gradient overwrites it
    const float lse = row_lse;
    const float c = valid ? sc : 0.0f;
    for (int j = 8 * tid; j < v8; j += 8 * CE_T) {
        float v[8];
        ce_ld8(x + j, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = c * (exp2f((v[e] - lse) * TT_LOG2E) - (j + e == lab ? 1.0f : 0.0f));
        ce_st8(g + j, v);
    }
    for (int j = v8 + tid; j < V; j += CE_T) {
        const float v = (float)x[j];
        g[j] = (T)(c * (exp2f((v - lse) * TT_LOG2E) - (j == lab ? 1.0f : 0.0f)));
    }
}

// The same for rows that fit the register files: 1024 threads hold the row as
// NV vectors of 16 bytes each, so the logits are read once (2 x row bytes of
// traffic) and no exponential is taken against a running maximum.
constexpr int CE_TR = 1024;

template <typename T, int NV>
__global__ __launch_bounds__(CE_TR) void ce_rows_reg_kernel(const T* logits, int64_t ld, int V,
                                                            const int32_t* __restrict__ labels,
                                                            const float* __restrict__ row_scale, int ignore_index,
                                                            float* __restrict__ loss, T* grad, int64_t ldg) {
    constexpr int VE = 16 / sizeof(T);
    typedef T TV __attribute__((ext_vector_type(VE)));
    union Vec {
        TV t;
        uint32_t w[4];
    };
    __shared__ float red_m[CE_TR / 64], red_s[CE_TR / 64];
    const int row = blockIdx.x, tid = threadIdx.x;
    const T* x = logits + (int64_t)row * ld;
    T* g = grad + (int64_t)row * ldg;
    const int n_v = V / VE;                       // whole vectors; the rest, one element a thread
    const int jt = n_v * VE + tid;
    Vec v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = i * CE_TR + tid;
        if (j < n_v) v[i].t = *(const TV*)(x + (int64_t)j * VE);
        else
#pragma unroll
            for (int e = 0; e < VE; ++e) v[i].t[e] = (T)-INFINITY;
    }
    // Between the passes over the row its registers are opaque to the compiler,
    // which would else keep the passes' unpacked floats (twice the registers).
    const auto opaque = [&]() {
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(v[i].w[e]));
    };
    const float vt = jt < V ? (float)x[jt] : -INFINITY;
    const int lab = labels[row];
    const bool ignore = lab == ignore_index;
    const bool valid = !ignore && lab >= 0 && lab < V;
    const float sc = row_scale[row];
    const float xl = valid ? (float)x[lab] : 0.0f;

    float m = vt;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < VE; ++e) m = fmaxf(m, (float)v[i].t[e]);
    opaque();
    // a thread without a logit above -inf adds nothing; the hardware exponential's
    // flushed denormals are lost beside the maximum's 1
    float s = 0.0f;
    const float ms = m == -INFINITY ? 0.0f : m;
    if (jt < V) s = fast_exp2((vt - ms) * TT_LOG2E);
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < VE; ++e) s += fast_exp2(((float)v[i].t[e] - ms) * TT_LOG2E);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float m2 = __shfl_xor(m, o), s2 = __shfl_xor(s, o);
        merge_ms(m, s, m2, s2);
    }
    if ((tid & 63) == 0) {
        red_m[tid >> 6] = m;
        red_s[tid >> 6] = s;
    }
    opaque();
    __syncthreads();   // also: the label's logit is read before any gradient overwrites it
    m = red_m[0];
    s = red_s[0];
#pragma unroll
    for (int w = 1; w < CE_TR / 64; ++w) merge_ms(m, s, red_m[w], red_s[w]);
    const float lse = m + logf(s);
    if (tid == 0) loss[row] = ignore ? 0.0f : (valid ? sc * (lse - xl) : __builtin_nanf(""));
    const float c = valid ? sc : 0.0f;
    const int lab_t = valid ? lab - VE * tid : -1;   // the label's column counted from the thread's first
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int j = i * CE_TR + tid;
        if (j < n_v) {
            TV o;
#pragma unroll
            for (int e = 0; e < VE; ++e)
                o[e] = (T)(c * (exp2f(((float)v[i].t[e] - lse) * TT_LOG2E) - (i * CE_TR * VE + e == lab_t ? 1.0f : 0.0f)));
            *(TV*)(g + (int64_t)j * VE) = o;
        }
    }
    if (jt < V) g[jt] = (T)(c * (exp2f((vt - lse) * TT_LOG2E) - (jt == lab ? 1.0f : 0.0f)));
}

// The register kernel where it is the faster one: from more than 4 vectors a
// thread in bf16, 4 in fp32, to the 20 that leave its 16 waves a CU. 4,096 rows,
// two-pass against registers (us): bf16 vocab 32,000 122 / 135, 32,776 130 / 125,
// 40,960 161 / 142, 50,304 230 / 173, 65,536 304 / 213, 128,256 648 / 438,
// 151,936 759 / 539 (4.6 TB/s); fp32 8,192 59 / 78, 12,292 91 / 82, 16,384
// 119 / 90, 32,000 288 / 204, 65,536 630 / 414. Five vectors have an instance of
// their own: in that of eight their three empty ones cost more than the second
// read (vocab 32,776: 145 us).
template <typename T>
void ce_launch(const void* logits, int64_t ld, int n_rows, int vocab, const int32_t* labels, const float* row_scale,
               int ignore_index, float* loss, void* grad, int64_t ldg, hipStream_t s) {
    const int nv = tt_cdiv(vocab / (16 / (int)sizeof(T)), CE_TR);   // vectors a thread
#define CE_REG(NV)                                                                                                  \
    hipLaunchKernelGGL((ce_rows_reg_kernel<T, NV>), dim3(n_rows), dim3(CE_TR), 0, s, (const T*)logits, ld, vocab,   \
                       labels, row_scale, ignore_index, loss, (T*)grad, ldg)
    if (nv > 20)
        hipLaunchKernelGGL(ce_rows_kernel<T>, dim3(n_rows), dim3(CE_T), 0, s, (const T*)logits, ld, vocab, labels,
                           row_scale, ignore_index, loss, (T*)grad, ldg);
    else if (nv > 16) CE_REG(20);
    else if (nv > 12) CE_REG(16);
    else if (nv > 8) CE_REG(12);
    else if (nv > 5) CE_REG(8);
    else if (nv > 4) CE_REG(5);
    else if (nv > 3 && sizeof(T) == 4) CE_REG(4);
    else
        hipLaunchKernelGGL(ce_rows_kernel<T>, dim3(n_rows), dim3(CE_T), 0, s, (const T*)logits, ld, vocab, labels,
                           row_scale, ignore_index, loss, (T*)grad, ldg);
#undef CE_REG
}

}  // namespace

int tt_ce_rows_launch(int dtype, const void* logits, int64_t ld, int n_rows, int vocab, const int32_t* labels,
                      const float* row_scale, int ignore_index, float* loss, void* grad, int64_t ldg,
                      hipStream_t s) {
    if (dtype == TT_DTYPE_BF16)
        ce_launch<__bf16>(logits, ld, n_rows, vocab, labels, row_scale, ignore_index, loss, grad, ldg, s);
    else
        ce_launch<float>(logits, ld, n_rows, vocab, labels, row_scale, ignore_index, loss, grad, ldg, s);
    return hipGetLastError() == hipSuccess ? TT_OK : TT_E_HIP;
}
