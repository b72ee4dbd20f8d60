// SPDX-License-Identifier: MIT
// 16-bit GEMM for few rows, C[M,N] = A[M,K] * W[N,K]^T with FP32 accumulation and the
// epilogues of gemm16_pp.hip: products of at most 16 rows, and plain ones without split
// scratch of up to 128 rows and not too many columns (gemm16_pingpong decides).
//
// With at most 16 rows the product is bound by reading W once. The 256 x 256 tiles of the
// general kernel stage it through LDS for mostly empty rows and need a split along K, with
// a reduction launch, to fill the chip. Here a workgroup owns 16 or 32 columns and all
// rows; its 8 waves cut K between them, each reading its operands straight into MFMA
// fragments (no LDS, no barrier in the loop, two groups of K steps in flight), and their
// sums are added through LDS in wave order, so that one launch stores the result. Every
// workgroup reads all of A, which is what bounds it with more rows and many columns.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace ehip {
namespace skinny {

constexpr int WAVES = 8;

struct Params {
    const void* A;
    const void* W;
    int M, N, nk;
    int a_row, a_kstep, w_row, w_kstep;  // byte distances of rows and of 32-column K steps
    void* C;
    long ldc, c_rs, c_ss;  // c_rs, c_ss: GLU output, distance of rows and of 32-column groups
    const float* bias;
    const float* resid;
    long ld_resid;
    const float* gate;
    int vec;  // 16-byte aligned rows and vectors (8-byte for 16-bit outputs), N a multiple of 4
};

template <typename T> struct Mfma;
template <> struct Mfma<f16> {
    typedef f16x8 vec;
    static __device__ __forceinline__ f32x4 run(vec a, vec b, f32x4 c)
    { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <> struct Mfma<bf16> {
    typedef bf16x8 vec;
    static __device__ __forceinline__ f32x4 run(vec a, vec b, f32x4 c)
    { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

// MB row blocks and NB column blocks of 16. A GLU epilogue takes NB = 2: 16 up columns
// and the 16 gate columns 32 further on. U: K steps per group.
template <typename T, typename OutT, int EPI, int MB, int NB, int U>
__global__ void __launch_bounds__(64 * WAVES) kernel(Params p)
{
    static_assert(!epi_glu(EPI) || NB == 2, "a GLU tile is one up and one gate block");
    typedef typename Mfma<T>::vec vec8;
    typedef OutT out4 __attribute__((ext_vector_type(4)));
    __shared__ f32x4 red[WAVES][MB * NB][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q16 = lane >> 4;
    const int b = blockIdx.x;
    // W row of column block j's first column.
    auto col0 = [&](int j) { return epi_glu(EPI) ? (b >> 1) * 64 + (b & 1) * 16 + 32 * j : (b * NB + j) * 16; };

    uint32_t ao[MB], wo[NB];
#pragma unroll
    for (int i = 0; i < MB; ++i) ao[i] = (uint32_t)(min(16 * i + r16, p.M - 1) * (long)p.a_row) + 16 * q16;
#pragma unroll
    for (int j = 0; j < NB; ++j) wo[j] = (uint32_t)(min(col0(j) + r16, p.N - 1) * (long)p.w_row) + 16 * q16;
    const char* A = static_cast<const char*>(p.A);
    const char* W = static_cast<const char*>(p.W);
    f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Groups of U consecutive K steps, dealt to the waves in turn, so that a workgroup
    // reads whole pieces of each row; each workgroup starts at another group, so that all
    // of them together do not walk the same few memory channels.
    const int groups = (p.nk + U - 1) / U, n = (groups - wave + WAVES - 1) / WAVES;
    vec8 af[2][U][MB], wf[2][U][NB];
    auto load = [&](int k, vec8 (&a)[U][MB], vec8 (&w)[U][NB]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kt = min(k + u, p.nk - 1);  // past the end: read again, not used
            const char* wk = W + (long)kt * p.w_kstep;
            const char* ak = A + (long)kt * p.a_kstep;
#pragma unroll
            for (int j = 0; j < NB; ++j) w[u][j] = *reinterpret_cast<const vec8*>(wk + wo[j]);
#pragma unroll
            for (int i = 0; i < MB; ++i) a[u][i] = *reinterpret_cast<const vec8*>(ak + ao[i]);
        }
    };
    auto mul = [&](int k, const vec8 (&a)[U][MB], const vec8 (&w)[U][NB]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < p.nk)
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j) acc[i][j] = Mfma<T>::run(w[u][j], a[u][i], acc[i][j]);
    };
    if (n > 0) {
        int at = b % n;
        auto next = [&]() {
            const int k = (wave + WAVES * at) * U;
            at = at + 1 < n ? at + 1 : 0;
            return k;
        };
        int k = next(), k2;
        load(k, af[0], wf[0]);
        for (int i = 0; i < n; i += 2) {
            load(k2 = next(), af[1], wf[1]);
            mul(k, af[0], wf[0]);
            if (i + 1 == n) break;
            load(k = next(), af[0], wf[0]);
            mul(k2, af[1], wf[1]);
        }
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) red[wave][i * NB + j][lane] = acc[i][j];
    __syncthreads();
    // Element group: block (i, j), lane l: row 16 i + l % 16, columns 4 (l / 16) .. + 3.
    constexpr int JS = epi_glu(EPI) ? 1 : NB;  // a GLU's up block takes its gate block along
#pragma unroll
    for (int x = threadIdx.x; x < MB * JS * 64; x += 64 * WAVES) {
        const int blk = x >> 6, i = blk / JS, j = blk - i * JS;
        const int m = 16 * i + r16, n = col0(j) + 4 * q16;
        if (m >= p.M || n >= p.N) continue;
        f32x4 v = red[0][i * NB + j][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += red[w][i * NB + j][lane];
        if constexpr (epi_glu(EPI)) {
            f32x4 g = red[0][i * NB + 1][lane];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) g += red[w][i * NB + 1][lane];
            OutT* c = static_cast<OutT*>(p.C) + (size_t)m * p.c_rs + (size_t)(n >> 6) * p.c_ss + (n & 31);
            out4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = OutT(v[r] * glu_act<EPI == EPI_SWIGLU>(g[r]));
            if (p.vec) *reinterpret_cast<out4*>(c) = o;
            else
#pragma unroll
                for (int r = 0; r < 4; ++r) c[r] = o[r];
        } else {
            OutT* c = static_cast<OutT*>(p.C) + (size_t)m * p.ldc + n;
            if (p.vec) {
                if (EPI == EPI_GATE_RESID) {
                    const f32x4 g = *reinterpret_cast<const f32x4*>(p.gate + n);
                    const f32x4 res = *reinterpret_cast<const f32x4*>(p.resid + (size_t)m * p.ld_resid + n);
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = __builtin_fmaf(g[r], v[r], res[r]);
                } else if (p.bias) {
                    v += *reinterpret_cast<const f32x4*>(p.bias + n);
                }
                *reinterpret_cast<out4*>(c) = out4{OutT(v[0]), OutT(v[1]), OutT(v[2]), OutT(v[3])};
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (n + r >= p.N) continue;
                    float y = v[r];
                    if (EPI == EPI_GATE_RESID) y = __builtin_fmaf(p.gate[n + r], y, p.resid[(size_t)m * p.ld_resid + n + r]);
                    else if (p.bias) y += p.bias[n + r];
                    c[r] = OutT(y);
                }
            }
        }
    }
}

template <typename T, typename OutT, int EPI, int MB>
void launch_mb(const Params& p, hipStream_t s)
{
    constexpr int U = MB == 8 ? 1 : 2;
    const dim3 block(64 * WAVES);
    if constexpr (epi_glu(EPI)) {
        hipLaunchKernelGGL((kernel<T, OutT, EPI, MB, 2, U>), dim3(p.N / 32), block, 0, s, p);
    } else if (p.N <= kSkinnyNarrow) {
        hipLaunchKernelGGL((kernel<T, OutT, EPI, MB, 1, U>), dim3(skinny_workgroups(p.N)), block, 0, s, p);
    } else {
        hipLaunchKernelGGL((kernel<T, OutT, EPI, MB, 2, U>), dim3(skinny_workgroups(p.N)), block, 0, s, p);
    }
}

// More than 16 rows: plain products only. Returns -1 for others.
template <typename T, typename OutT, int EPI>
int launch(const Params& p, hipStream_t s)
{
    if (p.M <= 16) {
        launch_mb<T, OutT, EPI, 1>(p, s);
        return 0;
    }
    if constexpr (EPI == EPI_STORE) {
        if (p.M <= 32) launch_mb<T, OutT, EPI, 2>(p, s);
        else if (p.M <= 64) launch_mb<T, OutT, EPI, 4>(p, s);
        else launch_mb<T, OutT, EPI, 8>(p, s);
        return 0;
    }
    return -1;
}

template <typename T>
int launch_dtype(const GemmArgs& a, const Params& p, hipStream_t s)
{
    if (a.epilogue == EPI_GATE_RESID) return launch<T, float, EPI_GATE_RESID>(p, s);
    if (a.epilogue == EPI_SWIGLU) return launch<T, T, EPI_SWIGLU>(p, s);
    if (a.epilogue == EPI_GEGLU) return launch<T, T, EPI_GEGLU>(p, s);
    if (a.c_dtype == DT_F32) return launch<T, float, EPI_STORE>(p, s);
    return launch<T, T, EPI_STORE>(p, s);
}

}  // namespace skinny

int gemm16_skinny(const GemmArgs& a, bool vec, hipStream_t s)
{
    skinny::Params p{};
    p.A = a.A; p.W = a.W; p.M = a.M; p.N = a.N; p.nk = a.K / 32;
    p.a_row = a.a_k32_rows ? 64 : (int)(a.lda * 2);
    p.a_kstep = a.a_k32_rows ? a.a_k32_rows * 64 : 64;
    p.w_row = a.w_k32 ? 64 : (int)(a.ldw * 2);
    p.w_kstep = a.w_k32 ? a.N * 64 : 64;
    p.C = a.C; p.ldc = a.ldc;
    p.c_rs = a.c_k32_rows ? 32 : a.ldc;
    p.c_ss = a.c_k32_rows ? 32L * a.c_k32_rows : 32;
    p.bias = a.bias; p.resid = a.resid; p.ld_resid = a.ld_resid; p.gate = a.gate;
    p.vec = vec;
    int rc = a.dtype == DT_F16 ? skinny::launch_dtype<f16>(a, p, s) : skinny::launch_dtype<bf16>(a, p, s);
    if (rc) return rc;
    if (a.epilogue == EPI_QKROPE) {
        // Q and K columns were stored permuted and rounded: normalised, rotated and put in
        // natural order as for the split rows of the general kernel.
        rc = qk_norm_rope_permuted(a.C, a.dtype, 0, a.M, (int)(a.k_col / 128), (int)((a.qk_cols - a.k_col) / 128),
                                             a.ldc, a.k_col, a.gq, a.gk, a.cs_t, a.qk_eps, s);
        if (rc) return rc;
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : -int(e);
}

}  // namespace ehip
