/* Small projections of the DiT path on the matrix cores: the F32 linears of
 * the timestep MLP.
 *
 * F32 MFMAs (v_mfma_f32_16x16x4_f32) multiply and add in full F32: measured
 * on the card, each of their k steps is one fmaf of the accumulator, in k
 * order, denormals, overflow and NaN included.
 */
#include "hk_common.h"
#include "hk_internal.h"

typedef int hk_v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t hk_proj_rsrc(const void *p,
                                                               uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0,
                                             (int)n, 0x00020000);
}

/* ------------------------------------------------------------ F32 linear
 *
 * C[M, N] = X[M, K] . W[N, K]^T (+ bias), all F32.  Few rows (the time rows
 * of a schedule), so it is bound by streaming W once; one thread per output
 * walked W with a row stride between lanes and a serial chain of K fmaf.
 *
 * A workgroup owns 16 columns and up to 16 MB rows, and its eight waves
 * split K: 168 workgroups (the 2688 columns of the time MLP's second layer)
 * then keep 1344 waves loading.  Each lane loads 16 bytes of a W row (and of
 * MB X rows, which L2 serves), DEPTH steps of 16 k ahead of the MFMAs;
 * component j of the four k quarters goes into MFMA j, the same permutation
 * of k on both operands.  The waves' sums meet in LDS in wave order, then
 * the bias is added.  The sum of 8 chains has a smaller rounding error than
 * the single chain had.
 *
 * Measured (39 rows, 256 -> 5376 and 5376 -> 2688): 10.4 and 41.6 us, from
 * 211 and 2284 us. */
enum { HK_LF_WAVES = 8 };

template <int MB, int DEPTH>
__global__ void __launch_bounds__(HK_LF_WAVES * 64)
hk_linear_f32_mfma(const float *x, const float *w, const float *bias,
                   float *c, uint32_t m, uint32_t n, uint32_t k,
                   uint32_t x_bytes, uint32_t w_bytes) {
    extern __shared__ __attribute__((aligned(16))) float hk_lf_red[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, quad = lane >> 4;
    const uint32_t n0 = blockIdx.x * 16u, m0 = blockIdx.y * (16u * MB);
    const __amdgpu_buffer_rsrc_t xr = hk_proj_rsrc(x, x_bytes);
    const __amdgpu_buffer_rsrc_t wr = hk_proj_rsrc(w, w_bytes);
    /* this wave's 16-wide k steps */
    const uint32_t steps = (k + 15u) / 16u;
    const uint32_t first = steps * wave / HK_LF_WAVES;
    const uint32_t last = steps * (wave + 1u) / HK_LF_WAVES;
    /* rows past the end start at the buffer's end and read zeros; so does
     * the part of a last step past K, on both operands */
    const uint32_t w_off = min(n0 + r16, n) * k * 4u + quad * 16u;
    uint32_t x_off[MB];
#pragma unroll
    for (int b = 0; b < MB; b++)
        x_off[b] = min(m0 + 16u * b + r16, m) * k * 4u + quad * 16u;
    hk_v4i wf[DEPTH], xf[DEPTH][MB];
    auto load = [&](int slot, uint32_t step) {
        const bool in = step < last && step * 16u + quad * 4u < k;
        wf[slot] = __builtin_amdgcn_raw_buffer_load_b128(
            wr, in ? w_off + step * 64u : w_bytes, 0, 0);
#pragma unroll
        for (int b = 0; b < MB; b++)
            xf[slot][b] = __builtin_amdgcn_raw_buffer_load_b128(
                xr, in ? x_off[b] + step * 64u : x_bytes, 0, 0);
    };
    hk_f32x4 acc[MB];
#pragma unroll
    for (int b = 0; b < MB; b++) acc[b] = hk_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < DEPTH; d++) load(d, first + d);
    for (uint32_t s = first; s < last; s += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            /* steps past the range hold zeros */
            const hk_f32x4 wv = __builtin_bit_cast(hk_f32x4, wf[d]);
            hk_f32x4 xv[MB];
#pragma unroll
            for (int b = 0; b < MB; b++)
                xv[b] = __builtin_bit_cast(hk_f32x4, xf[d][b]);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int b = 0; b < MB; b++)
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        wv[j], xv[b][j], acc[b], 0, 0, 0);
            load(d, s + DEPTH + d);
        }
    }
    /* acc[b][i] = C[m0 + 16 b + r16][n0 + 4 quad + i], summed over waves */
    hk_f32x4 *red = (hk_f32x4 *)hk_lf_red;
#pragma unroll
    for (int b = 0; b < MB; b++)
        red[(wave * MB + b) * 64u + lane] = acc[b];
    __syncthreads();
    for (uint32_t t = tid; t < MB * 64u; t += HK_LF_WAVES * 64u) {
        hk_f32x4 sum = red[t];
#pragma unroll
        for (int v = 1; v < HK_LF_WAVES; v++) sum += red[v * MB * 64u + t];
        const uint32_t row = m0 + (t >> 6) * 16u + (t & 15u);
        const uint32_t col = n0 + ((t >> 4) & 3u) * 4u;
        if (row >= m) continue;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (col + i < n)
                c[(size_t)row * n + col + i] =
                    sum[i] + (bias ? bias[col + i] : 0.0f);
    }
}

template <int MB, int DEPTH>
static void hk_linear_f32_run(struct h3_gpu *gpu, const float *x,
                              const float *w, const float *bias, float *c,
                              uint32_t m, uint32_t n, uint32_t k) {
    hipLaunchKernelGGL((hk_linear_f32_mfma<MB, DEPTH>),
                       dim3((n + 15) / 16, (m + 16 * MB - 1) / (16 * MB)),
                       dim3(HK_LF_WAVES * 64),
                       HK_LF_WAVES * MB * 64 * sizeof(hk_f32x4), gpu->stream,
                       x, w, bias, c, m, n, k, (uint32_t)((uint64_t)m * k * 4),
                       (uint32_t)((uint64_t)n * k * 4));
}

bool hk_linear_f32(struct h3_gpu *gpu, const float *x, const float *w,
                   const float *bias, float *c, uint32_t m, uint32_t n,
                   uint32_t k) {
    /* 16-byte loads; offsets up to a step past the end of a row past the
     * end stay below 2^32 */
    const uint64_t margin = 4ull * k + 4096;
    if (!k || k % 4 || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) ||
        (uint64_t)m * k * 4 + margin >= 0x100000000ull ||
        (uint64_t)n * k * 4 + margin >= 0x100000000ull || m > 65535u * 64u)
        return false;
    if (m <= 16)
        hk_linear_f32_run<1, 8>(gpu, x, w, bias, c, m, n, k);
    else if (m <= 32)
        hk_linear_f32_run<2, 6>(gpu, x, w, bias, c, m, n, k);
    else if (m <= 48)
        hk_linear_f32_run<3, 4>(gpu, x, w, bias, c, m, n, k);
    else
        hk_linear_f32_run<4, 4>(gpu, x, w, bias, c, m, n, k);
    return true;
}
