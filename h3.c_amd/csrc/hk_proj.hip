/* Small projections of the DiT path on the matrix cores: the F32 linears of
 * the timestep MLP, the F32 patch projections and the final adaLN heads.
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
 * of a schedule), so it should be bound by streaming W once; one thread per
 * output walked W with a row stride between lanes and a serial chain of K
 * fmaf.
 *
 * A workgroup owns 32 columns, up to 16 MB rows and, where that leaves CUs
 * idle, one of a few pieces of K (blockIdx.z); its eight waves split the K
 * range again.  Each lane loads 16 bytes of two W rows and of MB X rows,
 * DEPTH steps of 32 k ahead of the MFMAs; component j of the four k quarters
 * goes into MFMA j, the same permutation of k on both operands.  The waves'
 * sums meet in LDS in wave order; pieces leave partial sums that
 * hk_linear_f32_reduce adds in piece order, and the bias comes last.  The sum
 * of many short chains has a smaller rounding error than the single chain
 * had.
 *
 * X, re-read by every workgroup, is what its rate hangs on: with 16 columns
 * and all of K per workgroup (168 of them for 5376 -> 2688) 39 rows took 41
 * us, 10 more for every 16 rows, deeper pipelines or whole-line loads made no
 * difference; 32 columns and three pieces read half of it, on all CUs.
 * Measured (39 rows, 256 -> 5376 and 5376 -> 2688, with the reduction):
 * 8.7 and 27.6 us (22.9 and 4.7), from 211 and 2284. */
enum { HK_LF_WAVES = 8, HK_LF_BLOCKS = 2 };

struct hk_linear_f32_args {
    const float *x, *w, *bias;
    float *c;         /* [M, N], or with pieces their sums [piece][M, N] */
    uint32_t m, n, k, x_bytes, w_bytes;
    uint32_t piece_steps; /* 32-wide k steps of a piece */
};

template <int MB, int DEPTH>
__global__ void __launch_bounds__(HK_LF_WAVES * 64)
hk_linear_f32_mfma(hk_linear_f32_args g) {
    constexpr int NB = HK_LF_BLOCKS;
    extern __shared__ __attribute__((aligned(16))) float hk_lf_red[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, quad = lane >> 4;
    const uint32_t n0 = blockIdx.x * (16u * NB);
    const uint32_t m0 = blockIdx.y * (16u * MB);
    const uint32_t m = g.m, n = g.n, k = g.k;
    const __amdgpu_buffer_rsrc_t xr = hk_proj_rsrc(g.x, g.x_bytes);
    const __amdgpu_buffer_rsrc_t wr = hk_proj_rsrc(g.w, g.w_bytes);
    /* this wave's 32-wide k steps of the workgroup's piece */
    const uint32_t begin = blockIdx.z * g.piece_steps;
    const uint32_t steps = min(g.piece_steps, (k + 31u) / 32u - begin);
    const uint32_t first = begin + steps * wave / HK_LF_WAVES;
    const uint32_t last = begin + steps * (wave + 1u) / HK_LF_WAVES;
    /* rows past the end start at the buffer's end and read zeros; so does
     * the part of a last step past K, on both operands */
    uint32_t w_off[NB], x_off[MB];
#pragma unroll
    for (int a = 0; a < NB; a++)
        w_off[a] = min(n0 + 16u * a + r16, n) * k * 4u + quad * 16u;
#pragma unroll
    for (int b = 0; b < MB; b++)
        x_off[b] = min(m0 + 16u * b + r16, m) * k * 4u + quad * 16u;
    hk_v4i wf[DEPTH][NB][2], xf[DEPTH][MB][2];
    auto load = [&](int slot, uint32_t step) {
        bool in[2];
#pragma unroll
        for (uint32_t h = 0; h < 2; h++)
            in[h] = step < last && step * 32u + h * 16u + quad * 4u < k;
#pragma unroll
        for (int a = 0; a < NB; a++)
#pragma unroll
            for (uint32_t h = 0; h < 2; h++)
                wf[slot][a][h] = __builtin_amdgcn_raw_buffer_load_b128(
                    wr, in[h] ? w_off[a] + step * 128u + h * 64u : g.w_bytes,
                    0, 0);
#pragma unroll
        for (int b = 0; b < MB; b++)
#pragma unroll
            for (uint32_t h = 0; h < 2; h++)
                xf[slot][b][h] = __builtin_amdgcn_raw_buffer_load_b128(
                    xr, in[h] ? x_off[b] + step * 128u + h * 64u : g.x_bytes,
                    0, 0);
    };
    hk_f32x4 acc[NB][MB];
#pragma unroll
    for (int a = 0; a < NB; a++)
#pragma unroll
        for (int b = 0; b < MB; b++)
            acc[a][b] = hk_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
        load(d, first + d);
        __builtin_amdgcn_sched_barrier(0); /* in this order: see below */
    }
    for (uint32_t s = first; s < last; s += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            if (s + d >= last) break;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                hk_f32x4 wv[NB], xv[MB];
#pragma unroll
                for (int a = 0; a < NB; a++)
                    wv[a] = __builtin_bit_cast(hk_f32x4, wf[d][a][h]);
#pragma unroll
                for (int b = 0; b < MB; b++)
                    xv[b] = __builtin_bit_cast(hk_f32x4, xf[d][b][h]);
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int a = 0; a < NB; a++)
#pragma unroll
                        for (int b = 0; b < MB; b++)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                wv[a][j], xv[b][j], acc[a][b], 0, 0, 0);
            }
            load(d, s + DEPTH + d);
            /* keeps the loads here: gathered at the loop's end, they were
             * all waited for at its top */
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    /* acc[a][b][i] = C[m0 + 16 b + r16][n0 + 16 a + 4 quad + i], summed over
     * the waves */
    hk_f32x4 *red = (hk_f32x4 *)hk_lf_red;
#pragma unroll
    for (int a = 0; a < NB; a++)
#pragma unroll
        for (int b = 0; b < MB; b++)
            red[((wave * NB + a) * MB + b) * 64u + lane] = acc[a][b];
    __syncthreads();
    float *c = g.c + (size_t)blockIdx.z * m * n;
    for (uint32_t t = tid; t < NB * MB * 64u; t += HK_LF_WAVES * 64u) {
        hk_f32x4 sum = red[t];
#pragma unroll
        for (int v = 1; v < HK_LF_WAVES; v++)
            sum += red[v * NB * MB * 64u + t];
        const uint32_t block = t >> 6;
        const uint32_t row = m0 + block % MB * 16u + (t & 15u);
        const uint32_t col =
            n0 + block / MB * 16u + ((t >> 4) & 3u) * 4u;
        if (row >= m) continue;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (col + i < n)
                c[(size_t)row * n + col + i] =
                    sum[i] + (g.bias ? g.bias[col + i] : 0.0f);
    }
}

/* C = the pieces' sums, in piece order, + bias. */
__global__ void __launch_bounds__(256)
hk_linear_f32_reduce(const float *partial, const float *bias, float *c,
                     uint32_t m, uint32_t n, uint32_t pieces) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= m * n) return;
    float sum = partial[i];
    for (uint32_t p = 1; p < pieces; p++) sum += partial[(size_t)p * m * n + i];
    c[i] = sum + (bias ? bias[i % n] : 0.0f);
}

bool hk_linear_f32(struct h3_gpu *gpu, const float *x, const float *w,
                   const float *bias, float *c, uint32_t m, uint32_t n,
                   uint32_t k) {
    /* 16-byte loads; offsets up to a step past the end of a row past the
     * end stay below 2^32 */
    const uint64_t margin = 4ull * k + 4096;
    if (gpu->reference_kernels || !k || k % 4 || ((uintptr_t)x & 15) ||
        ((uintptr_t)w & 15) || (uint64_t)m * k * 4 + margin >= 0x100000000ull ||
        (uint64_t)n * k * 4 + margin >= 0x100000000ull || m > 65535u * 64u)
        return false;
    /* a handful of products each: one thread an output is done before eight
     * waves have met (K = 16, 128 x 64 outputs 3.5 us against 4.6, 128 x 512
     * 3.5 against 4.8; 300 x 512 7.1 against 4.9) */
    if (k <= 16 && (uint64_t)m * n <= 65536) return false;
    struct {
        uint32_t blocks;
        void (*kernel)(hk_linear_f32_args);
    } const sizes[] = {{1, hk_linear_f32_mfma<1, 4>},
                       {2, hk_linear_f32_mfma<2, 3>},
                       {3, hk_linear_f32_mfma<3, 3>},
                       {4, hk_linear_f32_mfma<4, 2>},
                       {6, hk_linear_f32_mfma<6, 2>},
                       {8, hk_linear_f32_mfma<8, 1>}};
    /* the fewest row blocks of 16 that hold m, at most 8 a workgroup */
    uint32_t at = 0;
    while (at < 5 && sizes[at].blocks * 16u < m) at++;
    const uint32_t gx = (n + 16 * HK_LF_BLOCKS - 1) / (16 * HK_LF_BLOCKS);
    const uint32_t cus = gpu->num_cus > 0 ? (uint32_t)gpu->num_cus : 256u;
    const uint32_t steps = (k + 31u) / 32u;
    /* a K too short for pieces: fewer rows a workgroup, from 32 on, while one
     * round of CUs holds them (128 rows x 64 -> 64 5.0 us against 9.2 with all
     * rows in one, and 7.4 of one thread an output; 300 x 256 -> 512 6.4
     * against 11.5; beyond a round 1000 x 128 -> 5376 66 against 56) */
    for (uint32_t few = 1; few < at && steps < 8 * HK_LF_WAVES; few++)
        if ((uint64_t)gx * ((m + 16 * sizes[few].blocks - 1) /
                            (16 * sizes[few].blocks)) <= cus)
            at = few;
    const uint32_t mb = sizes[at].blocks;
    const uint32_t lds =
        HK_LF_WAVES * HK_LF_BLOCKS * mb * 64 * (uint32_t)sizeof(hk_f32x4);
    const uint32_t gy = (m + 16 * mb - 1) / (16 * mb);
    /* pieces of at least 4 steps a wave, while they find idle CUs */
    uint32_t pieces = gx * gy <= cus ? cus / (gx * gy) : 1u;
    if (pieces > steps / (4 * HK_LF_WAVES)) pieces = steps / (4 * HK_LF_WAVES);
    hk_linear_f32_args g = {x, w, bias, c, m, n, k,
                            (uint32_t)((uint64_t)m * k * 4),
                            (uint32_t)((uint64_t)n * k * 4), steps};
    if (pieces > 1) {
        g.piece_steps = (steps + pieces - 1) / pieces;
        pieces = (steps + g.piece_steps - 1) / g.piece_steps;
        float *partial = (float *)hk_splitk_try(
            gpu, (size_t)pieces * m * n * sizeof(float));
        if (partial) {
            g.c = partial;
            g.bias = NULL;
        } else { /* no scratch: in one piece */
            g.piece_steps = steps;
            pieces = 1;
        }
    }
    if (pieces < 1) pieces = 1;
    static uint64_t ready[2]; /* devices whose limit is raised: 96, 128 rows */
    const uint64_t bit = 1ull << (gpu->device & 63);
    if (lds > 64 * 1024 && !(ready[at - 4] & bit)) {
        (void)hipFuncSetAttribute((const void *)sizes[at].kernel,
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds);
        ready[at - 4] |= bit;
    }
    hipLaunchKernelGGL(sizes[at].kernel, dim3(gx, gy, pieces),
                       dim3(HK_LF_WAVES * 64), lds, gpu->stream, g);
    if (pieces > 1)
        hipLaunchKernelGGL(hk_linear_f32_reduce, dim3((m * n + 255) / 256),
                           dim3(256), 0, gpu->stream, g.c, bias, c, m, n,
                           pieces);
    return true;
}

/* ------------------------------------------------------ patch projection
 *
 * F32 in, bf16 out, and bit for bit the reference's hand kernel
 * (h3_cuda_core.cu:374-403): fmaf from the bias in k order.  The F32 MFMA
 * keeps that order (above), so each accumulator starts at the bias and runs
 * through k four at a time, lane quarter q holding k = 4 s + q.
 *
 * Bound by the F32 MFMA rate (1.85 GFLOP for 1792 x 96 -> 5376, 12 us at
 * 155 TFLOP/s; its bytes take 4 us) and a fixed 7 us of starting, filling LDS
 * and storing.  A 64-column x 64-row tile per workgroup (four waves of
 * 32 x 32) needs 18 KiB of LDS and 72 registers, so seven share a CU and
 * one's loads overlap the others' MFMAs; 128 columns (three or four a CU)
 * took 26.8 us and 7.8 at 192 rows, this 26.1 and 5.4.  LDS holds each row's
 * 32-deep k chunk quarter by quarter (k % 4, then k / 4), so that one 16-byte
 * read feeds four MFMAs; a row pitch of 36 floats spreads 16 rows over all
 * banks.  One thread per output had read W rows with a 384-byte stride
 * between lanes: 493 us at 1792 rows. */
enum { HK_PL_COLS = 64, HK_PL_ROWS = 64, HK_PL_K = 32, HK_PL_PITCH = 36 };

__global__ void __launch_bounds__(256)
hk_patch_linear_mfma(const float *x, const float *w, const float *bias,
                     uint16_t *out, const uint32_t *row_map, uint32_t m,
                     uint32_t n, uint32_t k) {
    __shared__ __attribute__((aligned(16)))
    float lds[(HK_PL_COLS + HK_PL_ROWS) * HK_PL_PITCH];
    float *lds_x = lds + HK_PL_COLS * HK_PL_PITCH;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r16 = lane & 15u, quad = lane >> 4;
    const uint32_t n0 = blockIdx.x * HK_PL_COLS, m0 = blockIdx.y * HK_PL_ROWS;
    const uint32_t wn = (wave >> 1) * 32u, wm = (wave & 1u) * 32u;
    /* staging: thread t takes 16-byte piece t % 8 of rows t / 8 + 32 i;
     * rows past the end repeat the last one (their outputs are dropped) */
    const uint32_t piece = tid & 7u, srow = tid >> 3;
    const float *wp[2], *xp[2];
#pragma unroll
    for (uint32_t i = 0; i < 2; i++)
        wp[i] = w + (size_t)min(n0 + srow + 32u * i, n - 1u) * k + piece * 4u;
#pragma unroll
    for (uint32_t i = 0; i < 2; i++)
        xp[i] = x + (size_t)min(m0 + srow + 32u * i, m - 1u) * k + piece * 4u;
    hk_f32x4 wv[2], xv[2];
    auto load = [&](uint32_t k0) {
        if (k0 + piece * 4u >= k) return;
#pragma unroll
        for (int i = 0; i < 2; i++) wv[i] = *(const hk_f32x4 *)(wp[i] + k0);
#pragma unroll
        for (int i = 0; i < 2; i++) xv[i] = *(const hk_f32x4 *)(xp[i] + k0);
    };
    auto put = [&](float *base, hk_f32x4 v) {
#pragma unroll
        for (int e = 0; e < 4; e++) base[e * 8 + piece] = v[e];
    };
#pragma unroll
    for (int i = 0; i < 2; i++) wv[i] = hk_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    xv[0] = xv[1] = wv[0];
    load(0);
    hk_f32x4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const uint32_t col = n0 + wn + 16u * a + quad * 4u;
        acc[a][0] = bias && col < n ? *(const hk_f32x4 *)(bias + col)
                                    : hk_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        acc[a][1] = acc[a][0];
    }
    for (uint32_t k0 = 0; k0 < k; k0 += HK_PL_K) {
#pragma unroll
        for (uint32_t i = 0; i < 2; i++)
            put(lds + (srow + 32u * i) * HK_PL_PITCH, wv[i]);
#pragma unroll
        for (uint32_t i = 0; i < 2; i++)
            put(lds_x + (srow + 32u * i) * HK_PL_PITCH, xv[i]);
        __syncthreads();
        if (k0 + HK_PL_K < k) load(k0 + HK_PL_K);
        const uint32_t steps = min((k - k0) / 4u, 8u);
#pragma unroll
        for (uint32_t g = 0; g < 2; g++) {
            hk_f32x4 wf[2], xf[2];
#pragma unroll
            for (int a = 0; a < 2; a++)
                wf[a] = *(const hk_f32x4 *)(
                    lds + (wn + 16u * a + r16) * HK_PL_PITCH + quad * 8u +
                    g * 4u);
#pragma unroll
            for (int b = 0; b < 2; b++)
                xf[b] = *(const hk_f32x4 *)(
                    lds_x + (wm + 16u * b + r16) * HK_PL_PITCH + quad * 8u +
                    g * 4u);
#pragma unroll
            for (uint32_t s = 0; s < 4; s++)
                if (g * 4u + s < steps)
#pragma unroll
                    for (int a = 0; a < 2; a++)
#pragma unroll
                        for (int b = 0; b < 2; b++)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                wf[a][s], xf[b][s], acc[a][b], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const uint32_t row = m0 + wm + 16u * b + r16;
        if (row >= m) continue;
        uint16_t *dst = out + (size_t)(row_map ? row_map[row] : row) * n;
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const uint32_t col = n0 + wn + 16u * a + quad * 4u;
            if (col < n)
                *(uint2 *)(dst + col) =
                    make_uint2(hk_pack2(acc[a][b][0], acc[a][b][1]),
                               hk_pack2(acc[a][b][2], acc[a][b][3]));
        }
    }
}

bool hk_patch_linear(struct h3_gpu *gpu, const float *x, const float *w,
                     const float *bias, uint16_t *out,
                     const uint32_t *row_map, uint32_t m, uint32_t n,
                     uint32_t k) {
    if (gpu->reference_kernels || !k || k % 4 || n % 4 ||
        ((uintptr_t)x & 15) || ((uintptr_t)w & 15) ||
        ((uintptr_t)bias & 15) || ((uintptr_t)out & 7) ||
        m > 65535u * HK_PL_ROWS)
        return false;
    hipLaunchKernelGGL(hk_patch_linear_mfma,
                       dim3((n + HK_PL_COLS - 1) / HK_PL_COLS,
                            (m + HK_PL_ROWS - 1) / HK_PL_ROWS),
                       dim3(256), 0, gpu->stream, x, w, bias, out, row_map, m,
                       n, k);
    return true;
}

/* ------------------------------------------------------ final adaLN head
 *
 * RMS adaLN of a row, rounded to bf16, times a [N, width] weight (reference
 * h3_cuda_dit.cu:183-234).  One workgroup per row had each row read the
 * whole weight (1 MiB for 96 x 5376) with 2-byte loads.
 *
 * Here a workgroup of sixteen waves takes ROWS rows and 16 NB columns.  Each
 * thread keeps its 8 columns of all the rows in registers, so x is read once
 * and the norm weight and (when the rows share a modulation row, as a
 * target's rows do) the shift and scale once for all of them; the
 * normalised rows go through LDS half a width at a time (16 rows of 5376
 * are 168 KiB) to be MFMA operands (v_mfma_f32_16x16x32_bf16), and the waves
 * split the half's 32-wide k steps, reading weight rows from L2.
 *
 * What bounds it is a workgroup's one dependent chain: x from memory, the
 * statistics, two barriers, the normalised rows to LDS, then the weights
 * (three quarters of the 0.7 MiB that a workgroup reads with NB = 3, which
 * alone takes 5 us of a CU's 64 bytes a clock).  Loading x, norm, shift and
 * scale as MFMA fragments instead (16 lanes repeating each modulation piece)
 * took 41-44 us at 1792 rows x 96 outputs and 21 us at 74 rows x 32; this
 * takes 24.2 and 15.4 us, with the modulation rows' numbers, the modulation
 * and a half's first weights loaded ahead of their use (28.7 and 16.7
 * without).  One workgroup per row: 563 and 198. */
enum { HK_HEAD_WAVES = 16 };

struct hk_head_args {
    const uint16_t *x, *norm, *mod, *w, *bias;
    const uint32_t *row_map;
    float *inverse;
    uint16_t *out;
    uint32_t rows, width, n, slots, shift_slot, scale_slot;
    float epsilon;
};

/* bytes of a normalised row's half in LDS: 16 more than its data, so that
 * the 16 rows of a fragment read start on different banks */
static __host__ __device__ uint32_t hk_head_pitch(uint32_t width) {
    return (width / 32u + 1u) / 2u * 64u + 16u;
}

template <int NB, int ROWS>
__global__ void __launch_bounds__(HK_HEAD_WAVES * 64)
hk_adaln_head_mfma(hk_head_args a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t hk_head_lds[];
    __shared__ float squares[HK_HEAD_WAVES][ROWS];
    __shared__ float inverses[ROWS];
    /* weight steps in flight: as many as the 128 registers hold (of NB = 6
     * even one spills ten; it is still the faster there, see hk_adaln_head) */
    constexpr uint32_t AHEAD = NB > 3 ? 1 : NB * ROWS > 32 ? 2 : 3;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, quad = lane >> 4;
    const uint32_t row0 = blockIdx.x * ROWS;
    const uint32_t n0 = blockIdx.y * (16u * NB);
    const uint32_t steps = a.width / 32u, half_steps = (steps + 1u) / 2u;
    const uint32_t pitch = hk_head_pitch(a.width);
    const uint32_t col = tid * 8u;
    const bool mine = col < a.width;
    /* rows past the end repeat the last one; their outputs are dropped */
    auto row_of = [&](uint32_t r) { return min(row0 + r, a.rows - 1u); };
    /* weight rows past N repeat the last one; those columns are dropped */
    const uint16_t *wr[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
        wr[b] = a.w + (size_t)min(n0 + 16u * b + r16, a.n - 1u) * a.width +
                quad * 8u;
    /* AHEAD steps' weights in flight, a half's first ones from before its
     * rows are ready; steps past the half repeat its last one */
    hk_bf16x8 wf[AHEAD][NB];
    auto load = [&](uint32_t first, uint32_t count, uint32_t s0) {
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; u++)
#pragma unroll
            for (int b = 0; b < NB; b++)
                wf[u][b] = *(const hk_bf16x8 *)(
                    wr[b] +
                    (first + min(s0 + u * HK_HEAD_WAVES, count - 1u)) * 32u);
    };
    if (ROWS == 4) load(0, half_steps, wave); /* the registers allow it */
    const uint32_t at = min(col, a.width - 8u); /* loads without a branch */
    /* every row's modulation row, one a lane: loaded row by row, they were
     * a chain of ROWS loads */
    const uint32_t maps = a.row_map[row_of(lane % ROWS)];
    uint4 xv[ROWS];
#pragma unroll
    for (uint32_t r = 0; r < ROWS; r++)
        xv[r] = *(const uint4 *)(a.x + (size_t)row_of(r) * a.width + at);
    const uint4 nw = *(const uint4 *)(a.norm + at);
    uint4 sh, sc;
    auto load_mod = [&](uint32_t map) {
        const uint16_t *mod = a.mod + (size_t)map * a.slots * a.width + at;
        sh = *(const uint4 *)(mod + (size_t)a.shift_slot * a.width);
        sc = *(const uint4 *)(mod + (size_t)a.scale_slot * a.width);
    };
    /* readlane: a branch on the map must not become a lane mask */
    uint32_t map = __builtin_amdgcn_readlane(maps, 0);
    load_mod(map);
    /* ROWS sums over the wave's 64 lanes: each exchange halves the rows a
     * lane carries, so that the lane's top bits end up naming the row; the
     * other bits are summed as usual */
    float sum[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        float v[8];
        hk_unpack8(xv[r], v);
        sum[r] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) sum[r] = fmaf(v[e], v[e], sum[r]);
        if (!mine) sum[r] = 0.0f;
    }
#pragma unroll
    for (int width = ROWS / 2, bit = 32; width; width >>= 1, bit >>= 1)
#pragma unroll
        for (int r = 0; r < width; r++) {
            const bool high = lane & bit;
            const float keep = high ? sum[r + width] : sum[r];
            const float send = high ? sum[r] : sum[r + width];
            sum[r] = keep + __shfl_xor(send, bit, 64);
        }
#pragma unroll
    for (int bit = 32 / ROWS; bit; bit >>= 1)
        sum[0] += __shfl_xor(sum[0], bit, 64);
    constexpr uint32_t SPAN = 64 / ROWS; /* lanes that hold one row's sum */
    if (lane % SPAN == 0) squares[wave][lane / SPAN] = sum[0];
    /* x stays packed until it is normalised (unpacked, it spilled) */
#pragma unroll
    for (int r = 0; r < ROWS; r++)
        asm volatile("" : "+v"(xv[r].x), "+v"(xv[r].y), "+v"(xv[r].z),
                          "+v"(xv[r].w));
    __syncthreads();
    if (tid < ROWS) {
        float total = 0.0f;
#pragma unroll
        for (int v = 0; v < HK_HEAD_WAVES; v++) total += squares[v][tid];
        const float inverse =
            1.0f / sqrtf(total / (float)a.width + a.epsilon);
        inverses[tid] = inverse;
        if (blockIdx.y == 0 && row0 + tid < a.rows)
            a.inverse[row0 + tid] = inverse;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < ROWS; r++) {
        const uint32_t next = __builtin_amdgcn_readlane(maps, r);
        if (next != map) {
            map = next;
            load_mod(map);
        }
        /* opaque at both ends: many unpacked rows at a time would spill */
        asm volatile("" : "+v"(xv[r].x), "+v"(xv[r].y), "+v"(xv[r].z),
                          "+v"(xv[r].w));
        const float inverse = inverses[r];
        float v[8], w8[8], s8[8], c8[8], y[8];
        hk_unpack8(xv[r], v);
        hk_unpack8(nw, w8);
        hk_unpack8(sh, s8);
        hk_unpack8(sc, c8);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float n = v[e] * inverse * w8[e];
            y[e] = n * (1.0f + c8[e]) + s8[e];
        }
        xv[r] = hk_pack8(y);
        asm volatile("" : "+v"(xv[r].x), "+v"(xv[r].y), "+v"(xv[r].z),
                          "+v"(xv[r].w));
    }
    hk_f32x4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) acc[b] = hk_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (ROWS != 4) load(0, half_steps, wave);
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) {
        const uint32_t first = h * half_steps;
        const uint32_t count = h ? steps - half_steps : half_steps;
        if (h) __syncthreads(); /* the first half has been read */
        if (mine && col / 32u >= first && col / 32u < first + count) {
            uint8_t *dst = hk_head_lds + (col - first * 32u) * 2u;
#pragma unroll
            for (uint32_t r = 0; r < ROWS; r++)
                *(uint4 *)(dst + r * pitch) = xv[r];
        }
        __syncthreads();
        for (uint32_t s0 = wave; s0 < count; s0 += AHEAD * HK_HEAD_WAVES) {
#pragma unroll
            for (uint32_t u = 0; u < AHEAD; u++) {
                const uint32_t s = s0 + u * HK_HEAD_WAVES;
                if (s >= count) break;
                const hk_bf16x8 xf = *(const hk_bf16x8 *)(
                    hk_head_lds + (r16 % ROWS) * pitch + s * 64u +
                    quad * 16u);
#pragma unroll
                for (int b = 0; b < NB; b++)
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        wf[u][b], xf, acc[b], 0, 0, 0);
            }
            if (s0 + AHEAD * HK_HEAD_WAVES < count)
                load(first, count, s0 + AHEAD * HK_HEAD_WAVES);
        }
        if (!h && steps > half_steps)
            load(half_steps, steps - half_steps, wave);
    }
    __syncthreads();
    /* acc[b][i] = out[row0 + r16][n0 + 16 b + 4 quad + i], summed over the
     * waves in wave order */
    hk_f32x4 *red = (hk_f32x4 *)hk_head_lds;
#pragma unroll
    for (int b = 0; b < NB; b++)
        red[(wave * NB + b) * 64u + lane] = acc[b];
    __syncthreads();
    if (tid >= NB * 64u || r16 >= ROWS || row0 + r16 >= a.rows) return;
    hk_f32x4 total = red[tid];
#pragma unroll
    for (int v = 1; v < HK_HEAD_WAVES; v++) total += red[v * NB * 64u + tid];
    const uint32_t c = n0 + (tid >> 6) * 16u + quad * 4u;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (c + i < a.n)
            a.out[(size_t)(row0 + r16) * a.n + c + i] = hk_f2bf(
                a.bias ? total[i] + hk_bf2f(a.bias[c + i]) : total[i]);
}

template <int NB, int ROWS>
static void hk_head_run(struct h3_gpu *gpu, const hk_head_args &a) {
    const size_t tile = (size_t)ROWS * hk_head_pitch(a.width);
    const size_t sums = (size_t)HK_HEAD_WAVES * NB * 64 * sizeof(hk_f32x4);
    const size_t lds = tile > sums ? tile : sums;
    /* over 64 KiB with its static LDS (squares and inverses), the kernel's
     * limit is raised (each process and device once, to the most that a
     * width can need) */
    const size_t fixed = (HK_HEAD_WAVES + 1) * ROWS * sizeof(float);
    static uint64_t ready = 0;
    const uint64_t bit = 1ull << (gpu->device & 63);
    if (lds + fixed > 64 * 1024 && !(ready & bit)) {
        (void)hipFuncSetAttribute(
            (const void *)hk_adaln_head_mfma<NB, ROWS>,
            hipFuncAttributeMaxDynamicSharedMemorySize,
            (int)((size_t)ROWS * hk_head_pitch(HK_HEAD_WAVES * 64 * 8)));
        ready |= bit;
    }
    hipLaunchKernelGGL((hk_adaln_head_mfma<NB, ROWS>),
                       dim3((a.rows + ROWS - 1) / ROWS,
                            (a.n + 16 * NB - 1) / (16 * NB)),
                       dim3(HK_HEAD_WAVES * 64), lds, gpu->stream, a);
}

bool hk_adaln_head(struct h3_gpu *gpu, const uint16_t *x, float *inverse,
                   const uint16_t *norm, const uint16_t *mod,
                   const uint32_t *row_map, const uint16_t *w,
                   const uint16_t *bias, uint16_t *out, uint32_t rows,
                   uint32_t width, uint32_t n, uint32_t slots,
                   uint32_t shift_slot, uint32_t scale_slot, float epsilon) {
    /* a thread per 8 columns, loaded 16 bytes at a time; of a small weight,
     * smaller with many rows, one workgroup a row is faster (us at 74, 1792
     * and 6000 rows, here and there: 64 -> 4 6.8, 10.5 and 19.8, 4.0, 4.1 and
     * 8.1; 64 -> 64 11.3, 12.5 and 26.3, 9.4, 11.9 and 33.5; 256 -> 32 9.5,
     * 12.2 and 23.0, 8.5, 10.7 and 27.8; 128 -> 96 11.4, 12.5 and 28.8, 15.5,
     * 19.4 and 54.4) */
    if (gpu->reference_kernels || width % 32 ||
        (uint64_t)width * n < (rows <= 2048 ? 12288u : 4096u) ||
        width > HK_HEAD_WAVES * 64 * 8 || !n || n > 65535u * 32u ||
        ((uintptr_t)x & 15) || ((uintptr_t)norm & 15) ||
        ((uintptr_t)mod & 15) || ((uintptr_t)w & 15))
        return false;
    const hk_head_args a = {x,       norm, mod, w,     bias,  row_map,
                            inverse, out,  rows, width, n,    slots,
                            shift_slot, scale_slot, epsilon};
    /* 4 rows a workgroup while one round of workgroups covers them (15.4 us
     * against 22 with 16 at 74 rows x 32, where a workgroup's own chain of
     * steps is all that counts), else 16, which read the weights a quarter
     * as often; 96 columns a workgroup where 48 would need a second round
     * (2835 rows: 40.4 us against 50.7), else 48 (1792: 24.2) */
    const uint32_t cus = gpu->num_cus > 0 ? (uint32_t)gpu->num_cus : 256u;
    const uint32_t groups = n <= 32 ? 1u : (n + 47u) / 48u;
    if (n <= 32 && (rows + 3u) / 4u <= cus) hk_head_run<2, 4>(gpu, a);
    else if (n <= 32) hk_head_run<2, 16>(gpu, a);
    else if ((rows + 3u) / 4u * groups <= cus) hk_head_run<3, 4>(gpu, a);
    else if ((rows + 15u) / 16u * groups <= cus) hk_head_run<3, 16>(gpu, a);
    else hk_head_run<6, 16>(gpu, a);
    return true;
}
