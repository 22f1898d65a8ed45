// Kernel-level C ABI for the Q8_0 activation quantizer and the lane GEMV (the device
// counterparts of the reference's quantize_row_q8_0 and oxe_vl_gemv / ggml_gemv_q8_0_4x8_q8_0).
#include "oxe_gemv.h"
#include "oxe_kernels.h"

#include <algorithm>

namespace oxe {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Eight threads per block of 32, four values each: 16-byte loads and 4-byte stores of neighbouring
// threads are neighbours, and a few rows already give every CU some waves (45 rows of 4096: 2.6 us
// with a thread per block, 1.9 so; 2048 rows 7.8, 7.9). The arithmetic is quant_block_q8_0's.
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float *__restrict__ x, int64_t n, int8_t *__restrict__ q,
                                                            uint16_t *__restrict__ d) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;   // whole blocks: a block's eight threads stay together
    const float4 f = *(const float4 *)(x + i);
    const float v[4] = {f.x, f.y, f.z, f.w};
    float am = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) am = fmaxf(am, __builtin_fabsf(v[e]));
    am = fmaxf(am, dpp_f<DPP_XOR1>(am));
    am = fmaxf(am, dpp_f<DPP_XOR2>(am));
    am = fmaxf(am, dpp_f<DPP_HALF_MIRROR>(am));
    const float dd = am / 127.0f;
    const float id = dd != 0.0f ? 1.0f / dd : 0.0f;
    uint32_t u = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) u |= ((uint32_t)((int32_t)__builtin_rintf(v[e] * id) & 0xff)) << (8 * e);
    *(uint32_t *)(q + i) = u;
    if ((threadIdx.x & 7) == 0) d[i / 32] = f2h(dd);
}

int quantize_q8_0(const float *x, int64_t n, int8_t *q, uint16_t *d, hipStream_t st) {
    if (n <= 0 || n % 32 != 0) return -1;
    hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, st, x, n, q, d);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Q8_0 lane GEMV for any k that is a multiple of 32 (the row lengths without a tuned kernel). A
// workgroup's R rows are one run of bytes: thread t takes its 16-byte chunks t, t + 256, ..., four in flight,
// so loads are whole lines for every k (a wave per row read 64 blocks of 32 bytes apart). A chunk's activations
// come from LDS; the two halves of a block are neighbouring lanes' (k / 16 is even). Then one thread per (row,
// lane) runs the fp32 chain over the blocks in order from +0 (ggml_gemv_q8_0_4x8_q8_0, repack_subset.cpp:1672:
// acc = fma(isum, d_x * d_w, acc)), its scales from LDS too. Bound by the latency of one workgroup at the sizes
// that a few workgroups per CU cover. Two lanes, a wave per row before: 3001 x 1120
// 6.3 -> 4.9 us, 4096 x 5120 23.1 -> 13.9, 151936 x 1024 148 -> 34.
template <int NL>
__global__ __launch_bounds__(256) void gemv_any_kernel(int64_t k, int64_t nr, int R, const int8_t *__restrict__ wq,
                                                       const uint16_t *__restrict__ wd, const int8_t *__restrict__ xq,
                                                       const uint16_t *__restrict__ xd, float *__restrict__ y,
                                                       int32_t *__restrict__ isum_out) {
    extern __shared__ __align__(16) uint8_t ga_lds[];
    const int nb = (int)(k / 32), kch = 2 * nb, t = threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.x * R;
    const int rows = (int)(nr - r0 < R ? nr - r0 : R), n = rows * kch;
    u32x4 *s_x = (u32x4 *)ga_lds;                        // [NL][kch]
    int32_t *s_is = (int32_t *)(s_x + NL * kch);         // [NL][R][nb + 1]
    uint16_t *s_xd = (uint16_t *)(s_is + NL * R * (nb + 1));   // [NL][nb]
    uint16_t *s_wd = s_xd + NL * nb;                     // [R][nb]
    const u32x4 *wp = (const u32x4 *)(wq + r0 * k);
    constexpr int U = 4;
    u32x4 w[U];
#pragma unroll
    for (int u = 0; u < U; u++) w[u] = __builtin_nontemporal_load(wp + (t + 256 * u < n ? t + 256 * u : n - 1));
    for (int i = t; i < NL * kch; i += 256) s_x[i] = ((const u32x4 *)xq)[i];
    for (int i = t; i < NL * nb; i += 256) s_xd[i] = xd[i];
    for (int i = t; i < rows * nb; i += 256) s_wd[i] = wd[r0 * nb + i];
    __syncthreads();
    int r = t / kch, c = t % kch;                        // row and chunk of i
    const int dr = 256 / kch, dc = 256 % kch;
    for (int i0 = 0; i0 < n; i0 += 256 * U) {
        u32x4 nx[U];
        const int j0 = i0 + 256 * U + t;
#pragma unroll
        for (int u = 0; u < U; u++) nx[u] = __builtin_nontemporal_load(wp + (j0 + 256 * u < n ? j0 + 256 * u : n - 1));
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (i0 + 256 * u + t < n) {
#pragma unroll
                for (int l = 0; l < NL; l++) {
                    const u32x4 x = s_x[l * kch + c];
                    int32_t s = dot4(w[u][0], x[0], 0);
                    s = dot4(w[u][1], x[1], s);
                    s = dot4(w[u][2], x[2], s);
                    s = dot4(w[u][3], x[3], s);
                    s += dpp_i<DPP_XOR1>(s);   // n is even: both halves of a block are live
                    if ((c & 1) == 0) s_is[(l * R + r) * (nb + 1) + (c >> 1)] = s;
                }
            }
            r += dr;
            c += dc;
            if (c >= kch) {
                c -= kch;
                r++;
            }
            w[u] = nx[u];
        }
    }
    __syncthreads();
    if (t < NL * rows) {
        const int l = t / rows, rr = t % rows;
        const int32_t *is = s_is + (l * R + rr) * (nb + 1);
        float acc = 0.0f;
#pragma unroll 8
        for (int b = 0; b < nb; b++) acc = __builtin_fmaf((float)is[b], h2f(s_xd[l * nb + b]) * h2f(s_wd[rr * nb + b]), acc);
        y[(int64_t)l * nr + r0 + rr] = acc;
    }
    if (isum_out)
        for (int i = t; i < NL * rows * nb; i += 256) {
            const int l = i / (rows * nb), rr = (i / nb) % rows, b = i % nb;
            isum_out[((int64_t)l * nr + r0 + rr) * nb + b] = s_is[(l * R + rr) * (nb + 1) + b];
        }
}
inline size_t gemv_any_lds(int64_t k, int nl, int R) {
    const size_t nb = (size_t)(k / 32);
    return (size_t)nl * k + (size_t)nl * R * (nb + 1) * 4 + (nl * nb + R * nb) * 2;
}
template <int NL>
static void gemv_any_launch(int64_t k, int64_t nr, int R, size_t lds, const int8_t *wq, const uint16_t *wd, const int8_t *xq,
                            const uint16_t *xd, float *y, int32_t *isum, hipStream_t st) {
    hipLaunchKernelGGL(gemv_any_kernel<NL>, dim3((unsigned)((nr + R - 1) / R)), dim3(256), lds, st, k, nr, R, wq, wd, xq, xd, y,
                       isum);
}

// Rows too long for that kernel's LDS or, with their lanes, for enough of its workgroups, and small matrices (700 x 320: 3.3 us against 3.7): one wave per row; lane i forms the exact int32 dots of blocks i, i + 64, ...
// for every activation lane, then thread l of the wave runs lane l's chain over the blocks.
constexpr int GG_ROWS = 4;
__global__ __launch_bounds__(64 * GG_ROWS) void gemv_long_kernel(int64_t k, int64_t nr, int nl, const int8_t *__restrict__ wq,
                                                               const uint16_t *__restrict__ wd, const int8_t *__restrict__ xq,
                                                               const uint16_t *__restrict__ xd, float *__restrict__ y,
                                                               int32_t *__restrict__ isum_out) {
    extern __shared__ int32_t gg_isum[];   // [GG_ROWS][nl][nb]
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t nb = k / 32, r = (int64_t)blockIdx.x * GG_ROWS + w;
    int32_t *is = gg_isum + (int64_t)w * nl * nb;
    if (r < nr) {
        for (int64_t b = lane; b < nb; b += 64) {
            const uint4 *wp = (const uint4 *)(wq + r * k + 32 * b);
            const uint4 w0 = wp[0], w1 = wp[1];
            for (int l = 0; l < nl; l++) {
                const uint4 *xp = (const uint4 *)(xq + l * k + 32 * b);
                is[l * nb + b] = dot16(w1, xp[1], dot16(w0, xp[0], 0));
            }
        }
    }
    __syncthreads();
    if (r < nr && lane < nl) {
        const int l = lane;
        float acc = 0.0f;
        for (int64_t b = 0; b < nb; b++) {
            const int32_t v = is[l * nb + b];
            acc = __builtin_fmaf((float)v, h2f(xd[l * nb + b]) * h2f(wd[r * nb + b]), acc);
            if (isum_out) isum_out[((int64_t)l * nr + r) * nb + b] = v;
        }
        y[(int64_t)l * nr + r] = acc;
    }
}

}  // namespace oxe

extern "C" {

int oxe_hip_quantize_row_q8_0(const float *x, int64_t k, int64_t nrows, int8_t *q, uint16_t *d, void *stream) {
    if (k <= 0 || k % 32 != 0 || nrows <= 0) return -1;
    return oxe::quantize_q8_0(x, k * nrows, q, d, (hipStream_t)stream);
}

// oxe_vl_gemv's contract (crates/kernels-sys/csrc/oxe_vl.inc:78-107, bound as `!= 0` by
// gemv_lanes_raw, crates/kernels-sys/src/lib.rs:652-666): 1 when done; 0 with nothing written when
// there is no kernel for the call (lanes outside 1..4, no rows, k not a positive multiple of 32 or
// past the one-wave-per-row kernel's LDS); -2 on a launch error
int oxe_hip_gemv_q8_0(int64_t k, int64_t nr, int nl, const int8_t *wq, const uint16_t *wd, const int8_t *xq,
                      const uint16_t *xd, float *y, int32_t *isum, void *stream) {
    if (nr <= 0 || nl < 1 || nl > oxe::GEMV_MAX_LANES || k <= 0 || k % 32 != 0) return 0;
    if (k != 512 && k != 2048 && k != 4096) {
        // about 1024 chunks of 16 bytes per workgroup (its threads' first loads hold most of its rows), fewer rows
        // where that leaves CUs without a workgroup
        int R = (int)std::min<int64_t>(16, std::max<int64_t>(1, (16 * 1024 + k / 2) / k));
        R = (int)std::min<int64_t>(R, std::max<int64_t>(2, nr / 512));
        while (R > 1 && oxe::gemv_any_lds(k, nl, R) > 64 * 1024) R--;
        const size_t need = oxe::gemv_any_lds(k, nl, R);
        // its workgroups stage the lanes' activations: over many rows that pays where the rows in flight on a CU, as many
        // workgroups as its LDS holds, come to 43 KB. Against a wave per row, us: 8192 x 8192, 4 lanes (48 KB) 61 / 80, 9216 x 8192,
        // 4 lanes (54) 69 / 91, 11008 x 8192, 3 lanes (43) 101 / 117 and
        // x 4096 58 / 56, 18944 x 4096, 2 lanes (56) 96 / 91; but 12288 x 4096, 4 lanes (24) 100 / 59, 16384 x 4096, 3 lanes (32)
        // 123 / 76, 12288 x 4096, 3 lanes (36) 72 / 59, 10240 x 4096, 4 lanes (40) 53 / 49. Up to 1536 rows its latency
        // is the shorter one all the same (10240 x 1500, 4 lanes 26 / 34, 16384 x 1024, 3 lanes 39 / 50)
        const bool pays = nr <= 1536 || (int64_t)(160 * 1024 / std::max<size_t>(1, need)) * R * k >= 43 * 1024;
        // its phases cost more than its lines save on a small matrix: 2^19 weights, 7 * 2^17 where rows are short but
        // hold a few blocks and the lanes are few (us, 2^19.3 weights: k 320, one lane 4.2 / 3.5, 448, four lanes 4.7 / 4.4; but k 160,
        // three 4.1 / 4.1, 64, one 3.4 / 4.9, 768, one 3.9 / 4.4)
        const int64_t small = k >= 128 && k <= 640 && 80 * nl <= k ? 7 << 17 : 1 << 19;
        if (nr * k > small && need <= 64 * 1024 && pays && ((uintptr_t)wq | (uintptr_t)xq) % 16 == 0) {
            const hipStream_t st = (hipStream_t)stream;
            if (nl == 1) oxe::gemv_any_launch<1>(k, nr, R, need, wq, wd, xq, xd, y, isum, st);
            else if (nl == 2) oxe::gemv_any_launch<2>(k, nr, R, need, wq, wd, xq, xd, y, isum, st);
            else if (nl == 3) oxe::gemv_any_launch<3>(k, nr, R, need, wq, wd, xq, xd, y, isum, st);
            else oxe::gemv_any_launch<4>(k, nr, R, need, wq, wd, xq, xd, y, isum, st);
            return hipGetLastError() == hipSuccess ? 1 : -2;
        }
        const size_t lds = (size_t)oxe::GG_ROWS * nl * (k / 32) * sizeof(int32_t);
        if (lds > 64 * 1024) return 0;   // k > 32768 with 4 lanes, 65536 with 2, 131072 with 1
        hipLaunchKernelGGL(oxe::gemv_long_kernel, dim3((unsigned)((nr + oxe::GG_ROWS - 1) / oxe::GG_ROWS)),
                           dim3(64 * oxe::GG_ROWS), lds, (hipStream_t)stream, k, nr, nl, wq, wd, xq, xd, y, isum);
        return hipGetLastError() == hipSuccess ? 1 : -2;
    }
    oxe::EpiStore epi{y, nr, nullptr, 0};
    if (oxe::gemv_launch_k(k, nl, wq, wd, nr, oxe::Acts{xq, xd}, isum, epi, (hipStream_t)stream) != 0) return 0;
    return hipGetLastError() == hipSuccess ? 1 : -2;
}

}  // extern "C"
