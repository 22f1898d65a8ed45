// Batched Q8_0 GEMM for prefill: y[t][r] = W[r] . x[t] for T tokens, the reference's
// ggml_gemm_q8_0_4x8_q8_0 (vendor/ggml-subset/generated/repack_subset.cpp:3804-3954), whose
// per (row, token) result equals the Q8_0 GEMV's bit for bit (docs/lab-notes/M3-PREFILL.md:70-71):
// for each 32-element block b in order, acc = fma(f32(isum_b), d_x[t][b] * d_w[r][b], acc) from +0,
// isum_b the exact int32 dot of the block's codes.
//
// The int32 block dots are int8 matrix-core products (v_mfma_i32_32x32x32_i8: a 32 x 32 tile of one
// block's dots per instruction, exact in any order; any split of the block's 32 codes over the
// lanes gives the same sums as long as weights and activations use the same split). The scale
// products d_x[t][b] * d_w[r][b] of both 32-token tiles of a block are one two-block fp32 matrix-core
// outer product (v_mfma_f32_32x32x1_2b_f32: one product per element and nothing added, so each
// element is the correctly rounded fp32 product, the value a VALU multiply gives), in the same
// 32 x 32 output layout as the dots. What is left for the VALU is the chain itself, two operations
// per output and block (convert the block sum, fused multiply-add), one value per (row, token) per
// lane, block by block in order, so the chain is the reference's. The VALU is the kernel's bound.
//
// Workgroup tile: 128 weight rows x 64 tokens, 4 waves of 32 rows x 64 tokens (two 32 x 32 tiles).
// K is staged 4 blocks (128 bytes per row) at a time, double-buffered in LDS and filled by
// direct global-to-LDS loads (global_load_lds_dwordx4 / _dword: no staging registers), so three
// workgroups fit a CU. Code rows (128 bytes) are stored unpadded with their 16-byte chunks
// XOR-swizzled by f(r) = (r & 7) ^ ((r >> 3) & 1): the 16-byte fragment reads of 8 consecutive rows
// cover 8 distinct chunk slots of 128 bytes, and those of 16 consecutive rows 16 distinct 16-byte
// slots of 256 bytes, so neither a 32-bank nor a 64-bank LDS sees a conflict.
// Scales are staged as the raw f16 (4 per row and stage) and converted when read.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/oxe_amd.h"
#include "oxe_common.h"
#include "oxe_gemm.h"

namespace oxe {

namespace gm {
constexpr int BM = 128, BN = 64;       // rows, tokens per workgroup
constexpr int KC = 128;                // K bytes (4 blocks) per stage
constexpr int NBC = KC / 32;           // blocks per stage
constexpr int NT = 256;                // threads
constexpr int WR = 32;                 // weight rows per wave
}  // namespace gm

// one stage of LDS: codes [row][KC] with chunk c of row r at slot c ^ f(r); scales [row][NBC] f16
struct GemmStage {
    int8_t w[gm::BM * gm::KC];
    int8_t x[gm::BN * gm::KC];
    uint16_t dw[gm::BM * gm::NBC];
    uint16_t dx[gm::BN * gm::NBC];
};

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void glb_void;

// global -> LDS, 16 or 4 bytes per lane; lane i's bytes land at dst + 16 i (4 i), dst wave-uniform
__device__ __forceinline__ void to_lds16(const void *src, void *dst) {
    __builtin_amdgcn_global_load_lds((glb_void *)src, (lds_void *)dst, 16, 0, 0);
}
__device__ __forceinline__ void to_lds4(const void *src, void *dst) {
    __builtin_amdgcn_global_load_lds((glb_void *)src, (lds_void *)dst, 4, 0, 0);
}

__global__ __launch_bounds__(gm::NT, 3) void gemm_q8_kernel(GemmArgs a, int vec4) {
    using namespace gm;
    __shared__ __align__(16) GemmStage st0, st1;
    __shared__ int64_t sxr[BN];   // activation row of each of the tile's output rows (-1: none)
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t k = a.k, nr = a.nr, nb = k / 32;
    // plain GEMMs with a partial last row tile dispatch its workgroups after all full ones, and its
    // waves without a valid row skip the arithmetic: the round that holds them is short
    int64_t bx = blockIdx.x, by = blockIdx.y;
    if (!a.tiles) {
        const int64_t nfull = nr / BM;
        if (nfull < (int64_t)gridDim.x) {
            const int64_t L = (int64_t)blockIdx.y * gridDim.x + blockIdx.x, nf = nfull * gridDim.y;
            if (L < nf) {
                bx = L % nfull;
                by = L / nfull;
            } else {
                bx = nfull;
                by = L - nf;
            }
        }
    }
    const int64_t r0 = bx * BM;
    const bool wave_on = r0 + WR * w < nr;   // wave-uniform
    int64_t p0, pn;
    const int8_t *wq = a.wq;
    const uint16_t *wd = a.wd;
    if (a.tiles) {
        if (a.tile_count && (int)blockIdx.y >= *a.tile_count) return;   // uniform: before any barrier
        const int4 tl = a.tiles[blockIdx.y];
        const bool last = a.last > 0 && tl.x == a.last;
        wq = last ? a.wq_last : wq + (int64_t)tl.x * a.wq_stride;
        wd = last ? a.wd_last : wd + (int64_t)tl.x * a.wd_stride;
        p0 = tl.y;
        pn = tl.z;
    } else {
        p0 = by * BN;
        pn = a.nt - p0 < BN ? a.nt - p0 : BN;
    }
    if (pn <= 0) return;   // uniform
    if (t < BN) sxr[t] = t < pn ? (a.xrow ? (int64_t)a.xrow[p0 + t] : p0 + t) : -1;
    __syncthreads();
    // Loads of one stage. Rows past the matrix (weights) or the tile (tokens) read a valid row
    // instead (the last weight row, the tile's first token): their outputs are never stored, and
    // each output element depends only on its own row's and token's codes and scales.
    // Wave w fills weight rows 32 w .. + 31 (4 x 8 rows of 128 bytes), token rows 16 w .. + 15 (2 x 8
    // rows), the weight scales of its 32 rows and (waves 0, 1) the token scales of rows 32 w .. + 31.
    // Lane L of a code load: row 8 q + (L >> 3) of the group, chunk (L & 7) ^ f(row) of the 128
    // bytes, stored at slot L & 7 (f(row) = (L >> 3) ^ (q & 1): each group starts at a multiple of
    // 8 rows, odd groups at an odd multiple); lane L of a scale load: row L >> 1, f16 pair L & 1.
    const int lr8 = lane >> 3, cch = (lane & 7) ^ lr8;
    const int64_t wlast = nr - 1;
    uint32_t wofs[4], xofs[2], wsofs, xsofs = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int64_t gr = r0 + WR * w + 8 * q + lr8;
        wofs[q] = (uint32_t)((gr < wlast ? gr : wlast) * k + 16 * (cch ^ (q & 1)));
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int64_t xr = sxr[16 * w + 8 * q + lr8];
        xofs[q] = (uint32_t)((xr >= 0 ? xr : sxr[0]) * k + 16 * (cch ^ (q & 1)));
    }
    {
        const int64_t gr = r0 + WR * w + (lane >> 1);
        wsofs = (uint32_t)(((gr < wlast ? gr : wlast) * nb) * 2 + 4 * (lane & 1));
        if (w < 2) {
            const int64_t xr = sxr[32 * w + (lane >> 1)];
            xsofs = (uint32_t)(((xr >= 0 ? xr : sxr[0]) * nb) * 2 + 4 * (lane & 1));
        }
    }
    auto fetch = [&](GemmStage &S, int64_t kc) {
        const int8_t *wb = wq + kc, *xb = a.xq + kc;
        const int8_t *wsb = (const int8_t *)wd + kc / 16, *xsb = (const int8_t *)a.xd + kc / 16;
        if (wave_on) {
#pragma unroll
            for (int q = 0; q < 4; q++) to_lds16(wb + wofs[q], S.w + (WR * w + 8 * q) * KC);
            to_lds4(wsb + wsofs, S.dw + WR * w * NBC);
        }
#pragma unroll
        for (int q = 0; q < 2; q++) to_lds16(xb + xofs[q], S.x + (16 * w + 8 * q) * KC);
        if (w < 2) to_lds4(xsb + xsofs, S.dx + 32 * w * NBC);
    };
    // wave w: rows 32 w .. + 31 of the tile; tile j: tokens 32 j .. + 31. Fragment of a code row:
    // row / token lane & 31, the 16 bytes 16 (lane >> 5) .. of the block, at slot (2 b + (lane >> 5))
    // ^ f(row); f(row) = f(lane & 31) for both operands (their row bases are multiples of 16).
    const int wr = WR * w, fr = lane & 31, fh = lane >> 5;
    int fofs[NBC];
#pragma unroll
    for (int bb = 0; bb < NBC; bb++) fofs[bb] = fr * KC + 16 * ((2 * bb + fh) ^ (fr & 7) ^ ((fr >> 3) & 1));
    float acc[2][16];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[j][v] = 0.0f;
    // one stage's chain: tile j's outputs in this lane are rows wr + 8 q + 4 (lane >> 5) + e
    // (v = 4 q + e), token 32 j + (lane & 31); the two-block scale product's block j is tile j
    auto compute = [&](const GemmStage &S, auto njc) {
        constexpr int NJ = decltype(njc)::value;
        if (!wave_on) return;
        const uint2 hw = *(const uint2 *)&S.dw[(wr + fr) * NBC];   // this lane's weight row, 4 blocks
        const uint2 hx = *(const uint2 *)&S.dx[lane * NBC];        // token `lane`, 4 blocks
        auto dots = [&](int bb, int j) {
            const i32x4 fa = *(const i32x4 *)(S.w + wr * KC + fofs[bb]);
            const i32x4 fb = *(const i32x4 *)(S.x + 32 * KC * j + fofs[bb]);
            const i32x16 zero = {};
            return __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb, zero, 0, 0, 0);
        };
        auto scales = [&](int bb) {
            const uint32_t pw = bb < 2 ? hw.x : hw.y, px = bb < 2 ? hx.x : hx.y;
            const float dw = h2f((uint16_t)(pw >> (16 * (bb & 1)))), dx = h2f((uint16_t)(px >> (16 * (bb & 1))));
            const f32x32 zero = {};
            return __builtin_amdgcn_mfma_f32_32x32x1f32(dw, dx, zero, 0, 0, 0);
        };
        i32x16 s[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) s[j] = dots(0, j);
        f32x32 d = scales(0);
#pragma unroll
        for (int bb = 0; bb < NBC; bb++) {
#pragma unroll
            for (int j = 0; j < NJ; j++) {
#pragma unroll
                for (int v = 0; v < 16; v++) acc[j][v] = __builtin_fmaf((float)s[j][v], d[16 * j + v], acc[j][v]);
                if (bb + 1 < NBC) s[j] = dots(bb + 1, j);
            }
            if (bb + 1 < NBC) d = scales(bb + 1);
        }
    };
    // every wave's loads of a stage done and visible before any wave reads it; every wave done with a
    // stage before it is refilled
    auto stage_sync = [&]() {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    };
    auto run = [&](auto njc) {
        const int64_t ns = k / KC;
        fetch(st0, 0);
        stage_sync();
        for (int64_t i = 0; i < ns; i += 2) {
            if (i + 1 < ns) fetch(st1, (i + 1) * KC);
            compute(st0, njc);
            stage_sync();
            if (i + 1 >= ns) break;
            if (i + 2 < ns) fetch(st0, (i + 2) * KC);
            compute(st1, njc);
            stage_sync();
        }
    };
    // tokens of the tile: a per-expert group fills a tile partly; an empty second tile is skipped
    // (uniform across the workgroup)
    if (pn > 32) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int tt = 32 * j + fr;
        if (tt >= pn) continue;
        const int64_t p = p0 + tt;
        float *yp = a.y + p * a.ldy;
        const float *rp = a.res ? a.res + p * a.ldr : nullptr;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int64_t gr = r0 + wr + 8 * q + 4 * fh;
            float o[4] = {acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
            if (vec4 && gr + 3 < nr) {
                if (rp) {
                    const float4 r4 = *(const float4 *)(rp + gr);
                    o[0] += r4.x; o[1] += r4.y; o[2] += r4.z; o[3] += r4.w;
                }
                *(float4 *)(yp + gr) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (gr + e < nr) yp[gr + e] = rp ? o[e] + rp[gr + e] : o[e];
            }
        }
    }
}

// ---- few tokens -------------------------------------------------------------------------------------
// The same products where the tiles above leave the chip idle (a short prompt: 2048 rows x 45 tokens are
// 16 workgroups, each walking K alone one stage ahead): one wave per TS x TS output tile, TS 16 or 32. A
// wave loads its rows' and tokens' blocks, four at a time, as whole 128-byte lines (8 rows a load) into
// registers, RD stages ahead, and turns each stage into fragments through LDS of its own: no barrier, and a
// wait for a stage leaves the later ones in flight. Fragments read straight from global memory, 16 or 32
// rows of 32 bytes a load, took about 4 cycles of the CU's load path per row; direct global-to-LDS loads
// about 190 cycles each for a lone wave. Scale products of four (TS 16) or two (TS 32) blocks come from one
// rank-1 matrix product: lane group g holds the scale of block b + g. The chain of an output is the one
// above. Bound by the latency of a stage's steps in a lone wave (LDS, matrix product, chain).
// K 4096 x 2048 rows, 45 tokens: 38.3 us by the large tile, 10.5 us.
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// LDS accesses of this wave before it come before those after it (one wave: the LDS runs them in order)
__device__ __forceinline__ void lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int TS>
struct SmallStage {
    static constexpr int RD = TS == 16 ? 6 : 3;                 // stages in flight
    static constexpr int BYTES = 2 * TS * 128 + 2 * TS * 8;     // codes of both operands, their scales
};

template <int TS>
__global__ __launch_bounds__(64) void gemm_q8_small_kernel(GemmArgs a, int vec4) {
    using R = SmallStage<TS>;
    constexpr int NG = 64 / TS;            // lanes per row: 4 of 8 bytes, or 2 of 16 bytes, per block
    constexpr int NV = TS * TS / 64;       // outputs per lane
    constexpr int NS = 4 / NG;             // scale products per stage of four blocks
    typedef typename std::conditional<TS == 16, u32x2, u32x4>::type frag_t;
    __shared__ __align__(16) int8_t sm[R::BYTES];   // one stage
    const int lane = threadIdx.x, fr = lane & (TS - 1), g = lane / TS;
    const int64_t k = a.k, nr = a.nr, nb = k / 32;
    const int64_t p0 = (int64_t)blockIdx.y * TS;
    int64_t pn = a.nt - p0;
    if (pn > TS) pn = TS;
    const int64_t r0 = (int64_t)blockIdx.x * TS;
    // rows past the matrix, tokens past the tile: a valid one, never stored
    auto wrow = [&](int i) { return r0 + i < nr ? r0 + i : nr - 1; };
    auto xrow = [&](int i) -> int64_t {
        const int64_t p = p0 + (i < pn ? i : 0);
        return a.xrow ? (int64_t)a.xrow[p] : p;
    };
    // code loads: lane L of load q fills row 8 q + (L >> 3), slot L & 7 with chunk (L & 7) ^ f(row);
    // scale loads: f16 pair L & 1 of row L >> 1 (TS 16: the weights' rows, then the tokens')
    const int lr8 = lane >> 3;
    uint32_t wofs[TS / 8], xofs[TS / 8], sofs[2 * TS / 32];
#pragma unroll
    for (int q = 0; q < TS / 8; q++) {
        const uint32_t c = 16 * ((lane & 7) ^ lr8 ^ (q & 1));
        wofs[q] = (uint32_t)(wrow(8 * q + lr8) * k) + c;
        xofs[q] = (uint32_t)(xrow(8 * q + lr8) * k) + c;
    }
    const int srow = lane >> 1;
    const bool sx = TS == 16 && lane >= 32;
    if constexpr (TS == 16) {
        sofs[0] = (uint32_t)((sx ? xrow(srow - 16) : wrow(srow)) * nb * 2 + 4 * (lane & 1));
    } else {
        sofs[0] = (uint32_t)(wrow(srow) * nb * 2 + 4 * (lane & 1));
        sofs[1] = (uint32_t)(xrow(srow) * nb * 2 + 4 * (lane & 1));
    }
    const int8_t *wq = a.wq, *wsb = (const int8_t *)a.wd, *xsb = (const int8_t *)a.xd;
    const int8_t *sb0 = TS == 16 && sx ? xsb : wsb;
    struct Stage {
        u32x4 w[TS / 8], x[TS / 8];
        uint32_t s[2 * TS / 32];
    } st[R::RD];
    auto fetch = [&](Stage &G, int64_t i) {
        const int8_t *wb = wq + 128 * i, *xb = a.xq + 128 * i;
#pragma unroll
        for (int q = 0; q < TS / 8; q++) G.w[q] = *(const u32x4 *)(wb + wofs[q]);
#pragma unroll
        for (int q = 0; q < TS / 8; q++) G.x[q] = *(const u32x4 *)(xb + xofs[q]);
        G.s[0] = *(const uint32_t *)(sb0 + 8 * i + sofs[0]);
        if constexpr (TS == 32) G.s[1] = *(const uint32_t *)(xsb + 8 * i + sofs[1]);
    };
    auto put = [&](const Stage &G) {
#pragma unroll
        for (int q = 0; q < TS / 8; q++) *(u32x4 *)(sm + 1024 * q + 16 * lane) = G.w[q];
#pragma unroll
        for (int q = 0; q < TS / 8; q++) *(u32x4 *)(sm + TS * 128 + 1024 * q + 16 * lane) = G.x[q];
        *(uint32_t *)(sm + 2 * TS * 128 + 4 * lane) = G.s[0];
        if constexpr (TS == 32) *(uint32_t *)(sm + 2 * TS * 128 + 256 + 4 * lane) = G.s[1];
    };
    float acc[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] = 0.0f;
    const int sw = (fr & 7) ^ ((fr >> 3) & 1);
    // a stage's fragments in registers; NG blocks' dots and scale products (one rank-1 product)
    struct Frag {
        frag_t w[4], x[4];
        uint16_t dw[NS], dx[NS];
    };
    struct Dots {
        int32_t s[NG][NV];
        float d[NG * NV];
    };
    auto read = [&](Frag &F) {
        const int8_t *S = sm;
        const uint16_t *sd = (const uint16_t *)(S + 2 * TS * 128);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            F.dw[s] = sd[4 * fr + NG * s + g];
            F.dx[s] = sd[4 * (TS + fr) + NG * s + g];
        }
#pragma unroll
        for (int b = 0; b < 4; b++) {
            // lane group g of a row: bytes 8 g .. (TS 16) or 16 g .. (TS 32) of the block
            const int at = fr * 128 + (TS == 16 ? 16 * ((2 * b + (g >> 1)) ^ sw) + 8 * (g & 1) : 16 * ((2 * b + g) ^ sw));
            F.w[b] = *(const frag_t *)(S + at);
            F.x[b] = *(const frag_t *)(S + TS * 128 + at);
        }
    };
    auto dots = [&](const Frag &F, int s, Dots &D) {
        const float dw = h2f(F.dw[s]), dx = h2f(F.dx[s]);
        if constexpr (TS == 16) {
            const f32x16 zero = {};
            const f32x16 t = __builtin_amdgcn_mfma_f32_16x16x1f32(dw, dx, zero, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < NG * NV; v++) D.d[v] = t[v];
        } else {
            const f32x32 zero = {};
            const f32x32 t = __builtin_amdgcn_mfma_f32_32x32x1f32(dw, dx, zero, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < NG * NV; v++) D.d[v] = t[v];
        }
#pragma unroll
        for (int b = 0; b < NG; b++) {
            if constexpr (TS == 16) {
                const i32x4 zero = {};
                const i32x4 t = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, F.w[NG * s + b]),
                                                                     __builtin_bit_cast(long, F.x[NG * s + b]), zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < NV; v++) D.s[b][v] = t[v];
            } else {
                const i32x16 zero = {};
                const i32x16 t = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, F.w[NG * s + b]),
                                                                      __builtin_bit_cast(i32x4, F.x[NG * s + b]), zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < NV; v++) D.s[b][v] = t[v];
            }
        }
    };
    auto chain = [&](const Dots &D) {
#pragma unroll
        for (int b = 0; b < NG; b++)
#pragma unroll
            for (int v = 0; v < NV; v++) acc[v] = __builtin_fmaf((float)D.s[b][v], D.d[NV * b + v], acc[v]);
    };
    const int ng = (int)(k / 128);
#pragma unroll
    for (int j = 0; j < R::RD; j++) {
        fetch(st[j], j < ng ? j : ng - 1);
        __builtin_amdgcn_sched_barrier(0);   // stage by stage, so that a wait covers its own stage only
    }
    // the next stage's fragments are on their way from LDS while the chain runs over the current dots
    Frag F;
    Dots D[NS];
    auto take = [&](Stage &G, int i) {
        lds_fence();   // the previous stage's reads come before these writes
        put(G);
        fetch(G, i + R::RD < ng ? i + R::RD : ng - 1);
        __builtin_amdgcn_sched_barrier(0);
        lds_fence();
        read(F);
        __builtin_amdgcn_sched_barrier(0);   // every read on its way before the chain
    };
    take(st[0], 0);
#pragma unroll
    for (int s = 0; s < NS; s++) dots(F, s, D[s]);
    for (int i = 0; i < ng; i += R::RD) {
#pragma unroll
        for (int j = 0; j < R::RD; j++) {
            const int at = i + j;   // chain of stage at, dots of stage at + 1
            if (at >= ng) break;
            take(st[(j + 1) % R::RD], at + 1);
#pragma unroll
            for (int s = 0; s < NS; s++) {
                chain(D[s]);
                dots(F, s, D[s]);
            }
        }
    }
    if (fr >= pn) return;
    // outputs of a lane: token fr, rows 8 q + 4 g + e (TS 32, v = 4 q + e) or 4 g + e (TS 16)
    const int64_t p = p0 + fr;
    float *yp = a.y + p * a.ldy;
    const float *rp = a.res ? a.res + p * a.ldr : nullptr;
#pragma unroll
    for (int q = 0; q < NV / 4; q++) {
        const int64_t gr0 = r0 + 8 * q + 4 * g;
        float o[4] = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
        if (vec4 && gr0 + 3 < nr) {
            if (rp) {
                const float4 r4 = *(const float4 *)(rp + gr0);
                o[0] += r4.x; o[1] += r4.y; o[2] += r4.z; o[3] += r4.w;
            }
            *(float4 *)(yp + gr0) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (gr0 + e < nr) yp[gr0 + e] = rp ? o[e] + rp[gr0 + e] : o[e];
        }
    }
}

// The tile of a plain GEMM: 16, 32 (one wave each) or 0 (the 128 x 64 workgroup tile). Time of one round of
// tiles at K 4096: 10 us (16), 21 us (32), 38 us (128 x 64, 768 of them resident); a round is about 600 wave tiles (more share
// a CU's load path). Measured, few tokens against the large tile (us): [2048 x 4096] 45 tokens 10.5 / 38, 200: 20 / 39, 701:
// 45 / 40 (stays large); [1024 x 2048] 64: 6.4 / 21.6, 701: 14.7 / 22.6; [12352 x 2048] 3: 9.8 / 18, 64: 17 / 23,
// 100: 28 / 24 (stays large).
static int small_tile(int64_t nr, int64_t nt) {
    auto rounds = [](int64_t tiles, int64_t per) { return tiles > per ? (double)tiles / (double)per : 1.0; };
    auto tiles = [&](int64_t r, int64_t t) { return ((nr + r - 1) / r) * ((nt + t - 1) / t); };
    const double c16 = 10.0 * rounds(tiles(16, 16), 600), c32 = 21.0 * rounds(tiles(32, 32), 600);
    const double big = 38.0 * rounds(tiles(gm::BM, gm::BN), 768);
    return c16 <= c32 && c16 < big ? 16 : c32 < big ? 32 : 0;
}

int gemm_launch(const GemmArgs &a, int64_t ntiles, hipStream_t st) {
    using namespace gm;
    if (a.k <= 0 || a.k % KC != 0 || a.nr <= 0 || a.ldy < a.nr) return -1;
    if (!a.wq || !a.wd || !a.xq || !a.xd || !a.y) return -1;
    // 16-byte loads of codes
    if (((uintptr_t)a.wq | (uintptr_t)a.wd | (uintptr_t)a.xq | (uintptr_t)a.xd) % 16 != 0) return -1;
    // the kernel addresses one weight group's and the activations' codes with 32-bit offsets
    if ((uint64_t)a.nr * (uint64_t)a.k > UINT32_MAX || (uint64_t)a.nt * (uint64_t)a.k > UINT32_MAX) return -1;
    const int64_t ny = a.tiles ? ntiles : (a.nt + BN - 1) / BN;
    if (ny <= 0) return 0;
    // 16-byte output (and residual) accesses where every row group of 4 starts 16-byte aligned
    const int vec4 = a.ldy % 4 == 0 && (uintptr_t)a.y % 16 == 0 && (!a.res || (a.ldr % 4 == 0 && (uintptr_t)a.res % 16 == 0));
    // grouped tiles stay with the large tile: a prompt of 61 tokens streams its experts at 5 TB/s with it (a
    // whole prefill 11.1 ms; their tiles by single waves of 16 or 32: 13.8, 12.7)
    const int ts = a.tiles ? 0 : small_tile(a.nr, a.nt);
    if (ts > 0) {
        const dim3 g((unsigned)((a.nr + ts - 1) / ts), (unsigned)((a.nt + ts - 1) / ts));
        if (ts == 16) hipLaunchKernelGGL(gemm_q8_small_kernel<16>, g, dim3(64), 0, st, a, vec4);
        else hipLaunchKernelGGL(gemm_q8_small_kernel<32>, g, dim3(64), 0, st, a, vec4);
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    hipLaunchKernelGGL(gemm_q8_kernel, dim3((unsigned)((a.nr + BM - 1) / BM), (unsigned)ny), dim3(NT), 0, st, a, vec4);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace oxe

extern "C" {

int oxe_hip_gemm_q8_0(int64_t k, int64_t nr, int64_t nt, const int8_t *wq, const uint16_t *wd, const int8_t *xq,
                      const uint16_t *xd, float *y, int64_t ldy, void *stream) {
    if (nt <= 0) return -1;
    oxe::GemmArgs a{wq, wd, xq, xd, y, nullptr, nr, nt, k, ldy, 0, nullptr, 0, 0, nullptr, nullptr, nullptr, nullptr, 0};
    return oxe::gemm_launch(a, 0, (hipStream_t)stream);
}

}  // extern "C"
