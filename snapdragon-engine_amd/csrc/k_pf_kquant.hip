// Batched prefill over K-quant matrices: y[t][r] = W[r] . x[t] for T tokens as matrix-core GEMMs,
// each (row, token) value the lane GEMV's bit for bit (k_kquant.hip: exact integers per sub-block,
// the reference's float chain per block in order), and the token-parallel kernels around them.
//
// Per type, what the matrix cores form exactly and what is left for the VALU, per output and block
// of 256 weights:
//   Q4_K, Q5_K  the chain takes f32(scale * dot32) per 32 weights. scale * code is at most 63 * 31 =
//               1953 and exact in f16, the activation codes are exact in f16, and every partial sum
//               is an integer below 2^24, so the f16 matrix product with f32 accumulators *is* that
//               float: one fused multiply-add per 32 weights remains (the int8 product would leave
//               a convert, a scale multiply and the fma). The min terms' integer sums are f16
//               products of the mins with the codes' sums of 16 the same way.
//   Q3_K        scale * (code - 4), negated, fits int8 (-128..124): the whole block's integer is one
//               int8 product chain, one convert and one fma per block remain.
//   Q6_K        scale * (code - 32) = 64 h + l with h and l in int8: two int8 product chains, then
//               64 h + l, a convert, a product and an add per block.
// The block scale products d_w * d_x are rank-1 f32 matrix products (nothing added to each product,
// so each is the correctly rounded one).
//
// Workgroup: NW waves of 32 weight rows x up to 64 tokens (two 32 x 32 tiles). A wave stages its own rows' blocks
// through LDS of its own (no barrier: no other wave reads them), loaded as whole lines one block ahead; unpacked straight
// from global memory, 32 rows apart per load, a single-wave workgroup ([2048 x 4096], 701 tokens, Q4_K) took 83 us against
// 55. The tokens' codes go through LDS shared by the waves, 256 bytes a row per stage, double buffered, by direct
// global-to-LDS loads; 128-byte code rows with their 16-byte chunks XOR-swizzled by f(r) = (r & 7) ^ ((r >> 3) & 1), as the
// Q8_0 GEMM's. Bound by the VALU (unpacking, and the chain): in the largest launches it issues in 48 to 59 % of the
// cycles (the Q8_0 GEMM's in 61 %), with the matrix cores busy 17 to 25 %, at two waves per SIMD (three for Q3_K; one for
// single-wave workgroups).
//
// Measured, 2048 tokens: [12352 x 2048] Q3_K 141 us, Q5_K 341, Q6_K 239; [9216 x 2048] Q4_K 165.
// A 701-token prompt through 8 layers of the Ornith file's types: 419 ms as decode runs of two positions, 4.9 ms.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/oxe_amd.h"
#include "oxe_kq_block.h"
#include "oxe_pf_kquant.h"
#include "oxe_prologue.h"
#include "oxe_shape.h"

namespace oxe {
namespace kqg {

using kq::QK;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void glb_void;

OXE_DEV void to_lds16(const void *src, void *dst) {
    __builtin_amdgcn_global_load_lds((glb_void *)src, (lds_void *)dst, 16, 0, 0);
}
OXE_DEV h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
OXE_DEV uint32_t as_u(h2 v) { return __builtin_bit_cast(uint32_t, v); }
OXE_DEV f32x16 mfma_f16(const uint32_t (&a)[4], i32x4 b, f32x16 c) {
    const i32x4 av = {(int)a[0], (int)a[1], (int)a[2], (int)a[3]};
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, av), __builtin_bit_cast(h8, b), c, 0, 0, 0);
}
OXE_DEV i32x16 mfma_i8(const uint32_t (&a)[4], i32x4 b, i32x16 c) {
    const i32x4 av = {(int)a[0], (int)a[1], (int)a[2], (int)a[3]};
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(av, b, c, 0, 0, 0);
}
// (byte i of w) as an f16 pair (b, b): 0x64 above a byte is 1024 + b in f16
template <int I>
OXE_DEV h2 byte_pair(uint32_t w) {
    const uint32_t u = __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u + 0x00010001u * I);
    return as_h2(u) - h2{(_Float16)1024.0f, (_Float16)1024.0f};
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// 16 bytes (and the two after them) at LDS address p + sh, p a multiple of 16, sh 0 or 2
struct Run {
    u32x4 w;
    uint32_t x;
    OXE_DEV void load(const uint8_t *p) {
        w = *(const u32x4 *)p;
        x = *(const uint32_t *)(p + 16);
    }
    OXE_DEV uint32_t get(int i, int sh) const { return __builtin_amdgcn_alignbyte(i < 3 ? w[i + 1] : x, w[i], sh); }
};

// A block's bytes as a wave stages them: 32 rows, CH chunks of 16 bytes each, STRIDE bytes apart in LDS (8 consecutive
// rows' 16-byte reads fall on distinct banks; the 4-byte reads behind them conflict, 13 % of Q3_K's LDS cycles and 29 % of
// Q6_K's). Q6_K's 14 chunks end 12 bytes past its block: past the matrix's last block they read its allocation's margin. Q3_K / Q6_K blocks (110 / 210 bytes) of odd index start 2 bytes past a
// dword (rows hold an even number of blocks): they are staged from the dword before, and read with that shift.
template <int TY> struct Geo;
template <> struct Geo<3> { static constexpr int BB = 110, CH = 7, STRIDE = 112; };
template <> struct Geo<4> { static constexpr int BB = 144, CH = 9, STRIDE = 144; };
template <> struct Geo<5> { static constexpr int BB = 176, CH = 11, STRIDE = 176; };
template <> struct Geo<6> { static constexpr int BB = 210, CH = 14, STRIDE = 240; };

// ---- one lane's share of a staged block: row lane & 31, half hf = lane >> 5 of every 32-weight sub-block -------
// Q3_K: bytes 16 hf .. of the high-bit mask and of each 128-weight half's codes; Q6_K: of each half's low and high
// code bits
struct Raw3 {
    Run hm, qs[2];
    OXE_DEV void load(const uint8_t *b, int hf) {
        hm.load(b + 16 * hf);
#pragma unroll
        for (int n = 0; n < 2; n++) qs[n].load(b + 32 + 32 * n + 16 * hf);
    }
};
struct Raw6 {
    Run ql[2], qh;
    OXE_DEV void load(const uint8_t *b, int hf, int n) {
        ql[0].load(b + 64 * n + 16 * hf);
        ql[1].load(b + 64 * n + 32 + 16 * hf);
        qh.load(b + 128 + 32 * n + 16 * hf);
    }
};

// the f16 fragments of one 64-weight step: lo / hi 32 weights (p), matrix product m of 16
// (qs: the lane's 16 nibble bytes of the step; qh: Q5_K's high-bit bytes)
template <int TY>
OXE_DEV void step_frags(u32x4 qs, u32x4 qh, int g, h2 s_lo, h2 s_hi, uint32_t (&lo)[2][4], uint32_t (&hi)[2][4]) {
    const h2 k1024 = h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
    const h2 c_lo = s_lo * k1024, c_hi = s_hi * k1024;   // exact: at most 63 * 2^10
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t w = qs[i];
        // pairs (code 0, code 2) and (code 1, code 3) of the dword's four bytes
        uint32_t l0 = (w & 0x000f000fu) | 0x64006400u, l1 = ((w >> 8) & 0x000f000fu) | 0x64006400u;
        uint32_t h0 = ((w >> 4) & 0x000f000fu) | 0x64006400u, h1 = ((w >> 12) & 0x000f000fu) | 0x64006400u;
        if constexpr (TY == 5) {
            const uint32_t q = qh[i];
            const uint32_t bl = (q >> (2 * g)) & 0x01010101u, bh = (q >> (2 * g + 1)) & 0x01010101u;
            l0 |= (bl & 0x00010001u) << 4;
            l1 |= (bl >> 4) & 0x00100010u;
            h0 |= (bh & 0x00010001u) << 4;
            h1 |= (bh >> 4) & 0x00100010u;
        }
        // (1024 + code) * s - 1024 * s = code * s, one rounding of an exact value
        lo[i >> 1][2 * (i & 1)] = as_u(__builtin_elementwise_fma(as_h2(l0), s_lo, c_lo));
        lo[i >> 1][2 * (i & 1) + 1] = as_u(__builtin_elementwise_fma(as_h2(l1), s_lo, c_lo));
        hi[i >> 1][2 * (i & 1)] = as_u(__builtin_elementwise_fma(as_h2(h0), s_hi, c_hi));
        hi[i >> 1][2 * (i & 1) + 1] = as_u(__builtin_elementwise_fma(as_h2(h1), s_hi, c_hi));
    }
}

// Q3_K, sub-block j of half n: the 16 codes' products with s = 32 - raw scale, by byte lookup:
// (code - 4) * s for code 0..7 in two dwords
OXE_DEV void q3_frag(const Raw3 &r, int sh, int n, int j, int s, uint32_t (&f)[4]) {
    const uint32_t s1 = (uint32_t)s & 255u, s2 = (uint32_t)(2 * s) & 255u, s3 = (uint32_t)(3 * s) & 255u;
    const uint32_t n1 = (uint32_t)-s & 255u, n2 = (uint32_t)(-2 * s) & 255u, n3 = (uint32_t)(-3 * s) & 255u;
    const uint32_t n4 = (uint32_t)(-4 * s) & 255u;
    const uint32_t thi = s1 << 8 | s2 << 16 | s3 << 24, tlo = n4 | n3 << 8 | n2 << 16 | n1 << 24;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t c = ((r.qs[n].get(i, sh) >> (2 * j)) & 0x03030303u) | (((r.hm.get(i, sh) >> (4 * n + j)) & 0x01010101u) << 2);
        f[i] = __builtin_amdgcn_perm(thi, tlo, c);
    }
}

typedef short s2v __attribute__((ext_vector_type(2)));
// Q6_K, sub-block q of half n: s * (code - 32) = 64 h + l of the 16 codes
OXE_DEV void q6_frag(const Raw6 &r, int sh, int q, int s, uint32_t (&fh)[4], uint32_t (&fl)[4]) {
    const s2v sv = {(short)s, (short)s}, off = {(short)(-32 * s), (short)(-32 * s)};
    const s2v six = {6, 6};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t a = r.ql[q & 1].get(i, sh) >> (q >= 2 ? 4 : 0), b = r.qh.get(i, sh);
        const uint32_t c = (a & 0x0f0f0f0fu) | (((b >> (2 * q)) & 0x03030303u) << 4);
        const s2v e = __builtin_bit_cast(s2v, c & 0x00ff00ffu), o = __builtin_bit_cast(s2v, (c >> 8) & 0x00ff00ffu);
        const s2v ve = e * sv + off, vo = o * sv + off;
        const uint32_t he = __builtin_bit_cast(uint32_t, ve >> six), ho = __builtin_bit_cast(uint32_t, vo >> six);
        const uint32_t le = __builtin_bit_cast(uint32_t, ve) & 0x003f003fu, lo = __builtin_bit_cast(uint32_t, vo) & 0x003f003fu;
        fh[i] = __builtin_amdgcn_perm(ho, he, 0x06020400u);   // bytes e0, o0, e1, o1
        fl[i] = le | (lo << 8);
    }
}

constexpr int BN = 64;   // tokens per workgroup

// LDS accesses of this wave before it come before those after it (wave-private rows: no barrier)
OXE_DEV void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// chunk swizzle of a 128-byte code row
OXE_DEV int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

template <int TY, int NW>
__global__ __launch_bounds__(64 * NW, 2) void kq_gemm_kernel(KqGemmArgs a) {
    constexpr bool F16 = TY == 4 || TY == 5;
    using G = Geo<TY>;
    constexpr int XB = F16 ? 512 : 256;   // code bytes of a token and block
    constexpr int SPB = XB / 256;         // token stages per block, of two 128-byte units
    constexpr int NLD = (32 * G::CH + 63) / 64;   // 16-byte weight loads per lane and block
    __shared__ __align__(16) uint8_t sx[2][2 * BN * 128];
    __shared__ __align__(16) uint8_t sw[NW][32 * G::STRIDE];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, fr = lane & 31, hf = lane >> 5;
    const int nb = a.nb;
    // the row tile's segment (fixed indices: the table stays in the kernel arguments)
    KqGemmSeg sg = a.seg[0];
    int tile = blockIdx.x;
#pragma unroll
    for (int j = 1; j < KQG_SEGS; j++)
        if (j < a.nseg && (int)blockIdx.x >= a.tile0[j]) {
            sg = a.seg[j];
            tile = (int)blockIdx.x - a.tile0[j];
        }
    int64_t p0, pn;
    const uint8_t *wb = sg.w;
    if (a.tiles) {
        if (a.tile_count && (int)blockIdx.y >= *a.tile_count) return;   // uniform: before any barrier
        const int4 tl = a.tiles[blockIdx.y];
        wb += (int64_t)tl.x * sg.gstride;
        p0 = tl.y;
        pn = tl.z;
    } else {
        p0 = (int64_t)blockIdx.y * BN;
        pn = a.nt - p0 < BN ? a.nt - p0 : BN;
    }
    if (pn <= 0) return;   // uniform
    const int64_t r0 = (int64_t)tile * (32 * NW) + 32 * w;
    const bool wave_on = r0 < sg.nr;   // wave-uniform
    // weight loads: lane's chunk i = lane + 64 j of the wave's 32 rows x CH chunks (past the rows: the last row's)
    uint32_t wofs[NLD];
    int wdst[NLD];
#pragma unroll
    for (int j = 0; j < NLD; j++) {
        const int i = lane + 64 * j < 32 * G::CH ? lane + 64 * j : 32 * G::CH - 1, r = i / G::CH, c = i % G::CH;
        const int64_t row = r0 + r < sg.nr ? r0 + r : sg.nr - 1;
        wofs[j] = (uint32_t)(row * (int64_t)nb * G::BB + 16 * c);
        wdst[j] = r * G::STRIDE + 16 * c;
    }
    // activation row of token slot i of the tile (past the tile: its first token, never stored)
    auto xrow = [&](int i) -> int64_t {
        const int64_t p = p0 + (i < pn ? i : 0);
        return a.xrow ? (int64_t)a.xrow[p] : p;
    };
    auto run = [&](auto njc) {
        constexpr int NJ = decltype(njc)::value;
        constexpr int RG = 4 * NJ;                       // 8-row groups of the stage
        constexpr int RPW = (RG + NW - 1) / NW;          // row groups per wave
        uint32_t xofs[RPW];
#pragma unroll
        for (int k = 0; k < RPW; k++) {
            const int row = 8 * (w * RPW + k) + (lane >> 3);
            xofs[k] = (uint32_t)(xrow(row) * (int64_t)nb * XB + 16 * ((lane & 7) ^ swz(row)));
        }
        const uint8_t *xc = F16 ? (const uint8_t *)a.x.c16 : (const uint8_t *)a.x.c8;
        auto fetch = [&](int buf, int st) {   // stage st: code bytes 256 st .. of every token row
#pragma unroll
            for (int k = 0; k < RPW; k++)
                if (w * RPW + k < RG) {
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        to_lds16(xc + (xofs[k] + (uint32_t)(st * 256 + 128 * u)), &sx[buf][(u * BN + 8 * (w * RPW + k)) * 128]);
                }
        };
        // block scale of token `lane` (both tiles in one rank-1 product) and, Q4_K / Q5_K, the sums of
        // 16 of token 32 j + fr, codes 8 hf ..
        const int64_t xr64 = xrow(NJ == 2 ? lane : fr);
        const float *xdp = a.x.d + xr64 * nb;
        const uint16_t *bsp[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) bsp[j] = F16 ? a.x.bs + xrow(32 * j + fr) * (int64_t)nb * 16 + 8 * hf : nullptr;
        u32x4 stg[NLD];
        float dx = 0.0f;
        i32x4 bs[NJ];
        auto wload = [&](int b) {
            const uint8_t *p = wb + (b * G::BB - (F16 ? 0 : 2 * (b & 1)));
#pragma unroll
            for (int j = 0; j < NLD; j++) __builtin_memcpy(&stg[j], __builtin_assume_aligned(p + wofs[j], F16 ? 16 : 4), 16);
            dx = xdp[b];
            if constexpr (F16) {
#pragma unroll
                for (int j = 0; j < NJ; j++) bs[j] = *(const i32x4 *)(bsp[j] + 16 * b);
            }
        };
        // the staged block to this wave's LDS rows: its reads of the block before come first, those of this one after
        auto wput = [&]() {
            wave_fence();
#pragma unroll
            for (int j = 0; j < NLD; j++) *(u32x4 *)&sw[w][wdst[j]] = stg[j];
            wave_fence();
        };
        const uint8_t *wl = &sw[w][fr * G::STRIDE];   // this lane's row
        float acc[NJ][16];
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[j][v] = 0.0f;
        const f32x32 zero32 = {};
        const f32x16 zero16 = {};
        auto frag = [&](int buf, int u, int c, int j) {
            return *(const i32x4 *)&sx[buf][(u * BN + 32 * j + fr) * 128 + 16 * (c ^ swz(fr))];
        };
        auto stage_sync = [&]() {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
        };
        const int ns = nb * SPB;
        fetch(0, 0);
        wload(0);
        for (int b = 0; b < nb; b++) {
            stage_sync();   // the stage's codes in LDS, every wave done with the other buffer
            const float dxb = dx;
            i32x4 bsb[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) bsb[j] = bs[j];
            if (SPB * b + 1 < ns) fetch((SPB * b + 1) & 1, SPB * b + 1);
            wput();
            if (b + 1 < nb) wload(b + 1);
            if constexpr (F16) {
                const u32x4 hdr = *(const u32x4 *)wl;
                u32x4 qh = {};
                if constexpr (TY == 5) qh = *(const u32x4 *)(wl + 16 + 16 * hf);
                const float dw = h2f((uint16_t)hdr[0]), dm = h2f((uint16_t)(hdr[0] >> 16));
                // the eight 6-bit scales and mins, four bytes a dword (get_scale_min_k4)
                const uint32_t s0 = hdr[1], s1 = hdr[2], s2 = hdr[3];
                const uint32_t sc[2] = {s0 & 0x3f3f3f3fu, (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u)};
                const uint32_t mn = hf ? ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u) : s1 & 0x3f3f3f3fu;
                const f32x32 ds = __builtin_amdgcn_mfma_f32_32x32x1f32(dw, dxb, zero32, 0, 0, 0);
                uint32_t mf[4] = {as_u(byte_pair<0>(mn)), as_u(byte_pair<1>(mn)), as_u(byte_pair<2>(mn)), as_u(byte_pair<3>(mn))};
                // acc -= (sum of mins * code sums) * (dmin * d_x)
                auto mins = [&](const uint32_t (&f)[4]) {
                    const f32x32 ms = __builtin_amdgcn_mfma_f32_32x32x1f32(dm, dxb, zero32, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < NJ; j++) {
                        const f32x16 B = mfma_f16(f, bsb[j], zero16);
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            const float tm = ms[16 * j + v] * B[v];
                            acc[j][v] = acc[j][v] - tm;
                        }
                    }
                };
                auto step = [&](int buf, auto gc) {
                    constexpr int g = decltype(gc)::value;
                    uint32_t lo[2][4], hi[2][4];
                    step_frags<TY>(*(const u32x4 *)(wl + (TY == 4 ? 16 : 48) + 32 * g + 16 * hf), qh, g,
                                   byte_pair<(2 * g) & 3>(sc[g >> 1]), byte_pair<(2 * g + 1) & 3>(sc[g >> 1]), lo, hi);
                    auto dots = [&](const uint32_t (&f)[2][4], int c, int j) {
                        const f32x16 S = mfma_f16(f[0], frag(buf, g & 1, c + hf, j), zero16);
                        return mfma_f16(f[1], frag(buf, g & 1, c + 2 + hf, j), S);
                    };
                    if constexpr (TY == 4) {
                        f32x16 S[NJ], H[NJ];
#pragma unroll
                        for (int j = 0; j < NJ; j++) S[j] = dots(lo, 0, j);
#pragma unroll
                        for (int j = 0; j < NJ; j++) H[j] = dots(hi, 4, j);
#pragma unroll
                        for (int j = 0; j < NJ; j++)
#pragma unroll
                            for (int v = 0; v < 16; v++) acc[j][v] = __builtin_fmaf(ds[16 * j + v], S[j][v], acc[j][v]);
#pragma unroll
                        for (int j = 0; j < NJ; j++)
#pragma unroll
                            for (int v = 0; v < 16; v++) acc[j][v] = __builtin_fmaf(ds[16 * j + v], H[j][v], acc[j][v]);
                    } else {
                        // mins 2 g, 2 g + 1 against sums 4 g .. 4 g + 3: the other slots are zero. One tile at a
                        // time: both at once do not fit the registers
                        uint32_t bf[4];
#pragma unroll
                        for (int i = 0; i < 4; i++) bf[i] = (hf == (g >> 1) && (i >> 1) == (g & 1)) ? mf[i] : 0u;
                        const f32x32 ms = __builtin_amdgcn_mfma_f32_32x32x1f32(dm, dxb, zero32, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            const f32x16 S = dots(lo, 0, j), H = dots(hi, 4, j), B = mfma_f16(bf, bsb[j], zero16);
#pragma unroll
                            for (int v = 0; v < 16; v++) {
                                acc[j][v] = __builtin_fmaf(ds[16 * j + v], S[v], acc[j][v]);
                                acc[j][v] = __builtin_fmaf(ds[16 * j + v], H[v], acc[j][v]);
                                const float tm = ms[16 * j + v] * B[v];
                                acc[j][v] = acc[j][v] - tm;
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                };
                if (wave_on) {
                    step(0, std::integral_constant<int, 0>{});
                    step(0, std::integral_constant<int, 1>{});
                }
                stage_sync();
                if (2 * b + 2 < ns) fetch(0, 2 * b + 2);
                if (wave_on) {
                    step(1, std::integral_constant<int, 2>{});
                    step(1, std::integral_constant<int, 3>{});
                    if constexpr (TY == 4) mins(mf);
                }
            } else if (wave_on) {
                const int buf = b & 1, sh = 2 * (b & 1);
                if constexpr (TY == 3) {
                    Raw3 r;
                    r.load(wl, hf);
                    Run sr;   // bytes 96..107 (scales), 108..109 (d)
                    sr.load(wl + 96);
                    uint32_t s[3];
#pragma unroll
                    for (int i = 0; i < 3; i++) s[i] = sr.get(i, sh);
                    const float dw = h2f((uint16_t)(sr.w[3] >> (8 * sh)));
                    // chain sign: the products below are negated, so is the scale
                    const f32x32 ds = __builtin_amdgcn_mfma_f32_32x32x1f32(-dw, dxb, zero32, 0, 0, 0);
                    i32x16 I[NJ];
#pragma unroll
                    for (int j = 0; j < NJ; j++) I[j] = i32x16{};
#pragma unroll
                    for (int n = 0; n < 2; n++)
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            // raw scale i = 8 n + 2 q + hf (q3k_raw_scales): low nibbles of bytes 0..7 then their
                            // high nibbles, top bits two by two in bytes 8..11
                            const int bi = 2 * q + hf;
                            const int lo = (int)((q < 2 ? s[0] : s[1]) >> (8 * (bi & 3) + (n ? 4 : 0))) & 15;
                            const int hi2 = (int)(s[2] >> (8 * (bi & 3) + 2 * (2 * n + (q >> 1)))) & 3;
                            uint32_t f[4];
                            q3_frag(r, sh, n, q, 32 - (lo | hi2 << 4), f);
#pragma unroll
                            for (int j = 0; j < NJ; j++) I[j] = mfma_i8(f, frag(buf, n, 2 * q + hf, j), I[j]);
                        }
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int v = 0; v < 16; v++) acc[j][v] = __builtin_fmaf((float)I[j][v], ds[16 * j + v], acc[j][v]);
                } else {
                    Run sr;   // bytes 192..207 (scales), 208..209 (d)
                    sr.load(wl + 192);
                    uint32_t s[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) s[i] = sr.get(i, sh);
                    const float dw = h2f((uint16_t)(sr.x >> (8 * sh)));
                    const f32x32 ds = __builtin_amdgcn_mfma_f32_32x32x1f32(dw, dxb, zero32, 0, 0, 0);
                    i32x16 Ih[NJ], Il[NJ];
#pragma unroll
                    for (int j = 0; j < NJ; j++) Ih[j] = Il[j] = i32x16{};
#pragma unroll
                    for (int n = 0; n < 2; n++) {
                        Raw6 r;
                        r.load(wl, hf, n);
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            const int i = 2 * q + hf;   // scale 8 n + i
                            const int sc = (int)(int8_t)((q < 2 ? s[2 * n] : s[2 * n + 1]) >> (8 * (i & 3)));
                            uint32_t fh[4], fl[4];
                            q6_frag(r, sh, q, sc, fh, fl);
#pragma unroll
                            for (int j = 0; j < NJ; j++) {
                                const i32x4 x = frag(buf, n, 2 * q + hf, j);
                                Ih[j] = mfma_i8(fh, x, Ih[j]);
                                Il[j] = mfma_i8(fl, x, Il[j]);
                            }
                        }
                    }
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            const int I = Ih[j][v] * 64 + Il[j][v];
                            const float tv = (float)I * ds[16 * j + v];
                            acc[j][v] = acc[j][v] + tv;
                        }
                }
            }
        }
        if (!wave_on) return;
        // tile j's outputs in this lane: rows 8 q + 4 hf + e (v = 4 q + e), token 32 j + fr
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int tt = 32 * j + fr;
            if (tt >= pn) continue;
            float *yp = a.y + (p0 + tt) * a.ldy + sg.off;
            const float *rp = a.res ? a.res + (p0 + tt) * a.ldr + sg.off : nullptr;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int64_t gr = r0 + 8 * q + 4 * hf;
                if (gr >= sg.nr) continue;   // the rows of every segment come in fours
                float4 o = make_float4(acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]);
                if (rp) {
                    const float4 r4 = *(const float4 *)(rp + gr);
                    o.x += r4.x; o.y += r4.y; o.z += r4.z; o.w += r4.w;
                }
                *(float4 *)(yp + gr) = o;
            }
        }
    };
    if (pn > 32) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
}

// ---- q8_K of activation rows in the GEMM's forms: one wave per block ------------------------------
// f16 codes: 128-byte units of 64 codes; chunk c = 4 p + 2 m + h (16 bytes) holds codes
// 32 p + 16 h + 8 m + {0, 2, 1, 3, 4, 6, 5, 7}, the order in which step_frags unpacks the weights
OXE_DEV void q8K_store(const float (&v)[4], int lane, int64_t blk, const KqAct &y) {
    int q[4];
    const float d = kq::q8K_codes(v, lane, q);
    const int s = kq::sum16(q);
    if (y.c8) *(uint32_t *)(y.c8 + blk * QK + 4 * lane) = kq::pack4(q);
    if (y.c16) {
        const int g = lane >> 4, p = (lane >> 3) & 1, h = (lane >> 2) & 1, m = (lane >> 1) & 1;
        // int8 codes and int16 sums, as the ggml block stores them
        const h2 a = {(_Float16)(float)(int8_t)q[0], (_Float16)(float)(int8_t)q[2]};
        const h2 b = {(_Float16)(float)(int8_t)q[1], (_Float16)(float)(int8_t)q[3]};
        *(uint2 *)(y.c16 + blk * QK + 64 * g + 8 * (4 * p + 2 * m + h) + 4 * (lane & 1)) = make_uint2(as_u(a), as_u(b));
        if ((lane & 3) == 0) y.bs[blk * 16 + (lane >> 2)] = __builtin_bit_cast(uint16_t, (_Float16)(float)(int16_t)s);
    }
    if (lane == 0) y.d[blk] = d;
}
__global__ __launch_bounds__(256) void quant_rows_kernel(const float *__restrict__ x, int64_t ldx, int64_t nblk, int nb, KqAct y) {
    const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (b >= nblk) return;
    const float4 f = *(const float4 *)(x + (b / nb) * ldx + (b % nb) * QK + 4 * lane);
    const float v[4] = {f.x, f.y, f.z, f.w};
    q8K_store(v, lane, b, y);
}

// ---- swiglu (ggml_vec_swiglu_f32: silu(gate) * up) of one row of 512 per wave ---------------------
// index of gate element i of a row: split [gate 512 | up 512], or 8 gate then 8 up values in turn
template <bool SPLIT>
OXE_DEV void swiglu4(const float *g, int i, float (&h)[4]) {
    const int at = SPLIT ? i : (i >> 3) * 16 + (i & 7);
    const float4 a = *(const float4 *)(g + at), u = *(const float4 *)(g + at + (SPLIT ? shp::FF : 8));
    h[0] = v_silu(a.x) * u.x;
    h[1] = v_silu(a.y) * u.y;
    h[2] = v_silu(a.z) * u.z;
    h[3] = v_silu(a.w) * u.w;
}
template <bool SPLIT>
__global__ __launch_bounds__(256) void swiglu_q8_K_kernel(const float *gu, int64_t rows, KqAct y) {
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= rows) return;
#pragma unroll
    for (int b = 0; b < shp::FF / QK; b++) {
        float h[4];
        swiglu4<SPLIT>(gu + r * (2 * shp::FF), QK * b + 4 * lane, h);
        q8K_store(h, lane, r * (shp::FF / QK) + b, y);
    }
}
template <bool SPLIT>
__global__ __launch_bounds__(256) void swiglu_q8_0_kernel(const float *gu, int64_t rows, int8_t *hq, uint16_t *hd) {
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= rows) return;
    float h0[4], h1[4];
    swiglu4<SPLIT>(gu + r * (2 * shp::FF), 8 * lane, h0);
    swiglu4<SPLIT>(gu + r * (2 * shp::FF), 8 * lane + 4, h1);
    const float v[8] = {h0[0], h0[1], h0[2], h0[3], h1[0], h1[1], h1[2], h1[3]};
    quant8(v, hq + r * shp::FF + 8 * lane, hd + r * (shp::FF / 32) + lane / 4);
}

__global__ __launch_bounds__(256) void embed_rows_kernel(const uint8_t *w, int type, int64_t row_bytes, const uint32_t *toks,
                                                         float *x) {
    const uint8_t *row = w + (int64_t)toks[blockIdx.x] * row_bytes;
    const int bb = kq_block_bytes(type);
    for (int i = threadIdx.x; i < shp::E; i += 256)
        x[(int64_t)blockIdx.x * shp::E + i] = kq::kq_elem(type, row + (i / QK) * bb, i % QK);
}

// waves (32-row slices) per workgroup: four share a token stage; one where four-wave workgroups would
// leave CUs without work
constexpr int64_t WIDE_MIN = 512;

template <int TY>
int launch_ty(KqGemmArgs &a, int64_t ny, hipStream_t st) {
    auto tiles = [&](int nw) {
        int n = 0;
        for (int i = 0; i < a.nseg; i++) {
            a.tile0[i] = n;
            n += (int)((a.seg[i].nr + 32 * nw - 1) / (32 * nw));
        }
        return n;
    };
    int nx = tiles(4);
    if ((int64_t)nx * ny >= WIDE_MIN) {
        hipLaunchKernelGGL((kq_gemm_kernel<TY, 4>), dim3((unsigned)nx, (unsigned)ny), dim3(256), 0, st, a);
    } else {
        nx = tiles(1);
        hipLaunchKernelGGL((kq_gemm_kernel<TY, 1>), dim3((unsigned)nx, (unsigned)ny), dim3(64), 0, st, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace kqg

int kq_gemm_launch(int type, KqGemmArgs a, int64_t ntiles, hipStream_t st) {
    if (a.nseg < 1 || a.nseg > KQG_SEGS || a.nb < 1 || !a.y || !a.x.d || a.ldy % 4 != 0 || (a.res && a.ldr % 4 != 0)) return -1;
    if (((uintptr_t)a.y | (uintptr_t)a.res) % 16 != 0) return -1;
    for (int i = 0; i < a.nseg; i++)
        if ((uint64_t)a.seg[i].nr * (uint64_t)a.nb * 210 > UINT32_MAX) return -1;   // 32-bit weight offsets
    for (int i = 0; i < a.nseg; i++)
        if (!a.seg[i].w || a.seg[i].nr < 4 || a.seg[i].nr % 4 != 0 || a.seg[i].off % 4 != 0 || (uintptr_t)a.seg[i].w % 16 != 0) return -1;
    const bool f16 = kqg_f16(type);
    if (f16 ? (!a.x.c16 || !a.x.bs) : !a.x.c8) return -1;
    if (!f16 && a.nb % 2 != 0) return -1;   // 110- and 210-byte blocks: every row starts on a dword
    if ((uint64_t)a.nt * (uint64_t)a.nb * (f16 ? 512 : 256) > UINT32_MAX) return -1;   // 32-bit code offsets
    const int64_t ny = a.tiles ? ntiles : (a.nt + kqg::BN - 1) / kqg::BN;
    if (ny <= 0) return 0;
    switch (type) {
        case 11: return kqg::launch_ty<3>(a, ny, st);
        case 12: return kqg::launch_ty<4>(a, ny, st);
        case 13: return kqg::launch_ty<5>(a, ny, st);
        case 14: return kqg::launch_ty<6>(a, ny, st);
        default: return -1;
    }
}

int kq_pf_quant(const float *x, int64_t ldx, int64_t rows, int64_t k, KqAct y, hipStream_t st) {
    const int64_t nblk = rows * (k / kq::QK);
    hipLaunchKernelGGL(kqg::quant_rows_kernel, dim3((unsigned)((nblk + 3) / 4)), dim3(256), 0, st, x, ldx, nblk,
                       (int)(k / kq::QK), y);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int kq_pf_swiglu_q8_0(const float *gu, bool split, int64_t rows, int8_t *hq, uint16_t *hd, hipStream_t st) {
    const dim3 g((unsigned)((rows + 3) / 4));
    if (split) hipLaunchKernelGGL(kqg::swiglu_q8_0_kernel<true>, g, dim3(256), 0, st, gu, rows, hq, hd);
    else hipLaunchKernelGGL(kqg::swiglu_q8_0_kernel<false>, g, dim3(256), 0, st, gu, rows, hq, hd);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}
int kq_pf_swiglu_q8_K(const float *gu, bool split, int64_t rows, KqAct h, hipStream_t st) {
    const dim3 g((unsigned)((rows + 3) / 4));
    if (split) hipLaunchKernelGGL(kqg::swiglu_q8_K_kernel<true>, g, dim3(256), 0, st, gu, rows, h);
    else hipLaunchKernelGGL(kqg::swiglu_q8_K_kernel<false>, g, dim3(256), 0, st, gu, rows, h);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int kq_pf_embed(const RawW &e, const uint32_t *toks, int64_t n, float *x, hipStream_t st) {
    hipLaunchKernelGGL(kqg::embed_rows_kernel, dim3((unsigned)n), dim3(256), 0, st, e.w, e.type, raw_row_bytes(e), toks, x);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int kq_head_one(const RawW &w, const float *xn, uint8_t *xk, float *logits, hipStream_t st) {
    int rc = oxe_hip_quantize_row_q8_K(xn, shp::E, 1, xk, st);
    if (rc) return rc;
    rc = oxe_hip_vl_gemv(w.type - 8, shp::E, w.rows, 1, w.w, xk, logits, st);
    return rc == 1 ? 0 : rc == 0 ? -1 : rc;
}

}  // namespace oxe
