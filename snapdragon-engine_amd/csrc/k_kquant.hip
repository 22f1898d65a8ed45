// K-quant kernels: the q8_K activation quantizer (quantize_row_q8_K) and the lane GEMVs over
// Q3_K / Q4_K / Q5_K / Q6_K weights (the reference's oxe_vl_gemv, crates/kernels-sys/csrc/
// oxe_vl.inc:78-107, types 3..6), bit for bit per (lane, row).
//
// Weights are the GGUF file's ggml blocks (no repack: the reference's 8-row interleave only serves
// its NEON SMMLA tiles). Integer parts are exact (codes repacked 4 per dword into v_dot4_i32_i8),
// so only the float chain per (lane, row), in the order and fusion the reference documents per
// type, fixes the bits; the kernel layout is free otherwise (see vl_gemv_kernel).
#include <algorithm>

#include "oxe_common.h"
#include "oxe_kq_block.h"
#include "oxe_model_kernels.h"
#include "oxe_prologue.h"

#include <mutex>

namespace oxe {
namespace kq {

constexpr int MAX_LANES = 4;

// B: block bytes; R: integers per (unit, lane) that the chain reads (kept in LDS between the units
// and the chains, so a smaller R leaves room for more waves per CU)
template <int TY> struct BT;
template <> struct BT<3> { static constexpr int B = 110, R = 1; };
template <> struct BT<4> { static constexpr int B = 144, R = 5; };
template <> struct BT<5> { static constexpr int B = 176, R = 6; };
template <> struct BT<6> { static constexpr int B = 210, R = 1; };

OXE_DEV uint32_t ld32(const uint8_t *p) { return *(const uint32_t *)p; }
OXE_DEV uint16_t ld16(const uint8_t *p) { return *(const uint16_t *)p; }
// N dwords from a 2-byte aligned LDS address (Q3_K / Q6_K blocks are 110 / 210 bytes, so every other
// block of a row starts 2 bytes off a dword boundary): N + 1 aligned dword reads, then each dword
// cut out of a neighbouring pair (v_alignbyte_b32)
template <int N>
OXE_DEV void ld_run(const uint8_t *p, uint32_t (&out)[N]) {
    const uint32_t sh = (uint32_t)(uintptr_t)p & 3u;
    const uint32_t *a = (const uint32_t *)(p - sh);
    uint32_t w[N + 1];
#pragma unroll
    for (int i = 0; i <= N; i++) w[i] = a[i];
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], sh);
}
// Activations in LDS: each q8_K block repacked as two halves (codes 128 h .. 128 h + 127 and their 8
// sums of 16), YH = 37 dwords apart (odd: the 16 threads of a row read one half each, at the same
// offset, on distinct banks), lanes YL(nb) dwords apart; the block scales in a separate array.
constexpr int YH = 37;
__host__ __device__ inline int y_lane_words(int nb) { return nb * 2 * YH; }
struct YView {
    const uint32_t *h;   // half (b, h) of lane 0
    int ls;              // lane stride in dwords
    OXE_DEV uint32_t q(int l, int j) const { return h[l * ls + j]; }   // code dword j (0..31)
    OXE_DEV int bsum(int l, int i) const { return (int)((const int16_t *)(h + l * ls + 32))[i]; }   // sum i (0..7)
};

__global__ __launch_bounds__(256) void quant_q8_K_kernel(const float *__restrict__ x, int64_t nblk,
                                                         uint8_t *__restrict__ y) {
    const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b >= nblk) return;
    q8K_block(x + b * QK, threadIdx.x & 63, y + b * Q8K_BYTES);
}

// the q8_K blocks of a workgroup's [NL][E] rows held in LDS (256 threads: wave w takes blocks w,
// w + 4, ...), after the barrier that completes the rows
template <int NL>
OXE_DEV void q8K_rows_lds(const float (&rows)[NL][shp::E], uint8_t *__restrict__ y) {
    __syncthreads();
    for (int b = threadIdx.x >> 6; b < NL * shp::E / QK; b += 4)
        q8K_block(&rows[0][0] + b * QK, threadIdx.x & 63, y + (int64_t)b * Q8K_BYTES);
}

// ---- integers of one half block (unit h: weights 128 h .. 128 h + 127), every lane ---------------
// y: the lanes' halves h of this block position (YView); out[l * BT<TY>::R + ...]

// Q4_K / Q5_K: for the unit's two 64-weight steps g: sc_lo * I_lo, sc_hi * I_hi (out[0..3]); Q4_K:
// out[4] = the unit's part of sum min_j * bsum32_j; Q5_K: out[4 + g'] = that sum per step
template <int TY, int NL>
OXE_DEV void unit_k45(const uint8_t *wb, YView y, int h, int *out) {
    constexpr int RES = BT<TY>::R;
    const uint8_t *sc = wb + 4;
    const uint8_t *qs = wb + (TY == 4 ? 16 : 48);
    const uint8_t *qh = wb + 16;
    int bias4[NL];
#pragma unroll
    for (int l = 0; l < NL; l++) bias4[l] = 0;
#pragma unroll
    for (int gg = 0; gg < 2; gg++) {
        const int g = 2 * h + gg;
        int lo[NL], hi[NL];
#pragma unroll
        for (int l = 0; l < NL; l++) lo[l] = hi[l] = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t w = ld32(qs + 32 * g + 4 * i);
            uint32_t cl = w & 0x0F0F0F0Fu, ch = (w >> 4) & 0x0F0F0F0Fu;
            if (TY == 5) {
                const uint32_t hb = ld32(qh + 4 * i);
                cl |= ((hb >> (2 * g)) & 0x01010101u) << 4;
                ch |= ((hb >> (2 * g + 1)) & 0x01010101u) << 4;
            }
#pragma unroll
            for (int l = 0; l < NL; l++) {
                lo[l] = dot4(cl, y.q(l, 16 * gg + i), lo[l]);
                hi[l] = dot4(ch, y.q(l, 16 * gg + 8 + i), hi[l]);
            }
        }
        int s_lo, m_lo, s_hi, m_hi;
        scale_min_k4(2 * g, sc, s_lo, m_lo);
        scale_min_k4(2 * g + 1, sc, s_hi, m_hi);
#pragma unroll
        for (int l = 0; l < NL; l++) {
            out[l * RES + 2 * gg] = s_lo * lo[l];
            out[l * RES + 2 * gg + 1] = s_hi * hi[l];
            const int bias = m_lo * (y.bsum(l, 4 * gg) + y.bsum(l, 4 * gg + 1)) + m_hi * (y.bsum(l, 4 * gg + 2) + y.bsum(l, 4 * gg + 3));
            if (TY == 5) out[l * RES + 4 + gg] = bias;
            bias4[l] += bias;
        }
    }
    if (TY == 4)
#pragma unroll
        for (int l = 0; l < NL; l++) out[l * RES + 4] = bias4[l];
}

// Q6_K: the unit's part of I = sum_i scale_i * (16 codes - 32) . q8 (the -32 through the q8 sums)
template <int NL>
OXE_DEV void unit_q6(const uint8_t *wb, YView y, int n, int *out) {
    constexpr int RES = BT<6>::R;
    const int8_t *sc = (const int8_t *)(wb + 192);
    uint32_t qlw[16], qhw[8];   // ql[64 n .. 64 n + 63], qh[32 n .. 32 n + 31]
    ld_run<16>(wb + 64 * n, qlw);
    ld_run<8>(wb + 128 + 32 * n, qhw);
    int d[NL][8];
#pragma unroll
    for (int l = 0; l < NL; l++)
#pragma unroll
        for (int i = 0; i < 8; i++) d[l][i] = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t a = qlw[i], a2 = qlw[8 + i], hb = qhw[i];
        const uint32_t c0 = (a & 0x0F0F0F0Fu) | ((hb & 0x03030303u) << 4);
        const uint32_t c1 = (a2 & 0x0F0F0F0Fu) | (((hb >> 2) & 0x03030303u) << 4);
        const uint32_t c2 = ((a >> 4) & 0x0F0F0F0Fu) | (((hb >> 4) & 0x03030303u) << 4);
        const uint32_t c3 = ((a2 >> 4) & 0x0F0F0F0Fu) | (((hb >> 6) & 0x03030303u) << 4);
        const int s = i >> 2;   // which 16 of the 32
#pragma unroll
        for (int l = 0; l < NL; l++) {
            d[l][0 + s] = dot4(c0, y.q(l, i), d[l][0 + s]);
            d[l][2 + s] = dot4(c1, y.q(l, 8 + i), d[l][2 + s]);
            d[l][4 + s] = dot4(c2, y.q(l, 16 + i), d[l][4 + s]);
            d[l][6 + s] = dot4(c3, y.q(l, 24 + i), d[l][6 + s]);
        }
    }
#pragma unroll
    for (int l = 0; l < NL; l++) {
        int I = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) I += (int)sc[8 * n + i] * (d[l][i] - 32 * y.bsum(l, i));
        out[l * RES] = I;
    }
}

// Q3_K: the unit's part of isum = sum_i (raw_i - 32) * dot16_i, codes (low 2 bits | hmask bit << 2) - 4
template <int NL>
OXE_DEV void unit_q3(const uint8_t *wb, YView y, int n, int *out) {
    constexpr int RES = BT<3>::R;
    uint32_t qsw[8], hmw[8];   // qs[32 n .. 32 n + 31], hmask[0..31]
    ld_run<8>(wb + 32 + 32 * n, qsw);
    ld_run<8>(wb, hmw);
    int d[NL][8];
#pragma unroll
    for (int l = 0; l < NL; l++)
#pragma unroll
        for (int i = 0; i < 8; i++) d[l][i] = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t qw = qsw[i], hw = hmw[i];
        const int half = i >> 2;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const uint32_t c = ((qw >> (2 * s)) & 0x03030303u) | (((hw >> (4 * n + s)) & 0x01010101u) << 2);
#pragma unroll
            for (int l = 0; l < NL; l++) d[l][2 * s + half] = dot4(c, y.q(l, 8 * s + i), d[l][2 * s + half]);
        }
    }
    int sc[8];
#pragma unroll
    for (int i = 0; i < 8; i++) sc[i] = q3_raw(wb + 96, 8 * n + i) - 32;
#pragma unroll
    for (int l = 0; l < NL; l++) {
        int I = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) I += sc[i] * (d[l][i] - 4 * y.bsum(l, i));
        out[l * RES] = I;
    }
}

template <int TY, int NL>
OXE_DEV void unit(const uint8_t *wb, YView y, int h, int *out) {
    if (TY == 4 || TY == 5) unit_k45<TY, NL>(wb, y, h, out);
    else if (TY == 6) unit_q6<NL>(wb, y, h, out);
    else unit_q3<NL>(wb, y, h, out);
}

// ---- the reference's float chain over one block (units r0: weights 0..127, r1: 128..255) ---------
template <int TY>
OXE_DEV float chain(float acc, const uint8_t *wb, float dx, const int *r0, const int *r1) {
    if (TY == 4 || TY == 5) {
        // oxe_vl_q4k.inc:1-7 / oxe_vl_q5k.inc:6-12
        const float sbs = h2f(ld16(wb)) * dx, sbm = h2f(ld16(wb + 2)) * dx;
        const int *r[2] = {r0, r1};
        for (int u = 0; u < 2; u++)
            for (int gg = 0; gg < 2; gg++) {
                acc = fmaf(sbs, (float)r[u][2 * gg], acc);
                acc = fmaf(sbs, (float)r[u][2 * gg + 1], acc);
                if (TY == 5) {
                    const float t = sbm * (float)r[u][4 + gg];
                    acc = acc - t;
                }
            }
        if (TY == 4) {
            const float t = (float)(r0[4] + r1[4]) * sbm;
            acc = acc - t;
        }
        return acc;
    }
    if (TY == 6) {   // oxe_vl_q6k.inc:1-8, 107-113: unfused
        const float sbs = h2f(ld16(wb + 208)) * dx;
        const float t = (float)(r0[0] + r1[0]) * sbs;
        return acc + t;
    }
    // Q3_K, oxe_vl_q3k.inc:1-10: fused
    const float sbd = dx * h2f(ld16(wb + 108));
    return fmaf((float)(r0[0] + r1[0]), sbd, acc);
}

// ---- the lane GEMV --------------------------------------------------------------------------------
// s[l * nr + r] = W[r] . y[l]; w: nr rows of nb blocks (row bytes a multiple of 4, w 16-byte
// aligned); y: NL lanes of nb q8_K blocks. Waves persistent over groups of 4 rows, NW of them to a workgroup
// (16 threads per row). Per group: the 4 rows' bytes (contiguous) go to LDS with 16-byte loads, the
// first PF x 1 KiB of them held in registers, two groups ahead (buffers a and b, alternating); then
// per chunk of up to 8 blocks thread (row ri, unit u) forms half block u % 2 of block u / 2 for
// every lane, and threads u < NL of each row run lane u's chain over the chunk's blocks in order.
// The register loads are unconditional (indices clamped into the group; a group past the end
// re-reads the last one and writes nothing): a load under a per-thread condition makes the
// compiler wait for every outstanding load before the first LDS store, which drains the second
// buffer (measured: 2-deep conditional 143.8 us, unconditional 130.6 us for the Q6_K LM head).
constexpr int GR = 4;     // rows per group
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));   // a plain vector (HIP's uint4 is a union
                                                              // type that keeps arrays of it in scratch)

__host__ __device__ inline int align16(int n) { return (n + 15) / 16 * 16; }

// the first PF x 1 KiB of group g's bytes (g < ngroups) into registers, non-temporal 16-byte loads
template <int PF>
OXE_DEV void pf_load(u32x4 (&pf)[PF], const uint8_t *w, int64_t g, int64_t nr, int row_bytes, int t) {
    const u32x4 *src = (const u32x4 *)(w + g * GR * row_bytes);
    const int n16 = (int)(min((int64_t)GR, nr - g * GR) * row_bytes) / 16;
#pragma unroll
    for (int j = 0; j < PF; j++) pf[j] = __builtin_nontemporal_load(src + min(t + 64 * j, n16 - 1));
}

// the consumer of an engine phase's GEMV, applied at its store (ctl null: lane u's value to s[u][r]):
// row r of lane u < ctl->nl, in an active run only, goes to dst[u][r] (lane stride ld), plus
// resid[u][r] when resid is given (one fp32 add, as a separate pass would make it), and as fp16 to
// the V^T cache row r at position pos0 + u when vt is given
struct KqEpi {
    const RunCtl *ctl = nullptr;
    float *dst = nullptr;
    int64_t ld = 0;
    const float *resid = nullptr;
    uint16_t *vt = nullptr;
    int64_t vt_ld = 0;
};

// up to four matrices of one type and row length over the same activation in one launch (a
// projection's parts): groups are numbered through the segments in order; segment i's rows go to
// dst at row offset off[i] (its lane values to s when there is no epilogue: one segment then), and
// segment vseg's also to V^T
constexpr int KQ_SEGS = 4;
struct KqSegs {
    int n = 0;
    int vseg = -1;
    int64_t ngroups = 0;
    const uint8_t *w[KQ_SEGS] = {};
    int64_t nr[KQ_SEGS] = {};
    int64_t g0[KQ_SEGS] = {};
    int64_t off[KQ_SEGS] = {};
};

struct SegRef {
    const uint8_t *w;
    int64_t nr, gl, off;   // rows, the group's index within the segment, row offset in dst
    bool v;
};

// the segment of group g (fixed indices only, so the table stays in the kernel arguments)
OXE_DEV SegRef seg_ref(const KqSegs &S, int64_t g) {
    SegRef r{S.w[0], S.nr[0], g, S.off[0], S.vseg == 0};
#pragma unroll
    for (int j = 1; j < KQ_SEGS; j++)
        if (j < S.n && g >= S.g0[j]) r = SegRef{S.w[j], S.nr[j], g - S.g0[j], S.off[j], S.vseg == j};
    return r;
}

// LDS accesses of this wave before it come before those after it (wave-private regions: no barrier)
OXE_DEV void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
template <int NW>
OXE_DEV void group_sync() {
    if (NW == 1) __syncthreads();   // one wave: a wait for its LDS accesses (the fence alone measured 5-10 % slower)
    else wave_fence();
}
// LDS of one wave: a group's rows and its units' integers
__host__ __device__ inline int vl_wave_lds(int bb, int rr, int nb, int nl) {
    return align16(GR * nb * bb) + align16(64 * ((nl * rr) | 1) * 4);
}

// one group of 4 rows (g may be past the end: then nothing is written): its prefetched bytes (pf)
// and the rest to LDS, pf refilled with group g_next, then the units and the chains
template <int TY, int NL, int PF, int NW>
OXE_DEV void vl_group(u32x4 (&pf)[PF], int64_t g, int64_t g_next, const KqSegs &S, int nb, float *__restrict__ s,
                      const KqEpi &epi, uint8_t *wl, const uint32_t *yh, const float *yd, int *res) {
    constexpr int BB = BT<TY>::B;
    constexpr int RES = BT<TY>::R;
    constexpr int RS = (NL * RES) | 1;   // odd per-thread stride: no bank conflicts between threads
    const int row_bytes = nb * BB, ls = y_lane_words(nb);
    const int t = NW == 1 ? threadIdx.x : threadIdx.x & 63, ri = t >> 4, u = t & 15;
    const int64_t ngroups = S.ngroups;
    const bool gin = g < ngroups;
    const SegRef sg = seg_ref(S, gin ? g : ngroups - 1);   // the group whose bytes pf holds
    const int64_t nr = sg.nr;
    const int sp = (int)(min((int64_t)GR, nr - sg.gl * GR) * row_bytes), n16 = sp / 16;
    const u32x4 *src = (const u32x4 *)(sg.w + sg.gl * GR * row_bytes);
    group_sync<NW>();   // the previous group's LDS reads come first
#pragma unroll
    for (int j = 0; j < PF; j++) ((u32x4 *)wl)[min(t + 64 * j, n16 - 1)] = pf[j];   // clamped: same bytes
    for (int i = t + 64 * PF; i < n16; i += 64) ((u32x4 *)wl)[i] = src[i];
    for (int i = n16 * 4 + t; i < sp / 4; i += 64) ((uint32_t *)wl)[i] = ((const uint32_t *)src)[i];   // tail
    group_sync<NW>();
    {
        const SegRef sn = seg_ref(S, g_next < ngroups ? g_next : ngroups - 1);
        pf_load(pf, sn.w, sn.gl, sn.nr, row_bytes, t);   // in flight meanwhile
    }
    const int64_t r = sg.gl * GR + ri;
    const bool live = gin && r < nr;
    float acc = 0.0f;
    for (int b0 = 0; b0 < nb; b0 += 8) {
        const int kc = min(8, nb - b0);
        const int bi = b0 + (u >> 1);
        if ((u >> 1) < kc && live)
            unit<TY, NL>(wl + ri * row_bytes + bi * BB, YView{yh + (2 * bi + (u & 1)) * YH, ls}, u & 1, res + t * RS);
        group_sync<NW>();
        if (u < NL && live)
            for (int b = 0; b < kc; b++) {
                const int *r0 = res + (ri * 16 + 2 * b) * RS + u * RES;
                const int *r1 = res + (ri * 16 + 2 * b + 1) * RS + u * RES;
                acc = chain<TY>(acc, wl + ri * row_bytes + (b0 + b) * BB, yd[u * nb + b0 + b], r0, r1);
            }
        group_sync<NW>();
    }
    if (u < NL && live) {
        if (!epi.ctl) {
            s[(int64_t)u * nr + r] = acc;
        } else if (epi.ctl->active && u < epi.ctl->nl) {
            const int64_t i = (int64_t)u * epi.ld + sg.off + r;
            const float v = epi.resid ? acc + epi.resid[i] : acc;
            epi.dst[i] = v;
            if (sg.v && epi.vt) epi.vt[r * epi.vt_ld + epi.ctl->pos0 + u] = f2h(v);
        }
    }
}

template <int TY, int NL, int PF, int NW>
__global__ __launch_bounds__(64 * NW) void vl_gemv_kernel(KqSegs S, int nb, const uint8_t *__restrict__ y,
                                                          float *__restrict__ s, KqEpi epi) {
    constexpr int BB = BT<TY>::B;
    extern __shared__ __align__(16) uint8_t lds[];
    const int row_bytes = nb * BB;
    const int t = NW == 1 ? threadIdx.x : threadIdx.x & 63, w = NW == 1 ? 0 : threadIdx.x >> 6;
    // the lanes' activations, shared; then per wave a group's rows and the units' integers
    const int ys = align16(NL * nb * (2 * YH + 1) * 4);
    uint8_t *wl = lds + (NW == 1 ? 0 : ys + (size_t)w * vl_wave_lds(BB, BT<TY>::R, nb, NL));   // [GR][row_bytes]
    uint32_t *yh = (uint32_t *)(lds + (NW == 1 ? align16(GR * row_bytes) : 0));   // [NL][nb][2][YH]
    float *yd = (float *)(yh + NL * y_lane_words(nb));                   // [NL][nb]
    int *res = (int *)(wl + align16(GR * row_bytes) + (NW == 1 ? ys : 0));   // [64][(NL * R) | 1]
    const int64_t ngroups = S.ngroups, G = (int64_t)gridDim.x * NW, g0 = (int64_t)blockIdx.x * NW + w;
    // the lanes' q8_K blocks (lane l block b is block l nb + b) repacked into halves and scales
    for (int i = threadIdx.x; i < NL * nb * 2 * 36; i += 64 * NW) {
        const int wd = i % 36, hb = i / 36, h = hb & 1;
        const uint32_t *src = (const uint32_t *)(y + (int64_t)(hb >> 1) * Q8K_BYTES);
        yh[hb * YH + wd] = wd < 32 ? src[1 + 32 * h + wd] : src[65 + 4 * h + (wd - 32)];
    }
    for (int i = threadIdx.x; i < NL * nb; i += 64 * NW) yd[i] = *(const float *)(y + (int64_t)i * Q8K_BYTES);
    // two register buffers (fixed indices only: they stay in registers), groups g and g + G in
    // flight from the start; the scheduling barrier keeps buffer a's loads ahead of b's, so the
    // first LDS stores wait for a's only
    u32x4 pa[PF], pb[PF];
    {
        const SegRef sa = seg_ref(S, min(g0, ngroups - 1)), sb = seg_ref(S, min(g0 + G, ngroups - 1));
        pf_load(pa, sa.w, sa.gl, sa.nr, row_bytes, t);
        __builtin_amdgcn_sched_barrier(0);
        pf_load(pb, sb.w, sb.gl, sb.nr, row_bytes, t);
    }
    if (NW > 1) __syncthreads();
    for (int64_t g = g0; g < ngroups; g += 2 * G) {
        vl_group<TY, NL, PF, NW>(pa, g, g + 2 * G, S, nb, s, epi, wl, yh, yd, res);
        vl_group<TY, NL, PF, NW>(pb, g + G, g + 3 * G, S, nb, s, epi, wl, yh, yd, res);
    }
}

size_t vl_gemv_lds(int bb, int rr, int nb, int nl, int nw) {
    return (size_t)align16(nl * nb * (2 * YH + 1) * 4) + (size_t)nw * vl_wave_lds(bb, rr, nb, nl);
}

constexpr int KQ_MAX_DEV = 64;
template <int TY, int NL, int PF, int NW>
int vl_gemv_launch_nw(const KqSegs &S, int nb, const uint8_t *y, float *s, hipStream_t st, const KqEpi &epi) {
    constexpr int BB = BT<TY>::B;
    const size_t lds = vl_gemv_lds(BB, BT<TY>::R, nb, NL, NW);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= KQ_MAX_DEV) return -2;
    // per instantiation and device: the dynamic LDS the kernel is configured for (above 64 KiB it
    // needs the attribute; 160 KiB per CU), the CU count, and the occupancy per LDS size, each asked
    // of the runtime once (a query per launch would sit on the decode path)
    struct Cache {
        size_t configured = 65536;
        int ncu = 0;
        size_t lds[8] = {};
        int occ[8] = {};
    };
    static Cache cache[KQ_MAX_DEV];
    static std::mutex mu;
    int ncu = 256, occ = 0;
    {
        std::lock_guard<std::mutex> lk(mu);
        Cache &cc = cache[dev];
        if (lds > cc.configured) {
            if (hipFuncSetAttribute((const void *)vl_gemv_kernel<TY, NL, PF, NW>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)lds) != hipSuccess)
                return -2;
            cc.configured = lds;
        }
        if (cc.ncu == 0 && hipDeviceGetAttribute(&cc.ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            cc.ncu = 256;
        ncu = cc.ncu;
        int slot = -1;
        for (int i = 0; i < 8 && slot < 0; i++)
            if (cc.lds[i] == lds || cc.lds[i] == 0) slot = i;
        if (slot >= 0 && cc.lds[slot] == lds) {
            occ = cc.occ[slot];
        } else {
            // exactly the waves a CU holds, by LDS and registers both: a grid beyond them leaves its
            // last waves to start after others finish, one below them leaves SIMDs short of a wave
            // (measured on the Q6_K LM head, 12 resident per CU: 11 per CU 131 us, 13 per CU 116 us,
            // 12 per CU 92.5 us)
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, vl_gemv_kernel<TY, NL, PF, NW>, 64 * NW, lds) != hipSuccess ||
                occ < 1)
                occ = (int)std::max<size_t>(1, (160 * 1024) / lds);
            if (slot >= 0) {
                cc.lds[slot] = lds;
                cc.occ[slot] = occ;
            }
        }
    }
    const int64_t grid = std::min<int64_t>((S.ngroups + NW - 1) / NW, (int64_t)ncu * std::max(1, std::min(16 / NW, occ)));
    hipLaunchKernelGGL((vl_gemv_kernel<TY, NL, PF, NW>), dim3((unsigned)grid), dim3(64 * NW), lds, st, S, nb, y, s, epi);
    return hipGetLastError() == hipSuccess ? 1 : -2;
}
// Four waves share the lanes' activations in LDS where staging them is what a workgroup spends its time on: at
// least two lanes of rows of 2048 (Q3_K, whose waves need the most registers: 24 blocks in all; Q6_K also one lane of 3072).
// Rows set no line: a few workgroups of four waves are still the shorter latency. Measured, one wave against four (us):
//   Q4_K, 2048 long, 2 lanes: 32 rows 7.1 / 6.6, 512 7.0 / 7.0, 2048 7.7 / 6.7, 8192 10.7 / 9.0, 32768 19.7 / 19.0
//   2048 x 4096, 2 / 4 lanes: Q3_K 12.2 / 9.9, 18.4 / 12.0; Q4_K 13.5 / 11.0, 18.8 / 12.5; Q5_K 15.1 / 12.7; Q6_K 15.0 / 12.2,
//   20.8 / 14.4, one lane 12.3 / 10.8
//   2048 x 2048, 4 lanes: Q3_K 10.5 / 7.6, Q4_K 10.5 / 7.6, Q5_K 10.9 / 8.2, Q6_K 10.4 / 7.8; 3 lanes Q3_K 9.1 / 7.3
//   100000 rows: Q4_K 4096 long, 4 lanes 160 / 106; Q6_K 3072 long, 2 lanes 113 / 68
// and the other side: one lane 700 x 2048 Q4_K 6.2 / 7.3, 100000 x 1024 24.3 / 27.1; Q5_K 512 x 2048, 2 lanes 7.5 / 7.8
template <int TY, int NL, int PF>
int vl_gemv_launch_pf(const KqSegs &S, int nb, const uint8_t *y, float *s, hipStream_t st, const KqEpi &epi) {
    if constexpr (PF >= 4 && (NL >= 2 || TY == 6)) {
        const bool wide = NL >= 2 ? nb >= 8 && (TY != 3 || NL * nb >= 24) : nb >= 12;
        if (wide && vl_gemv_lds(BT<TY>::B, BT<TY>::R, nb, NL, 4) <= 80 * 1024)
            return vl_gemv_launch_nw<TY, NL, PF, 4>(S, nb, y, s, st, epi);
    }
    return vl_gemv_launch_nw<TY, NL, PF, 1>(S, nb, y, s, st, epi);
}

// registers per prefetch buffer: the smallest of 2, 4, a row-of-2048 group's, 8 KiB per wave that holds a whole group
// (the rest of a larger group is copied to LDS directly)
template <int TY, int NL>
int vl_gemv_launch(const KqSegs &S, int nb, const uint8_t *y, float *s, hipStream_t st, const KqEpi &epi) {
    const int n16 = GR * nb * BT<TY>::B / 16;
    if (n16 <= 128) return vl_gemv_launch_pf<TY, NL, 2>(S, nb, y, s, st, epi);
    if (n16 <= 256) return vl_gemv_launch_pf<TY, NL, 4>(S, nb, y, s, st, epi);
    constexpr int P = (GR * 8 * BT<TY>::B / 16 + 63) / 64;   // a group of rows of 2048
    if constexpr (P > 4)
        if (n16 <= 64 * P) return vl_gemv_launch_pf<TY, NL, P>(S, nb, y, s, st, epi);
    return vl_gemv_launch_pf<TY, NL, 8>(S, nb, y, s, st, epi);
}

// one matrix [nr rows of nb blocks] as a one-segment table
inline KqSegs one_seg(const uint8_t *w, int64_t nr) {
    KqSegs S;
    S.n = 1;
    S.w[0] = w;
    S.nr[0] = nr;
    S.ngroups = (nr + GR - 1) / GR;
    return S;
}

template <int TY>
int vl_gemv_segs(const KqSegs &S, int nb, const uint8_t *y, int nl, float *s, hipStream_t st, const KqEpi &epi) {
    switch (nl) {
        case 1: return vl_gemv_launch<TY, 1>(S, nb, y, s, st, epi);
        case 2: return vl_gemv_launch<TY, 2>(S, nb, y, s, st, epi);
        case 3: return vl_gemv_launch<TY, 3>(S, nb, y, s, st, epi);
        default: return vl_gemv_launch<TY, 4>(S, nb, y, s, st, epi);
    }
}

template <int TY>
int vl_gemv_type(const uint8_t *w, int nb, int64_t nr, const uint8_t *y, int nl, float *s, hipStream_t st) {
    return vl_gemv_segs<TY>(one_seg(w, nr), nb, y, nl, s, st, KqEpi{});
}


// ==== K-quant and F32 matrices in the engine's per-phase runs ======================================
// (the reference's mv / mv_lanes over any qtype, crates/model/src/engine.rs:2270-2343; MoE phases
// engine.rs:3437-3625; LM head 3630-3715). Every (lane, row) value is the lane GEMV's: the same
// block units and float chain as vl_gemv_kernel, on the activation quantised as the weight's type
// asks (q8_K for K-quants, Q8_0 for Q8_0, the f32 vector itself for F32 rows).

// ggml type id (11..14) -> the units / chain of that type
template <int NL>
OXE_DEV void unit_rt(int type, const uint8_t *wb, YView y, int h, int *out) {
    switch (type) {
        case 11: unit<3, NL>(wb, y, h, out); break;
        case 12: unit<4, NL>(wb, y, h, out); break;
        case 13: unit<5, NL>(wb, y, h, out); break;
        default: unit<6, NL>(wb, y, h, out); break;
    }
}
OXE_DEV float chain_rt(int type, float acc, const uint8_t *wb, float dx, const int *r0, const int *r1) {
    switch (type) {
        case 11: return chain<3>(acc, wb, dx, r0, r1);
        case 12: return chain<4>(acc, wb, dx, r0, r1);
        case 13: return chain<5>(acc, wb, dx, r0, r1);
        default: return chain<6>(acc, wb, dx, r0, r1);
    }
}
OXE_DEV int res_of(int type) { return type == 12 ? BT<4>::R : type == 13 ? BT<5>::R : 1; }
constexpr int RES_MAX = 6;

// q8_K of NBLK blocks of floats by a workgroup of W waves into LDS, as halves (YH words apart) and scales, every load in
// flight at once. Each workgroup of gate / up and of down quantises what it reads, 1.5 us more of a launch each (the
// launches that did it before them took 4.3 and 4.5)
template <int W, int NBLK>
OXE_DEV void quant_q8k_lds(const float *x, uint32_t *yh, float *yd) {
    constexpr int I = (NBLK + W - 1) / W;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float4 f[I];
#pragma unroll
    for (int k = 0; k < I; k++) f[k] = *(const float4 *)(x + min(w + W * k, NBLK - 1) * QK + 4 * lane);
#pragma unroll
    for (int k = 0; k < I; k++) {
        const int b = w + W * k;
        if (b >= NBLK) break;   // wave-uniform
        const float v[4] = {f[k].x, f[k].y, f[k].z, f[k].w};
        int q[4];
        const float d = q8K_codes(v, lane, q);
        const int s = sum16(q);
        uint32_t *y = yh + (2 * b + (lane >> 5)) * YH;
        y[lane & 31] = pack4(q);
        if ((lane & 3) == 0) ((int16_t *)(y + 32))[(lane >> 2) & 7] = (int16_t)s;
        if (lane == 0) yd[b] = d;
    }
}

OXE_DEV uint32_t ordered_bits(float f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// ---- F32 ssm_beta / ssm_alpha rows: x -> rms_norm * attn_norm (every workgroup, exact), then
// oxe_vec_dot_f32 per (row, lane) in ggml_vec_dot_f32's order (vec.cpp:104-125): lane c of a
// 16-lane group runs chain c over elements c + 16 s; xor 8, 4, 1, 2 is the NEON reduction tree.
// Workgroup b: rows 16 b .. 16 b + 15 of [beta rows | alpha rows]; outputs into the projection
// buffer at DN_BETA / DN_ALPHA, where the delta-net phase reads them.
template <int NL>
__global__ __launch_bounds__(256) void ba_f32_kernel(const RunCtl *__restrict__ ctl, const float *x, const float *norm_w,
                                                     float eps, const float *beta, const float *alpha, float *proj) {
    __shared__ float s_xn[NL][shp::E];
    __shared__ NormScratch ns;
    if (!ctl->active) return;
    const int nl = ctl->nl, t = threadIdx.x;
#pragma unroll
    for (int l = 0; l < NL; l++) {
        float v[EPT];
        if (l < nl) {
            load8(x + (int64_t)l * shp::E, v);
            rms_norm_mul_e(v, x + (int64_t)l * shp::E, norm_w, eps, ns);
        } else {
#pragma unroll
            for (int i = 0; i < EPT; i++) v[i] = 0.0f;
        }
        store8(s_xn[l], v);
    }
    __syncthreads();
    const int c = t & 15, row = blockIdx.x * 16 + (t >> 4);
    const bool is_beta = row < shp::NVH;
    const float *w = (is_beta ? beta + (int64_t)row * shp::E : alpha + (int64_t)(row - shp::NVH) * shp::E);
    float acc[NL];
#pragma unroll
    for (int l = 0; l < NL; l++) acc[l] = 0.0f;
#pragma unroll 32
    for (int s = 0; s < shp::E / 16; s++) {
        const float wv = w[c + 16 * s];
#pragma unroll
        for (int l = 0; l < NL; l++) acc[l] = __builtin_fmaf(wv, s_xn[l][c + 16 * s], acc[l]);
    }
#pragma unroll
    for (int l = 0; l < NL; l++) {
        float v = acc[l];
        v = v + shfl_xor_f(v, 8);
        v = v + shfl_xor_f(v, 4);
        v = v + shfl_xor_f(v, 1);
        v = v + shfl_xor_f(v, 2);
        if (c == 0 && l < nl) proj[(int64_t)l * shp::DN_ROWS + (is_beta ? shp::DN_BETA + row : shp::DN_ALPHA + row - shp::NVH)] = v;
    }
}

// ---- MoE gate / up over K-quant matrices: workgroup (unit u, tile of 8 rows), u < OXE_MAX_UNION
// the union's expert u, u = OXE_MAX_UNION the shared expert. Thread (matrix t / 128: gate, up; row
// t / 16 % 8, half block t % 16) forms its half block's integers for every lane; threads t % 16 < NL
// then run lane t % 16's chain over the row's 8 blocks, gate and up at once; then silu(g) * u
// (ggml_v_silu, as swiglu) for every lane that routed to the expert (the shared expert: every lane).
// A tile's rows are one run of bytes per matrix: they come as whole lines, before the activations, and are read from
// LDS (each thread reading its half block from global memory after the activations, 64 threads 72 bytes apart: 18.4 us a
// launch with Q4_K experts of two lanes, 14.2 so, both after a launch that quantised xn). Bound by the latency of one round of workgroups.
struct KqGuArgs {
    const float *xn;            // [NL][E]
    RawW gate, up, sh_gate, sh_up;
    const int32_t *uni, *route_ids;
    float *hexp;                // [NL][KUSED][FF]
    float *hsh;                 // [NL][FFSH]
    int do_exp, do_sh;
    uint32_t *stats;            // [0] sum of union sizes, [1] launches (as the Q8_0 experts phase counts)
};
constexpr int GU_NB = shp::E / QK;   // 8 blocks per row
constexpr int GU_R = 8;              // rows per workgroup
constexpr int GU_LD = (GU_R * GU_NB * 210 / 16 + 127) / 128;   // 16-byte loads per thread: a tile of one matrix, Q6_K's blocks
static_assert(GU_NB * 2 == 16 && shp::FF == shp::FFSH, "16 half blocks per row; one tiling for both");

template <int NL>
__global__ __launch_bounds__(256) void kq_gu_kernel(const RunCtl *__restrict__ ctl, KqGuArgs a) {
    constexpr int RS = (NL * RES_MAX) | 1;
    extern __shared__ __align__(16) uint8_t gu_w[];   // the gate rows, then the up rows
    __shared__ uint32_t yh[NL * GU_NB * 2 * YH];
    __shared__ float yd[NL * GU_NB];
    __shared__ int res[256 * RS];
    __shared__ float s_gu[2][GU_R][NL];
    const int t = threadIdx.x, which = t >> 7, ri = (t >> 4) & (GU_R - 1), hu = t & 15;
    const int u = blockIdx.x / (shp::FF / GU_R), tile = blockIdx.x % (shp::FF / GU_R);
    const bool sh = u == OXE_MAX_UNION;
    // one round trip for all that says which rows to read
    const int active = ctl->active, nl = ctl->nl, nu = a.uni[0];
    int e = a.uni[1 + (sh ? 0 : u)];
    if (!active) return;
    if (a.do_exp && blockIdx.x == 0 && t == 0) {
        atomicAdd(a.stats, (uint32_t)nu);
        atomicAdd(a.stats + 1, 1u);
    }
    if (sh ? !a.do_sh : !a.do_exp) return;
    if (!sh && u >= nu) return;
    e = sh || e < 0 ? 0 : (e >= shp::NEXP ? shp::NEXP - 1 : e);
    const RawW &W = sh ? (which ? a.sh_up : a.sh_gate) : (which ? a.up : a.gate);
    const int type = W.type, rs = res_of(type), rb = (int)raw_row_bytes(W), n16 = GU_R * rb / 16;
    const u32x4 *src = (const u32x4 *)(W.w + ((int64_t)e * W.rows + tile * GU_R) * rb);
    u32x4 pf[GU_LD];
#pragma unroll
    for (int k = 0; k < GU_LD; k++) pf[k] = __builtin_nontemporal_load(src + min((t & 127) + 128 * k, n16 - 1));
    __builtin_amdgcn_sched_barrier(0);   // the weights before the activations
    quant_q8k_lds<4, NL * GU_NB>(a.xn, yh, yd);
    int slot = -1;
    if (which == 0 && hu < NL && hu < nl && !sh)
#pragma unroll
        for (int jj = 0; jj < shp::KUSED; jj++)
            if (a.route_ids[hu * shp::KUSED + jj] == e) slot = jj;
    uint8_t *wl = gu_w + (which ? GU_R * (int)raw_row_bytes(sh ? a.sh_gate : a.gate) : 0);
#pragma unroll
    for (int k = 0; k < GU_LD; k++) ((u32x4 *)wl)[min((t & 127) + 128 * k, n16 - 1)] = pf[k];   // clamped: same bytes
    __syncthreads();
    const int row = tile * GU_R + ri;
    {
        const uint8_t *wr = wl + ri * rb;
        unit_rt<NL>(type, wr + (hu >> 1) * kq_block_bytes(type), YView{yh + (2 * (hu >> 1) + (hu & 1)) * YH, GU_NB * 2 * YH},
                    hu & 1, res + t * RS);
        __syncthreads();
        if (hu < NL) {
            float acc = 0.0f;
            for (int b = 0; b < GU_NB; b++) {
                const int *r0 = res + ((t & ~15) + 2 * b) * RS + hu * rs, *r1 = res + ((t & ~15) + 2 * b + 1) * RS + hu * rs;
                acc = chain_rt(type, acc, wr + b * kq_block_bytes(type), yd[hu * GU_NB + b], r0, r1);
            }
            s_gu[which][ri][hu] = acc;
        }
        __syncthreads();
    }
    if (which == 0 && hu < NL && hu < nl) {
        const float h = v_silu(s_gu[0][ri][hu]) * s_gu[1][ri][hu];
        if (sh) a.hsh[(int64_t)hu * shp::FFSH + row] = h;
        else if (slot >= 0) a.hexp[((int64_t)hu * shp::KUSED + slot) * shp::FF + row] = h;
    }
}

// ---- MoE down + combine with any mix of K-quant and Q8_0 down matrices: workgroup = 8 output
// rows; units 0..nu-1 the union's experts, unit OXE_MAX_UNION the shared expert. Each (unit, lane,
// row) value is that matrix's row dot with the lane's h (slot j of the lane's top-k, or the shared
// h): K-quants on h's q8_K blocks (2 per row of 512), Q8_0 on h quantised to Q8_0 in LDS. Then the
// reference's combine (engine.rs:3591-3601): m = d0 w0; m += dj wj; f = m + dsh * g; x2 = f + x1.
// 32 threads per unit, every unit at once: a unit's 8 rows are one run of bytes, requested as whole lines before
// anything else and read from LDS, so the launch waits for memory once (256 workgroups, one per CU, whose 125 KB
// of LDS and registers nothing else wants). Eight units a pass from global memory, the Q8_0 unit's blocks by one
// thread per row: 17.2 us a launch with Q5_K experts and a Q8_0 shared matrix, two lanes; 8.8 so, both after
// a launch that quantised h.
struct KqDownArgs {
    const int32_t *uni, *route_ids;
    const float *route_w, *sh_gate;
    const float *hexp, *hsh;        // f32 h, quantised here
    Q8W exp_down, shexp_down;
    RawW exp_down_r, sh_down_r;
    const float *x1;
    float *x2;
    unsigned long long *amax_key;
};
constexpr int DN_R = 8;                      // output rows per workgroup (E / 8 = 256 workgroups)
constexpr int DN_NB = shp::FF / QK;          // 2 blocks per down row
constexpr int DN_U = OXE_MAX_UNION + 1;
constexpr int DN_A = shp::KUSED + 1;         // activation rows per lane: the k slots, then the shared h
constexpr int DN_T = 64 * ((DN_U + 1) / 2);  // 32 threads per unit
constexpr int DN_SLAB = DN_R * (shp::FF + shp::FF / 16);   // most bytes of a unit's rows: Q8_0 codes, then scales
constexpr int DN_LD = (DN_SLAB / 16 + 31) / 32;            // 16-byte loads per thread of a unit

template <int NL>
__global__ __launch_bounds__(DN_T) void kq_down_kernel(const RunCtl *__restrict__ ctl, KqDownArgs a) {
    constexpr int RS = (NL * RES_MAX) | 1;   // odd per-thread stride of the unit integers
    constexpr int QB = shp::FF / 32;         // Q8_0 blocks of a row
    static_assert(DN_R == 8 && OXE_MAX_UNION % 2 == 0, "32 threads per unit; the shared unit in a wave of its own");
    static_assert(DN_SLAB % 16 == 0 && DN_SLAB >= DN_R * DN_NB * 210 && 32 * RS >= NL * DN_R * QB, "a unit's LDS");
    __shared__ __align__(16) uint8_t s_wl[DN_U][DN_SLAB];
    __shared__ uint32_t yh[NL * DN_A * DN_NB * 2 * YH];
    __shared__ float yd[NL * DN_A * DN_NB];
    __shared__ __align__(16) int8_t s_q[NL * DN_A][shp::FF];
    __shared__ uint16_t s_d[NL * DN_A][QB];
    __shared__ int res[DN_T * RS];
    __shared__ float s_dn[NL][DN_A][DN_R];
    __shared__ int32_t s_slot[DN_U][NL];
    __shared__ float s_w[NL][shp::KUSED], s_sg[NL];
    const int t = threadIdx.x, u = t >> 5, ti = t & 31;
    const bool shu = __builtin_amdgcn_readfirstlane(t >> 6) == OXE_MAX_UNION / 2;
    const int active = ctl->active, nl = ctl->nl, nu = a.uni[0], e0 = shu ? 0 : a.uni[1 + u];
    if (!active) return;
    const int64_t row0 = (int64_t)blockIdx.x * DN_R;
    const bool live = u < DN_U && (shu || u < nu);
    const RawW &W = shu ? a.sh_down_r : a.exp_down_r;
    const int type = W.type, bb = type != 8 ? kq_block_bytes(type) : 0;
    const int64_t e = e0 < 0 ? 0 : (e0 < shp::NEXP ? e0 : shp::NEXP - 1);   // slots below compare the unclamped id
    // the unit's 8 rows (one run of bytes), on their way before anything else
    u32x4 pf[DN_LD];
    if (live) {
        if (type == 8) {
            const Q8W &Q = shu ? a.shexp_down : a.exp_down;
            const u32x4 *q = (const u32x4 *)(Q.q + (e * shp::E + row0) * shp::FF), *d = (const u32x4 *)(Q.d + (e * shp::E + row0) * QB);
#pragma unroll
            for (int k = 0; k < DN_LD - 1; k++) pf[k] = __builtin_nontemporal_load(q + ti + 32 * k);
            pf[DN_LD - 1] = __builtin_nontemporal_load(d + (ti & 15));
        } else {
            const u32x4 *src = (const u32x4 *)(W.w + (e * W.rows + row0) * raw_row_bytes(W));   // 16 blocks: bb chunks
#pragma unroll
            for (int k = 0; k < 7; k++) pf[k] = __builtin_nontemporal_load(src + min(ti + 32 * k, bb - 1));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (blockIdx.x == 0 && t < NL) a.amax_key[t] = 0ull;   // the LM head that follows starts clean
    const bool exp_kq = a.exp_down_r.type != 8, sh_kq = a.sh_down_r.type != 8;
    if (t < DN_U) {
        const int ue = t < OXE_MAX_UNION ? (t < nu ? a.uni[1 + t] : -1) : 0;
        for (int l = 0; l < NL; l++) {
            int j = -1;
            if (l < nl) {
                if (t == OXE_MAX_UNION) j = shp::KUSED;
                else if (ue >= 0)
                    for (int jj = 0; jj < shp::KUSED; jj++)
                        if (a.route_ids[l * shp::KUSED + jj] == ue) j = jj;
            }
            s_slot[t][l] = j;
        }
    }
    if (t < NL * shp::KUSED) s_w[t / shp::KUSED][t % shp::KUSED] = t / shp::KUSED < nl ? a.route_w[t] : 0.0f;
    if (t < NL) s_sg[t] = t < nl ? a.sh_gate[t] : 0.0f;
    // activations: q8_K rows of every lane's slots, then of every lane's shared h; Q8_0 row l * DN_A + j (j = KUSED: the
    // shared h)
    constexpr int YSH = NL * shp::KUSED;   // first shared row
    if (exp_kq) quant_q8k_lds<DN_T / 64, NL * shp::KUSED * DN_NB>(a.hexp, yh, yd);
    if (sh_kq) quant_q8k_lds<DN_T / 64, NL * DN_NB>(a.hsh, yh + YSH * DN_NB * 2 * YH, yd + YSH * DN_NB);
    if (!exp_kq || !sh_kq) {
        for (int i = t; i < NL * DN_A * QB; i += DN_T) {
            const int ar = i / QB, b = i % QB, l = ar / DN_A, j = ar % DN_A;
            const bool want = j < shp::KUSED ? !exp_kq : !sh_kq;
            if (want && l < nl) {
                const float *src = j < shp::KUSED ? a.hexp + ((int64_t)l * shp::KUSED + j) * shp::FF + 32 * b
                                                  : a.hsh + (int64_t)l * shp::FFSH + 32 * b;
                quant_block_q8_0(src, &s_q[ar][32 * b], &s_d[ar][b]);
            }
        }
    }
    uint8_t *wl = s_wl[u < DN_U ? u : 0];
    if (live) {
        if (type == 8) {
#pragma unroll
            for (int k = 0; k < DN_LD - 1; k++) ((u32x4 *)wl)[ti + 32 * k] = pf[k];
            ((u32x4 *)wl)[DN_R * shp::FF / 16 + (ti & 15)] = pf[DN_LD - 1];
        } else {
#pragma unroll
            for (int k = 0; k < 7; k++) ((u32x4 *)wl)[min(ti + 32 * k, bb - 1)] = pf[k];   // clamped: same bytes
        }
    }
    __syncthreads();
    // Integers of a unit: K-quant, thread (row ti / 4, half block ti % 4) for every lane with a slot there; Q8_0, block
    // ti % 16 of rows ti / 16, + 2, ... Then threads ti % 4 < NL run lane ti % 4's chain over row ti / 4's blocks.
    const int rr = ti >> 2, hu = ti & 3, rs = type != 8 ? res_of(type) : 0;
    int *ru = res + (t & ~31) * RS;   // the unit's
    if (live) {
        for (int l = 0; l < NL; l++) {
            const int j = s_slot[u][l];
            if (j < 0) continue;
            if (type != 8) {
                const int ar = shu ? YSH + l : l * shp::KUSED + j;
                unit_rt<1>(type, wl + (rr * DN_NB + (hu >> 1)) * bb, YView{yh + (ar * DN_NB * 2 + hu) * YH, 0}, hu & 1,
                           res + t * RS + l * rs);
            } else {
                const int b = ti & 15;
                for (int r = ti >> 4; r < DN_R; r += 2) {
                    const u32x4 *wp = (const u32x4 *)(wl + r * shp::FF + 32 * b), *xp = (const u32x4 *)&s_q[l * DN_A + j][32 * b];
                    int32_t s = 0;
#pragma unroll
                    for (int k = 0; k < 8; k++) s = dot4(wp[k >> 2][k & 3], xp[k >> 2][k & 3], s);
                    ru[(l * DN_R + r) * QB + b] = s;
                }
            }
        }
    }
    __syncthreads();
    if (live && hu < NL && s_slot[u][hu] >= 0) {
        const int j = s_slot[u][hu];
        float acc = 0.0f;
        if (type != 8) {
            const int ar = shu ? YSH + hu : hu * shp::KUSED + j;
            for (int b = 0; b < DN_NB; b++) {
                const int *r0 = res + ((t & ~3) + 2 * b) * RS + hu * rs, *r1 = res + ((t & ~3) + 2 * b + 1) * RS + hu * rs;
                acc = chain_rt(type, acc, wl + (rr * DN_NB + b) * bb, yd[ar * DN_NB + b], r0, r1);
            }
        } else {
            const uint16_t *wd = (const uint16_t *)(wl + DN_R * shp::FF) + rr * QB, *xd = s_d[hu * DN_A + j];
            const int *is = ru + (hu * DN_R + rr) * QB;
#pragma unroll
            for (int b = 0; b < QB; b++) acc = __builtin_fmaf((float)is[b], h2f(xd[b]) * h2f(wd[b]), acc);
        }
        s_dn[hu][j][rr] = acc;
    }
    __syncthreads();
    if (t < NL * DN_R) {
        const int l = t / DN_R, rr = t % DN_R;
        if (l < nl) {
            float m = s_dn[l][0][rr] * s_w[l][0];
            for (int j = 1; j < shp::KUSED; j++) {
                const float pp = s_dn[l][j][rr] * s_w[l][j];
                m = m + pp;
            }
            const float sv = s_dn[l][shp::KUSED][rr] * s_sg[l];
            const float f = m + sv;
            a.x2[(int64_t)l * shp::E + row0 + rr] = f + a.x1[(int64_t)l * shp::E + row0 + rr];
        }
    }
}

// ---- LM head over a K-quant matrix: the normed x2 (h_nextn) of every lane, q8_K blocks of it, the
// lane GEMV into the logits, then the first strict maximum per wanted lane (NaN never wins; all
// -inf: no key, argmax 0), packed as the per-phase head packs it: (ordered value << 32) | ~row.
template <int NL>
__global__ __launch_bounds__(256) void kq_head_norm_kernel(const RunCtl *__restrict__ ctl, const float *x2,
                                                           const float *norm_w, float eps, float *hid, float *xn,
                                                           uint8_t *xk) {
    __shared__ NormScratch ns;
    __shared__ float s_n[NL][shp::E];
    if (!ctl->active) return;
    const int nl = ctl->nl, t = threadIdx.x;
#pragma unroll
    for (int l = 0; l < NL; l++) {
        float v[EPT];
        if (l < nl) {
            load8(x2 + (int64_t)l * shp::E, v);
            rms_norm_mul_e(v, x2 + (int64_t)l * shp::E, norm_w, eps, ns);
            store8(hid + (int64_t)l * shp::E, v);
        } else {
#pragma unroll
            for (int i = 0; i < EPT; i++) v[i] = 0.0f;
        }
        store8(xn + (int64_t)l * shp::E, v);
        store8(s_n[l], v);
    }
    q8K_rows_lds<NL>(s_n, xk);   // the head GEMV's activation
}

// workgroup (slice of the rows, lane): 16-byte reads of a slice, then one key per workgroup into the lane's (two
// workgroups of 1024 threads for both lanes' 248320 logits took 77 us, these 5)
constexpr int AM_WG = 128;
template <int NL>
__global__ __launch_bounds__(256) void kq_argmax_kernel(const RunCtl *__restrict__ ctl, const float *logits, int64_t nv,
                                                        unsigned long long *amax_key, const uint32_t *ids) {
    __shared__ unsigned long long red[4];
    if (!ctl->active) return;
    const int l = blockIdx.y, t = threadIdx.x;
    if (l >= ctl->nl || !((ctl->head_mask >> l) & 1)) return;
    float best = -__builtin_inff();
    int64_t bi = -1;
    for (int64_t r = 4 * (blockIdx.x * 256 + t); r < nv; r += 4 * 256 * AM_WG) {
        const float4 v = *(const float4 *)(logits + (int64_t)l * nv + r);
        if (v.x > best) { best = v.x; bi = r; }
        if (v.y > best) { best = v.y; bi = r + 1; }
        if (v.z > best) { best = v.z; bi = r + 2; }
        if (v.w > best) { best = v.w; bi = r + 3; }
    }
    // a restricted draft head's rows are ascending token ids: the first maximum by row is the first by id
    const uint32_t id = bi < 0 ? 0u : (ids ? ids[bi] : (uint32_t)bi);
    unsigned long long key = bi >= 0 ? ((unsigned long long)ordered_bits(best) << 32) | (0xffffffffu - id) : 0ull;
    for (int m = 32; m >= 1; m >>= 1) {
        const unsigned long long o = __shfl_xor(key, m, 64);
        key = o > key ? o : key;
    }
    if ((t & 63) == 0) red[t >> 6] = key;
    __syncthreads();
    if (t == 0) {
        unsigned long long k = 0ull;
        for (int i = 0; i < 4; i++) k = red[i] > k ? red[i] : k;
        if (k) atomicMax(&amax_key[l], k);
    }
}

// ---- K-quant mixer matrices and token embedding in the per-phase runs ----------------------------
// the lanes' token rows of a K-quant embedding (engine.rs:2251-2256): workgroup l = lane
template <int NL>
__global__ __launch_bounds__(256) void kq_embed_kernel(const RunCtl *__restrict__ ctl, const uint8_t *w, int type,
                                                       int64_t row_bytes, float *out) {
    if (!ctl->active) return;
    const int l = blockIdx.x;
    if (l >= ctl->nl) return;
    const uint8_t *row = w + (int64_t)ctl->tok[l] * row_bytes;
    const int bb = kq_block_bytes(type);
    for (int i = threadIdx.x; i < shp::E; i += 256) out[(int64_t)l * shp::E + i] = kq_elem(type, row + (i / QK) * bb, i % QK);
}

// the lanes' projection input: xn = rms_norm(x) * attn_norm (oxe_ops.cpp:32-42), x the embedding
// (Q8_0 emb, or the dequantised rows embf; stored to x_store, the residual of layer 0) or x; lanes
// past the run's are zero
template <int NL>
__global__ __launch_bounds__(256) void kq_norm_kernel(const RunCtl *__restrict__ ctl, const float *x, Q8W emb,
                                                      const float *embf, float *x_store, const float *norm_w, float eps,
                                                      float *xn, uint8_t *xk) {
    __shared__ NormScratch ns;
    __shared__ float s_x[shp::E];
    __shared__ float s_n[NL][shp::E];
    if (!ctl->active) return;
    const int nl = ctl->nl;
#pragma unroll
    for (int l = 0; l < NL; l++) {
        float v[EPT];
        if (l < nl) {
            if (embf) load8(embf + (int64_t)l * shp::E, v);
            else if (emb.q) embed8(emb, ctl->tok[l], v);
            else load8(x + (int64_t)l * shp::E, v);
            if (x_store && (embf || emb.q)) store8(x_store + (int64_t)l * shp::E, v);
            store8(s_x, v);   // the replay source of the exact-sum fallback
            __syncthreads();
            rms_norm_mul_e(v, s_x, norm_w, eps, ns);
            __syncthreads();
        } else {
#pragma unroll
            for (int i = 0; i < EPT; i++) v[i] = 0.0f;
        }
        store8(xn + (int64_t)l * shp::E, v);
        store8(s_n[l], v);
    }
    q8K_rows_lds<NL>(s_n, xk);   // the GEMV's activation: q8_K blocks of xn
}

}  // namespace kq

int launch_ba_f32(const RunCtl *ctl, const ModelRt &m, const LayerW &w, const float *x, const ActBufs &b, hipStream_t st) {
    hipLaunchKernelGGL(kq::ba_f32_kernel<OXE_NL>, dim3(2 * shp::NVH / 16), dim3(256), 0, st, ctl, x, w.attn_norm, m.eps,
                       (const float *)w.beta_r.w, (const float *)w.alpha_r.w, b.proj);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// q8_K blocks of nblk consecutive 256-value blocks of x (every lane of a [NL][n] buffer at once)
static void quant_k(const float *x, int64_t nblk, uint8_t *y, hipStream_t st) {
    hipLaunchKernelGGL(kq::quant_q8_K_kernel, dim3((unsigned)((nblk + 3) / 4)), dim3(256), 0, st, x, nblk, y);
}

int launch_kq_moe(const RunCtl *ctl, const ModelRt &m, const LayerW &w, const ActBufs &b, hipStream_t st) {
    (void)m;
    const bool exp_gu = w.exp_gate_r.type != 8, sh_gu = w.sh_gate_r.type != 8;
    if (!exp_gu) launch_experts(ctl, w, b, st);
    if (exp_gu || sh_gu) {
        kq::KqGuArgs a{};
        a.xn = b.xn;
        a.gate = w.exp_gate_r;
        a.up = w.exp_up_r;
        a.sh_gate = w.sh_gate_r;
        a.sh_up = w.sh_up_r;
        a.uni = b.uni;
        a.route_ids = b.route_ids;
        a.hexp = b.hexp;
        a.hsh = b.hsh;
        a.do_exp = exp_gu;
        a.do_sh = sh_gu;
        a.stats = b.counters + CNT_UNI_SUM;
        // a tile's gate and up rows in LDS, of whichever unit is larger
        const int64_t le = exp_gu ? raw_row_bytes(a.gate) + raw_row_bytes(a.up) : 0;
        const int64_t ls = sh_gu ? raw_row_bytes(a.sh_gate) + raw_row_bytes(a.sh_up) : 0;
        hipLaunchKernelGGL(kq::kq_gu_kernel<OXE_NL>, dim3((OXE_MAX_UNION + 1) * (shp::FF / kq::GU_R)), dim3(256),
                           (size_t)(kq::GU_R * std::max(le, ls)), st, ctl, a);
    }
    kq::KqDownArgs d{};
    d.uni = b.uni;
    d.route_ids = b.route_ids;
    d.route_w = b.route_w;
    d.sh_gate = b.sh_gate;
    d.hexp = b.hexp;
    d.hsh = b.hsh;
    d.exp_down = w.exp_down;
    d.shexp_down = w.shexp_down;
    d.exp_down_r = w.exp_down_r;
    d.sh_down_r = w.sh_down_r;
    d.x1 = b.x1;
    d.x2 = b.x2;
    d.amax_key = b.amax_key;
    hipLaunchKernelGGL(kq::kq_down_kernel<OXE_NL>, dim3(shp::E / kq::DN_R), dim3(kq::DN_T), 0, st, ctl, d);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_kq_head(const RunCtl *ctl, const ModelRt &m, const float *norm_w, const ActBufs &b, hipStream_t st,
                   const RawW *w, const uint32_t *ids) {
    hipLaunchKernelGGL(kq::kq_head_norm_kernel<OXE_NL>, dim3(1), dim3(256), 0, st, ctl, b.x2, norm_w, m.eps, b.hid, b.xn,
                       b.xk);
    const int nb = shp::E / kq::QK;
    const RawW &o = w ? *w : m.output_r;
    int rc;
    switch (o.type) {
        case 11: rc = kq::vl_gemv_type<3>(o.w, nb, o.rows, b.xk, OXE_NL, b.logits, st); break;
        case 12: rc = kq::vl_gemv_type<4>(o.w, nb, o.rows, b.xk, OXE_NL, b.logits, st); break;
        case 13: rc = kq::vl_gemv_type<5>(o.w, nb, o.rows, b.xk, OXE_NL, b.logits, st); break;
        default: rc = kq::vl_gemv_type<6>(o.w, nb, o.rows, b.xk, OXE_NL, b.logits, st); break;
    }
    if (rc != 1) return -2;
    hipLaunchKernelGGL(kq::kq_argmax_kernel<OXE_NL>, dim3(kq::AM_WG, OXE_NL), dim3(256), 0, st, ctl, b.logits, o.rows, b.amax_key, ids);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// the lane GEMV over a matrix of ggml type 11..14 (nb blocks per row), s[l * rows + r]; 1: done
static int vl_gemv_any(int type, const kq::KqSegs &S, int nb, const uint8_t *y, hipStream_t st, const kq::KqEpi &epi) {
    switch (type) {
        case 11: return kq::vl_gemv_segs<3>(S, nb, y, OXE_NL, nullptr, st, epi);
        case 12: return kq::vl_gemv_segs<4>(S, nb, y, OXE_NL, nullptr, st, epi);
        case 13: return kq::vl_gemv_segs<5>(S, nb, y, OXE_NL, nullptr, st, epi);
        case 14: return kq::vl_gemv_segs<6>(S, nb, y, OXE_NL, nullptr, st, epi);
        default: return 0;
    }
}

int launch_kq_embed(const RunCtl *ctl, const ModelRt &m, float *out, hipStream_t st) {
    const RawW &e = m.tok_embd_r;
    if (e.type < 11 || e.type > 14) return -1;
    hipLaunchKernelGGL(kq::kq_embed_kernel<OXE_NL>, dim3(OXE_NL), dim3(256), 0, st, ctl, e.w, e.type, raw_row_bytes(e), out);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_kq_proj(const RunCtl *ctl, const ModelRt &m, const LayerW &w, const float *x, bool embed, float *x_store,
                   const ActBufs &b, hipStream_t st, int64_t row_begin) {
    using namespace shp;
    const bool kemb = embed && m.tok_embd_r.type != 8;
    hipLaunchKernelGGL(kq::kq_norm_kernel<OXE_NL>, dim3(1), dim3(256), 0, st, ctl, x, embed && !kemb ? m.tok_embd : Q8W{},
                       kemb ? b.emb : nullptr, x_store, w.attn_norm, m.eps, b.xn, b.xk);
    struct Part {
        const RawW *r;
        int64_t off;
        bool v;
    };
    const Part dn[4] = {{&w.qkv_r, 0, false}, {&w.z_r, DN_Z, false}, {&w.beta_r, DN_BETA, false}, {&w.alpha_r, DN_ALPHA, false}};
    const Part at[3] = {{&w.q_r, 0, false}, {&w.k_r, AT_K, false}, {&w.v_r, AT_V, true}};
    const Part *ps = w.att ? at : dn;
    const int np = w.att ? 3 : 4;
    kq::KqEpi epi;       // the rows straight into the run's projection buffer (V rows also to V^T)
    epi.ctl = ctl;
    epi.dst = b.proj;
    epi.ld = DN_ROWS;
    epi.vt = w.att ? m.vcache + (int64_t)w.index * NKV * HD * m.n_ctx : nullptr;
    epi.vt_ld = m.n_ctx;
    // consecutive parts of one K-quant type share a launch
    kq::KqSegs S;
    int ty = 0;
    auto flush = [&]() {
        const int rc = S.n ? vl_gemv_any(ty, S, (int)(E / kq::QK), b.xk, st, epi) : 1;
        S = kq::KqSegs{};
        return rc == 1;
    };
    for (int i = 0; i < np; i++) {
        const RawW &r = *ps[i].r;
        if (ps[i].off < row_begin || r.type < 11 || r.type > 14) continue;   // F32 beta / alpha: launch_ba_f32
        if (S.n && r.type != ty && !flush()) return -2;
        ty = r.type;
        const int j = S.n++;
        S.w[j] = (const uint8_t *)r.w;
        S.nr[j] = r.rows;
        S.g0[j] = S.ngroups;
        S.off[j] = ps[i].off;
        if (ps[i].v) S.vseg = j;
        S.ngroups += (r.rows + kq::GR - 1) / kq::GR;
    }
    if (!flush()) return -2;
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_kq_out(const RunCtl *ctl, const ModelRt &m, const LayerW &w, const float *x, const ActBufs &b, hipStream_t st) {
    (void)m;
    using namespace shp;
    const RawW &r = w.out_r;
    quant_k(b.o32, (int64_t)OXE_NL * MIX_W / kq::QK, b.ok, st);
    kq::KqEpi epi;       // mixer_out's residual (engine.rs:2573-2609) at the store: x1 = out + x
    epi.ctl = ctl;
    epi.dst = b.x1;
    epi.ld = E;
    epi.resid = x;
    if (vl_gemv_any(r.type, kq::one_seg((const uint8_t *)r.w, E), (int)(MIX_W / kq::QK), b.ok, st, epi) != 1) return -2;
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace oxe

extern "C" {

int oxe_hip_quantize_row_q8_K(const float *x, int64_t k, int64_t nrows, void *y, void *stream) {
    if (!x || !y || k <= 0 || k % oxe::kq::QK != 0 || nrows <= 0) return -1;
    if (((uintptr_t)x & 15) != 0 || ((uintptr_t)y & 3) != 0) return -1;
    const int64_t nblk = k / oxe::kq::QK * nrows;
    hipLaunchKernelGGL(oxe::kq::quant_q8_K_kernel, dim3((unsigned)((nblk + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, x, nblk, (uint8_t *)y);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int oxe_hip_vl_gemv(int type, int64_t k, int64_t nr, int nl, const void *w, const void *y, float *s, void *stream) {
    using namespace oxe::kq;
    if (nl < 1 || nl > MAX_LANES || nr <= 0 || k <= 0 || k % QK != 0 || k > 8192 || !w || !y || !s) return 0;
    if (((uintptr_t)w & 15) != 0 || ((uintptr_t)y & 3) != 0) return 0;
    const int nb = (int)(k / QK);
    const hipStream_t st = (hipStream_t)stream;
    const uint8_t *wb = (const uint8_t *)w, *yb = (const uint8_t *)y;
    switch (type) {
        case 4: return vl_gemv_type<4>(wb, nb, nr, yb, nl, s, st);
        case 5: return vl_gemv_type<5>(wb, nb, nr, yb, nl, s, st);
        // 110- and 210-byte blocks: rows of an even block count keep every 4-row group 16-byte aligned
        case 3: return nb % 2 ? 0 : vl_gemv_type<3>(wb, nb, nr, yb, nl, s, st);
        case 6: return nb % 2 ? 0 : vl_gemv_type<6>(wb, nb, nr, yb, nl, s, st);
        default: return 0;
    }
}

}  // extern "C"
