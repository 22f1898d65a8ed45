// K-quant block arithmetic shared by the decode kernels (k_kquant.hip) and the batched prefill
// (k_pf_kquant.hip): the q8_K quantiser of one block and single-element dequantisation.
#pragma once
#include "oxe_common.h"

namespace oxe {
namespace kq {

constexpr int QK = 256;
constexpr int Q8K_BYTES = 292;   // block_q8_K: float d, int8 qs[256], int16 bsums[16]
constexpr int Q8K_QS = 4, Q8K_BS = 260;

// ---- quantize_row_q8_K_ref (vendor/ggml-subset/generated/quants_base.c:14-48) --------------------
// One wave per 256-value block; thread t holds values 4 t .. 4 t + 3. The block maximum is the
// first value of largest magnitude (the reference's strict > scan); iscale = -127 / max (f32
// division), codes = nearest_int(iscale * x) (the float add of 1.5 * 2^23: round half to even),
// clamped above at 127; bsums = sums of 16 codes; d = 1 / iscale. An all-zero block gets d = 0 and
// zero codes and sums.
// (v: this lane's four values; every lane of one wave) the lane's codes; returns d
OXE_DEV float q8K_codes(const float (&v)[4], int lane, int (&q)[4]) {
    float am = 0.0f, mx = 0.0f;
    for (int e = 0; e < 4; e++) {
        const float ax = fabsf(v[e]);
        if (ax > am) {
            am = ax;
            mx = v[e];
        }
    }
    // the wave's largest magnitude by lane moves, then the first lane that holds it (lanes hold values in order)
    const float top = wave_max_any(am);
    const unsigned long long at = __ballot(am == top);
    mx = readlane_f(mx, __builtin_ctzll(at));
    am = top;
    q[0] = q[1] = q[2] = q[3] = 0;
    if (am == 0.0f) return 0.0f;
    const float iscale = -127.f / mx;
    for (int e = 0; e < 4; e++) {
        const float p = iscale * v[e];
        const float t = p + 12582912.f;
        const int r = (int)(__builtin_bit_cast(uint32_t, t) & 0x007fffffu) - 0x00400000;
        q[e] = r < 127 ? r : 127;
    }
    return 1 / iscale;
}
OXE_DEV uint32_t pack4(const int (&q)[4]) {
    return (uint32_t)(q[0] & 255) | (uint32_t)(q[1] & 255) << 8 | (uint32_t)(q[2] & 255) << 16 | (uint32_t)(q[3] & 255) << 24;
}
// the lane's sum of 16 codes (every lane of four holds it)
OXE_DEV int sum16(const int (&q)[4]) {
    int s = q[0] + q[1] + q[2] + q[3];
    s += dpp_i<DPP_XOR1>(s);
    s += dpp_i<DPP_XOR2>(s);
    return s;
}
// the same into a ggml block_q8_K (xb: the block's 256 values)
OXE_DEV void q8K_block(const float *xb, int lane, uint8_t *__restrict__ yb) {
    const float4 v4 = *(const float4 *)(xb + 4 * lane);
    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
    int q[4];
    const float d = q8K_codes(v, lane, q);
    *(uint32_t *)(yb + Q8K_QS + 4 * lane) = pack4(q);
    const int s = sum16(q);
    if ((lane & 3) == 0) *(int16_t *)(yb + Q8K_BS + 2 * (lane >> 2)) = (int16_t)s;
    if (lane == 0) *(float *)yb = d;
}

// get_scale_min_k4 (quants_base.c:50-57)
OXE_DEV void scale_min_k4(int j, const uint8_t *q, int &d, int &m) {
    if (j < 4) {
        d = q[j] & 63;
        m = q[j + 4] & 63;
    } else {
        d = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
        m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
}

// q3k_raw_scales (repack_subset.cpp:575-587): raw 6-bit scale i of a Q3_K block
OXE_DEV int q3_raw(const uint8_t *s12, int i) {
    const int lo = i < 8 ? (s12[i] & 15) : (s12[i - 8] >> 4);
    const int hi = (s12[8 + (i & 3)] >> (2 * (i >> 2))) & 3;
    return lo | hi << 4;
}

// dequantize_row_q{3,4,5,6}_K (vendor/ggml-subset/generated/quants_base.c:80-230) of element i of
// one 256-weight block b (type 11..14), as the reference builds it: GCC's default contraction
// (crates/kernels-sys/build.rs:5-7) makes the Q4_K / Q5_K element (d * scale) * code - dmin * min
// one fused multiply-subtract; Q3_K and Q6_K are products in source order.
OXE_DEV float ld_f16u(const uint8_t *p) { return h2f((uint16_t)(p[0] | (p[1] << 8))); }
OXE_DEV float kq_elem(int type, const uint8_t *b, int i) {
    switch (type) {
        case 12:
        case 13: {
            const float d = ld_f16u(b), mn = ld_f16u(b + 2);
            const int c = i >> 6, hi = (i >> 5) & 1, l = i & 31;
            const uint8_t *q = b + (type == 12 ? 16 : 48) + 32 * c;
            int sc, mi;
            scale_min_k4(2 * c + hi, b + 4, sc, mi);
            int qq = hi ? (q[l] >> 4) : (q[l] & 0xF);
            if (type == 13 && (b[16 + l] & ((1 + hi) << (2 * c)))) qq += 16;
            return __builtin_fmaf(d * (float)sc, (float)qq, -(mn * (float)mi));
        }
        case 14: {
            const float d = ld_f16u(b + 208);
            const int n = i >> 7, r = i & 127, qd = r >> 5, l = r & 31;
            const uint8_t *ql = b + 64 * n, *qh = b + 128 + 32 * n;
            const int8_t sc = (int8_t)b[192 + 8 * n + (l >> 4) + 2 * qd];
            const int lo = (qd & 1) ? ql[l + 32] : ql[l];
            const int q = ((qd >> 1) ? (lo >> 4) : (lo & 0xF)) | (((qh[l] >> (2 * qd)) & 3) << 4);
            return d * (float)sc * (float)(q - 32);
        }
        default: {   // 11: Q3_K
            const float dall = ld_f16u(b + 108);
            const int n = i >> 7, r = i & 127, j = r >> 5, hf = (r >> 4) & 1, idx = (r & 15) + 16 * hf;
            const float dl = dall * (float)(q3_raw(b + 96, 8 * n + 2 * j + hf) - 32);
            const int code = (b[32 + 32 * n + idx] >> (2 * j)) & 3;
            return dl * (float)(code - ((b[idx] & (1 << (4 * n + j))) ? 0 : 4));
        }
    }
}

}  // namespace kq
}  // namespace oxe
