// Batched prefill over K-quant matrices (k_pf_kquant.hip), callable from the host side of the engine.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oxe_engine.h"

namespace oxe {

// q8_K activations of the K-quant GEMM, rows of nb blocks of 256 values. One code array per kind of
// weight: f16 (Q4_K, Q5_K) in the GEMM's fragment order, int8 (Q3_K, Q6_K) in order; either may be
// null when no consumer of that kind follows.
struct KqAct {
    uint16_t *c16;   // [rows][nb][256]
    int8_t *c8;      // [rows][nb][256]
    float *d;        // [rows][nb] block scales
    uint16_t *bs;    // [rows][nb][16] sums of 16 codes, f16 (exact: at most 16 * 127)
};

// one matrix of a GEMM launch: rows go to y at column offset off; group g's rows at w + g * gstride
constexpr int KQG_SEGS = 4;
struct KqGemmSeg {
    const uint8_t *w;
    int64_t nr, off, gstride;
};
// y[p][off + r] = W[r] . x[xrow ? xrow[p] : p] (+ res[p][off + r]), token rows and tiles as GemmArgs
struct KqGemmArgs {
    KqGemmSeg seg[KQG_SEGS];
    int32_t tile0[KQG_SEGS];   // first row tile of each segment
    int32_t nseg, nb;
    KqAct x;
    float *y;
    const float *res;
    int64_t ldy, ldr, nt;
    const int4 *tiles;
    const int32_t *xrow;
    const int32_t *tile_count;
};

// whether a matrix of ggml type t reads the f16 codes (else the int8 ones)
inline bool kqg_f16(int t) { return t == 12 || t == 13; }

// every segment of ggml type `type` (11..14); grouped: ntiles tiles. 0, -1 (bad shape), -2
int kq_gemm_launch(int type, KqGemmArgs a, int64_t ntiles, hipStream_t st);
// q8_K of rows of k values at x (row stride ldx)
int kq_pf_quant(const float *x, int64_t ldx, int64_t rows, int64_t k, KqAct y, hipStream_t st);
// swiglu of gate / up rows (512 values each; split: [gate | up], else interleaved 8 by 8) and its
// Q8_0 or q8_K codes
int kq_pf_swiglu_q8_0(const float *gu, bool split, int64_t rows, int8_t *hq, uint16_t *hd, hipStream_t st);
int kq_pf_swiglu_q8_K(const float *gu, bool split, int64_t rows, KqAct h, hipStream_t st);
// dequantised token rows of a K-quant embedding
int kq_pf_embed(const RawW &e, const uint32_t *toks, int64_t n, float *x, hipStream_t st);
// the LM head of one normed row over a K-quant matrix: its q8_K blocks (292-byte form) at xk, the
// lane GEMV's values at logits
int kq_head_one(const RawW &w, const float *xn, uint8_t *xk, float *logits, hipStream_t st);

}  // namespace oxe
