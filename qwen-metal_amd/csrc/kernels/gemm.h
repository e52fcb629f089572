/* Pieces shared by the linears (the GEMM kernels themselves are in
 * gemm_q.h):
 *   out[m, n] = epilogue( sum_k A[m, k] * W[n, k] )
 * A bf16 row-major (row stride lda), W in the checkpoint's native [out, in]
 * layout (bf16, or int8 with one fp32 scale per output row), fp32
 * accumulation.
 *
 * - int8 -> bf16 widening (exact for |q| <= 127): a whole-weight pass
 *   (qw_widen_i8_bf16) and the per-fragment form the int8 GEMM uses; the
 *   per-row scale multiplies the fp32 sums in the epilogue, so the
 *   contraction equals the dequantised product.
 * - the streaming GEMV kernels for linears of at most 8 rows;
 * - the tile order (XCD-aware) and the direct-to-LDS load helpers;
 * - the epilogue (scale, bias, GELU, residual gate, q/k norm + RoPE), which
 *   stages the fp32 sums through LDS and writes whole 256-byte row runs.
 */
#pragma once
#include "common.h"

#define GBK 64
/* End of a K-slice: its direct loads landed
 * (vmcnt(0)) and this wave's LDS reads done, then a bare s_barrier. The
 * direct loads are issued from inline assembly, so the compiler's own wait
 * insertion does not know them; this wait is the one that covers them. */
#define QW_SLICE_END() asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory")
/* floats per split-tile partial (one 256 x 256 tile) */
#define QW_SPLIT_PART (256u * 256u)
/* buffer cache policy sc0 | sc1: coherent at device scope */
#define QW_CPOL_COHERENT 17
/* buffer cache policy nt: non-temporal */
#define QW_CPOL_NT 2

/* int8 x16 -> bf16 x16 (exact: bf16 holds every 8-bit integer), as two
 * 16-byte chunks: byte-select conversions to fp32, packed pairwise. */
__device__ __forceinline__ void i8x16_to_bf16(u32x4 q, u32x4 &lo, u32x4 &hi) {
    uint32_t o[8];
#pragma unroll
    for (int w = 0; w < 4; w++) {
        int32_t x = (int32_t)q[w];
        o[2 * w] = pack_bf((float)((x << 24) >> 24), (float)((x << 16) >> 24));
        o[2 * w + 1] = pack_bf((float)((x << 8) >> 24), (float)(x >> 24));
    }
    lo = u32x4{o[0], o[1], o[2], o[3]};
    hi = u32x4{o[4], o[5], o[6], o[7]};
}

/* int8 x8 -> bf16 x8 (one MFMA fragment), exact */
__device__ __forceinline__ bf16x8 i8x8_to_bf16(u32x2 q) {
    uint32_t o[4];
#pragma unroll
    for (int w = 0; w < 2; w++) {
        const int32_t x = (int32_t)q[w];
        o[2 * w] = pack_bf((float)((x << 24) >> 24), (float)((x << 16) >> 24));
        o[2 * w + 1] = pack_bf((float)((x << 8) >> 24), (float)(x >> 24));
    }
    return __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
}

/* out[i] = bf16(q[i]) for count int8 weights (count % 16 == 0): the
 * unscaled widening that lets int8 linears run on the bf16 GEMM, whose
 * epilogue then applies the per-row scale to the fp32 sums. 8 weights per
 * thread and step (an 8-byte load, a 16-byte store): measured 17-19%
 * faster than 16 per step on the step's three weights. */
QW_KERNEL void __launch_bounds__(256) qw_widen_i8_bf16(qw_widen_args a) {
    const uint64_t n8 = a.count / 8;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
         i += (uint64_t)gridDim.x * blockDim.x)
        ((u32x4 *)a.out)[i] = __builtin_bit_cast(u32x4, i8x8_to_bf16(((const u32x2 *)a.in)[i]));
}

/* Linears with at most QW_GEMV_MAX_ROWS rows (the timestep / modulation
 * MLP runs on 1-2 rows): a 256 x 256 tile would be almost all padding and
 * its K loop latency-bound, so each wave instead streams QW_GEMV_COLS weight
 * rows (bf16, or int8 widened in registers) once, 16 bytes per lane, against
 * the same k chunks of every input row, with fp32 FMAs and a wave-shuffle
 * sum. The epilogue is the GEMM's: y = bf16(acc * wscale + bias) (the int8
 * scale multiplies the finished sum, as in the tiled kernels), then GELU or
 * a plain store. */
#define QW_GEMV_MAX_ROWS 8
#define QW_GEMV_COLS 2
template <int INT8, int EPI>
__device__ __forceinline__ void qw_gemv_impl(const qw_gemm_args &a) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t c0 = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * QW_GEMV_COLS;
    if (c0 >= a.n) return; /* whole waves */
    const uint32_t m = a.m, kc = a.k / 8;
    const u16 *A = (const u16 *)a.a;
    float acc[QW_GEMV_MAX_ROWS][QW_GEMV_COLS];
#pragma unroll
    for (int r = 0; r < QW_GEMV_MAX_ROWS; r++)
#pragma unroll
        for (int c = 0; c < QW_GEMV_COLS; c++) acc[r][c] = 0.0f;
    for (uint32_t j = lane; j < kc; j += 64) {
        float w[QW_GEMV_COLS][8];
#pragma unroll
        for (int c = 0; c < QW_GEMV_COLS; c++) {
            const uint32_t col = min(c0 + c, a.n - 1);
            if (INT8) {
                const u32x2 q = *(const u32x2 *)((const int8_t *)a.w + (size_t)col * a.k + 8 * j);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int32_t x = (int32_t)q[h];
                    w[c][4 * h] = (float)((x << 24) >> 24);
                    w[c][4 * h + 1] = (float)((x << 16) >> 24);
                    w[c][4 * h + 2] = (float)((x << 8) >> 24);
                    w[c][4 * h + 3] = (float)(x >> 24);
                }
            } else {
                const u32x4 q = *(const u32x4 *)((const u16 *)a.w + (size_t)col * a.k + 8 * j);
#pragma unroll
                for (int i = 0; i < 4; i++) w[c][2 * i] = lo_bf(q[i]), w[c][2 * i + 1] = hi_bf(q[i]);
            }
        }
#pragma unroll
        for (int r = 0; r < QW_GEMV_MAX_ROWS; r++) {
            if ((uint32_t)r >= m) break;
            const u32x4 x = *(const u32x4 *)(A + (size_t)r * a.lda + 8 * j);
            float xf[8];
#pragma unroll
            for (int i = 0; i < 4; i++) xf[2 * i] = lo_bf(x[i]), xf[2 * i + 1] = hi_bf(x[i]);
#pragma unroll
            for (int c = 0; c < QW_GEMV_COLS; c++)
#pragma unroll
                for (int i = 0; i < 8; i++) acc[r][c] = fmaf(xf[i], w[c][i], acc[r][c]);
        }
    }
#pragma unroll
    for (int r = 0; r < QW_GEMV_MAX_ROWS; r++) {
        if ((uint32_t)r >= m) break;
#pragma unroll
        for (int c = 0; c < QW_GEMV_COLS; c++) {
            float t = wave_sum(acc[r][c]);
            const uint32_t col = c0 + c;
            if (lane != 0 || col >= a.n) continue;
            if (a.wscale) t *= a.wscale[col];
            float y = bf2f(f2bf(t + (a.bias ? bf2f(a.bias[col]) : 0.0f)));
            if (EPI == QW_EPI_GELU) y = gelu_tanh_f(y);
            a.out[(size_t)r * a.ldc + col] = f2bf(y);
        }
    }
}
QW_KERNEL void __launch_bounds__(256) qw_gemv_bf16_store(qw_gemm_args a) {
    qw_gemv_impl<0, QW_EPI_STORE>(a);
}
QW_KERNEL void __launch_bounds__(256) qw_gemv_bf16_gelu(qw_gemm_args a) {
    qw_gemv_impl<0, QW_EPI_GELU>(a);
}
QW_KERNEL void __launch_bounds__(256) qw_gemv_i8_store(qw_gemm_args a) {
    qw_gemv_impl<1, QW_EPI_STORE>(a);
}
QW_KERNEL void __launch_bounds__(256) qw_gemv_i8_gelu(qw_gemm_args a) {
    qw_gemv_impl<1, QW_EPI_GELU>(a);
}

/* Workgroup id -> (tile row, tile column). Ids are dealt round-robin to the
 * 8 XCDs; the id is remapped so each XCD owns a contiguous range of tiles,
 * walked in groups of 4 tile-rows (column-major inside a group), so the A
 * and W panels an XCD touches stay hot in its L2. */
__device__ __forceinline__ void gemm_tile_in(uint32_t tiles_m, uint32_t tiles_n, uint32_t pid,
                                             uint32_t &tm, uint32_t &tn) {
#ifndef QW_GEMM_GROUP
/* 4 against 8 (same box, alternating, M = 8704): QKV 381 / 388, out 150 /
 * 152, up 509 / 514, down 572 / 578 us (medians), steps 66.15 / 66.62 ms */
#define QW_GEMM_GROUP 4
#endif
    const uint32_t G = QW_GEMM_GROUP;
    const uint32_t per_group = G * tiles_n;
    const uint32_t first_m = (pid / per_group) * G;
    const uint32_t gsize = min(tiles_m - first_m, G);
    const uint32_t inner = pid % per_group;
    tm = first_m + inner % gsize;
    tn = inner / gsize;
}
__device__ __forceinline__ void gemm_tile_at(const qw_gemm_args &a, uint32_t pid, uint32_t &tm,
                                             uint32_t &tn) {
    gemm_tile_in(a.tiles_m, a.tiles_n, pid, tm, tn);
}
/* id -> its place among n when each residue class mod 8 (one XCD, as ids are
 * dealt) takes one contiguous range, for any n */
__device__ __forceinline__ uint32_t gemm_xcd_range(uint32_t id, uint32_t n) {
    const uint32_t x = id & 7u;
    return x * (n >> 3) + min(x, n & 7u) + (id >> 3);
}
/* Epilogue through LDS: the fp32 sums of each 32-row slab of the wave's
 * block are first written to a wave-private LDS region (row stride
 * NI*32 + 4 floats: the 16 lanes of a ds_write_b128 pass land on 16
 * distinct 4-bank groups), then read back row-contiguous: 16 lanes per row,
 * 8 columns (one 16-byte store) per lane, so every output row segment is
 * written by whole 256-byte runs, and the residual/gate reads of the GATE
 * epilogue are coalesced the same way. A lane keeps the same 8 columns for
 * every row, so it loads their scale and bias once.
 *
 * write_slab(mi) stages slab mi (SR rows) of the wave's fp32 sums; read_row(lr,
 * v) returns this lane's 8 sums of row lr of the staged slab.
 *
 * Rows are processed RP at a time without branches: a lane outside the
 * output (row >= m, or its columns >= n) addresses its output and residual
 * past the end of a buffer resource, so its loads return zeros and its
 * stores are dropped. The per-row operands of the RP rows (residual, gate,
 * RoPE table rows) are issued before their LDS reads, so the rows' memory
 * latencies overlap each other instead of adding up row by row.
 *
 * MODE 0: a finished tile. MODE 1: a piece of a split tile, whose fp32 sums
 * are stored to its partial slot. MODE 2: the last piece of a split tile,
 * which adds all pieces' sums in piece order (its own from LDS) and runs
 * the epilogue. */
template <int EPI, int INT8, int NSLAB, int SR, int RP, int MODE, class SlabWriter,
          class SlabReader>
__device__ __forceinline__ void gemm_epilogue_mode(const qw_gemm_args &a, SlabWriter write_slab,
                                                   SlabReader lds_row, uint32_t row0,
                                                   uint32_t col0, uint32_t lane, float *pst,
                                                   const float *pld, uint32_t npart,
                                                   uint32_t own) {
#pragma clang fp contract(off)
    static_assert((SR / 4) % RP == 0, "rows per pass");
    const bool scaled = INT8 || a.wscale != nullptr;
    /* split-tile partials go through device-coherent buffer accesses (write
     * through / read past the XCD's L2), so pieces on different XCDs see
     * each other's sums without any L2 write-back or invalidate */
    const __amdgpu_buffer_rsrc_t part_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)a.sk_part, (short)0, (int)0x7FFFFFF0, 0x00020000);
    /* read-back geometry: lane -> (row within a 4-row group, 8-column chunk
     * of the wave's 128 columns) */
    const uint32_t rr = lane >> 4, cc = lane & 15;
    const uint32_t col = col0 + cc * 8;
    const bool col_ok = col < a.n;                 /* n % 8 == 0 */
    /* where this wave's columns go: with separate k and v outputs, one head of
     * 128 columns lies in one of them */
    void *out = (void *)a.out;
    uint32_t out_bytes = a.out_bytes, ldc = a.ldc, out_col = col;
    if (EPI == QW_EPI_QKNORM && MODE != 1 && a.out_k && col0 >= a.qk_cols / 2) {
        const bool v = col0 >= a.qk_cols;
        out = v ? (void *)a.out_v : (void *)a.out_k;
        out_bytes = a.kv_bytes;
        ldc = a.ld_kv;
        out_col = col - (v ? a.qk_cols : a.qk_cols / 2);
    }
    const __amdgpu_buffer_rsrc_t out_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(out, (short)0, (int)out_bytes, 0x00020000);
    const uint32_t colc = col_ok ? col : a.n - 8;  /* in-range column for operand loads */
    float sc[8], bias[8];
#pragma unroll
    for (int j = 0; j < 8; j++) sc[j] = 1.0f, bias[j] = 0.0f;
    if (MODE != 1) {
        if (scaled) {
            const floatx4 s0 = *(const floatx4 *)(a.wscale + colc);
            const floatx4 s1 = *(const floatx4 *)(a.wscale + colc + 4);
#pragma unroll
            for (int j = 0; j < 4; j++) sc[j] = s0[j], sc[4 + j] = s1[j];
        }
        if (a.bias) {
            const u32x4 bb = *(const u32x4 *)(a.bias + colc);
#pragma unroll
            for (int j = 0; j < 4; j++) bias[2 * j] = lo_bf(bb[j]), bias[2 * j + 1] = hi_bf(bb[j]);
        }
    }
    /* QW_EPI_QKNORM: this wave's 128 columns are one head (tiles start at
     * multiples of 128); q or k heads get the norm weight of their kind */
    const bool qk_head = EPI == QW_EPI_QKNORM && MODE != 1 && col0 < a.qk_cols;
    float nw[8];
    if (EPI == QW_EPI_QKNORM && qk_head) {
        const u32x4 wn = *(const u32x4 *)((col0 < a.qk_cols / 2 ? a.norm_q : a.norm_k) + 8 * cc);
#pragma unroll
        for (int i = 0; i < 4; i++) nw[2 * i] = lo_bf(wn[i]), nw[2 * i + 1] = hi_bf(wn[i]);
    }
    /* RoPE table row (row % rope_rows) of this lane's row row0 + rr + off,
     * from one division per tile: the rows are consecutive and off < 128,
     * and the host sends only tables of at least 128 rows here, so one
     * subtraction wraps each. Rows past the output read a row of the table
     * and are not stored. */
    const uint32_t rope_base = EPI == QW_EPI_QKNORM && qk_head ? (row0 + rr) % a.rope_rows : 0;
    auto rope_row = [&](uint32_t off) __attribute__((always_inline)) {
        const uint32_t r = rope_base + off;
        return r >= a.rope_rows ? r - a.rope_rows : r;
    };
#pragma unroll
    for (int mi = 0; mi < NSLAB; mi++) {
        write_slab(mi); /* fp32 sums of rows [SR mi, SR mi + SR) into the LDS region */
#pragma unroll
        for (int p0 = 0; p0 < SR / 4; p0 += RP) {
            uint32_t ooff[RP];
            u32x4 gv[RP], rv[RP];
            floatx4 rc[RP], rs[RP];
#pragma unroll
            for (int i = 0; i < RP; i++) {
                const uint32_t row = row0 + mi * SR + 4 * (p0 + i) + rr;
                ooff[i] = col_ok && row < a.m ? (row * ldc + out_col) * 2 : 0x80000000u;
                if (EPI == QW_EPI_GATE && MODE != 1) {
                    const uint32_t mrow = a.row_map[min(row, a.m - 1)];
                    gv[i] = *(const u32x4 *)(a.gate + (size_t)mrow * a.gate_row_stride + colc);
                    rv[i] = __builtin_bit_cast(
                        u32x4, __builtin_amdgcn_raw_buffer_load_b128(out_rsrc, ooff[i], 0, 0));
                }
            }
            if (EPI == QW_EPI_QKNORM && qk_head) {
#pragma unroll
                for (int i = 0; i < RP; i++) {
                    const size_t t = (size_t)rope_row(mi * SR + 4 * (p0 + i)) * 64 + 4 * cc;
                    rc[i] = *(const floatx4 *)(a.rope_cos + t);
                    rs[i] = *(const floatx4 *)(a.rope_sin + t);
                }
            }
            float y[RP][8];
            if (MODE == 2) { /* all pieces of a split tile, summed in piece order */
#pragma unroll
                for (int i = 0; i < RP; i++)
#pragma unroll
                    for (int j = 0; j < 8; j++) y[i][j] = 0.0f;
                for (uint32_t pc = 0; pc < npart; pc++) {
                    if (pc == own) {
#pragma unroll
                        for (int i = 0; i < RP; i++) {
                            float v[8];
                            lds_row(4 * (p0 + i) + rr, v);
#pragma unroll
                            for (int j = 0; j < 8; j++) y[i][j] += v[j];
                        }
                    } else {
#pragma unroll
                        for (int i = 0; i < RP; i++) {
                            const uint32_t poff = (mi * SR + 4 * (p0 + i) + rr) * 256 + cc * 8;
                            const uint32_t bo =
                                (uint32_t)((pld - a.sk_part) + pc * QW_SPLIT_PART + poff) * 4;
                            const floatx4 q0 = __builtin_bit_cast(
                                floatx4, __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, bo, 0,
                                                                               QW_CPOL_COHERENT));
                            const floatx4 q1 = __builtin_bit_cast(
                                floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                             part_rsrc, bo + 16, 0, QW_CPOL_COHERENT));
#pragma unroll
                            for (int j = 0; j < 4; j++) y[i][j] += q0[j], y[i][4 + j] += q1[j];
                        }
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < RP; i++) lds_row(4 * (p0 + i) + rr, y[i]);
            }
            if constexpr (MODE == 1) { /* piece of a split tile: keep the fp32 sums */
#pragma unroll
                for (int i = 0; i < RP; i++) {
                    const uint32_t poff = (mi * SR + 4 * (p0 + i) + rr) * 256 + cc * 8;
                    const uint32_t bo = (uint32_t)((pst - a.sk_part) + poff) * 4;
                    __builtin_amdgcn_raw_buffer_store_b128(
                        __builtin_bit_cast(u32x4, floatx4{y[i][0], y[i][1], y[i][2], y[i][3]}),
                        part_rsrc, bo, 0, QW_CPOL_COHERENT);
                    __builtin_amdgcn_raw_buffer_store_b128(
                        __builtin_bit_cast(u32x4, floatx4{y[i][4], y[i][5], y[i][6], y[i][7]}),
                        part_rsrc, bo + 16, 0, QW_CPOL_COHERENT);
                }
                continue;
            }
            /* y = bf16(sum * scale + bias): the packed words are the STORE
             * epilogue's output; the other epilogues continue from y */
            uint32_t pk[RP][4];
#pragma unroll
            for (int i = 0; i < RP; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    /* sc is 1 where there is no scale: the product is exact */
                    const float t0 = y[i][2 * j] * sc[2 * j], t1 = y[i][2 * j + 1] * sc[2 * j + 1];
                    pk[i][j] = pack_bf(t0 + bias[2 * j], t1 + bias[2 * j + 1]);
                    y[i][2 * j] = lo_bf(pk[i][j]);
                    y[i][2 * j + 1] = hi_bf(pk[i][j]);
                }
            if (EPI == QW_EPI_QKNORM && qk_head) {
                /* the 16 lanes of a row hold one head, 8 elements each
                 * (lane cc: elements 8 cc..8 cc + 7), as qw_qk_norm_rope_bf16
                 * holds it: the same sum order, shuffles and roundings */
                float ss[RP];
#pragma unroll
                for (int i = 0; i < RP; i++) {
                    ss[i] = 0.0f;
#pragma unroll
                    for (int j = 0; j < 8; j++) ss[i] = fmaf(y[i][j], y[i][j], ss[i]);
                }
#pragma unroll
                for (int i = 0; i < RP; i++) ss[i] = row16_sum(ss[i]);
#pragma unroll
                for (int i = 0; i < RP; i++) {
                    const float inv = head_rms_inv(ss[i], a.eps);
#pragma unroll
                    for (int q = 0; q < 4; q++) { /* rounded to bf16 in pairs */
                        const uint32_t w = pack_bf(y[i][2 * q] * inv * nw[2 * q],
                                                   y[i][2 * q + 1] * inv * nw[2 * q + 1]);
                        y[i][2 * q] = lo_bf(w);
                        y[i][2 * q + 1] = hi_bf(w);
                    }
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float y0 = y[i][2 * q] * rc[i][q] - y[i][2 * q + 1] * rs[i][q];
                        const float y1 = y[i][2 * q] * rs[i][q] + y[i][2 * q + 1] * rc[i][q];
                        y[i][2 * q] = y0;
                        y[i][2 * q + 1] = y1;
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < RP; i++) {
                if (EPI == QW_EPI_GELU) {
#pragma unroll
                    for (int j = 0; j < 8; j++) y[i][j] = gelu_tanh_f(y[i][j]);
                } else if (EPI == QW_EPI_GATE) {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        y[i][2 * j] = lo_bf(rv[i][j]) + y[i][2 * j] * lo_bf(gv[i][j]);
                        y[i][2 * j + 1] = hi_bf(rv[i][j]) + y[i][2 * j + 1] * hi_bf(gv[i][j]);
                    }
                }
                /* non-temporal store (cache policy NT): measured 3% faster
                 * on the up projection and 8% on 8192^3 than a
                 * default-policy store */
                if (EPI != QW_EPI_STORE) {
#pragma unroll
                    for (int j = 0; j < 4; j++) pk[i][j] = pack_bf(y[i][2 * j], y[i][2 * j + 1]);
                }
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{pk[i][0], pk[i][1], pk[i][2], pk[i][3]},
                                                       out_rsrc, ooff[i], 0, QW_CPOL_NT);
            }
        }
    }
}

/* SwiGLU (EPI_SWIGLU): the wave's 128 columns are the gate rows f0..f0 + 63
 * of W, then the up rows F + f0..F + f0 + 63 (qg_wrow), so one lane finds a
 * gate and its up value 64 staged columns apart: 8 lanes per output row, 8
 * output columns (one 16-byte store) per lane, 8 rows per pass. The same
 * rounding points as the linear followed by qw_swiglu_bf16: g and u to bf16,
 * silu(g) to bf16, the product to bf16.
 *
 * Fused because the separate pass writes and re-reads the [M, 2F] linear
 * output: at M = 4119, F = 12288 the pass took 120-123 us after a 625 us
 * linear that also had twice the output to store.
 *
 * MODE 0: a finished tile; MODE 2: the last piece of a split tile, which
 * adds all pieces' sums in piece order. read_half(lr, half, v): this lane's
 * 8 sums of gate (half 0) or up (half 1) columns of staged row lr. */
template <int INT8, int NSLAB, int SR, int MODE, class SlabWriter, class HalfReader>
__device__ __forceinline__ void gemm_epilogue_swiglu(const qw_gemm_args &a, SlabWriter write_slab,
                                                     HalfReader read_half, uint32_t row0,
                                                     uint32_t f0, uint32_t lane,
                                                     const float *pld, uint32_t npart,
                                                     uint32_t own) {
#pragma clang fp contract(off)
    const bool scaled = INT8 || a.wscale != nullptr;
    const __amdgpu_buffer_rsrc_t part_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)a.sk_part, (short)0, (int)0x7FFFFFF0, 0x00020000);
    const __amdgpu_buffer_rsrc_t out_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void *)a.out, (short)0, (int)a.out_bytes, 0x00020000);
    const uint32_t F = a.n / 2, rr = lane >> 3, cc = lane & 7;
    const uint32_t col = f0 + cc * 8;
    const bool col_ok = col < F;             /* F % 8 == 0 */
    const uint32_t colc = col_ok ? col : F - 8; /* in-range column for operand loads */
    float sc[2][8], bias[2][8];
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int j = 0; j < 8; j++) sc[h][j] = 1.0f, bias[h][j] = 0.0f;
        if (scaled) {
            const floatx4 s0 = *(const floatx4 *)(a.wscale + h * F + colc);
            const floatx4 s1 = *(const floatx4 *)(a.wscale + h * F + colc + 4);
#pragma unroll
            for (int j = 0; j < 4; j++) sc[h][j] = s0[j], sc[h][4 + j] = s1[j];
        }
        if (a.bias) {
            const u32x4 bb = *(const u32x4 *)(a.bias + h * F + colc);
#pragma unroll
            for (int j = 0; j < 4; j++)
                bias[h][2 * j] = lo_bf(bb[j]), bias[h][2 * j + 1] = hi_bf(bb[j]);
        }
    }
#pragma unroll
    for (int mi = 0; mi < NSLAB; mi++) {
        write_slab(mi);
#pragma unroll
        for (int p = 0; p < SR / 8; p++) {
            const uint32_t lr = 8 * p + rr, row = row0 + mi * SR + lr;
            const uint32_t ooff = col_ok && row < a.m ? (row * a.ldc + col) * 2 : 0x80000000u;
            float y[2][8];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (MODE == 0) {
                    read_half(lr, h, y[h]);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; j++) y[h][j] = 0.0f;
                    for (uint32_t pc = 0; pc < npart; pc++) {
                        float v[8];
                        if (pc == own) {
                            read_half(lr, h, v);
                        } else {
                            const uint32_t poff = (mi * SR + lr) * 256 + h * 64 + cc * 8;
                            const uint32_t bo =
                                (uint32_t)((pld - a.sk_part) + pc * QW_SPLIT_PART + poff) * 4;
                            const floatx4 q0 = __builtin_bit_cast(
                                floatx4, __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, bo, 0,
                                                                               QW_CPOL_COHERENT));
                            const floatx4 q1 = __builtin_bit_cast(
                                floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                             part_rsrc, bo + 16, 0, QW_CPOL_COHERENT));
#pragma unroll
                            for (int j = 0; j < 4; j++) v[j] = q0[j], v[4 + j] = q1[j];
                        }
#pragma unroll
                        for (int j = 0; j < 8; j++) y[h][j] += v[j];
                    }
                }
#pragma unroll
                for (int j = 0; j < 8; j += 2) {
                    const float t0 = y[h][j] * sc[h][j], t1 = y[h][j + 1] * sc[h][j + 1];
                    const uint32_t w = pack_bf(t0 + bias[h][j], t1 + bias[h][j + 1]);
                    y[h][j] = lo_bf(w);
                    y[h][j + 1] = hi_bf(w);
                }
            }
            uint32_t pk[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t g =
                    pack_bf(silu_epi_f(y[0][2 * j]), silu_epi_f(y[0][2 * j + 1]));
                pk[j] = pack_bf(lo_bf(g) * y[1][2 * j], hi_bf(g) * y[1][2 * j + 1]);
            }
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{pk[0], pk[1], pk[2], pk[3]}, out_rsrc,
                                                   ooff, 0, QW_CPOL_NT);
        }
    }
}

template <int EPI, int INT8, int NSLAB, int SR, int RP, class SlabWriter, class SlabReader>
__device__ __forceinline__ void gemm_epilogue_lds(const qw_gemm_args &a, SlabWriter write_slab,
                                                  SlabReader read_row, uint32_t row0,
                                                  uint32_t col0, uint32_t lane, float *pst,
                                                  const float *pld, uint32_t npart,
                                                  uint32_t own) {
    if (pst)
        gemm_epilogue_mode<EPI, INT8, NSLAB, SR, RP, 1>(a, write_slab, read_row, row0, col0, lane, pst,
                                                     pld, npart, own);
    else if (pld)
        gemm_epilogue_mode<EPI, INT8, NSLAB, SR, RP, 2>(a, write_slab, read_row, row0, col0, lane, pst,
                                                     pld, npart, own);
    else
        gemm_epilogue_mode<EPI, INT8, NSLAB, SR, RP, 0>(a, write_slab, read_row, row0, col0, lane, pst,
                                                     pld, npart, own);
}

/* buffer_load_dwordx4 ... lds from inline assembly: M0 = LDS address,
 * lane l writes M0 + 16 l */
__device__ __forceinline__ void gemm_dma16(u32x4 rsrc, uint32_t lds, uint32_t voff, uint32_t soff) {
    /* s_nop 0: an LDS-direct load reads M0 at least one wait state after
     * an SALU write of it (gfx9); inside the asm the compiler cannot add it */
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                 : "m0");
}
__device__ __forceinline__ u32x4 gemm_rs4(const void *p, uint32_t bytes) {
    const uint64_t b = (uint64_t)p;
    return u32x4{(uint32_t)b, (uint32_t)(b >> 32) & 0xffffu, bytes, 0x00020000u};
}
