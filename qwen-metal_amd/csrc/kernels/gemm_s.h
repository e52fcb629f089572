/* Narrow tiles for linears of few rows (bf16 W): 64 MB rows x 128 columns
 * per workgroup of 4 waves stacked along the rows, each wave 16 MB rows x
 * 128 columns (MB x 8 v_mfma_f32_16x16x32_bf16 blocks), so a launch that
 * has few 256 x 256 tiles still has a workgroup for every CU.
 *
 * What bounds them is the way from L2 and HBM into LDS: a slice of 64 k
 * moves 8 MB + 16 KB for 16 MB MFMAs per wave, and the time from a load's
 * issue to its landing (1.2-1.5 us, measured as the time of a slice with one
 * slice ahead) is several slices long. So the K-slices go through a ring of
 * NST stages, NST - 1 of them in flight; the rest is the wide kernels'
 * pipeline (gemm_q.h): direct loads, XOR-swizzled chunks, and each slice's
 * second sub-step held back under the next slice's loads and reads.
 *
 * Where the tiles are fewer than the CUs, a tile is cut into k-ranges. A
 * piece stores its accumulators as they sit in the registers (1 KB per
 * instruction, no staging); the last piece in adds all pieces' in piece
 * order, again in the registers, and runs the plain epilogue. */
#pragma once

#define QS_W_BYTES (128 * 128) /* W stage: 128 rows x 64 bf16 */

struct QsCtx {
    u32x4 a_rs4, w_rs4;
    uint32_t a_dvoff[8], w_dvoff[4];
    uint32_t a_dst, w_dst;   /* this wave's share of a stage */
    uint32_t a_frag, w_frag; /* fragment row base (rows + lane % 16) in bytes */
    uint32_t ch[2];          /* swizzled 16-byte chunk of sub-step 0 / 1 */
};

/* how many of n fragment reads are issued before MFMA i of m: all of them
 * under the first half, so the last ones have landed by the sub-step's end
 * (4-5% of a linear at MB = 2 and 4 against reads spread evenly) */
constexpr int qs_at(int i, int n, int m) { return 2 * i * n / m < n ? 2 * i * n / m : n; }
/* One 64-k slice, multiplied from stage `cur` while the slice at byte offset
 * ko of its rows streams into stage `nxt`; off: 0, or 2^31 for a slice past
 * the last, whose loads then lie past the ends of their buffers. */
template <bool PREV, int MB>
__device__ __forceinline__ void qs_slice(const QsCtx &c, floatx4 (&acc)[MB][8], bf16x8 (&pa)[MB],
                                         bf16x8 (&pw)[8], const unsigned char *cur, uint32_t nxt,
                                         uint32_t ko, uint32_t off) {
    constexpr int AB = MB * 64 * 128, NM = 8 * MB, ND = 2 * MB + 4, NR = MB + 8;
    auto dma = [&](int j) __attribute__((always_inline)) {
        if (j < 4)
            gemm_dma16(c.w_rs4, nxt + AB + c.w_dst + j * 1024, c.w_dvoff[j] | off, ko);
        else
            gemm_dma16(c.a_rs4, nxt + c.a_dst + (j - 4) * 1024, c.a_dvoff[j - 4] | off, ko);
    };
    auto rd = [&](int j, uint32_t ch, bf16x8 (&af)[MB], bf16x8 (&bw)[8])
        __attribute__((always_inline)) {
        if (j == 0)
            bw[0] = *(const bf16x8 *)(cur + AB + c.w_frag + ch);
        else if (j <= MB)
            af[j - 1] = *(const bf16x8 *)(cur + c.a_frag + (j - 1) * 2048 + ch);
        else
            bw[j - MB] = *(const bf16x8 *)(cur + AB + c.w_frag + (j - MB) * 2048 + ch);
    };
    bf16x8 af[MB], bw[8], af1[MB], bw1[8];
    if (PREV) {
        asm volatile("s_nop 1" ::"v"(pw[0]), "v"(pw[1]), "v"(pw[2]), "v"(pw[3]), "v"(pw[4]),
                     "v"(pw[5]), "v"(pw[6]), "v"(pw[7]));
#pragma unroll
        for (int i = 0; i < MB; i++) asm volatile("s_nop 1" ::"v"(pa[i]));
#pragma unroll
        for (int i = 0; i < NM; i++) {
            QG_MFMA(acc[i % MB][i / MB], pw[i / MB], pa[i % MB]);
#pragma unroll
            for (int j = qs_at(i, NR, NM); j < qs_at(i + 1, NR, NM); j++)
                rd(j, c.ch[0], af, bw);
#pragma unroll
            for (int j = i * ND / NM; j < (i + 1) * ND / NM; j++) dma(j);
        }
    } else {
#pragma unroll
        for (int j = 0; j < ND; j++) dma(j);
#pragma unroll
        for (int j = 0; j < NR; j++) rd(j, c.ch[0], af, bw);
    }
#pragma unroll
    for (int i = 0; i < NM; i++) {
        if (PREV)
            QG_MFMA(acc[i % MB][i / MB], bw[i / MB], af[i % MB]);
        else
            QG_MFMA0(acc[i % MB][i / MB], bw[i / MB], af[i % MB]);
#pragma unroll
        for (int j = qs_at(i, NR, NM); j < qs_at(i + 1, NR, NM); j++)
            rd(j, c.ch[1], af1, bw1);
    }
#pragma unroll
    for (int i = 0; i < MB; i++) pa[i] = af1[i];
#pragma unroll
    for (int i = 0; i < 8; i++) pw[i] = bw1[i];
}

/* Sums of the tile at rows m0, W rows n0 over k-steps [kb, ke) into acc;
 * ends with the LDS free. Slices past ke - 1 are asked for past the ends of
 * their buffers (in the vector offset, which the buffer's bounds check
 * covers), where a load moves nothing, so that every slice issues the same
 * number of loads and one vmcnt serves every wait. */
template <int MB, int NST, bool GLU>
__device__ __forceinline__ void qs_mainloop(const qw_gemm_args &a, unsigned char *lds, uint32_t m0,
                                            uint32_t n0, uint32_t kb, uint32_t ke,
                                            floatx4 (&acc)[MB][8]) {
    constexpr uint32_t AB = MB * 64 * 128, STAGE = AB + QS_W_BYTES;
    constexpr int ND = 2 * MB + 4, PF = NST - 1;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    QsCtx c;
    const uint32_t lrow = lane >> 3, lp = lane & 7;
#pragma unroll
    for (int j = 0; j < 2 * MB; j++) {
        const uint32_t r = wave * (16 * MB) + j * 8 + lrow;
        c.a_dvoff[j] = (min(m0 + r, a.m - 1) * a.lda + (lp ^ ((r >> 1) & 7u)) * 8) * 2;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t r = wave * 32 + j * 8 + lrow;
        c.w_dvoff[j] = (qg_wrow<GLU>(a, n0, r) * a.k + (lp ^ ((r >> 1) & 7u)) * 8) * 2;
    }
    c.a_rs4 = gemm_rs4(a.a, a.a_bytes);
    c.w_rs4 = gemm_rs4(a.w, a.w_bytes);
    c.a_dst = wave * (16 * MB) * 128;
    c.w_dst = wave * 32 * 128;
    const uint32_t l16 = lane & 15, h = lane >> 4, swz = (l16 >> 1) & 7u;
    c.a_frag = (wave * (16 * MB) + l16) * 128;
    c.w_frag = l16 * 128;
    c.ch[0] = ((0 + h) ^ swz) << 4;
    c.ch[1] = ((4 + h) ^ swz) << 4;
    const uint32_t base =
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
    auto ko = [&](uint32_t k) __attribute__((always_inline)) { return k < ke ? k * (GBK * 2) : 0u; };
    auto off = [&](uint32_t k) __attribute__((always_inline)) { return k < ke ? 0u : 0x80000000u; };
#pragma unroll
    for (int p = 0; p < PF; p++) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            gemm_dma16(c.w_rs4, base + p * STAGE + AB + c.w_dst + j * 1024, c.w_dvoff[j] | off(kb + p),
                       ko(kb + p));
#pragma unroll
        for (int j = 0; j < 2 * MB; j++)
            gemm_dma16(c.a_rs4, base + p * STAGE + c.a_dst + j * 1024, c.a_dvoff[j] | off(kb + p),
                       ko(kb + p));
    }
    /* all but the newest PF - 1 slices' loads landed, in every wave */
    auto landed = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((PF - 1) * ND) : "memory");
    };
    bf16x8 pa[MB], pw[8];
    landed();
    qs_slice<false, MB>(c, acc, pa, pw, lds, base + PF * STAGE, ko(kb + PF), off(kb + PF));
    uint32_t kt = kb + 1;
    if constexpr (MB >= 3) {
        /* NST slices a turn, so that the stages are constants */
        while (kt < ke) {
#pragma unroll
            for (int st = 1; st <= NST; st++) {
                if (kt >= ke) break;
                landed();
                qs_slice<true, MB>(c, acc, pa, pw, lds + (st % NST) * STAGE,
                                   base + ((st + PF) % NST) * STAGE, ko(kt + PF), off(kt + PF));
                kt++;
            }
        }
    } else {
        uint32_t cur = STAGE, nxt = 0; /* stages of slices kt and kt + PF */
        for (; kt < ke; kt++) {
            landed();
            qs_slice<true, MB>(c, acc, pa, pw, lds + cur, base + nxt, ko(kt + PF), off(kt + PF));
            nxt = cur;
            cur = cur + STAGE == NST * STAGE ? 0u : cur + STAGE;
        }
    }
    asm volatile("s_nop 1" ::"v"(pw[0]), "v"(pw[1]), "v"(pw[2]), "v"(pw[3]), "v"(pw[4]),
                 "v"(pw[5]), "v"(pw[6]), "v"(pw[7]));
#pragma unroll
    for (int i = 0; i < MB; i++) asm volatile("s_nop 1" ::"v"(pa[i]));
#pragma unroll
    for (int i = 0; i < 8 * MB; i++) QG_MFMA(acc[i % MB][i / MB], pw[i / MB], pa[i % MB]);
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
    /* no read of an accumulator moves above the wait for the last MFMAs */
#pragma unroll
    for (int i = 0; i < 8 * MB; i++) asm volatile("" : "+a"(acc[i % MB][i / MB]));
    QW_SLICE_END(); /* the last stages' loads land before the epilogue uses the LDS */
}

template <int EPI, int MB, int NST>
__device__ __forceinline__ void qs_impl(const qw_gemm_args &a, unsigned char *lds) {
    constexpr bool GLU = EPI == QW_EPI_SWIGLU;
    const uint32_t KT = a.k / GBK, R = a.tiles_m * a.tiles_n, S = a.split, np = R * S;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    /* ids are dealt round-robin to the 8 XCDs: each XCD takes one contiguous
     * range of the pieces (numbered k-range-major, tile rows first), so the
     * tile rows that share a W panel read it through one L2 */
    const uint32_t q = gemm_xcd_range(blockIdx.x, np);
    const uint32_t piece = q / R, r = q % R;
    const uint32_t kb = piece * KT / S, ke = (piece + 1) * KT / S;
    uint32_t tm, tn;
    gemm_tile_at(a, r, tm, tn);
    const uint32_t m0 = a.m_base + tm * (64 * MB), n0 = tn * 128;
    floatx4 acc[MB][8];
    qs_mainloop<MB, NST, GLU>(a, lds, m0, n0, kb, ke, acc);
    if (S > 1) {
        const __amdgpu_buffer_rsrc_t part = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(a.sk_part + (size_t)r * S * (MB * 64 * 128)), (short)0,
            (int)(S * (MB * 64 * 128 * 4)), 0x00020000);
        /* block (mb, nb) of this wave in piece pc: 1 KB */
        auto at = [&](uint32_t pc, int mb, int nb) __attribute__((always_inline)) {
            return pc * (MB * 64 * 128 * 4) + ((wave * MB + mb) * 8 + nb) * 1024 + lane * 16;
        };
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < 8; nb++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[mb][nb]), part,
                                                       at(piece, mb, nb), 0, QW_CPOL_COHERENT);
        uint32_t &ticket = *(uint32_t *)lds;
        __builtin_amdgcn_s_waitcnt(0x0F70); /* vmcnt(0): the partial's stores are done */
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        if (threadIdx.x == 0)
            ticket = __hip_atomic_fetch_add(a.sk_flag + r, 1u, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (ticket != S - 1) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        __syncthreads(); /* the ticket is read before the staging overwrites it */
        floatx4 own[MB][8];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < 8; nb++) own[mb][nb] = acc[mb][nb];
        for (uint32_t pc = 0; pc < S; pc++) {
            floatx4 v[MB][8];
            if (pc == piece) {
#pragma unroll
                for (int mb = 0; mb < MB; mb++)
#pragma unroll
                    for (int nb = 0; nb < 8; nb++) v[mb][nb] = own[mb][nb];
            } else {
#pragma unroll
                for (int mb = 0; mb < MB; mb++)
#pragma unroll
                    for (int nb = 0; nb < 8; nb++)
                        v[mb][nb] = __builtin_bit_cast(
                            floatx4, __builtin_amdgcn_raw_buffer_load_b128(part, at(pc, mb, nb), 0,
                                                                           QW_CPOL_COHERENT));
            }
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int nb = 0; nb < 8; nb++)
                    acc[mb][nb] = pc ? acc[mb][nb] + v[mb][nb] : v[mb][nb];
        }
        if (threadIdx.x == 0)
            __hip_atomic_store(a.sk_flag + r, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    qg_finish_wave<EPI, 0, MB>(a, (float *)(lds + wave * QG_REGION), m0 + wave * (16 * MB), n0,
                               n0 / 2, 0, acc);
}

/* stages of each tile height: as many as hide the loads (a fifth or sixth
 * stage of the lower tiles measured no faster) */
#define QS_NST(MB) ((MB) <= 2 ? 4 : 3)
#define QS_ENTRY(name, EPI, MB)                                                                \
    QW_KERNEL void __launch_bounds__(256, 1) name(qw_gemm_args a) {                            \
        __shared__ __attribute__((aligned(16))) unsigned char                                  \
            smem[QS_NST(MB) * (MB * 64 * 128 + QS_W_BYTES)];                                   \
        static_assert(sizeof(smem) >= 4 * QG_REGION, "staging");                               \
        qs_impl<EPI, MB, QS_NST(MB)>(a, smem);                                                 \
    }
#define QS_ENTRIES(MB)                                                                         \
    QS_ENTRY(qw_gemm_bf16_store_n##MB, QW_EPI_STORE, MB)                                       \
    QS_ENTRY(qw_gemm_bf16_gelu_n##MB, QW_EPI_GELU, MB)                                         \
    QS_ENTRY(qw_gemm_bf16_gate_n##MB, QW_EPI_GATE, MB)                                         \
    QS_ENTRY(qw_gemm_bf16_qkn_n##MB, QW_EPI_QKNORM, MB)                                        \
    QS_ENTRY(qw_gemm_bf16_swiglu_n##MB, QW_EPI_SWIGLU, MB)
QS_ENTRIES(1)
QS_ENTRIES(2)
QS_ENTRIES(3)
QS_ENTRIES(4)
