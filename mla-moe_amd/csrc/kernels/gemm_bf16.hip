/* gemm_bf16.hip -- dense y = x . W^T on v_mfma_f32_16x16x32_bf16 (matmul of
 * src/run.c:29-37 batched over T rows).
 *
 * W is bf16 row-major [d_out, n_in] exactly as the reference stores it: a B
 * operand fragment (16 output columns x 32 inputs, lane l holding column
 * l % 16 and inputs 8*(l/16) .. +7) is 16 contiguous bytes of one weight row
 * per lane, so B stages into LDS by direct global -> LDS loads in operand
 * order.  x is fp32: mm_cvt_bf16 first writes it as bf16 rows, either
 * truncated (the config that casts activations on the input side,
 * include/tensor.h:16-20) or split into a bf16 hi/lo pair (two MFMAs, ~2^-17
 * relative) so the result tracks the fp32 reference; A then stages exactly
 * like B.
 *
 * See mm_gemm_bf16 for the tile and the two kinds of waves.
 */
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

#define GB_BM MM_GB_BM
#define GB_BK 64
#define GB_COPY (128 * 128)             /* A of one stage: 128 rows x 128 B */

/* x -> bf16 rows of stride kp (zeros past n_in), 8 values per thread:
 * truncation (the reference's cast, include/tensor.h:16-20) or the RNE
 * hi/lo split. */
extern "C" __global__ __launch_bounds__(256) void mm_cvt_bf16(mm_cvt_bf16_args a) {
    const size_t i8 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;   /* 8-value chunk */
    const int cpr = a.kp / 8;
    if (i8 >= (size_t)a.T * cpr) return;
    const int t = (int)(i8 / cpr), k = (int)(i8 % cpr) * 8;
    u16x8 hi = {0, 0, 0, 0, 0, 0, 0, 0}, lo = {0, 0, 0, 0, 0, 0, 0, 0};
    if (k < a.n_in) {   /* n_in is a multiple of 8 */
        const float *p = a.x + (size_t)t * a.n_in + k;
        const f32x4 x0 = *(const f32x4 *)p, x1 = *(const f32x4 *)(p + 4);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float v = e < 4 ? x0[e] : x1[e - 4];
            if (a.split) {
                const uint16_t h16 = rne16(v);
                hi[e] = h16;
                lo[e] = rne16(v - bf16_f32(h16));
            } else {
                hi[e] = (uint16_t)(__float_as_uint(v) >> 16);
            }
        }
    }
    *(u16x8 *)(a.xh + i8 * 8) = hi;
    if (a.split) *(u16x8 *)(a.xl + i8 * 8) = lo;
}

/* Block tile 128 rows x BN columns (128, 64 or 32), K chunks of 64, both
 * operands global -> LDS by direct loads into a ring of NS stages [A hi][A lo
 * (split mode)][B].  Eight waves, two per SIMD: four multiply (a 2 x 2 grid,
 * 64 x BN / 2 each), four only load, NS - 1 chunks ahead.  A multiplying
 * wave's instruction stream then holds nothing but LDS reads and MFMAs, the
 * reads of the next 32-wide K step (the next chunk's first included: the
 * barrier comes before a chunk's last MFMAs) between the MFMAs of the
 * current one.  With four waves doing both in turn, the loads' issue, the
 * reads' round trip and the MFMAs of a chunk added up (split mode, 2,048
 * rows: 2,048 x 2,048 49 us, 2,048 x 10,944 209, 10,944 x 2,048 270; now 32,
 * 153 and 178: 1,030-1,200 TFLOP/s of MFMAs, what a library product of 8,192
 * cubed reaches here; 512 truncated rows through the four projections 58 us
 * -> 53).  Its parts alone, 2,048 x 10,944: the loads 108 us (48 KB per chunk
 * and CU: 20 TB/s out of L2), the MFMAs 100, both 153: they share the LDS.
 *
 * GB_FLUSH: the accumulators are added to a second set every 512 values of
 * K (2,048 values, truncated input: error against 64 bits 2.7e-7 -> 1.3e-7).
 *
 * A load instruction moves 8 rows x 128 B (whole cache lines; half-line
 * accesses measured ~2.6x slower): lane l carries row 8 i + l / 8 and stores
 * at position l % 8 of that row's 128 B the 16 B piece (l % 8) ^ s(row), s(R)
 * = (R / 2) % 8.  The XOR swizzle makes the operand reads (16 rows, one piece
 * each) conflict-free.  Rows past T and columns past d_out, and weight pieces
 * past n_in, are out of the buffers' range: nothing is read, zeros staged.
 * Offsets within a tile's rows are 32 bits: where 128 rows of n_in values pass
 * 4 GB (2^24 values) the tile takes fewer of them, down to one. */
__device__ __forceinline__ int gb_swz(int R) { return (R >> 1) & 7; }
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
#define GB_OOB 0xFFFFFFF0u
#define GB_FLUSH 8                /* chunks summed in one accumulator (512 values of K) */

/* Waits until at most min(n, N) chunks of LPW loads are out (n < 0: none): a
 * chunk has landed when only those after it are, of which few follow near K's
 * end.  (With loads of the last chunk again in their place, so that the count
 * holds, one chunk of K took seven: 64 x 64, 400 truncated rows 7.2 us, 6.8 now,
 * 1,328 x 152, 640 rows 8.4 and 8.0.) */
template <int LPW, int N>
__device__ __forceinline__ void gb_wait(int n) {
    if constexpr (N > 0) {
        if (n < N) return gb_wait<LPW, N - 1>(n);
    }
    VMCNT_WAIT(LPW * N);
}

template <bool HL, int BN>
__device__ __forceinline__ void gemm_block(const mm_gemm_bf16_args &a, uint8_t *lds) {
    constexpr int NP = HL ? 2 : 1;                 /* A planes: hi (and lo) */
    constexpr int BOFF = NP * GB_COPY;
    constexpr int SB = MM_GB_STAGE(HL, BN);
    constexpr int NS = MM_GB_NS(HL, BN);
    constexpr int LPW = 4 * NP + BN / 32;          /* loads per loading wave per chunk */
    static_assert(SB == BOFF + BN * 128 && LPW * (NS - 2) < 64, "ring");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    /* 1-D grid: blocks are dealt to the 8 XCDs round robin (block b -> XCD
     * b % 8).  The XCDs split the tile grid into xr x 8 / xr rectangles, so
     * that an XCD's L2 takes in 1 / xr of x and xr / 8 of the weights (the host
     * chooses xr).  Column blocks from nb0 on are the second matrix's. */
    const int nb1 = a.w1 ? (a.d_out1 + a.cols - 1) / a.cols : 0;
    const int nbx = a.nb0 + nb1, nby = (a.T + a.rows - 1) / a.rows;
    const int xcd = blockIdx.x % 8, loc = blockIdx.x / 8, xc = 8 / a.xr;
    const int pr = (nby + a.xr - 1) / a.xr, pc = (nbx + xc - 1) / xc;
    const int rb = xcd / xc * pr + loc % pr;
    int cb = xcd % xc * pc + loc / pr;
    if (rb >= nby || loc % pr >= pr || loc / pr >= pc || cb >= nbx) return;
    const bool second = cb >= a.nb0;
    if (second) cb -= a.nb0;
    const uint16_t *w = second ? a.w1 : a.w;
    const int d_out = second ? a.d_out1 : a.d_out;
    const int m0 = rb * a.rows, n0 = cb * a.cols;
    const int mrows = min(a.T - m0, a.rows), ncols = min(d_out - n0, a.cols);
    const int K = a.n_in, KB = a.kp / GB_BK;
    const uint32_t lds0 = lds_addr(lds);

    if (wave >= 4) {   /* a loading wave: a quarter of each plane and of the weights */
        const int lw = wave - 4;
        rsrc_t rs[NP + 1];
#pragma unroll
        for (int q = 0; q < NP; q++)
            rs[q] = raw_rsrc((q ? a.xl : a.xh) + (size_t)m0 * a.kp, (uint32_t)mrows * (uint32_t)a.kp * 2u);
        rs[NP] = raw_rsrc(w + (size_t)n0 * K, (uint32_t)ncols * (uint32_t)K * 2u);
        constexpr int WL = BN / 32;                /* weight loads per wave: 8 rows each */
        uint32_t ao[4], wo[WL];
        int wk[WL];                                /* first K value of the lane's weight piece */
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int R = 8 * (4 * lw + u) + (lane >> 3), kq = 8 * ((lane & 7) ^ gb_swz(R));
            ao[u] = R < mrows ? ((uint32_t)R * (uint32_t)a.kp + (uint32_t)kq) * 2u : GB_OOB;
        }
#pragma unroll
        for (int u = 0; u < WL; u++) {
            const int R = 8 * (WL * lw + u) + (lane >> 3);
            wk[u] = 8 * ((lane & 7) ^ gb_swz(R));
            wo[u] = R < ncols ? ((uint32_t)R * (uint32_t)K + (uint32_t)wk[u]) * 2u : GB_OOB;
        }
        auto issue = [&](int kb, int st) {
            const int k0 = kb * GB_BK;
            const uint32_t sb = lds0 + (uint32_t)(st * SB);
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int q = 0; q < NP; q++)
                    lds_dma16_buf(ao[u] != GB_OOB ? ao[u] + 2u * (uint32_t)k0 : GB_OOB, rs[q],
                                  sb + (uint32_t)(q * GB_COPY + (4 * lw + u) * 1024));
#pragma unroll
            for (int u = 0; u < WL; u++)
                lds_dma16_buf(wo[u] != GB_OOB && k0 + wk[u] < K ? wo[u] + 2u * (uint32_t)k0 : GB_OOB, rs[NP],
                              sb + (uint32_t)(BOFF + (WL * lw + u) * 1024));
        };
#pragma unroll 1
        for (int s = 0; s < min(NS - 1, KB); s++) issue(s, s);
        gb_wait<LPW, NS - 2>(KB - 1);              /* chunk 0 */
        __builtin_amdgcn_s_barrier();
        int st = NS - 1, kb = 0;
        for (; kb + NS - 1 < KB; kb++) {           /* one barrier per chunk */
            issue(kb + NS - 1, st);                /* the slot of chunk kb - 1 */
            st = st + 1 == NS ? 0 : st + 1;
            VMCNT_WAIT(LPW * (NS - 2));            /* chunk kb + 1 */
            __builtin_amdgcn_s_barrier();
        }
        for (; kb < KB; kb++) {
            gb_wait<LPW, NS - 2>(KB - 2 - kb);
            __builtin_amdgcn_s_barrier();
        }
        VMCNT_WAIT(0);
        if (BN < 64) __builtin_amdgcn_s_barrier();   /* before the multiplying waves' exchange */
        return;
    }

    /* v_mfma_f32_32x32x16_bf16: operand lane l holds row (column) l % 32, K
     * values 8 (l / 32) .. + 7 of a 16-wide step.  Row tile t (column tile j),
     * step s: row 32 t + l % 32, piece 2 s + l / 32.  BN = 32: the waves of a
     * row share its one column tile and split K's steps between them. */
    constexpr int WT = BN >= 64 ? BN / 64 : 1;     /* 32-column tiles per wave */
    constexpr int KH = BN >= 64 ? 1 : 2;           /* waves splitting a chunk's K */
    constexpr int KS = 4 / KH;                     /* 16-wide steps per wave per chunk */
    typedef const __attribute__((address_space(3))) i32x4 *lds_cp;
    const int wm = wave >> 1, wn = wave & 1, c32 = lane & 31, hi = lane >> 5;
    uint32_t rd[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) rd[s] = c32 * 128 + 16 * ((2 * (KS * (KH > 1 ? wn : 0) + s) + hi) ^ gb_swz(c32));
    const int cw = KH > 1 ? 0 : wn * (BN / 2);     /* the wave's first column */
    i32x4 x[2][2][NP], wv[2][WT];
    auto read = [&](int st, int s) {
        const uint32_t sa = lds0 + (uint32_t)(st * SB) + rd[s] + wm * 64 * 128;
        const uint32_t sw = lds0 + (uint32_t)(st * SB) + BOFF + rd[s] + cw * 128;
#pragma unroll
        for (int j = 0; j < WT; j++) wv[s & 1][j] = *(lds_cp)(sw + j * 4096);
#pragma unroll
        for (int q = 0; q < NP; q++)
#pragma unroll
            for (int t = 0; t < 2; t++) x[s & 1][t][q] = *(lds_cp)(sa + q * GB_COPY + t * 4096);
    };
    f32x16 acc[2][WT], sum[2][WT];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < WT; j++) acc[t][j] = sum[t][j] = (f32x16){};
    auto mfma = [&](int s) {
#pragma unroll
        for (int q = 0; q < NP; q++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < WT; j++)
                    acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wv[s & 1][j]),
                                                                        __builtin_bit_cast(bf16x8, x[s & 1][t][q]),
                                                                        acc[t][j], 0, 0, 0);
        /* the reads between the MFMAs */
        constexpr int RD = 2 * NP + WT, MF = 2 * NP * WT, PER = MF / RD > 0 ? MF / RD : 1;
#pragma unroll
        for (int i = 0; i < RD; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
    };
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    int st = 0;
    for (int kb = 0; kb < KB; kb++) {
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (s + 1 < KS) {
                read(st, s + 1);
            } else {
                /* this chunk's reads are done, so its slot may be refilled
                 * after the barrier, which also shows every loading wave's
                 * part of the next chunk */
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                st = st + 1 == NS ? 0 : st + 1;
                read(st, 0);
            }
            mfma(s);
        }
        if (kb % GB_FLUSH == GB_FLUSH - 1) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < WT; j++) {
                    sum[t][j] += acc[t][j];
                    acc[t][j] = (f32x16){};
                }
        }
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < WT; j++) sum[t][j] += acc[t][j];
    if (KH > 1) {
        /* the odd wave's sums to the even one through the ring's LDS: free
         * after a barrier (every load landed, every read done) */
        typedef __attribute__((address_space(3))) float lds_f;
        lds_f *red = (lds_f *)(lds0 + (uint32_t)(wm * 2 * 16 * MM_WAVE * 4 + lane * 4));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (wn == 1) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) red[(16 * t + i) * MM_WAVE] = sum[t][0][i];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (wn == 1) return;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) sum[t][0][i] += red[(16 * t + i) * MM_WAVE];
    }

    /* lane l holds row l % 32 and, in registers 4 g + i, columns 8 g + 4 (l /
     * 32) + i of each 32 x 32 tile (the weights are the first operand).  With
     * accumulate, the wave's old outputs are all loaded (clamped addresses,
     * unconditionally) before any is added, four at a time in a tile of whole
     * columns (2,048 rows, accumulated: 64 x 64 7.9 us, 4096 x 512 38; one value
     * at a time, a row tile after the other, 9.3 and 46). */
    float *y = second ? a.y1 : a.y;
    const int mend = m0 + mrows, nend = n0 + ncols;
    auto row_of = [&](int t) { return y + (size_t)min(m0 + 64 * wm + 32 * t + c32, mend - 1) * d_out; };
    if (a.accumulate && !second) {   /* uniform */
        f32x16 prev[2][WT];
        if (n0 + cw + 32 * WT <= nend) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < WT; j++)
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const f32x4 v = *(const f32x4_a4 *)(row_of(t) + n0 + cw + 32 * j + 8 * g + 4 * hi);
#pragma unroll
                        for (int i = 0; i < 4; i++) prev[t][j][4 * g + i] = v[i];
                    }
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < WT; j++)
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        prev[t][j][i] = row_of(t)[min(n0 + cw + 32 * j + 8 * (i >> 2) + 4 * hi + (i & 3), nend - 1)];
        }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int j = 0; j < WT; j++) sum[t][j] = prev[t][j] + sum[t][j];
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int m = m0 + 64 * wm + 32 * t + c32;
        float *row = row_of(t);
#pragma unroll
        for (int j = 0; j < WT; j++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int n = n0 + cw + 32 * j + 8 * g + 4 * hi;
                if (m >= mend || n >= nend) continue;
                if (n + 3 < nend) {
                    *(f32x4_a4 *)(row + n) = (f32x4){sum[t][j][4 * g], sum[t][j][4 * g + 1], sum[t][j][4 * g + 2],
                                                     sum[t][j][4 * g + 3]};
                } else {
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        if (n + i < nend) row[n + i] = sum[t][j][4 * g + i];
                }
            }
    }
}

/* 1-D grid of 8 * ceil(row blocks / xr) * ceil(column blocks / (8 / xr))
 * blocks, 512 threads, dynamic LDS: MM_GB_NS stages of MM_GB_STAGE bytes. */
extern "C" __global__ __launch_bounds__(512, 1) void mm_gemm_bf16(mm_gemm_bf16_args a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t glds[];
    if (a.split) {
        if (a.bn == 128) gemm_block<true, 128>(a, glds);
        else if (a.bn == 64) gemm_block<true, 64>(a, glds);
        else gemm_block<true, 32>(a, glds);
    } else {
        if (a.bn == 128) gemm_block<false, 128>(a, glds);
        else if (a.bn == 64) gemm_block<false, 64>(a, glds);
        else gemm_block<false, 32>(a, glds);
    }
}

/* ---- skinny-M GEMM: T <= 64 rows of x (batched decode) ------------------------
 *
 * Every weight row is read from HBM once per K split.  Block = 4 waves x
 * 16 SK_WC output columns; a wave holds C[64 tokens][16 SK_WC columns] (4
 * token groups x SK_WC column groups of v_mfma_f32_16x16x32_bf16, x as the
 * A operand -- each x fragment read from LDS feeds SK_WC MFMAs -- and W as
 * the B operand).  The
 * W fragments of the block's K range stream straight into registers, SK_D
 * 64-input chunks ahead of their MFMAs; fp32 x is loaded two chunks ahead
 * into registers and staged into LDS as bf16 (hi and lo) one 64-input chunk
 * at a time, so no separate conversion pass runs (double-buffered; rows
 * padded to 72 bf16 against bank conflicts; token rows past T read row
 * T - 1 and are not stored).  With
 * nsplit > 1 the K range is split over grid.y and mm_skinny_reduce sums the
 * partials in split order. */
/* Two forms: 64 output columns per block (one 16-column group per wave,
 * 4 chunks of W in flight), and for long outputs (the LM head) 64 *
 * MM_SKINNY_WIDE_WC columns per block (MM_SKINNY_WIDE_WC groups per wave, 2
 * chunks in flight), which stages each x chunk (64 rows x 64 inputs, fp32:
 * twice the bytes of one wave-group's weights) once for more weights.  LM
 * head at 64 rows (102400 x 2048): 154.6 -> ~136 us with 2 or 4 groups. */
#define SK_WC1 (MM_SKINNY_BN / 64)   /* 16-column groups per wave */
#define SK_D1 4                      /* chunks of W in flight per wave */
#define SK_DW 2
#define SK_ROW 72                    /* LDS row stride (bf16) of a staged x chunk */
#define SK_STAGE (2 * 64 * SK_ROW)   /* bf16 per stage: hi rows then lo rows */

template <bool SPLIT, int SK_WC, int SK_D>
__device__ __forceinline__ void skinny(const mm_gemm_skinny_args &a, uint16_t (*xs)[SK_STAGE]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    /* column block bx of matrix `seg` (the second one past nb0 blocks) */
    const bool seg = (int)blockIdx.x >= a.nb0;
    const int bx = seg ? blockIdx.x - a.nb0 : blockIdx.x;
    const int d_out = seg ? a.d_out1 : a.d_out;
    const uint16_t *wm = seg ? a.w1 : a.w;
    const int n0 = bx * (64 * SK_WC) + wave * (16 * SK_WC);
    const int kb = blockIdx.y * a.kr;
    const int nch = (min(a.n_in, kb + a.kr) - kb) / 64;    /* 64-input chunks of this split */
    const uint16_t *wrow[SK_WC];
#pragma unroll
    for (int j = 0; j < SK_WC; j++) {
        const int col = min(n0 + 16 * j + (lane & 15), d_out - 1);   /* past d_out: not stored */
        wrow[j] = wm + (size_t)col * a.n_in + kb + 8 * (lane >> 4);
    }

    /* x chunk c (fp32) -> registers, two slots: chunks are loaded two ahead
     * of their use.  Thread t holds the 16 B pieces p = t + 256 j (64 rows x
     * 16 pieces); staging converts them to bf16 -- the hi/lo pair of
     * mm_cvt_bf16 (RNE hi, RNE of the remainder) or the truncation -- and
     * writes hi rows then lo rows. */
    f32x4 xr[2][4];
    auto load_x = [&](int slot, int c) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int p = tid + 256 * j, r = p >> 4, q = p & 15;
            xr[slot][j] = *(const f32x4 *)(a.x + (size_t)min(r, a.T - 1) * a.n_in + kb + 64 * c + 4 * q);
        }
    };
    auto store_x = [&](int slot, int st) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int p = tid + 256 * j, r = p >> 4, q = p & 15;
            typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
            u16x4 hi, lo;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float v = xr[slot][j][e];
                if (SPLIT) {
                    hi[e] = rne16(v);
                    lo[e] = rne16(v - bf16_f32(hi[e]));
                } else {
                    hi[e] = (uint16_t)(__float_as_uint(v) >> 16);
                }
            }
            *(u16x4 *)&xs[st][r * SK_ROW + 4 * q] = hi;
            if (SPLIT) *(u16x4 *)&xs[st][(64 + r) * SK_ROW + 4 * q] = lo;
        }
    };
    bf16x8 wr[SK_D][SK_WC][2];
    auto load_w = [&](int slot, int c) {
        const int cc = min(c, nch - 1);                     /* past the end: reload the last */
#pragma unroll
        for (int j = 0; j < SK_WC; j++)
#pragma unroll
            for (int s = 0; s < 2; s++)
                wr[slot][j][s] = __builtin_bit_cast(bf16x8, __builtin_nontemporal_load(
                                                                (const u16x8 *)(wrow[j] + 64 * cc + 32 * s)));
    };
#pragma unroll
    for (int d = 0; d < SK_D; d++) load_w(d, d);
    load_x(0, 0);
    if (nch > 1) load_x(1, 1);
    store_x(0, 0);
    __syncthreads();

    f32x4 acc[SK_WC][4];
#pragma unroll
    for (int j = 0; j < SK_WC; j++)
#pragma unroll
        for (int g = 0; g < 4; g++) acc[j][g] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    static_assert(SK_D % 2 == 0, "the x slots alternate with the chunk parity");
    for (int c0 = 0; c0 < nch; c0 += SK_D) {
#pragma unroll
        for (int d = 0; d < SK_D; d++) {
            const int c = c0 + d;
            /* slot d & 1 held chunk c (in LDS since the last barrier): refill it with c + 2 */
            if (c + 2 < nch) load_x(d & 1, c + 2);
            if (c < nch) {
                const uint16_t *xb = xs[d & 1];
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const int ko = 32 * s + 8 * (lane >> 4);
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const int r = 16 * g + (lane & 15);
                        const bf16x8 ah = *(const bf16x8 *)&xb[r * SK_ROW + ko];
                        bf16x8 al;
                        if (SPLIT) al = *(const bf16x8 *)&xb[(64 + r) * SK_ROW + ko];
#pragma unroll
                        for (int j = 0; j < SK_WC; j++) {
                            acc[j][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, wr[d][j][s], acc[j][g], 0, 0, 0);
                            if (SPLIT)
                                acc[j][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, wr[d][j][s], acc[j][g], 0, 0, 0);
                        }
                    }
                }
            }
            load_w(d, c + SK_D);
            if (c + 1 < nch) store_x((d + 1) & 1, (d + 1) & 1);
            __syncthreads();
        }
    }
    /* C[token 16 g + 4 (l / 16) + i][column n0 + 16 j + l % 16] */
#pragma unroll
    for (int j = 0; j < SK_WC; j++) {
        const int n = n0 + 16 * j + (lane & 15);
        if (n >= d_out) continue;
        float *part = a.part + (seg ? (size_t)a.nsplit * a.T * a.d_out : 0);
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int t = 16 * g + 4 * (lane >> 4) + i;
                if (t >= a.T) continue;
                if (a.nsplit > 1 || a.part_out) {
                    part[((size_t)blockIdx.y * a.T + t) * d_out + n] = acc[j][g][i];
                } else {
                    float *y = (seg ? a.y1 : a.y) + (size_t)t * d_out + n;
                    *y = a.accumulate ? *y + acc[j][g][i] : acc[j][g][i];
                }
            }
    }
}

extern "C" __global__ __launch_bounds__(256) void mm_gemm_skinny(mm_gemm_skinny_args a) {
    __shared__ __attribute__((aligned(16))) uint16_t xs[2][SK_STAGE];
    if (a.split)
        skinny<true, SK_WC1, SK_D1>(a, xs);
    else
        skinny<false, SK_WC1, SK_D1>(a, xs);
}

extern "C" __global__ __launch_bounds__(256) void mm_gemm_skinny_wide(mm_gemm_skinny_args a) {
    __shared__ __attribute__((aligned(16))) uint16_t xs[2][SK_STAGE];
    if (a.split)
        skinny<true, MM_SKINNY_WIDE_WC, SK_DW>(a, xs);
    else
        skinny<false, MM_SKINNY_WIDE_WC, SK_DW>(a, xs);
}

/* y (+)= sum over splits s = 0 .. nsplit-1 of part[s], in that order. */
/* ---- skinny-M GEMM over pre-split x ------------------------------------------
 *
 * The mm_gemm_skinny computation (same column blocks, K splits, partials and
 * MFMA sequence per output: per 32-wide K step the hi product, then the lo
 * product) with x arriving as bf16 hi/lo planes written by its producer.
 * Both operands then go global -> LDS by direct loads into one ring of
 * HL_NS stages of a 64-wide K chunk (W: 64 rows x 128 B; x: 64 rows x 128 B
 * per plane), two chunks ahead: every load of the loop belongs to the ring,
 * so no wait for an x chunk (an L2 hit) also waits for weight loads issued
 * before it, as the register staging of fp32 x did (vector memory counts
 * complete in order; measured 0.75 us per chunk at q_proj + kv_a_proj,
 * B = 64).  Wave w owns token rows 16 w .. + 15 and the block's 64 columns
 * (4 x 16-column MFMA tiles).  LDS rows are 128 B of 8 pieces; piece p of
 * row r sits in slot p ^ swz(r) (16 consecutive rows, one piece: 16
 * distinct bank groups).  Two blocks per CU. */
#define HL_NS 3
#define HL_WB (64 * 128)                 /* W bytes per stage */
#define HL_STAGE (HL_WB + 2 * 64 * 128)  /* + the x planes: 24 KB */
#define HL_LPW 6                         /* direct loads per wave per stage: 2 of W, 4 of x */

__device__ __forceinline__ int hl_swz(int r) { return (r >> 1) & 7; }

extern "C" __global__ __launch_bounds__(256) void mm_gemm_hl(mm_gemm_hl_args a) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[HL_NS * HL_STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    /* column block bx of matrix `seg` (the second one past nb0 blocks) */
    const bool seg = (int)blockIdx.x >= a.nb0;
    const int bx = seg ? blockIdx.x - a.nb0 : blockIdx.x;
    const int d_out = seg ? a.d_out1 : a.d_out;
    const uint16_t *wm = seg ? a.w1 : a.w;
    const int n0 = bx * 64, K = a.n_in, T = a.T, q = lane & 7;
    const int kb = blockIdx.y * a.kr;
    const int nch = (min(K, kb + a.kr) - kb) / 64;      /* 64-input chunks of this split */

    /* direct loads of a chunk: W instruction 2 wave + u covers weight rows
     * (output columns) 8 (2 wave + u) .. + 7 of the block, x instruction
     * 4 wave + u plane (4 wave + u) / 8, token rows 8 ((4 wave + u) % 8) ..
     * + 7; lane l loads row + l / 8, slot q = l % 8, i.e. piece q ^ swz(row).
     * Rows past d_out or T load the last one (not stored). */
    const uint16_t *wp[2], *xp[4];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int c = 8 * (2 * wave + u) + (lane >> 3);
        wp[u] = wm + (size_t)min(n0 + c, d_out - 1) * K + kb + 8 * (q ^ hl_swz(c));
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int i = 4 * wave + u, r = 8 * (i & 7) + (lane >> 3);
        xp[u] = a.xhl + (size_t)(i >> 3) * T * K + (size_t)min(r, T - 1) * K + kb + 8 * (q ^ hl_swz(r));
    }
    auto issue = [&](int c, int st) {
        uint8_t *sb = lds + st * HL_STAGE;
#pragma unroll
        for (int u = 0; u < 2; u++) lds_dma16(wp[u] + 64 * c, sb + (2 * wave + u) * 1024);
#pragma unroll
        for (int u = 0; u < 4; u++) lds_dma16(xp[u] + 64 * c, sb + HL_WB + (4 * wave + u) * 1024);
    };
    /* operand reads (bytes within a stage), K half s: A row 16 wave + l % 16,
     * B row (column) 16 j + l % 16, piece 4 s + l / 16 */
    uint32_t ao[2], bo[2][4];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int p = 4 * s + (lane >> 4), r = 16 * wave + (lane & 15);
        ao[s] = HL_WB + r * 128 + 16 * (p ^ hl_swz(r));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int c = 16 * j + (lane & 15);
            bo[s][j] = c * 128 + 16 * (p ^ hl_swz(c));
        }
    }
    f32x4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

    const uint32_t l0 = lds_addr(lds);
    issue(0, 0);
    if (nch > 1) issue(1, 1);
    for (int c = 0; c < nch; c++) {
        /* chunk c landed (chunk c + 1's loads, issued after, may stay out);
         * the barrier shows every wave's loads of chunk c and frees the stage
         * of chunk c - 1 for chunk c + 2 */
        if (c + 1 < nch) VMCNT_WAIT(HL_LPW);
        else VMCNT_WAIT(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (c + 2 < nch) issue(c + 2, (c + 2) % HL_NS);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t sb = l0 + (uint32_t)((c % HL_NS) * HL_STAGE);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            i32x4 xa[2], wb[4];
            xa[0] = ds_read16(sb + ao[s]);
            xa[1] = ds_read16(sb + ao[s] + 64 * 128);
#pragma unroll
            for (int j = 0; j < 4; j++) wb[j] = ds_read16(sb + bo[s][j]);
            asm volatile("s_waitcnt lgkmcnt(0)"
                         : "+v"(xa[0]), "+v"(xa[1]), "+v"(wb[0]), "+v"(wb[1]), "+v"(wb[2]), "+v"(wb[3]));
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, xa[h]), __builtin_bit_cast(bf16x8, wb[j]), acc[j], 0, 0, 0);
        }
    }
    /* C[token 16 wave + 4 (l / 16) + i][column n0 + 16 j + l % 16] */
    float *part = a.part + (seg ? (size_t)a.nsplit * T * a.d_out : 0);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int n = n0 + 16 * j + (lane & 15);
        if (n >= d_out) continue;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = 16 * wave + 4 * (lane >> 4) + i;
            if (t >= T) continue;
            if (a.nsplit > 1 || a.part_out) {
                part[((size_t)blockIdx.y * T + t) * d_out + n] = acc[j][i];
            } else {
                float *y = (seg ? a.y1 : a.y) + (size_t)t * d_out + n;
                *y = a.accumulate ? *y + acc[j][i] : acc[j][i];
            }
        }
    }
}

extern "C" __global__ __launch_bounds__(256) void mm_skinny_reduce(mm_skinny_reduce_args a) {
    const size_t n0 = (size_t)a.T * a.d_out, n1 = a.y1 ? (size_t)a.T * a.d_out1 : 0;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n0 + n1;
         k += (size_t)gridDim.x * blockDim.x) {
        const bool seg = k >= n0;
        const size_t n = seg ? n1 : n0, i = seg ? k - n0 : k;
        const float *part = a.part + (seg ? (size_t)a.nsplit * n0 : 0);
        float *y = seg ? a.y1 : a.y;
        float v = part[i];
        for (int s = 1; s < a.nsplit; s++) v += part[(size_t)s * n + i];
        y[i] = a.accumulate ? y[i] + v : v;
    }
}
