/* moe_bf16_mm.h -- MoE expert FFN with bf16 weights and fp32 activations
 * for more than a few tokens: grouped GEMMs on v_mfma_f32_16x16x32_bf16.
 *
 * The GEMV stages (moe_bf16.hip, whose module
 * these kernels share) read a token's experts once per token; here
 * every touched expert's weights are read once per BM rows that chose it.
 * fp32 activations travel as three bf16 planes whose sum is exactly the fp32
 * value (split3: 8 + 8 + 8 significant bits), so every product is exact and
 * only the fp32 sums round, as in the GEMV.
 *
 *   mm_bf16_rows   routes sorted by expert: the sorted position of every
 *                  route, and x's planes gathered into that order (and in
 *                  token order for the shared expert)
 *   mm_bf16_gu     h = silu(gate . x) * (up . x) per sorted route, written as
 *                  planes again (down's operand)
 *   mm_bf16_dn     y = down . h per sorted route, fp32
 *   (then mm_i8_combine: the weighted sum over a token's routes)
 *
 * With the rows of an expert next to each other a tile's activation rows are
 * one contiguous run: no row lists inside the GEMM's load loop.
 *
 * Measured on a DeepSeek-V2-Lite layer, GEMV stages -> these kernels: 64
 * tokens 1430 -> 245 us, 515 tokens 11,440 -> 431 us.  At 64 tokens the weight
 * stream bounds them: gate/up 761 MB in 144 us (5.3 TB/s), down 381 MB in 78
 * us (4.9 TB/s); with more rows per expert LDS reads and MFMAs share the time.
 */
#pragma once
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

/* x = hi + mid + lo, each a bf16 of x's sign, exactly: truncations of 8
 * significant bits each (a rounded hi could overflow to infinity).  Where a
 * part would end the sum it is taken one step nearer to zero, so that no
 * part of a nonzero x is zero: an infinite weight then gives infinity in
 * every product, as in fp32, and not infinity + infinity * 0 (parts below
 * 2^-133, of values below 2^-117, are zero all the same).  An infinite x gives
 * infinity times whatever the weight is. */
__device__ __forceinline__ void split3(float x, uint16_t *hi, uint16_t *mid, uint16_t *lo) {
    const uint32_t u = __float_as_uint(x);
    const bool fin = (u & 0x7f800000u) != 0x7f800000u;
    auto part = [](uint32_t v) { return (v >> 16) - ((v & 0xffffu) == 0 && (v << 1) != 0 ? 1u : 0u); };
    const uint32_t h = part(u);
    const float r1 = x - __uint_as_float(h << 16);
    const uint32_t m = part(__float_as_uint(r1));
    const float r2 = r1 - __uint_as_float(m << 16);
    const uint16_t one = (uint16_t)(((u >> 16) & 0x8000u) | 0x3f80u);
    *hi = fin ? (uint16_t)h : x != x ? (uint16_t)0x7fc0u : (uint16_t)(u >> 16);
    *mid = fin ? (uint16_t)m : one;
    *lo = fin ? (uint16_t)(__float_as_uint(r2) >> 16) : one;
}

/* ---- sorted rows ------------------------------------------------------------ */

/* Block s < R (R = sum of the counts): the route at sorted position s.
 * Blocks R .. R + T - 1 (with a shared expert): token s - R.  Each block
 * finds its expert by a wave scan over the counts (64 per step). */
extern "C" __global__ __launch_bounds__(256) void mm_bf16_rows(mm_bf16_rows_args a) {
    const int s = blockIdx.x;
    __shared__ int s_rid;
    int tok = s - a.R;
    if (s < a.R) {
        if (threadIdx.x < MM_WAVE) {
            const int lane = threadIdx.x;
            int base = 0;
            for (int e0 = 0; e0 < a.E; e0 += MM_WAVE) {
                const int e = e0 + lane;
                const int n = e < a.E ? min(a.cnt[e * MM_CNT_STRIDE], a.T) : 0;
                int incl = n;
#pragma unroll
                for (int off = 1; off < MM_WAVE; off <<= 1) {
                    const int v = __shfl_up(incl, off, MM_WAVE);
                    if (lane >= off) incl += v;
                }
                const int st = base + incl - n;
                if (s >= st && s < st + n) s_rid = a.rows[(size_t)e * a.T + (s - st)];
                base += __shfl(incl, MM_WAVE - 1, MM_WAVE);
            }
            if (lane == 0 && s >= base) s_rid = -1;   /* fewer routes listed than R */
        }
        __syncthreads();
        const int rid = s_rid;
        if (rid < 0) return;
        tok = rid / a.K;
        if (threadIdx.x == 0) a.inv[rid] = s;
    }
    const size_t row = s < a.R ? (size_t)s : (size_t)(s - a.R);
    uint16_t *dst = (s < a.R ? a.xs : a.xt) + row * a.H;
    const size_t plane = (size_t)(s < a.R ? a.R : a.T) * a.H;
    const float *x = a.x + (size_t)tok * a.H;
    for (int i = 4 * threadIdx.x; i < a.H; i += 4 * blockDim.x) {
        const f32x4 v = *(const f32x4 *)(x + i);
        u16x4 h, m, l;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint16_t h16, m16, l16;
            split3(v[j], &h16, &m16, &l16);
            h[j] = h16;
            m[j] = m16;
            l[j] = l16;
        }
        *(u16x4 *)(dst + i) = h;
        *(u16x4 *)(dst + plane + i) = m;
        *(u16x4 *)(dst + 2 * plane + i) = l;
    }
}

/* ---- grouped GEMM -------------------------------------------------------------- */

/* A block tile: BM activation rows of one expert x 128 weight rows (gate/up:
 * 64 gate and the same 64 up columns; down: 128 columns), K in chunks of KB.
 * Both operands go global -> LDS by direct loads of whole 128-byte lines, in
 * two rings: weights NSW stages, activation planes NSA.  The grid is
 * persistent, one block per CU, and the rings run across tile boundaries, so
 * the weight stream does not pause at a tile's start or end.  Four waves only
 * read LDS and multiply, two load weights and two load planes: a wave's vector
 * memory operations complete in order, so a wave loading both could not wait
 * for planes (an L2 hit, needed soon) without waiting for weights issued
 * before them (from HBM, wanted as far ahead as LDS allows), nor a multiplying
 * wave load without waiting for its stores.  With the weights loaded by the
 * multiplying waves and one wave for the planes, 515 tokens took 451 us; the
 * loading waves give 446, the reads between the MFMAs 431.  LDS rows are
 * KB * 2 bytes of 16-byte pieces, piece p of row r in slot p ^ swz(r): 16
 * rows at one piece fall on distinct bank groups.  BM 16 or 32: each
 * multiplying wave owns all rows and a quarter of the weight rows; BM 64: a
 * 2 x 2 grid of waves, which reads 10 operand fragments per 24 MFMAs instead
 * of 14.  Loads past a matrix (rows past the tile's, columns past N, K pieces
 * past Kd) are out of the buffer's range: no memory is read and zeros are
 * staged.
 *
 * The operands of the next 32-wide K step are read from LDS between the
 * current step's MFMAs (plain loads, which the compiler counts), the first
 * step of the next chunk included: the wait for that chunk and the block's
 * barrier come before a chunk's last MFMAs.
 *
 * The sums of the hi planes move to a second set of registers every GRP_FLUSH
 * values of K, those of the small planes have their own: one chain of K =
 * 2048 rounds to twice the error of the GEMV's 64 short chains. */
#define GRP_NB 128                /* weight rows per tile */
#define GRP_OOB 0xFFFFFFF0u           /* past every buffer range */
#define GRP_FLUSH 256
#define GRP_MMW 4                     /* multiplying waves */
#define GRP_WLD 2                     /* weight-loading waves */
#define GRP_ALD 2                     /* plane-loading waves */
static_assert(MM_BF16_MM_THREADS == (GRP_MMW + GRP_WLD + GRP_ALD) * MM_WAVE, "threads known to the host");

template <int BM> struct shape {
    static constexpr int KB = MM_BF16_MM_KB(BM);
    static constexpr int ROWB = 2 * KB;                /* LDS bytes per row */
    static constexpr int RPI = 1024 / ROWB;            /* rows per load instruction */
    static constexpr int W_LPW = GRP_NB / RPI / GRP_WLD;       /* loads per weight-loading wave per chunk */
    static constexpr int AP = BM / RPI / GRP_ALD;      /* loads per plane-loading wave, plane and chunk */
    static constexpr int A_LPW = 3 * AP;
    static constexpr int W_BYTES = GRP_NB * ROWB, A_BYTES = 3 * BM * ROWB;
    static constexpr int NSW = MM_BF16_MM_NSW(BM), NSA = MM_BF16_MM_NSA(BM);
    static constexpr int WN = BM == 64 ? 2 : 4;        /* waves over the weight rows */
    static constexpr int TT = BM == 64 ? 2 : BM / 16;  /* 16-row tiles per wave */
    static constexpr int WT = GRP_NB / 16 / WN;            /* 16-column weight tiles per wave */
    static constexpr int KS = KB / 32;                 /* MFMA steps per chunk */
    static_assert(NSW * W_BYTES + NSA * A_BYTES == MM_BF16_MM_LDS(BM), "ring sizes known to the host");
    static_assert(W_LPW * (NSW - 2) < 64 && A_LPW * (NSA - 2) < 64 && KS % 2 == 0 && GRP_FLUSH % KB == 0, "");
    static __device__ int swz(int r) { return KB == 64 ? (r >> 1) & 7 : r & 15; }
};

/* Exclusive prefixes over the experts (16 bits: a pass has at most
 * MM_BF16_MM_T_CHUNK * 16 = 32768 rows). */
struct grp_shared {
    uint16_t gstart[MM_EMAX + 1];  /* BM-row groups */
    uint16_t rstart[MM_EMAX + 1];  /* rows */
};
static_assert(MM_BF16_MM_T_CHUNK * 16 < 65536, "row prefixes in 16 bits");

struct grp_tile {
    int si, e, slab, m0, M;        /* segment, expert, column slab, first row, the expert's rows */
    int row0;                      /* sorted position of the expert's first row */
};

template <int V> struct const_int { static constexpr int v = V; };

template <int BM, bool GU>
__device__ __forceinline__ grp_tile grp_decode(const mm_bf16_mm_args &a, const grp_shared &sh, int n0, int t) {
    constexpr int CPT = GU ? GRP_NB / 2 : GRP_NB;
    grp_tile id;
    if (t < n0) {
        const int nslab = (a.seg[0].N + CPT - 1) / CPT;
        int lo = 0, hi = a.E;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (nslab * sh.gstart[mid] <= t) lo = mid; else hi = mid;
        }
        const int ge = sh.gstart[lo + 1] - sh.gstart[lo], loc = t - nslab * sh.gstart[lo];
        id.si = 0;
        id.e = lo;
        id.slab = loc / ge;
        id.m0 = (loc % ge) * BM;
        id.M = sh.rstart[lo + 1] - sh.rstart[lo];
        id.row0 = sh.rstart[lo];
    } else {
        const int g1 = (a.T + BM - 1) / BM, loc = t - n0;
        id.si = 1;
        id.e = 0;
        id.slab = loc / g1;
        id.m0 = (loc % g1) * BM;
        id.M = a.T;
        id.row0 = 0;
    }
    id.si = __builtin_amdgcn_readfirstlane(id.si);
    id.e = __builtin_amdgcn_readfirstlane(id.e);
    id.slab = __builtin_amdgcn_readfirstlane(id.slab);
    id.m0 = __builtin_amdgcn_readfirstlane(id.m0);
    id.M = __builtin_amdgcn_readfirstlane(id.M);
    id.row0 = __builtin_amdgcn_readfirstlane(id.row0);
    return id;
}

template <int BM, bool GU>
__device__ __forceinline__ void grp_run(const mm_bf16_mm_args &a) {
    using sp = shape<BM>;
    constexpr int CPT = GU ? GRP_NB / 2 : GRP_NB;              /* output columns per tile */
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    __shared__ grp_shared sh;
    const int tid = threadIdx.x, lane = tid & (MM_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / MM_WAVE);
    const int l16 = lane & 15, g4 = lane >> 4;

    /* prefix sums of the experts' rows and row groups */
    if (tid < MM_WAVE) {
        int rb = 0, gb = 0;
        for (int e0 = 0; e0 < a.E; e0 += MM_WAVE) {
            const int e = e0 + lane;
            const int M = e < a.E ? min(a.cnt[e * MM_CNT_STRIDE], a.T) : 0;
            const int G = (M + BM - 1) / BM;
            int ri = M, gi = G;
#pragma unroll
            for (int off = 1; off < MM_WAVE; off <<= 1) {
                const int v = __shfl_up(ri, off, MM_WAVE), u = __shfl_up(gi, off, MM_WAVE);
                if (lane >= off) {
                    ri += v;
                    gi += u;
                }
            }
            if (e < a.E) {
                sh.rstart[e] = (uint16_t)(rb + ri - M);
                sh.gstart[e] = (uint16_t)(gb + gi - G);
            }
            rb += __shfl(ri, MM_WAVE - 1, MM_WAVE);
            gb += __shfl(gi, MM_WAVE - 1, MM_WAVE);
        }
        if (lane == 0) {
            sh.rstart[a.E] = (uint16_t)rb;
            sh.gstart[a.E] = (uint16_t)gb;
        }
    }
    __syncthreads();
    const int n0 = sh.gstart[a.E] * ((a.seg[0].N + CPT - 1) / CPT);
    const int n1 = a.nseg > 1 ? (a.T + BM - 1) / BM * ((a.seg[1].N + CPT - 1) / CPT) : 0;
    /* XCD x (block b runs on XCD b % 8) takes the x-th eighth of each
     * segment's tiles, its blocks neighbouring tiles at the same time: an
     * expert's row groups of one slab meet in that XCD's L2 */
    const int xcd = blockIdx.x % 8, nbx = gridDim.x / 8;
    const int lo0 = n0 * xcd / 8, len0 = n0 * (xcd + 1) / 8 - lo0;
    const int lo1 = n0 + n1 * xcd / 8, len = len0 + n0 + n1 * (xcd + 1) / 8 - lo1;
    auto tile_at = [&](int t) { return grp_decode<BM, GU>(a, sh, n0, t < len0 ? lo0 + t : lo1 + (t - len0)); };
    int ct = blockIdx.x / 8;
    if (ct >= len) return;

    /* ---- loads ----
     * a load instruction covers RPI LDS rows; lane l carries row + l / LPR,
     * slot l % LPR, i.e. K piece slot ^ swz(row).  Load u of loading wave lw
     * covers the rows from RPI (W_LPW lw + u) of the weights, or from RPI (AP
     * lw + u) of each plane. */
    constexpr int RPI = sp::RPI, LPR = MM_WAVE / RPI, KB = sp::KB;
    const uint32_t ldsw = lds_addr(lds), ldsa = ldsw + sp::NSW * sp::W_BYTES;
    auto piece = [&](int r) { return 8 * ((lane % LPR) ^ sp::swz(r)); };   /* first K value */
    int it = ct, ic = 0, inch, kd;                     /* tile and chunk of the next issue */
    /* next chunk of the ring; true when the tile has changed.  Past the last
     * tile its last chunk again, read by nobody. */
    auto advance = [&]() {
        if (++ic < inch) return false;
        if (it + nbx >= len) {
            ic = inch - 1;
            return false;
        }
        it += nbx;
        ic = 0;
        return true;
    };

    /* A loading wave's ring of NS stages, LPW loads each: NS - 1 chunks are
     * out before the first barrier, and each chunk's barrier shows that the
     * next one has landed (only those of the NS - 2 chunks after it are out)
     * and that every read of the chunk is done, whose slot the issues after
     * the barrier take. */
    auto load_ring = [&](auto ns, auto lpw, auto &issue) {
        constexpr int NS = decltype(ns)::v, OUT = decltype(lpw)::v * (NS - 2);
#pragma unroll 1
        for (int s = 0; s < NS - 1; s++) issue(s);
        VMCNT_WAIT(OUT);
        __builtin_amdgcn_s_barrier();
        int slot = NS - 1;
        for (; ct < len; ct += nbx) {
            const int nch = (a.seg[tile_at(ct).si].Kd + KB - 1) / KB;
            for (int cc = 0; cc < nch; cc++) {
                issue(slot);
                slot = slot + 1 == NS ? 0 : slot + 1;
                VMCNT_WAIT(OUT);
                __builtin_amdgcn_s_barrier();
            }
        }
        VMCNT_WAIT(0);
    };
    if (wave >= GRP_MMW + GRP_WLD) {   /* a planes' wave */
        const int lw = wave - GRP_MMW - GRP_WLD;
        rsrc_t ar[3];
        constexpr int AP = sp::AP;
        uint32_t ao[AP];
        auto row_of = [&](int u) { return RPI * (AP * lw + u) + lane / LPR; };
        auto set_issue = [&](const grp_tile &id) {
            const mm_bf16_mm_seg &g = a.seg[id.si];
            kd = g.Kd;
            inch = (kd + KB - 1) / KB;
            const int rows = min(id.M - id.m0, BM);
#pragma unroll
            for (int q = 0; q < 3; q++)
                ar[q] = raw_rsrc(g.a + (size_t)q * g.aplane + (size_t)(id.row0 + id.m0) * kd,
                                 (uint32_t)rows * (uint32_t)kd * 2u);
#pragma unroll
            for (int u = 0; u < AP; u++) {
                const int R = row_of(u);
                ao[u] = R < rows ? ((uint32_t)R * (uint32_t)kd + (uint32_t)piece(R)) * 2u : GRP_OOB;
            }
        };
        auto issue = [&](int slot) {
            const uint32_t sb = ldsa + (uint32_t)(slot * sp::A_BYTES + AP * lw * 1024);
            const int k0 = ic * KB;
#pragma unroll
            for (int u = 0; u < AP; u++) {
                const uint32_t o = ao[u] != GRP_OOB && k0 + piece(row_of(u)) < kd ? ao[u] + (uint32_t)(2 * k0) : GRP_OOB;
#pragma unroll
                for (int q = 0; q < 3; q++) lds_dma16_buf(o, ar[q], sb + (uint32_t)((q * (BM / RPI) + u) * 1024));
            }
            if (advance()) set_issue(tile_at(it));
        };
        set_issue(tile_at(it));
        load_ring(const_int<sp::NSA>(), const_int<sp::A_LPW>(), issue);
        return;
    }

    if (wave >= GRP_MMW) {   /* a weights' wave */
        const int lw = wave - GRP_MMW;
        rsrc_t wr[GU ? 2 : 1];
        uint32_t wo[sp::W_LPW];
        auto row_of = [&](int u) { return RPI * (sp::W_LPW * lw + u) + lane / LPR; };
        auto up = [&](int u) { return GU && RPI * (sp::W_LPW * lw + u) >= GRP_NB / 2; };   /* uniform */
        auto set_issue = [&](const grp_tile &id) {
            const mm_bf16_mm_seg &g = a.seg[id.si];
            kd = g.Kd;
            inch = (kd + KB - 1) / KB;
            wr[0] = raw_rsrc(g.w0 + (size_t)id.e * g.wstride, (uint32_t)g.N * (uint32_t)kd * 2u);
            if (GU) wr[GU ? 1 : 0] = raw_rsrc(g.w1 + (size_t)id.e * g.wstride, (uint32_t)g.N * (uint32_t)kd * 2u);
#pragma unroll
            for (int u = 0; u < sp::W_LPW; u++) {
                const int R = row_of(u), col = id.slab * CPT + (GU ? R & 63 : R);
                wo[u] = col < g.N ? ((uint32_t)col * (uint32_t)kd + (uint32_t)piece(R)) * 2u : GRP_OOB;
            }
        };
        auto issue = [&](int slot) {
            const uint32_t sb = ldsw + (uint32_t)(slot * sp::W_BYTES + sp::W_LPW * lw * 1024);
            const int k0 = ic * KB;
#pragma unroll
            for (int u = 0; u < sp::W_LPW; u++)
                lds_dma16_buf_nt(wo[u] != GRP_OOB && k0 + piece(row_of(u)) < kd ? wo[u] + (uint32_t)(2 * k0) : GRP_OOB,
                                 up(u) ? wr[GU ? 1 : 0] : wr[0], sb + (uint32_t)(u * 1024));
            if (advance()) set_issue(tile_at(it));
        };
        set_issue(tile_at(it));
        load_ring(const_int<sp::NSW>(), const_int<sp::W_LPW>(), issue);
        return;
    }

    /* ---- operand reads ----
     * weight tile j of this wave: LDS rows wrow(j) + l % 16; row tile t: plane
     * p, row 16 (TT wm + t) + l % 16; K step s: piece 4 s + l / 16 */
    const int wn = BM == 64 ? wave & 1 : wave, wm = BM == 64 ? wave >> 1 : 0;
    constexpr int WT = sp::WT, TT = sp::TT, KS = sp::KS;
    auto wrow = [&](int j) {
        return GU ? (j & 1) * 64 + 8 * WT * wn + 16 * (j >> 1) : 16 * WT * wn + 16 * j;
    };
    typedef const __attribute__((address_space(3))) i32x4 *lds_cp;
    const int swz = sp::swz(l16);
    i32x4 rw[2][WT], rx[2][TT][3];
    auto read = [&](int sw, int sa, int s) {
        const uint32_t p = 16 * ((4 * s + g4) ^ swz) + l16 * sp::ROWB;
        const uint32_t wb = ldsw + (uint32_t)(sw * sp::W_BYTES) + p, ab = ldsa + (uint32_t)(sa * sp::A_BYTES) + p;
#pragma unroll
        for (int j = 0; j < WT; j++) rw[s & 1][j] = *(lds_cp)(wb + (uint32_t)(wrow(j) * sp::ROWB));
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int q = 0; q < 3; q++)
                rx[s & 1][t][q] = *(lds_cp)(ab + (uint32_t)((q * BM + 16 * (TT * wm + t)) * sp::ROWB));
    };
    f32x4 acch[TT][WT], accl[TT][WT], accm[TT][WT];
    auto zero = [&]() {
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int j = 0; j < WT; j++) acch[t][j] = accl[t][j] = accm[t][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    };
    auto mfma = [&](int s) {
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int j = 0; j < WT; j++) {
                    f32x4 &c = q == 0 ? acch[t][j] : accl[t][j];
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, rw[s & 1][j]),
                                                                __builtin_bit_cast(bf16x8, rx[s & 1][t][q]), c, 0, 0, 0);
                }
        /* the next step's reads between the MFMAs */
        constexpr int RD = WT + 3 * TT, MF = 3 * TT * WT, PER = MF / RD > 0 ? MF / RD : 1;
#pragma unroll
        for (int i = 0; i < RD; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
    };
    auto flush = [&]() {
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int j = 0; j < WT; j++) {
                accm[t][j] += acch[t][j];
                acch[t][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
            }
    };
    /* lane l holds row l % 16 of each row tile, columns 4 (l / 16) + i of
     * each column tile (the weights are the first operand) */
    auto store = [&](const grp_tile &id) {
        const mm_bf16_mm_seg &g = a.seg[id.si];
#pragma unroll
        for (int t = 0; t < TT; t++) {
            const int m = id.m0 + 16 * (TT * wm + t) + l16;
            const size_t row = (size_t)(id.row0 + m);
#pragma unroll
            for (int j = 0; j < WT; j += GU ? 2 : 1) {
                const int col = id.slab * CPT + wrow(j) + 4 * g4;
                if (m >= id.M || col >= g.N) continue;
                const f32x4 v0 = accm[t][j] + (acch[t][j] + accl[t][j]);
                if (GU) {
                    const f32x4 v1 = accm[t][j + 1] + (acch[t][j + 1] + accl[t][j + 1]);
                    u16x4 h, md, lo;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        uint16_t h16, m16, l16_;
                        split3(swiglu_f(v0[i], v1[i]), &h16, &m16, &l16_);
                        h[i] = h16;
                        md[i] = m16;
                        lo[i] = l16_;
                    }
                    uint16_t *o = g.h + row * g.N + col;
                    *(u16x4 *)o = h;
                    *(u16x4 *)(o + g.hplane) = md;
                    *(u16x4 *)(o + 2 * g.hplane) = lo;
                } else {
                    *(f32x4 *)(g.y + row * g.N + col) = v0;
                }
            }
        }
    };

    grp_tile cur = tile_at(ct);
    int nch = (a.seg[cur.si].Kd + KB - 1) / KB, cc = 0, sw = 0, sa = 0;
    zero();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0, 0);
    for (;;) {
        const int nw = sw + 1 == sp::NSW ? 0 : sw + 1, na = sa + 1 == sp::NSA ? 0 : sa + 1;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (s + 1 < KS) {
                read(sw, sa, s + 1);
            } else {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                read(nw, na, 0);
            }
            mfma(s);
            __builtin_amdgcn_sched_barrier(0);
        }
        sw = nw;
        sa = na;
        if (++cc == nch) {
            store(cur);
            ct += nbx;
            if (ct >= len) break;
            cur = tile_at(ct);
            nch = (a.seg[cur.si].Kd + KB - 1) / KB;
            cc = 0;
            zero();
        } else if (cc % (GRP_FLUSH / KB) == 0) {
            flush();
        }
    }
}

#define GRP_KERNEL(name, BM, GU)                                                            \
    extern "C" __global__ __launch_bounds__(MM_BF16_MM_THREADS, 1) void name(mm_bf16_mm_args a) { grp_run<BM, GU>(a); }
GRP_KERNEL(mm_bf16_gu_16, 16, true)
GRP_KERNEL(mm_bf16_gu_32, 32, true)
GRP_KERNEL(mm_bf16_gu_64, 64, true)
GRP_KERNEL(mm_bf16_dn_16, 16, false)
GRP_KERNEL(mm_bf16_dn_32, 32, false)
GRP_KERNEL(mm_bf16_dn_64, 64, false)
