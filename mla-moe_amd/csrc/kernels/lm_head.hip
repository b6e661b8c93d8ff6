/* lm_head.hip -- the decode step's LM head on gfx950: final RMSNorm, logits
 * over the vocabulary, greedy argmax.
 *
 * Reference semantics (src/run.c):
 *   rmsnorm  run.c:22-27   y = (x * inv) * w, inv = 1 / sqrtf(ss / n + eps),
 *                          ss the sum of squares
 *   logits   run.c:493-494 matmul(logits, xb, lm_head, vocab, hidden)
 *   sample   run.c:503-508 first index of the maximum under a strict '>'
 *                          scan from index 0
 * The sum of squares and the logit dot products are reduced in parallel
 * (fp32, a different association than the reference's sequential loops):
 * results agree to ~1e-6 relative, which the tests bound.
 *
 * Kernels:
 *   mm_lm_gemv   for up to MM_LM_NB tokens: rmsnorm, logits (every weight
 *                row read once: HBM-bound, 2 bytes per weight) and per-wave
 *                argmax partials in one pass (the GEMV core of gemv.h)
 *   mm_rmsnorm_hl + mm_lm_gemm  for up to 64 tokens: the same split, logits on
 *                the matrix cores
 *   mm_rmsnorm   one block per token (the GEMM path for more tokens)
 *   mm_argmax_part / mm_argmax_final   segments of every row in parallel
 *                (mm_lm_gemv and mm_lm_gemm write their partials themselves),
 *                then one block per row over the partials
 */
#include "gemv.h"

/* ---- RMSNorm ---------------------------------------------------------------- */

/* 1 / sqrt(sum / n + eps) over the block's NT threads, ss = this thread's
 * sum of squares (every thread calls it). */
template <int NT>
__device__ __forceinline__ float rms_inv_block(float ss, int n, float eps) {
    __shared__ float red[NT / MM_WAVE];
    ss = wave_sum(ss);
    const int lane = threadIdx.x & (MM_WAVE - 1), wave = threadIdx.x / MM_WAVE;
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int w = 0; w < NT / MM_WAVE; w++) tot += red[w];
    return 1.0f / sqrtf(tot / (float)n + eps);
}

extern "C" __global__ __launch_bounds__(256) void mm_rmsnorm(mm_rmsnorm_args a) {
    const int t = blockIdx.x;
    const float *x = a.x + (size_t)t * a.n;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < a.n; i += 256) ss += x[i] * x[i];
    const float inv = rms_inv_block<256>(ss, a.n, a.eps);
    float *y = a.y + (size_t)t * a.n;
    for (int i = threadIdx.x; i < a.n; i += 256) y[i] = x[i] * inv * bf16_f32(a.w[i]);
}

/* As mm_rmsnorm (the same arithmetic), the normalised row written as bf16
 * hi/lo planes: hi = rne16(y), lo = rne16(y - hi), the split the bf16 GEMMs
 * apply to fp32 activations.  grid (T). */
extern "C" __global__ __launch_bounds__(256) void mm_rmsnorm_hl(mm_rmsnorm_hl_args a) {
    const int t = blockIdx.x;
    const float *x = a.x + (size_t)t * a.n;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < a.n; i += 256) ss += x[i] * x[i];
    const float inv = rms_inv_block<256>(ss, a.n, a.eps);
    uint16_t *hi = a.yhl + (size_t)t * a.n, *lo = hi + (size_t)gridDim.x * a.n;
    /* 8 consecutive values per thread (n is a multiple of 8): 16-byte
     * stores of each plane */
    typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
    for (int i = 8 * threadIdx.x; i < a.n; i += 8 * 256) {
        const f32x4 x0 = *(const f32x4 *)(x + i), x1 = *(const f32x4 *)(x + i + 4);
        const u16x8_t w8 = *(const u16x8_t *)(a.w + i);
        u16x8_t h8, l8;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            /* no contraction: lo splits the rounded fp32 y, as the GEMMs
             * that split a stored row do (y - hi fused with y's last
             * product would split the unrounded product) */
#pragma clang fp contract(off)
            const float v = (k < 4 ? x0[k & 3] : x1[k & 3]) * inv * bf16_f32(w8[k]);
            h8[k] = rne16(v);
            l8[k] = rne16(v - bf16_f32(h8[k]));
        }
        *(u16x8_t *)(hi + i) = h8;
        *(u16x8_t *)(lo + i) = l8;
    }
}

/* mm_reduce_rmsnorm_args: one block of RRN_T threads per row, each thread
 * RRN_PT elements (n <= RRN_T * RRN_PT) kept in registers between the sum
 * and the norm.  The partial loads of up to RRN_SU splits are issued
 * together: a row block is one latency-bound pass, so the loads must not
 * wait for each other. */
#define RRN_T MM_RRN_THREADS
#define RRN_PT MM_RRN_PT
#define RRN_SU 8
extern "C" __global__ __launch_bounds__(RRN_T) void mm_reduce_rmsnorm(mm_reduce_rmsnorm_args a) {
    const int t = blockIdx.x, n = a.n;
    const size_t plane = (size_t)a.T * n;
    float *x = a.x + (size_t)t * n;
    const float *p0 = a.part + (size_t)t * n;
    float v[RRN_PT];
#pragma unroll
    for (int k = 0; k < RRN_PT; k++) v[k] = 0.0f;
    for (int s0 = 0; s0 < a.nsplit; s0 += RRN_SU) {
        float pv[RRN_SU][RRN_PT];
#pragma unroll
        for (int u = 0; u < RRN_SU; u++)
#pragma unroll
            for (int k = 0; k < RRN_PT; k++) {
                const int i = threadIdx.x + RRN_T * k;
                pv[u][k] = (s0 + u < a.nsplit && i < n) ? p0[(size_t)(s0 + u) * plane + i] : 0.0f;
            }
#pragma unroll
        for (int u = 0; u < RRN_SU; u++)
#pragma unroll
            for (int k = 0; k < RRN_PT; k++)
                if (s0 + u < a.nsplit) v[k] = (s0 + u == 0) ? pv[u][k] : v[k] + pv[u][k];
    }
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < RRN_PT; k++) {
        const int i = threadIdx.x + RRN_T * k;
        if (i < n) {
            const float xv = x[i] + v[k];
            x[i] = xv;
            v[k] = xv;
            ss += xv * xv;
        }
    }
    const float inv = rms_inv_block<RRN_T>(ss, n, a.eps);
    float *xn = a.xn + (size_t)t * n;
#pragma unroll
    for (int k = 0; k < RRN_PT; k++) {
        const int i = threadIdx.x + RRN_T * k;
        if (i < n) xn[i] = v[k] * inv * bf16_f32(a.w[i]);
    }
}

/* ---- greedy argmax ---------------------------------------------------------- */

/* (v, i) beats (bv, bi) when v is a number and bv is not, or v > bv, or
 * v == bv at a lower index: the first maximum of the sequential strict-'>'
 * scan, NaNs never winning.  A NaN at index 0 is the scan's start value and
 * is never beaten (handled by the caller). */
__device__ __forceinline__ bool am_better(float v, int i, float bv, int bi) {
    if (v != v) return false;
    if (bv != bv) return true;
    return v > bv || (v == bv && i < bi);
}

/* ---- logits GEMV -------------------------------------------------------------- */

/* The register-resident GEMV core (gemv.h) over the vocabulary with the
 * final norm applied to the activations in registers, so no separate norm
 * pass runs.  Each wave keeps its best (logit, row) per token; the block's
 * best goes to part_v / part_i [t][block]: the argmax then only reduces
 * those partials. */
template <int NB>
struct lm_sink {
    float *y;
    int V, B;
    float bv[NB];
    int bi[NB];
    __device__ __forceinline__ void operator()(int row, int t, float v) {
        if ((threadIdx.x & (MM_WAVE - 1)) == 0 && t < B) y[(size_t)t * V + row] = v;
        if (am_better(v, row, bv[t], bi[t])) { bv[t] = v; bi[t] = row; }
    }
};

template <int NB>
__device__ __forceinline__ void lm_gemv(const mm_lm_gemv_args &a) {
    f32x4 xv[NB][GV_PPL][2];
    gemv_load_x<NB>(xv, a.x, a.B, a.H, a.norm, a.eps, false);
    lm_sink<NB> sk;
    sk.y = a.y;
    sk.V = a.V;
    sk.B = a.B;
#pragma unroll
    for (int t = 0; t < NB; t++) { sk.bv[t] = __builtin_nanf(""); sk.bi[t] = 0x7fffffff; }
    const uint16_t *w = a.w;
    const int H = a.H;
    gemv_rows<NB>(xv, H, a.V, [=](int r) { return w + (size_t)r * H; }, sk);
    /* the block's best per token: one partial per block */
    __shared__ float sv[NB][256 / MM_WAVE];
    __shared__ int si[NB][256 / MM_WAVE];
    const int lane = threadIdx.x & (MM_WAVE - 1), wave = threadIdx.x / MM_WAVE;
    if (lane == 0)
#pragma unroll
        for (int t = 0; t < NB; t++) { sv[t][wave] = sk.bv[t]; si[t][wave] = sk.bi[t]; }
    __syncthreads();
    if (threadIdx.x < NB && (int)threadIdx.x < a.B) {
        const int t = threadIdx.x;
        float v = sv[t][0];
        int i = si[t][0];
        for (int w2 = 1; w2 < 256 / MM_WAVE; w2++)
            if (am_better(sv[t][w2], si[t][w2], v, i)) { v = sv[t][w2]; i = si[t][w2]; }
        a.part_v[(size_t)t * gridDim.x + blockIdx.x] = v;
        a.part_i[(size_t)t * gridDim.x + blockIdx.x] = i;
    }
}

/* one entry point per token count (register allocation per instance) */
extern "C" __global__ __launch_bounds__(256) void mm_lm_gemv_1(mm_lm_gemv_args a) { lm_gemv<1>(a); }
extern "C" __global__ __launch_bounds__(256) void mm_lm_gemv_2(mm_lm_gemv_args a) { lm_gemv<2>(a); }
extern "C" __global__ __launch_bounds__(256) void mm_lm_gemv_4(mm_lm_gemv_args a) { lm_gemv<4>(a); }

/* Pass 1: block (seg, t) scans its contiguous segment of row t and writes
 * the segment's best (value, index) to part[t][seg]. */
extern "C" __global__ __launch_bounds__(256) void mm_argmax_part(mm_argmax_args a) {
    __shared__ float sv[256 / MM_WAVE];
    __shared__ int si[256 / MM_WAVE];
    const int t = blockIdx.y, seg = blockIdx.x;
    const float *lg = a.logits + (size_t)t * a.n;
    const int len = (a.n + a.nseg - 1) / a.nseg;
    const int i0 = seg * len, i1 = min(a.n, i0 + len);
    float bv = __builtin_nanf("");
    int bi = 0x7fffffff;
    for (int i = i0 + threadIdx.x; i < i1; i += 256) {
        const float v = lg[i];
        if (am_better(v, i, bv, bi)) { bv = v; bi = i; }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, MM_WAVE);
        const int oi = __shfl_xor(bi, off, MM_WAVE);
        if (am_better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
    }
    const int lane = threadIdx.x & (MM_WAVE - 1), wave = threadIdx.x / MM_WAVE;
    if (lane == 0) { sv[wave] = bv; si[wave] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 256 / MM_WAVE; w++)
            if (am_better(sv[w], si[w], sv[0], si[0])) { sv[0] = sv[w]; si[0] = si[w]; }
        a.part_v[(size_t)t * a.nseg + seg] = sv[0];
        a.part_i[(size_t)t * a.nseg + seg] = si[0];
    }
}

/* Pass 2: one block per row reduces the partials (8 loads per thread in
 * flight) in the same order-independent rule, then applies the scan's
 * start at index 0. */
extern "C" __global__ __launch_bounds__(256) void mm_argmax_final(mm_argmax_args a) {
    __shared__ float sv[256 / MM_WAVE];
    __shared__ int si[256 / MM_WAVE];
    const int t = blockIdx.x;
    const float *pv = a.part_v + (size_t)t * a.nseg;
    const int32_t *pi = a.part_i + (size_t)t * a.nseg;
    float bv = __builtin_nanf("");
    int bi = 0x7fffffff;
    for (int s0 = 0; s0 < a.nseg; s0 += 8 * 256) {
        float v[8];
        int i[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int s = s0 + k * 256 + threadIdx.x;
            v[k] = s < a.nseg ? pv[s] : __builtin_nanf("");
            i[k] = s < a.nseg ? pi[s] : 0x7fffffff;
        }
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (am_better(v[k], i[k], bv, bi)) { bv = v[k]; bi = i[k]; }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, MM_WAVE);
        const int oi = __shfl_xor(bi, off, MM_WAVE);
        if (am_better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
    }
    const int lane = threadIdx.x & (MM_WAVE - 1), wave = threadIdx.x / MM_WAVE;
    if (lane == 0) { sv[wave] = bv; si[wave] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 256 / MM_WAVE; w++)
            if (am_better(sv[w], si[w], bv, bi)) { bv = sv[w]; bi = si[w]; }
        const float v0 = a.logits[(size_t)t * a.n];
        /* run.c:504-508 starts its scan at logits[0]: a NaN there is never
         * replaced; no number at all (every entry NaN) also leaves 0 */
        a.tokens[t] = (v0 != v0 || bi == 0x7fffffff) ? 0 : bi;
    }
}

/* ---- logits GEMM for 5..64 rows ----------------------------------------------
 *
 * y[T, N] = x . W^T for the LM head's batch rows, and every block's best
 * logit per token for the argmax.  Bound by the weight stream (2 N K bytes).
 *
 * Persistent, one block per CU: the vocabulary's 16-column units are dealt out
 * evenly in contiguous ranges (102400 columns: 25 units for each of 256
 * blocks), and a block takes its range in equal passes of at most MM_LMG_MU
 * units.  (One 256-column tile per block left 400 blocks on 256 CUs: the
 * second turn filled 56% of them.)
 *
 * Eight waves multiply, two load W, one loads x's bf16 hi/lo planes, into two
 * LDS rings that run on across passes: W in stages of four 64-wide K chunks, x
 * one chunk at a time.  A wave's vector memory operations complete in order,
 * so a wave that loaded both operands could not wait for x (an L2 hit) without
 * waiting for weights (HBM, wanted far ahead), and a multiplying wave that
 * loaded any would wait behind its stores of y.  Loads of rows past the pass's
 * columns or T are out of the buffer's range: no memory is read, zeros are
 * staged.
 *
 * W streams faster in longer pieces of a row (loads alone, 64 x 102400 x 2048:
 * 83 us in 128-byte pieces, 74 us in 512-byte pieces), which is why a pass is
 * only 112 columns wide although x (512 KB) is then read from L2 four times
 * per block: whole LM head 111.2 us, 112.5 us with two passes of 208 columns
 * in 128-byte pieces, 147 us with a tile per block.
 *
 * Multiplying wave w owns units w % 4, w % 4 + 4, .. of the pass for 32 rows:
 * v_mfma_f32_16x16x32_bf16 with W as the first operand, so that a lane holds 4
 * consecutive columns of one row; per 32-wide K step every output takes its hi
 * product, then its lo product (mm_gemm_skinny's sequence).  The operands of
 * the next step are read during the current step's MFMAs.
 *
 * LDS rows are 16-byte pieces, piece p of row r in slot p ^ swz(r): the 16
 * lanes of an operand read (16 consecutive rows, one piece) hit distinct
 * 16-byte bank groups. */
#define LMG_MMW 8                     /* multiplying waves: 4 over the units x 2 over the rows */
#define LMG_WLD 2                     /* W-loading waves */
#define LMG_PPR (8 * MM_LMG_WC)       /* 16-byte pieces per W row in LDS */
#define LMG_RPL (MM_WAVE / LMG_PPR)   /* W rows per load */
#define LMG_W_LPW (16 * MM_LMG_MU / LMG_RPL / LMG_WLD)   /* loads per W-loading wave per stage */
#define LMG_X_LPW 16                  /* loads of the x-loading wave per chunk */
#define LMG_UPW ((MM_LMG_MU + 3) / 4)   /* units per multiplying wave */
#define LMG_GPW 2                     /* 16-row groups per multiplying wave */
#define LMG_OOB 0xFFFFFFF0u           /* past every buffer range */
static_assert(MM_LMG_THREADS == (LMG_MMW + LMG_WLD + 1) * MM_WAVE, "threads known to the host");
static_assert(LMG_W_LPW * LMG_RPL * LMG_WLD == 16 * MM_LMG_MU && LMG_W_LPW * (MM_LMG_NSW - 1) < 64 && LMG_X_LPW * (MM_LMG_NSX - 1) < 64, "loads in flight: vmcnt");
typedef __bf16 lmg_bf16x8 __attribute__((ext_vector_type(8)));
typedef const __attribute__((address_space(3))) i32x4 *lmg_lds_cp;

/* the slots' swizzle for rows of 16-byte pieces, 8 or more of them */
__device__ __forceinline__ int lmg_swz(int r, int pieces) { return pieces == 8 ? (r >> 1) & 7 : r & 15; }

/* A loading wave: NI loads per stage, a stage being CPS 64-wide chunks of K;
 * byte offsets vo[] within a buffer whose base moves one stage at a time, NS
 * ring stages of `stage` bytes.  One barrier per chunk, as the multiplying
 * waves have. */
template <int NI, int NS, int CPS, bool NT, class F>
__device__ __forceinline__ void lmg_load(int np, int nch, uint32_t lds0, uint32_t stage, F pass_of) {
    const uint16_t *base;
    uint32_t range, vo[NI];
    const int nst = (nch + CPS - 1) / CPS, total = np * nst;
    int ip = 0, is = 0, slot = 0;                  /* pass, stage and slot of the next issue */
    auto issue = [&]() {
        if (is == 0) pass_of(ip, base, range, vo);
        const rsrc_t r = raw_rsrc(base + 64 * CPS * (size_t)is,
                                  __builtin_amdgcn_readfirstlane(range - 128u * CPS * (uint32_t)is));
        const uint32_t sb = lds0 + (uint32_t)slot * stage;
#pragma unroll
        for (int u = 0; u < NI; u++) {
            if (NT) lds_dma16_buf_nt(vo[u], r, sb + (uint32_t)u * 1024u);
            else lds_dma16_buf(vo[u], r, sb + (uint32_t)u * 1024u);
        }
        slot = slot + 1 == NS ? 0 : slot + 1;
        if (++is == nst) {
            is = 0;
            ip++;
        }
    };
#pragma unroll 1
    for (int i = 0; i < NS - 1 && i < total; i++) issue();
    int cs = 0;
    for (int i = 0; i < total; i++) {
        /* stage i landed: only the loads of the NS - 2 stages after it may be out */
        if (i + NS - 2 < total) VMCNT_WAIT(NI * (NS - 2));
        else VMCNT_WAIT(0);
        __builtin_amdgcn_s_barrier();
        if (i + NS - 1 < total) issue();   /* into the slot of stage i - 1, read before the barrier */
        for (int c = CPS * cs + 1; c < min(CPS * (cs + 1), nch); c++) __builtin_amdgcn_s_barrier();
        cs = cs + 1 == nst ? 0 : cs + 1;
    }
}

extern "C" __global__ __launch_bounds__(MM_LMG_THREADS, 1) void mm_lm_gemm(mm_lm_gemm_args a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & (MM_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / MM_WAVE);
    const int K = a.K, T = a.T, N = a.N, nch = K / 64;
    const int nu = (N + 15) / 16;
    /* (integer divisions run on the vector unit: back to scalars) */
    const int ub = __builtin_amdgcn_readfirstlane((int)((int64_t)nu * blockIdx.x / gridDim.x));
    const int un = __builtin_amdgcn_readfirstlane((int)((int64_t)nu * (blockIdx.x + 1) / gridDim.x)) - ub;
    const int np = (un + MM_LMG_MU - 1) / MM_LMG_MU;
    auto first = [&](int p) { return ub + __builtin_amdgcn_readfirstlane(un * p / np); };   /* first unit of pass p */
    const uint32_t ldsw = lds_addr(lds), ldsx = ldsw + MM_LMG_NSW * MM_LMG_WB;

    if (wave >= LMG_MMW + LMG_WLD) {   /* x: load i is plane i / 8, rows from 8 (i % 8) */
        lmg_load<LMG_X_LPW, MM_LMG_NSX, 1, false>(
            np, nch, ldsx, MM_LMG_XB, [&](int, const uint16_t *&base, uint32_t &range, uint32_t *vo) {
                base = a.xhl;
                range = 4u * (uint32_t)T * (uint32_t)K;
#pragma unroll
                for (int i = 0; i < LMG_X_LPW; i++) {
                    const int r = 8 * (i & 7) + (lane >> 3);
                    vo[i] = r < T ? 2u * (uint32_t)((i >> 3) * T + r) * (uint32_t)K + 16u * (uint32_t)((lane & 7) ^ lmg_swz(r, 8)) : LMG_OOB;
                }
            });
    } else if (wave >= LMG_MMW) {
        const int w0 = LMG_W_LPW * (wave - LMG_MMW);
        lmg_load<LMG_W_LPW, MM_LMG_NSW, MM_LMG_WC, true>(
            np, nch, ldsw + 1024u * (uint32_t)w0, MM_LMG_WB,
            [&](int p, const uint16_t *&base, uint32_t &range, uint32_t *vo) {
                const int n0 = 16 * first(p), cols = min(16 * first(p + 1), N) - n0;
                base = a.w + (size_t)n0 * K;
                range = 2u * (uint32_t)cols * (uint32_t)K;
#pragma unroll
                for (int u = 0; u < LMG_W_LPW; u++) {
                    const int r = LMG_RPL * (w0 + u) + lane / LMG_PPR;
                    vo[u] = r < cols ? 2u * (uint32_t)r * (uint32_t)K + 16u * (uint32_t)(lane % LMG_PPR ^ lmg_swz(r, LMG_PPR)) : LMG_OOB;
                }
            });
    }

    const int l16 = lane & 15, g4 = lane >> 4;
    const int wu = wave & 3, g0 = wave / 4 * LMG_GPW;   /* a multiplying wave's units (mod 4), 16-row groups */
    float bv[LMG_GPW];
    int bi[LMG_GPW];
#pragma unroll
    for (int g = 0; g < LMG_GPW; g++) { bv[g] = __builtin_nanf(""); bi[g] = 0x7fffffff; }
    if (wave < LMG_MMW) {
        const bool v4 = N % 4 == 0;   /* rows of y 16-byte aligned */
        const int total = np * nch;
        i32x4 wv[2][LMG_UPW], xa[2][2][LMG_GPW];
        auto read = [&](int sw, int sc, int sx, int s) {
            /* rows of all fragments agree mod 16: one swizzle per operand */
            const uint32_t q = (uint32_t)(l16 * 128 + 16 * ((4 * s + g4) ^ lmg_swz(l16, 8)));
            const uint32_t qw = (uint32_t)(l16 * 16 * LMG_PPR + 16 * ((8 * sc + 4 * s + g4) ^ lmg_swz(l16, LMG_PPR)));
            const uint32_t wb = ldsw + (uint32_t)(sw * MM_LMG_WB) + qw, xb = ldsx + (uint32_t)(sx * MM_LMG_XB) + q;
#pragma unroll
            for (int j = 0; j < LMG_UPW; j++)   /* a wave with fewer units repeats the last one, unused */
                wv[s][j] = *(lmg_lds_cp)(wb + (uint32_t)(min(wu + 4 * j, MM_LMG_MU - 1) * 256 * LMG_PPR));
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int g = 0; g < LMG_GPW; g++) xa[s][h][g] = *(lmg_lds_cp)(xb + (uint32_t)((64 * h + 16 * (g0 + g)) * 128));
        };
        f32x4 acc[LMG_UPW][LMG_GPW];
        auto zero = [&]() {
#pragma unroll
            for (int j = 0; j < LMG_UPW; j++)
#pragma unroll
                for (int g = 0; g < LMG_GPW; g++) acc[j][g] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        };
        auto mfma = [&](int s) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int g = 0; g < LMG_GPW; g++)
#pragma unroll
                    for (int j = 0; j < LMG_UPW; j++)
                        acc[j][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(lmg_bf16x8, wv[s][j]),
                            __builtin_bit_cast(lmg_bf16x8, xa[s][h][g]), acc[j][g], 0, 0, 0);
        };
        int sw = 0, sc = 0, sx = 0, c = 0, p = 0;   /* W slot, chunk within it, x slot; chunk, pass */
        zero();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read(0, 0, 0, 0);
        for (int i = 0; i < total; i++) {
            read(sw, sc, sx, 1);
            __builtin_amdgcn_sched_barrier(0);
            mfma(0);
            __builtin_amdgcn_sched_barrier(0);
            /* this wave's reads of the slots are done before the barrier that
             * frees them and makes the next chunk's loads visible */
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const bool last = ++c == nch;
            sx = sx + 1 == MM_LMG_NSX ? 0 : sx + 1;
            if (++sc == MM_LMG_WC || last) {
                sc = 0;
                sw = sw + 1 == MM_LMG_NSW ? 0 : sw + 1;
            }
            if (i + 1 < total) {
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                read(sw, sc, sx, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            mfma(1);
            __builtin_amdgcn_sched_barrier(0);
            if (!last) continue;
            /* C[column 16 u + 4 (l / 16) + i][token 16 g + l % 16] */
            const int u0 = first(p), un_p = first(p + 1) - u0;
#pragma unroll
            for (int j = 0; j < LMG_UPW; j++) {
                const int u = wu + 4 * j, n = 16 * (u0 + u) + 4 * g4;
                if (u >= un_p) continue;
#pragma unroll
                for (int g = 0; g < LMG_GPW; g++) {
                    const int t = 16 * (g0 + g) + l16;
                    if (t >= T || n >= N) continue;
                    float *y = a.y + (size_t)t * N + n;
                    if (v4) __builtin_nontemporal_store(acc[j][g], (f32x4 *)y);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        if (n + k >= N) continue;
                        if (!v4) y[k] = acc[j][g][k];
                        if (am_better(acc[j][g][k], n + k, bv[g], bi[g])) { bv[g] = acc[j][g][k]; bi[g] = n + k; }
                    }
                }
            }
            c = 0;
            p++;
            zero();
        }
#pragma unroll
        for (int off = 16; off < MM_WAVE; off <<= 1)
#pragma unroll
            for (int g = 0; g < LMG_GPW; g++) {
                const float ov = __shfl_xor(bv[g], off, MM_WAVE);
                const int oi = __shfl_xor(bi[g], off, MM_WAVE);
                if (am_better(ov, oi, bv[g], bi[g])) { bv[g] = ov; bi[g] = oi; }
            }
    }
    /* the waves' bests meet in the (drained) ring's LDS */
    __syncthreads();
    float *sv = (float *)lds;             /* [4][64] */
    int *si = (int *)(lds + 4 * 64 * 4);
    if (wave < LMG_MMW && g4 == 0)
#pragma unroll
        for (int g = 0; g < LMG_GPW; g++) {
            sv[wu * 64 + 16 * (g0 + g) + l16] = bv[g];
            si[wu * 64 + 16 * (g0 + g) + l16] = bi[g];
        }
    __syncthreads();
    if (tid < T) {
        float v = sv[tid];
        int ix = si[tid];
        for (int w = 1; w < 4; w++)
            if (am_better(sv[w * 64 + tid], si[w * 64 + tid], v, ix)) { v = sv[w * 64 + tid]; ix = si[w * 64 + tid]; }
        a.part_v[(size_t)tid * gridDim.x + blockIdx.x] = v;
        a.part_i[(size_t)tid * gridDim.x + blockIdx.x] = ix;
    }
}
