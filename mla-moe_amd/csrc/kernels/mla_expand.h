/* mla_expand.h -- MLA attention of a prompt's rows in the expanded form
 * (part of mla.hip): keys and values per head, as forward_unabsorbed has them
 * (src/run.c:189-370), instead of the latent vectors.
 *
 * A row of a prompt meets every earlier key.  Absorbed, a (row, key, head)
 * triple costs 576 + 512 latent products, times two for the bf16 pair that
 * carries the fp32 operand: 2,176.  Expanded it costs 128 + 64 + 128 products,
 * times four where both operands are pairs and two for the rope part: 1,152;
 * and the absorbed queries and W_UV products of every row go.  The price is
 * one pass over the latent cache per layer (mm_mla_expand: 2 x 128 x 512
 * products per key and head, both operands bf16, no pairs), so it pays from
 * 65 rows on, and from one row per 20 keys (MM_MLA_EXPAND_MIN,
 * MM_MLA_EXPAND_KEYS).
 *
 * All four products of two pairs are kept: without lo * lo the error against
 * 64 bits is 15% above the absorbed form's (emulated, 700 random keys: 4.9e-6
 * against 4.2e-6; with it 4.0e-6).
 *
 * Layout of the expanded keys and values, per 32-key block and head, 32 KB:
 *   K hi [32 keys][128], K lo, V hi [128 dims][32 keys], V lo
 * 16-byte pieces swizzled for the LDS reads below (the block is copied to LDS
 * as it is): K piece p of key r in slot p ^ (r % 16); V piece p of dim d in
 * slot p ^ (d / 4 % 4).  V piece 2 s + h holds keys 16 s + 4 h + {0..3, 8..11}:
 * the keys whose probabilities lane half h holds as the second operand of
 * v_mfma_f32_32x32x16_bf16 after the score product (result register 4 g + i
 * of lane l is key 8 g + 4 (l / 32) + i). */
#define XD 128                    /* nope and value dimensions per head */
#define XB 32                     /* keys per block */
#define XBLK MM_MLA_XBLK          /* bytes per block and head */
#define XT (XB * XD * 2)          /* bytes of one of its four tiles */
static_assert(XBLK == 4 * XT, "expanded block");
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(3))) i32x4 *lds_c4;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

/* The bf16 pair of two values, (hi, lo) packed two to a word: v_cvt_pk_bf16_f32
 * rounds to nearest even, as split_bf16 does, in a tenth of its instructions. */
__device__ __forceinline__ void split_pk(float a, float b, uint32_t *hi, uint32_t *lo) {
    const bf16x2 h = __builtin_convertvector((f32x2){a, b}, bf16x2);
    const uint32_t w = __builtin_bit_cast(uint32_t, h);
    *hi = w;
    *lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a - bf16_lo(w), b - bf16_hi(w)}, bf16x2));
}

/* Bits 15 and 31: whether the low and the high bf16 of a word are not finite. */
__device__ __forceinline__ uint32_t nonfinite2(uint32_t w) {
    return ((w & 0x7f807f80u) + 0x00800080u) & 0x80008000u;
}

__device__ __forceinline__ f32x16 mfma32(i32x4 a, i32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

/* Keys (part 0) or values (part 1) of 128 cache rows and one head: 128 x 128
 * x 512, four multiplying waves (2 x 2, 64 x 64 each) and four loading, a
 * ring of XNS chunks of 64 latent values; two blocks per CU, one's products
 * and output beside the other's loads.  16 heads: one prompt of 2,048 rows
 * (512 blocks, two per CU) 20 us; prompts of 1,364 and 683 rows (544 blocks:
 * 32 run in a second turn) 24.  Which operand comes first is a matter of
 * addresses: as a choice at each product it took a branch each and spilled 10
 * registers (23 and 33 us).  In that form one block per CU with four chunks in
 * flight took 31 us for the 2,048 rows, and the pairs stored from the
 * accumulators, 8 bytes at a time, 32: they leave through LDS in whole lines.
 * Rows at or past the tile's length are zeros: a value of an unwritten cache
 * row must not meet a probability of zero as an infinity. */
#define XNS MM_MLA_XNS
extern "C" __global__ __launch_bounds__(512, 4) void mm_mla_expand(mm_mla_expand_args a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t xlds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.x, part = blockIdx.y;
    const int32_t *tl = a.tiles + 4 * blockIdx.z;      /* slot, first key, keys of the sequence, first block */
    const int slot = tl[0], key0 = tl[1], len = tl[2], blk0 = tl[3];
    const uint32_t lds0 = lds_addr(xlds);
    constexpr int SB = 2 * 16384, NC = KVL / 64;
    if (wave >= 4) {
        const int lw = wave - 4, rows = min(len - key0, 128);
        const rsrc_t rx = raw_rsrc(a.cache + ((size_t)slot * a.seq_stride + key0) * KVD, (uint32_t)rows * KVD * 2);
        const rsrc_t rw = raw_rsrc(a.kv_b + ((size_t)h * 2 * XD + part * XD) * KVL, XD * KVL * 2);
        uint32_t xo[4], wo[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int R = 8 * (4 * lw + u) + (lane >> 3), p = 16 * ((lane & 7) ^ ((R >> 1) & 7));
            xo[u] = R < rows ? (uint32_t)(R * KVD * 2 + p) : 0xFFFFF000u;   /* past the range: zeros */
            wo[u] = (uint32_t)(R * KVL * 2 + p);
        }
        auto issue = [&](int c, int st) {
            const uint32_t sb = lds0 + (uint32_t)(st * SB + 4 * lw * 1024);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                lds_dma16_buf(xo[u] + (uint32_t)(128 * c), rx, sb + u * 1024);
                lds_dma16_buf(wo[u] + (uint32_t)(128 * c), rw, sb + 16384 + u * 1024);
            }
        };
#pragma unroll
        for (int s = 0; s < XNS - 1; s++) issue(s, s);
#pragma unroll
        for (int c = 0; c < NC; c++) {                 /* one barrier per chunk: chunk c has landed */
            VMCNT_WAIT(8 * (XNS - 2));
            __builtin_amdgcn_s_barrier();
            issue(min(c + XNS - 1, NC - 1), (c + XNS - 1) % XNS);   /* chunk c - 1's slot */
        }
        VMCNT_WAIT(0);
    } else {
        const int wm = wave >> 1, wn = wave & 1, c32 = lane & 31, hi = lane >> 5;
        /* the first operand's rows are a result's registers, the second's its
         * lanes: keys have lanes for keys (the weights first), values lanes for
         * dims (the latent rows first) -- one code for both, by the addresses */
        const uint32_t ax = (uint32_t)(64 * wm * 128), aw = (uint32_t)(16384 + 64 * wn * 128);
        const uint32_t a0 = part == 0 ? aw : ax, a1 = part == 0 ? ax : aw;
        f32x16 acc[2][2] = {};                             /* [first operand's tile][second's] */
#pragma unroll
        for (int c = 0; c < NC; c++) {
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const uint32_t sb = lds0 + (uint32_t)(c % XNS * SB) + c32 * 128;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const uint32_t p = 16 * ((2 * s + hi) ^ ((c32 >> 1) & 7));
                i32x4 f0[2], f1[2];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    f0[t] = *(lds_c4)(sb + p + a0 + 32 * t * 128);
                    f1[t] = *(lds_c4)(sb + p + a1 + 32 * t * 128);
                }
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int v = 0; v < 2; v++) acc[u][v] = mfma32(f0[u], f1[v], acc[u][v]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        /* the pairs into LDS as they lie in memory (the ring is free: every
         * load landed, every read done), then out in whole lines */
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int v = 0; v < 2; v++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                    uint32_t h0, h1, l0, l1;
                    split_pk(acc[u][v][4 * g], acc[u][v][4 * g + 1], &h0, &l0);
                    split_pk(acc[u][v][4 * g + 2], acc[u][v][4 * g + 3], &h1, &l1);
                    /* key c32 of tile v, dims 64 wn + 32 u + 8 g + 4 hi .. + 3 */
                    const uint32_t ok = (2 * wm + v) * 2 * XT + c32 * 256 + 16 * (((64 * wn + 32 * u) / 8 + g) ^ (c32 & 15)) + 8 * hi;
                    /* dim d, keys 8 g + 4 hi .. + 3 of tile u */
                    const int d = 64 * wn + 32 * v + c32;
                    const uint32_t ov = (2 * wm + u) * 2 * XT + d * 64 + 16 * ((2 * (g >> 1) + hi) ^ ((d >> 2) & 3)) + 8 * (g & 1);
                    const uint32_t o = part == 0 ? ok : ov;
                    *(u32x2 *)(xlds + o) = (u32x2){h0, h1};
                    *(u32x2 *)(xlds + o + XT) = (u32x2){l0, l1};
                }
    }
    if (wave >= 4) __builtin_amdgcn_s_barrier();
    __syncthreads();
    /* key block b of the tile: 16 KB of pairs, two waves each */
    const int b = wave >> 1, kb = key0 / XB + b;       /* key0 is a multiple of 128 */
    if (kb * XB >= len) return;
    uint8_t *dst = a.kv + ((size_t)(blk0 + kb) * a.NH + h) * XBLK + part * 2 * XT + (wave & 1) * XT;
    const uint8_t *src = xlds + b * 2 * XT + (wave & 1) * XT;
    u32x4 v[XT / 1024];
    uint32_t any = 0;
#pragma unroll
    for (int u = 0; u < XT / 1024; u++) {
        v[u] = *(const u32x4 *)(src + u * 1024 + lane * 16);
        any |= nonfinite2(v[u].x) | nonfinite2(v[u].y) | nonfinite2(v[u].z) | nonfinite2(v[u].w);
    }
    if (part == 1) {
        /* zero times a later key's infinity or NaN must not reach the rows
         * before it: such a value is stored as zero (its low part is no number
         * either) and its key's bit set, for the rows that do see it */
        uint32_t keys = 0;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(any != 0) != 0, 0)) {
#pragma unroll 1
            for (int u = 0; u < XT / 1024; u++) {
                const int d = 16 * u + (lane >> 2), p = (lane & 3) ^ ((d >> 2) & 3);
                u32x4 w = *(const u32x4 *)(src + u * 1024 + lane * 16);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t n = nonfinite2(w[i]);
                    w[i] &= ~((n >> 15) * 0xffffu);
                    keys |= ((n >> 15 & 1u) | (n >> 30 & 2u)) << (16 * (p >> 1) + 4 * (p & 1) + 2 * (i & 1) + 8 * (i >> 1));
                }
                *(u32x4 *)(dst + u * 1024 + lane * 16) = w;
            }
#pragma unroll
            for (int off = 1; off < MM_WAVE; off <<= 1) keys |= (uint32_t)__shfl_xor((int)keys, off, MM_WAVE);
        }
        if (lane == 0 && (wave & 1) == 0) a.nf[(size_t)(blk0 + kb) * a.NH + h] = keys;
        if (keys) return;
    }
#pragma unroll
    for (int u = 0; u < XT / 1024; u++) *(u32x4 *)(dst + u * 1024 + lane * 16) = v[u];
}

/* Flash attention of 64 rows (consecutive positions of one sequence) and one
 * head per block: four waves, wave w rows 32 (w % 2) .. + 31 over the even
 * (w < 2) or odd 32-key blocks, merged through LDS at the end.  One stage of
 * two key blocks (72 KB: K and V pairs, the cache's k_pe); two blocks share a
 * CU, and one's products cover the other's loads.  Scores transposed (K as the first
 * operand): a lane holds 16 of a block's 32 keys of one row, so a row's
 * maximum takes one exchange between lane halves and the probabilities are
 * the second operand of the value product as they stand.  Lazy rescaling as
 * in mm_mla_attn.
 *
 * Bound by the MFMAs of the longest rows: 72 of 32 cycles per key block and
 * wave.  Two prompts of 1,364 and 683 rows: 63 us per layer, one of 2,048: 88
 * (absorbed, with its query and W_UV products: 286 and 420).  128-row blocks
 * of eight waves, one per CU, with two whole steps in LDS took 84 and 114:
 * a CU's one long block set the time.  With one load phase per step instead of
 * keys and values in turn: 71 and 102. */
#define XTAU 11.0f                /* RESCALE_TAU in units of ln 2 */
#define XSTAGE (XBLK + XB * 128)  /* one key block: K, V, k_pe */
static_assert(2 * XSTAGE == MM_MLA_XATTN_LDS, "one stage of two key blocks");
extern "C" __global__ __launch_bounds__(256, 2) void mm_mla_attn_expanded(mm_mla_xattn_args a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t xlds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c32 = lane & 31, hi = lane >> 5, wr = wave & 1, kw = wave >> 1;
    /* tiles in the host's order, a tile's heads next to each other: head h of
     * every tile of a sequence runs on XCD h % 8 */
    const int h = blockIdx.x % a.NH;
    const int32_t *tl = a.tiles + 5 * (blockIdx.x / a.NH);
    const int row0 = tl[0], nrows = tl[1], pos0 = tl[2], slot = tl[3], blk0 = tl[4];
    const int nblk = (pos0 + nrows + XB - 1) / XB;     /* key blocks of the tile's last row */
    const int nst = (nblk + 1) / 2;
    const uint32_t lds0 = lds_addr(xlds);

    /* this wave's share of a step: half of its key block's keys (and k_pe rows)
     * or values.  The values load during the scores' products and the next
     * step's keys during the values', each into the place that the barrier
     * before has freed. */
    const rsrc_t rp = raw_rsrc(a.cache + (size_t)slot * a.seq_stride * KVD, (uint32_t)(pos0 + nrows) * KVD * 2);
    const uint32_t sb = lds0 + (uint32_t)(kw * XSTAGE);
    auto issue = [&](int j, bool values) {
        const int kb = min(2 * j + kw, nblk - 1);
        const rsrc_t rk = raw_rsrc(a.kv + ((size_t)(blk0 + kb) * a.NH + h) * XBLK, XBLK);
        const uint32_t o = (uint32_t)((values ? 2 * XT : 0) + wr * XT);
#pragma unroll
        for (int u = 0; u < 8; u++) lds_dma16_buf(o + (uint32_t)(u * 1024 + lane * 16), rk, sb + o + u * 1024);
        if (values) return;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int r = 8 * (2 * wr + u) + (lane >> 3);   /* rows past the sequence: zeros */
            lds_dma16_buf((uint32_t)((kb * XB + r) * KVD + KVL) * 2 + 16 * ((lane & 7) ^ ((r >> 1) & 7)), rp,
                          sb + XBLK + (2 * wr + u) * 1024);
        }
    };

    issue(0, false);
    /* Q of the wave's rows (row l % 32, dims 16 s + 8 (l / 32) .. + 7) as pairs */
    const int myrow = 32 * wr + c32;
    const float *qp = a.q + ((size_t)(row0 + min(myrow, nrows - 1)) * a.NH + h) * (XD + MM_MLA_QKR) + 8 * hi;
    i32x4 qh[12], ql[12];
#pragma unroll
    for (int s = 0; s < 12; s++) {
        const f32x4 x0 = *(const f32x4 *)(qp + 16 * s), x1 = *(const f32x4 *)(qp + 16 * s + 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t vh, vl;
            split_pk(j < 2 ? x0[2 * j] : x1[2 * j - 4], j < 2 ? x0[2 * j + 1] : x1[2 * j - 3], &vh, &vl);
            qh[s][j] = (int)vh;
            ql[s][j] = (int)vl;
        }
    }
    const int pos = pos0 + min(myrow, nrows - 1);      /* this lane's row */
    const int wlast = pos0 + min(32 * wr + 31, nrows - 1), wfirst = pos0 + min(32 * wr, nrows - 1);
    /* the first key with a value that is not finite (mm_mla_expand stored
     * zeros): the rows that see it give NaN, as its infinity or NaN would */
    int kbad = INT32_MAX;
    for (int b0 = 0; b0 < nblk && kbad == INT32_MAX; b0 += MM_WAVE) {
        const uint32_t nf = b0 + lane < nblk ? a.nf[(size_t)(blk0 + b0 + lane) * a.NH + h] : 0;
        const uint64_t any = __builtin_amdgcn_ballot_w64(nf != 0);
        if (any) {
            const int f = __builtin_ctzll(any);
            kbad = XB * (b0 + f) + __builtin_ctz(__builtin_amdgcn_readlane((int)nf, f));
        }
    }
    const float scale2 = a.scale * 1.44269504088896341f;   /* scores in units of ln 2: e^x is one v_exp */
    float m = -INFINITY, l = 0.0f;
    f32x16 O[4] = {};
    const int swk = c32 & 15, swp = (c32 >> 1) & 7, swv = (c32 >> 2) & 3;
    VMCNT_WAIT(0);
    __builtin_amdgcn_s_barrier();                      /* every wave's part of the first keys */
    asm volatile("" ::: "memory");
    for (int j = 0; j < nst; j++) {
        issue(j, true);
        const int k0 = (2 * j + kw) * XB;
        const bool on = k0 <= wlast && 2 * j + kw < nblk;   /* uniform: some row of the wave sees a key */
        i32x4 ph[2], pl[2];
        f32x16 sa = {};
        if (on) {
            f32x16 sc = {};                            /* sa: hi * hi, sc: the smaller products */
            const uint32_t kr = sb + c32 * 256, pr = sb + XBLK + c32 * 128;
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const i32x4 kh = *(lds_c4)(kr + 16 * ((2 * s + hi) ^ swk));
                const i32x4 kl = *(lds_c4)(kr + XT + 16 * ((2 * s + hi) ^ swk));
                sa = mfma32(kh, qh[s], sa);
                sc = mfma32(kl, qh[s], sc);
                sc = mfma32(kh, ql[s], sc);
                sc = mfma32(kl, ql[s], sc);
            }
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const i32x4 kp = *(lds_c4)(pr + 16 * ((2 * s + hi) ^ swp));
                sa = mfma32(kp, qh[8 + s], sa);
                sc = mfma32(kp, ql[8 + s], sc);
            }
#pragma unroll
            for (int i = 0; i < 16; i++) sa[i] += sc[i];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        VMCNT_WAIT(0);
        __builtin_amdgcn_s_barrier();                  /* the keys read, every wave's values there */
        asm volatile("" ::: "memory");
        issue(j + 1 < nst ? j + 1 : j, false);         /* (after the last step its keys again, read by nobody) */
        if (on) {
            float mx = -INFINITY;
            if (k0 + XB - 1 <= wfirst) {               /* uniform: no masked key */
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    sa[i] *= scale2;
                    mx = fmaxf(mx, sa[i]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int key = k0 + 8 * (i >> 2) + 4 * hi + (i & 3);
                    sa[i] = key <= pos ? sa[i] * scale2 : -INFINITY;
                    mx = fmaxf(mx, sa[i]);
                }
            }
            if (__builtin_amdgcn_ballot_w64(mx > m + XTAU)) {
                mx = fmaxf(mx, __shfl_xor(mx, 32, MM_WAVE));
                const float mn = fmaxf(m, mx);
                const float cr = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
                l *= cr;
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int i = 0; i < 16; i++) O[t][i] *= cr;
                m = mn;
            }
            const float mz = m == -INFINITY ? 0.0f : m;   /* rows with no key yet: probabilities 0 */
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float p0 = __builtin_amdgcn_exp2f(sa[8 * s + 2 * i] - mz);
                    const float p1 = __builtin_amdgcn_exp2f(sa[8 * s + 2 * i + 1] - mz);
                    l += p0 + p1;
                    uint32_t vh, vl;
                    split_pk(p0, p1, &vh, &vl);
                    ph[s][i] = (int)vh;
                    pl[s][i] = (int)vl;
                }
            const uint32_t vr = sb + 2 * XT + c32 * 64;
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const i32x4 vh = *(lds_c4)(vr + t * 2048 + 16 * ((2 * s + hi) ^ swv));
                    const i32x4 vl = *(lds_c4)(vr + XT + t * 2048 + 16 * ((2 * s + hi) ^ swv));
                    O[t] = mfma32(vh, ph[s], O[t]);
                    O[t] = mfma32(vl, ph[s], O[t]);
                    O[t] = mfma32(vh, pl[s], O[t]);
                    O[t] = mfma32(vl, pl[s], O[t]);
                }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        VMCNT_WAIT(0);
        __builtin_amdgcn_s_barrier();                  /* the values read, every wave's next keys there */
        asm volatile("" ::: "memory");
    }
    asm volatile("" ::: "memory");
    if (pos >= kbad) l = __builtin_nanf("");

    /* the odd blocks' (m, l, O) to the wave of the same rows; both halves of a
     * row's lanes hold the same m, each its own share of l */
    float *ex = (float *)xlds + (size_t)wr * 66 * MM_WAVE + lane;
    if (kw == 1) {
        ex[0] = m;
        ex[MM_WAVE] = l;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) ex[(2 + 16 * t + i) * MM_WAVE] = O[t][i];
    }
    __syncthreads();
    if (kw == 1 || myrow >= nrows) return;             /* a row's two lanes leave together */
    const float m1 = ex[0], mm = fmaxf(m, m1);
    const float w0 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mm);
    const float w1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mm);
    l = l * w0 + ex[MM_WAVE] * w1;
    l += __shfl_xor(l, 32, MM_WAVE);
    const float inv = 1.0f / l, f0 = w0 * inv, f1 = w1 * inv;
    float *out = a.ctx + ((size_t)(row0 + myrow) * a.NH + h) * XD + 4 * hi;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; i++)
                v[i] = O[t][4 * g + i] * f0 + ex[(2 + 16 * t + 4 * g + i) * MM_WAVE] * f1;
            *(f32x4 *)(out + 32 * t + 8 * g) = v;
        }
}
