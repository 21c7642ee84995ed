// Prompt prefill at large M: the reference runs the prompt one token per
// forward (src/speculative.c:100-107, src/model.c:450-616); here a chunk of
// up to a few thousand prompt rows runs as one batch.
//
//   vx_pf_panel_kernel   rows, their RMSNorm or SwiGLU as the GEMM's operand
//   vx_pf_gemm_kernel    Y = X W^T (+ R) for M rows, compute-bound MFMA tiles
//   vx_pf_rope_kv_kernel RoPE of q|k rows and the k/v cache store (fp32 rows)
//   vx_pf_swiglu_kernel  h = |silu(g)| < thr ? 0 : silu(g) * u
//
// GEMM arithmetic.  A Q4_0/Q8_0 block is d * q with q = s - 8 (resp. the int8)
// exact in fp16 and d an fp16 scale.  Activations are split into two fp16
// parts, x_hi + x_lo (22 bits).  Per block of 32 the MFMAs sum x_lo q and
// x_hi q from zero, and one fp32 fma per output adds d times that block sum to
// the running sum: two MFMA products per weight and a VALU fma that runs in
// their shadow.  (The scheme before it folded d into the weights as an exact
// fp16 pair and took three products, x_hi w_hi + x_lo w_hi + x_hi w_lo, with
// no rescaling: 1.5 times the MFMA work, and its one long fp32 chain over K
// was three times as far from the 64-bit result: 6.6e-7 against 2.3e-7 at
// K = 4096.)
#include "vxh_internal.h"
#include "vxh_gemm_core.h"

#define PF_BM 64                 // activation rows per workgroup (a row group of the panel)
#define PF_MT (PF_BM / 32)       // 32-row MFMA tiles per workgroup
#define PF_STAGE (PF_MT * 2 * 2 * 2 * 64)   // A units (8 fp16) of one block pair: [mt][blk][s][hl][lane]

typedef uint32_t vx_u32x4 __attribute__((ext_vector_type(4)));

struct vx_pf_args {
    const uint4 *wq;
    const uint32_t *wd;
    int n_tiles, n_pairs;
    const uint4 *px;   // rows panel (vxh_rows_panel): [row group][pair][PF_STAGE units]
    const float *rs;   // [M] power-of-two row scales of the panel
    int M;
    float *y;
    int ldy, n_out;
    const float *r;
    int ldr;
    float scale;
};

// Wavefront tile: 32 MT activation rows x 32 NT weight rows (MT = 2, or 1 in
// a last row group of <= 32 rows).  Workgroup = CW x KS wavefronts: CW of
// them side by side over the weight tiles, KS over the K range (block pairs
// p with p % KS = ks), whose sums meet in LDS at the end in a fixed order.
// Per step the workgroup copies the activation stages of its next KS pairs
// from the rows panel into LDS (already in MFMA operand order), double-
// buffered with one barrier per step; with CW = 1 no two wavefronts share a
// stage and each loads its operands straight into registers.
//
// Bound by the matrix cores once the chip is full (launches of the GEMM alone,
// back to back): 2048 x 22016 x 4096 Q4_0 1714 -> 670 us (2 products: 1.10
// PFLOP/s, 95% of what a large library fp16 product reaches here), 512 x 22016 x
// 4096 441 -> 191 us.  64 x 64 per
// wavefront because an operand read from LDS then feeds two MFMAs (at 64 x 32
// LDS reads took as long as the products); the block sums of one tile are
// scaled and added between the MFMAs of the next, so neither pipe waits.
template <int QT, int NT, int CW, int KS, int MT>
__device__ __forceinline__ void vx_pf_gemm_body(const vx_pf_args &a, int rg, int cg, vx_u32x4 *lds, float *s_rs)
{
    constexpr int WPP = QT == 2 ? 1 : 2;
    constexpr int RING = QT == 2 && CW != 2 ? 3 : 2;   // weight pairs in flight (register room)
    constexpr bool DIRECT = CW == 1;
    constexpr int NTHR = 64 * CW * KS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cw = wave % CW, ks = wave / CW;
    const int T0 = (cg * CW + cw) * NT;
    const int c = lane & 31, h = lane >> 5;
    const uint32_t magic = 0x64006400u;
    const vx_u32x4 *wp[NT];
    const uint32_t *sp[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int Tc = min(T0 + nt, a.n_tiles - 1);
        wp[nt] = (const vx_u32x4 *)a.wq + (size_t)Tc * a.n_pairs * WPP * 64 + lane;
        sp[nt] = a.wd + (size_t)Tc * a.n_pairs * 32 + c;
    }
    const vx_u32x4 *xg = (const vx_u32x4 *)a.px + (size_t)rg * a.n_pairs * PF_STAGE;

    vx_u32x4 w[RING][NT][WPP];
    uint32_t sc[RING][NT];
    auto load_w = [&](int i, int p) {
        const int pc = min(p, a.n_pairs - 1);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
#pragma unroll
            for (int q = 0; q < WPP; q++) w[i][nt][q] = wp[nt][((size_t)pc * WPP + q) * 64];
            sc[i][nt] = sp[nt][(size_t)pc * 32];
        }
    };
    // LDS staging: XU units of a step per thread
    constexpr int XU = DIRECT ? 1 : KS * PF_STAGE / NTHR;
    vx_u32x4 xa[XU];
    auto load_x = [&](int st) {
#pragma unroll
        for (int j = 0; j < XU; j++) {
            const int u = threadIdx.x + NTHR * j;
            const int p = min(st * KS + u / PF_STAGE, a.n_pairs - 1);
            xa[j] = xg[(size_t)p * PF_STAGE + u % PF_STAGE];
        }
    };
    auto store_x = [&](vx_u32x4 *buf) {
#pragma unroll
        for (int j = 0; j < XU; j++) buf[threadIdx.x + NTHR * j] = xa[j];
    };
    // DIRECT: the operands of one pair in registers, refilled block by block
    vx_half8 xf[2][MT][2][2];   // [blk][mt][s][hi, lo]
    auto load_f = [&](int blk, int p) {
        const vx_u32x4 *xp = xg + (size_t)min(p, a.n_pairs - 1) * PF_STAGE + lane;
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int hl = 0; hl < 2; hl++)
                    xf[blk][mt][s][hl] = __builtin_bit_cast(vx_half8, xp[(((mt * 2 + blk) * 2 + s) * 2 + hl) * 64]);
    };

    // K whole: the row scales to LDS, for the epilogue (behind the first barrier)
    const int m0 = rg * PF_BM;
    if (KS == 1 && threadIdx.x < PF_BM) s_rs[threadIdx.x] = a.rs[min(m0 + (int)threadIdx.x, a.M - 1)];
    vx_f32x16 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[nt][mt] = vx_f32x16{};
    // block products of the last tile issued and the scale they wait for
    vx_f32x16 S = vx_f32x16{};
    float Sd = 0.0f;
    auto add4 = [&](vx_f32x16 &P, int r0) {
#pragma unroll
        for (int r = r0; r < r0 + 4; r++) P[r] = fmaf(Sd, S[r], P[r]);
    };
    const int n_steps = (a.n_pairs + KS - 1) / KS;
#pragma unroll
    for (int i = 0; i < RING; i++) load_w(i, i * KS + ks);
    if constexpr (DIRECT) {
        load_f(0, ks);
        load_f(1, ks);
    } else {
        load_x(0);
        store_x(lds);
        if (n_steps > 1) load_x(1);
        __syncthreads();
    }
    for (int s0 = 0; s0 < n_steps; s0 += RING) {
#pragma unroll
        for (int i = 0; i < RING; i++) {
            const int st = s0 + i, p = st * KS + ks;
            if (st >= n_steps) break;
            const vx_u32x4 *cur = lds + ((st & 1) * KS + ks) * PF_STAGE;
            if constexpr (!DIRECT) {
                // the next step's activations into the other buffer (free
                // since the barrier that ended step st-1), then the one after
                // in flight
                if (st + 1 < n_steps) {
                    store_x(lds + ((st + 1) & 1) * KS * PF_STAGE);
                    if (st + 2 < n_steps) load_x(st + 2);
                }
            }
            if (KS == 1 || p < a.n_pairs) {
#pragma unroll
                for (int blk = 0; blk < 2; blk++) {
                    vx_half8 A[MT][2][2];
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
#pragma unroll
                        for (int s = 0; s < 2; s++)
#pragma unroll
                            for (int hl = 0; hl < 2; hl++)
                                A[mt][s][hl] = DIRECT ? xf[blk][mt][s][hl]
                                                      : __builtin_bit_cast(vx_half8, cur[(((mt * 2 + blk) * 2 + s) * 2 +
                                                                                          hl) * 64 + lane]);
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) {
                        vx_half8 b0, b1;
                        if constexpr (QT == 2) {
                            const vx_u32x4 v = w[i][nt][0];
                            b0 = vx_unpack_q4(blk ? v.z : v.x, magic);
                            b1 = vx_unpack_q4(blk ? v.w : v.y, magic);
                        } else {
                            const vx_u32x4 v = w[i][nt][blk];
                            b0 = vx_unpack_q8(v.x, v.y, magic);
                            b1 = vx_unpack_q8(v.z, v.w, magic);
                        }
                        const float d = vx_half_bits_to_float((sc[i][nt] >> (16 * blk)) & 0xFFFFu);
#pragma unroll
                        for (int mt = 0; mt < MT; mt++) {
                            // this tile's block products; the tile before it
                            // is scaled and added in the MFMAs' shadow
                            vx_f32x16 N = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[mt][0][1], b0, vx_f32x16{}, 0, 0, 0);
                            const vx_half8 first = A[mt][0][1];
                            constexpr int TILES = NT * MT;
                            vx_f32x16 &P = acc[((nt * MT + mt + TILES - 1) % TILES) / MT][(mt + MT - 1) % MT];
                            add4(P, 0);
                            N = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[mt][1][1], b1, N, 0, 0, 0);
                            add4(P, 4);
                            N = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[mt][0][0], b0, N, 0, 0, 0);
                            add4(P, 8);
                            N = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[mt][1][0], b1, N, 0, 0, 0);
                            add4(P, 12);
                            // an MFMA that starts a chain must not write over its
                            // own sources: keep them live past it
                            asm volatile("" : "+v"(N) : "v"(first), "v"(b0));
                            S = N;
                            Sd = d;
                        }
                    }
                    if constexpr (DIRECT) load_f(blk, p + KS);
                }
                load_w(i, p + RING * KS);
            }
            if constexpr (!DIRECT) __syncthreads();
        }
    }

#pragma unroll
    for (int r = 0; r < 16; r += 4) add4(acc[NT - 1][MT - 1], r);
    // Output (nt, mt, r) of a lane.  Row scales (with K whole from LDS) and
    // residual elements of a batch are read before its first store: behind a
    // store that may alias them each would be a round trip of its own (2048 x
    // 4096 x 4096 with the residual 161 -> 138 us, 2048 x 22016 x 128 80 -> 67)
    auto row_of = [&](int mt, int r) { return mt * 32 + 8 * (r / 4) + 4 * h + (r % 4); };
    auto col_of = [&](int nt) { return (T0 + nt) * 32 + c; };
    auto resid = [&](int nt, int mt, int r) {
        return a.r[(size_t)min(m0 + row_of(mt, r), a.M - 1) * a.ldr + min(col_of(nt), a.n_out - 1)];
    };
    auto put = [&](int nt, int mt, int r, float sum, float rsv, float rv) {
        const int n = col_of(nt), row = m0 + row_of(mt, r);
        if (n >= a.n_out || row >= a.M) return;
        const float v = (sum * (KS == 1 ? s_rs[row_of(mt, r)] : rsv)) * a.scale;   // the row scale is a power of two
        a.y[(size_t)row * a.ldy + n] = a.r ? rv + v : v;
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                float rv[16];
#pragma unroll
                for (int r = 0; r < 16; r++) rv[r] = a.r ? resid(nt, mt, r) : 0.0f;
#pragma unroll
                for (int r = 0; r < 16; r++) put(nt, mt, r, acc[nt][mt][r], 0.0f, rv[r]);
            }
    } else {
        // [ks][cw][register][lane]; the last step's barrier freed the stages
        constexpr int R = NT * MT * 16, RK = R / KS;
        static_assert(R % KS == 0, "registers of a tile over the K slices");
        float *red = (float *)lds;
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int r = 0; r < 16; r++) red[(wave * R + (nt * MT + mt) * 16 + r) * 64 + lane] = acc[nt][mt][r];
        __syncthreads();
        float rsv[RK], rv[RK];
#pragma unroll
        for (int j = 0; j < RK; j++) {
            const int reg = ks * RK + j;
            rsv[j] = a.rs[min(m0 + row_of((reg / 16) % MT, reg % 16), a.M - 1)];
            rv[j] = a.r ? resid(reg / (16 * MT), (reg / 16) % MT, reg % 16) : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < RK; j++) {
            const int reg = ks * RK + j;
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < KS; k++) v += red[((k * CW + cw) * R + reg) * 64 + lane];
            put(reg / (16 * MT), (reg / 16) % MT, reg % 16, v, rsv[j], rv[j]);
        }
    }
}

// LDS units of a workgroup: two steps' stages, or the K slices' sums
template <int NT, int CW, int KS>
static constexpr int vx_pf_lds_units()
{
    const int stage = CW == 1 ? 1 : 2 * KS * PF_STAGE, red = KS == 1 ? 0 : KS * CW * NT * PF_MT * 16 * 16;
    return stage > red ? stage : red;
}

template <int QT, int NT, int CW, int KS>
__global__ __launch_bounds__(64 * CW *KS, 2) void vx_pf_gemm_kernel(vx_pf_args a, int n_cg, int n_rg)
{
    __shared__ vx_u32x4 lds[vx_pf_lds_units<NT, CW, KS>()];
    __shared__ float s_rs[KS == 1 ? PF_BM : 1];
    // workgroup id -> tile: ids go round the 8 XCDs, so every XCD takes a
    // contiguous run of tiles, in blocks of 8 row groups: the row groups of a
    // block share weight tiles and the columns share activation stages in L2
    const int nb = n_cg * n_rg, x = blockIdx.x % 8, per = nb / 8, rem = nb % 8;
    const int id = x * per + min(x, rem) + blockIdx.x / 8;
    const int sup = id / (8 * n_cg), rs = min(8, n_rg - 8 * sup), in = id - sup * 8 * n_cg;
    const int rg = 8 * sup + in % rs, cg = in / rs;
    if (a.M - rg * PF_BM > 32)
        vx_pf_gemm_body<QT, NT, CW, KS, 2>(a, rg, cg, lds, s_rs);
    else
        vx_pf_gemm_body<QT, NT, CW, KS, 1>(a, rg, cg, lds, s_rs);
}

template <int QT, int NT, int CW, int KS>
static int vx_pf_gemm_launch(const vx_pf_args &a, hipStream_t s)
{
    const int n_cg = (a.n_tiles + NT * CW - 1) / (NT * CW), n_rg = (a.M + PF_BM - 1) / PF_BM;
    vx_pf_gemm_kernel<QT, NT, CW, KS><<<(unsigned)(n_cg * n_rg), 64 * CW * KS, 0, s>>>(a, n_cg, n_rg);
    VXH_LAUNCHED();
    return VXH_OK;
}

// Which split: the estimated time in rounds of workgroups over the 256 CUs.
// Each weight is the time of one round relative to the others' at K = 4096
// (from there all splits scale with K alike), as measured with an epilogue that
// loaded element by element; with today's they are 3.1 (a last round 2.0), 1.0,
// 0.55 and 0.36.  Weights refitted to 323 measured points chose splits 0.1%
// faster on average, so these stay.  us back to back, Q4_0, before the K splits
// and now:
//   64 x 256, K whole: two workgroups to a CU; a full round of 512 takes 4.05,
//     a last one of up to 256 (one to a CU) 2.  The best rate per tile, but
//     M = 512, N = 4096 would leave half the CUs empty.
//   64 x 128, K over 4: 1.1 a round.  512 x 4096 x 4096 100 -> 42 (78 with K
//     whole); 2048 x 4096 x 4096 160, where K whole takes 132.
//   64 x 64, K over 8: 0.65 a round.  512 x 2048 x 5632 135 -> 32 (51 with
//     64 x 128); 128 x 22016 x 4096 150 -> 62 (78 with K whole).
//   64 x 32, K over 8: 0.38 a round.  77 x 4096 x 11008 Q8_0 260 -> 35 (55
//     with 64 x 64); 48 x 4096 x 4096 90 -> 12.7.
template <int QT>
static int vx_pf_gemm(const vx_pf_args &a, hipStream_t s)
{
    const long n_rg = (a.M + PF_BM - 1) / PF_BM;
    auto groups = [&](int tiles) { return n_rg * ((a.n_tiles + tiles - 1) / tiles); };
    auto rounds = [&](long n) { return (float)((n + 255) / 256); };
    const long n0 = groups(8), rest = n0 % 512;
    // Below K = 4096 a round has a part that does not shrink with K (output
    // rows, join of the K slices).  Fitted to 100 shapes of K = 32 to 2048: the
    // split taken is within 11% of the best one at each.  512 x 11008 x 128 with
    // K whole 15.0 us, by 64 x 128 (its split at 4096) 18.5; 700 x 6000 x 128
    // with K whole 14.6, by 64 x 64 23.9.
    const float k = fminf((float)a.n_pairs / 64.0f, 1.0f);
    auto weight = [&](float at4096, float fixed) { return k < 1.0f ? fixed + (at4096 - fixed) * k : at4096; };
    const float full = weight(4.05f, 0.2f), half = weight(2.0f, 0.29f);
    const float t0 = full * (float)(n0 / 512) + (rest == 0 ? 0.0f : rest <= 256 ? half : full);
    const float t1 = weight(1.1f, 0.15f) * rounds(groups(4)), t2 = weight(0.65f, 0.1f) * rounds(groups(2)),
                t3 = weight(0.38f, 0.07f) * rounds(groups(1));
    const float best = fminf(fminf(t0, t1), fminf(t2, t3));
    if (t0 == best) return vx_pf_gemm_launch<QT, 2, 4, 1>(a, s);
    if (t1 == best) return vx_pf_gemm_launch<QT, 2, 2, 4>(a, s);
    if (t2 == best) return vx_pf_gemm_launch<QT, 2, 1, 8>(a, s);
    return vx_pf_gemm_launch<QT, 1, 1, 8>(a, s);
}

// Rows panel: fp32 rows as the GEMM's LDS stages.  Unit u of a (row group
// rg, pair p) stage, u = ((mt*2 + blk)*2 + s)*128 + ln, holds row 64 rg + 32 mt
// + ln % 32, elements 64 p + 32 blk + 16 (ln/32) + 8 s .. + 7, as hi = fp16(x')
// and (64 units further) lo = fp16(x' - hi).  x' = x 2^-e with e from the row's
// largest magnitude (vx_row_scale: |x'| < 1), so no element overflows fp16 and
// a row of small values keeps the low parts' bits; rs[row] = 2^e goes back in
// in the GEMM epilogue, exactly.  Rows past M (up to the 64-row group) and
// columns past K are zeros.
//
// The rows are x[M][ldx] as they are (PF_ROWS), their RMSNorm (PF_RMS), or the
// SwiGLU with the FFN gate-skip (src/model.c:582-585) of the interleaved
// gate/up product (PF_SWIGLU; 16 gate then 16 up columns per tile of 32).
//
// Bound by memory.  A workgroup takes PR rows, WPR wavefronts each.  Many
// rows: 8 and 2, as the 16-byte units of 8 rows are one 128-byte line; with a
// workgroup per row the rows of a line go to 8 XCDs, whose L2s each write back
// a part of it (2048 x 4096: 33 -> 19 us; norm and panel 50 -> 21; SwiGLU and
// panel of 2048 x 11008 153 -> 70).  Few rows: a workgroup each (77 x 11008
// 7.4 us, 22 with 8 rows: only 16 workgroups), of 4 wavefronts up to their
// register window of 12288 columns, of 16 beyond (SwiGLU of 17 x 18944 21.0 ->
// 12.1 us, 512 x 18944 50 -> 42), and SwiGLU rows of 16 from 8192 columns on
// while a CU gets two of them or fewer (17 x 11008 10.8 -> 8.8 us, 512 x 11008
// 28.4 -> 26.4; 1000 x 12288 52.6 against 55.9).  A row stays in registers, up
// to KEEP groups of 8 columns per lane (2 up to 4096 columns, as groups past
// the row's end cost their loads: norm of 1000 x 1024 8.4 -> 6.6 us); what is
// left is read again (the sum of squares and the maximum come first), SwiGLU
// evaluated again.
enum { PF_ROWS = 0, PF_RMS = 1, PF_SWIGLU = 2 };

template <int SRC, int KEEP, int PR, int WPR>
__global__ __launch_bounds__(64 * PR *WPR) void vx_pf_panel_kernel(const float *__restrict__ x, int ldx, int M, int K,
                                                                    int n_pairs, const float *__restrict__ w, float thr,
                                                                    uint4 *__restrict__ px, float *__restrict__ rs)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = wave % PR, part = wave / PR;
    const int row = blockIdx.x * PR + r;
    const int rg = row / PF_BM, mt = (row % PF_BM) / 32, l32 = row % 32;
    const bool live = row < M;
    const float *xr = x + (size_t)(live ? row : 0) * ldx;
    __shared__ float red[2][WPR][PR];
    const int k0 = 8 * (lane + 64 * part), step = 8 * 64 * WPR;
    // the 8 columns from k on, before any norm; zeros past K and M (K % 32 ==
    // 0: wholly in or out), read from a clamped address so that the loads of
    // all groups leave together
    auto load = [&](int k, float v[8]) {
        const bool ok = live && k < K;
        const int kc = min(k, K - 8);
        const float *p = SRC == PF_SWIGLU ? xr + 32 * (kc / 16) + kc % 16 : xr + kc;
        const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
        const float t[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        if constexpr (SRC == PF_SWIGLU) {
            const float4 ua = *(const float4 *)(p + 16), ub = *(const float4 *)(p + 20);
            const float u[8] = {ua.x, ua.y, ua.z, ua.w, ub.x, ub.y, ub.z, ub.w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float g = vx_silu(t[e]);
                v[e] = !ok || fabsf(g) < thr ? 0.0f : g * u[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = ok ? t[e] : 0.0f;
        }
    };
    // the norm's weights of the same columns (1 without them)
    auto load_w = [&](int k, float wv[8]) {
        float4 a = make_float4(1.f, 1.f, 1.f, 1.f), b = a;
        if (w) {
            const float *p = w + min(k, K - 8);
            a = *(const float4 *)p;
            b = *(const float4 *)(p + 4);
        }
        wv[0] = a.x; wv[1] = a.y; wv[2] = a.z; wv[3] = a.w;
        wv[4] = b.x; wv[5] = b.y; wv[6] = b.z; wv[7] = b.w;
    };
    float inv = 1.0f;
    auto norm = [&](const float wv[8], float v[8]) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = wv[e] * (v[e] * inv);
    };
    auto load_normed = [&](int k, float v[8]) {
        load(k, v);
        if constexpr (SRC == PF_RMS) {
            float wv[8];
            load_w(k, wv);
            norm(wv, v);
        }
    };
    // the values of a row's wavefronts joined
    auto join = [&](int slot, float v, bool sum) {
        if (lane == 0) red[slot][part][r] = v;
        __syncthreads();
        float j = red[slot][0][r];
#pragma unroll
        for (int i = 1; i < WPR; i++) j = sum ? j + red[slot][i][r] : fmaxf(j, red[slot][i][r]);
        return j;
    };
    float keep[KEEP][8];
    float wk[SRC == PF_RMS ? KEEP : 1][8];
#pragma unroll
    for (int i = 0; i < KEEP; i++) {
        load(k0 + i * step, keep[i]);
        if constexpr (SRC == PF_RMS) load_w(k0 + i * step, wk[i]);
    }
    if constexpr (SRC == PF_RMS) {
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < KEEP; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) ss += keep[i][e] * keep[i][e];
        for (int k = k0 + KEEP * step; k < K; k += step) {
            float v[8];
            load(k, v);
#pragma unroll
            for (int e = 0; e < 8; e++) ss += v[e] * v[e];
        }
        inv = vx_rms_inv(join(0, vx_wave_sum64(ss), true), K);
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < KEEP; i++) {
        if constexpr (SRC == PF_RMS) norm(wk[i], keep[i]);
#pragma unroll
        for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(keep[i][e]));
    }
    for (int k = k0 + KEEP * step; k < K; k += step) {
        float v[8];
        load_normed(k, v);
#pragma unroll
        for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
    }
    amax = join(1, vx_wave_max64(amax), false);
    float rsv;
    const float sc = live ? vx_row_scale(amax, &rsv) : 1.0f;
    if (live && lane == 0 && part == 0) rs[row] = rsv;
    auto put = [&](int k, const float v[8]) {
        vx_half8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float t = v[e] * sc;
            const _Float16 f = (_Float16)t;
            hi[e] = f;
            lo[e] = (_Float16)(t - (float)f);
        }
        const int p = k / 64, blk = (k / 32) & 1, half = (k / 16) & 1, s = (k / 8) & 1;
        uint4 *o = px + ((size_t)rg * n_pairs + p) * PF_STAGE + ((mt * 2 + blk) * 2 + s) * 128 + l32 + 32 * half;
        o[0] = __builtin_bit_cast(uint4, hi);
        o[64] = __builtin_bit_cast(uint4, lo);
    };
#pragma unroll
    for (int i = 0; i < KEEP; i++)
        if (k0 + i * step < n_pairs * 64) put(k0 + i * step, keep[i]);
    for (int k = k0 + KEEP * step; k < n_pairs * 64; k += step) {
        float v[8];
        load_normed(k, v);
        put(k, v);
    }
}

// the row scales follow the stages (16-byte aligned)
static size_t vx_pf_stage_bytes(int M, int K)
{
    return (size_t)((M + PF_BM - 1) / PF_BM) * ((K + 63) / 64) * PF_STAGE * sizeof(uint4);
}

extern "C" size_t vxh_rows_panel_bytes(int M, int K)
{
    if (M < 1 || K < 1) return 0;
    return vx_pf_stage_bytes(M, K) + ((size_t)M * sizeof(float) + 15) / 16 * 16;
}

// from here 8 rows to a workgroup (1024 x 4096: 17.3 us with one each, 12.2;
// below, they would leave more than half of the CUs idle)
#define PF_MANY_ROWS 1024

template <int SRC>
static int vx_pf_panel(const float *x, int ldx, int M, int K, const float *w, float thr, void *px, vxh_stream s)
{
    const int n_pairs = (K + 63) / 64;
    const unsigned rows = (unsigned)((M + PF_BM - 1) / PF_BM * PF_BM);
    float *rs = (float *)((char *)px + vx_pf_stage_bytes(M, K));
    const bool wide = K > 12 * 1024 || (SRC == PF_SWIGLU && K > 8 * 1024 && rows <= 512);
    if (M < PF_MANY_ROWS && K <= 4 * 1024)
        vx_pf_panel_kernel<SRC, 2, 1, 4><<<rows, 256, 0, vxh_hs(s)>>>(x, ldx, M, K, n_pairs, w, thr, (uint4 *)px, rs);
    else if (M < PF_MANY_ROWS && !wide)
        vx_pf_panel_kernel<SRC, 6, 1, 4><<<rows, 256, 0, vxh_hs(s)>>>(x, ldx, M, K, n_pairs, w, thr, (uint4 *)px, rs);
    else if (M < PF_MANY_ROWS)
        vx_pf_panel_kernel<SRC, 3, 1, 16><<<rows, 1024, 0, vxh_hs(s)>>>(x, ldx, M, K, n_pairs, w, thr, (uint4 *)px, rs);
    else if (K <= 4 * 1024)
        vx_pf_panel_kernel<SRC, 4, 8, 2><<<rows / 8, 1024, 0, vxh_hs(s)>>>(x, ldx, M, K, n_pairs, w, thr, (uint4 *)px,
                                                                         rs);
    else
        vx_pf_panel_kernel<SRC, SRC == PF_RMS ? 6 : 11, 8, 2><<<rows / 8, 1024, 0, vxh_hs(s)>>>(
            x, ldx, M, K, n_pairs, w, thr, (uint4 *)px, rs);
    VXH_LAUNCHED();
    return VXH_OK;
}

extern "C" int vxh_rows_panel(const float *X, int ldx, int M, int K, void *px, vxh_stream s)
{
    if (!X || !px || M < 1 || K < 32 || K % 32 || ldx < K || ldx % 4 || ((uintptr_t)X & 15) || ((uintptr_t)px & 15))
        return vxh_fail(VXH_ERR_PARAM, "rows_panel: M %d K %d ldx %d", M, K, ldx);
    return vx_pf_panel<PF_ROWS>(X, ldx, M, K, nullptr, 0.0f, px, s);
}

extern "C" int vxh_rmsnorm_rows_panel(const float *X, int ldx, int M, int K, const float *w, void *px, vxh_stream s)
{
    if (!X || !px || M < 1 || K < 32 || K % 32 || ldx < K || ldx % 4 || ((uintptr_t)X & 15) || ((uintptr_t)px & 15) ||
        ((uintptr_t)w & 15))
        return vxh_fail(VXH_ERR_PARAM, "rmsnorm_rows_panel: M %d K %d ldx %d", M, K, ldx);
    return vx_pf_panel<PF_RMS>(X, ldx, M, K, w, 0.0f, px, s);
}

extern "C" int vxh_swiglu_rows_panel(const float *gu, int ld_gu, int M, int F, float thr, void *px, vxh_stream s)
{
    if (!gu || !px || M < 1 || F < 32 || F % 32 || ld_gu < 2 * F || ld_gu % 4 || ((uintptr_t)gu & 15) ||
        ((uintptr_t)px & 15))
        return vxh_fail(VXH_ERR_PARAM, "swiglu_rows_panel: M %d F %d ld %d", M, F, ld_gu);
    return vx_pf_panel<PF_SWIGLU>(gu, ld_gu, M, F, nullptr, thr, px, s);
}

extern "C" int vxh_gemm_rows(const vxh_qmat *W, const void *px, int M, float *Y, int ldy, int n_out,
                             const float *R, int ldr, float scale, vxh_stream s)
{
    if (!W || !px || !Y || M < 1 || n_out < 1 || n_out > W->n_rows || ldy < n_out || (R && ldr < n_out) ||
        ((uintptr_t)px & 15))
        return vxh_fail(VXH_ERR_PARAM, "gemm_rows: M %d n_out %d (rows %d, K %d, ldy %d)", M, n_out, W->n_rows,
                        W->n_cols, ldy);
    if (W->type != 2 && W->type != 8) return vxh_fail(VXH_ERR_UNSUPPORTED, "gemm_rows: type %d", W->type);
    vx_pf_args a;
    a.wq = (const uint4 *)W->qs;
    a.wd = (const uint32_t *)W->d;
    a.n_tiles = W->n_rows / 32;
    a.n_pairs = W->n_pairs;
    a.px = (const uint4 *)px;
    a.rs = (const float *)((const char *)px + vx_pf_stage_bytes(M, W->n_cols));
    a.M = M;
    a.y = Y;
    a.ldy = ldy;
    a.n_out = n_out;
    a.r = R;
    a.ldr = ldr;
    a.scale = scale;
    return W->type == 2 ? vx_pf_gemm<2>(a, vxh_hs(s)) : vx_pf_gemm<8>(a, vxh_hs(s));
}

// ---------------------------------------------------------------------------
// RoPE + KV store for fp32 q|k|v rows (the same per-pair arithmetic as the
// verify path's vx_rope_kv_kernel, src/tensor.c:249-270): one thread per
// (row, pair) of q and k, v copied.
// ---------------------------------------------------------------------------
__global__ void vx_pf_rope_kv_kernel(const float *__restrict__ qkv, int ld_qkv, int M, int n_past, int n_ctx,
                                     int n_heads, int n_kv_heads, int hd, const float *__restrict__ bq,
                                     const float *__restrict__ bk, const float *__restrict__ bv,
                                     const float *__restrict__ cs, const float *__restrict__ sn,
                                     float *__restrict__ q_out, int ldq, float *__restrict__ kc,
                                     float *__restrict__ vc)
{
    const int qd = n_heads * hd, kvd = n_kv_heads * hd;
    const int half = hd / 2;
    const int per_row = (qd + kvd) / 2 + kvd;
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)M * per_row) return;
    const int m = (int)(idx / per_row), r = (int)(idx % per_row);
    const int rope_pos = n_past + m;
    const int pos = rope_pos < n_ctx ? rope_pos : n_ctx - 1;
    const float *row = qkv + (size_t)m * ld_qkv;
    if (r < (qd + kvd) / 2) {
        const int e = 2 * r;
        const bool isq = e < qd;
        const int el = isq ? e : e - qd;
        const int i = (el % hd) / 2;
        const float *bias = isq ? bq : bk;
        const float a = vx_norm_bias((double)row[e], 1.0f, bias, el);
        const float b = vx_norm_bias((double)row[e + 1], 1.0f, bias, el + 1);
        const float2 o = vx_rope_rot(a, b, cs[(size_t)rope_pos * half + i], sn[(size_t)rope_pos * half + i]);
        if (isq) *(float2 *)(q_out + (size_t)m * ldq + el) = o;
        else *(float2 *)(kc + (size_t)pos * kvd + el) = o;
    } else {
        const int el = r - (qd + kvd) / 2;
        vc[(size_t)pos * kvd + el] = vx_norm_bias((double)row[qd + kvd + el], 1.0f, bv, el);
    }
}

extern "C" int vxh_rope_kv_rows(const float *qkv, int ld_qkv, int M, int n_past, int n_ctx, int n_heads,
                                int n_kv_heads, int head_dim, const float *bq, const float *bk, const float *bv,
                                const float *cos_tab, const float *sin_tab, int n_pos, float *q_out, int ldq,
                                float *k_cache_layer, float *v_cache_layer, vxh_stream s)
{
    if (M < 1 || head_dim % 2 || ld_qkv % 2 || ldq % 2 || n_past < 0 || n_past + M - 1 >= n_pos ||
        ld_qkv < (n_heads + 2 * n_kv_heads) * head_dim || ldq < n_heads * head_dim)
        return vxh_fail(VXH_ERR_PARAM, "rope_kv_rows: M %d n_past %d n_pos %d", M, n_past, n_pos);
    const int qd = n_heads * head_dim, kvd = n_kv_heads * head_dim;
    const long n = (long)M * ((qd + kvd) / 2 + kvd);
    vx_pf_rope_kv_kernel<<<(unsigned)((n + 255) / 256), 256, 0, vxh_hs(s)>>>(
        qkv, ld_qkv, M, n_past, n_ctx, n_heads, n_kv_heads, head_dim, bq, bk, bv, cos_tab, sin_tab, q_out, ldq,
        k_cache_layer, v_cache_layer);
    VXH_LAUNCHED();
    return VXH_OK;
}

// ---------------------------------------------------------------------------
// SwiGLU with the FFN gate-skip (src/model.c:582-585) from the interleaved
// gate/up product (16 gate then 16 up columns per tile of 32): row m, column
// i reads gate at 32(i/16) + i%16 and up 16 further.
// ---------------------------------------------------------------------------
__global__ void vx_pf_swiglu_kernel(const float *__restrict__ gu, int ld_gu, int M, int F, float thr,
                                    float *__restrict__ h, int ldh)
{
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)M * F) return;
    const int m = (int)(idx / F), i = (int)(idx % F);
    const float *pg = gu + (size_t)m * ld_gu + 32 * (i / 16) + i % 16;
    const float g = vx_silu(pg[0]), u = pg[16];
    h[(size_t)m * ldh + i] = fabsf(g) < thr ? 0.0f : g * u;
}

extern "C" int vxh_swiglu_rows(const float *gu, int ld_gu, int M, int F, float thr, float *h, int ldh,
                               vxh_stream s)
{
    if (M < 1 || F < 1 || ldh < F || ld_gu < (F + 15) / 16 * 32)
        return vxh_fail(VXH_ERR_PARAM, "swiglu_rows: M %d F %d", M, F);
    const long n = (long)M * F;
    vx_pf_swiglu_kernel<<<(unsigned)((n + 255) / 256), 256, 0, vxh_hs(s)>>>(gu, ld_gu, M, F, thr, h, ldh);
    VXH_LAUNCHED();
    return VXH_OK;
}
