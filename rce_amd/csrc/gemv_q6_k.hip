// gemv_q6_k.hip -- the Q6_K decode kernels (EXACT: one chain lane per row; Q8: one
// lane per row and super-block).
#include "gemv_chain_pipe.h"
#include "lds_limit.h"
#include "qmm_gemv_kernels.h"

namespace rce_qmm {
namespace {

// ---------------------------------------------------------------------------
// Q6_K EXACT: one lane per row (the row sum is a single chain); this form,
// which also forms its own products, serves rows longer than the LDS holds.
// ---------------------------------------------------------------------------

// rce-op-qmm/src/lib.rs L425-454, L1667-1705: per half o, l in 0..32, the
// positions l, l+32, l+64, l+96 in order: sumf += ((d sc) q) a.
__device__ __forceinline__ float q6_exact_superblock(const RawQ6_K &b, const float *as, float sumf) {
    const float d = h2f(b.d);
#pragma unroll
    for (int o = 0; o < 2; o++) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const float ds1 = d * (float)q6_sc(b.c[12], 8 * o + c), ds2 = d * (float)q6_sc(b.c[12], 8 * o + c + 2);
            const float ds3 = d * (float)q6_sc(b.c[12], 8 * o + c + 4), ds4 = d * (float)q6_sc(b.c[12], 8 * o + c + 6);
            const float n1 = -32.0f * ds1, n2 = -32.0f * ds2, n3 = -32.0f * ds3, n4 = -32.0f * ds4;
#pragma unroll
            for (int lq = 4 * c; lq < 4 * c + 4; lq++) {
                uint32_t u1, u2, u3, u4;
                q6_words(b, o, lq, u1, u2, u3, u4);
                const float *al = as + 128 * o + 4 * lq;
                float x[4][4];  // activations of positions 4 lq + J + 32 m
#pragma unroll
                for (int m = 0; m < 4; m++)
#pragma unroll
                    for (int j = 0; j < 4; j++) x[m][j] = al[j + 32 * m];
#define Q6_STEP(J)                                                                   \
    sumf = sumf + __builtin_fmaf(ubyte<J>(u1), ds1, n1) * x[0][J];                     \
    sumf = sumf + __builtin_fmaf(ubyte<J>(u2), ds2, n2) * x[1][J];                     \
    sumf = sumf + __builtin_fmaf(ubyte<J>(u3), ds3, n3) * x[2][J];                     \
    sumf = sumf + __builtin_fmaf(ubyte<J>(u4), ds4, n4) * x[3][J];
                Q6_STEP(0) Q6_STEP(1) Q6_STEP(2) Q6_STEP(3)
#undef Q6_STEP
            }
        }
    }
    return sumf;
}

// Rows longer than Q6_EXACT_LDS_K: the activations are read from global
// memory (each lane the same addresses) instead of LDS.
constexpr size_t Q6_EXACT_LDS_K = 16384;
__global__ __launch_bounds__(256) void k_gemv_exact_q6k(DevWeight w, const float *__restrict__ A,
                                                        float *__restrict__ out) {
    const size_t row = (size_t)blockIdx.x * 256 + threadIdx.x;
    // Lanes past the end recompute the last row (no branch around loads).
    const size_t rr = row < w.n_rows ? row : w.n_rows - 1;
    const int nsb = (int)(w.n_cols / 256);
    const float *a = A + (size_t)blockIdx.y * w.n_cols;
    float sumf = 0.0f;
    RawQ6_K b0, b1;
    ld_q6_k(w, rr, 0, b0);
    int sb = 0;
    for (; sb + 1 < nsb; sb += 2) {
        ld_q6_k(w, rr, sb + 1, b1);
        sumf = q6_exact_superblock(b0, a + 256 * sb, sumf);
        if (sb + 2 < nsb) ld_q6_k(w, rr, sb + 2, b0);
        sumf = q6_exact_superblock(b1, a + 256 * (sb + 1), sumf);
    }
    if (sb < nsb) sumf = q6_exact_superblock(b0, a + 256 * sb, sumf);
    if (row < w.n_rows) out[(size_t)blockIdx.y * w.n_rows + row] = sumf;
}

// The same row chains with the products formed by helper waves (the
// pipeline of gemv_chain_pipe.h), for k <= Q6_EXACT_LDS_K.  A block serves
// 64 rows of a group with four waves, one per SIMD: wave 0 holds the chains,
// waves 1..3 form the products (a fifth wave would share the chain's SIMD
// and the chain, which every barrier waits for, would get half its issue
// slots).  The unit of work is a pair: steps l = 8 p .. 8 p + 7, m = 0..3
// (positions 128 o + l + 32 m) of half o of a super-block, pairs numbered
// g = 8 sb + 4 o + p in the chain's order.  Stage s is pairs 3 s .. 3 s + 2,
// helper h forming pair 3 s + h - 1 from 8-byte slices of its ql, qh and
// scale chunks and the rows' d; pairs past the row give +0.0 products, which
// leave a chain (from +0.0, never -0.0) unchanged.
constexpr int Q6_DS = 8;  // stages of loads a helper keeps in flight

// GROUP (grouped experts): blockIdx.y is a tile of tiles[0 .. n_tiles[0]),
// blockIdx.z the slot in it.
template <bool GROUP>
__global__ __launch_bounds__(256) void k_gemv_exact_q6k_split(DevWeight w, const float *__restrict__ A,
                                                              float *__restrict__ out, const DevWeight *__restrict__ wtab,
                                                              const MoeTile *__restrict__ tiles,
                                                              const int *__restrict__ n_tiles) {
    constexpr int SV = 96;  // chain steps per stage: 3 pairs
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    size_t t = blockIdx.y;
    const size_t row0 = (size_t)blockIdx.x * 64;
    if constexpr (GROUP) {
        if ((int)blockIdx.y >= n_tiles[0]) return;
        const MoeTile tl = tiles[blockIdx.y];
        if ((int)blockIdx.z >= tl.rows) return;
        w = wtab[tl.e];
        t = (size_t)tl.r0 + blockIdx.z;
    }
    const size_t k = w.n_cols;
    const int np = (int)(k / 256) * 8;  // pairs in a row
    const int ns = (np + 2) / 3;
    const int s_tot = (ns + Q6_DS - 1) / Q6_DS * Q6_DS;
    extern __shared__ __align__(16) unsigned char lds[];
    float *act = reinterpret_cast<float *>(lds);  // k values, then a 16-byte dump slot
    float4 *prod = reinterpret_cast<float4 *>(act + k + 4);  // [2][24][64]
    const int hw = wv - 1;
    const uint8_t *gb = w.base + (row0 / 64) * w.group_stride;
    const WBuf wq = make_wbuf(gb, (uint32_t)lane * 16);  // chunk slices
    const WBuf wd = make_wbuf(gb, (uint32_t)lane * 2);   // d
    struct Slice { uint2 qa, qb, qh, sc; uint32_t d; };
    // pair g's slices (g past the row: the last pair's, not used)
    auto load = [&](int s, Slice &v) {
        const int g = min(3 * s + hw, np - 1), o = (g >> 2) & 1, p = g & 3, c = p >> 1;
        const uint32_t so = (uint32_t)(g >> 3) * (uint32_t)IL64_Q6K_SB, b8 = 8u * (uint32_t)(p & 1);
        v.qa = bld8(wq, (uint32_t)(4 * o + c) * 1024u + b8, so);
        v.qb = bld8(wq, (uint32_t)(4 * o + 2 + c) * 1024u + b8, so);
        v.qh = bld8(wq, (uint32_t)(8 + 2 * o + c) * 1024u + b8, so);
        v.sc = bld8(wq, 12u * 1024u + 8u * (uint32_t)o, so);
        v.d = bld2(wd, (uint32_t)IL64_Q6K_D, so);
    };
    Slice ring[Q6_DS];
    if (wv != 0) {
#pragma unroll
        for (int j = 0; j < Q6_DS; j++) load(j, ring[j]);
    }
    stage_act<256, 16>(A + t * k, k, k, act, [](size_t i) { return i; });
    __syncthreads();
    if (wv == 0) {
        const float acc = run_chain<SV, 64>(prod + lane, ns, s_tot);
        const size_t row = row0 + lane;
        if (row < w.n_rows) out[t * w.n_rows + row] = acc;
        return;
    }
    // the pair's 32 activations (positions 8 p + 4 h + 32 m .. + 3 of its
    // half, h = 0, 1), read during the stage before
    float4 an[2][2][4];
    auto read_act = [&](int s, float4 (*dst)[4]) {
        const int g = min(3 * s + hw, np - 1);
        const float *ah = act + (size_t)(g >> 3) * 256 + 128 * ((g >> 2) & 1) + 8 * (g & 3);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int m = 0; m < 4; m++) dst[h][m] = *reinterpret_cast<const float4 *>(ah + 4 * h + 32 * m);
    };
    read_act(0, an[0]);
    for (int s0 = 0; s0 < s_tot; s0 += Q6_DS) {
#pragma unroll
        for (int u = 0; u < Q6_DS; u++) {
            const int s = s0 + u;
            read_act(s + 1, an[(u + 1) & 1]);
            const Slice v = ring[u];
            const int g = 3 * s + hw, c = (g & 3) >> 1;
            // (d sc) per m as the reference forms it, and -32 (d sc) for the
            // fma that rounds (q - 32) (d sc) once
            const float d = h2f(v.d);
            float ds[4], nn[4];
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const int bi = c + 2 * m;  // scale byte 8 o + is + 2 m within the half's 8 bytes
                const uint32_t wsc = (bi >> 2) ? v.sc.y : v.sc.x;
                ds[m] = d * (float)(int)(int8_t)((wsc >> (8 * (bi & 3))) & 0xFFu);
                nn[m] = -32.0f * ds[m];
            }
            float4 pr[2][4];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t qa = h ? v.qa.y : v.qa.x, qb = h ? v.qb.y : v.qb.x, qh = h ? v.qh.y : v.qh.x;
                const uint32_t uq[4] = {(qa & NIB) | ((qh & 0x03030303u) << 4), (qb & NIB) | ((qh & 0x0C0C0C0Cu) << 2),
                                        ((qa >> 4) & NIB) | (qh & 0x30303030u),
                                        ((qb >> 4) & NIB) | ((qh >> 2) & 0x30303030u)};
                float pj[4][4];  // [J][m]
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const float4 x = an[u & 1][h][m];
                    const float xa[4] = {x.x, x.y, x.z, x.w};
                    pj[0][m] = __builtin_fmaf(ubyte<0>(uq[m]), ds[m], nn[m]) * xa[0];
                    pj[1][m] = __builtin_fmaf(ubyte<1>(uq[m]), ds[m], nn[m]) * xa[1];
                    pj[2][m] = __builtin_fmaf(ubyte<2>(uq[m]), ds[m], nn[m]) * xa[2];
                    pj[3][m] = __builtin_fmaf(ubyte<3>(uq[m]), ds[m], nn[m]) * xa[3];
                }
#pragma unroll
                for (int j = 0; j < 4; j++) pr[h][j] = make_float4(pj[j][0], pj[j][1], pj[j][2], pj[j][3]);
            }
            load(s + Q6_DS, ring[u]);  // the slot's next stage once this one is used
            float4 *pp = prod + ((size_t)(s & 1) * (SV / 4) + 8 * hw) * 64 + lane;
            if (g < np) {
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int j = 0; j < 4; j++) pp[(size_t)(4 * h + j) * 64] = pr[h][j];
            } else {  // past the row: +0.0 steps
#pragma unroll
                for (int j = 0; j < 8; j++) pp[(size_t)j * 64] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------
// Q6_K Q8: a block owns R rows (R consecutive lanes of a 64-row group) and TB
// tokens; thread (r = tid % R, sb = tid / R) forms the sum of super-block sb,
// then sb + 256 / R, ... of row r, and the row's sums are folded in
// super-block order (rce-op-qmm/src/lib.rs L1667-1705's order).  A load
// instruction's R lanes read R * 16 contiguous bytes of one chunk plane, whole
// lines, where the activation-stationary form (a lane per super-block of a
// row, consecutive lanes a super-block apart) touched a line per lane for 16
// bytes of it; and the activations stay in LDS (a super-block's 256 values
// are one address for its R lanes) instead of 64 registers per token, so a
// SIMD holds five or six waves instead of two.  Bound by the weight's bytes
// at 32000x2048, by latency (quantize, barrier, 13 chunks, fold) below.
// Measured (us, that form / this one): 2048x5632 at 1 / 2 / 4 / 8 tokens
// 12.6 / 14.2 / 18.6 / 34.4 against 6.2 / 9.1 / 9.0 / 11.5; 32000x2048 at 1 / 2 /
// 4 / 8 11.8 / 26 / 50 / 95 against 9.1 (5.9 TB/s, cache included) / 10.4 / 16.8 /
// 28.8; 4096x14336 at 1 / 8 39 / 156 against 14.3 / 32.8.
// FX: the decode step's fused forms and grouped experts, as in k_gemv_as
// (FX_SWIGLU: lanes r < R / 2 gate rows, the others the same up rows).
// ---------------------------------------------------------------------------
template <int TB, int R, int FX>
__global__ __launch_bounds__(256) void k_gemv_q8_q6k(DevWeight w, const float *__restrict__ A, float *__restrict__ out,
                                                     int t_rows, GemvFx fx) {
    constexpr int NT = 256, NS = NT / R, KIND = FX & 7;
    constexpr bool NORM = (FX & FX_NORM) != 0, GROUP = (FX & FX_GROUP) != 0;
    static_assert(64 % R == 0 && (!GROUP || FX == FX_GROUP) && (!NORM || TB == 1), "forms");
    constexpr int RO = KIND == FX_SWIGLU ? R / 2 : R;  // output rows of the block
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, r = tid % R, sb0 = tid / R;
    unsigned bx = blockIdx.x;
    if constexpr (KIND == FX_SEG) {  // block-uniform choice of the segment
        if (fx.pos && bx == 0 && tid == 0 && fx.status[2] == 0) {  // the step's last kernel: advance the position
            const int p = fx.pos[0];
            if (p >= fx.ctx_len && fx.status[0] == 0) fx.status[0] = 2;
            fx.pos[0] = p + 1;
        }
        if (bx >= fx.blk3) { w = fx.w3; out = fx.out3; bx -= fx.blk3; }
        else if (bx >= fx.blk2) { w = fx.w2; out = fx.out2; bx -= fx.blk2; }
    }
    int t0 = blockIdx.y * TB, tv = min(TB, t_rows - t0);
    if constexpr (GROUP) {
        if ((int)blockIdx.y >= fx.n_tiles[0]) return;
        const MoeTile tl = fx.tiles[blockIdx.y];
        w = blockIdx.z ? fx.wtab2[tl.e] : fx.wtab[tl.e];
        if (blockIdx.z) out = fx.out2;
        t0 = tl.r0;
        tv = tl.rows;
    }
    const size_t row0 = (size_t)bx * RO, k = w.n_cols;
    const int nsb = (int)(k / 256);
    // RO divides 64, so the block's rows lie in one 64-row group, which the
    // layout holds whole: rows past n_rows are its padding.  Super-blocks
    // past the row repeat its last; neither is folded.
    const uint8_t *base = w.base;
    if constexpr (KIND == FX_SWIGLU) base = r >= RO ? fx.w2.base : base;
    base += (row0 / 64) * w.group_stride;
    const size_t ln = (row0 & 63) + r % RO;
    v4u32 c[13];
    uint32_t dr;
    auto load = [&](int sb) {
        const uint8_t *sp = base + (size_t)min(sb, nsb - 1) * IL64_Q6K_SB;
#pragma unroll
        for (int j = 0; j < 13; j++)
            c[j] = __builtin_nontemporal_load(reinterpret_cast<const v4u32 *>(sp + ((size_t)j * 64 + ln) * 16));
        dr = ldw2(sp + IL64_Q6K_D + ln * 2);
    };
    // the activations' loads go out first (they are waited for first)
    const int kq = (int)(k / 8), total = GROUP ? 0 : tv * kq;
    QuantTask q0, q1;
    if constexpr (!GROUP) {
        quant_task_load(A, kq, t0, total, tid, q0);
        quant_task_load(A, kq, t0, total, tid + NT, q1);
        if constexpr (NORM) {
            quant_task_load_g(fx.norm_w, kq, total, tid, q0);
            quant_task_load_g(fx.norm_w, kq, total, tid + NT, q1);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    load(sb0);
    __builtin_amdgcn_sched_barrier(0);
    ActLds L(lds, k, TB);
    if constexpr (GROUP) {
        const ActLds G(const_cast<unsigned char *>(fx.preq), k, fx.preq_t);
        for (int t = 0; t < tv; t++) {
            const int4 *gx = reinterpret_cast<const int4 *>(G.xq + (size_t)(t0 + t) * (k / 4));
            const int4 *gd = reinterpret_cast<const int4 *>(G.dx + (size_t)(t0 + t) * (k / 32));
            const int4 *gs = reinterpret_cast<const int4 *>(G.s16 + (size_t)(t0 + t) * (k / 16));
            int4 *lx = reinterpret_cast<int4 *>(L.xq + t * (k / 4)), *ld = reinterpret_cast<int4 *>(L.dx + t * (k / 32));
            int4 *ls = reinterpret_cast<int4 *>(L.s16 + t * (k / 16));
            for (int i = tid; i < (int)(k / 16); i += NT) lx[i] = gx[i];
            for (int i = tid; i < (int)(k / 128); i += NT) ld[i] = gd[i];
            for (int i = tid; i < (int)(k / 64); i += NT) ls[i] = gs[i];
        }
    } else {
        float inv = 0.0f;
        if constexpr (NORM) {  // rms_norm's scale from the whole row (kq <= 2 NT), as k_gemv_as
            __shared__ float red[NT / 64];
            float ss = quant_task_ssq(q0, tid < total);
            ss = ss + quant_task_ssq(q1, tid + NT < total);
            ss = wave_sum(ss);
            if ((tid & 63) == 0) red[tid >> 6] = ss;
            __syncthreads();
            float tot = 0.0f;
#pragma unroll
            for (int i = 0; i < NT / 64; i++) tot = tot + red[i];
            const float mean_sq = tot / (float)k;
            inv = 1.0f / sqrtf(mean_sq + fx.eps);
        }
        quant_task_finish<NORM>(q0, k, total, tid, L, inv);
        quant_task_finish<NORM>(q1, k, total, tid + NT, L, inv);
        for (int i = 2 * NT; i < total; i += NT) {
            QuantTask q;
            quant_task_load(A, kq, t0, total, i + tid, q);
            quant_task_finish(q, k, total, i + tid, L);
        }
    }
    __syncthreads();
    // [super-block, padded to whole passes][token][row]: every lane stores, so
    // no arithmetic is sunk into a branch
    float *part = reinterpret_cast<float *>(lds + act_lds_bytes(k, TB));
    for (int s0 = 0; s0 < nsb; s0 += NS) {
        const int sb = min(s0 + sb0, nsb - 1);
        RawQ6_K raw;
        // the chunks enter the body as whole register quadruples: passed in
        // word by word, the compiler reused their registers before the reads
#pragma unroll
        for (int j = 0; j < 13; j++) {
            asm volatile("" : "+v"(c[j]));
            raw.c[j] = make_uint4(c[j].x, c[j].y, c[j].z, c[j].w);
        }
        const float d = h2f(dr);
        float ssb[TB];
#pragma unroll
        for (int t = 0; t < TB; t++) ssb[t] = 0.0f;
#pragma unroll
        for (int o = 0; o < 2; o++) {
            int acc[TB][8];  // sub-block 8 o + 2 m + h -> index 2 m + h
#pragma unroll
            for (int h = 0; h < 2; h++) {  // words 4 h .. 4 h + 3 of the half's quarters
                asm volatile("" ::: "memory");  // only their activations in registers at a time
                uint32_t u[4][4];
#pragma unroll
                for (int j = 0; j < 4; j++) q6_words(raw, o, 4 * h + j, u[0][j], u[1][j], u[2][j], u[3][j]);
#pragma unroll
                for (int m = 0; m < 4; m++)
#pragma unroll
                    for (int t = 0; t < TB; t++) {
                        const int4 x = *reinterpret_cast<const int4 *>(L.xq + t * (k / 4) + 64 * (size_t)sb + 32 * o +
                                                                       8 * m + 4 * h);
                        int a = __builtin_amdgcn_sdot4((int)u[m][0], x.x, 0, false);
                        a = __builtin_amdgcn_sdot4((int)u[m][1], x.y, a, false);
                        a = __builtin_amdgcn_sdot4((int)u[m][2], x.z, a, false);
                        acc[t][2 * m + h] = __builtin_amdgcn_sdot4((int)u[m][3], x.w, a, false);
                    }
            }
#pragma unroll
            for (int bb = 0; bb < 8; bb++) {  // sub-blocks in order: s += (d sc) (dx (dot - 32 sum))
                const int sbk = 8 * o + bb;
                const float ds = d * (float)q6_sc(raw.c[12], sbk);
#pragma unroll
                for (int t = 0; t < TB; t++) {
                    const int isum = acc[t][bb] - 32 * L.s16[t * (k / 16) + 16 * (size_t)sb + sbk];
                    const float ab = L.dx[t * (k / 32) + 8 * (size_t)sb + (sbk >> 1)] * (float)isum;
                    ssb[t] = ssb[t] + ds * ab;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TB; t++) part[((s0 + sb0) * TB + t) * R + r] = ssb[t];
        asm volatile("" ::: "memory");  // the next loads go into the registers just used
        if (s0 + NS < nsb) load(s0 + NS + sb0);
    }
    __syncthreads();
    auto fold = [&](int t, int rr) {
        float s = 0.0f;
#pragma unroll 8
        for (int sb = 0; sb < nsb; sb++) s = s + part[(sb * TB + t) * R + rr];
        return s;
    };
    for (int j = tid; j < tv * RO; j += NT) {
        const int t = j / RO, rr = j % RO;
        if (row0 + rr < w.n_rows) {
            const size_t o = ((size_t)t0 + t) * w.n_rows + row0 + rr;
            if constexpr (KIND == FX_SWIGLU) {
                const float g = fold(t, rr), u = fold(t, RO + rr);
                out[o] = silu_ref(g) * u;  // rce-tinyllama L320: h = silu(g) * u
            } else if constexpr (KIND == FX_RESIDUAL) {
                out[o] = fx.res[o] + fold(t, rr);  // rce-tinyllama L318, L323: x += ...
            } else {
                out[o] = fold(t, rr);
            }
        }
    }
}

size_t q6_q8_lds(size_t k, int tb, int r) {
    const size_t ns = 256 / (size_t)r;
    return act_lds_bytes(k, tb) + (k / 256 + ns - 1) / ns * ns * tb * r * sizeof(float);
}

// Rows per block: 16 spreads a row's super-blocks over 16 threads, 32 halves
// the blocks' repeated quantization and activation staging, so 32 where it
// still leaves two blocks per CU.  `units` is tokens / TB (times matrices).
// Measured, 16 / 32 rows (us, a separate quantization launch of about 3
// included): 512 blocks of 32 rows: 4096x4096 at 8 tokens 14.6 / 13.0, 4096x14336
// at 8 46 / 37; 256 blocks: 4096x4096 at 4 10.4 / 11.0, 4096x14336 at 4 28 / 28.
bool q6_rows32(size_t n_rows, size_t k, int tb, size_t units) {
    return (n_rows + 31) / 32 * units >= 512 && q6_q8_lds(k, tb, 32) <= LDS_MAX;
}

template <int TB, int R, int FX>
hipError_t launch_q6_q8(const DevWeight &w, const float *a, size_t t_rows, float *out, const GemvFx &fx, dim3 grid,
                        hipStream_t s) {
    // 16 rows, two tokens, the longest row (act_lds_bytes(k, 1) = LDS_MAX): 151 KB
    // (past 64 KB: q6_prepare_lds has raised the limit)
    const size_t lds = q6_q8_lds(w.n_cols, TB, R);
    hipLaunchKernelGGL((k_gemv_q8_q6k<TB, R, FX>), grid, dim3(256), lds, s, w, a, out, (int)t_rows, fx);
    return hipGetLastError();
}

template <int TB>
hipError_t launch_q6_q8_plain(const DevWeight &w, const float *a, size_t t_rows, float *out, hipStream_t s) {
    const size_t tg = (t_rows + TB - 1) / TB;
    if (q6_rows32(w.n_rows, w.n_cols, TB, tg))
        return launch_q6_q8<TB, 32, 0>(w, a, t_rows, out, GemvFx{}, dim3((unsigned)((w.n_rows + 31) / 32), (unsigned)tg), s);
    return launch_q6_q8<TB, 16, 0>(w, a, t_rows, out, GemvFx{}, dim3((unsigned)((w.n_rows + 15) / 16), (unsigned)tg), s);
}

template <int TB>
hipError_t launch_q6_q8_grouped(const DevWeight &w, const MoeGroup &m, const void *a, float *out, hipStream_t s) {
    GemvFx fx{};
    fx.wtab = m.wtab;
    fx.wtab2 = m.wtab2;
    fx.out2 = m.out2;
    fx.tiles = m.tiles;
    fx.n_tiles = m.n_tiles;
    fx.preq = static_cast<const unsigned char *>(a);
    fx.preq_t = m.n_slots_max;
    const unsigned y = (unsigned)m.max_tiles, z = m.wtab2 ? 2u : 1u;
    if (q6_rows32(w.n_rows, w.n_cols, TB, (size_t)y * z))
        return launch_q6_q8<TB, 32, FX_GROUP>(w, nullptr, 0, out, fx, dim3((unsigned)((w.n_rows + 31) / 32), y, z), s);
    return launch_q6_q8<TB, 16, FX_GROUP>(w, nullptr, 0, out, fx, dim3((unsigned)((w.n_rows + 15) / 16), y, z), s);
}

// The decode step's fused forms (launch_gemv_fx has checked dtypes, columns
// and the normalizing forms' row length).
template <int FX>
hipError_t launch_q6_q8_fx(const FxLaunch &f, const float *a, hipStream_t s) {
    GemvFx fx{};
    fx.norm_w = f.norm_w;
    fx.eps = f.eps;
    fx.pos = f.pos;
    fx.status = f.status;
    fx.ctx_len = f.ctx_len;
    fx.res = f.res;
    constexpr bool SEG = (FX & 7) == FX_SEG, PAIR = (FX & 7) == FX_SWIGLU;
    if (f.pos && (!SEG || !f.status)) return hipErrorInvalidValue;
    if ((FX & FX_NORM) && !f.norm_w) return hipErrorInvalidValue;
    size_t rows = f.w[0].n_rows;
    if (SEG)
        for (int i = 1; i < f.nw; i++) rows += f.w[i].n_rows;
    const bool r32 = q6_rows32(PAIR ? 2 * rows : rows, f.w[0].n_cols, 1, 1);
    const size_t ro = (r32 ? 32 : 16) / (PAIR ? 2 : 1);
    auto nblk = [&](const DevWeight &w) { return (unsigned)((w.n_rows + ro - 1) / ro); };
    unsigned blocks = nblk(f.w[0]);
    fx.blk2 = fx.blk3 = ~0u;
    if (SEG) {
        if (f.nw < 1 || f.nw > 3) return hipErrorInvalidValue;
        if (f.nw >= 2) { fx.w2 = f.w[1]; fx.out2 = f.out[1]; fx.blk2 = blocks; blocks += nblk(f.w[1]); }
        if (f.nw >= 3) { fx.w3 = f.w[2]; fx.out3 = f.out[2]; fx.blk3 = blocks; blocks += nblk(f.w[2]); }
    }
    if (PAIR) {
        if (f.nw != 2 || f.w[1].n_rows != f.w[0].n_rows) return hipErrorInvalidValue;
        fx.w2 = f.w[1];
    }
    return r32 ? launch_q6_q8<1, 32, FX>(f.w[0], a, 1, f.out[0], fx, dim3(blocks), s)
               : launch_q6_q8<1, 16, FX>(f.w[0], a, 1, f.out[0], fx, dim3(blocks), s);
}

size_t q6_split_lds(size_t k) { return (k + 4) * sizeof(float) + 2 * 96 * 64 * sizeof(float); }

hipError_t launch_q6_split(const DevWeight &w, const float *a, size_t t_rows, float *out, hipStream_t s) {
    const size_t lds = q6_split_lds(w.n_cols);
    if (lds > 64 * 1024) {  // activations of a long row: more than the default 64 KB
        const hipError_t e = ensure_lds_limit((const void *)k_gemv_exact_q6k_split<false>, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    const dim3 grid((unsigned)((w.n_rows + 63) / 64), (unsigned)t_rows);
    hipLaunchKernelGGL(k_gemv_exact_q6k_split<false>, grid, dim3(256), lds, s, w, a, out, (const DevWeight *)nullptr,
                       (const MoeTile *)nullptr, (const int *)nullptr);
    return hipGetLastError();
}

}  // namespace

hipError_t q6_prepare_lds() {
    // Q8: the forms with 16 rows per block (with 32, q6_rows32 keeps to 64 KB;
    // the normalizing forms' rows are short)
    for (const void *fn : {(const void *)k_gemv_exact_q6k_split<false>, (const void *)k_gemv_exact_q6k_split<true>,
                           (const void *)k_gemv_q8_q6k<1, 16, 0>, (const void *)k_gemv_q8_q6k<2, 16, 0>,
                           (const void *)k_gemv_q8_q6k<1, 16, FX_GROUP>, (const void *)k_gemv_q8_q6k<2, 16, FX_GROUP>,
                           (const void *)k_gemv_q8_q6k<1, 16, FX_SEG>, (const void *)k_gemv_q8_q6k<1, 16, FX_RESIDUAL>,
                           (const void *)k_gemv_q8_q6k<1, 16, FX_SWIGLU>}) {
        const hipError_t e = ensure_lds_limit(fn, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_gemv_grouped_q6_k(const DevWeight &w, const MoeGroup &m, const void *a, float *out, int mode, hipStream_t s) {
    if (mode != 0) {
        if (m.tb == 1) return launch_q6_q8_grouped<1>(w, m, a, out, s);
        return m.tb == 2 ? launch_q6_q8_grouped<2>(w, m, a, out, s) : hipErrorInvalidValue;
    }
    if (w.n_cols > Q6_EXACT_LDS_K) return hipErrorInvalidValue;
    const size_t lds = q6_split_lds(w.n_cols);
    if (lds > 64 * 1024) {
        const hipError_t e = ensure_lds_limit((const void *)k_gemv_exact_q6k_split<true>, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    const dim3 grid((unsigned)((w.n_rows + 63) / 64), (unsigned)m.max_tiles, (unsigned)m.tb);
    for (int i = 0; i < (m.wtab2 ? 2 : 1); i++) {
        hipLaunchKernelGGL(k_gemv_exact_q6k_split<true>, grid, dim3(256), lds, s, w, static_cast<const float *>(a),
                           i ? m.out2 : out, i ? m.wtab2 : m.wtab, m.tiles, m.n_tiles);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_gemv_q6_k(const DevWeight &w, const float *a, size_t t_rows, float *out, int mode,
                            hipStream_t s) {
    if (mode == 0) {
        if (w.n_cols <= Q6_EXACT_LDS_K) return launch_q6_split(w, a, t_rows, out, s);
        dim3 grid((unsigned)((w.n_rows + 255) / 256), (unsigned)t_rows);
        hipLaunchKernelGGL(k_gemv_exact_q6k, grid, dim3(256), 0, s, w, a, out);
        return hipGetLastError();
    }
    // one token or two per block: four hold the block's LDS and registers for
    // the gain of a weight read from the Infinity Cache (us, two / four per
    // block at 4 tokens: 4096x4096 10.4 / 11.1, 2048x5632 11.9 / 15.8,
    // 32000x2048 20.5 / 18.9)
    return t_rows == 1 ? launch_q6_q8_plain<1>(w, a, t_rows, out, s) : launch_q6_q8_plain<2>(w, a, t_rows, out, s);
}
hipError_t launch_gemv_fx_q6_k(const FxLaunch &f, const float *a, int mode, hipStream_t s) {
    if (mode == 0) return hipErrorInvalidValue;  // EXACT Q6_K is one lane per row
    switch (f.kind) {
    case FX_SEG: return launch_q6_q8_fx<FX_SEG>(f, a, s);
    case FX_SEG | FX_NORM: return launch_q6_q8_fx<FX_SEG | FX_NORM>(f, a, s);
    case FX_RESIDUAL: return launch_q6_q8_fx<FX_RESIDUAL>(f, a, s);
    case FX_SWIGLU: return launch_q6_q8_fx<FX_SWIGLU>(f, a, s);
    case FX_SWIGLU | FX_NORM: return launch_q6_q8_fx<FX_SWIGLU | FX_NORM>(f, a, s);
    default: return hipErrorInvalidValue;
    }
}
}  // namespace rce_qmm
