// gemv_q8_mfma.hip -- the Q8-activation product of several tokens (mode Q8)
// on the int8 matrix cores, for one weight (mm_batched) and for grouped
// experts (MoE).  Every block of 32's exact int32 dot of the weight's
// integers with a token's Q8 integers is one lane's element of a
// v_mfma_i32_16x16x32_i8 (16 weight rows x 16 tokens, K = one block), and
// the rest is the decode kernels' f32 arithmetic in their order
// (qmm_gemv_kernels.h: Q32Q8, Q4_KQ8, Q5_KQ8; gemv_q6_k.hip), the row sum folded
// over units in order from +0.0 in registers.  So the result is bit-identical
// to the decode kernels' Q8 mode and to the oracle's orc_mm_batched_q8.
//
// What bounds it: 4 (Q8_0) to 12 (Q4_K, per 64) f32 operations per (row,
// token, unit), each rounded, whatever computes the dots, and the unpacking:
// Q4_K 14336x4096 at 32 tokens counts 8.6 M vector instructions, 8400 per SIMD (14
// us of the kernel's 25 at four cycles each and 2.4 GHz), no LDS bank
// conflicts.  The decode kernels hold a token's activations in registers, at most four at a time, so
// they dequantize the weight again for every four tokens and send every
// addend through LDS to a fold thread.
//
// Work mapping: a block of four waves owns 16 rows and one tile of 16
// tokens.  K is cut into chunks of four units (CK = 256 for the K-quants, 128
// for blocks of 32), chunk c to wave c % 4: a row's sum is a chain over all
// of K, and one wave walking it alone took 1 us per 256 of K whatever the
// problem size.  Each wave forms its chunk's addends (lane l: A operand row
// l % 16, positions 8 kq .. 8 kq + 7, kq = l / 16, of a block of 32; B operand
// token l % 16, the same positions; accumulator element i is row 4 kq + i,
// token l % 16) and stores them to LDS; then thread (row, token) adds the
// four chunks' addends in unit order, the reference's sequential sum, with
// the running sum in a register.
//
// Each wave fills its own LDS ring of RING chunks with direct global -> LDS
// loads of its rows' weight bytes, so no barrier orders them, and takes its
// activation operands (which k_quantize_tiles lays out so that a lane's is
// one 16-byte load per 64 of K) from the L2 into registers one chunk ahead.
// vmcnt retires in order: the operand loads go out before the ring's newest
// chunk, so that waiting for them does not drain it.  The wave forms its rows' f32 scales
// once per chunk into a small LDS table.
//
// Measured (us, decode kernels / this form, quantization included): see
// gemv_q8_mfma_preferred.
#include "lds_limit.h"
#include "mfma_util.h"
#include "qmm_gemv_kernels.h"

#include <algorithm>

namespace rce_qmm {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int QK = 256;          // K of an activation stage: two halves of ACT_HALF bytes
constexpr int ACT_HALF = 2560;   // 128 of K of a tile: operands [pair of blocks][lane] 16 B, then {dx, sums} [pair][token] 16 B
constexpr int ACT_STAGE = 2 * ACT_HALF;

// s_waitcnt vmcnt(N) alone (gfx9 encoding: expcnt and lgkmcnt not waited for)
template <int N>
__device__ __forceinline__ void q8_wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
template <int N>
__device__ __forceinline__ void q8_wait_lgkm() {
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
template <int OFF>
__device__ __forceinline__ u32x4 ds_read16(uint32_t a) {
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF) : "memory");
    return v;
}
template <int OFF>
__device__ __forceinline__ void ds_write4(uint32_t a, float v) {
    asm volatile("ds_write_b32 %0, %1 offset:%2" ::"v"(a), "v"(v), "n"(OFF) : "memory");
}
__device__ __forceinline__ void ds_write16(uint32_t a, f32x4 v) { asm volatile("ds_write_b128 %0, %1" ::"v"(a), "v"(v) : "memory"); }

// --- formats -----------------------------------------------------------------
// Per chunk and 16 rows: NSEG 1 KB loads of weight bytes (64 bytes per row;
// Q6_K: four chunks of its 64-row groups each), one header of 16 bytes per
// row and, with fifth bits, FB bytes per row.  UNITS: addends per chunk.
enum Q8Fmt { QF_Q4_0, QF_Q8_0, QF_Q5_0, QF_Q4_1, QF_Q4_K, QF_Q5_K, QF_Q6_K };
template <Q8Fmt F>
struct QFmt {
    static constexpr bool Q6 = F == QF_Q6_K, KQ = F == QF_Q4_K || F == QF_Q5_K;
    static constexpr bool FIFTH = F == QF_Q5_0 || F == QF_Q5_K;
    static constexpr int CK = Q6 || KQ ? 256 : 128, NP = CK / 64;  // K of a chunk, its pairs of blocks
    static constexpr int UNITS = Q6 ? 1 : 4;
    static constexpr int NSEG = Q6 ? 3 : KQ || F == QF_Q8_0 ? 2 : 1;
    static constexpr int FB = F == QF_Q5_K ? 32 : F == QF_Q5_0 ? 16 : 0;
    static constexpr int OFF_H = NSEG * 1024;
    static constexpr int OFF_F = OFF_H + (Q6 ? 288 : 256);      // Q6_K: the scales chunk (16 B x 16 rows), then d (2 B x 16)
    static constexpr int W_ROWS = (OFF_F + 16 * FB + 127) / 128 * 128;  // per 16 rows
    static constexpr int W_LOADS = NSEG + 1 + (FIFTH ? 1 : 0);
    static constexpr int ACT = CK / 128 * ACT_HALF, META = CK / 128 * 512;
    static constexpr int LOADS = W_LOADS + 1;                   // to LDS, per wave and chunk
    static constexpr int SLOT = META + W_ROWS;
    static constexpr int SCT = Q6 || KQ ? 1024 : F == QF_Q4_1 ? 512 : 256;
    static constexpr int PART = UNITS * 1024;                   // a wave's addends
    static constexpr int FIX = 4 * (SCT + PART);
    // chunks in each wave's ring: three where four blocks still share a CU
    static constexpr int RING = 3 * 4 * SLOT + FIX <= 40 * 1024 ? 3 : 2;
    static constexpr int LDS = RING * 4 * SLOT + FIX;
    static_assert(LDS <= 160 * 1024, "LDS budget");
    static constexpr int NIBC = F == QF_Q4_0 ? 8 : F == QF_Q5_0 ? 16 : 0;  // the block formats' value offset
};

// One pair of blocks of 32 (a 64-group): what a lane reads from LDS for it.
template <Q8Fmt F>
struct QPair {
    u32x4 m;         // {dx, s16 pair} of both blocks
    u32x2 w[QFmt<F>::KQ ? 1 : QFmt<F>::Q6 ? 3 : 2];
    uint32_t fb[2];  // fifth-bit bytes
    u32x4 sc[QFmt<F>::KQ ? 4 : QFmt<F>::Q6 || F == QF_Q4_1 ? 4 : 2];
};

__device__ __forceinline__ i32x4 dot16(u32x2 a, uint32_t b0, uint32_t b1) {
    const u32x2 b = {b0, b1};
    long A, B;
    __builtin_memcpy(&A, &a, 8);
    __builtin_memcpy(&B, &b, 8);
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(A, B, i32x4{0, 0, 0, 0}, 0, 0, 0);
}

struct Q8Out {  // blockIdx.y's weight, expert table and output
    DevWeight w;
    const DevWeight *wtab;
    float *out;
};

template <Q8Fmt F>
__global__ __launch_bounds__(256, 3) void k_gemv_q8_mfma(Q8Out o0, Q8Out o1, const unsigned char *__restrict__ acts, int T,
                                                      int n_tile_max, const MoeTile *__restrict__ tiles,
                                                      const int *__restrict__ n_tiles) {
    using Q = QFmt<F>;
    constexpr int ROWS = 16, UNITS = Q::UNITS;
    extern __shared__ __align__(16) unsigned char lds[];
    // Block L: XCD L % 8; its blocks take the tiles of one row slice one after
    // the other, so the weight rows that several tiles read come from that
    // XCD's L2.
    const int L = blockIdx.x, tile = (L / 8) % n_tile_max;
    const size_t slice = (size_t)(L / 8 / n_tile_max) * 8 + L % 8;
    const Q8Out &o = blockIdx.y ? o1 : o0;
    DevWeight w = o.w;
    float *out = o.out;
    size_t orow = (size_t)tile * 16;  // first output row (token, or slot)
    int tokens = 16;
    if (n_tiles) {
        if (tile >= n_tiles[0]) return;
        const MoeTile tl = tiles[tile];
        w = o.wtab[tl.e];
        orow = (size_t)tl.r0;
        tokens = tl.rows;
    } else {
        tokens = T - (int)orow < 16 ? T - (int)orow : 16;
    }
    const size_t n = w.n_rows, k = w.n_cols, row0 = slice * ROWS;
    if (row0 >= n) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int nch = (int)(k / Q::CK);

    // ---- loads
    const __amdgpu_buffer_rsrc_t ab = byte_buffer(acts + (size_t)tile * (k / QK) * ACT_STAGE, (uint32_t)(k / QK * ACT_STAGE));
    __amdgpu_buffer_rsrc_t wb;
    uint32_t seg_off, h_off, f_off = 0;
    if constexpr (Q::Q6) {  // rows row0 .. of one 64-row group (rows padded to 64)
        wb = byte_buffer(w.base + (row0 >> 6) * w.group_stride, (uint32_t)w.group_stride);
        const uint32_t rg = (uint32_t)(row0 & 63);
        seg_off = (uint32_t)(kq * 1024) + 16u * (rg + (uint32_t)r16);  // chunk 4 j + kq
        h_off = lane < 16 ? 12u * 1024u + 16u * (rg + (uint32_t)r16) : (uint32_t)IL64_Q6K_D + 2u * rg + 16u * (uint32_t)(lane & 1);
    } else {
        const int rows = (int)(n - row0 < (size_t)ROWS ? n - row0 : ROWS);
        wb = byte_buffer(w.base + row0 * w.row_stride, (uint32_t)((size_t)rows * w.row_stride));
        auto rel = [&](int r) { return (uint32_t)((size_t)(r < rows ? r : rows - 1) * w.row_stride); };  // rows past n: the last
        const int sr = lane >> 2;
        seg_off = rel(sr) + 16u * (uint32_t)((lane & 3) ^ ((sr >> 2) & 3));
        h_off = rel(r16);
        f_off = Q::FB == 16 ? h_off : rel((lane >> 1) & 15) + 16u * (uint32_t)(lane & 1);
    }
    unsigned char *ring = lds + wave * (Q::RING * Q::SLOT);
    // Loads of the wave's chunk c (past the end: its last chunk again, into
    // a slot nothing reads any more).
    auto issue = [&](int c, int slot) {
        const int cc = c < nch ? c : nch - 1;
        unsigned char *d = ring + slot * Q::SLOT;
        const uint32_t as = (uint32_t)cc * (uint32_t)Q::ACT;
        // the scales and sums of the chunk's halves
        if (Q::META == 1024 || lane < 32)
            buf_load_lds16(ab, 2048u + 16u * (uint32_t)(lane & 31) + (lane < 32 ? 0u : (uint32_t)ACT_HALF), as, d);
        unsigned char *wd = d + Q::META;
        if constexpr (Q::Q6) {
            const uint32_t sb = (uint32_t)cc * (uint32_t)IL64_Q6K_SB;
#pragma unroll
            for (int j = 0; j < 3; j++) buf_load_lds16(wb, seg_off, sb + (uint32_t)j * 4096u, wd + j * 1024);
            if (lane < 18) buf_load_lds16(wb, h_off, sb, wd + Q::OFF_H);
        } else {
#pragma unroll
            for (int j = 0; j < Q::NSEG; j++)
                buf_load_lds16(wb, seg_off, (uint32_t)(j ? w.plane2 : w.plane1) + 64u * (uint32_t)cc, wd + j * 1024);
            // 16 header bytes: a super-block's, a chunk's four {d, m}, or the
            // f16 scales of two chunks
            const uint32_t hs = 16u * (uint32_t)(Q::KQ || F == QF_Q4_1 ? cc : cc >> 1);
            if (lane < 16) buf_load_lds16(wb, h_off, hs, wd + Q::OFF_H);
            if constexpr (Q::FIFTH)
                if (lane < Q::FB)
                    buf_load_lds16(wb, f_off, (uint32_t)(F == QF_Q5_K ? w.plane3 : w.plane2) + (uint32_t)(Q::FB * cc), wd + Q::OFF_F);
        }
    };

    // The operand of the wave's chunk c, one 16-byte load per pair of blocks
    // (from the L2, every block of the tile reads them).
    u32x4 xr[Q::NP];
    auto load_x = [&](int c) {
        const uint32_t as = (uint32_t)(c < nch ? c : nch - 1) * (uint32_t)Q::ACT;
#pragma unroll
        for (int p = 0; p < Q::NP; p++)
            xr[p] = __builtin_amdgcn_raw_buffer_load_b128(ab, 16 * lane, (int)(as + (uint32_t)((p >> 1) * ACT_HALF + (p & 1) * 1024)), 0);
    };

    // ---- LDS addresses (slot 0; offsets within a chunk are immediates)
    const uint32_t a0 = lds_addr(ring), w0 = a0 + (uint32_t)Q::META;
    unsigned char *fix = lds + 4 * Q::RING * Q::SLOT;
    const uint32_t sct = lds_addr(fix) + (uint32_t)(wave * Q::SCT);
    const uint32_t part0 = lds_addr(fix + 4 * Q::SCT) + 4u * (uint32_t)tid;                        // fold
    const uint32_t part_wr = lds_addr(fix + 4 * Q::SCT) + (uint32_t)(wave * Q::PART) + 4u * (uint32_t)lane;
    const uint32_t m_rd = a0 + 16u * (uint32_t)r16;
    const uint32_t h_rd = w0 + Q::OFF_H + 16u * (uint32_t)r16;
    // weight bytes of piece p (16-byte part of a segment): Q4_K / Q5_K / Q8_0
    // k-slice kq in plane kq / 2, bytes 8 (kq & 1); Q6_K: of its chunk kq / 2
    uint32_t w_rd[4];
#pragma unroll
    for (int p = 0; p < 4; p++)
        w_rd[p] = w0 + (Q::Q6 ? (uint32_t)((kq >> 1) * 256 + r16 * 16 + 8 * (kq & 1))
                              : (Q::KQ || F == QF_Q8_0 ? (uint32_t)(kq >> 1) * 1024u : 0u) + (uint32_t)r16 * 64u +
                                    16u * (uint32_t)(p ^ ((r16 >> 2) & 3)) + 8u * (uint32_t)(kq & 1));
    const uint32_t f_rd = w0 + (uint32_t)(Q::OFF_F + r16 * Q::FB + kq);
    const int nsh = F == QF_Q8_0 || Q::KQ ? 0 : 4 * (kq >> 1);
    // scale table: lane (row r16, part kq) writes, rows 4 kq .. are read
    const uint32_t sc_wr = sct + (Q::KQ ? (uint32_t)(kq * 16 + r16) * 16u
                                  : Q::Q6 ? (uint32_t)(kq * 64 + r16) * 4u
                                          : (uint32_t)(kq * (F == QF_Q4_1 ? 32 : 16) + r16) * 4u);
    const uint32_t sc_rd = sct + (Q::KQ ? 64u : 16u) * (uint32_t)kq;

    // The rows' scales of chunk c (in the slot at byte `so`) to the wave's table.
    auto scales = [&](int c, uint32_t so) {
        if constexpr (Q::KQ) {  // 64-group kq of row r16: {d1, min1, d2, min2} to [group][row]
            u32x4 hv = ds_read16<0>(h_rd + so);
            q8_wait_lgkm<0>();
            pin(hv);
            const uint4 h = make_uint4(hv[0], hv[1], hv[2], hv[3]);
            const float d = h2f(h.x & 0xFFFFu), dmin = h2f(h.x >> 16);
            int sc1, m1, sc2, m2;
            k4_scale_min_pair(h, kq, sc1, m1, sc2, m2);
            ds_write16(sc_wr, f32x4{d * (float)sc1, dmin * (float)m1, d * (float)sc2, dmin * (float)m2});
        } else if constexpr (Q::Q6) {  // sub-blocks 4 kq .. + 3 of row r16 to [sub-block][row]
            uint32_t sv = lds_read4<0>(h_rd + so + 4u * (uint32_t)kq);
            uint32_t dv = lds_read_u16<256>(h_rd + so - 14u * (uint32_t)r16);
            q8_wait_lgkm<0>();
            pin(sv);
            pin(dv);
            const float d = h2f(dv);
            ds_write4<0>(sc_wr, d * (float)(int8_t)(sv & 0xFFu));
            ds_write4<64>(sc_wr, d * (float)(int8_t)((sv >> 8) & 0xFFu));
            ds_write4<128>(sc_wr, d * (float)(int8_t)((sv >> 16) & 0xFFu));
            ds_write4<192>(sc_wr, d * (float)(int8_t)(sv >> 24));
        } else if constexpr (F == QF_Q4_1) {  // block kq's {d, m} to [block][d, m][row]
            uint32_t sv = lds_read4<0>(h_rd + so + 4u * (uint32_t)kq);
            q8_wait_lgkm<0>();
            pin(sv);
            ds_write4<0>(sc_wr, h2f(sv & 0xFFFFu));
            ds_write4<64>(sc_wr, h2f(sv >> 16));
        } else {  // block kq's d to [block][row]
            uint32_t sv = lds_read_u16<0>(h_rd + so + 8u * (uint32_t)(c & 1) + 2u * (uint32_t)kq);
            q8_wait_lgkm<0>();
            pin(sv);
            ds_write4<0>(sc_wr, h2f(sv));
        }
    };

    // LDS reads of pair p of the chunk in the slot at byte `so`.  Q6_K: pair p
    // is quarters 2 (p & 1), 2 (p & 1) + 1 of half p / 2.
    auto read_pair = [&](auto pc, QPair<F> &q, uint32_t so) {
        constexpr int p = decltype(pc)::value;
        q.m = ds_read16<p * 256>(m_rd + so);
        if constexpr (Q::Q6) {
            // k-slice kq: ql chunks 4 o + c and 4 o + 2 + c, qh chunk 8 + 2 o
            // + c (c = kq / 2), bytes 8 (kq & 1) of row r16
            constexpr int oh = p >> 1, so6 = (8 * oh + 4 * (p & 1)) * 64;
            q.w[0] = lds_read8<oh * 1024>(w_rd[0] + so);
            q.w[1] = lds_read8<oh * 1024 + 512>(w_rd[0] + so);
            q.w[2] = lds_read8<2048 + oh * 512>(w_rd[0] + so);
            static_for<4>([&](auto i) { q.sc[decltype(i)::value] = ds_read16<so6 + 64 * decltype(i)::value>(sc_rd); });
        } else if constexpr (Q::KQ) {
            q.w[0] = lds_read8<0>(w_rd[p] + so);
            static_for<4>([&](auto i) { q.sc[decltype(i)::value] = ds_read16<256 * p + 16 * decltype(i)::value>(sc_rd); });
        } else {
            q.w[0] = lds_read8<0>(w_rd[2 * p] + so);
            q.w[1] = lds_read8<0>(w_rd[2 * p + 1] + so);
            constexpr int ns = F == QF_Q4_1 ? 4 : 2;
            static_for<ns>([&](auto i) { q.sc[decltype(i)::value] = ds_read16<64 * (ns * p + decltype(i)::value)>(sc_rd); });
        }
        if constexpr (Q::FIFTH) {
            q.fb[0] = lds_read_u8<8 * p>(f_rd + so);
            q.fb[1] = lds_read_u8<8 * p + 4>(f_rd + so);
        }
    };
    auto pin_pair = [&](QPair<F> &q) {
        pin(q.m);
        for (auto &v : q.w) pin(v);
        for (auto &v : q.sc) pin(v);
        if constexpr (Q::FIFTH) {
            pin(q.fb[0]);
            pin(q.fb[1]);
        }
    };
    auto f = [](uint32_t u) { return __uint_as_float(u); };
    auto lo16 = [](uint32_t u) { return (int)(int16_t)(u & 0xFFFFu); };
    auto hi16 = [](uint32_t u) { return (int)u >> 16; };

    // The addends of pair p: ad[unit][i], row 4 kq + i.
    auto compute = [&](auto pc, const QPair<F> &q, float (&ad)[UNITS][4]) {
        constexpr int p = decltype(pc)::value;
        const float dx0 = f(q.m[0]), dx1 = f(q.m[2]);
        const u32x4 x = xr[p];
        if constexpr (Q::KQ) {
            u32x2 lo = {q.w[0].x & NIB, q.w[0].y & NIB}, hi = {(q.w[0].x >> 4) & NIB, (q.w[0].y >> 4) & NIB};
            if constexpr (F == QF_Q5_K) {
                lo.x |= spread4_bit4(q.fb[0] & 15u);
                lo.y |= spread4_bit4(q.fb[0] >> 4);
                hi.x |= spread4_bit4(q.fb[1] & 15u);
                hi.y |= spread4_bit4(q.fb[1] >> 4);
            }
            const i32x4 il = dot16(lo, x[0], x[1]), ih = dot16(hi, x[2], x[3]);
            const float al = dx0 * (float)(lo16(q.m[1]) + hi16(q.m[1])), ah = dx1 * (float)(lo16(q.m[3]) + hi16(q.m[3]));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float va_lo = dx0 * (float)il[i], va_hi = dx1 * (float)ih[i];
                float s = f(q.sc[i][0]) * va_lo;
                s = s - f(q.sc[i][1]) * al;
                s = s + f(q.sc[i][2]) * va_hi;
                s = s - f(q.sc[i][3]) * ah;
                ad[p][i] = s;
            }
        } else if constexpr (Q::Q6) {
#pragma unroll
            for (int b = 0; b < 2; b++) {  // quarter 2 (p & 1) + b
                // low nibbles of the two ql chunks for quarters 0, 1; high for 2, 3
                const uint32_t sh = 4u * (p & 1), qs = 2u * (2 * (p & 1) + b);
                const u32x2 v = {((q.w[b].x >> sh) & NIB) | (((q.w[2].x >> qs) & 0x03030303u) << 4),
                                 ((q.w[b].y >> sh) & NIB) | (((q.w[2].y >> qs) & 0x03030303u) << 4)};
                const uint32_t x0 = x[2 * b], x1 = x[2 * b + 1];
                const float dx = b ? dx1 : dx0;
#pragma unroll
                for (int c = 0; c < 2; c++) {  // sub-block: the k-slices 2 c, 2 c + 1
                    const bool on = (kq >> 1) == c;
                    const i32x4 acc = dot16(v, on ? x0 : 0u, on ? x1 : 0u);
                    const float off = 32.0f * (float)(c ? hi16(q.m[2 * b + 1]) : lo16(q.m[2 * b + 1]));
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float t = dx * ((float)acc[i] - off);  // integers below 2^24: exact
                        ad[0][i] = ad[0][i] + f(q.sc[2 * b + c][i]) * t;
                    }
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < 2; b++) {
                u32x2 v = q.w[b];
                if constexpr (F != QF_Q8_0) v = u32x2{(v.x >> nsh) & NIB, (v.y >> nsh) & NIB};
                if constexpr (F == QF_Q5_0) {
                    v.x |= spread4_bit4(q.fb[b] & 15u);
                    v.y |= spread4_bit4(q.fb[b] >> 4);
                }
                const i32x4 acc = dot16(v, x[2 * b], x[2 * b + 1]);
                const float dx = b ? dx1 : dx0;
                const int xs = lo16(q.m[2 * b + 1]) + hi16(q.m[2 * b + 1]);
                if constexpr (F == QF_Q4_1) {
                    const float a = dx * (float)xs;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float va = dx * (float)acc[i];
                        const float u = f(q.sc[2 * b][i]) * va, m = f(q.sc[2 * b + 1][i]) * a;
                        ad[2 * p + b][i] = u + m;
                    }
                } else {
                    const float off = (float)(Q::NIBC * xs);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float iv = Q::NIBC ? (float)acc[i] - off : (float)acc[i];  // integers below 2^24: exact
                        const float sub = dx * iv;
                        ad[2 * p + b][i] = f(q.sc[b][i]) * sub;
                    }
                }
            }
        }
    };

    float sum = 0.0f;  // of row 4 (lane / 16) + wave, token lane % 16
    for (int r = 0; r < Q::RING; r++) {
        if (r == Q::RING - 1) load_x(wave);  // before the last chunk's loads, as in the loop
        issue(4 * r + wave, r);
    }
    int slot = 0;
    for (int c0 = 0; c0 < nch; c0 += 4) {
        const int c = c0 + wave;
        const uint32_t so = (uint32_t)(slot * Q::SLOT);
        // This chunk's operand has arrived, and so (in order) has every load
        // issued before it; the ring's last chunk, issued after it, need not.
        q8_wait_vm<Q::LOADS>();
        float ad[UNITS][4];
#pragma unroll
        for (int i = 0; i < 4; i++) ad[0][i] = 0.0f;
        scales(c, so);
        q8_wait_lgkm<0>();  // the table is written
        // each pair's reads in flight over the previous one's arithmetic
        QPair<F> q[2];
        read_pair(ic<0>{}, q[0], so);
        static_for<Q::NP>([&](auto pc) {
            constexpr int p = decltype(pc)::value;
            q8_wait_lgkm<0>();
            pin_pair(q[p & 1]);
            if constexpr (p + 1 < Q::NP) read_pair(ic<p + 1>{}, q[(p + 1) & 1], so);
            __builtin_amdgcn_sched_barrier(0);
            compute(pc, q[p & 1], ad);
            __builtin_amdgcn_sched_barrier(0);
        });
        __builtin_amdgcn_sched_barrier(0);
        load_x(c + 4);
        issue(c + 4 * Q::RING, slot);
        slot = slot == Q::RING - 1 ? 0 : slot + 1;
        __builtin_amdgcn_s_barrier();  // the previous round's addends are read
        static_for<4 * UNITS>([&](auto j) {
            constexpr int u = decltype(j)::value / 4, i = decltype(j)::value % 4;
            ds_write4<(4 * u + i) * 256>(part_wr, ad[u][i]);
        });
        q8_wait_lgkm<0>();
        __builtin_amdgcn_s_barrier();
        // thread (i = wave, lane): row 4 (lane / 16) + i; the round's chunks in order
        const int nv = nch - c0 < 4 ? nch - c0 : 4;
        uint32_t v[4 * UNITS];
        static_for<4 * UNITS>([&](auto j) {
            constexpr int x = decltype(j)::value / UNITS, u = decltype(j)::value % UNITS;
            v[x * UNITS + u] = lds_read4<x * Q::PART + u * 1024>(part0);
        });
        q8_wait_lgkm<0>();
#pragma unroll
        for (int j = 0; j < 4 * UNITS; j++) pin(v[j]);
#pragma unroll
        for (int x = 0; x < 4; x++)
            if (x < nv) {
#pragma unroll
                for (int u = 0; u < UNITS; u++) sum = sum + f(v[x * UNITS + u]);
            }
    }
    __builtin_amdgcn_s_waitcnt(0);  // no load still writing LDS when the wave ends
    const size_t row = row0 + (size_t)(4 * kq + wave);
    if (r16 < tokens && row < n) out[(orow + r16) * n + row] = sum;
}

// One stage (256 values) of one tile of 16 activation rows, quantized as the
// decode kernels do (quant_task_finish) into the tile layout: lane (token j,
// k-slice q) of block b writes its 8 bytes at [pair][16 q + j][b & 1] of the
// half stage, the block's {dx, sums of its two halves as int16} go to
// [pair][j][b & 1].
// SRC: the rows are activations (of token, or of the slot's token), or
// silu(A) or silu(A) * A2 of the slots.  Tokens past the tile's get zeros.
template <int SRC>
__global__ __launch_bounds__(512) void k_quantize_tiles(const float *__restrict__ A, const float *__restrict__ A2, size_t k,
                                                        int T, unsigned char *__restrict__ acts,
                                                        const MoeTile *__restrict__ tiles, const int *__restrict__ n_tiles,
                                                        const int *__restrict__ tok_of_slot) {
    const int tile = blockIdx.y, s = blockIdx.x, tid = threadIdx.x;
    int first = tile * 16, rows = T - first;
    if (n_tiles) {
        if (tile >= n_tiles[0]) return;
        first = tiles[tile].r0;
        rows = tiles[tile].rows;
    }
    const int j = tid >> 5, b = (tid >> 2) & 7, q = tid & 3;  // token, block of 32, k-slice
    const bool ok = j < rows;
    size_t r = (size_t)(first + (ok ? j : 0));
    if (SRC == Q8SRC_ROWS && tok_of_slot) r = (size_t)tok_of_slot[r];
    const size_t e = r * k + (size_t)s * QK + 32 * b + 8 * q;
    float v[8];
    load_f32x(A + e, v, 8);
    if constexpr (SRC == Q8SRC_SILU) {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = silu_ref(v[i]);
    }
    if constexpr (SRC == Q8SRC_SWIGLU) {
        float u[8];
        load_f32x(A2 + e, u, 8);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = silu_ref(v[i]) * u[i];
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        v[i] = ok ? v[i] : 0.0f;
        amax = fmaxf(amax, fabsf(v[i]));
    }
    amax = fmaxf(amax, quad_xor1f(amax));
    amax = fmaxf(amax, quad_xor2f(amax));
    const float d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    uint32_t w0 = 0, w1 = 0;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int qi = round_half_away(v[i] * id);  // |v * id| <= 127
        sum += qi;
        if (i < 4) w0 |= ((uint32_t)qi & 0xFFu) << (8 * i);
        else w1 |= ((uint32_t)qi & 0xFFu) << (8 * (i - 4));
    }
    const int half = sum + quad_xor1(sum);        // this lane's half-block of 16
    const int other = quad_xor2(half);
    unsigned char *st = acts + ((size_t)tile * gridDim.x + s) * ACT_STAGE + (b >> 2) * ACT_HALF;
    const int p = (b >> 1) & 1;  // pair of blocks of the half stage
    *reinterpret_cast<uint2 *>(st + (p * 64 + 16 * q + j) * 16 + 8 * (b & 1)) = make_uint2(w0, w1);
    if (q == 0)
        *reinterpret_cast<uint2 *>(st + 2048 + (p * 16 + j) * 16 + 8 * (b & 1)) =
            make_uint2(__float_as_uint((float)(_Float16)d), ((uint32_t)half & 0xFFFFu) | ((uint32_t)other << 16));
}

// HIP takes fewer than 2^32 threads in a dimension of a grid.
constexpr size_t MAX_BLOCKS = ((size_t)1 << 24) - 1;
// Slices of 16 rows, padded to whole turns of the XCDs.
size_t row_slices(const DevWeight &w) { return ((w.n_rows + 15) / 16 + 7) / 8 * 8; }

bool weight_ok(const DevWeight &w) {
    switch (w.dtype) {
    case T_Q4_0: case T_Q8_0: case T_Q5_0: case T_Q4_1: case T_Q4_K: case T_Q5_K: case T_Q6_K: break;
    default: return false;
    }
    // a wave's 16 rows (a 64-row group) within 32-bit offsets
    return gpu_supports(w.dtype, w.n_cols, 1) && w.n_cols % QK == 0 && 16 * w.row_stride < ((size_t)1 << 31) &&
           w.group_stride < ((size_t)1 << 31);
}

template <Q8Fmt F>
hipError_t launch_fmt(const Q8Out &o0, const Q8Out &o1, int nw, const unsigned char *acts, int T, int n_tile_max,
                      const MoeTile *tiles, const int *n_tiles, hipStream_t s) {
    const size_t blocks = row_slices(o0.w) * (size_t)n_tile_max;
    if (blocks > MAX_BLOCKS) return hipErrorInvalidValue;
    constexpr int LDS = QFmt<F>::LDS;
    hipError_t e = ensure_lds_limit((const void *)k_gemv_q8_mfma<F>, LDS);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_gemv_q8_mfma<F>, dim3((unsigned)blocks, (unsigned)nw), dim3(256), LDS, s, o0, o1, acts, T, n_tile_max,
                       tiles, n_tiles);
    return hipGetLastError();
}

hipError_t launch_any(const Q8Out &o0, const Q8Out &o1, int nw, const unsigned char *acts, int T, int n_tile_max,
                      const MoeTile *tiles, const int *n_tiles, hipStream_t s) {
    if (!weight_ok(o0.w)) return hipErrorInvalidValue;
    switch (o0.w.dtype) {
    case T_Q4_0: return launch_fmt<QF_Q4_0>(o0, o1, nw, acts, T, n_tile_max, tiles, n_tiles, s);
    case T_Q8_0: return launch_fmt<QF_Q8_0>(o0, o1, nw, acts, T, n_tile_max, tiles, n_tiles, s);
    case T_Q5_0: return launch_fmt<QF_Q5_0>(o0, o1, nw, acts, T, n_tile_max, tiles, n_tiles, s);
    case T_Q4_1: return launch_fmt<QF_Q4_1>(o0, o1, nw, acts, T, n_tile_max, tiles, n_tiles, s);
    case T_Q4_K: return launch_fmt<QF_Q4_K>(o0, o1, nw, acts, T, n_tile_max, tiles, n_tiles, s);
    case T_Q5_K: return launch_fmt<QF_Q5_K>(o0, o1, nw, acts, T, n_tile_max, tiles, n_tiles, s);
    case T_Q6_K: return launch_fmt<QF_Q6_K>(o0, o1, nw, acts, T, n_tile_max, tiles, n_tiles, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

// The formats and shapes of this form (t_rows: the decode kernels' own bound).
bool gemv_q8_mfma_supports(const DevWeight &w, size_t t_rows) {
    return weight_ok(w) && row_slices(w) <= MAX_BLOCKS && t_rows >= 2 && t_rows <= 65535 * 8;
}

bool gemv_q8_grouped_supports(const DevWeight &w, size_t n_tile_max) {
    return weight_ok(w) && n_tile_max <= 65535 && row_slices(w) * n_tile_max <= MAX_BLOCKS;
}

// Where this form is the faster one, by estimates fitted to both forms'
// times (us, quantization included) at 2-128 tokens, N 512-14336, K
// 512-14336, every format.  With t tokens, M = N K / 10^6 and tiles of 16 tokens:
//   decode kernels, the formats quantized once per launch (a row of at most
//     256 units): 5.4 + 0.022 M per token (Q8_0 past K 4096 0.032), K-quants 6.2 +
//     0.0225 M + 1.5e-5 N; tokens in fours, few rows longer (a round of
//     blocks is not full): times 1 + 256 / N;
//   Q5_0, Q4_1 (quantized inside every block, one launch less): 3.3 + the larger of a
//     chain of 0.21 per 1024 of K for each of up to eight tokens of a block and
//     M t times 0.03 (K to 512), 0.037 (2048), 0.066 (4096) or, past that, 0.08-0.2 by the
//     tokens per block (their registers spill); the smaller adds 0.6 (0.3) of itself;
//   rows of more than 256 units (blocks of 32: K > 8192, 64-groups: K > 16384), no
//     pre-quantized form: 4 + 0.2 M t, up to 3 tokens 5 + 0.1 M t;
//   Q6_K: 5 + 0.05 M t (K to 2048 0.038, 1024 0.07, 512 0.13: passes over super-blocks part filled);
//   this form: its chain over K, 1.17 (K-quants), 1.55, 1.45 (Q8_0), 1.65 (Q5_0, Q4_1), 2.5 (Q6_K) per
//     1024 of K, or its arithmetic per tile, 0.18 M + 1e-4 N, 0.215 M, 0.43 M + 3e-4 N
//     (Q6_K), whichever is larger, and 5.2-5.6; at least 7 (Q6_K 8.2).
// Measured, decode kernels / this form: Q4_K 14336x4096 at 8 / 16 / 32 / 64
// tokens 19.2 / 28.3 / 47.2 / 87.0 against 18.3 / 18.4 / 25.9 / 44.1; Q4_0 4096x14336 at
// 4 / 16 / 64 54 / 194 / 768 against 28 / 28 / 48; Q5_0 4096x512 at 4 / 32 4.1 /
// 5.3 against 6.9 / 6.9, 4096x4096 at 4 / 16 8.6 / 23.4 against 12.0 / 12.1; Q6_K 2048x5632
// at 8 / 24 / 32 11.5 / 18.5 / 22.0 against 20.2 / 20.6 / 20.6.  Of the
// 3528 shapes timed, the form taken is within 10 % of the faster one at 3489 (with one set of
// decode costs for all formats 3077: Q5_0 and Q4_1 came here at short K, 4.1 -> 7.0 us).
// RCE_QMM_Q8_MFMA: 0 = never this form, 2 = always where it applies (tests of
// both forms on the same shapes).  Read at every call, so a test can switch it.
bool gemv_q8_mfma_preferred(const DevWeight &w, size_t t_rows) {
    const char *e = getenv("RCE_QMM_Q8_MFMA");
    const int mode = e ? atoi(e) : 1;
    if (mode != 1) return mode == 2;
    const size_t K = w.n_cols;
    const double n = (double)w.n_rows, m = n * (double)K * 1e-6, t = (double)t_rows, k = (double)K / 1024.0;
    const double t4 = t_rows < 4 ? t : (double)((t_rows + 3) / 4 * 4), tiles = (double)((t_rows + 15) / 16);
    const bool q6 = w.dtype == T_Q6_K, kq = w.dtype == T_Q4_K || w.dtype == T_Q5_K;
    const bool inl = w.dtype == T_Q5_0 || w.dtype == T_Q4_1;
    double decode, self;
    if (q6) {
        decode = 5.0 + (K <= 512 ? 0.13 : K <= 1024 ? 0.07 : K <= 2048 ? 0.038 : 0.05) * m * t;
        self = std::max(8.2, 5.6 + std::max(2.5 * k, (0.43 * m + 3e-4 * n) * tiles));
    } else if (kq) {
        decode = std::max(t_rows < 4 ? 6.3 : 7.1, 6.2 + (0.0225 * m + 1.5e-5 * n) * t4 * (1.0 + 256.0 / n));
        self = std::max(7.0, 5.2 + std::max(1.17 * k, (0.18 * m + 1e-4 * n) * tiles));
    } else {
        const double chain = 0.21 * k * std::min(t, 8.0);
        const double slope = K <= 512 ? 0.03 : K <= 2048 ? 0.037 : K <= 4096 ? 0.066 : t_rows >= 8 ? 0.2 : t_rows >= 4 ? 0.13 : 0.08;
        if (inl) decode = 3.3 + std::max(chain, slope * m * t) + (K <= 2048 ? 0.6 : K <= 4096 ? 0.3 : 0.0) * std::min(chain, slope * m * t);
        else decode = std::max(6.4, 5.4 + (w.dtype == T_Q8_0 && K > 4096 ? 0.032 : 0.022) * m * t4 * (1.0 + 256.0 / n));
        self = std::max(6.9, 5.6 + std::max((inl ? 1.65 : w.dtype == T_Q8_0 ? 1.45 : 1.55) * k, 0.215 * m * tiles));
    }
    if (!q6 && nt_for(units_per_row(w.dtype, K)) != 256) decode = t_rows >= 4 ? 4.0 + 0.2 * m * t : 5.0 + 0.1 * m * t;
    return self < decode;
}

size_t gemv_q8_tile_bytes(size_t n_cols) { return n_cols / QK * ACT_STAGE; }

hipError_t launch_quantize_tiles(int src, const float *a, const float *a2, size_t k, size_t t_rows, int n_tile_max,
                                 const MoeTile *tiles, const int *n_tiles, const int *tok_of_slot, void *acts,
                                 hipStream_t s) {
    unsigned char *q = static_cast<unsigned char *>(acts);
    const dim3 grid((unsigned)(k / QK), (unsigned)n_tile_max);
    if (n_tile_max > 65535) return hipErrorInvalidValue;
    if (src == Q8SRC_ROWS)
        hipLaunchKernelGGL(k_quantize_tiles<Q8SRC_ROWS>, grid, dim3(512), 0, s, a, a2, k, (int)t_rows, q, tiles, n_tiles, tok_of_slot);
    else if (src == Q8SRC_SILU)
        hipLaunchKernelGGL(k_quantize_tiles<Q8SRC_SILU>, grid, dim3(512), 0, s, a, a2, k, (int)t_rows, q, tiles, n_tiles, tok_of_slot);
    else
        hipLaunchKernelGGL(k_quantize_tiles<Q8SRC_SWIGLU>, grid, dim3(512), 0, s, a, a2, k, (int)t_rows, q, tiles, n_tiles, tok_of_slot);
    return hipGetLastError();
}

hipError_t launch_gemv_q8_mfma(const DevWeight &w, const float *a, size_t t_rows, float *out, void *acts, hipStream_t s) {
    if (t_rows == 0 || w.n_rows == 0) return hipSuccess;
    if (!gemv_q8_mfma_supports(w, t_rows)) return hipErrorInvalidValue;
    const int nt = (int)((t_rows + 15) / 16);
    hipError_t e = launch_quantize_tiles(Q8SRC_ROWS, a, nullptr, w.n_cols, t_rows, nt, nullptr, nullptr, nullptr, acts, s);
    if (e != hipSuccess) return e;
    // as many tiles a launch as its grid takes
    const int per = (int)std::min<size_t>(MAX_BLOCKS / row_slices(w), (size_t)nt);
    const unsigned char *q = static_cast<const unsigned char *>(acts);
    for (int g = 0; g < nt && e == hipSuccess; g += per) {
        const size_t t0 = 16 * (size_t)g;
        const Q8Out o{w, nullptr, out + t0 * w.n_rows};
        e = launch_any(o, o, 1, q + (size_t)g * gemv_q8_tile_bytes(w.n_cols), (int)(t_rows - t0), std::min(per, nt - g), nullptr,
                       nullptr, s);
    }
    return e;
}

hipError_t launch_gemv_q8_grouped(const DevWeight &w, const DevWeight *wtab, float *out, const DevWeight *wtab2, float *out2,
                                  const void *acts, int n_tile_max, const MoeTile *tiles, const int *n_tiles, hipStream_t s) {
    const Q8Out o0{w, wtab, out}, o1{w, wtab2, out2};
    return launch_any(o0, o1, wtab2 ? 2 : 1, static_cast<const unsigned char *>(acts), 0, n_tile_max, tiles, n_tiles, s);
}

hipError_t q8_mfma_prepare_lds() {
    hipError_t e = hipSuccess;
    auto one = [&](const void *fn, int bytes) {
        if (e == hipSuccess) e = ensure_lds_limit(fn, bytes);
    };
    one((const void *)k_gemv_q8_mfma<QF_Q4_0>, QFmt<QF_Q4_0>::LDS);
    one((const void *)k_gemv_q8_mfma<QF_Q8_0>, QFmt<QF_Q8_0>::LDS);
    one((const void *)k_gemv_q8_mfma<QF_Q5_0>, QFmt<QF_Q5_0>::LDS);
    one((const void *)k_gemv_q8_mfma<QF_Q4_1>, QFmt<QF_Q4_1>::LDS);
    one((const void *)k_gemv_q8_mfma<QF_Q4_K>, QFmt<QF_Q4_K>::LDS);
    one((const void *)k_gemv_q8_mfma<QF_Q5_K>, QFmt<QF_Q5_K>::LDS);
    one((const void *)k_gemv_q8_mfma<QF_Q6_K>, QFmt<QF_Q6_K>::LDS);
    return e;
}

}  // namespace rce_qmm
