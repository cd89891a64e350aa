// gemm_wide.hip -- the prefill GEMM for many tokens on the CDNA4 matrix
// cores: out[M, N] = A[M, K] . W[N, K]^T in tiles of up to 256 x 256, W in
// GGUF blocks (Q4_K, Q5_K, Q4_0, Q4_1, Q5_0, Q8_0, Q6_K) dequantized to
// binary16 fragments in registers, or plain F16, contracted with
// v_mfma_f32_32x32x16_f16 (f32 accumulation).
//
// The 128 x 64 tile of gemm_f16.hip copies 18 KB into LDS per 64-wide chunk
// for 256 MFMA cycles per SIMD, 70 B/clk per CU, and waits for those copies.
// Here a 256 x 256 tile copies 41 KB (Q4_K) for 2048 MFMA cycles, 20 B/clk.
// Counted at 4096 x 14336 x 4096 (Q4_K, 463 us at the 1.6 GHz the chip holds):
// the matrix cores busy 63 % of the cycles, 4.9 other vector instructions and
// 1.1 LDS instructions per MFMA, LDS bank conflicts (the reads of raw weight bytes; A's
// have none) 18 % of a CU's cycles, A and W read 6 times from HBM between the eight L2s.
//
// Work split.  Eight waves, 2 (M) x 4 (N): a wave owns RB x CB blocks of
// 32 x 32 outputs (tile 64 RB x 128 CB) over all of K, one accumulator
// chain per output (k-steps of 16 in order).  Each wave dequantizes the W
// fragments it consumes (each weight twice per tile, once per M half: four
// vector instructions per MFMA at RB = 4) from the raw bytes in LDS, so no
// binary16 W tile is written.
//
// Pipeline.  K runs in chunks of 64 (four k-steps).  A is staged NSA - 1
// chunks ahead, W one stage of SK (128 or 64) K ahead, all with direct
// global -> LDS loads spread evenly over the waves.  One barrier per chunk,
// before its last k-step: by then every wave holds that k-step's fragments
// in registers, so the barrier frees the chunk's stage and the 8 MFMAs of
// the last k-step hide the first LDS reads of the next chunk.  Within a
// k-step the next one's raw weights and A fragments are read first, half of
// the MFMAs run while they arrive, and the dequantization is spread between
// the other half.
//
// A: 128 bytes per row and chunk, 16-byte column g of row r at slot
// g ^ f(r) (f(r) = (r & 7) ^ ((r >> 3) & 1)), the swizzle of gemm_f16.hip:
// fragment reads are conflict free.  Rows past M read past the buffer's end
// and land zeros.  W: per field of FB bytes per row and stage, 16-byte
// pieces rotated by the row; rows past N repeat the last row (never
// stored).
#include "lds_limit.h"
#include "mfma_util.h"
#include "qmm_internal.h"

#include <algorithm>

namespace rce_qmm {
namespace {

constexpr int WKC = 64;          // K per chunk
constexpr int WNT = 512;         // threads: 8 waves
constexpr int WIDE_LDS = 160 * 1024;

// --- weight formats ------------------------------------------------------------
// Per stage of SK K positions a row has up to three fields of FB[i] bytes
// (a multiple of 16, at most 64) at byte src(w, i, stage) of the row; the
// tile's rows of field i lie at foff<BN>(i) of the stage in LDS.  For k-step
// kq of chunk u of the stage: the lane's eight weights are the 8 bytes at
// piece wpiece(u, kq), lane half h, of field wfield(kq) (4-bit formats: one
// nibble, shift wshift(kq)); acol(kq) is the 16-byte A column of lane half
// 0; the {scale, bias} word (SBW bytes zero-extended) is at byte
// sbyte(par, u, kq) of the row's field SF, par = stage & 1; formats with
// fifth bits (HB) keep them in field 2, the lane's eight at byte hbyte(u,
// kq) + h.
enum WideKind { WK_SPLIT, WK_Q6K, WK_F16 };

struct WQ4K {
    static constexpr WideKind KIND = WK_SPLIT;
    static constexpr int SK = 128, OFF = 1024, SBW = 4, NF = 3, SF = 2;
    static constexpr bool HB = false;
    static constexpr int fb(int i) { return i < 2 ? 32 : 16; }
    __device__ static size_t src(const DevWeight &w, int i, int s) {
        return i == 0 ? w.plane1 + 32 * (size_t)s : i == 1 ? w.plane2 + 32 * (size_t)s : w.plane4 + 16 * (size_t)s;
    }
    static constexpr int wfield(int kq) { return kq >> 1; }
    static constexpr int wpiece(int u, int) { return u; }
    static constexpr int wshift(int kq) { return 4 * (kq & 1); }
    static constexpr int acol(int kq) { return (kq & 1) * 4 + (kq >> 1) * 2; }
    static constexpr int sbyte(int, int u, int kq) { return 4 * (2 * u + (kq & 1)); }
    static constexpr int hbyte(int, int) { return 0; }
    __device__ static uint32_t vals(uint32_t x, int sh) { return (x >> sh) & 0x0F0F0F0Fu; }
};
// Q5_K: Q4_K's fields and, per 64-group, the 8-byte word of fifth bits.
struct WQ5K : WQ4K {
    static constexpr int NF = 4;
    static constexpr bool HB = true;
    static constexpr int fb(int i) { return i < 2 ? 32 : 16; }
    __device__ static size_t src(const DevWeight &w, int i, int s) {
        return i == 3 ? w.plane3 + 16 * (size_t)s : WQ4K::src(w, i, s);
    }
    static constexpr int hbyte(int u, int kq) { return 8 * u + 4 * (kq & 1) + 2 * (kq >> 1); }
};
// Q4_0: the stage's four blocks are 64 contiguous nibble bytes; the header
// field is the 16 bytes of f16 scales of the stage pair's eight blocks.
struct WQ40 {
    static constexpr WideKind KIND = WK_SPLIT;
    static constexpr int SK = 128, OFF = 1032, SBW = 2, NF = 2, SF = 1;
    static constexpr bool HB = false;
    static constexpr int fb(int i) { return i == 0 ? 64 : 16; }
    __device__ static size_t src(const DevWeight &w, int i, int s) {
        return i == 0 ? w.plane1 + 64 * (size_t)s : 16 * (size_t)(s >> 1);
    }
    static constexpr int wfield(int) { return 0; }
    static constexpr int wpiece(int u, int kq) { return 2 * u + (kq >> 1); }
    static constexpr int wshift(int kq) { return 4 * (kq & 1); }
    static constexpr int acol(int kq) { return 2 * kq; }
    static constexpr int sbyte(int par, int u, int kq) { return 8 * par + 2 * (2 * u + (kq >> 1)); }
    static constexpr int hbyte(int, int) { return 0; }
    __device__ static uint32_t vals(uint32_t x, int sh) { return (x >> sh) & 0x0F0F0F0Fu; }
};
// Q4_1: the header field is the stage's four {d, m} words.
struct WQ41 : WQ40 {
    static constexpr int OFF = 1024, SBW = 4;
    __device__ static size_t src(const DevWeight &w, int i, int s) {
        return i == 0 ? w.plane1 + 64 * (size_t)s : 16 * (size_t)s;
    }
    static constexpr int sbyte(int, int u, int kq) { return 4 * (2 * u + (kq >> 1)); }
};
// Q5_0: Q4_0's fields and the stage's four qh words.
struct WQ50 : WQ40 {
    static constexpr int OFF = 1040, NF = 3;
    static constexpr bool HB = true;
    static constexpr int fb(int i) { return i == 0 ? 64 : 16; }
    __device__ static size_t src(const DevWeight &w, int i, int s) {
        return i == 2 ? w.plane2 + 16 * (size_t)s : WQ40::src(w, i, s);
    }
    static constexpr int hbyte(int u, int kq) { return 4 * (2 * u + (kq >> 1)) + 2 * (kq & 1); }
};
// Q8_0: bytes 0..15 and 16..31 of the stage's four blocks, 64 contiguous
// bytes of either plane.
struct WQ80 {
    static constexpr WideKind KIND = WK_SPLIT;
    static constexpr int SK = 128, OFF = 1152, SBW = 2, NF = 3, SF = 2;
    static constexpr bool HB = false;
    static constexpr int fb(int i) { return i < 2 ? 64 : 16; }
    __device__ static size_t src(const DevWeight &w, int i, int s) {
        return i == 0 ? w.plane1 + 64 * (size_t)s : i == 1 ? w.plane2 + 64 * (size_t)s : 16 * (size_t)(s >> 1);
    }
    static constexpr int wfield(int kq) { return kq & 1; }
    static constexpr int wpiece(int u, int kq) { return 2 * u + (kq >> 1); }
    static constexpr int wshift(int) { return 0; }
    static constexpr int acol(int kq) { return (kq >> 1) * 4 + (kq & 1) * 2; }
    static constexpr int sbyte(int par, int u, int kq) { return 8 * par + 2 * (2 * u + (kq >> 1)); }
    static constexpr int hbyte(int, int) { return 0; }
    __device__ static uint32_t vals(uint32_t x, int) { return x ^ 0x80808080u; }
};
// Q6_K (64-row groups): per group and half super-block 6 KB of ql (4
// chunks) and qh (2), then 2 KB of pairs [pair][row]; k-step kq of chunk u:
// ql chunk kq, nibble u; qh chunk kq & 1, bits 2 (2u + kq / 2); pair 4u + kq.
struct WQ6K {
    static constexpr WideKind KIND = WK_Q6K;
    static constexpr int SK = 128, OFF = 1024, NF = 0;
    static constexpr bool HB = false;
    static constexpr int fb(int) { return 0; }
    static constexpr int acol(int kq) { return (kq >> 1) * 4 + (kq & 1) * 2; }
};
// F16 (64-row groups of 16-byte chunks): a 64-K stage is eight contiguous KB
// per group, read as fragments as they stand.
struct WF16 {
    static constexpr WideKind KIND = WK_F16;
    static constexpr int SK = 64, OFF = 0, NF = 0;
    static constexpr bool HB = false;
    static constexpr int fb(int) { return 0; }
    static constexpr int acol(int kq) { return 2 * kq; }
};

template <class F, int RB, int CB>
struct WideTile {
    static constexpr int BM = 64 * RB, BN = 128 * CB;
    static constexpr int CPS = F::SK / WKC;  // chunks per W stage
    static constexpr int field_off(int i) {
        int o = 0;
        for (int j = 0; j < i; j++) o += BN * F::fb(j);
        return o;
    }
    static constexpr int W_STAGE = F::KIND == WK_SPLIT ? field_off(F::NF) : BN / 64 * 8192;
    static constexpr int A_STAGE = BM * WKC * 2;
    // Stages: A NSA, W NSW (each the most that fit: the ring of four needs
    // no wait for the LDS reads in flight before a barrier, below), loaded
    // APD chunks / WPD W stages ahead; D: k-steps the LDS reads of A run
    // ahead of their MFMAs.
    static constexpr bool F16W = F::KIND == WK_F16;
    static constexpr int NSW = F16W ? (4 * A_STAGE + 4 * W_STAGE <= WIDE_LDS ? 4 : 3 * A_STAGE + 3 * W_STAGE <= WIDE_LDS ? 3 : 2) : 2;
    static constexpr int NSA = 4 * A_STAGE + NSW * W_STAGE <= WIDE_LDS ? 4 : 3 * A_STAGE + NSW * W_STAGE <= WIDE_LDS ? 3 : 2;
    static constexpr int APD = NSA > 2 ? 2 : 1, WPD = NSW > 2 ? 2 : 1;
    static constexpr int D = APD == 2 && (!F16W || WPD == 2) ? 2 : 1;
    static constexpr bool PREWAIT = D == 1 || NSA < 4 || (F16W && NSW < 4);
    static constexpr int OFF_W = NSA * A_STAGE;
    static constexpr int LDS = OFF_W + NSW * W_STAGE;
    static_assert(LDS <= WIDE_LDS, "LDS budget");
    // accumulator chains per output: F16 weights, whose only rounding is the
    // accumulation's, add two (even and odd k-steps) at the end
    static constexpr int NCH = F16W ? 2 : 1;
    static constexpr int RW = BN / 8;      // W rows per wave and field
    static constexpr int A_LOADS = RB;     // per wave and chunk (1 KB each)
    static constexpr int field_loads(int i) { return RW * F::fb(i) > 1024 ? RW * F::fb(i) / 1024 : 1; }
    static constexpr int first_load(int f) {
        int n = 0;
        for (int i = 0; i < f; i++) n += field_loads(i);
        return n;
    }
    static constexpr int load_field(int l) {
        int f = 0;
        while (first_load(f + 1) <= l) f++;
        return f;
    }
    static constexpr int W_LOADS = F::KIND == WK_SPLIT ? first_load(F::NF) : BN / 64;  // per wave and stage
    // Loads a wave may still have in flight at the barrier of chunk u of a
    // stage.  Chunk c issues [W stage s + WPD at the stage's first chunk],
    // then A of chunk c + APD; past the barrier A of chunk c + 1 is read,
    // and W of the next stage from the barrier of the stage's last chunk
    // (D = 2) or, the raw weights being read two k-steps ahead, one k-step
    // before it (D = 1), so from the barrier one chunk earlier.
    static constexpr int vm_after(int u) {
        if (APD == 1) return 0;
        const bool w_open = F16W ? WPD == 2 : D == 2 && u == 0 && CPS > 1;
        return A_LOADS + (w_open ? W_LOADS : 0);
    }
};

template <int N>
__device__ __forceinline__ void wait_lgkm() {
    static_assert(N >= 0 && N < 16, "lgkmcnt range");
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
// Tile p of a band-ordered numbering: bands of four row tiles, column tiles
// next, so that the tiles an XCD runs together share four row tiles of A and
// a few of W in its L2.
__device__ __forceinline__ void wide_tile(int p, int m_tiles, int n_tiles, int &mt, int &nt) {
    const int band = p / (4 * n_tiles), r = p - band * 4 * n_tiles;
    const int bm = m_tiles - 4 * band < 4 ? m_tiles - 4 * band : 4;
    mt = 4 * band + r % bm;
    nt = r / bm;
}

// Block L of n: XCD x (blocks x, x + 8, ..) takes a contiguous run.
__device__ __forceinline__ int xcd_run(int L, int n) {
    const int q = n / 8, r = n % 8, x = L % 8;
    return x * q + (x < r ? x : r) + L / 8;
}

// One output tile: rows m0 .. m0 + BM - 1 (those below M), columns n0 ..
template <class F, int RB, int CB>
__device__ __forceinline__ void wide_body(const DevWeight &w, const _Float16 *__restrict__ A, size_t M,
                                          float *__restrict__ out, size_t m0, size_t n0, unsigned char *lds) {
    using T = WideTile<F, RB, CB>;
    constexpr int BM = T::BM, BN = T::BN, NSA = T::NSA, CPS = T::CPS, NSW = T::NSW, D = T::D, NCH = T::NCH;
    const size_t N = w.n_rows, K = w.n_cols;
    const int rows = (int)(M - m0 < (size_t)BM ? M - m0 : BM);
    const int cols = (int)(N - n0 < (size_t)BN ? N - n0 : BN);
    const int nchunks = (int)(K / WKC), nstages = nchunks / CPS;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 2, wn = wave & 3, l32 = lane & 31, h = lane >> 5;
    const uint32_t lds0 = lds_addr(lds);

    // ---- loads: per-lane offsets
    const __amdgpu_buffer_rsrc_t abuf = byte_buffer(A + m0 * K, (uint32_t)((size_t)rows * K * 2));
    uint32_t a_off[T::A_LOADS];
#pragma unroll
    for (int i = 0; i < T::A_LOADS; i++) {  // 8 rows x 128 bytes per load
        const int r = 8 * (wave * T::A_LOADS + i) + (lane >> 3), f = (r & 7) ^ ((r >> 3) & 1);
        a_off[i] = (uint32_t)r * (uint32_t)(2 * K) + 16u * (uint32_t)((lane & 7) ^ f);
    }
    const __amdgpu_buffer_rsrc_t wbuf =
        F::KIND == WK_SPLIT ? byte_buffer(w.base + n0 * w.row_stride, (uint32_t)((size_t)cols * w.row_stride))
                            : byte_buffer(w.base + (n0 >> 6) * w.group_stride,
                                          (uint32_t)((size_t)((cols + 63) >> 6) * w.group_stride));
    // split formats: row and rotated piece of this lane for 16-, 32- and
    // 64-byte fields (one load covers 64, 32 or 16 rows)
    uint32_t w_off[3][2];
    if constexpr (F::KIND == WK_SPLIT) {
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int lpr = 1 << c, r = wave * T::RW + i * (64 / lpr) + lane / lpr;
                const int rot = c == 2 ? (r >> 2) & 3 : c == 1 ? (r >> 3) & 1 : 0;
                const int rc = r < cols ? r : cols - 1;
                w_off[c][i] = (uint32_t)((size_t)rc * w.row_stride) + 16u * (uint32_t)((lane & (lpr - 1)) ^ rot);
            }
    }
    // W stage s's slot in the ring (NSW = 3 counts through a carried index)
    auto wslot = [&](int s) { return NSW == 3 ? s % 3 : s & (NSW - 1); };
    // A load i of chunk c into stage `stage`; W load i of stage s.
    auto load_a = [&](auto ic_, int c, int stage) {
        constexpr int i = decltype(ic_)::value;
        const uint32_t soff = (uint32_t)(c < nchunks ? c : nchunks - 1) * (WKC * 2);
        buf_load_lds16(abuf, a_off[i], soff, lds + stage * T::A_STAGE + wave * (T::A_LOADS * 1024) + i * 1024);
    };
    auto load_w = [&](auto ic_, int s) {
        constexpr int i = decltype(ic_)::value;
        unsigned char *dst = lds + T::OFF_W + wslot(s) * T::W_STAGE;
        const int ss = s < nstages ? s : nstages - 1;
        if constexpr (F::KIND == WK_SPLIT) {
            constexpr int f = T::load_field(i), k = i - T::first_load(f), fb = F::fb(f), c = fb == 64 ? 2 : fb == 32 ? 1 : 0;
            constexpr int RW = T::RW;
            if (RW * fb >= 1024 || lane < RW * fb / 16)
                buf_load_lds16(wbuf, w_off[c][k], (uint32_t)F::src(w, f, ss),
                               dst + T::field_off(f) + wave * RW * fb + k * 1024);
        } else {
            // KB `wave` of the stage's eight of group i
            const int ngroups = (cols + 63) >> 6;
            const uint32_t gb = (uint32_t)((size_t)(i < ngroups ? i : ngroups - 1) * w.group_stride);
            uint32_t kb;
            if constexpr (F::KIND == WK_Q6K) {
                const int n = ss & 1;
                const uint32_t sb = (uint32_t)(ss >> 1) * (uint32_t)IL64_Q6K_SB;
                kb = sb + (wave < 4   ? (uint32_t)(4 * n + wave) * 1024u
                           : wave < 6 ? (uint32_t)(8 + 2 * n + wave - 4) * 1024u
                                      : (uint32_t)IL64_Q6K_P + (uint32_t)(2 * n + wave - 6) * 1024u);
            } else {
                kb = (uint32_t)(8 * ss + wave) * 1024u;
            }
            buf_load_lds16(wbuf, 16u * (uint32_t)lane, gb + kb, dst + i * 8192 + wave * 1024);
        }
    };

    // ---- LDS read addresses (stage 0); 32-row and 32-column blocks are
    // immediates
    uint32_t a_rd[4];
    {
        const uint32_t f = (uint32_t)((l32 & 7) ^ ((l32 >> 3) & 1)) ^ (uint32_t)h;
        const uint32_t row = lds0 + (uint32_t)((wm * 32 * RB + l32) * 128);
#pragma unroll
        for (int kq = 0; kq < 4; kq++) a_rd[kq] = row + 16u * (f ^ (uint32_t)F::acol(kq));
    }
    const int ncol = wn * 32 * CB + l32;  // tile column of this lane in column block 0
    // split formats: byte 8h of piece p of the column's row (64-byte fields:
    // p = 0..3; 32-byte: p = 0, 1), its scale word and fifth bits;
    // 64-row groups: byte 8h (Q6_K) or 0 (F16) of the column in its group
    uint32_t w_rd[4], s_rd = 0, h_rd = 0;
    constexpr int WFB = F::KIND == WK_SPLIT ? F::fb(0) : 16;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        if constexpr (F::KIND == WK_SPLIT) {
            const int rot = WFB == 64 ? (ncol >> 2) & 3 : (ncol >> 3) & 1, np = WFB / 16;
            w_rd[p] = lds0 + T::OFF_W + (uint32_t)(ncol * WFB + 16 * ((p & (np - 1)) ^ rot) + 8 * h);
        } else if constexpr (F::KIND == WK_Q6K) {
            w_rd[p] = lds0 + T::OFF_W + (uint32_t)((ncol >> 6) * 8192 + (ncol & 63) * 16 + 8 * h);
        } else {
            w_rd[p] = lds0 + T::OFF_W + (uint32_t)((ncol >> 6) * 8192 + (ncol & 63) * 16 + 1024 * h);
        }
    }
    if constexpr (F::KIND == WK_SPLIT) {
        s_rd = lds0 + T::OFF_W + (uint32_t)(T::field_off(F::SF) + ncol * F::fb(F::SF));
        if constexpr (F::HB) h_rd = lds0 + T::OFF_W + (uint32_t)(T::field_off(F::NF - 1) + ncol * 16 + h);
    } else if constexpr (F::KIND == WK_Q6K) {
        s_rd = lds0 + T::OFF_W + (uint32_t)((ncol >> 6) * 8192 + 6144 + (ncol & 63) * 4);
    }

    f32x16 acc[NCH][RB][CB];
#pragma unroll
    for (int k = 0; k < NCH; k++)
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int j = 0; j < CB; j++) acc[k][i][j] = f32x16{};

    // One k-step's raw weights of this lane, per column block.
    struct Raw {
        u32x2 l[CB], q[CB];   // bytes; Q6_K: and qh bytes
        uint32_t s[CB], b[CB];  // scale word; fifth bits
        half8 f[CB];          // F16: the fragment itself
    };
    // Read k-step kq of chunk u (of a stage of parity par, W buffer base
    // wb): the weights, then the A fragments (stage base ab).
    auto read_w = [&](auto uc, auto kc, Raw &r, uint32_t wb, int par) {
        constexpr int u = decltype(uc)::value, kq = decltype(kc)::value;
        if constexpr (F::KIND == WK_SPLIT) {
            constexpr int fo = T::field_off(F::wfield(kq)), pc = F::wpiece(u, kq);
            const uint32_t a = w_rd[pc] + wb;
            r.l[0] = lds_read8<fo>(a);
            if constexpr (CB > 1) r.l[1] = lds_read8<fo + 32 * WFB>(a);
            constexpr int so = F::sbyte(0, u, kq);
            const uint32_t sa = s_rd + wb + (F::SBW == 2 ? 8u * (uint32_t)par : 0u);
            if constexpr (F::SBW == 2) {
                r.s[0] = lds_read_u16<so>(sa);
                if constexpr (CB > 1) r.s[1] = lds_read_u16<so + 32 * F::fb(F::SF)>(sa);
            } else {
                r.s[0] = lds_read4<so>(sa);
                if constexpr (CB > 1) r.s[1] = lds_read4<so + 32 * F::fb(F::SF)>(sa);
            }
            if constexpr (F::HB) {
                constexpr int ho = F::hbyte(u, kq);
                r.b[0] = lds_read_u8<ho>(h_rd + wb);
                if constexpr (CB > 1) r.b[1] = lds_read_u8<ho + 32 * 16>(h_rd + wb);
            }
        } else if constexpr (F::KIND == WK_Q6K) {
            const uint32_t a = w_rd[0] + wb, sa = s_rd + wb;
            r.l[0] = lds_read8<kq * 1024>(a);
            r.q[0] = lds_read8<(4 + (kq & 1)) * 1024>(a);
            r.s[0] = lds_read4<(4 * u + kq) * 256>(sa);
            if constexpr (CB > 1) {
                r.l[1] = lds_read8<kq * 1024 + 512>(a);
                r.q[1] = lds_read8<(4 + (kq & 1)) * 1024 + 512>(a);
                r.s[1] = lds_read4<(4 * u + kq) * 256 + 128>(sa);
            }
        } else {
            const uint32_t a = w_rd[0] + wb;
            r.f[0] = lds_read_frag<kq * 2048>(a);
            if constexpr (CB > 1) r.f[1] = lds_read_frag<kq * 2048 + 512>(a);
        }
    };
    auto read_a = [&](half8 *a, uint32_t addr) {
        a[0] = lds_read_frag<0>(addr);
        a[1] = lds_read_frag<4096>(addr);
        if constexpr (RB > 2) a[2] = lds_read_frag<8192>(addr);
        if constexpr (RB > 3) a[3] = lds_read_frag<12288>(addr);
    };
    auto pin_raw = [&](Raw &r) {
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            if constexpr (F::KIND == WK_F16) {
                pin(r.f[cb]);
            } else {
                pin(r.l[cb]);
                pin(r.s[cb]);
                if constexpr (F::KIND == WK_Q6K) pin(r.q[cb]);
                if constexpr (F::HB) pin(r.b[cb]);
            }
        }
    };
    // word i (0, 1) of the eight weights of column block cb as byte values
    auto bytes = [&](auto uc, auto kc, const Raw &r, int cb, int i) -> uint32_t {
        constexpr int u = decltype(uc)::value, kq = decltype(kc)::value;
        const uint32_t x = i ? r.l[cb].y : r.l[cb].x;
        if constexpr (F::KIND == WK_Q6K) {
            const uint32_t y = i ? r.q[cb].y : r.q[cb].x;
            return ((x >> (4 * u)) & 0x0F0F0F0Fu) | (((y >> (2 * (2 * u + (kq >> 1)))) & 0x03030303u) << 4);
        } else if constexpr (F::HB) {
            const uint32_t b4 = i ? (r.b[cb] >> 4) & 15u : r.b[cb] & 15u;
            return F::vals(x, F::wshift(kq)) | (((b4 * 0x00204081u) & 0x01010101u) << 4);
        } else if constexpr (F::KIND == WK_SPLIT) {
            return F::vals(x, F::wshift(kq));
        } else {
            return x;
        }
    };

    // Half p of word i: two weights as a packed binary16 pair.
    auto deq2 = [&](uint32_t x, uint32_t sb, int p) -> half2v {
        const half2v moff = {(_Float16)(-(float)F::OFF), (_Float16)(-(float)F::OFF)}, v = as_h2(sb);
        const half2v sc = __builtin_shufflevector(v, v, 0, 0), bias = __builtin_shufflevector(v, v, 1, 1);
        const uint32_t u = __builtin_amdgcn_perm(x, 0x64646464u, p ? 0x00070006u : 0x00050004u);
        return __builtin_elementwise_fma(as_h2(u) + moff, sc, bias);
    };

    // ---- prologue: the first APD chunks of A and WPD stages of W
    static_for<T::W_LOADS>([&](auto i) { load_w(i, 0); });
    static_for<T::A_LOADS>([&](auto i) { load_a(i, 0, 0); });
    if constexpr (T::WPD == 2) static_for<T::W_LOADS>([&](auto i) { load_w(i, 1); });
    if constexpr (T::APD == 2) static_for<T::A_LOADS>([&](auto i) { load_a(i, 1, 1); });
    wait_vm_barrier<(T::APD - 1) * T::A_LOADS + (T::WPD - 1) * T::W_LOADS>();
    // K-step j's A fragments (F16: and W fragments) live in slot j, its raw
    // weights and dequantized fragments in slot j & 1: fixed registers over
    // the chunks, so a read in flight is never copied.
    half8 a[4][RB], b[F::KIND == WK_F16 ? 4 : 2][CB];
    Raw raw[2];
    {
        read_w(ic<0>{}, ic<0>{}, raw[0], 0, 0);
        read_w(ic<0>{}, ic<1>{}, raw[1], 0, 0);
        read_a(a[0], a_rd[0]);
        read_a(a[1], a_rd[1]);
        wait_lgkm<0>();
        pin_raw(raw[0]);
        pin_raw(raw[1]);
#pragma unroll
        for (int i = 0; i < RB; i++) {
            pin(a[0][i]);
            pin(a[1][i]);
        }
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            if constexpr (F::KIND == WK_F16) {
                b[0][cb] = raw[0].f[cb];
                b[1][cb] = raw[1].f[cb];
            } else {
                const uint32_t x0 = bytes(ic<0>{}, ic<0>{}, raw[0], cb, 0), x1 = bytes(ic<0>{}, ic<0>{}, raw[0], cb, 1);
                const uint32_t sc = raw[0].s[cb];
                b[0][cb] = join8(deq2(x0, sc, 0), deq2(x0, sc, 1), deq2(x1, sc, 0), deq2(x1, sc, 1));
            }
        }
    }

    constexpr int JB = 4 - D;  // the barrier's k-step: before the first read of the next chunk's A
    constexpr int LOAD_STEPS = T::APD == 2 ? JB : 2;
    int st = 0, ws = 0;  // A stage of chunk c, W slot of stage s
    for (int c = 0, s = 0; c < nchunks; c += CPS, s++) {
        const int ws1 = ws == NSW - 1 ? 0 : ws + 1;
        auto chunk = [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            const int cu = c + u, st1 = st == NSA - 1 ? 0 : st + 1;  // chunk, stage of the next chunk
            // The loads go out one at a time between the MFMAs of k-steps
            // 0 .. LOAD_STEPS - 1: [W stage s + WPD], then A of chunk cu +
            // APD.  The slots they fill were read last in chunk cu - 1
            // (NSA = 4: cu - 2) or before and freed by that chunk's barrier.
            constexpr int WL = u == 0 ? T::W_LOADS : 0, NL = WL + T::A_LOADS;
            const int ca = cu + T::APD, sta = st + T::APD >= NSA ? st + T::APD - NSA : st + T::APD;
            auto step = [&](auto jc) {
                constexpr int j = decltype(jc)::value;
                constexpr int ja = (j + D) & 3, jn = (j + 1) & 3, j2 = (j + 2) & 3;
                constexpr bool a_over = j + D > 3, n_over = j == 3, w_over = j + 2 > 3;  // of the next chunk
                constexpr int un = n_over ? (u + 1) % CPS : u, u2 = w_over ? (u + 1) % CPS : u;
                if constexpr (j == JB) wait_vm_barrier<T::vm_after(u)>();
                constexpr int NM = RB * CB, ND = F::KIND == WK_F16 ? 0 : 4 * CB;  // MFMAs, weight pairs of the step
                half2v hq[CB][4];
                uint32_t x = 0;
                auto slice = [&](auto tc) {
                    constexpr int t = decltype(tc)::value, cb = t / RB, rb = t % RB, ch = j % NCH;
                    acc[ch][rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[j][rb], b[F::KIND == WK_F16 ? j : j & 1][cb],
                                                                             acc[ch][rb][cb], 0, 0, 0);
                    if constexpr (t == 0) {  // LDS reads
                        if constexpr (F::KIND == WK_F16) {
                            Raw r;
                            read_w(ic<0>{}, ic<ja>{}, r, (uint32_t)((a_over ? ws1 : ws) * T::W_STAGE), 0);
#pragma unroll
                            for (int i = 0; i < CB; i++) b[ja][i] = r.f[i];
                        } else {
                            constexpr bool nxt = w_over && u == CPS - 1;
                            read_w(ic<u2>{}, ic<j2>{}, raw[j & 1], (uint32_t)((nxt ? ws1 : ws) * T::W_STAGE), (nxt ? s + 1 : s) & 1);
                        }
                        read_a(a[ja], a_rd[ja] + (uint32_t)((a_over ? st1 : st) * T::A_STAGE));
                    }
                    if constexpr (j < LOAD_STEPS) {
                        constexpr int g = j * NM + t, l0 = g * NL / (LOAD_STEPS * NM), l1 = (g + 1) * NL / (LOAD_STEPS * NM);
                        static_for<l1 - l0>([&](auto i) {
                            constexpr int l = l0 + decltype(i)::value;
                            if constexpr (l < WL) load_w(ic<l>{}, s + T::WPD);
                            else load_a(ic<l - WL>{}, ca, sta);
                        });
                    }
                    // weight pairs [t ND / NM, (t + 1) ND / NM) of the next k-step
#pragma unroll
                    for (int e = t * ND / NM; e < (t + 1) * ND / NM; e++) {
                        const Raw &r = raw[(j + 1) & 1];
                        if ((e & 1) == 0) x = bytes(ic<un>{}, ic<jn>{}, r, e >> 2, (e >> 1) & 1);
                        hq[e >> 2][e & 3] = deq2(x, r.s[e >> 2], e & 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                static_for<NM>(slice);
                // D = 2: this step's reads of A (issued after the raw ones)
                // stay in flight, except before a barrier that frees their
                // slot within a chunk.
                constexpr int OPEN = F::KIND == WK_F16 ? RB + CB : RB;
                if constexpr (D == 1 || (T::PREWAIT && j == JB - 1)) wait_lgkm<0>();
                else wait_lgkm<OPEN>();
#pragma unroll
                for (int i = 0; i < RB; i++) pin(a[jn][i]);
                if constexpr (F::KIND == WK_F16) {
#pragma unroll
                    for (int i = 0; i < CB; i++) pin(b[jn][i]);
                } else {
                    pin_raw(raw[j & 1]);
#pragma unroll
                    for (int cb = 0; cb < CB; cb++) b[jn & 1][cb] = join8(hq[cb][0], hq[cb][1], hq[cb][2], hq[cb][3]);
                }
            };
            static_for<4>(step);
            st = st1;
        };
        static_for<CPS>(chunk);
        ws = ws1;
    }
    wait_lgkm<0>();  // the reads past the end
#pragma unroll
    for (int i = 0; i < RB; i++) {
        pin(a[0][i]);
        pin(a[1][i]);
    }
    if constexpr (F::KIND == WK_F16) {
#pragma unroll
        for (int i = 0; i < CB; i++) {
            pin(b[0][i]);
            pin(b[1][i]);
        }
    }
    if constexpr (NCH > 1) {
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int j = 0; j < CB; j++) acc[0][i][j] += acc[1][i][j];
    }
    __builtin_amdgcn_s_waitcnt(0);  // the loads past the end

    // Element r of acc[rb][cb] in lane l is row 8 (r / 4) + 4 (l / 32) + r % 4,
    // column l % 32 of the 32 x 32 block.
    const int wrow = wm * 32 * RB;
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
        const int col = wn * 32 * CB + 32 * cb + l32;
        float *o = out + (m0 + (size_t)(wrow + 4 * h)) * N + n0 + col;
        if (col < cols) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int m = 32 * rb + 8 * (r >> 2) + (r & 3);
                    if (wrow + 4 * h + m < rows) o[(size_t)m * N] = acc[0][rb][cb][r];
                }
        }
    }
}

template <class F, int RB, int CB>
__global__ __launch_bounds__(WNT) void k_gemm_wide(DevWeight w, const _Float16 *__restrict__ A, size_t M,
                                                   float *__restrict__ out, int m_tiles, int n_tiles) {
    using T = WideTile<F, RB, CB>;
    extern __shared__ __align__(16) unsigned char lds[];
    int mt, nt;
    wide_tile(xcd_run(blockIdx.x, gridDim.x), m_tiles, n_tiles, mt, nt);
    wide_body<F, RB, CB>(w, A, M, out, (size_t)mt * T::BM, (size_t)nt * T::BN, lds);
}

// 256 x 256 tiles for the first `full` tiles (whole rounds over the CUs),
// the rest as two 128 x 256 tiles each: a last round that would leave half
// of the CUs idle runs on all of them.
template <class F>
__global__ __launch_bounds__(WNT) void k_gemm_wide_tail(DevWeight w, const _Float16 *__restrict__ A, size_t M,
                                                        float *__restrict__ out, int m_tiles, int n_tiles, int full) {
    extern __shared__ __align__(16) unsigned char lds[];
    int mt, nt;
    const int L = blockIdx.x;
    if (L < full) {
        wide_tile(xcd_run(L, full), m_tiles, n_tiles, mt, nt);
        wide_body<F, 4, 2>(w, A, M, out, (size_t)mt * 256, (size_t)nt * 256, lds);
    } else {
        const int h = xcd_run(L - full, gridDim.x - full);
        wide_tile(full + h / 2, m_tiles, n_tiles, mt, nt);
        const size_t m0 = (size_t)mt * 256 + 128 * (h & 1);
        if (m0 < M) wide_body<F, 2, 2>(w, A, M, out, m0, (size_t)nt * 256, lds);
    }
}

template <class F, int RB, int CB>
hipError_t wide_lds() {
    return ensure_lds_limit((const void *)k_gemm_wide<F, RB, CB>, WideTile<F, RB, CB>::LDS);
}
template <class F>
constexpr int TAIL_LDS = WideTile<F, 4, 2>::LDS > WideTile<F, 2, 2>::LDS ? WideTile<F, 4, 2>::LDS : WideTile<F, 2, 2>::LDS;
template <class F>
hipError_t wide_tail_lds() {
    return ensure_lds_limit((const void *)k_gemm_wide_tail<F>, TAIL_LDS<F>);
}

template <class F, int RB, int CB>
hipError_t launch_wide(const DevWeight &w, const _Float16 *a, size_t M, float *out, hipStream_t s) {
    using T = WideTile<F, RB, CB>;
    const size_t mt = (M + T::BM - 1) / T::BM, nt = (w.n_rows + T::BN - 1) / T::BN;
    hipError_t e = wide_lds<F, RB, CB>();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_gemm_wide<F, RB, CB>), dim3((unsigned)(mt * nt)), dim3(WNT), T::LDS, s, w, a, M, out, (int)mt,
                       (int)nt);
    return hipGetLastError();
}

template <class F>
hipError_t launch_wide_tail(const DevWeight &w, const _Float16 *a, size_t M, float *out, int cus, hipStream_t s) {
    const size_t mt = (M + 255) / 256, nt = (w.n_rows + 255) / 256, full = mt * nt / cus * cus;
    hipError_t e = wide_tail_lds<F>();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_gemm_wide_tail<F>), dim3((unsigned)(full + 2 * (mt * nt - full))), dim3(WNT), TAIL_LDS<F>, s, w, a, M,
                       out, (int)mt, (int)nt, (int)full);
    return hipGetLastError();
}

}  // namespace

namespace {

enum WideShape { WIDE_NONE, WIDE_256x256, WIDE_256x256_TAIL, WIDE_128x256, WIDE_256x128, WIDE_128x128 };

// Estimated time of `tiles` tiles on `cus` CUs, one tile per CU at a time:
// `full` a round on all CUs, `lo` one on at most half of them (a part-filled
// chip holds a higher clock).
double wide_rounds(size_t tiles, size_t cus, double full, double lo) {
    const size_t r = tiles / cus, m = tiles % cus, knee = cus / 2;
    return (double)r * full + (m == 0 ? 0.0 : m <= knee ? lo : lo + (full - lo) * (double)(m - knee) / (double)(cus - knee));
}

// Microseconds of one round of tiles at K 4096 on 256 CUs, {every CU busy, at
// most half of them}: 128 x 128, 128 x 256, 256 x 128 and 256 x 256 here, 128 x 64
// and (a full round) 96 x 128 in gemm_f16.hip.  Fitted to every shape of every format
// at M 128-2048, N 1024-14336.  Fifth bits cost a multiply per four weights in each
// of the waves that share a column, Q6_K's two bit planes less.
struct WideCost {
    double t128[2], t128x256[2], t256x128[2], t256[2], t128x64[2], t96x128;
};
const WideCost &wide_cost(uint32_t dtype) {
    static const WideCost plain = {{46.5, 38.0}, {79.0, 60.0}, {72.0, 52.0}, {126.0, 83.0}, {25.0, 19.0}, 34.5};
    static const WideCost fifth = {{52.0, 45.0}, {86.0, 72.0}, {73.5, 57.0}, {132.5, 96.0}, {25.0, 18.0}, 35.0};
    static const WideCost q6 = {{46.5, 40.5}, {81.0, 69.0}, {69.0, 49.5}, {126.0, 88.5}, {24.0, 18.0}, 0.0};
    return dtype == T_Q5_K || dtype == T_Q5_0 ? fifth : dtype == T_Q6_K ? q6 : plain;
}

// The estimated time of gemm_f16.hip's tiles.  Its last row tile runs a 64- or
// 96-row body where it holds no more rows; a round there has a fixed part
// (measured against the tiles here: +24 % at K 1024, -6 % at K 14336).
double small_tile_cost(const DevWeight &w, size_t M, size_t cus, const WideCost &c) {
    const size_t N = w.n_rows, n64 = (N + 63) / 64, t = (M + 127) / 128 * n64, rounds = (t + cus - 1) / cus, rem = M % 128;
    double v = wide_rounds(t, cus, c.t128x64[0], c.t128x64[1]);
    if (rounds > 1 && rem > 0 && rem <= 96 && n64 >= t - (rounds - 1) * cus) v -= (rem <= 64 ? 0.45 : 0.2) * c.t128x64[0];
    if (w.dtype != T_Q8_0 && w.dtype != T_Q6_K)
        v = std::min(v, c.t96x128 * (double)(((M + 95) / 96 * ((N + 127) / 128) + cus - 1) / cus));
    return v * (0.92 + 0.08 * 4096.0 / (double)w.n_cols);
}

// The tile shape for out[M, N], or WIDE_NONE where gemm_f16.hip's tiles are
// estimated faster.  Per 128 x 128 outputs a plain format's full round is 31 us in
// 256 x 256 tiles, 36 in 256 x 128, 40 in 128 x 256, 46 in 128 x 128 and 50 in 128 x 64, so
// the larger tiles win as soon as they fill the chip: M 1024 x N 4096 50 -> 47
// us on 128 x 128, M 2048 x N 4096 103 -> 75 on 256 x 128, M 4096 x N 14336
// 1070 -> 447 on 256 x 256 with the last half round as 128 x 256.  With one
// set of costs for all formats, Q5_K, Q5_0 and Q6_K came here where the small
// tiles are faster: Q5_K M 200 x N 14336 at K 14336 131 us there, 176 here.
// F16 weights always come here (K 2560, M 333, N 6912: 45 us in
// gemm_gen.hip, 20 here; M 16, N 2048: 21 / 15; M 16, K 14336, N 512, four
// blocks: 93 / 70; none of 506 shapes slower by more than 1.2 us).
WideShape wide_shape(const DevWeight &w, size_t M, size_t cus) {
    const size_t N = w.n_rows;
    auto tiles = [&](size_t bm, size_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    WideShape best = WIDE_NONE;
    double cost = 0.0;
    auto offer = [&](WideShape sh, double c) {
        if (best == WIDE_NONE ? (cost == 0.0 || c < cost) : c < cost) { best = sh; cost = c; }
    };
    if (w.dtype == T_F16) {
        offer(WIDE_128x128, wide_rounds(tiles(128, 128), cus, 22.0, 15.5));
        offer(WIDE_128x256, wide_rounds(tiles(128, 256), cus, 43.0, 25.0));
        offer(WIDE_256x128, wide_rounds(tiles(256, 128), cus, 43.5, 26.0));
        return best;
    }
    const WideCost &c = wide_cost(w.dtype);
    cost = small_tile_cost(w, M, cus, c);
    offer(WIDE_128x128, wide_rounds(tiles(128, 128), cus, c.t128[0], c.t128[1]));
    offer(WIDE_128x256, wide_rounds(tiles(128, 256), cus, c.t128x256[0], c.t128x256[1]));
    offer(WIDE_256x128, wide_rounds(tiles(256, 128), cus, c.t256x128[0], c.t256x128[1]));
    const size_t t = tiles(256, 256), rem = t % cus;
    offer(WIDE_256x256, wide_rounds(t, cus, c.t256[0], c.t256[1]));
    if (t > cus && rem && 2 * rem <= cus)
        offer(WIDE_256x256_TAIL, (double)(t / cus) * c.t256[0] + wide_rounds(2 * rem, cus, c.t128x256[0], c.t128x256[1]));
    return best;
}

bool wide_dtype(const DevWeight &w) {
    return gemm_supports(w.dtype, w.n_cols) || gemm_q8_supports(w.dtype, w.n_cols) ||
           (w.dtype == T_F16 && gemm_gen_supports(w.dtype, w.n_cols));
}

// Call f with the format tag of a weight type.
template <class Fn>
hipError_t wide_fmt(uint32_t dtype, Fn &&f) {
    switch (dtype) {
    case T_Q4_K: return f(WQ4K{});
    case T_Q5_K: return f(WQ5K{});
    case T_Q4_0: return f(WQ40{});
    case T_Q4_1: return f(WQ41{});
    case T_Q5_0: return f(WQ50{});
    case T_Q8_0: return f(WQ80{});
    case T_Q6_K: return f(WQ6K{});
    case T_F16: return f(WF16{});
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

// The kernel's load offsets are 32-bit within a tile's 256 rows of A and W.
bool gemm_wide_preferred(const DevWeight &w, size_t M) {
    const size_t lim = (size_t)1 << 32, cus = cu_count() ? (size_t)cu_count() : 256;
    if (M == 0 || w.n_rows == 0 || !wide_dtype(w)) return false;
    if (256 * w.n_cols * 2 >= lim || 256 * w.row_stride >= lim || 4 * w.group_stride >= lim) return false;
    if (w.n_rows >= (size_t)1 << 31 || M >= (size_t)1 << 31 || (M / 128 + 1) * (w.n_rows / 128 + 1) >= (size_t)1 << 30) return false;
    return wide_shape(w, M, cus) != WIDE_NONE;
}

hipError_t launch_gemm_wide(const DevWeight &w, const void *a_f16, size_t M, float *out, hipStream_t s) {
    if (!gemm_wide_preferred(w, M)) return hipErrorInvalidValue;
    const _Float16 *a = static_cast<const _Float16 *>(a_f16);
    const size_t cus = cu_count() ? (size_t)cu_count() : 256;
    const WideShape sh = wide_shape(w, M, cus);
    return wide_fmt(w.dtype, [&](auto fmt) {
        using F = decltype(fmt);
        if constexpr (F::KIND != WK_F16) {
            if (sh == WIDE_256x256) return launch_wide<F, 4, 2>(w, a, M, out, s);
            if (sh == WIDE_256x256_TAIL) return launch_wide_tail<F>(w, a, M, out, (int)cus, s);
        }
        if (sh == WIDE_128x256) return launch_wide<F, 2, 2>(w, a, M, out, s);
        if (sh == WIDE_256x128) return launch_wide<F, 4, 1>(w, a, M, out, s);
        return launch_wide<F, 2, 1>(w, a, M, out, s);
    });
}

hipError_t gemm_wide_prepare_lds() {
    for (uint32_t t : {T_Q4_K, T_Q5_K, T_Q4_0, T_Q4_1, T_Q5_0, T_Q8_0, T_Q6_K, T_F16}) {
        const hipError_t e = wide_fmt(t, [&](auto fmt) {
            using F = decltype(fmt);
            hipError_t r = wide_lds<F, 2, 2>();
            if (r == hipSuccess) r = wide_lds<F, 4, 1>();
            if (r == hipSuccess) r = wide_lds<F, 2, 1>();
            if constexpr (F::KIND != WK_F16) {
                if (r == hipSuccess) r = wide_lds<F, 4, 2>();
                if (r == hipSuccess) r = wide_tail_lds<F>();
            }
            return r;
        });
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace rce_qmm
