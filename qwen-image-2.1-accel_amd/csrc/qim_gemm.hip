// MXFP8 GEMM on CDNA4 scaled MFMA with fused epilogues.
//
//   Y[m, n] = sum_k (A[m, k] 2^(sa[m, k/32] - 127)) (B[n, k] 2^(sb[n, k/32] - 127))
//
// A: (Mp, K) E4M3 codes, B: (N, K) E4M3 codes (both K-contiguous), scales in
// the 128x4 swizzled layout.  fp32 accumulation in v_mfma_scale_f32_32x32x64_
// f8f6f4, which applies the E8M0 block scales inside the instruction.  Lane l
// of a 32x32x64 step holds row l%32 of A (column l%32 of B); with h = l/32 its
// bytes 0-15 are K [16h, 16h+16) and bytes 16-31 are K [32+16h, 32+16h+16), so
// bytes 0-15 of both half-waves form scale block 0 and bytes 16-31 block 1, and
// lane l supplies the E8M0 exponent of (row l%32, block h).  (Measured with
// qim_debug_mfma_probe: one-hot operands against per-lane exponents.)
//
// Workgroup tile 256 x 256, 4 waves in a 2 x 2 grid, each wave a 128 x 128
// block of 4 x 4 MFMA tiles (256 fp32 accumulators per lane, in AGPRs).
// K advances 64 bytes per stage through a 4-deep LDS ring (34 KiB per stage:
// A 256 x 64, B 256 x 64, and the 1 KiB A / B scale chunks of the stage's
// 128-K group).  Operands move global -> LDS with global_load_lds_dwordx4
// (no register staging): lane i of an instruction writes LDS bytes
// [16i, 16i+16) of a 1 KiB segment, so the bank swizzle is applied to the
// source address instead -- LDS holds logical 16-byte chunk c of tile row r at
// chunk c ^ (((r >> 1) ^ (r >> 2)) & 3), which makes 8 (and 16) lanes reading
// 8 (16) consecutive rows at one chunk hit distinct banks.  Stage s+4 is
// issued at the top of stage s, right after the barrier that proves every wave
// has consumed ring slot s % 4; the fragments of stage s+1 are read from LDS
// while the 16 MFMAs of stage s run.
#include <type_traits>

#include "qim_device.h"
#include "qim_runtime.h"

namespace qim {

typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void gbl_void_t;

constexpr int BM = 256, BN = 256, BK = 64, NSTAGE = 4;
constexpr int TILE_BYTES = BM * BK;                          // 16 KiB per operand per stage
constexpr int SCALE_BYTES = 1024;                            // two 512-byte chunks per operand
constexpr int STAGE_BYTES = 2 * TILE_BYTES + 2 * SCALE_BYTES;  // 34 KiB
constexpr int LDS_BYTES = NSTAGE * STAGE_BYTES;              // 136 KiB
// Loads per wave per stage: 4 A + 4 B (16 B each), plus 2 of 4 B for the
// scales in even stages only: a 128-K scale group spans two stages, and odd
// stages reuse the even stage's scales from registers.
constexpr int LOADS_EVEN = 10, LOADS_ODD = 8;

struct GemmArgs {
    const uint8_t *aq, *as, *bq, *bs;
    int64_t M, Mp, N, K;
    const uint16_t *bias, *gate, *res;
    int64_t seq;
    void *out;
    int64_t ldo;
    uint8_t *out_scales;
    int tiles_m, tiles_n;  // 256 x 256 tiles (tiles_n: whole 256-column blocks)
    int main_tiles;  // whole tiles; workgroups past them compute quarter tiles of the rest
    int quarters;    // quarter tiles of whole tiles; the ones after them cover a last
                     // 128-column block (N % 256 == 128), 128 rows each
    int a_tiled, b_tiled, out_tiled;  // code layouts (mxt_offset) of A, B and a quantized output
    // QIM_EPI_QK_NORM_ROPE: head weights, RoPE table (seq rows of 128 fp32),
    // and the column ends of Q (H * 128) and K (2 * H * 128).
    const uint16_t *wq, *wk;
    const float *freqs;
    float epsq, epsk;
    int64_t q_cols, qk_cols;
    // With vt set, the V columns leave as the attention's V^T tiles instead:
    // tile (batch, head, key block) of 128 rows (d) x 64 keys at
    // ((batch * H + head) * vt_nkb + key block) * 8192 elements, vt_nkb =
    // seq / 64 (seq % 64 == 0).
    uint16_t *vt;
    int64_t vt_nkb;
    // Split K (qim_mxfp8_gemm_ws): with ksplit > 1 each quarter tile is computed
    // by ksplit workgroups over disjoint ranges of K, which write their fp32
    // accumulators to ws; k_mx_gemm_sum then sums them in a fixed order and
    // runs the epilogue.
    float *ws;
    int ksplit;
    int qrows, qcols;  // a grid of quarter tiles only: its rows and columns (qrows 0 otherwise)
    int tile_rows;     // rows of a whole tile: 256, or 192 (k_mx_gemm_192; tiles_m counts those)
};

// qim_mxfp8_gemm_qk_norm_rope_vt: the QK-norm + RoPE epilogue whose V columns
// leave as V^T tiles (an instantiation of its own, so the plain QKV kernel
// carries none of it).  Its outputs are read next by the attention core, so
// it stores through the caches (block @1024^2 with attention: 881 -> 874 us)
// where every other epilogue streams its output past them.
constexpr int EPI_QKV_VT = 6;
template <int EPI>
constexpr bool is_qk_epi() { return EPI == QIM_EPI_QK_NORM_ROPE || EPI == EPI_QKV_VT; }
// QIM_EPI_NONE with an fp32 or fp16 output (QIM_GEMM_OUT_F32 / _F16): the
// reference's out_dtype of torch._scaled_mm.
constexpr int EPI_F32 = 7, EPI_F16 = 8;

template <typename V>
__device__ __forceinline__ void st_out(bool cached, void *ptr, const V &v) {
    if (cached)
        *reinterpret_cast<V *>(ptr) = v;
    else
        st_nt(ptr, v);
}

__device__ __forceinline__ int kswz(int row) { return mx_chunk_swizzle(row); }
// LDS byte offset of logical 16-byte chunk c of tile row `row` (64-byte rows).
__device__ __forceinline__ int lds_off(int row, int c) { return row * BK + ((c ^ kswz(row)) << 4); }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N < 64, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void block_barrier() { asm volatile("s_barrier" ::: "memory"); }

// Stage-0 source offset of this lane's 16 bytes in the DMA of the 16 tile
// rows [grp, grp + 16) of an (R, K) code matrix whose tile starts at row m0:
// lane i lands at row grp + i/4, physical LDS chunk i%4.  Row-major codes:
// the lane's logical chunk of its row.  Tiled codes (mxt_offset): the group is
// already the LDS image, 1 KiB contiguous.  Rows past R are clamped into the
// matrix; they only feed output rows that are never stored.
__device__ __forceinline__ uint32_t opnd_offset(int64_t m0, int grp, int lane, int64_t R, int64_t K, bool tiled) {
    if (!tiled) {
        const int row = grp + (lane >> 2);
        int64_t r = m0 + row;
        r = r < R ? r : R - 1;
        return (uint32_t)(r * K + (((lane & 3) ^ kswz(row)) << 4));
    }
    int64_t rg = m0 + grp;
    rg = rg <= R - 16 ? rg : R - 16;
    const int64_t r0 = rg & ~int64_t(255);
    return (uint32_t)(r0 * K + (rg - r0) * 64 + lane * 16);
}
// Advance of those offsets per 64-byte K stage (wave-uniform).
__device__ __forceinline__ uint32_t opnd_step(int64_t m0, int64_t R, bool tiled) {
    if (!tiled) return BK;
    const int64_t r0 = m0 & ~int64_t(255);
    return (uint32_t)((R - r0 < 256 ? R - r0 : 256) * 64);
}

// Per-lane source offsets of the 10 load instructions of a stage (stage 0);
// stage s adds s * astep / s * bstep (operands) or (s / 2) * 512 (scales).
struct LoadPlan {
    uint32_t a[4], b[4];      // byte offsets into aq / bq
    uint32_t sc[2];           // byte offsets into sc_base
    const uint8_t *sc_base[2];  // as (A scale quarter) or bs (B scale quarter); wave-uniform
    uint32_t astep, bstep;
    int wave;
};

__device__ __forceinline__ LoadPlan make_plan(const GemmArgs &p, int64_t m0, int64_t n0) {
    LoadPlan L;
    const int lane = threadIdx.x & 63;
    L.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int grp = (L.wave * 4 + j) * 16;
        L.a[j] = opnd_offset(m0, grp, lane, p.Mp, p.K, p.a_tiled);
        L.b[j] = opnd_offset(n0, grp, lane, p.N, p.K, p.b_tiled);
    }
    L.astep = opnd_step(m0, p.Mp, p.a_tiled);
    L.bstep = opnd_step(n0, p.N, p.b_tiled);
    const int64_t kt = p.K / 128;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int idx = L.wave * 2 + j;          // 0..3: A scale quarter, 4..7: B scale quarter
        const int off = (idx & 3) * 256 + lane * 4;
        const int g = off >> 9, o = off & 511;
        L.sc_base[j] = idx >= 4 ? p.bs : p.as;
        int64_t grow;
        if (idx < 4) {
            grow = m0 / 128 + g;
            grow = grow < p.Mp / 128 ? grow : p.Mp / 128 - 1;
        } else {
            grow = n0 / 128 + g;
        }
        L.sc[j] = (uint32_t)(grow * kt * 512 + o);
    }
    return L;
}

// LDS DMA through inline asm: the compiler does not see these as LDS writes,
// so it does not force vmcnt(0) before every LDS read (it cannot prove the
// ring slots disjoint); the ring's own vmcnt waits and s_barrier order them.
// M0 holds the wave-uniform LDS destination; lane i lands at M0 + 16i (4i for
// the dword form).  The destination is an "{m0}" operand, so the compiler
// writes M0 itself and knows its value at every statement; the s_nop covers
// the wait state between that write and the DMA's read of M0.
__device__ __forceinline__ void dma16(const uint8_t *base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base),
                 "{m0}"(lds_addr)
                 : "memory");
}
__device__ __forceinline__ void dma4(const uint8_t *base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base),
                 "{m0}"(lds_addr)
                 : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const uint8_t *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)p;
}

template <bool SCALES>
__device__ __forceinline__ void issue_stage(const GemmArgs &p, const LoadPlan &L, uint8_t *slot, int s) {
    const uint32_t ka = (uint32_t)s * L.astep, kb = (uint32_t)s * L.bstep;
    const uint32_t base = lds_addr(slot);
#pragma unroll
    for (int j = 0; j < 4; ++j) dma16(p.aq, L.a[j] + ka, base + (L.wave * 4 + j) * 1024);
#pragma unroll
    for (int j = 0; j < 4; ++j) dma16(p.bq, L.b[j] + kb, base + TILE_BYTES + (L.wave * 4 + j) * 1024);
    if constexpr (SCALES) {
        const uint32_t gofs = (uint32_t)(s >> 1) * 512;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            dma4(L.sc_base[j], L.sc[j] + gofs, base + 2 * TILE_BYTES + (L.wave * 2 + j) * 256);
    }
}

struct Frags {
    i32x8_t a[4], b[4];
    uint4 sa, sb;  // scale dwords of row tiles 0..3 (exponents of the 128-K group's 4 blocks)
};

// Fragment reads of one ring slot (stage), one operand tile at a time.
__device__ __forceinline__ i32x8_t read_tile(const uint8_t *base, int row, int kh) {
    const uint4 lo = *reinterpret_cast<const uint4 *>(base + lds_off(row, kh));
    const uint4 hi = *reinterpret_cast<const uint4 *>(base + lds_off(row, 2 + kh));
    return i32x8_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}
// The four scale dwords of a wave's row tiles t = 0..3 (local rows
// r = h*128 + t*32 + lr of a 1 KiB scale tile, whose dword for row r sits at
// (r/128)*512 + (r%32)*16 + ((r%128)/32)*4 = h*512 + lr*16 + t*4): contiguous,
// so one 16-byte read.
__device__ __forceinline__ uint4 read_scales(const uint8_t *base, int h, int lr) {
    return *reinterpret_cast<const uint4 *>(base + h * 512 + lr * 16);
}

__device__ __forceinline__ void read_frags(const uint8_t *slot, int wm, int wn, int lr, int kh, Frags &f) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        f.a[t] = read_tile(slot, wm * 128 + t * 32 + lr, kh);
        f.b[t] = read_tile(slot + TILE_BYTES, wn * 128 + t * 32 + lr, kh);
    }
    f.sa = read_scales(slot + 2 * TILE_BYTES, wm, lr);
    f.sb = read_scales(slot + 2 * TILE_BYTES + SCALE_BYTES, wn, lr);
}

// Every stage issues its loads unconditionally (past the end of K they
// re-read the last stage into a ring slot that is never read again), so at
// the top of stage s the outstanding loads are always those of stages s+1,
// s+2, s+3, and "stage s+1 landed" is always vmcnt(LOADS_EVEN + LOADS_ODD).  Keeping the stage
// free of branches keeps it one basic block, which the explicit schedule
// below needs.

#define QIM_SCHED() __builtin_amdgcn_sched_barrier(0)

// One pipeline step with an explicit instruction order (the scheduler may not
// move anything across QIM_SCHED()).  With one wave per SIMD the MFMA pipe
// idles whenever the wave stalls, so the 16 MFMAs of stage s (operands in
// `cur`) are spread around everything else the stage has to do:
//   MFMA 0 | wait for stage s+1's DMA and this wave's reads of stage s, barrier | MFMA 1-3, each followed by a
//   third of the 10 DMA issues of stage s+4 | MFMA 4-15, each followed by two
//   of the 24 LDS reads of stage s+1's operands into `nxt`.
// The scale dwords hold the exponents of K blocks 0..3 of the stage's 128-K
// group; the upper half-wave's are shifted down one byte so that byte
// (s % 2) * 2 is every lane's own block and op_sel can select it uniformly.
template <int PAR>
__device__ __forceinline__ void pipeline_step(const GemmArgs &p, const LoadPlan &L, uint8_t *lds, int s, int S,
                                              f32x16_t (&acc)[4][4], const Frags &cur, Frags &nxt, int wm,
                                              int wn, int lr, int kh) {
    int sa[4], sb[4];
    const uint32_t ca[4] = {cur.sa.x, cur.sa.y, cur.sa.z, cur.sa.w}, cb[4] = {cur.sb.x, cur.sb.y, cur.sb.z, cur.sb.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        sa[t] = (int)(ca[t] >> (8 * kh));
        sb[t] = (int)(cb[t] >> (8 * kh));
    }
#define QIM_MF(i, j)                                                                                          \
    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(cur.a[i], cur.b[j], acc[i][j], 0, 0, PAR * 2, \
                                                                sa[i], PAR * 2, sb[j])
    uint8_t *fill = lds + (s & 3) * STAGE_BYTES;
    const uint8_t *next = lds + ((s + 1) & 3) * STAGE_BYTES;  // stale at the last stage; unused then
    const int sl = s + 4 < S ? s + 4 : S - 1;                 // stage to load (clamped)
    const uint32_t ka = (uint32_t)sl * L.astep, kb = (uint32_t)sl * L.bstep, gofs = (uint32_t)(sl >> 1) * 512;
    const uint32_t fb = lds_addr(fill);
    const int ra0 = wm * 128 + lr, rb0 = wn * 128 + lr;

    const uint8_t *nsa = next + 2 * TILE_BYTES, *nsb = nsa + SCALE_BYTES;
    const uint8_t *scb0 = L.sc_base[0], *scb1 = L.sc_base[1];
    const uint32_t w4 = L.wave * 4;
#define QIM_STEP(mi, mj, work) QIM_MF(mi, mj); QIM_SCHED(); work; QIM_SCHED()
    QIM_MF(0, 0);
    QIM_SCHED();
    wait_vmcnt<LOADS_EVEN + LOADS_ODD>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    QIM_SCHED();
    QIM_STEP(0, 1, dma16(p.aq, L.a[0] + ka, fb + (w4 + 0) * 1024));
    // The next stage's scales: the same 128-K group after an even stage (kept
    // in registers), a new group after an odd one (one 16-byte read each).
    QIM_STEP(0, 2, dma16(p.aq, L.a[1] + ka, fb + (w4 + 1) * 1024);
             if constexpr (PAR == 0) nxt.sa = cur.sa; else nxt.sa = read_scales(nsa, wm, lr));
    QIM_STEP(0, 3, dma16(p.aq, L.a[2] + ka, fb + (w4 + 2) * 1024);
             if constexpr (PAR == 0) nxt.sb = cur.sb; else nxt.sb = read_scales(nsb, wn, lr));
    QIM_STEP(1, 0, dma16(p.aq, L.a[3] + ka, fb + (w4 + 3) * 1024); nxt.a[0] = read_tile(next, ra0, kh));
    QIM_STEP(1, 1, dma16(p.bq, L.b[0] + kb, fb + TILE_BYTES + (w4 + 0) * 1024);
             nxt.b[0] = read_tile(next + TILE_BYTES, rb0, kh));
    QIM_STEP(1, 2, dma16(p.bq, L.b[1] + kb, fb + TILE_BYTES + (w4 + 1) * 1024);
             nxt.b[1] = read_tile(next + TILE_BYTES, rb0 + 32, kh));
    QIM_STEP(1, 3, dma16(p.bq, L.b[2] + kb, fb + TILE_BYTES + (w4 + 2) * 1024);
             nxt.b[2] = read_tile(next + TILE_BYTES, rb0 + 64, kh));
    QIM_STEP(2, 0, dma16(p.bq, L.b[3] + kb, fb + TILE_BYTES + (w4 + 3) * 1024);
             nxt.b[3] = read_tile(next + TILE_BYTES, rb0 + 96, kh));
    // Logical stage s + 4 has this stage's parity: scales in even stages only.
    QIM_STEP(2, 1, if constexpr (PAR == 0) dma4(scb0, L.sc[0] + gofs, fb + 2 * TILE_BYTES + (L.wave * 2 + 0) * 256);
             nxt.a[1] = read_tile(next, ra0 + 32, kh));
    QIM_STEP(2, 2, if constexpr (PAR == 0) dma4(scb1, L.sc[1] + gofs, fb + 2 * TILE_BYTES + (L.wave * 2 + 1) * 256);
             nxt.a[2] = read_tile(next, ra0 + 64, kh));
    QIM_STEP(2, 3, nxt.a[3] = read_tile(next, ra0 + 96, kh));
    QIM_MF(3, 0);
    QIM_MF(3, 1);
    QIM_MF(3, 2);
    QIM_MF(3, 3);
    QIM_SCHED();
#undef QIM_STEP
#undef QIM_MF
}

// Tile id -> (tile row, tile column): groups of 4 tile-rows, column-major
// inside a group, so consecutive tiles share B columns and, within a group, A
// rows in L2.
__device__ __forceinline__ void tile_coords(const GemmArgs &p, int t, int &tm, int &tn) {
    constexpr int GM = 4;
    const int per_group = GM * p.tiles_n;
    const int group = t / per_group, first = group * GM;
    const int gm = p.tiles_m - first < GM ? p.tiles_m - first : GM;
    const int r = t - group * per_group;
    tm = first + r % gm;
    tn = r / gm;
}

// Workgroup -> tile.  Workgroups are dispatched round-robin over the 8 XCDs,
// so workgroup w runs on XCD w % 8; tile ids are remapped so that each XCD
// owns one contiguous range, walked in groups of 4 tile-rows (column-major
// inside a group) so the tiles resident on one XCD share A rows and B columns
// in that XCD's L2.
__device__ __forceinline__ void tile_of(const GemmArgs &p, int &tm, int &tn) {
    const int nt = p.main_tiles;
    int t = blockIdx.x;
    if ((nt & 7) == 0) t = (t & 7) * (nt >> 3) + (t >> 3);
    tile_coords(p, t, tm, tn);
}

// ------------------------------------------------------------ SiLU table --
// The SwiGLU epilogues look bf16(silu(g)) up instead of computing it (the
// estimate, its band test and the rounding cost ~14 vector instructions per
// output, on one wave per SIMD with nothing to hide them).  The table holds
// every bf16 g with biased exponent 101..132 (2^-26 <= |g| < 64): entry i of
// a sign is g = bits 0x3280 + i, positive at byte 2i, negative at 8192 + 2i,
// so for the packed bf16 pair G the two byte addresses come from
// P = G - 0x3280 (per half) as (P << 1) for bits 0..12 and (P >> 2) for the
// sign at bit 13; a value is in the table when bits 12..14 of P are clear.
// Entries are computed with silu_bf16 (bit-identical to the reference's
// rounding) by each workgroup while its first stages' loads are in flight;
// the rest (|g| < 2^-26, |g| >= 64, NaN) takes silu_bf16 itself.
constexpr int SILU_TAB_BYTES = 16384;
constexpr uint16_t SILU_TAB_BASE = 0x3280;
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

template <int EPI>
constexpr int ring_offset() { return (EPI == QIM_EPI_SWIGLU || EPI == QIM_EPI_SWIGLU_QUANT) ? SILU_TAB_BYTES : 0; }

__device__ __forceinline__ void fill_silu_table(uint8_t *tab) {
    // 256 threads x 16 dwords (two entries each), dword d = c * 256 + t.
#pragma unroll
    for (int c0 = 0; c0 < 16; c0 += 4) {
        float g[8], y[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t e = 2 * ((c0 + j / 2) * 256 + threadIdx.x) + (j & 1);  // entry 0..8191
            const uint32_t b = SILU_TAB_BASE + (e & 4095) + ((e >> 12) << 15);
            g[j] = __uint_as_float(b << 16);
        }
        silu_bf16_n<8>(g, y);
#pragma unroll
        for (int j = 0; j < 8; j += 2)
            *reinterpret_cast<uint32_t *>(tab + 4 * ((c0 + j / 2) * 256 + threadIdx.x)) = pack_bf16x2(y[j], y[j + 1]);
    }
}

// bf16(silu(g)) for the two bf16 values of gp (low half first), from the
// table, as bf16 bits; `bad` collects the bits that mark a value outside it.
__device__ __forceinline__ void silu_lookup2(const uint8_t *tab, uint32_t gp, uint32_t &y0, uint32_t &y1,
                                             uint32_t &bad) {
    const u16x2_t P = __builtin_bit_cast(u16x2_t, gp) - (u16x2_t){SILU_TAB_BASE, SILU_TAB_BASE};
    bad |= __builtin_bit_cast(uint32_t, P) & 0x70007000u;
    const uint32_t a = __builtin_bit_cast(uint32_t, (u16x2_t)(P << (u16x2_t){1, 1}));
    const uint32_t b = __builtin_bit_cast(uint32_t, (u16x2_t)(P >> (u16x2_t){2, 2}));
    uint32_t w;  // bits 0..12 of each half from a, bit 13 (and the zero bits above it) from b
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(w) : "s"(0x1fff1fffu), "v"(a), "v"(b));
    y0 = *reinterpret_cast<const uint16_t *>(tab + (w & 0xffffu));
    y1 = *reinterpret_cast<const uint16_t *>(tab + (w >> 16));
}

// ------------------------------------------------------------- epilogue --
// Two passes per 64 rows (two MFMA row tiles) of the wave's block, through a
// wave-private LDS region (the ring is free once the main loop has drained):
//  1. registers -> LDS: the per-element part of the epilogue (bias add, or
//     SwiGLU of the gate/up tile pair), then bf16.  Accumulators i = 4g'..4g'+3
//     of an MFMA tile are 4 consecutive rows of one column, so they are packed
//     two rows per dword (v_cvt_pk_bf16_f32) and stored with one 8-byte write:
//     the region holds, per group of 4 rows and per column, the column's 4
//     values (8 bytes).
//  2. LDS -> global: each lane reads the 4 x 8 block of 4 rows x 8 columns
//     (4 x 16 bytes), regroups it into the 4 rows' 16-byte vectors with byte
//     permutes, applies the per-row part (gated residual with coalesced
//     res/gate loads, or MXFP8 quantization of 32-column blocks = 4 lanes) and
//     stores each row vector (8 bytes for codes).
// Accumulator i of MFMA tile (ti, tj) is row 32ti + 8(i/4) + 4(l/32) + i%4,
// column 32tj + l%32 of the wave's block of TI x TJ MFMA tiles, whose first
// row is row0 and first GEMM column gcol0.  Within a row group, column c sits
// at 8c + 16(c/8) bytes: the pass-2 lanes of a 16-lane read group start 80
// bytes apart, on disjoint banks.
template <int W>
__device__ __forceinline__ int epi_col_offset(int c) { return c * 8 + (c >> 3) * 16; }

template <int EPI, int TI, int TJ>
__device__ __forceinline__ void epilogue(const GemmArgs &p, f32x16_t (&acc)[TI][TJ], uint8_t *lds,
                                         [[maybe_unused]] const uint8_t *tab, int64_t row0, int64_t gcol0, int lane,
                                         int wave) {
    if constexpr (EPI == EPI_F32 || EPI == EPI_F16) {
        // Straight from the accumulators: for each register, 32 lanes store
        // 32 consecutive columns of one row (128 or 64 contiguous bytes).
        const int lr = lane & 31, kh = lane >> 5;
#pragma unroll
        for (int ti = 0; ti < TI; ++ti)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int64_t row = row0 + 32 * ti + 8 * (i / 4) + 4 * kh + (i % 4);
                if (row >= p.M) continue;
#pragma unroll
                for (int tj = 0; tj < TJ; ++tj) {
                    const int64_t o = row * p.ldo + gcol0 + 32 * tj + lr;
                    if constexpr (EPI == EPI_F32)
                        __builtin_nontemporal_store(acc[ti][tj][i], reinterpret_cast<float *>(p.out) + o);
                    else
                        __builtin_nontemporal_store((_Float16)acc[ti][tj][i], reinterpret_cast<_Float16 *>(p.out) + o);
                }
            }
        return;
    } else {
    constexpr bool SWI = EPI == QIM_EPI_SWIGLU || EPI == QIM_EPI_SWIGLU_QUANT;
    constexpr int W = SWI ? 16 * TJ : 32 * TJ;  // output columns of this wave
    constexpr int RGS = W * 8 + (W / 8) * 16;   // bytes per group of 4 rows
    constexpr int LPR = W / 8;                  // lanes per row group in pass 2
    constexpr int GPI = 64 / LPR;               // row groups per pass-2 step
    const int lr = lane & 31, kh = lane >> 5;
    uint8_t *reg = lds + wave * (16 * RGS);
    const int64_t col0 = SWI ? gcol0 / 2 : gcol0;  // first output column
    // SwiGLU -> MXFP8 in a whole tile (TI = 4): the two waves of a 128-row
    // block (wave & 1 = 0, 1) together produce its 512-byte scale chunk (128
    // rows x the tile's 4 blocks of 32 output columns).  Their exponent bytes
    // are staged in LDS, after every wave's staging region, and the chunk
    // leaves as 32 whole 16-byte stores: byte stores straight to memory wrote
    // each 64-byte segment of the scales in many partial writes (+45 % of the
    // kernel's HBM writes at 4352 x 24576 x 3072).
    constexpr bool STAGE_SC = EPI == QIM_EPI_SWIGLU_QUANT && TI == 4;
    [[maybe_unused]] uint8_t *const sc_stage = lds + 4 * 16 * RGS + (wave >> 1) * 512;
    const int64_t F = p.N / 2;
    // QKV projection with vt: this wave's V columns are staged per column (64
    // keys, VT_COL bytes apart; the odd stride spreads the pass-1 writes of a
    // 32-lane group over all banks) and leave as V^T tiles.
    [[maybe_unused]] constexpr int VT_COL = 136;
    static_assert(W * VT_COL <= 16 * RGS, "V^T staging fits the wave's region");
    const bool vtw = EPI == EPI_QKV_VT && col0 >= p.qk_cols;
    float bias[TJ] = {};
    if constexpr (EPI == QIM_EPI_BIAS) {
#pragma unroll
        for (int tj = 0; tj < TJ; ++tj) bias[tj] = bf16_to_f32(p.bias[gcol0 + tj * 32 + lr]);
    }
#pragma unroll
    for (int half = 0; half < TI / 2; ++half) {
        // The residual rows of this half's pass 2, loaded before pass 1 so that
        // their latency overlaps it (rows past M: clamped, not stored).
        [[maybe_unused]] uint4 rpre[16 / GPI][4];
        // The gate vector of this half's rows when they are one batch's (a
        // per-row load in pass 2 would sit between stores: see pass 2).
        [[maybe_unused]] uint4 gpre = make_uint4(0, 0, 0, 0);
        [[maybe_unused]] bool gate_once = false;
        if constexpr (EPI == QIM_EPI_GATED_RESIDUAL) {
            const int cl = lane % LPR, gl = lane / LPR;
            // Row h0 + lr, clamped to M - 1: a uniform base row hc and
            // min(lr, M - 1 - hc) rows past it (32-bit per row).
            const int64_t h0 = row0 + half * 64, hc = h0 < p.M ? h0 : p.M - 1;
            const uint16_t *rb = p.res + hc * p.N;
            const uint32_t lmax = (uint32_t)(p.M - 1 - hc), rcol = (uint32_t)(col0 + cl * 8);
#pragma unroll
            for (int it = 0; it < 16 / GPI; ++it)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t lr = (uint32_t)(4 * (it * GPI + gl) + r);
                    rpre[it][r] = ld_nt(rb + ((lr < lmax ? lr : lmax) * (uint32_t)p.N + rcol));
                }
            const int64_t h1 = h0 + 63 < p.M ? h0 + 63 : p.M - 1;
            const uint32_t b0 = (uint32_t)hc / (uint32_t)p.seq;
            gate_once = b0 == (uint32_t)h1 / (uint32_t)p.seq;
            gpre = *reinterpret_cast<const uint4 *>(p.gate + (int64_t)b0 * p.N + col0 + cl * 8);
        }
        // pass 1
        if constexpr (SWI && TI == 2) {
            // Quarter tiles compute the SiLU (32 values per lane; filling the
            // table below would compute as many).
            static_assert(TJ == 2, "one gate / up tile pair");
#pragma unroll
            for (int tl = 0; tl < 2; ++tl) {
                float g[16], y[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) g[i] = acc[tl][0][i];
#pragma unroll
                for (int i = 0; i < 16; i += 2) rbf2(g[i], g[i + 1]);
                silu_bf16_n<16>(g, y);
#pragma unroll
                for (int i = 0; i < 16; ++i) y[i] *= rbf(acc[tl][1][i]);
#pragma unroll
                for (int ig = 0; ig < 4; ++ig)
                    *reinterpret_cast<uint2 *>(reg + (tl * 8 + ig * 2 + kh) * RGS + epi_col_offset<W>(lr)) =
                        make_uint2(pack_bf16x2(y[4 * ig], y[4 * ig + 1]), pack_bf16x2(y[4 * ig + 2], y[4 * ig + 3]));
            }
        } else if constexpr (SWI) {
            // bf16(bf16(silu(g)) * v) for the half's 8 row groups: g and v
            // rounded to bf16 in pairs, every table read of the half issued
            // before the first is used (their latency overlaps the rest), one
            // rarely taken branch for values outside the table (recomputed
            // from the accumulators), then the products; the store's bf16
            // packing is the final rounding.
            constexpr int NP = TJ;  // pairs per row group: TJ / 2 column pairs x 2 row pairs
            uint32_t up[2][4][NP], bad = 0;
            uint32_t y[2][4][2 * NP];  // bf16 bits
#pragma unroll
            for (int tl = 0; tl < 2; ++tl)
#pragma unroll
                for (int ig = 0; ig < 4; ++ig)
#pragma unroll
                    for (int u = 0; u < TJ / 2; ++u)
#pragma unroll
                        for (int e = 0; e < 4; e += 2) {
                            const int ti = half * 2 + tl, k = 2 * u + e / 2;
                            const uint32_t gp = pack_bf16x2(acc[ti][2 * u][4 * ig + e], acc[ti][2 * u][4 * ig + e + 1]);
                            up[tl][ig][k] =
                                pack_bf16x2(acc[ti][2 * u + 1][4 * ig + e], acc[ti][2 * u + 1][4 * ig + e + 1]);
                            silu_lookup2(tab, gp, y[tl][ig][2 * k], y[tl][ig][2 * k + 1], bad);
                        }
            // Keep the conversions below from being scheduled up against
            // their reads.
            __builtin_amdgcn_sched_barrier(0);
            if (__builtin_expect(bad != 0, 0)) {
#pragma unroll
                for (int tl = 0; tl < 2; ++tl)
#pragma unroll
                    for (int ig = 0; ig < 4; ++ig)
#pragma unroll
                        for (int u = 0; u < TJ / 2; ++u)
#pragma unroll
                            for (int e = 0; e < 4; e += 2) {
                                const int ti = half * 2 + tl, k = 2 * u + e / 2;
                                const uint32_t gp =
                                    pack_bf16x2(acc[ti][2 * u][4 * ig + e], acc[ti][2 * u][4 * ig + e + 1]);
#pragma unroll
                                for (int h = 0; h < 2; ++h) {
                                    const uint32_t gb = (gp >> (16 * h)) & 0xffffu;
                                    if (((gb - SILU_TAB_BASE) & 0x7000u) != 0)
                                        y[tl][ig][2 * k + h] = __float_as_uint(silu_bf16(__uint_as_float(gb << 16))) >> 16;
                                }
                            }
            }
#pragma unroll
            for (int tl = 0; tl < 2; ++tl)
#pragma unroll
                for (int ig = 0; ig < 4; ++ig) {
                    uint8_t *grp = reg + (tl * 8 + ig * 2 + kh) * RGS;  // rows 32tl + 8ig + 4kh + 0..3
                    float yy[2 * NP];
#pragma unroll
                    for (int i = 0; i < 2 * NP; ++i) yy[i] = __uint_as_float(y[tl][ig][i] << 16);
#pragma unroll
                    for (int u = 0; u < TJ / 2; ++u) {
                        const uint32_t v0 = up[tl][ig][2 * u], v1 = up[tl][ig][2 * u + 1];
                        *reinterpret_cast<uint2 *>(grp + epi_col_offset<W>(u * 32 + lr)) =
                            make_uint2(pack_bf16x2(yy[4 * u] * __uint_as_float(v0 << 16),
                                                   yy[4 * u + 1] * __uint_as_float(v0 & 0xffff0000u)),
                                       pack_bf16x2(yy[4 * u + 2] * __uint_as_float(v1 << 16),
                                                   yy[4 * u + 3] * __uint_as_float(v1 & 0xffff0000u)));
                    }
                }
        } else
#pragma unroll
        for (int tl = 0; tl < 2; ++tl) {
            const int ti = half * 2 + tl;
#pragma unroll
            for (int ig = 0; ig < 4; ++ig) {
                uint8_t *grp = reg + (tl * 8 + ig * 2 + kh) * RGS;  // rows 32tl + 8ig + 4kh + 0..3
                if (vtw) {
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj)
                        *reinterpret_cast<uint2 *>(reg + (tj * 32 + lr) * VT_COL + (32 * tl + 8 * ig + 4 * kh) * 2) =
                            make_uint2(pack_bf16x2(acc[ti][tj][4 * ig + 0], acc[ti][tj][4 * ig + 1]),
                                       pack_bf16x2(acc[ti][tj][4 * ig + 2], acc[ti][tj][4 * ig + 3]));
                } else {
#pragma unroll
                    for (int tj = 0; tj < TJ; ++tj) {
                        float y[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            y[e] = acc[ti][tj][4 * ig + e];
                            if constexpr (EPI == QIM_EPI_BIAS) y[e] = y[e] + bias[tj];
                        }
                        *reinterpret_cast<uint2 *>(grp + epi_col_offset<W>(tj * 32 + lr)) =
                            make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
                    }
                }
            }
        }
        // pass 2 (LDS operations of one wave complete in order: no wait needed)
        if (vtw) {
            // V^T tiles: this half's 64 rows are one key block (seq % 64 ==
            // 0).  Tile row d is 8 chunks of 16 bytes; physical chunk pc holds
            // logical chunk c = pc ^ ((d >> 1) & 7): keys 16(c/2) + 4(c%2) +
            // 0..3, then the same 8 keys later.  Eight lanes per row: each
            // store instruction writes 1 KiB contiguous.
            const int64_t R = row0 + half * 64;
            if (R < p.M) {
                const int64_t bt = R / p.seq, kb = (R - bt * p.seq) / 64, vc = col0 - p.qk_cols;
                uint16_t *tile = p.vt + ((bt * (p.q_cols / 128) + vc / 128) * p.vt_nkb + kb) * (64 * 128);
#pragma unroll
                for (int it = 0; it < W / 8; ++it) {
                    const int dl = it * 8 + (lane >> 3), pc = lane & 7, d = (int)(vc & 127) + dl;
                    const int c = pc ^ ((d >> 1) & 7), k0 = 16 * (c >> 1) + 4 * (c & 1);
                    const uint2 lo = *reinterpret_cast<const uint2 *>(reg + dl * VT_COL + k0 * 2);
                    const uint2 hi = *reinterpret_cast<const uint2 *>(reg + dl * VT_COL + (k0 + 8) * 2);
                    *reinterpret_cast<uint4 *>(tile + d * 64 + pc * 8) = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
            }
            continue;
        }
        // Pass 2.  Loads issued between one row group's stores and the next
        // group's use would make the compiler wait for those stores too (the
        // vector-memory counter drains in issue order and counts stores), and
        // a per-row "row < M" branch makes every wait after it assume the
        // fewest outstanding operations.  So: the per-half gate vector and the
        // head weights are loaded before the loop, the QK epilogue's RoPE
        // rows one row group ahead (before the current group's stores), and a
        // half whose 64 rows are all below M takes a version of the loop
        // without per-row checks (every half, when M % 64 == 0).
        const int cl = lane % LPR, gl = lane / LPR;
        const int64_t col = col0 + cl * 8;
        [[maybe_unused]] const bool isq = col0 < p.q_cols;
        [[maybe_unused]] const int hc = (int)(col0 & 127) + cl * 8;  // column within the head
        [[maybe_unused]] float wt[8];
        [[maybe_unused]] float4 fr[2][4][2];  // RoPE (cos, sin) of 4 rows: this group's and the next's
        [[maybe_unused]] const bool qk_cols = is_qk_epi<EPI>() && col0 < p.qk_cols;
        auto load_freqs = [&](int it, float4 (&f)[4][2]) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t tok = (uint32_t)(row0 + half * 64 + 4 * (it * GPI + gl) + r) % (uint32_t)p.seq;
                const float4 *fp = reinterpret_cast<const float4 *>(p.freqs + (int64_t)tok * 128 + hc);
                f[r][0] = fp[0];
                f[r][1] = fp[1];
            }
        };
        if constexpr (is_qk_epi<EPI>()) {
            if (qk_cols) {
                unpack8(*reinterpret_cast<const uint4 *>((isq ? p.wq : p.wk) + hc), wt);
                load_freqs(0, fr[0]);
            }
        }
        // MXFP8 output: the half's 64 rows lie in one 256-row group of the
        // tiled layout and one 128-row block of the scales, so each row's
        // code and scale offsets are a uniform base plus a per-lane 32-bit
        // offset plus a compile-time row term (times a uniform row step for
        // the codes): no 64-bit arithmetic per row.  Local row
        // lr = 4 (it GPI + gl) + r; with GPI % 4 == 0 its chunk swizzle
        // ((lr >> 1) ^ (lr >> 2)) & 3 is ((2 gl + r / 2) ^ gl) & 3.  Mp is a
        // multiple of 128, so a half is stored whole or not at all.
        // bf16 output rows: the same split, row h0 + lr at obase + ooff + lr * ldo.
        [[maybe_unused]] uint16_t *const obase = reinterpret_cast<uint16_t *>(p.out) + (row0 + half * 64) * p.ldo;
        [[maybe_unused]] const uint32_t ooff = (uint32_t)(col + 4 * gl * p.ldo);
        [[maybe_unused]] uint8_t *qbase = nullptr, *sbase = nullptr;
        [[maybe_unused]] uint32_t qoff[2] = {0, 0}, soff = 0, sst = 0, qstep = 0;
        [[maybe_unused]] bool qlive = false;
        if constexpr (EPI == QIM_EPI_SWIGLU_QUANT) {
            static_assert(GPI % 8 == 0, "row terms below assume whole groups of 8 row groups");
            const int64_t h0 = row0 + half * 64, kb = col >> 5;
            qlive = h0 < p.Mp;
            sbase = p.out_scales + (h0 >> 7) * (F >> 7) * 512 + ((h0 & 127) >> 5) * 4;
            soff = (uint32_t)((kb >> 2) * 512 + (kb & 3) + (gl & 7) * 64 + (gl >> 3) * 4);
            sst = (uint32_t)((kb & 3) + (gl & 7) * 64 + (gl >> 3) * 4 + ((h0 & 127) >> 5) * 4);
            if (p.out_tiled) {
                const int64_t r0 = h0 & ~int64_t(255);
                const int64_t n = p.Mp - r0 < 256 ? p.Mp - r0 : 256;
                qbase = reinterpret_cast<uint8_t *>(p.out) + r0 * F + (h0 - r0) * 64;
                qstep = 64;
                const uint32_t lo = (uint32_t)((col >> 6) * n * 64 + (col & 15) + gl * 4 * 64);
                const int ch = (int)(col >> 4) & 3;
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) qoff[hb] = lo + ((ch ^ (((2 * gl + hb) ^ gl) & 3)) << 4);
            } else {
                qbase = reinterpret_cast<uint8_t *>(p.out) + h0 * F;
                qstep = (uint32_t)F;
                qoff[0] = qoff[1] = (uint32_t)(col + gl * 4 * F);
            }
        }
        auto pass2 = [&](auto all_rows, auto one_gate) {
            constexpr bool ALL_ROWS = decltype(all_rows)::value, ONE_GATE = decltype(one_gate)::value;
#pragma unroll
        for (int it = 0; it < 16 / GPI; ++it) {
            const int g = it * GPI + gl;  // row group: rows 4g .. 4g+3 of this half
            const uint8_t *src = reg + g * RGS + epi_col_offset<W>(cl * 8);
            uint4 q[4];  // q[k]: columns 8cl + 2k, 2k+1; .x/.y rows 0-1/2-3 of the first, .z/.w of the second
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = *reinterpret_cast<const uint4 *>(src + k * 16);
            uint4 rowv[4];
            {
                uint32_t w[4][4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    w[0][k] = __builtin_amdgcn_perm(q[k].z, q[k].x, 0x05040100u);  // row 0: low halves
                    w[1][k] = __builtin_amdgcn_perm(q[k].z, q[k].x, 0x07060302u);  // row 1: high halves
                    w[2][k] = __builtin_amdgcn_perm(q[k].w, q[k].y, 0x05040100u);
                    w[3][k] = __builtin_amdgcn_perm(q[k].w, q[k].y, 0x07060302u);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) rowv[r] = make_uint4(w[r][0], w[r][1], w[r][2], w[r][3]);
            }
            if constexpr (is_qk_epi<EPI>()) {
                // Q and K head columns: RMSNorm + RoPE of each row's 128-wide
                // head, as k_norm_rope computes it on the stored output.  A
                // wave holds W columns of the head; with W = 64 (quarter tiles)
                // the other half is the partner wave's (wave ^ 1, same rows),
                // whose row sums come through LDS.  The Q/K/V class is uniform
                // over a quarter tile's four waves (one head), so its barriers
                // are too.  So it is over the four waves of a 192-row tile (two
                // heads): H is even, so both heads are of one class.
                if (qk_cols) {
                    float x[4][8];
                    double ss[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        unpack8(rowv[r], x[r]);
                        ss[r] = group_sum<LPR>(head_sumsq8(x[r]));
                    }
                    if constexpr (W < 128) {
                        static_assert(W == 64, "a head spans two waves at most");
                        double *xs = reinterpret_cast<double *>(lds + 4 * 16 * RGS) + (it & 1) * (4 * GPI * 4);
                        if (cl == 0) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) xs[(wave * GPI + gl) * 4 + r] = ss[r];
                        }
                        __syncthreads();
#pragma unroll
                        for (int r = 0; r < 4; ++r) ss[r] += xs[((wave ^ 1) * GPI + gl) * 4 + r];
                    }
                    const float eps = isq ? p.epsq : p.epsk;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        head_rmsnorm8(x[r], ss[r], 128, eps, wt);
                        head_rope8(x[r], fr[it & 1][r][0], fr[it & 1][r][1]);
                        rowv[r] = pack8(x[r]);
                    }
                    if (it + 1 < 16 / GPI) load_freqs(it + 1, fr[(it + 1) & 1]);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t grow = row0 + half * 64 + 4 * g + r;
                const uint4 v = rowv[r];
                if constexpr (EPI == QIM_EPI_SWIGLU_QUANT) {
                    int e;
                    const uint2 c = quantize8_bf16(v, e);
                    // Cached, not streaming: a store instruction covers half of
                    // each 128-byte line (rows 4 apart), and streamed half-line
                    // writes reached memory as 1.5x the code bytes (WRITE_SIZE
                    // 78207 vs 53952 KiB at 4352 x 24576 x 3072); through the
                    // cache the two halves merge.
                    *reinterpret_cast<uint2 *>(qbase + (qoff[r >> 1] + (uint32_t)(4 * it * GPI + r) * qstep)) = c;
                    if ((cl & 3) == 0) {
                        if constexpr (STAGE_SC)
                            sc_stage[sst + (uint32_t)(16 * r + it * (GPI / 8) * 4)] = (uint8_t)e;
                        else
                            sbase[soff + (uint32_t)(16 * r + it * (GPI / 8) * 4)] = (uint8_t)e;
                    }
                } else {
                    if (!ALL_ROWS && grow >= p.M) continue;
                    uint4 o = v;
                    if constexpr (EPI == QIM_EPI_GATED_RESIDUAL) {
                        const uint4 hv = rpre[it][r];
                        const uint4 gv = ONE_GATE ? gpre
                                                  : *reinterpret_cast<const uint4 *>(p.gate + (grow / p.seq) * p.N + col);
                        float y[8], h[8], gg[8], z[8];
                        unpack8(v, y);
                        unpack8(hv, h);
                        unpack8(gv, gg);
#pragma unroll
                        for (int t = 0; t < 8; ++t) z[t] = h[t] + rbf(gg[t] * y[t]);
                        o = pack8(z);
                    }
                    st_out(EPI == EPI_QKV_VT, obase + (ooff + (uint32_t)(4 * it * GPI + r) * (uint32_t)p.ldo), o);
                }
            }
        }
        };
        // Two versions only where pass 2 loads (gated residual, QK): the
        // epilogues without loads wait for nothing there, and a second copy of
        // their loop only lengthens live ranges across the main loop.
        const bool all_rows = row0 + half * 64 + 64 <= p.M;  // uniform
        if constexpr (EPI == QIM_EPI_GATED_RESIDUAL) {
            if (all_rows && gate_once)
                pass2(std::true_type{}, std::true_type{});
            else
                pass2(std::false_type{}, std::false_type{});
        } else if constexpr (is_qk_epi<EPI>()) {
            if (all_rows)
                pass2(std::true_type{}, std::false_type{});
            else
                pass2(std::false_type{}, std::false_type{});
        } else if constexpr (EPI == QIM_EPI_SWIGLU_QUANT) {
            if (qlive) pass2(std::false_type{}, std::false_type{});
        } else {
            pass2(std::false_type{}, std::false_type{});
        }
    }
    if constexpr (STAGE_SC) {
        // Both halves of both waves of each 128-row block staged (a block
        // below Mp is live in both halves: Mp % 128 == 0).
        __syncthreads();
        if ((wave & 1) == 0 && lane < 32 && row0 < p.Mp) {
            uint8_t *chunk = p.out_scales + ((row0 >> 7) * (F >> 7) + (col0 >> 7)) * 512;
            *reinterpret_cast<uint4 *>(chunk + lane * 16) = *reinterpret_cast<const uint4 *>(sc_stage + lane * 16);
        }
    }
    }
}

// --------------------------------------------------------- quarter tiles --
// Quarter tiles of 128 x 128: 4 waves in a 2 x 2 grid, each a 64 x 64 block of
// 2 x 2 MFMA tiles.  They compute
//  - the last r tiles (r <= CUs / 2) of a grid of whole tiles (4352 x 12288: 816
//    tiles = 3.19 rounds of 256), as 4r quarter tiles by as many extra
//    workgroups of k_mx_gemm, so the last round takes about a quarter of a
//    tile's time instead of a whole one;
//  - whole problems whose 256 x 256 tiles would leave most CUs idle
//    (k_mx_gemm_quarter, gemm_plan).
// A quarter tile reads twice a whole tile's operand bytes per MFMA from L2 and
// from LDS, and LDS bounds it: per 128 of K, 33 KiB of DMA writes and 64 KiB of
// fragment reads against 512 MFMA cycles (measured 0.36 us, ~800 cycles, with the
// operands in L2; 0.5 us with weights from HBM, where a CU draws 50-70 GB/s
// however much it has in flight).  So what counts is that its waits overlap: K
// advances in pairs of 64-byte stages (a pair is one 128-K scale group) with one
// barrier per pair, each half pair's fragments are read while the other half's
// MFMAs run, and the pairs go through a ring of NP slots of 33 KiB: NP = 4 where
// a workgroup has the CU to itself, 2 where two share it (the other's MFMAs then
// cover its waits).  (Fragments loaded straight into registers, the four waves
// splitting K and summing their accumulators through LDS at the end, ran the main
// loop at the MFMA rate from L2 but cost 5.5 us per tile for the exchange: 1280 x
// 3072 x 3072 19.8 against 16.4 us, x 12288 54.5 against 59 us.)
constexpr int QTILE_BYTES = 128 * BK;                             // 8 KiB per operand per stage
constexpr int QSCALE_BYTES = 512;                                 // per operand per pair
constexpr int QPAIR_BYTES = 4 * QTILE_BYTES + 2 * QSCALE_BYTES;   // A, B of both stages, A and B scales: 33 KiB
constexpr int QLOADS = 9;  // per wave per pair: 2 x (2 A + 2 B) of 16 B, 1 of 4 B (scales)
static_assert(4 * QPAIR_BYTES <= LDS_BYTES, "the 4-pair ring fits the whole tile's");

struct QPlan {
    uint32_t a[2], b[2];   // byte offsets into aq / bq (stage 0)
    uint32_t sc;           // byte offset of this wave's 256 scale bytes (stage 0)
    const uint8_t *sc_base;
    uint32_t astep, bstep;
    int wave;
};

__device__ __forceinline__ QPlan make_qplan(const GemmArgs &p, int64_t m0, int64_t n0) {
    QPlan Q;
    const int lane = threadIdx.x & 63;
    Q.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int grp = (Q.wave * 2 + j) * 16;
        Q.a[j] = opnd_offset(m0, grp, lane, p.Mp, p.K, p.a_tiled);
        Q.b[j] = opnd_offset(n0, grp, lane, p.N, p.K, p.b_tiled);
    }
    Q.astep = opnd_step(m0, p.Mp, p.a_tiled);
    Q.bstep = opnd_step(n0, p.N, p.b_tiled);
    // Waves 0, 1 load the A scale chunk of rows [m0, m0 + 128), waves 2, 3 the B chunk.
    const int64_t kt = p.K / 128;
    const int64_t grow = Q.wave < 2 ? m0 / 128 : n0 / 128;
    Q.sc_base = Q.wave < 2 ? p.as : p.bs;
    Q.sc = (uint32_t)(grow * kt * 512 + (Q.wave & 1) * 256 + lane * 4);
    return Q;
}

// LDS of a pair: stage h (0, 1) has A at h * 16 KiB and B 8 KiB after it; the
// scales follow both.
__device__ __forceinline__ void issue_qhalf(const GemmArgs &p, const QPlan &Q, uint8_t *slot, int s) {
    const uint32_t ka = (uint32_t)s * Q.astep, kb = (uint32_t)s * Q.bstep, w2 = Q.wave * 2;
    const uint32_t base = lds_addr(slot) + (s & 1) * 2 * QTILE_BYTES;
    dma16(p.aq, Q.a[0] + ka, base + (w2 + 0) * 1024);
    dma16(p.aq, Q.a[1] + ka, base + (w2 + 1) * 1024);
    dma16(p.bq, Q.b[0] + kb, base + QTILE_BYTES + (w2 + 0) * 1024);
    dma16(p.bq, Q.b[1] + kb, base + QTILE_BYTES + (w2 + 1) * 1024);
}
__device__ __forceinline__ void issue_qscales(const QPlan &Q, uint8_t *slot, int t) {
    dma4(Q.sc_base, Q.sc + (uint32_t)t * 512,
         lds_addr(slot) + 4 * QTILE_BYTES + (Q.wave < 2 ? 0 : QSCALE_BYTES) + (Q.wave & 1) * 256);
}
__device__ __forceinline__ void issue_qpair(const GemmArgs &p, const QPlan &Q, uint8_t *slot, int t) {
    issue_qhalf(p, Q, slot, 2 * t);
    issue_qscales(Q, slot, t);
    issue_qhalf(p, Q, slot, 2 * t + 1);
}

struct QFrags {
    i32x8_t a[2], b[2];
};

// The fragments of half h of a pair, in the order its MFMAs use them.
__device__ __forceinline__ void read_qfrags(const uint8_t *slot, int h, int wm, int wn, int lr, int kh, QFrags &f) {
    const uint8_t *A = slot + h * 2 * QTILE_BYTES + 0, *B = A + QTILE_BYTES;
    f.a[0] = read_tile(A, wm * 64 + lr, kh);
    f.b[0] = read_tile(B, wn * 64 + lr, kh);
    f.b[1] = read_tile(B, wn * 64 + 32 + lr, kh);
    f.a[1] = read_tile(A, wm * 64 + 32 + lr, kh);
}

// Scale dwords of row tiles 0, 1 of the wave's rows (x, y: A; z, w: B).  Rows
// h*64 + t*32 + lr (t = 0, 1) of a 128-row scale chunk: dwords at lr*16 + (2h +
// t)*4, contiguous.
__device__ __forceinline__ uint4 read_qscales(const uint8_t *slot, int wm, int wn, int lr) {
    const uint8_t *sc = slot + 4 * QTILE_BYTES;
    const uint2 a = *reinterpret_cast<const uint2 *>(sc + lr * 16 + wm * 8);
    const uint2 b = *reinterpret_cast<const uint2 *>(sc + QSCALE_BYTES + lr * 16 + wn * 8);
    return make_uint4(a.x, a.y, b.x, b.y);
}

// One pair of stages of a quarter tile.  On entry fa holds the even stage's
// fragments and sc the pair's scales.  First half: the even stage's MFMAs beside
// the reads of the odd stage.  Then every wave's reads of this slot are done
// (waited for here) and pair t + 1 has landed for every wave.  Second half: the
// odd stage's MFMAs beside the reads of pair t + 1 and the issue of pair t + NP
// into this slot.  REM = 0: inside the K range (pairs t + 1 .. t + NP - 1 are in
// flight); REM > 0: the REM-th pair from its end, with nothing left to issue and
// the REM - 1 later pairs in flight.
template <int NP, int REM>
__device__ __forceinline__ void qpair_step(const GemmArgs &p, const QPlan &Q, uint8_t *lds, int t, f32x16_t (&acc)[2][2],
                                           QFrags &fa, uint4 &sc, int wm, int wn, int lr, int kh) {
    uint8_t *const slot = lds + (t & (NP - 1)) * QPAIR_BYTES;
    const int sa[2] = {(int)(sc.x >> (8 * kh)), (int)(sc.y >> (8 * kh))};
    const int sb[2] = {(int)(sc.z >> (8 * kh)), (int)(sc.w >> (8 * kh))};
    QFrags fb;
#define QIM_QMF(f, h, i, j)                                                                                        \
    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.a[i], f.b[j], acc[i][j], 0, 0, (h) * 2, sa[i], \
                                                                (h) * 2, sb[j])
    QIM_QMF(fa, 0, 0, 0);
    QIM_SCHED();
    read_qfrags(slot, 1, wm, wn, lr, kh, fb);
    QIM_SCHED();
    QIM_QMF(fa, 0, 0, 1);
    QIM_QMF(fa, 0, 1, 0);
    QIM_QMF(fa, 0, 1, 1);
    QIM_SCHED();
    if constexpr (REM != 1) {
        wait_vmcnt<(REM ? REM - 2 : NP - 2) * QLOADS>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        QIM_SCHED();
    }
    QIM_QMF(fb, 1, 0, 0);
    QIM_SCHED();
    if constexpr (REM != 1) {
        const uint8_t *next = lds + ((t + 1) & (NP - 1)) * QPAIR_BYTES;
        sc = read_qscales(next, wm, wn, lr);
        read_qfrags(next, 0, wm, wn, lr, kh, fa);
        QIM_SCHED();
    }
    QIM_QMF(fb, 1, 0, 1);
    QIM_SCHED();
    if constexpr (REM == 0) issue_qhalf(p, Q, slot, 2 * (t + NP));
    QIM_SCHED();
    QIM_QMF(fb, 1, 1, 0);
    QIM_SCHED();
    if constexpr (REM == 0) {
        issue_qscales(Q, slot, t + NP);
        issue_qhalf(p, Q, slot, 2 * (t + NP) + 1);
    }
    QIM_SCHED();
    QIM_QMF(fb, 1, 1, 1);
    QIM_SCHED();
#undef QIM_QMF
}

// The last min(NP, K range) pairs.
template <int NP, int REM>
__device__ __forceinline__ void qtail(const GemmArgs &p, const QPlan &Q, uint8_t *lds, int te, int left,
                                      f32x16_t (&acc)[2][2], QFrags &fa, uint4 &sc, int wm, int wn, int lr, int kh) {
    if constexpr (REM > 0) {
        if (REM <= left) qpair_step<NP, REM>(p, Q, lds, te - REM, acc, fa, sc, wm, wn, lr, kh);
        qtail<NP, REM - 1>(p, Q, lds, te, left, acc, fa, sc, wm, wn, lr, kh);
    }
}

// fp32 words of one split-K partial: a quarter tile, row-major.
constexpr int QPART_WORDS = 128 * 128;

// Corner of quarter tile q (of the last whole tiles, or a 128-row piece of a
// last 128-column block).
__device__ __forceinline__ void quarter_origin(const GemmArgs &p, int q, int64_t &m0, int64_t &n0) {
    if (p.qrows) {             // a grid of quarter tiles: groups of 8 tile-rows, column-major inside a group
        const int per_group = 8 * p.qcols, group = q / per_group, first = group * 8;
        const int gm = p.qrows - first < 8 ? p.qrows - first : 8;
        const int r = q - group * per_group;
        m0 = (int64_t)(first + r % gm) * 128;
        n0 = (int64_t)(r / gm) * 128;
    } else if (q < p.quarters) {  // a quarter of one of the last whole tiles
        const int tile = p.main_tiles + q / 4, quarter = q & 3;
        int tm, tn;
        tile_coords(p, tile, tm, tn);
        m0 = (int64_t)tm * BM + (quarter >> 1) * 128;
        n0 = (int64_t)tn * BN + (quarter & 1) * 128;
    } else {               // 128 rows of the last 128-column block
        m0 = (int64_t)(q - p.quarters) * 128;
        n0 = (int64_t)p.tiles_n * BN;
    }
}

// Quarter-tile unit u: quarter tile u % quarters over the stage pairs
// [kp * P / ksplit, (kp + 1) * P / ksplit), kp = u / quarters, P = K / 128 (the
// whole of K when ksplit == 1).
template <int EPI, int NP>
__device__ __forceinline__ void quarter_tile(const GemmArgs &p, uint8_t *lds, int u) {
    const int split = p.ksplit > 1 ? p.ksplit : 1;
    const int q = split > 1 ? u % p.quarters : u, kp = split > 1 ? u / p.quarters : 0;
    int64_t m0, n0;
    quarter_origin(p, q, m0, n0);
    if (m0 >= p.Mp) return;  // padding rows only (whole workgroup)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1, lr = lane & 31, kh = lane >> 5;
    const int P = (int)(p.K / (2 * BK));
    const int tb = kp * P / split, te = (kp + 1) * P / split;
    f32x16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x16_t{};
    const QPlan Q = make_qplan(p, m0, n0);
    const int left = te - tb < NP ? te - tb : NP;  // pairs of the prologue (ksplit <= P: at least one)
#pragma unroll
    for (int i = 0; i < NP; ++i)
        if (i < left) issue_qpair(p, Q, lds + ((tb + i) & (NP - 1)) * QPAIR_BYTES, tb + i);
    // Pair tb landed: the left - 1 pairs after it may be in flight.
    if (left == NP)
        wait_vmcnt<(NP - 1) * QLOADS>();
    else
        wait_vmcnt<0>();
    block_barrier();
    QFrags fa;
    const uint8_t *first = lds + (tb & (NP - 1)) * QPAIR_BYTES;
    uint4 sc = read_qscales(first, wm, wn, lr);
    read_qfrags(first, 0, wm, wn, lr, kh, fa);
    for (int t = tb; t < te - NP; ++t) qpair_step<NP, 0>(p, Q, lds, t, acc, fa, sc, wm, wn, lr, kh);
    qtail<NP, NP>(p, Q, lds, te, left, acc, fa, sc, wm, wn, lr, kh);
    if (split > 1) {  // a partial sum: to the workspace, the epilogue runs in k_mx_gemm_sum
        float *w = p.ws + (int64_t)u * QPART_WORDS + (wm * 64 + 4 * kh) * 128 + wn * 64 + lr;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (m0 + wm * 64 + i * 32 >= p.M) break;  // rows nobody reads
#pragma unroll
            for (int r = 0; r < 16; ++r)
#pragma unroll
                for (int j = 0; j < 2; ++j) w[(32 * i + 8 * (r / 4) + r % 4) * 128 + 32 * j] = acc[i][j][r];
        }
        return;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    block_barrier();
    epilogue<EPI, 2, 2>(p, acc, lds, nullptr, m0 + wm * 64, n0 + wn * 64, lane, wave);
}

template <int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_mx_gemm(GemmArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    // The SwiGLU kernels keep their SiLU table in the first 16 KiB; the ring
    // (and the epilogue's staging) follows it.
    uint8_t *const tab = smem, *const lds = smem + ring_offset<EPI>();
    if ((int)blockIdx.x >= p.main_tiles) {  // a quarter tile of the last partial round
        quarter_tile<EPI, 4>(p, lds, (int)blockIdx.x - p.main_tiles);
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    int tm, tn;
    tile_of(p, tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int S = (int)(p.K / BK);
    const int lr = lane & 31, kh = lane >> 5;

    f32x16_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x16_t{};

    const LoadPlan L = make_plan(p, m0, n0);
    issue_stage<true>(p, L, lds, 0);
    issue_stage<false>(p, L, lds + STAGE_BYTES, 1 < S ? 1 : S - 1);
    issue_stage<true>(p, L, lds + 2 * STAGE_BYTES, 2 < S ? 2 : S - 1);
    issue_stage<false>(p, L, lds + 3 * STAGE_BYTES, 3 < S ? 3 : S - 1);
    if constexpr (ring_offset<EPI>() > 0) fill_silu_table(tab);
    wait_vmcnt<LOADS_ODD + LOADS_EVEN + LOADS_ODD>();  // stage 0 landed
    block_barrier();
    Frags fa, fb;
    read_frags(lds, wm, wn, lr, kh, fa);

    // S = K / 64 is even (K % 128 == 0): stages come in (even, odd) pairs.
    for (int s = 0; s < S; s += 2) {
        pipeline_step<0>(p, L, lds, s, S, acc, fa, fb, wm, wn, lr, kh);
        pipeline_step<1>(p, L, lds, s + 1, S, acc, fb, fa, wm, wn, lr, kh);
    }
    wait_vmcnt<0>();  // the clamped tail loads must land before LDS is reused
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    block_barrier();

    epilogue<EPI, 4, 4>(p, acc, lds, tab, m0 + wm * 128, n0 + wn * 128, lane, wave);
}

// A grid of quarter tiles only (gemm_plan): NP = 4 while the units are no more
// than the CUs; else NP = 2, two per CU.
constexpr int qlds_bytes(int np) { return np * QPAIR_BYTES; }

template <int EPI, int NP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_mx_gemm_quarter(GemmArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    // Contiguous ranges of units per XCD (workgroup ids go round-robin over 8).
    const int n = gridDim.x, xcd = blockIdx.x & 7, base = n >> 3, rem = n & 7;
    quarter_tile<EPI, NP>(p, smem, xcd * base + (xcd < rem ? xcd : rem) + (int)(blockIdx.x >> 3));
}

// ---------------------------------------------------------- 192-row tiles --
// Whole tiles of 192 x 256 for grids of 256 x 256 tiles that leave CUs idle in
// their one round while three quarters of a tile per CU would not (gemm_plan):
// 2381 x 4096 x 12288 has 160 whole tiles or 208 of these, 109.3 -> 102.1 us (2.35
// PFLOP/s: from there the power limit holds it, as it does the largest grids).  4 waves side by side, each
// a 192 x 64 block of 6 x 2 MFMA tiles (the epilogues work in 64-row halves of a
// wave, so the rows stay together).  A stage's 92 KiB of LDS traffic (28 KiB of
// DMA writes, 64 KiB of fragment reads) against 768 MFMA cycles is the most the
// LDS moves in that time.  The ring, its waits and the schedule are the whole
// tile's; a 192-row tile may start in the middle of a 128-row scale chunk or a
// 256-row super-block of the tiled layout, so each A load has its own K step and
// the six scale dwords come in three 8-byte reads.  (A fifth ring slot: the same
// times within 1 %.)
constexpr int TBM = 192, TA_BYTES = TBM * BK;
constexpr int TSTAGE_BYTES = TA_BYTES + TILE_BYTES + 2 * SCALE_BYTES;  // 30 KiB
constexpr int TLDS_BYTES = NSTAGE * TSTAGE_BYTES;                      // 120 KiB
constexpr int TLOADS_EVEN = 9, TLOADS_ODD = 7;  // per wave per stage: 3 A + 4 B (16 B), 2 of scales (4 B)

struct TPlan {
    uint32_t a[3], b[4], astep[3], bstep;
    uint32_t sc[2];
    const uint8_t *sc_base[2];
    uint32_t sa[3], sb;  // LDS offsets, in a stage, of this lane's scale dword pairs
    int wave;
};

__device__ __forceinline__ TPlan make_tplan(const GemmArgs &p, int64_t m0, int64_t n0) {
    TPlan L;
    const int lane = threadIdx.x & 63, lr = lane & 31;
    L.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int grp = (L.wave * 3 + j) * 16;
        const int64_t rg = m0 + grp <= p.Mp - 16 ? m0 + grp : p.Mp - 16;
        L.a[j] = opnd_offset(m0, grp, lane, p.Mp, p.K, p.a_tiled);
        L.astep[j] = opnd_step(rg, p.Mp, p.a_tiled);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) L.b[j] = opnd_offset(n0, (L.wave * 4 + j) * 16, lane, p.N, p.K, p.b_tiled);
    L.bstep = opnd_step(n0, p.N, p.b_tiled);
    const int64_t kt = p.K / 128;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int idx = L.wave * 2 + j;  // 0..3: A scale quarter, 4..7: B scale quarter
        const int off = (idx & 3) * 256 + lane * 4;
        int64_t grow = (idx < 4 ? m0 : n0) / 128 + (off >> 9);
        if (idx < 4 && grow >= p.Mp / 128) grow = p.Mp / 128 - 1;  // rows past Mp: never stored
        L.sc_base[j] = idx < 4 ? p.as : p.bs;
        L.sc[j] = (uint32_t)(grow * kt * 512 + (off & 511));
    }
    // Row tiles 2u, 2u + 1 are the 32-row groups pt, pt + 1 from the start of
    // m0's scale chunk; pt is even, so both dwords are in one aligned 8 bytes.
    const int first = (int)(m0 & 127) / 32;  // 0 or 2
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int pt = first + 2 * u;
        L.sa[u] = (uint32_t)(TA_BYTES + TILE_BYTES + (pt >> 2) * 512 + lr * 16 + (pt & 3) * 4);
    }
    L.sb = (uint32_t)(TA_BYTES + TILE_BYTES + SCALE_BYTES + (L.wave >> 1) * 512 + lr * 16 + (L.wave & 1) * 8);
    return L;
}

template <bool SCALES>
__device__ __forceinline__ void issue_tstage(const GemmArgs &p, const TPlan &L, uint8_t *slot, int s) {
    const uint32_t kb = (uint32_t)s * L.bstep, base = lds_addr(slot);
#pragma unroll
    for (int j = 0; j < 3; ++j) dma16(p.aq, L.a[j] + (uint32_t)s * L.astep[j], base + (L.wave * 3 + j) * 1024);
#pragma unroll
    for (int j = 0; j < 4; ++j) dma16(p.bq, L.b[j] + kb, base + TA_BYTES + (L.wave * 4 + j) * 1024);
    if constexpr (SCALES) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            dma4(L.sc_base[j], L.sc[j] + (uint32_t)(s >> 1) * 512,
                 base + TA_BYTES + TILE_BYTES + (L.wave * 2 + j) * 256);
    }
}

struct TFrags {
    i32x8_t a[6], b[2];
    uint2 sa[3], sb;
};

__device__ __forceinline__ void read_tscales(const uint8_t *slot, const TPlan &L, TFrags &f) {
#pragma unroll
    for (int u = 0; u < 3; ++u) f.sa[u] = *reinterpret_cast<const uint2 *>(slot + L.sa[u]);
    f.sb = *reinterpret_cast<const uint2 *>(slot + L.sb);
}

// One stage: as pipeline_step, 12 MFMAs with 7 or 9 DMA issues of stage s + 4 and
// the reads of stage s + 1 between them.  The wait before the barrier covers
// this wave's reads of the slot that stage s + 4 overwrites.
template <int PAR>
__device__ __forceinline__ void tstep(const GemmArgs &p, const TPlan &L, uint8_t *lds, int s, int S,
                                      f32x16_t (&acc)[6][2], const TFrags &cur, TFrags &nxt, int lr, int kh) {
    int sa[6], sb[2];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        sa[2 * u] = (int)(cur.sa[u].x >> (8 * kh));
        sa[2 * u + 1] = (int)(cur.sa[u].y >> (8 * kh));
    }
    sb[0] = (int)(cur.sb.x >> (8 * kh));
    sb[1] = (int)(cur.sb.y >> (8 * kh));
    const uint8_t *next = lds + ((s + 1) & 3) * TSTAGE_BYTES;  // stale at the last stage; unused then
    const uint8_t *nextb = next + TA_BYTES;
    const int sl = s + 4 < S ? s + 4 : S - 1;  // stage to load (clamped)
    const uint32_t kb = (uint32_t)sl * L.bstep, gofs = (uint32_t)(sl >> 1) * 512;
    const uint32_t fb = lds_addr(lds + (s & 3) * TSTAGE_BYTES), fbb = fb + TA_BYTES, fbs = fbb + TILE_BYTES;
    const uint32_t w3 = L.wave * 3, w4 = L.wave * 4;
    const int rb = L.wave * 64 + lr;
#define QIM_TMF(i, j)                                                                                         \
    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(cur.a[i], cur.b[j], acc[i][j], 0, 0, PAR * 2, \
                                                                sa[i], PAR * 2, sb[j])
#define QIM_TSTEP(mi, mj, work) QIM_TMF(mi, mj); QIM_SCHED(); work; QIM_SCHED()
    QIM_TMF(0, 0);
    QIM_SCHED();
    wait_vmcnt<TLOADS_EVEN + TLOADS_ODD>();  // stage s + 1 landed
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    QIM_SCHED();
    QIM_TSTEP(0, 1, dma16(p.aq, L.a[0] + (uint32_t)sl * L.astep[0], fb + (w3 + 0) * 1024);
              nxt.a[0] = read_tile(next, lr, kh));
    QIM_TSTEP(1, 0, dma16(p.aq, L.a[1] + (uint32_t)sl * L.astep[1], fb + (w3 + 1) * 1024);
              nxt.b[0] = read_tile(nextb, rb, kh));
    QIM_TSTEP(1, 1, dma16(p.aq, L.a[2] + (uint32_t)sl * L.astep[2], fb + (w3 + 2) * 1024);
              nxt.b[1] = read_tile(nextb, rb + 32, kh));
    QIM_TSTEP(2, 0, dma16(p.bq, L.b[0] + kb, fbb + (w4 + 0) * 1024);
              if constexpr (PAR == 0) {
                  nxt.sa[0] = cur.sa[0]; nxt.sa[1] = cur.sa[1]; nxt.sa[2] = cur.sa[2]; nxt.sb = cur.sb;
              } else read_tscales(next, L, nxt));
    QIM_TSTEP(2, 1, dma16(p.bq, L.b[1] + kb, fbb + (w4 + 1) * 1024); nxt.a[1] = read_tile(next, 32 + lr, kh));
    QIM_TSTEP(3, 0, dma16(p.bq, L.b[2] + kb, fbb + (w4 + 2) * 1024); nxt.a[2] = read_tile(next, 64 + lr, kh));
    QIM_TSTEP(3, 1, dma16(p.bq, L.b[3] + kb, fbb + (w4 + 3) * 1024); nxt.a[3] = read_tile(next, 96 + lr, kh));
    QIM_TSTEP(4, 0, if constexpr (PAR == 0) dma4(L.sc_base[0], L.sc[0] + gofs, fbs + (L.wave * 2 + 0) * 256);
              nxt.a[4] = read_tile(next, 128 + lr, kh));
    QIM_TSTEP(4, 1, if constexpr (PAR == 0) dma4(L.sc_base[1], L.sc[1] + gofs, fbs + (L.wave * 2 + 1) * 256);
              nxt.a[5] = read_tile(next, 160 + lr, kh));
    QIM_TMF(5, 0);
    QIM_TMF(5, 1);
    QIM_SCHED();
#undef QIM_TSTEP
#undef QIM_TMF
}

template <int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_mx_gemm_192(GemmArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    // Contiguous ranges of tiles per XCD, as in k_mx_gemm_quarter.
    const int n = gridDim.x, xcd = blockIdx.x & 7, base = n >> 3, rem = n & 7;
    int tm, tn;
    tile_coords(p, xcd * base + (xcd < rem ? xcd : rem) + (int)(blockIdx.x >> 3), tm, tn);
    const int64_t m0 = (int64_t)tm * TBM, n0 = (int64_t)tn * BN;
    const int lane = threadIdx.x & 63, lr = lane & 31, kh = lane >> 5;
    const int S = (int)(p.K / BK);
    f32x16_t acc[6][2];
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x16_t{};
    const TPlan L = make_tplan(p, m0, n0);
    uint8_t *const lds = smem;
    issue_tstage<true>(p, L, lds, 0);
    issue_tstage<false>(p, L, lds + TSTAGE_BYTES, 1);  // S is even
    issue_tstage<true>(p, L, lds + 2 * TSTAGE_BYTES, 2 < S ? 2 : S - 1);
    issue_tstage<false>(p, L, lds + 3 * TSTAGE_BYTES, 3 < S ? 3 : S - 1);
    wait_vmcnt<TLOADS_ODD + TLOADS_EVEN + TLOADS_ODD>();  // stage 0 landed
    block_barrier();
    TFrags fa, fb;
#pragma unroll
    for (int t = 0; t < 6; ++t) fa.a[t] = read_tile(lds, t * 32 + lr, kh);
#pragma unroll
    for (int t = 0; t < 2; ++t) fa.b[t] = read_tile(lds + TA_BYTES, L.wave * 64 + t * 32 + lr, kh);
    read_tscales(lds, L, fa);
    for (int s = 0; s < S; s += 2) {
        tstep<0>(p, L, lds, s, S, acc, fa, fb, lr, kh);
        tstep<1>(p, L, lds, s + 1, S, acc, fb, fa, lr, kh);
    }
    wait_vmcnt<0>();  // the clamped tail loads must land before LDS is reused
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    block_barrier();
    epilogue<EPI, 6, 2>(p, acc, lds, nullptr, m0, n0 + L.wave * 64, lane, L.wave);
}

// The split-K second launch: sums each quarter tile's ksplit partials in order
// kp = 0, 1, ... and runs the plain, bias or gated-residual epilogue.  One
// lane per 8 columns of a row (16 lanes per row of a quarter, 16 rows per
// workgroup), so that a few rows still spread over many waves; a lane's loads of
// four partials are in flight together.
// (The bias may start at any element: a slice of a larger buffer.)
typedef uint32_t u32x4_any_t __attribute__((ext_vector_type(4), aligned(2)));

template <int EPI>
__global__ __launch_bounds__(256) void k_mx_gemm_sum(GemmArgs p) {
    static_assert(ring_offset<EPI>() == 0, "the split runs the plain, bias and gated-residual epilogues");
    const int q = (int)blockIdx.x, r = (int)blockIdx.y * 16 + (threadIdx.x >> 4), c = (threadIdx.x & 15) * 8;
    int64_t m0, n0;
    quarter_origin(p, q, m0, n0);
    const int64_t row = m0 + r, col = n0 + c;
    if (row >= p.M) return;
    [[maybe_unused]] uint4 hv, gv;
    if constexpr (EPI == QIM_EPI_GATED_RESIDUAL) {
        hv = ld_nt(p.res + row * p.N + col);
        gv = *reinterpret_cast<const uint4 *>(p.gate + ((uint32_t)row / (uint32_t)p.seq) * p.N + col);
    } else if constexpr (EPI == QIM_EPI_BIAS) {
        const u32x4_any_t b = *reinterpret_cast<const u32x4_any_t *>(p.bias + col);
        gv = make_uint4(b.x, b.y, b.z, b.w);
    }
    const float4 *w = reinterpret_cast<const float4 *>(p.ws + (int64_t)q * QPART_WORDS + r * 128 + c);
    const int64_t step = (int64_t)p.quarters * (QPART_WORDS / 4);
    float y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int kp = 0; kp < p.ksplit; kp += 4) {
        float4 a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (kp + i < p.ksplit) {
                a[i] = w[(kp + i) * step];
                b[i] = w[(kp + i) * step + 1];
            } else {
                a[i] = b[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            y[0] += a[i].x; y[1] += a[i].y; y[2] += a[i].z; y[3] += a[i].w;
            y[4] += b[i].x; y[5] += b[i].y; y[6] += b[i].z; y[7] += b[i].w;
        }
    }
    const int64_t o = row * p.ldo + col;
    if constexpr (EPI == EPI_F32) {
        float *out = reinterpret_cast<float *>(p.out) + o;
#pragma unroll
        for (int t = 0; t < 8; ++t) out[t] = y[t];
    } else if constexpr (EPI == EPI_F16) {
        _Float16 *out = reinterpret_cast<_Float16 *>(p.out) + o;
#pragma unroll
        for (int t = 0; t < 8; ++t) out[t] = (_Float16)y[t];
    } else {
        if constexpr (EPI == QIM_EPI_BIAS) {
            float bv[8];
            unpack8(gv, bv);
#pragma unroll
            for (int t = 0; t < 8; ++t) y[t] += bv[t];
        } else if constexpr (EPI == QIM_EPI_GATED_RESIDUAL) {
            float h[8], g[8];
            unpack8(hv, h);
            unpack8(gv, g);
#pragma unroll
            for (int t = 0; t < 8; ++t) y[t] = h[t] + rbf(g[t] * rbf(y[t]));
        }
        st_nt(reinterpret_cast<uint16_t *>(p.out) + o, pack8(y));
    }
}

// CUs the work split plans for: the current device's, or MI355X's 256 when no
// device answers (sizes queried without a GPU).
static int64_t plan_cus() {
    const int c = device_cus();
    return c > 0 ? c : 256;
}

// Whole tiles to launch: all of them, or all but the last r when the last
// round of the CUs would hold r <= CUs / 2 tiles (those become 4r quarters).
static int64_t main_tile_count(int64_t tiles) {
    const int64_t cus = plan_cus();
    if (tiles <= cus) return tiles;
    const int64_t r = tiles % cus;
    return (r > 0 && 2 * r <= cus) ? tiles - r : tiles;
}

template <int EPI, int NP>
static int launch_quarters(const GemmArgs &a, int64_t units, hipStream_t st) {
    static std::atomic<bool> configured[QIM_MAX_DEVICES] = {};
    if (const int rc = reserve_lds(reinterpret_cast<const void *>(&k_mx_gemm_quarter<EPI, NP>), qlds_bytes(NP), configured,
                                   "qim_mxfp8_gemm"))
        return rc;
    launch(k_mx_gemm_quarter<EPI, NP>, dim3((unsigned)units), dim3(256), qlds_bytes(NP), st, a);
    return QIM_OK;
}

template <int EPI>
static int launch_gemm(const GemmArgs &a, hipStream_t st) {
    static std::atomic<bool> configured[QIM_MAX_DEVICES] = {};
    const int64_t split = a.ksplit > 1 ? a.ksplit : 1;
    if (a.qrows) {
        const int64_t units = a.quarters * split;
        if (const int rc = units <= plan_cus() ? launch_quarters<EPI, 4>(a, units, st) : launch_quarters<EPI, 2>(a, units, st))
            return rc;
    } else if (a.tile_rows == TBM) {
        if constexpr (ring_offset<EPI>() == 0) {
            static std::atomic<bool> configured192[QIM_MAX_DEVICES] = {};
            if (const int rc = reserve_lds(reinterpret_cast<const void *>(&k_mx_gemm_192<EPI>), TLDS_BYTES, configured192,
                                           "qim_mxfp8_gemm"))
                return rc;
            launch(k_mx_gemm_192<EPI>, dim3((unsigned)a.main_tiles), dim3(256), TLDS_BYTES, st, a);
        }
    } else {
        constexpr int lds_bytes = LDS_BYTES + ring_offset<EPI>();
        if (const int rc = reserve_lds(reinterpret_cast<const void *>(&k_mx_gemm<EPI>), lds_bytes, configured,
                                       "qim_mxfp8_gemm"))
            return rc;
        const int64_t half_column = a.tiles_n * BN < a.N ? (a.Mp + 127) / 128 : 0;
        const int64_t grid = a.main_tiles + a.quarters * split + half_column;
        launch(k_mx_gemm<EPI>, dim3((unsigned)grid), dim3(256), lds_bytes, st, a);
    }
    if constexpr (ring_offset<EPI>() == 0 && !is_qk_epi<EPI>()) {
        if (split > 1) launch(k_mx_gemm_sum<EPI>, dim3((unsigned)a.quarters, 8), dim3(256), 0, st, a);
    }
    return QIM_OK;
}

static bool splits_k(int epilogue) {
    return epilogue == QIM_EPI_NONE || epilogue == QIM_EPI_BIAS || epilogue == QIM_EPI_GATED_RESIDUAL;
}

// How one problem runs: main_tiles whole tiles, then the quarter tiles of the
// other whole tiles (times ksplit) and those of a last 128-column block; or,
// with qrows set, quarters = qrows x qcols quarter tiles only (times ksplit); or,
// with tile_rows 192, main_tiles tiles of 192 x 256 only.
struct GemmPlan {
    int64_t main_tiles, quarters, qrows, qcols;
    int ksplit;
    int tile_rows = BM;
    int64_t ws_bytes() const { return ksplit > 1 ? quarters * ksplit * (int64_t)QPART_WORDS * 4 : 0; }
};

// K-splits of a grid of quarter tiles, from a cost model in microseconds fitted
// to sweeps over M 40..512 (weights cold, each time best of the splits within 10 %):
// 0.5 per stage pair (a CU draws ~66 GB/s of operands while few CUs run), 5
// for the summing launch, and the partials' traffic (32-row groups below M,
// written and read) at 5 TB/s.  40 x 3072 x 12288: 48.7 us unsplit, 15.5 us in 8;
// 512 x 4096 x 4096: 17.6 us unsplit, 19.9 us in 2 (kept unsplit).
static int quarter_ksplit(int64_t quarters, int64_t M, int64_t N, int64_t pairs) {
    const double partial = (double)((M + 31) / 32 * 32) * (double)N * 8.0 / 5e6;
    double best = 0.5 * (double)pairs;
    int64_t ksplit = 1;
    for (int64_t k = 2; k <= 8 && k <= pairs && k * quarters <= plan_cus(); ++k) {
        const double cost = 0.5 * (double)((pairs + k - 1) / k) + 5.0 + (double)k * partial;
        if (cost < best) {
            best = cost;
            ksplit = k;
        }
    }
    return (int)ksplit;
}

static GemmPlan gemm_plan(int64_t M, int64_t N, int64_t K, int epilogue) {
    const int64_t cus = plan_cus(), pairs = K / (2 * BK);
    const int64_t Mp = (M + 127) / 128 * 128, tiles_n = N / BN, tiles = (Mp + BM - 1) / BM * tiles_n;
    const int64_t qrows = Mp / 128, qcols = N / 128;
    // Quarter tiles only, when all of them fit the chip at once, two per CU: at
    // most half as many whole tiles as CUs would run.  1280 x 3072 x 3072 (60 whole
    // tiles) 28.3 -> 15.0 us, x 12288 104.7 -> 59 us; 2048 x 4096 x 4096 (128)
    // 38.5 -> 32.6 us; 1024 x 9216 x 3072 (144) 32.6 -> 35.9 us (kept whole).
    if (qrows * qcols <= 2 * cus) {
        const int64_t q = qrows * qcols;
        return GemmPlan{0, q, qrows, qcols, splits_k(epilogue) ? quarter_ksplit(q, M, N, pairs) : 1};
    }
    // One partial round of whole tiles: tiles of 192 x 256 instead, when those fit
    // one round too (a 192-row tile runs at the whole tile's rate and takes
    // three quarters of its work).  256- against 192-row tiles, operands rotated:
    // 1280 x 9216 x 3072 (180 / 252 tiles) 35.5 -> 32.9 us, 2381 x 4096 x 12288 (160 /
    // 208) 109.3 -> 102.1, 3072 x 4096 x 4096 (192 / 256) 44.2 -> 40.7, x 12288 117.7 ->
    // 113.2, 2816 x 3072 x 3072 (132 / 180) 29.3 -> 26.4 us.  Above 256 of them a second
    // round costs more than the whole tiles' one.  The SwiGLU epilogues keep whole
    // tiles: their scale staging and SiLU table are laid out for 128 x 128 waves.
    const int64_t tiles192 = (Mp + TBM - 1) / TBM * tiles_n;
    if (tiles < cus && tiles192 <= cus && tiles_n * BN == N && epilogue != QIM_EPI_SWIGLU &&
        epilogue != QIM_EPI_SWIGLU_QUANT)
        return GemmPlan{tiles192, 0, 0, 0, 1, TBM};
    const int64_t main = main_tile_count(tiles);
    GemmPlan pl{main, 4 * (tiles - main), 0, 0, 1};
    // K-splits of the tail's quarter tiles: as many as fill the CUs' one round
    // (quarters * ksplit <= CUs), at most one stage pair each and at most 8; 1
    // (no split) when the quarters alone hold more than half the CUs, when a last
    // 128-column block is there, or for an epilogue other than the plain, bias
    // and gated-residual ones.  Unlike quarter_ksplit this asks for no gain, and
    // below about K 4096 there is none: unsplit / split (bias), 4352 x 4096: K 1024
    // 24.2 / 28.3 us, 3072 49.6 / 50.4, 4096 62.7 / 61.9, 12288 164.7 / 153.5; 4608 x 4096
    // (128 quarters in 2): K 4096 63.5 / 67.0, 12288 166.6 / 165.7; 16640 x 3072 (48
    // in 5): K 3072 120.8 / 121.7, 12288 414.8 / 408.2 us.
    if (pl.quarters > 0 && tiles_n * BN == N && splits_k(epilogue)) {
        int64_t k = cus / pl.quarters;
        k = k < pairs ? k : pairs;
        pl.ksplit = (int)(k > 8 ? 8 : k >= 2 ? k : 1);
    }
    return pl;
}

}  // namespace qim

using namespace qim;

// Operands of the QK-norm-RoPE epilogue (qim_mxfp8_gemm_qk_norm_rope).
struct QKNormRope {
    const void *wq, *wk, *freqs;
    float epsq, epsk;
    int64_t heads;
    void *vt;  // V^T tiles instead of the V columns of out, or null
};

static int gemm_run(const void *aq, const void *as, const void *bq, const void *bs, int64_t M, int64_t N, int64_t K,
                    int epilogue, int layouts, const void *bias, const void *gate, const void *res, int64_t seq,
                    void *out, int64_t ldo, void *out_scales, const QKNormRope *qk, void *stream,
                    void *ws = nullptr, int64_t ws_bytes = 0) {
    QIM_REQUIRE(aq && as && bq && bs && out, QIM_ERR_ARG, "qim_mxfp8_gemm: null pointer");
    constexpr int KNOWN = QIM_GEMM_A_TILED | QIM_GEMM_B_TILED | QIM_GEMM_OUT_TILED | QIM_GEMM_OUT_F32 | QIM_GEMM_OUT_F16;
    QIM_REQUIRE((layouts & ~KNOWN) == 0, QIM_ERR_ARG, "qim_mxfp8_gemm: unknown layout flags 0x%x", layouts);
    const int out_format = layouts & (QIM_GEMM_OUT_F32 | QIM_GEMM_OUT_F16);
    QIM_REQUIRE(out_format != (QIM_GEMM_OUT_F32 | QIM_GEMM_OUT_F16), QIM_ERR_ARG,
                "qim_mxfp8_gemm: QIM_GEMM_OUT_F32 and QIM_GEMM_OUT_F16 exclude each other");
    QIM_REQUIRE(!out_format || epilogue == QIM_EPI_NONE, QIM_ERR_ARG,
                "qim_mxfp8_gemm: an fp32 / fp16 output is available with QIM_EPI_NONE only");
    QIM_REQUIRE(!(layouts & QIM_GEMM_OUT_TILED) || epilogue == QIM_EPI_SWIGLU_QUANT, QIM_ERR_ARG,
                "qim_mxfp8_gemm: a tiled output needs the quantized SwiGLU epilogue");
    QIM_REQUIRE(M > 0 && N > 0 && K > 0, QIM_ERR_SHAPE, "qim_mxfp8_gemm: empty problem");
    QIM_REQUIRE(K % 128 == 0, QIM_ERR_SHAPE, "qim_mxfp8_gemm: K=%lld is not a multiple of 128", (long long)K);
    QIM_REQUIRE(N % 128 == 0, QIM_ERR_SHAPE, "qim_mxfp8_gemm: N=%lld is not a multiple of 128", (long long)N);
    const int64_t Mp = (M + 127) / 128 * 128;
    const int64_t tiles_m = (Mp + BM - 1) / BM, tiles_n = N / BN;
    QIM_REQUIRE(4 * tiles_m * tiles_n < (1ll << 31), QIM_ERR_SHAPE, "qim_mxfp8_gemm: too many tiles");
    QIM_REQUIRE(aligned16(aq) && aligned16(bq) && aligned16(as) && aligned16(bs) && aligned16(out) &&
                    (!res || aligned16(res)) && (!gate || aligned16(gate)) && (!out_scales || aligned16(out_scales)),
                QIM_ERR_LAYOUT, "qim_mxfp8_gemm: operands must be 16-byte aligned");
    QIM_REQUIRE(epilogue == QIM_EPI_SWIGLU_QUANT || ldo % 8 == 0, QIM_ERR_LAYOUT,
                "qim_mxfp8_gemm: ldo=%lld is not a multiple of 8", (long long)ldo);
    // The epilogues address a 64-row half's outputs with 32-bit offsets.
    QIM_REQUIRE(ldo < (1ll << 25), QIM_ERR_LAYOUT, "qim_mxfp8_gemm: ldo=%lld too large", (long long)ldo);
    QIM_REQUIRE(Mp / 128 < (1ll << 30), QIM_ERR_SHAPE, "qim_mxfp8_gemm: M=%lld too large", (long long)M);
    QIM_REQUIRE(Mp * K < (1ll << 31) && N * K < (1ll << 31), QIM_ERR_SHAPE,
                "qim_mxfp8_gemm: operands above 2 GiB are not supported");
    GemmArgs a{(const uint8_t *)aq, (const uint8_t *)as, (const uint8_t *)bq, (const uint8_t *)bs, M, Mp, N, K,
               (const uint16_t *)bias, (const uint16_t *)gate, (const uint16_t *)res, seq > 0 ? seq : M, out, ldo,
               (uint8_t *)out_scales, (int)tiles_m, (int)tiles_n, 0, 0,
               (layouts & QIM_GEMM_A_TILED) != 0, (layouts & QIM_GEMM_B_TILED) != 0,
               (layouts & QIM_GEMM_OUT_TILED) != 0,
               nullptr, nullptr, nullptr, 0.0f, 0.0f, 0, 0, nullptr, 0};
    if (qk) {
        a.wq = (const uint16_t *)qk->wq;
        a.wk = (const uint16_t *)qk->wk;
        a.freqs = (const float *)qk->freqs;
        a.epsq = qk->epsq;
        a.epsk = qk->epsk;
        a.q_cols = qk->heads * 128;
        a.qk_cols = 2 * qk->heads * 128;
        a.vt = static_cast<uint16_t *>(qk->vt);
        a.vt_nkb = seq / 64;
    }
    const GemmPlan pl = gemm_plan(M, N, K, epilogue);
    a.main_tiles = (int)pl.main_tiles;
    a.quarters = (int)pl.quarters;
    a.qrows = (int)pl.qrows;
    a.qcols = (int)pl.qcols;
    a.tile_rows = pl.tile_rows;
    if (pl.tile_rows != BM) a.tiles_m = (int)((Mp + pl.tile_rows - 1) / pl.tile_rows);
    if (ws) {
        QIM_REQUIRE(aligned16(ws), QIM_ERR_LAYOUT, "qim_mxfp8_gemm_ws: ws must be 16-byte aligned");
        if (pl.ksplit > 1 && ws_bytes >= pl.ws_bytes()) {
            a.ws = static_cast<float *>(ws);
            a.ksplit = pl.ksplit;
        }
    }
    int rc;
    switch (epilogue) {
        case QIM_EPI_NONE:
            QIM_REQUIRE(ldo >= N, QIM_ERR_LAYOUT, "qim_mxfp8_gemm: ldo=%lld < N", (long long)ldo);
            if (out_format == QIM_GEMM_OUT_F32)
                rc = launch_gemm<EPI_F32>(a, as_stream(stream));
            else if (out_format == QIM_GEMM_OUT_F16)
                rc = launch_gemm<EPI_F16>(a, as_stream(stream));
            else
                rc = launch_gemm<QIM_EPI_NONE>(a, as_stream(stream));
            break;
        case QIM_EPI_BIAS:
            QIM_REQUIRE(bias, QIM_ERR_ARG, "qim_mxfp8_gemm: bias epilogue without bias");
            QIM_REQUIRE(ldo >= N, QIM_ERR_LAYOUT, "qim_mxfp8_gemm: ldo=%lld < N", (long long)ldo);
            rc = launch_gemm<QIM_EPI_BIAS>(a, as_stream(stream));
            break;
        case QIM_EPI_GATED_RESIDUAL:
            QIM_REQUIRE(gate && res, QIM_ERR_ARG, "qim_mxfp8_gemm: gated residual needs gate and res");
            QIM_REQUIRE(ldo >= N, QIM_ERR_LAYOUT, "qim_mxfp8_gemm: ldo=%lld < N", (long long)ldo);
            rc = launch_gemm<QIM_EPI_GATED_RESIDUAL>(a, as_stream(stream));
            break;
        case QIM_EPI_SWIGLU:
            QIM_REQUIRE(N % 512 == 0, QIM_ERR_SHAPE, "qim_mxfp8_gemm: SwiGLU needs N %% 512 == 0");
            QIM_REQUIRE(ldo >= N / 2, QIM_ERR_LAYOUT, "qim_mxfp8_gemm: ldo=%lld < N/2", (long long)ldo);
            rc = launch_gemm<QIM_EPI_SWIGLU>(a, as_stream(stream));
            break;
        case QIM_EPI_SWIGLU_QUANT:
            QIM_REQUIRE(N % 512 == 0, QIM_ERR_SHAPE, "qim_mxfp8_gemm: SwiGLU needs N %% 512 == 0");
            QIM_REQUIRE(out_scales, QIM_ERR_ARG, "qim_mxfp8_gemm: quantized output needs out_scales");
            rc = launch_gemm<QIM_EPI_SWIGLU_QUANT>(a, as_stream(stream));
            break;
        case QIM_EPI_QK_NORM_ROPE:
            QIM_REQUIRE(qk, QIM_ERR_ARG, "qim_mxfp8_gemm: the QK epilogue is qim_mxfp8_gemm_qk_norm_rope's");
            QIM_REQUIRE(ldo >= N, QIM_ERR_LAYOUT, "qim_mxfp8_gemm: ldo=%lld < N", (long long)ldo);
            rc = qk->vt ? launch_gemm<EPI_QKV_VT>(a, as_stream(stream))
                        : launch_gemm<QIM_EPI_QK_NORM_ROPE>(a, as_stream(stream));
            break;
        default:
            return fail(QIM_ERR_ARG, "qim_mxfp8_gemm: unknown epilogue %d", epilogue);
    }
    return rc ? rc : check_launch("qim_mxfp8_gemm");
}

extern "C" int qim_mxfp8_gemm(const void *aq, const void *as, const void *bq, const void *bs, int64_t M, int64_t N,
                              int64_t K, int epilogue, const void *bias, const void *gate, const void *res,
                              int64_t seq, void *out, int64_t ldo, void *out_scales, void *stream) {
    return qim_mxfp8_gemm_ex(aq, as, bq, bs, M, N, K, epilogue, 0, bias, gate, res, seq, out, ldo, out_scales,
                             stream);
}

extern "C" int qim_mxfp8_gemm_ex(const void *aq, const void *as, const void *bq, const void *bs, int64_t M,
                                 int64_t N, int64_t K, int epilogue, int layouts, const void *bias, const void *gate,
                                 const void *res, int64_t seq, void *out, int64_t ldo, void *out_scales,
                                 void *stream) {
    return gemm_run(aq, as, bq, bs, M, N, K, epilogue, layouts, bias, gate, res, seq, out, ldo, out_scales, nullptr,
                    stream);
}

extern "C" int64_t qim_mxfp8_gemm_ws_bytes(int64_t M, int64_t N, int64_t K, int epilogue) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 128 || N % 128) return 0;
    return gemm_plan(M, N, K, epilogue).ws_bytes();
}

extern "C" int qim_mxfp8_gemm_ws(const void *aq, const void *as, const void *bq, const void *bs, int64_t M,
                                 int64_t N, int64_t K, int epilogue, int layouts, const void *bias, const void *gate,
                                 const void *res, int64_t seq, void *out, int64_t ldo, void *out_scales, void *ws,
                                 int64_t ws_bytes, void *stream) {
    return gemm_run(aq, as, bq, bs, M, N, K, epilogue, layouts, bias, gate, res, seq, out, ldo, out_scales, nullptr,
                    stream, ws, ws_bytes);
}

static int qk_norm_rope_run(const char *who, const void *aq, const void *as, const void *bq, const void *bs, int64_t M,
                            int64_t K, int64_t H, int layouts, const void *wq, const void *wk, const void *freqs,
                            int64_t seq, float epsq, float epsk, void *out, int64_t ldo, void *vt, void *stream) {
    QIM_REQUIRE(wq && wk && freqs, QIM_ERR_ARG, "%s: null pointer", who);
    QIM_REQUIRE(H > 0 && H % 2 == 0 && H < (1 << 20), QIM_ERR_SHAPE,
                "%s: H=%lld must be even (N = 3 H 128 %% 256 == 0)", who, (long long)H);
    QIM_REQUIRE(seq > 0 && seq < (1ll << 31) && M < (1ll << 31), QIM_ERR_SHAPE, "%s: seq=%lld / M=%lld out of range",
                who, (long long)seq, (long long)M);
    QIM_REQUIRE(aligned16(wq) && aligned16(wk) && aligned16(freqs) && aligned16(vt), QIM_ERR_LAYOUT,
                "%s: wq, wk, freqs (and vt) must be 16-byte aligned", who);
    QIM_REQUIRE((layouts & QIM_GEMM_OUT_TILED) == 0, QIM_ERR_ARG, "%s: the output is bf16 (no tiled output)", who);
    const QKNormRope qk{wq, wk, freqs, epsq, epsk, H, vt};
    return gemm_run(aq, as, bq, bs, M, 3 * H * 128, K, QIM_EPI_QK_NORM_ROPE, layouts, nullptr, nullptr, nullptr, seq,
                    out, ldo, nullptr, &qk, stream);
}

extern "C" int qim_mxfp8_gemm_qk_norm_rope(const void *aq, const void *as, const void *bq, const void *bs,
                                           int64_t M, int64_t K, int64_t H, int layouts, const void *wq,
                                           const void *wk, const void *freqs, int64_t seq, float epsq, float epsk,
                                           void *out, int64_t ldo, void *stream) {
    return qk_norm_rope_run("qim_mxfp8_gemm_qk_norm_rope", aq, as, bq, bs, M, K, H, layouts, wq, wk, freqs, seq, epsq,
                            epsk, out, ldo, nullptr, stream);
}

extern "C" int qim_mxfp8_gemm_qk_norm_rope_vt(const void *aq, const void *as, const void *bq, const void *bs,
                                              int64_t M, int64_t K, int64_t H, int layouts, const void *wq,
                                              const void *wk, const void *freqs, int64_t seq, float epsq,
                                              float epsk, void *out, int64_t ldo, void *vt, void *stream) {
    QIM_REQUIRE(vt, QIM_ERR_ARG, "qim_mxfp8_gemm_qk_norm_rope_vt: null vt");
    QIM_REQUIRE(seq > 0 && seq % 64 == 0 && M % seq == 0, QIM_ERR_SHAPE,
                "qim_mxfp8_gemm_qk_norm_rope_vt: seq=%lld must be a multiple of 64 dividing M=%lld", (long long)seq,
                (long long)M);
    return qk_norm_rope_run("qim_mxfp8_gemm_qk_norm_rope_vt", aq, as, bq, bs, M, K, H, layouts, wq, wk, freqs, seq,
                            epsq, epsk, out, ldo, vt, stream);
}
