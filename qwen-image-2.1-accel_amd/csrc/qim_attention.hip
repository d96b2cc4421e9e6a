// Attention core of the MMDiT block: O = softmax(Q K^T * scale) V per (batch,
// head), head dim 128, bf16 in and out, fp32 scores, softmax statistics and
// accumulation, in the online-softmax (flash) form: K/V are streamed in blocks
// of 64 keys and never materialise the score matrix.  No mask (bidirectional
// attention over [prefix + target] keys, the reference's SDPA call of
// optimizations/quantized_decode.py:70-77).
//
// Transposed formulation on v_mfma_f32_32x32x16_bf16: S^T = K Q^T (32 keys x 32
// queries per MFMA tile) and O^T = V^T P^T (32 head dims x 32 queries), so
// lane l owns query l % 32 in both: the running max and sum and the rescale
// of O are lane-local; the two half-waves, which hold different keys of one
// query, exchange one value per block.  An S^T accumulator is already the B
// operand of the P V product: lane (q, h = l / 32) holds keys
// {8(i/4) + 4h + i%4}, i = 0..15, of its 32-key tile, so values 0-7 are its 8
// keys of the first 16-key MFMA step and 8-15 of the second.  The A operand of
// lane (d, h) is the same 8 keys of V's column d.  (An MFMA pairs the K slots of A
// and B by position, so any key order works as long as A and B agree.)
//
// V comes in one of two forms.  Rows: loaded straight from the V tensor and
// transposed by the LDS reads (two ds_read_b64_tr_b16 of 4 keys per operand).  V^T
// tiles: written to the workspace by the QKV GEMM's epilogue, or by a transpose
// pass (k_attn_vt) where the queries are many (ATT_VROWS_MAX_S): one 16 KiB tile
// per (batch, head, 64-key block), 128 rows (d) of 64 keys with each 16-key group
// in the operand order ([0-3, 8-11 | 4-7, 12-15]), so that an operand is one
// 16-byte read, and the 16-byte chunk c of row d at chunk c ^ ((d >> 1) & 7)
// (conflict-free reads of 16 lanes with consecutive d).  K is loaded straight from
// the K tensor, with chunk c of key r at chunk c ^ (r & 15) in LDS.
//
// What bounds it: the clock, 1.84-1.87 GHz of 2.4 in long runs (power limit), and
// the cycles beyond the matrix cores' own.  Counters, per 32-cycle MFMA of a wave:
// S = T = 16640, 24 heads, V^T tiles 44.9 cycles, of which the matrix core is busy
// 34.0 (2 for the row sums; 76 %); the wave issues in 25.2, has an instruction ready
// that cannot issue in 13.0 and waits (barrier, LDS, loads) in 6.7.  S 4096 x T 8392,
// 32 heads, V rows: 49.6, busy 34.0 (69 %), 28.3, 13.1 and 8.2.  No LDS bank
// conflicts in either.  How much of the waits are barriers and how much are loads was
// not separated.  Against the schedule the compiler made with every call
// transposing V (same box each): S = T = 16640 2785 -> 2600 us, S 4096 x T 8392 496 ->
// 443 us, S = T = 4352 (24 heads) 231 -> 208 us, S 1024 x T 1101 (2 x 32 heads) 54.7 ->
// 40.5 us.
#include <type_traits>

#include "qim_attention.h"
#include "qim_device.h"
#include "qim_runtime.h"

namespace qim {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16a_t __attribute__((ext_vector_type(16)));
typedef float f32x4a_t __attribute__((ext_vector_type(4)));

constexpr int ATT_D = 128;          // head dim
constexpr int ATT_KB = 64;          // keys per block
constexpr int ATT_BQ = 256;         // queries per workgroup: 4 waves x 2 tiles of 32
constexpr int ATT_TILE = ATT_KB * ATT_D * 2;  // 16 KiB: one K block or one V^T block
constexpr int ATT_NSTAGE = 4;
constexpr int ATT_LDS = ATT_NSTAGE * 2 * ATT_TILE;  // 128 KiB

struct AttnArgs {
    const uint16_t *q, *k;
    const uint16_t *vt;  // V^T tiles (k_attn_fwd<., true>)
    const uint16_t *v;   // V rows (k_attn_fwd<., false>)
    uint16_t *o;
    int64_t ldq, ldk, ldv, ldo;  // elements between consecutive tokens
    int S, T, H, nkb;       // queries, keys, heads, key blocks
    int nq;                 // query blocks per (batch, head)
    // Work split (att_plan): workgroups [0, nfull) each run one whole work item
    // (query block, head, batch); the remaining ntail items run as nsplit
    // chunks of kbc key blocks each, writing partial results (part_o: each
    // chunk's normalised output rows O_c / l_c in bf16, part_ml: (m, l) per
    // query in fp32) that k_attn_merge combines.
    int nfull, ntail, nsplit, kbc;
    uint16_t *part_o;
    float *part_ml;
    float scale_log2e;
    // MXFP8 output (qim_attention_mxfp8) instead of o: E4M3 codes of the
    // (B*S, H*128) output, row-major or in the GEMM's tiled layout over Mp
    // rows (mxt_offset), and its swizzled E8M0 scales.
    uint8_t *qcodes, *qscales;
    int64_t Mp;
    int tiled;
    int o_vec16;  // rows of o are 16-byte aligned
};

// One query row's 4-column group of an MXFP8 output: code byte offset.
__device__ __forceinline__ int64_t att_code_offset(const AttnArgs &p, int64_t row, int64_t k) {
    const int64_t K = (int64_t)p.H * ATT_D;
    return p.tiled ? mxt_offset(row, k, p.Mp, K) : row * K + k;
}

// ---------------------------------------------------------- V transpose --
// One workgroup per (batch, head, key block): 64 keys x 128 d through LDS.
__global__ __launch_bounds__(256) void k_attn_vt(const uint16_t *__restrict__ v, int64_t ldv, uint16_t *__restrict__ vt,
                                                 int T, int H, int nkb) {
    __shared__ uint16_t s[ATT_KB][ATT_D + 8];  // +8: stagger rows across banks
    const int kb = blockIdx.x, h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x;
    // Load: 64 keys x 16 chunks of 16 bytes; zeros past the last key.
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int idx = it * 256 + tid, key = idx >> 4, c = idx & 15;
        const int t = kb * ATT_KB + key;
        uint4 x = make_uint4(0, 0, 0, 0);
        if (t < T) x = ld_nt(v + ((int64_t)b * T + t) * ldv + (int64_t)h * ATT_D + c * 8);
        *reinterpret_cast<uint4 *>(&s[key][c * 8]) = x;
    }
    __syncthreads();
    // Store: 128 rows (d) x 8 chunks; physical chunk pc of row d holds logical
    // chunk c = pc ^ ((d >> 1) & 7): keys 16g + [4hh, 4hh+4) and 16g + 8 + [4hh, 4hh+4)
    // with g = c / 2, hh = c % 2.
    uint16_t *tile = vt + (((int64_t)b * H + h) * nkb + kb) * (ATT_KB * ATT_D);
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int idx = it * 256 + tid, d = idx >> 3, pc = idx & 7;
        const int c = pc ^ ((d >> 1) & 7), g = c >> 1, hh = c & 1;
        const int k0 = 16 * g + 4 * hh;
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int key_lo = (e < 2) ? k0 + 2 * e : k0 + 8 + 2 * (e - 2);
            w[e] = (uint32_t)s[key_lo][d] | ((uint32_t)s[key_lo + 1][d] << 16);
        }
        *reinterpret_cast<uint4 *>(tile + d * ATT_KB + pc * 8) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// ------------------------------------------------------------- forward --
template <int N>
__device__ __forceinline__ void att_wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// LDS: a ring of 4 K blocks (16 KiB each), then a ring of 4 V blocks.  Block n
// is in slot gray(n % 4) (0, 1, 3, 2), so going to the next block flips one
// address bit: 14 after even blocks, 15 after odd ones.
constexpr int ATT_VRING = ATT_NSTAGE * ATT_TILE;
__device__ __forceinline__ uint32_t att_flip(int n) { return (uint32_t)ATT_TILE << (n & 1); }
typedef __attribute__((address_space(3))) const u32x4_t *att_lds_vec_t;
typedef short i16x4_t __attribute__((ext_vector_type(4)));

// DMA addressing of one wave's share of a key block: 4 instructions of K and
// 4 of V (1 KiB each).  Instruction j (n = 4 wave + j) covers keys 4n..4n+3 of
// the block: lane i lands at LDS row r = 4n + i/16, physical chunk i % 16, whose
// source is the row's logical chunk (i % 16) ^ (r & 15) for K and
// (i % 16) ^ 4 (r & 3) for V rows; V^T tiles are copied as they are.  An
// instruction's offset field moves its LDS and its global address alike, so the
// four share one M0; the per-lane offsets are reduced by 1 KiB j and raised by
// ATT_BIAS, which the base pointers are lowered by.  Per block only the
// (wave-uniform) bases move; before the last block its rows past T - 1 are
// clamped to T - 1 (their scores are masked; V rows are zeroed in LDS).
constexpr int ATT_BIAS = 3072;
struct AttLoader {
    const uint8_t *kp, *vp;    // K and V of the next block to issue
    int64_t kstep, vstep;      // bytes per block
    uint32_t koff[4], voff[4]; // per-lane offsets (voff[0] only for V^T tiles)
    uint32_t lds;              // LDS address of this wave's share of the next slot
    int next, last;            // the next block and the range's last one
    int rmax;                  // last valid row of the range's last block (>= 63: whole)
};

template <bool VT>
__device__ __forceinline__ void att_offsets(const AttnArgs &p, AttLoader &L, int wave, int lane, int rmax) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = 4 * (wave * 4 + j) + (lane >> 4), rl = r < rmax ? r : rmax;
        const int adj = ATT_BIAS - 1024 * j;
        L.koff[j] = (uint32_t)(((int64_t)rl * p.ldk + ((lane & 15) ^ (r & 15)) * 8) * 2 + adj);
        L.voff[j] = VT ? (uint32_t)(wave * 4096 + lane * 16 + ATT_BIAS)
                       : (uint32_t)(((int64_t)rl * p.ldv + ((lane & 15) ^ ((r & 3) << 2)) * 8) * 2 + adj);
    }
}

// A wave-uniform pointer in scalar registers (the DMA's base operand).
__device__ __forceinline__ const uint8_t *att_uniform(const uint8_t *ptr) {
    const uint64_t a = reinterpret_cast<uint64_t>(ptr);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    return reinterpret_cast<const uint8_t *>((uint64_t)hi << 32 | lo);
}

template <bool VT>
__device__ __forceinline__ AttLoader att_loader(const AttnArgs &p, int b, int h, int kb0, int nkb, int wave, int lane) {
    AttLoader L;
    L.kstep = (int64_t)ATT_KB * p.ldk * 2;
    L.vstep = VT ? ATT_TILE : (int64_t)ATT_KB * p.ldv * 2;
    L.kp = reinterpret_cast<const uint8_t *>(p.k + (int64_t)b * p.T * p.ldk + (int64_t)h * ATT_D) + kb0 * L.kstep - ATT_BIAS;
    L.vp = (VT ? reinterpret_cast<const uint8_t *>(p.vt + ((int64_t)b * p.H + h) * p.nkb * (ATT_KB * ATT_D))
               : reinterpret_cast<const uint8_t *>(p.v + (int64_t)b * p.T * p.ldv + (int64_t)h * ATT_D)) +
           kb0 * L.vstep - ATT_BIAS;
    L.kp = att_uniform(L.kp);
    L.vp = att_uniform(L.vp);
    L.lds = wave * 4096;
    L.next = 0;
    L.last = nkb - 1;
    L.rmax = p.T - 1 - (kb0 + nkb - 1) * ATT_KB;
    att_offsets<VT>(p, L, wave, lane, ATT_KB);
    return L;
}

template <int OFF>
__device__ __forceinline__ void att_dma16(const uint8_t *base, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3" ::"v"(voff), "s"(base), "{m0}"(lds_addr), "n"(OFF)
                 : "memory");
}

// Before a block's DMA: the clamped offsets of a last block that is not whole.
template <bool VT>
__device__ __forceinline__ void att_issue_begin(const AttnArgs &p, AttLoader &L, int wave, int lane) {
    if (L.next == L.last && L.rmax < ATT_KB - 1) att_offsets<VT>(p, L, wave, lane, L.rmax);
}
// DMA instruction `part` of the next block (0-3: K, 4-7: V).
template <bool VT>
__device__ __forceinline__ void att_issue_part(const AttLoader &L, int part) {
    const uint32_t k = L.lds, v = L.lds + ATT_VRING;
    if (part == 0) att_dma16<0>(L.kp, L.koff[0], k);
    if (part == 1) att_dma16<1024>(L.kp, L.koff[1], k);
    if (part == 2) att_dma16<2048>(L.kp, L.koff[2], k);
    if (part == 3) att_dma16<3072>(L.kp, L.koff[3], k);
    if (part == 4) att_dma16<0>(L.vp, L.voff[0], v);
    if (part == 5) att_dma16<1024>(L.vp, VT ? L.voff[0] : L.voff[1], v);
    if (part == 6) att_dma16<2048>(L.vp, VT ? L.voff[0] : L.voff[2], v);
    if (part == 7) att_dma16<3072>(L.vp, VT ? L.voff[0] : L.voff[3], v);
}
// After it: on to the next block (the last one again past the end, into a slot
// that is never read).
__device__ __forceinline__ void att_issue_end(AttLoader &L, uint32_t flip) {
    const bool more = L.next < L.last;
    L.kp += more ? L.kstep : 0;
    L.vp += more ? L.vstep : 0;
    L.next += more ? 1 : 0;
    L.lds ^= flip;
}

// LDS addresses of a lane's fragments in the current slots (the kernel's LDS
// starts at address 0); sub-blocks and V's head-dim tiles (V^T) or key steps (V
// rows) are offsets of the reads themselves.
//   K, head-dim step j: lane (r = key % 32, hf) reads d [16j + 8hf, +8) of key r.
//   V^T, 16-key step kk of the block: lane (d % 32, hf) reads the 8 keys that
//     pair with its P^T operand; head dims 32 dt + d % 32.
//   V rows, head-dim tile dt: the transposing read gives lane i of a 16-lane
//     group column i of the 4 x 16 block whose row j is held by lanes 4j..4j+3,
//     so lane l addresses 8 bytes of key 4hf + (l % 16) / 4 (and 8 keys later),
//     d 32 dt + 16 ((l / 16) % 2) + 4 (l % 4); the chunk swizzle 4 (key % 4)
//     spreads the 4 keys over all banks.
struct AttAddr {
    uint32_t k[8], v[4];
};
template <bool VT>
__device__ __forceinline__ AttAddr att_addr(int lane) {
    AttAddr A;
    const int lq = lane & 31, hf = lane >> 5, i = lane & 15;
#pragma unroll
    for (int j = 0; j < 8; ++j) A.k[j] = lq * 256 + (((2 * j + hf) ^ (lq & 15)) << 4);
#pragma unroll
    for (int t = 0; t < 4; ++t)
        A.v[t] = ATT_VRING +
                 (VT ? lq * (ATT_KB * 2) + (((2 * t + hf) ^ ((lq >> 1) & 7)) << 4)
                     : (4 * hf + (i >> 2)) * 256 + ((t ^ (i >> 2)) << 6) + ((lane >> 4) & 1) * 32 + (i & 3) * 8);
    return A;
}
__device__ __forceinline__ bf16x8_t att_read_k(const AttAddr &A, int j, int off) {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<att_lds_vec_t>((uintptr_t)(A.k[j] + off)));
}
// V fragment of 16-key step kk, head-dim tile dt.
template <bool VT>
__device__ __forceinline__ bf16x8_t att_read_v(const AttAddr &A, int kk, int dt) {
    if constexpr (VT) {
        return __builtin_bit_cast(bf16x8_t,
                                  *reinterpret_cast<att_lds_vec_t>((uintptr_t)(A.v[kk] + dt * (32 * ATT_KB * 2))));
    } else {
        typedef __attribute__((address_space(3))) i16x4_t *ptr_t;
        const uint32_t at = A.v[dt] + kk * (16 * ATT_D * 2);
        const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<ptr_t>((uintptr_t)at));
        const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<ptr_t>((uintptr_t)(at + 8 * ATT_D * 2)));
        return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
}

// The loader of a range, its first three blocks issued.
template <bool VT>
__device__ __forceinline__ AttLoader att_start(const AttnArgs &p, int b, int h, int kb0, int nkb, int wave, int lane) {
    AttLoader ld = att_loader<VT>(p, b, h, kb0, nkb, wave, lane);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        att_issue_begin<VT>(p, ld, wave, lane);
#pragma unroll
        for (int part = 0; part < 8; ++part) att_issue_part<VT>(ld, part);
        att_issue_end(ld, att_flip(i));
    }
    return ld;
}

// Keys at or past T (the partial last block) get a score of -inf.
__device__ __forceinline__ void att_mask(f32x16a_t &s, int kbase, int T, int hf) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int key = kbase + 8 * (i >> 2) + 4 * hf + (i & 3);
        if (key >= T) s[i] = -__builtin_inff();
    }
}

__device__ __forceinline__ float att_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// The (unscaled) row max of a score tile over both half-waves (the other
// half-wave holds the other 16 keys of the same query).
__device__ __forceinline__ float att_rowmax(const f32x16a_t &s) {
    float a0 = att_max(s[0], s[1]), a1 = att_max(s[2], s[3]);
#pragma unroll
    for (int i = 4; i < 16; i += 4) {
        a0 = att_max(a0, att_max(s[i], s[i + 1]));
        a1 = att_max(a1, att_max(s[i + 2], s[i + 3]));
    }
    const float mx0 = att_max(a0, a1);
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx0), __float_as_uint(mx0), false, false);
    return att_max(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
}

// One 32-query tile of a wave: scores, P^T operands, O^T and the statistics.
// P of 16 keys x 32 queries per MFMA step: w[0..3] and w[4..7], packed bf16.
struct AttTile {
    f32x16a_t s, o[4];
    uint32_t w[8];
    float e[2];     // P of a pair not yet packed
    float m;        // reference max (log2 units)
    float l;        // this lane's sum of P (of the bf16 values used), sub-blocks before the last one's
    f32x4a_t r;     // the last sub-block's sum, in every element: added to l by att_sum
};
__device__ __forceinline__ bf16x8_t att_p(const AttTile &t, int u) {
    const u32x4_t v = {t.w[4 * u], t.w[4 * u + 1], t.w[4 * u + 2], t.w[4 * u + 3]};
    return __builtin_bit_cast(bf16x8_t, v);
}

// P = 2^(s c - m) of score k of a tile (called for k = 0..17 in order): the
// exponential of score k, and for even k the packing of the pair before it (one
// slot later, so that nothing waits for an exponential).  One slot after every
// second pair its and the previous pair's four values are added to r: v_mfma_f32_4x4x4_16b_bf16 with an
// all-ones A is, for each lane, the sum of the lane's own four B values.  (As
// v_dot2c_f32_bf16, eight per 16 scores, the sums slowed the MFMAs beside them:
// 49.4 against 37.4 cycles per MFMA without them, loads left out.)  r starts at
// zero with each sub-block and is added to l once: 16 values whose exponents
// differ by at most 12 add up exactly, and l, which grows with the keys, is
// rounded once per 16 of them.
__device__ __forceinline__ void att_exp(AttTile &t, int k, float c, i16x4_t ones) {
    if (k > 0 && k <= 16 && (k & 1) == 0) {
        uint32_t w = pack_bf16x2(t.e[0], t.e[1]);
        // Keeps the work in its slot: it would otherwise sink to where P is used.
        asm volatile("" : "+v"(w));
        t.w[k / 2 - 1] = w;
    }
    if (k > 4 && (k & 3) == 1) {
        const u32x2_t v = {t.w[(k - 1) / 2 - 2], t.w[(k - 1) / 2 - 1]};
        t.r = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_bit_cast(i16x4_t, v), k == 5 ? f32x4a_t{} : t.r, 0, 0,
                                                     0);
    }
    if (k < 16) t.e[k & 1] = __builtin_amdgcn_exp2f(__builtin_fmaf(t.s[k], c, -t.m));
}

__device__ __forceinline__ void att_sum(AttTile &t) { t.l += t.r[0]; }

// Online softmax with a running max (the safe form).  Scores above the
// reference max m by at most ATT_RESCALE (log2 units) are exponentiated
// against m as they are (P <= 2^ATT_RESCALE); a sub-block whose max exceeds
// that moves m to its max and rescales l and O (skipped, wave-uniform, when no
// query of the wave moved its max).
constexpr float ATT_RESCALE = 8.0f;

__device__ __forceinline__ void att_softmax_safe(AttTile &t, float c, i16x4_t ones) {
    const float mx = att_rowmax(t.s) * c;
    const float mnew = mx > t.m + ATT_RESCALE ? mx : t.m;
    const float alpha = __builtin_amdgcn_exp2f(t.m - mnew);  // 1 if m stays, 0 on the first sub-block
    t.m = mnew;
    t.l *= alpha;
#pragma unroll
    for (int k = 0; k <= 17; ++k) att_exp(t, k, c, ones);
    att_sum(t);
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) t.o[dt] *= alpha;
    }
}

#define ATT_SCHED() __builtin_amdgcn_sched_barrier(0)

// Waits until at most N of this wave's LDS reads are outstanding.  A builtin,
// not assembly: the compiler sees it and adds no wait per fragment (each a
// 4-cycle instruction) after it.
template <int N>
__device__ __forceinline__ void att_wait_lds() {
    static_assert(N <= 15, "lgkmcnt is 4 bits");
    __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));
}

// One region: 16 MFMAs of tile A -- its scores with the K fragments `kf`, then
// O += V^T P^T with the V fragments `vf` -- beside the softmax of tile B, in 16
// slots of one MFMA and one score each.  A lone wave issues at most one
// instruction per 4.4 cycles (5.4 for an 8-byte one, 8.5 for an exponential), so
// a slot of one MFMA, a score's fma and exponential, half a pack and a row sum and
// one LDS read could fit the MFMA's 32 cycles; what the whole loop takes stands at
// the head of the file.  (Left to itself the compiler
// bunched the softmax into the first half of each region, left the rest to bare
// MFMAs, and waited for each fragment separately.)  `work(k)` is the slot's memory
// work.  LDSK: the fragments were read in the previous region, K first; at most
// LDSK reads (V's) may be outstanding at the first score, none at the first P V.
// FAST: B's reference max is fixed, nothing to rescale; its sum r is complete
// only at the region's end and is added to l in the next one (where the tile is
// A), so that nothing waits for it.  Otherwise the safe softmax runs whole,
// before the MFMAs.
template <bool FAST, bool SCORES, bool PV, bool SOFTMAX, int LDSK, class F>
__device__ __forceinline__ void att_region(AttTile &A, AttTile &B, const bf16x8_t (&q)[8], const bf16x8_t (&kf)[8],
                                           bf16x8_t (&vf)[2][4], float c, i16x4_t ones, F &&work) {
    if constexpr (!FAST && SOFTMAX) att_softmax_safe(B, c, ones);
    if constexpr (LDSK >= 0 && SCORES) att_wait_lds<LDSK>();
    if (FAST) ATT_SCHED();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (k < 8) {
            if constexpr (SCORES)
                A.s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[k], q[k], k == 0 ? f32x16a_t{} : A.s, 0, 0, 0);
        } else {
            if constexpr (PV) {
                const int u = (k - 8) / 4, dt = k & 3;
                A.o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[u][dt], att_p(A, u), A.o[dt], 0, 0, 0);
            }
        }
        if (FAST) ATT_SCHED();
        if constexpr (FAST && SOFTMAX) att_exp(B, k, c, ones);
        if constexpr (FAST && PV)
            if (k == 2) att_sum(A);
        work(k);
        if (LDSK >= 0 && PV && k == 7) {
            att_wait_lds<0>();
            // V fragments live in accumulation registers (MFMA operands only):
            // the architectural ones hold O, the scores and P.
#pragma unroll
            for (int i = 0; i < 8; ++i) asm volatile("" : "+a"(vf[i / 4][i & 3]));
        }
        if (FAST) ATT_SCHED();
    }
    if constexpr (FAST && SOFTMAX) {
        att_exp(B, 16, c, ones);
        att_exp(B, 17, c, ones);
    }
    if (FAST) ATT_SCHED();
}

// One pass over the key blocks of a range for this wave's 64 queries: two
// 32-query tiles (0, 1), keys in 32-key sub-blocks u (two per 64-key LDS
// block).  Per sub-block the work is S_t = K Q_t^T, the softmax SM_t and O_t +=
// V^T P_t^T; it runs software-pipelined in two regions so that each softmax
// runs on the vector ALU beside 16 MFMAs that do not depend on it:
//   Y(u): MFMA S_0(u + 1), PV_0(u)   | VALU SM_1(u) | DMA of block n + 3
//   X(u): MFMA S_1(u), PV_1(u - 1)   | VALU SM_0(u) | LDS reads of K(u + 1), V(u)
// Every K and V fragment is read from LDS once and used for both query tiles;
// its successor is read right after its last use (in X), 8 to 16 MFMAs before
// the successor's first (in Y).  Block n + 3 is issued into the ring slot of
// block n - 1 after the barrier before X(2n + 1), which follows the last read of
// that slot.
//
// FAST: after each tile's first sub-block (which sets m to its max) the
// reference max stays fixed, so a region has no max, no rescale and no branch.
// P may then exceed 1 by the growth of the scores past the first sub-block's
// max; the caller checks that l stayed below ATT_FAST_LMAX (so that P, l and O
// stayed finite) and otherwise reruns the pass with FAST = false.
template <bool FAST, bool VT>
__device__ __forceinline__ void att_pass(const AttnArgs &p, AttLoader ld, uint8_t *lds, const bf16x8_t (&qf)[2][8],
                                         int wave, int lane, int kb0, int nkb, AttTile &t0, AttTile &t1) {
    // Key blocks [kb0, kb0 + nkb); n below counts from kb0.  Keys past T exist
    // only in the last block of T; a sub-block there may be all masked, which
    // gives P = 0 and leaves m, l and O as they are.
    const int hf = lane >> 5, lastb = nkb - 1;
    const int kl = (kb0 + lastb) * ATT_KB;  // first key of the last block
    const bool ragged = p.T - kl < ATT_KB;
    const float c = p.scale_log2e;
    const i16x4_t ones = {0x3f80, 0x3f80, 0x3f80, 0x3f80};  // bf16 1.0
    AttAddr A = att_addr<VT>(lane);
    bf16x8_t kf[8], vf[2][4];
    t0.m = t1.m = -__builtin_inff();
    t0.l = t1.l = 0.f;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) t0.o[dt] = t1.o[dt] = f32x16a_t{};

    // V rows past the last key count as zeros (V^T tiles hold zeros there).
    auto zero_rows = [&](int slot) {
        if (VT) return;
        const int tail = p.T - kl;
        for (int i = threadIdx.x; i < (ATT_KB - tail) * 16; i += 256)
            *reinterpret_cast<uint4 *>(lds + ATT_VRING + slot * ATT_TILE + tail * 256 + i * 16) = make_uint4(0, 0, 0, 0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    // Block 0 landed for every wave: S_0(0), S_1(0), SM_0(0), which sets the
    // tiles' reference max.
    att_wait_vmcnt<16>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (lastb == 0 && ragged) zero_rows(0);
    auto none = [](int) {};
    auto kread = [&](int k, int off) {
        if (k < 8) kf[k] = att_read_k(A, k, off);
    };
    auto vread = [&](int k, int half) {
        if (k >= 8) vf[(k - 8) / 4][k & 3] = att_read_v<VT>(A, 2 * half + (k - 8) / 4, k & 3);
    };
#pragma unroll
    for (int k = 0; k < 8; ++k) kread(k, 0);
    att_region<false, true, false, false, -1>(t0, t1, qf[0], kf, vf, c, ones, none);
    att_region<false, true, false, false, -1>(t1, t0, qf[1], kf, vf, c, ones, none);
    if (lastb == 0 && ragged) {
        att_mask(t0.s, kl, p.T, hf);
        att_mask(t1.s, kl, p.T, hf);
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        kread(k, 32 * 256);
        vread(k, 0);
    }
    if (FAST) {
        t0.m = att_rowmax(t0.s) * c;
        t1.m = att_rowmax(t1.s) * c;
#pragma unroll
        for (int k = 0; k <= 17; ++k) att_exp(t0, k, c, ones);
    } else {
        att_softmax_safe(t0, c, ones);
    }

    constexpr int LDSK = VT ? 8 : 15;  // V reads after the K reads: 8 (V^T) or 16
    for (int n = 0; n < lastb; ++n) {
        const uint32_t flip = att_flip(n);
        // Y(2n)
        att_region<FAST, true, true, true, LDSK>(t0, t1, qf[0], kf, vf, c, ones, none);
        // Block n + 1 landed for every wave; the slot of block n - 1 is free.
        att_wait_vmcnt<8>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        att_issue_begin<VT>(p, ld, wave, lane);
#pragma unroll
        for (int j = 0; j < 8; ++j) A.k[j] ^= flip;
        // X(2n + 1)
        att_region<FAST, true, true, true, -1>(t1, t0, qf[1], kf, vf, c, ones, [&](int k) {
            kread(k, 0);
            vread(k, 1);
        });
        // Y(2n + 1)
        att_region<FAST, true, true, true, LDSK>(t0, t1, qf[0], kf, vf, c, ones, [&](int k) {
            if (k & 1) att_issue_part<VT>(ld, k / 2);
        });
        att_issue_end(ld, att_flip(n + 3));
        if (n + 1 == lastb && ragged) {
            att_mask(t0.s, kl, p.T, hf);
            zero_rows((lastb & 3) ^ ((lastb & 3) >> 1));
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) A.v[t] ^= flip;
        // X(2n + 2)
        att_region<FAST, true, true, true, -1>(t1, t0, qf[1], kf, vf, c, ones, [&](int k) {
            kread(k, 32 * 256);
            vread(k, 0);
        });
    }
    // Last block L: Y(2L), X(2L + 1), Y(2L + 1) without new scores, PV_1(2L + 1).
    if (ragged) att_mask(t1.s, kl, p.T, hf);
    att_region<FAST, true, true, true, LDSK>(t0, t1, qf[0], kf, vf, c, ones, none);
    if (ragged) att_mask(t0.s, kl + 32, p.T, hf);
    att_region<FAST, true, true, true, -1>(t1, t0, qf[1], kf, vf, c, ones, [&](int k) { vread(k, 1); });
    if (ragged) att_mask(t1.s, kl + 32, p.T, hf);
    att_region<FAST, false, true, true, 0>(t0, t1, qf[0], kf, vf, c, ones, none);
    att_region<FAST, false, true, false, -1>(t1, t0, qf[1], kf, vf, c, ones, none);
    att_wait_vmcnt<0>();  // the repeated tail loads land before the LDS is reused or released
}

// Bound on a lane's partial sum l after a FAST pass: below it, every P and
// every |O| (for |V| < 2^63) stayed finite.
constexpr float ATT_FAST_LMAX = 18446744073709551616.0f;  // 2^64

template <bool QOUT, bool VT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_attn_fwd(AttnArgs p) {
    // The kernel's only LDS, so it starts at address 0 (AttAddr, AttLoader::lds).
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lq = lane & 31, hf = lane >> 5;

    // Work item (query block, head, batch) and key-block range.  Workgroup ids
    // go to the XCDs round-robin (over 8); each range of workgroups (the whole
    // items, then the tail chunks) is remapped so that each XCD runs a
    // contiguous range of it: the query blocks of few heads at a time, which
    // share K and V^T in that XCD's L2.  Tail chunks are ordered chunk-major.
    int item, kb0 = 0, nkb = p.nkb, tail = -1;
    {
        int lin = blockIdx.x, nw = p.nfull;
        if (lin >= p.nfull) {
            lin -= p.nfull;
            nw = p.ntail * p.nsplit;
        }
        const int xcd = lin & 7, base = nw >> 3, rem = nw & 7;
        const int w = xcd * base + (xcd < rem ? xcd : rem) + (lin >> 3);
        if (blockIdx.x < (unsigned)p.nfull) {
            item = w;
        } else {
            const int chunk = w / p.ntail, ti = w % p.ntail;
            item = p.nfull + ti;
            kb0 = chunk * p.kbc;
            nkb = p.nkb - kb0 < p.kbc ? p.nkb - kb0 : p.kbc;
            tail = ti * p.nsplit + chunk;
        }
    }
    const int qblk = item % p.nq, h = (item / p.nq) % p.H, b = item / (p.nq * p.H);
    const int q0 = qblk * ATT_BQ + wave * 64;

    // The first key blocks are in flight while Q is loaded.
    const AttLoader ld = att_start<VT>(p, b, h, kb0, nkb, wave, lane);
    // Q^T operands: lane (q, hf) holds d [16j + 8hf, +8) of query q0 + 32t + q.
    bf16x8_t qf[2][8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        int qi = q0 + 32 * t + lq;
        qi = qi < p.S ? qi : p.S - 1;  // rows past the end: computed, not stored
        const uint16_t *qrow = p.q + ((int64_t)b * p.S + qi) * p.ldq + (int64_t)h * ATT_D + hf * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[t][j] = *reinterpret_cast<const bf16x8_t *>(qrow + 16 * j);
    }
    // Q^T is only ever an MFMA operand: keep it in accumulation registers, which
    // leaves the architectural ones to O, the scores, P and the softmax.
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(qf[t][j]));

    AttTile t0, t1;
    att_pass<true, VT>(p, ld, lds, qf, wave, lane, kb0, nkb, t0, t1);
    float l0 = t0.l, l1 = t1.l;
    // Rerun the whole workgroup in the safe form when any wave's sums left
    // the range the fixed reference max guarantees (scores that grew by more
    // than ~64 in log2 units past their first sub-block's max).
    const bool bad = !(l0 < ATT_FAST_LMAX && l1 < ATT_FAST_LMAX);
    const int wave_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    __syncthreads();  // every wave is done with the rings
    int *const redo = reinterpret_cast<int *>(lds);
    if (lane == 0) redo[wave] = wave_bad;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(redo[0] | redo[1] | redo[2] | redo[3])) {
        __syncthreads();  // read by every wave before the rings are filled again
        att_pass<false, VT>(p, att_start<VT>(p, b, h, kb0, nkb, wave, lane), lds, qf, wave, lane, kb0, nkb, t0, t1);
        l0 = t0.l;
        l1 = t1.l;
    }

    // O = O^T / l: lane (q, hf) holds dims 32dt + 8(i/4) + 4hf + i%4 of its query.
    // A tail chunk writes the same bf16 rows into its part_o slot (256 x 128)
    // and (m, l) of each query into part_ml, for k_attn_merge.
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const f32x16a_t(&o)[4] = t ? t1.o : t0.o;
        const float lf = t ? l1 : l0;
        const float lt = lf + __shfl_xor(lf, 32, 64);
        const float inv = 1.0f / lt;
        const int qi = q0 + 32 * t + lq;
        const bool live = qi < p.S;  // the same for both half-waves of a query
        if (QOUT && tail < 0) {
            // MXFP8: the bf16 values the plain output would hold, quantized as
            // qim_mx_quantize does.  A 32-column block (dt) is this lane's 16
            // values and its partner's (lane ^ 32).
            const int64_t row = (int64_t)b * p.S + qi;
            uint32_t sc = 0;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                float f[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) f[i] = rbf(o[dt][i] * inv);
                uint32_t m = absmax_bits8(f);
                const uint32_t m2 = absmax_bits8(f + 8);
                m = m2 > m ? m2 : m;
                const uint32_t mp = (uint32_t)__shfl_xor((int)m, 32, 64);
                m = mp > m ? mp : m;
                const int e = mx_exponent(__uint_as_float(m));
                const float s = mx_scale_operand(e);
#pragma unroll
                for (int g = 0; g < 4; g += 2) {
                    // Columns 8g + 4hf and 8(g + 1) + 4hf; after the exchange
                    // the 8 of group g + hf.
                    const auto c = __builtin_amdgcn_permlane32_swap(
                        cvt_e4m3x4_scaled(f[4 * g], f[4 * g + 1], f[4 * g + 2], f[4 * g + 3], s),
                        cvt_e4m3x4_scaled(f[4 * g + 4], f[4 * g + 5], f[4 * g + 6], f[4 * g + 7], s), false, false);
                    const int64_t k = (int64_t)h * ATT_D + 32 * dt + 8 * (g + hf);
                    if (live) *reinterpret_cast<uint2 *>(p.qcodes + att_code_offset(p, row, k)) = make_uint2(c[0], c[1]);
                }
                sc |= (uint32_t)e << (8 * dt);
            }
            if (live && hf == 0)
                *reinterpret_cast<uint32_t *>(p.qscales + mx_scale_offset(row, 4 * h, (int64_t)p.H * ATT_D)) = sc;
            continue;
        }
        uint16_t *orow = p.o + ((int64_t)b * p.S + qi) * p.ldo + (int64_t)h * ATT_D;
        bool vec16 = p.o_vec16;
        if (tail >= 0) {
            const int ql = wave * 64 + 32 * t + lq;
            orow = p.part_o + ((int64_t)tail * ATT_BQ + ql) * ATT_D;
            vec16 = true;
            if (live && hf == 0)
                *reinterpret_cast<float2 *>(p.part_ml + ((int64_t)tail * ATT_BQ + ql) * 2) =
                    make_float2(t ? t1.m : t0.m, lt);
        }
        // The half-waves exchange 4-column groups (8g + 4hf of an even and an odd
        // g) so that each lane stores the 16 bytes of group g + hf: half as many
        // stores, each instruction covering whole 32-byte sectors.
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int g = 0; g < 4; g += 2) {
                const auto x = __builtin_amdgcn_permlane32_swap(pack_bf16x2(o[dt][4 * g + 0] * inv, o[dt][4 * g + 1] * inv),
                                                                pack_bf16x2(o[dt][4 * g + 4] * inv, o[dt][4 * g + 5] * inv),
                                                                false, false);
                const auto y = __builtin_amdgcn_permlane32_swap(pack_bf16x2(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv),
                                                                pack_bf16x2(o[dt][4 * g + 6] * inv, o[dt][4 * g + 7] * inv),
                                                                false, false);
                uint16_t *at = orow + 32 * dt + 8 * (g + hf);
                if (live && vec16) {
                    *reinterpret_cast<uint4 *>(at) = make_uint4(x[0], y[0], x[1], y[1]);
                } else if (live) {  // ldo need only be a multiple of 4 elements
                    *reinterpret_cast<uint2 *>(at) = make_uint2(x[0], y[0]);
                    *reinterpret_cast<uint2 *>(at + 4) = make_uint2(x[1], y[1]);
                }
            }
    }
}

// Combine the chunks of each tail item from their normalised rows
// R_c = O_c / l_c: O = sum_c w_c R_c / sum_c w_c with w_c = 2^(m_c - M) l_c,
// M = max_c m_c (accumulated with a running max).  One thread per (item,
// query, 8 d).
__global__ __launch_bounds__(256) void k_attn_merge(AttnArgs p) {
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int dg = (int)(g & 15), ql = (int)((g >> 4) & (ATT_BQ - 1));
    const int ti = (int)(g >> 12);  // 16 x 256 threads per item
    if (ti >= p.ntail) return;
    const int item = p.nfull + ti;
    const int qblk = item % p.nq, h = (item / p.nq) % p.H, b = item / (p.nq * p.H);
    const int qi = qblk * ATT_BQ + ql;
    if (qi >= p.S) return;
    // One pass, rescaling the running sums when the max grows, so that each
    // chunk's loads do not wait for the previous chunks' arithmetic.
    const int nc = p.nsplit;
    float M = -__builtin_inff(), wsum = 0.f;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int c = 0; c < nc; ++c) {
        const int64_t tc = (int64_t)(ti * p.nsplit + c);
        const float2 ml = *reinterpret_cast<const float2 *>(p.part_ml + (tc * ATT_BQ + ql) * 2);
        float r[8];
        unpack8(*reinterpret_cast<const uint4 *>(p.part_o + (tc * ATT_BQ + ql) * ATT_D + dg * 8), r);
        const float Mn = ml.x > M ? ml.x : M;
        const float sc = __builtin_amdgcn_exp2f(M - Mn);  // 0 on the first chunk (M = -inf)
        const float w = __builtin_amdgcn_exp2f(ml.x - Mn) * ml.y;
        wsum = wsum * sc + w;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = acc[e] * sc + w * r[e];
        M = Mn;
    }
    const float inv = 1.0f / wsum;
    if (p.qcodes) {
        // MXFP8 output: a 32-column block is 4 adjacent threads (dg 4j .. 4j+3).
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = rbf(acc[e] * inv);
        int e;
        const uint2 c = quantize8(f, e);
        const int64_t row = (int64_t)b * p.S + qi;
        *reinterpret_cast<uint2 *>(p.qcodes + att_code_offset(p, row, (int64_t)h * ATT_D + dg * 8)) = c;
        if ((dg & 3) == 0) p.qscales[mx_scale_offset(row, 4 * h + (dg >> 2), (int64_t)p.H * ATT_D)] = (uint8_t)e;
        return;
    }
    uint16_t *orow = p.o + ((int64_t)b * p.S + qi) * p.ldo + (int64_t)h * ATT_D + dg * 8;
    // 8-byte stores: ldo need only be a multiple of 4 elements.
    *reinterpret_cast<uint2 *>(orow) = make_uint2(pack_bf16x2(acc[0] * inv, acc[1] * inv),
                                                  pack_bf16x2(acc[2] * inv, acc[3] * inv));
    *reinterpret_cast<uint2 *>(orow + 4) = make_uint2(pack_bf16x2(acc[4] * inv, acc[5] * inv),
                                                      pack_bf16x2(acc[6] * inv, acc[7] * inv));
}

// MXFP8 output rows [M, Mp) (the padding of the last 128-row scale block):
// zero codes and scales, as qim_mx_quantize writes them.  One thread per
// 16-byte code chunk.
__global__ __launch_bounds__(256) void k_attn_qpad(AttnArgs p, int64_t M) {
    const int64_t K = (int64_t)p.H * ATT_D, per_row = K / 16;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t r = M + i / per_row, c = i % per_row;
    if (r >= p.Mp) return;
    *reinterpret_cast<uint4 *>(p.qcodes + att_code_offset(p, r, c * 16)) = make_uint4(0, 0, 0, 0);
    if (c < K / 128) *reinterpret_cast<uint32_t *>(p.qscales + mx_scale_offset(r, 4 * c, K)) = 0;
}

}  // namespace qim

using namespace qim;

// Work split.  Every workgroup of k_attn_fwd runs for about the same time and
// one fits per CU, so W whole items take ceil(W / CUs) rounds; when the last
// round is partial, its items may run instead as chunks of kbc key blocks plus
// a merge pass.  Cost model, in units of one workgroup's time per 64-key
// block (1.75 us at 24 heads when the model was made, 1.6 now): whole rounds * nkb + chunk rounds *
// kbc + the partials' HBM traffic (written once, read once by the merge, at
// ~5 TB/s) + ~3 for the merge launch.  A split is taken when it saves >= 5 %;
// chunks have at least ATT_MIN_CHUNK blocks.  Partials are bf16 rows and
// fp32 (m, l): 66 KiB per chunk.  (At S = T = 16640 and 24 heads the 24 tail
// items run as 10 chunks each, ~10 % faster; at S = T = 4352 the 152 tail
// items of one image run as 3 chunks each, ~1 % faster.)
namespace qim {

constexpr int ATT_MIN_CHUNK = 8;
// Most queries per image for which V is read as rows: the transposing reads
// take two instructions per fragment, the transpose pass one trip of V through
// memory, and the reads are repeated by every query block.  Rows against V^T with
// its pass: S 1024, T 1101, B 2, H 32 42.7 / 52.9 us; S = T = 1280, H 24 32.3 / 37.7;
// S 4096, T 8392, H 32 463 / 477; S = T = 4352, H 24 212 / 217; S = T = 8192, H 24 672.0
// / 671.8, H 32 893.0 / 891.8; S = T = 16640, H 24 2765 / 2718 us.
constexpr int64_t ATT_VROWS_MAX_S = 8192;

AttPlan att_plan(int64_t B, int64_t S, int64_t T, int64_t H) {
    const int64_t nq = (S + ATT_BQ - 1) / ATT_BQ, nkb = (T + ATT_KB - 1) / ATT_KB, W = B * H * nq;
    const int64_t C = device_cus() > 0 ? device_cus() : 256;
    AttPlan pl{W, 0, 1, nkb, B * H * nkb * ATT_TILE, 0, 0};
    const int64_t R = W / C, Wr = W - R * C;
    if (Wr == 0) return pl;
    const double per_chunk_bytes = 2.0 * (ATT_BQ * ATT_D * 2 + ATT_BQ * 2 * 4);  // written + read
    const double bytes_per_block = 5e12 * 1.75e-6;
    double best = 0.95 * (double)((R + 1) * nkb);
    for (int64_t k = 2; k <= 16; ++k) {
        const int64_t kbc = (nkb + k - 1) / k;
        if (kbc < ATT_MIN_CHUNK) break;
        const int64_t keff = (nkb + kbc - 1) / kbc;
        const int64_t rounds = (Wr * keff + C - 1) / C;
        const double cost = (double)(R * nkb + rounds * kbc) + (double)(Wr * keff) * per_chunk_bytes / bytes_per_block + 3.0;
        if (cost < best) {
            best = cost;
            pl.nfull = R * C;
            pl.ntail = Wr;
            pl.nsplit = keff;
            pl.kbc = kbc;
        }
    }
    if (pl.ntail) {
        pl.part_o_bytes = pl.ntail * pl.nsplit * ATT_BQ * ATT_D * 2;
        pl.part_ml_bytes = pl.ntail * pl.nsplit * ATT_BQ * 2 * 4;
    }
    return pl;
}

static bool ranges_overlap(const void *a, int64_t a_bytes, const void *b, int64_t b_bytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + (uintptr_t)b_bytes && y < x + (uintptr_t)a_bytes;
}

// Whether rows of `width` bytes, `stride` bytes apart, from a and from b are column
// blocks of one buffer that share no column.
static bool columns_disjoint(const void *a, const void *b, int64_t stride, int64_t width) {
    const int64_t d = (int64_t)(reinterpret_cast<uintptr_t>(a) - reinterpret_cast<uintptr_t>(b));
    const int64_t r = (d % stride + stride) % stride;  // a's first column seen from b's
    return r >= width && r + width <= stride;
}

// The checks and launches the attention entry points share.  Output: bf16 rows
// of o (ldo elements apart), or MXFP8 codes and scales when qcodes is set.
// v null: the workspace already holds V^T (qim_mxfp8_gemm_qk_norm_rope_vt),
// T % 64 == 0.  The workspace always has the room for V^T, also where V is read as
// rows: its size is asked for before it is known whether the output overlaps V.
int attention_run(const char *who, const void *q, int64_t ldq, const void *k, int64_t ldk, const void *v,
                         int64_t ldv, void *o, int64_t ldo, void *qcodes, void *qscales, int tiled, void *workspace,
                         int64_t workspace_bytes, int64_t B, int64_t S, int64_t T, int64_t H, int64_t D, float scale,
                         void *stream) {
    QIM_REQUIRE(q && k && (o || (qcodes && qscales)) && workspace, QIM_ERR_ARG, "%s: null pointer", who);
    QIM_REQUIRE(D == ATT_D, QIM_ERR_SHAPE, "%s: head dim %lld (128 only)", who, (long long)D);
    QIM_REQUIRE(scale > 0.0f && scale < 1e30f, QIM_ERR_ARG, "%s: scale must be positive and finite", who);
    QIM_REQUIRE(B > 0 && S > 0 && T > 0 && H > 0, QIM_ERR_SHAPE, "%s: empty problem", who);
    QIM_REQUIRE(B < 65536 && H < 65536 && S < (1 << 30) && T < (1 << 30) && B * H * ((S + ATT_BQ - 1) / ATT_BQ) < (1 << 30),
                QIM_ERR_SHAPE, "%s: too large", who);
    QIM_REQUIRE(v || T % ATT_KB == 0, QIM_ERR_SHAPE, "%s: V^T from the workspace (v null) needs T %% 64 == 0", who);
    QIM_REQUIRE(ldq >= H * D && ldk >= H * D && (!v || (ldv >= H * D && ldv % 8 == 0)) && ldq % 8 == 0 &&
                    ldk % 8 == 0 &&
                    (qcodes || (ldo >= H * D && ldo % 4 == 0)),
                QIM_ERR_LAYOUT, "%s: token strides must cover H*D and be multiples of 8 (ldo: 4)", who);
    QIM_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(workspace) &&
                    (qcodes ? aligned16(qcodes) && aligned16(qscales) : (reinterpret_cast<uintptr_t>(o) & 7u) == 0),
                QIM_ERR_LAYOUT, "%s: q, k, v, workspace (and codes, scales) 16-byte aligned, o 8-byte aligned", who);
    QIM_REQUIRE(tiled == 0 || tiled == 1, QIM_ERR_ARG, "%s: tiled must be 0 or 1", who);
    const int64_t nkb = (T + ATT_KB - 1) / ATT_KB;
    QIM_REQUIRE(B * T * ldk < (1ll << 31), QIM_ERR_SHAPE, "%s: K above 4 GiB of offsets", who);
    const AttPlan pl = att_plan(B, S, T, H);
    QIM_REQUIRE(workspace_bytes >= pl.total(), QIM_ERR_ARG,
                "%s: workspace of %lld bytes, this problem needs %lld (qim_attention_workspace_bytes)", who,
                (long long)workspace_bytes, (long long)pl.total());
    // V rows read through the transposing LDS reads, or V^T tiles: from the
    // workspace when v is null, else made here.  V rows are read until the last
    // workgroup ends, so an output whose memory overlaps V's takes V^T tiles,
    // which are complete before the first output is written.
    const int64_t M = B * S, Mp = (M + 127) / 128 * 128;
    bool vt = !v || S > ATT_VROWS_MAX_S || ldv >= (1ll << 25);  // (32-bit row offsets)
    if (!vt) {
        const int64_t v_bytes = ((B * T - 1) * ldv + H * D) * 2;
        vt = qcodes ? ranges_overlap(v, v_bytes, qcodes, Mp * H * D) || ranges_overlap(v, v_bytes, qscales, Mp * H * D / 32)
                    : ranges_overlap(v, v_bytes, o, ((M - 1) * ldo + H * D) * 2) &&
                          !(ldo == ldv && columns_disjoint(o, v, ldo * 2, H * D * 2));
    }
    static std::atomic<bool> configured[4][QIM_MAX_DEVICES] = {};
    void (*const fwd)(AttnArgs) = qcodes ? (vt ? k_attn_fwd<true, true> : k_attn_fwd<true, false>)
                                         : (vt ? k_attn_fwd<false, true> : k_attn_fwd<false, false>);
    if (const int rc = reserve_lds(reinterpret_cast<const void *>(fwd), ATT_LDS, configured[(qcodes ? 2 : 0) + vt], who))
        return rc;
    hipStream_t st = as_stream(stream);
    uint8_t *ws = static_cast<uint8_t *>(workspace);
    if (v && vt)
        launch(k_attn_vt, dim3((unsigned)nkb, (unsigned)H, (unsigned)B), dim3(256), 0, st,
                           (const uint16_t *)v, ldv, (uint16_t *)ws, (int)T, (int)H, (int)nkb);
    AttnArgs a{};
    a.q = (const uint16_t *)q;
    a.k = (const uint16_t *)k;
    a.vt = (const uint16_t *)ws;
    a.v = (const uint16_t *)v;
    a.ldv = ldv;
    a.o = (uint16_t *)o;
    a.ldq = ldq;
    a.ldk = ldk;
    a.ldo = ldo;
    a.S = (int)S;
    a.T = (int)T;
    a.H = (int)H;
    a.nkb = (int)nkb;
    a.nq = (int)((S + ATT_BQ - 1) / ATT_BQ);
    a.nfull = (int)pl.nfull;
    a.ntail = (int)pl.ntail;
    a.nsplit = (int)pl.nsplit;
    a.kbc = (int)pl.kbc;
    a.part_o = reinterpret_cast<uint16_t *>(ws + pl.vt_bytes);
    a.part_ml = reinterpret_cast<float *>(ws + pl.vt_bytes + pl.part_o_bytes);
    a.scale_log2e = scale * 1.4426950408889634f;
    a.qcodes = static_cast<uint8_t *>(qcodes);
    a.qscales = static_cast<uint8_t *>(qscales);
    a.Mp = Mp;
    a.tiled = tiled;
    a.o_vec16 = o && aligned16(o) && ldo % 8 == 0;
    const int64_t nwg = pl.nfull + pl.ntail * pl.nsplit;
    launch(fwd, dim3((unsigned)nwg), dim3(256), ATT_LDS, st, a);
    if (pl.ntail) {
        const int64_t threads = pl.ntail * ATT_BQ * (ATT_D / 8);
        launch(k_attn_merge, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, a);
    }
    if (qcodes && a.Mp > M) {
        const int64_t threads = (a.Mp - M) * H * ATT_D / 16;
        launch(k_attn_qpad, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, a, M);
    }
    return check_launch(who);
}

}  // namespace qim

extern "C" int qim_attention(const void *q, int64_t ldq, const void *k, int64_t ldk, const void *v, int64_t ldv,
                             void *o, int64_t ldo, void *workspace, int64_t workspace_bytes, int64_t B, int64_t S,
                             int64_t T, int64_t H, int64_t D, float scale, void *stream) {
    if (!o) return qim::fail(QIM_ERR_ARG, "qim_attention: null pointer");
    return attention_run("qim_attention", q, ldq, k, ldk, v, ldv, o, ldo, nullptr, nullptr, 0, workspace,
                         workspace_bytes, B, S, T, H, D, scale, stream);
}

extern "C" int qim_attention_mxfp8(const void *q, int64_t ldq, const void *k, int64_t ldk, const void *v,
                                   int64_t ldv, void *codes, void *scales, int tiled, void *workspace,
                                   int64_t workspace_bytes, int64_t B, int64_t S, int64_t T, int64_t H, int64_t D,
                                   float scale, void *stream) {
    if (!codes || !scales) return qim::fail(QIM_ERR_ARG, "qim_attention_mxfp8: null pointer");
    return attention_run("qim_attention_mxfp8", q, ldq, k, ldk, v, ldv, nullptr, 0, codes, scales, tiled, workspace,
                         workspace_bytes, B, S, T, H, D, scale, stream);
}

extern "C" int64_t qim_attention_workspace_bytes(int64_t B, int64_t S, int64_t T, int64_t H, int64_t D) {
    if (B <= 0 || S <= 0 || T <= 0 || H <= 0 || D != ATT_D) return 0;
    return att_plan(B, S, T, H).total();
}
