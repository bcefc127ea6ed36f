// Ring / block attention for MI355X (gfx950, CDNA4): forward with online softmax across
// KV chunks resident in HBM, recompute backward, behind the C ABI of include/ltr_attn.h.
//
// Kernel map
//   fwd_bf16_kernel<D, RB>   S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_32x32x16_bf16; a block of
//                        8 waves owns 256 * RB query rows, a wave 32 * RB of them, so a lane owns ONE query per row block:
//                        the row sums are in-lane reductions (no running max: the reference of the
//                        exponent moves only when a row sum leaves its safe range), and P^T leaves the
//                        first GEMM already in the B-operand layout of the second.  64-key K
//                        and V tiles go global -> LDS directly (no staging registers) into
//                        unpadded, XOR-swizzled, double-buffered tiles, one barrier per tile;
//                        the V^T operand is read with ds_read_b64_tr_b16.  The (O, LSE) merge
//                        with an earlier partial result is part of the epilogue.
//                        fwd_bf16_kernel<64, 2>: two 32-row blocks per wave (512 rows per block, 64-key tiles): every K / V
//                        operand read from LDS feeds two MFMAs (chosen by the host, or forced with LTR_FWD_ROWS_512).
//                        fwd_bf16_w4_kernel<D>, bwd_dq_w4_kernel<D>: 128 rows and four waves per block, several blocks per CU (FourWaves).
//   fwd_f32_mfma_kernel<D, KS>  fp32 I/O and arithmetic on v_mfma_f32_32x32x2_f32: the forward of the 1e-4 cases (the reference's
//                        acceptance dtype) on the matrix pipe; KS key shares per 32-row group for launches with few rows, <64, 4> of 16-row
//                        groups for those with the fewest (F32Rows16) and fwd_f32_rows32_kernel<64, 4> where their blocks pass one round;
//                        bwd_dq_f32_mfma_kernel, bwd_dq_f32_rows32_kernel likewise.
//   fwd_f32_kernel<D>    the same in scalar fp32 (no MFMA): kept as the fallback, reached with LTR_FWD_F32_SCALAR.
//                        fwd_bf16_shares_kernel<D, KS>, bwd_dq_shares_kernel<D, KS>: KS waves share a row group's keys (launches with
//                        few rows, see key_shares and choose_rows); *_pad_kernel: head dims below the width D (LTR_HEAD_COLS).
//   delta_kernel, delta_bf16_kernel<LANES>  DELTA = rowsum(dO * O).
//   bwd_dkdv_kernel<D, KW>  a block of 8 waves owns 128 * KW keys of one kv head and loops over the
//                        query heads of the GQA group and over 64-row query tiles taken from
//                        lists (fully visible / partly masked) built once in LDS.  Two waves
//                        share each 32-key slice: one computes S, P and dV^T, the other dP,
//                        dS and dK^T one tile behind, P handed over through LDS.  Q / dO tiles
//                        go global -> LDS directly into three swizzled buffers, one barrier
//                        per tile; K, V operands and the dK^T / dV^T accumulators stay in
//                        registers for the whole block.
//                        bwd_dkdv_kernel<64, 2>: two 32-key halves per wave (256 keys per block): every Q / dO operand
//                        read from LDS feeds two MFMAs, and a block's transfers and per-step costs are spread over
//                        twice the matrix work.  The registers allow it at head dim 64 only; chosen by the host
//                        for long equal blocks without masked tiles (or forced with LTR_DKDV_KEYS_256).
//   bwd_dkdv_keywave_kernel<64>  head dim 64: a wave does both halves of the work of its 32 keys, four waves per block, two blocks per CU.
//   bwd_dkdv_reduce_kernel<D, KW>  sums the partial dK / dV of blocks that share a key tile (see KvSplit).
//   bwd_dq_kernel<D, RB> forward-shaped: a block owns 256 * RB query rows, loops over K/V tiles
//                        (same direct-to-LDS tiles as the forward), recomputes S and dP and
//                        accumulates dQ^T in registers.  No atomics anywhere: results are
//                        bitwise reproducible.  bwd_dq_kernel<64, 2>: two 32-row blocks per wave (a lane owns two
//                        query rows): every K / V operand read from LDS feeds two MFMAs; head dim 64 only, chosen by the
//                        host when the wider blocks still fill the device (or forced with LTR_DQ_ROWS_512).
//   bwd_joint_kernel<D, KS>  the blocks of bwd_dq_kernel (KS = 2: of two key shares) and of bwd_dkdv_kernel<D, 1> in one launch, where
//                        they are few (LTR_BWD_JOINT); bwd_joint_delta_kernel<D>: with DELTA by the blocks themselves.
//   bwd_dq_f32_mfma_kernel<D, KS>, bwd_dkdv_f32_mfma_kernel<D>
//                        the fp32 backward on v_mfma_f32_32x32x2_f32 (see there).
//   bwd_dq_f32_kernel<D>, bwd_dkdv_f32_kernel<D, DV>
//                        the same backward in scalar fp32 (no MFMA): the fallback, reached with LTR_BWD_F32_SCALAR.
//   The tile loops of the bf16 kernels are unrolled over their LDS buffers (or, where registers are short,
//   keep per-lane LDS addresses in registers): no address arithmetic is left between the MFMAs.
//   RoPE: with LTR_ROPE_Q the forward rotates each q row in its operand registers (rope_rotate8) and can store the
//   rotated row; with LTR_ROPE_DQ the dQ kernel's epilogue rotates dQ by the conjugate angles (rope_conj4).
//   Block scheduling under a causal mask: a forward / dQ block takes a late q tile and its early counterpart when the
//   host says so (q_tile_slots; every other block in the opposite order, so that equal blocks do not all change tiles
//   at once), and the dK/dV kernel's chunk table is sorted by position (longest blocks first).
//   ltr_attn_bwd_noalloc keeps its DELTA workspace in the fixed __device__ array `scratch` (see there).
//
// MFMA 32x32x16 operand layout used throughout (lane l, i = l % 32, h = l / 32):
//   A[i][8h .. 8h+7], B[8h .. 8h+7][i], C[8*(r/4) + 4h + r%4][i] for accumulator register r.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>
#include <stdio.h>
#include <string.h>
#include <type_traits>
#include <optional>
#include <atomic>
#include <algorithm>
#include "ltr_attn.h"
#include "ltr_blocks.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

#define LTR_LOG2E 1.4426950408889634f
#define LTR_LN2 0.6931471805599453f

struct ChunkDev {
    const void *k;
    const void *v;
    float *dk;
    float *dv;
    int sk;
    int pos0;
};

struct FwdParams {
    const void *q;
    void *o;
    float *lse;
    int B, Hq, Hkv, n_rep;
    int cols;              // head dim of the tensors (the kernel's own width, or less: PAD kernels)
    int Sq, n_qtiles;
    int n_slots;           // q tiles are handed out in slots: n_qtiles of one tile, or (n_qtiles + 1) / 2 of two (see q_tile_slots)
    BlockMap map;
    long long qs[3], os[3], ks[3], vs[3];
    int q_pos0[2];
    int q_split;
    float scale;
    unsigned flags;
    int o_f32;
    int n_chunks;
    const float *rope;     // LTR_ROPE_Q: (cos, sin) rows, cols floats per position, row 0 = position rope_pos0
    int rope_pos0;
    void *q_rot;           // optional bf16 output: the rotated q
    long long qrs[3];
    ChunkDev chunk[LTR_MAX_CHUNKS];
};

struct BwdParams {
    const void *q;
    const void *d_o;
    const float *lse;
    float *delta;      // read; written by the dQ kernel with LTR_DELTA_FROM_O
    const void *o;     // forward output, read with LTR_DELTA_FROM_O (bf16) and LTR_DQ_F32_RESULT (fp32) only
    long long os_[3];
    void *dq;          // fp32 accumulator, or bf16 result with LTR_DQ_BF16
    int B, Hq, Hkv, n_rep;
    BlockMap q_map, kv_map;   // of the dQ and the dK/dV kernel
    JointMap joint;    // of bwd_joint_kernel, which holds the blocks of both
    int cols;          // head dim of the tensors (the kernel's own width, or less: PAD kernels)
    int Sq, n_qtiles;
    long long qs[3], dos[3], dqs[3], ks[3], vs[3], dks[3], dvs[3];
    int q_pos0[2];
    int q_split;
    float scale;
    unsigned flags;
    int n_chunks;
    int tiles_total;  // key tiles over all chunks
    int tiles_seen;   // those that have blocks in the dK/dV kernel: all of them, or (shared tiles, causal mask) those a query sees
    int q_last;       // largest position that counts as a query's for that: see seen_tiles
    int split_log2;   // log2 of the blocks that share one key tile of the dK/dV kernel (0: a block owns its keys alone), see KvSplit
    int share_log2;   // log2 of those that share out the q tiles of a head; the others share out the group's q heads,
    int n_reps;       // of which a block walks this many
    float *part;      // n_split > 1: the blocks' partial dK / dV, summed by bwd_dkdv_reduce_kernel
    int n_slots;      // slots of 256-row q tiles of the dQ kernel (see q_tile_slots)
    const float *rope;     // LTR_ROPE_DQ: (cos, sin) rows, cols floats per position, row 0 = position rope_pos0
    int rope_pos0;
    ChunkDev chunk[LTR_MAX_CHUNKS];
};

struct DeltaParams {
    const void *o;
    const void *d_o;
    float *delta;
    int B, Hq, D, Sq;
    long long os[3], dos[3];
    int o_f32, do_f32;
    int vec;           // rows start 16-byte aligned: 16-byte loads
    int rows32;        // B * Sq < 2^31
};

__device__ __forceinline__ int q_position(int row, int split, int p0, int p1) {
    return row < split ? p0 + row : p1 + (row - split);
}

// min and max global position over local rows [r0, r1] (inclusive, r0 <= r1)
__device__ __forceinline__ void q_pos_range(int r0, int r1, int split, int p0, int p1, int &lo, int &hi) {
    int a = q_position(r0, split, p0, p1), b = q_position(r1, split, p0, p1);
    lo = min(a, b);
    hi = max(a, b);
    if (r0 < split && r1 >= split) {  // tile straddles the two segments
        int c = q_position(split - 1, split, p0, p1), d = q_position(split, split, p0, p1);
        lo = min(lo, min(c, d));
        hi = max(hi, max(c, d));
    }
}

// Masked tiles of the forward and dQ kernels: a key of the chunk is visible to a row up to the chunk's end and, under a causal mask, up to the
// row's position.  Which of the 32 keys from `first` on (keys of the chunk) are, as bits: a score then costs a bit-field extract and a bit-field
// insert.  (With the two comparisons per score it was six instructions, and 32 registers of the forward held the keys; a comparison with a
// constant and a select wait for each other through VCC.)
__device__ __forceinline__ unsigned visible_bits(bool causal, int row_pos, int chunk_pos0, int chunk_keys, int first) {
    int last = chunk_keys - 1;
    if (causal) last = min(last, __builtin_elementwise_sub_sat(row_pos, chunk_pos0));
    const int n = min(max(__builtin_elementwise_sub_sat(last, first), -1), 31) + 1;
    return (unsigned)((1ull << n) - 1);
}
__device__ __forceinline__ float visible_score(unsigned bits, int key, float s) {   // s, or -inf
    const unsigned keep = (unsigned)__builtin_amdgcn_sbfe((int)bits, key, 1);
    return __uint_as_float((keep & __float_as_uint(s)) | (~keep & 0xff800000u));
}

__device__ __forceinline__ BlockItem block_item(const BlockMap &m, int pairs) { return block_item_at(m, pairs, blockIdx.x, blockIdx.y, blockIdx.z); }

// both halves of the wave end up with combine(x[l], x[l ^ 32])
__device__ __forceinline__ float xhalf_max(float x) {
    unsigned u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
    unsigned u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// ds_read_b64_tr_b16: within each group of 16 lanes, lane i receives as element e the
// 16-bit value that lane (4e + i/4) of the group addressed at position i % 4.  With lane s
// of a group pointing at M[k0 + s/4][n0 + 4*(s%4)] of a row-major tile, lane i receives
// M[k0 + 0..3][n0 + i]: four consecutive rows of one column, i.e. the MFMA K-dim packing.
__device__ __forceinline__ i16x4 lds_read_tr16(const __bf16 *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((i16x4 __attribute__((address_space(3))) *)(p));
}

// Unpadded row-major LDS tile of D bf16 per row whose 16-byte chunks are XOR-swizzled: chunk c of row r
// lives at chunk position c ^ lds_swz<D>(r).  LDS has 64 banks of 4 bytes; a 128-bit read is served 16
// lanes at a time and a 64-bit (transpose) read 32 lanes at a time.  With this permutation both the MFMA
// operand read (16 consecutive rows, same logical chunk) and the transpose read (4 consecutive rows x 4
// consecutive chunks) touch every bank exactly once, and so does the staging store (one row per 16 lanes).
template <int D>
__device__ __forceinline__ int lds_swz(int row) {
    return D == 128 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}

template <int D>
__device__ __forceinline__ int lds_swz_off(int row, int chunk) {   // element offset of (row, 16-byte chunk)
    return row * D + ((chunk ^ lds_swz<D>(row)) << 3);
}

// 8 K-dim values for an MFMA operand whose K index runs over the ROWS of a row-major LDS
// tile: rows {k0 + 4h + 0..3} and {k0 + 8 + 4h + 0..3} at column n_base + (l % 32).
// This row set is the one the accumulator registers 8b..8b+7 of a 32x32 MFMA result
// hold (rows 16b + 4h + 0..3 and 16b + 8 + 4h + 0..3), so a result tile can feed the
// next GEMM as an operand without leaving registers.
// (tile = swizzled tile, see lds_swz)
template <int D>
__device__ __forceinline__ bf16x8 lds_operand_tr_swz(const __bf16 *tile, int k0, int n_base, int lane) {
    // k0 is a multiple of 16, which the swizzle of a row does not see: it is an immediate beside the lane's address, and one pair of addresses
    // per column block serves every k0 (left to the compiler each k0 had its own: 24 registers of the forward and dK/dV kernels)
    const int li = lane & 15, g = lane >> 4;
    const int hh = g >> 1;
    const int col = n_base + ((g & 1) << 4) + ((li & 3) << 2);
    const int row = 4 * hh + (li >> 2);
    const __bf16 *const block = tile + k0 * D;
    i16x4 lo = lds_read_tr16(block + lds_swz_off<D>(row, col >> 3) + (col & 7));
    i16x4 hi = lds_read_tr16(block + lds_swz_off<D>(row + 8, col >> 3) + (col & 7));
    union {
        struct { i16x4 a, b; } s;
        bf16x8 v;
    } u;
    u.s.a = lo;
    u.s.b = hi;
    return u.v;
}

// 16 bytes per lane from global memory straight into LDS: lane l's data lands at LDS byte address lds_byte_addr + 16*l
// (wave-uniform; lds_address() of a __shared__ object plus an offset).  No staging registers, no LDS store pass.  Written as inline assembly so that the compiler
// does not track the transfer: with the builtin it makes the next LDS read of ANY address wait for vmcnt(0),
// which would expose the whole global-memory latency in the middle of a tile.  The transfer is only complete
// after tile_barrier() (the only place that waits for it); nothing may read the destination before that.
__device__ __forceinline__ unsigned lds_address(const void *shared_object) {
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void *)shared_object;
}

__device__ __forceinline__ void global_to_lds_b128(const void *gptr, unsigned lds_byte_addr_uniform) {
    const unsigned lds_addr = __builtin_amdgcn_readfirstlane(lds_byte_addr_uniform);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gptr), "s"(lds_addr) : "memory", "m0");
}

// End of a tile: wait for every outstanding tile transfer and LDS access of this wave, then the block
// barrier.  The wait is the s_waitcnt builtin (vmcnt(0) lgkmcnt(0), expcnt left alone) so that the compiler's
// own counter bookkeeping knows that nothing is pending afterwards.
__device__ __forceinline__ void tile_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// PAD kernels serve head dims between the two instantiated widths (multiples of 8): the tensors have `cols` < D columns, the LDS
// tiles keep the width D.  The 16-byte chunks past the last column are cleared once (nothing else ever writes them: a tile
// transfer leaves its lanes out), so the padding costs neither memory traffic nor passes over the tensors.  Measured beside
// zero-padding q, k, v and slicing the results (B=2, 16 heads, D=96, S=777, forward + backward): 163 us with 11 pad, fill and slice
// launches (47 us of them), 80 us without.
// The kernels of width 128 skip the fourth block of 32 columns where the tensors end by column 96 (DC = 96 columns computed; tiles, swizzle and
// addresses stay those of the width): a quarter of the matrix work and of the LDS reads.  Kernel us, all four blocks -> three, forward / dQ / dK/dV:
//   2 x 16 heads of 96 S=777   18.8 / 25.6 / 31.1 -> 17.6 / 24.6 / 28.3     8 x 32 on 8 of 96 S=2048   280 / 416 / 510 -> 253 / 372 / 453
//   6 x 8 heads of 80 S=3000    114 / 159 / 218 -> 103 / 141 / 195          1 x 32 of 72, S=1000, no mask   23.0 / 31.5 / 38.9 -> 21.5 / 29.7 / 34.7
// Those are kernels of their own, told apart by the type of their argument: with both bodies in one kernel each had the registers of the larger
// and twice the spilled scalars (bwd_joint_pad_kernel<128, 2> 115 for 40, 256 vector registers for 215), head dims above 96 too.  In time
// it is 1 % at most (2 x 16 heads of 96, S=777, joint 37.3 -> 36.8 us; 8 x 32 on 8 of 96, S=2048 the same).
template <class Params>
struct Columns96 : Params {};   // the same bytes
template <int BYTES>
__device__ __forceinline__ void clear_lds(unsigned char *smem) {   // followed by a barrier: the fill covers the columns that transfers write
    for (int i = threadIdx.x * 16; i < BYTES; i += 512 * 16) *(uint4 *)(smem + i) = make_uint4(0, 0, 0, 0);
    __syncthreads();
}

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 x) {
    union { uint4 u; bf16x8 v; } c;
    c.u = x;
    return c.v;
}

// Rotary position embedding of 8 consecutive elements (4 adjacent (re, im) pairs) of one row: f0, f1 hold the pairs'
// (cos, sin).  The arithmetic of apply_rotary_emb (layers/layers.py:44-70) as the streaming kernel of ltr_rope_apply does
// it: fp32 complex multiply with the four products rounded separately, result rounded to bf16 - so a row rotated here has
// the bits that the separate pass would have written.
__device__ __forceinline__ bf16x8 rope_rotate8(bf16x8 x, f32x4 f0, f32x4 f1) {
#pragma clang fp contract(off)
    const float cs[4] = {f0[0], f0[2], f1[0], f1[2]}, sn[4] = {f0[1], f0[3], f1[1], f1[3]};
    bf16x8 out;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float re = (float)x[2 * i], im = (float)x[2 * i + 1];
        const float rr = re * cs[i], ii = im * sn[i];
        const float ri = re * sn[i], ir = im * cs[i];
        out[2 * i] = (__bf16)(rr - ii);
        out[2 * i + 1] = (__bf16)(ri + ir);
    }
    return out;
}

// Gradient of that rotation: 4 consecutive fp32 elements (2 pairs) times the CONJUGATE angles; f = (cos, sin, cos, sin).
__device__ __forceinline__ f32x4 rope_conj4(f32x4 v, f32x4 f) {
#pragma clang fp contract(off)
    f32x4 out;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const float re = v[2 * i], im = v[2 * i + 1], c = f[2 * i], sn = f[2 * i + 1];
        out[2 * i] = re * c + im * sn;
        out[2 * i + 1] = im * c - re * sn;
    }
    return out;
}

struct PackedTile {   // 16 bf16 values of one lane's 32x32 tile column, as the two B operands of K = 16
    unsigned u[8];
};

__device__ __forceinline__ unsigned pack2_bf16(float a, float b) {
    bf16x2 t;
    t[0] = (__bf16)a;
    t[1] = (__bf16)b;
    return __builtin_bit_cast(unsigned, t);
}

__device__ __forceinline__ bf16x8 operand_of(const PackedTile &t, int kb) {
    union { unsigned u[4]; bf16x8 v; } c;
    c.u[0] = t.u[4 * kb];
    c.u[1] = t.u[4 * kb + 1];
    c.u[2] = t.u[4 * kb + 2];
    c.u[3] = t.u[4 * kb + 3];
    return c.v;
}

typedef __attribute__((address_space(3))) const bf16x8 *lds_bf16x8_ptr;
typedef __attribute__((address_space(3))) i16x4 *lds_i16x4_ptr;
typedef __attribute__((address_space(3))) const f32x4 *lds_f32x4_ptr;
typedef __attribute__((address_space(3))) const i32x4 *lds_i32x4_ptr;

// GEMM loops of the kernels whose LDS addresses of the lane's operands are in registers (one per 16 columns of a tile's rows, or a pair per
// head-dimension block: the swizzle makes them differ per lane, not by a constant), plus an immediate for the rows and the buffer.
// A kernel that does not unroll its tile loop over the LDS buffers flips them between the buffers with one XOR each per tile.

// Two independent 32x32 accumulation chains over the head dimension (added to ra / rb as passed in), A operands from rows of swizzled LDS tiles,
// B operands from registers.  The chains alternate so no MFMA waits for its predecessor, and the operand reads
// run PF steps ahead of the MFMAs that use them; sched_barrier pins that order (left alone, the scheduler sinks
// each read to just before its use and the full LDS latency is exposed at every step).
template <int D, int DC = D>
__device__ __forceinline__ void lds_gemm_pair_at(const unsigned (&addr)[D / 16], int imm_a, int imm_b,
                                                 const bf16x8 (&ba)[D / 16], const bf16x8 (&bb)[D / 16], f32x16 &ra, f32x16 &rb) {
    constexpr int NK = DC / 16, PF = 2;
    bf16x8 xa[PF + 1], xb[PF + 1];
#pragma unroll
    for (int i = 0; i < PF; i++) {
        xa[i] = *(lds_bf16x8_ptr)(uintptr_t)(addr[i] + imm_a);
        xb[i] = *(lds_bf16x8_ptr)(uintptr_t)(addr[i] + imm_b);
    }
#pragma unroll
    for (int kb = 0; kb < NK; kb++) {
        if (kb + PF < NK) {
            xa[(kb + PF) % (PF + 1)] = *(lds_bf16x8_ptr)(uintptr_t)(addr[kb + PF] + imm_a);
            xb[(kb + PF) % (PF + 1)] = *(lds_bf16x8_ptr)(uintptr_t)(addr[kb + PF] + imm_b);
        }
        __builtin_amdgcn_sched_barrier(0);
        ra = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[kb % (PF + 1)], ba[kb], ra, 0, 0, 0);
        rb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xb[kb % (PF + 1)], bb[kb], rb, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// one such chain
template <int D, int DC = D>
__device__ __forceinline__ void lds_gemm_chain_at(const unsigned (&addr)[D / 16], int imm, const bf16x8 (&b)[D / 16], f32x16 &r) {
    constexpr int NK = DC / 16, PF = 2;
    bf16x8 x[PF + 1];
#pragma unroll
    for (int i = 0; i < PF; i++) x[i] = *(lds_bf16x8_ptr)(uintptr_t)(addr[i] + imm);
#pragma unroll
    for (int kb = 0; kb < NK; kb++) {
        if (kb + PF < NK) x[(kb + PF) % (PF + 1)] = *(lds_bf16x8_ptr)(uintptr_t)(addr[kb + PF] + imm);
        __builtin_amdgcn_sched_barrier(0);
        r = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[kb % (PF + 1)], b[kb], r, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// acc[db] (32 x 32 tiles over the head dimension) += T^T-operand x B for NKB blocks of 16 tile rows: the A operands are transpose reads of
// the swizzled LDS tile T (rows = contraction index), the B operands b[kb] come from registers; reads run PF MFMAs ahead.
// addr[j][h]: byte address of the lane's transpose-read element for head-dimension block j, rows +0 (h = 0) / +8 (h = 1)
template <int D, int NKB, int DC = D>
__device__ __forceinline__ void lds_tr_gemm_at(const unsigned (&addr)[D / 32][2], int imm, const bf16x8 (&b)[NKB], f32x16 (&acc)[D / 32]) {
    constexpr int ND = DC / 32, N = NKB * ND, PF = 3;
    auto operand = [&](int i) {
        const int off = imm + (i / ND) * 16 * D * 2;
        union {
            struct { i16x4 a, b; } s;
            bf16x8 v;
        } u;
        u.s.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(uintptr_t)(addr[i % ND][0] + off));
        u.s.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(uintptr_t)(addr[i % ND][1] + off));
        return u.v;
    };
    bf16x8 a[PF + 1];
#pragma unroll
    for (int i = 0; i < PF && i < N; i++) a[i] = operand(i);
#pragma unroll
    for (int step = 0; step < N; step++) {
        if (step + PF < N) a[(step + PF) % (PF + 1)] = operand(step + PF);
        __builtin_amdgcn_sched_barrier(0);
        acc[step % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[step % (PF + 1)], b[step / ND], acc[step % ND], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Epilogue helper: a wave turns its 32 x D result tile, held in MFMA accumulator layout (lane (row l32, half hh),
// accumulator (db, 4 g + e) -> column 32 db + 8 g + 4 hh + e), into row-major order through a wave-private LDS area, so
// that global memory is written (and, for accumulators, read) in runs of whole rows instead of 8-16 bytes per row
// and instruction.  emit(row, col, v) receives 4 consecutive columns of one row; 32 / (D / 4) ... rows per step.
template <int D>
struct WaveStage {
    static constexpr int ROW_BYTES = D * 4 + 16;          // padded rows: the 128-bit column writes hit every bank once
    static constexpr int BYTES = 32 * ROW_BYTES + 128;    // + one float per row (per-row factor of the caller)
};

// Wave-uniform values pinned in scalar registers: kernel arguments used inside the epilogue loops are otherwise
// re-read from the argument segment in every iteration (a scalar load and a wait each time).
__device__ __forceinline__ int uniform32(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long long uniform64(long long x) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)x), hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(x >> 32));
    return (long long)(((unsigned long long)hi << 32) | lo);
}

template <int D, class Emit>
__device__ __forceinline__ void wave_tile_rowmajor(unsigned char *stage, int lane, const f32x16 (&acc)[D / 32], float mul,
                                                   Emit emit) {
    const int l32 = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int db = 0; db < D / 32; db++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = acc[db][4 * g + e] * mul;
            *(f32x4 *)(stage + l32 * WaveStage<D>::ROW_BYTES + (32 * db + 8 * g + 4 * hh) * 4) = v;
        }
    constexpr int LPR = D / 4;                // lanes per row
#pragma unroll
    for (int it = 0; it < 32 * LPR / 64; it++) {
        const int idx = it * 64 + lane, row = idx / LPR, c4 = idx % LPR;
        emit(row, 4 * c4, *(const f32x4 *)(stage + row * WaveStage<D>::ROW_BYTES + c4 * 16));
    }
}

struct NoHook {
    __device__ __forceinline__ void operator()(int) const {}
};

// The chain and the transpose GEMM for a wave that owns KW 32-key halves (dK/dV kernel) or KW 32-row blocks (forward): every operand
// read from LDS feeds one MFMA per half (b[k], r[k] / acc[k] belong to half k).  row: the lane's row of a swizzled tile, sw = the row's
// swizzle word XOR the lane's half.  hook(step) follows the MFMAs of operand `step`: independent arithmetic of the same wave
// written there issues while the matrix pipe works (a wave issues one instruction per ~5 clocks, an MFMA occupies the pipe for 32).
template <int D, int KW, int DC = D, class Hook = NoHook>
__device__ __forceinline__ void lds_gemm_chain_kw(const __bf16 *row, int sw, const bf16x8 (&b)[KW][D / 16], f32x16 (&r)[KW],
                                                  Hook hook = Hook()) {
    constexpr int NK = DC / 16, PF = 2;
    bf16x8 x[PF + 1];
#pragma unroll
    for (int i = 0; i < PF; i++) x[i] = *(const bf16x8 *)(row + (((2 * i) ^ sw) << 3));
#pragma unroll
    for (int kb = 0; kb < NK; kb++) {
        if (kb + PF < NK) x[(kb + PF) % (PF + 1)] = *(const bf16x8 *)(row + (((2 * (kb + PF)) ^ sw) << 3));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < KW; k++) r[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[kb % (PF + 1)], b[k][kb], r[k], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        hook(kb);
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <int D, int NKB, int KW, int DC = D, class Hook = NoHook>
__device__ __forceinline__ void lds_tr_gemm_kw(const __bf16 *T, int row0, int lane, const bf16x8 (&b)[KW][NKB],
                                               f32x16 (&acc)[KW][D / 32], Hook hook = Hook()) {
    constexpr int ND = DC / 32, N = NKB * ND, PF = 3;
    bf16x8 a[PF + 1];
#pragma unroll
    for (int i = 0; i < PF && i < N; i++) a[i] = lds_operand_tr_swz<D>(T, row0 + (i / ND) * 16, (i % ND) * 32, lane);
#pragma unroll
    for (int step = 0; step < N; step++) {
        if (step + PF < N)
            a[(step + PF) % (PF + 1)] = lds_operand_tr_swz<D>(T, row0 + ((step + PF) / ND) * 16, ((step + PF) % ND) * 32, lane);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < KW; k++)
            acc[k][step % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[step % (PF + 1)], b[k][step / ND], acc[k][step % ND], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        hook(step);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// keys per K / V tile of the forward and dQ kernels
template <int D, int RB = 1, int KS = 1>
struct FwdTile {
    // two row blocks per wave: S^T of 128 keys would be 128 registers; key shares: the tile is KS times as long (LDS)
    static constexpr int BN = KS > 1 ? (D == 128 && KS == 4 ? 32 : 64) : (D == 64 && RB == 1) ? 128 : 64;
};

// Key shares of the forward and dQ kernels (KS waves per 32-row group, each with its own keys): at the end every wave collects CW of
// the D result columns from the KS partial results, which lie in LDS as they lie in registers (4 KB per 32 x 32 tile).
template <int D, int KS>
struct KeyShares {
    static constexpr int CW = D / KS > 32 ? D / KS : 32;
    static constexpr int PART_OFF = 8 * 64 * 4;                                    // after the forward's references and sums
    static constexpr int BYTES = KS > 1 ? PART_OFF + 8 * (D / 32) * 4096 : 0;
};
template <int D, int KS>
__device__ __forceinline__ void collect_shares(unsigned char *smem, int w, int ks, int lane, const f32x16 (&acc)[D / 32], float mul,
                                               f32x16 (&own)[KeyShares<D, KS>::CW / 32]) {
    constexpr int ND = D / 32, NC = KeyShares<D, KS>::CW / 32;
    float *const parts = (float *)(smem + KeyShares<D, KS>::PART_OFF);
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) own[j][r] = 0.f;
#pragma unroll
    for (int i = 0; i < ND; i++) {
        if (i / NC == ks) {   // wave-uniform
#pragma unroll
            for (int r = 0; r < 16; r++) own[i % NC][r] = acc[i][r] * mul;
        } else {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = acc[i][4 * g + e] * mul;
                *(f32x4 *)(parts + (((w * ND + i) * 4 + g) * 64 + lane) * 4) = v;
            }
        }
    }
    __syncthreads();
    if (ks * NC >= ND) return;
#pragma unroll
    for (int k = 1; k < KS; k++) {
        const int other = w - ks + ((ks + k) & (KS - 1));
#pragma unroll
        for (int j = 0; j < NC; j++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const f32x4 v = *(const f32x4 *)(parts + (((other * ND + ks * NC + j) * 4 + g) * 64 + lane) * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) own[j][4 * g + e] += v[e];
            }
    }
}

// ------------------------------------------------------------------------------ forward, bf16
// RB = 32-row blocks per wave.  With two (head dim 64) every K / V operand read from LDS feeds two MFMAs and a tile of
// 64 keys serves 512 query rows: half the LDS reads and half the tile transfers per MFMA.
// KS = waves that share a 32-row group: each takes its own BN keys of every tile of KS * BN keys, and their partial (reference, row
// sum, O) are merged through LDS at the end.  For launches with too few query rows to give every CU a block (see FwdPlan).
// NW = waves: eight (one block per CU, two waves per SIMD), or four with 64-key tiles (FourWaves), where several blocks share a CU.
template <int D, int RB, int KS, bool PAD, int NW = 8, int BN = FwdTile<D, RB, KS>::BN, int DC = D>
__device__ __forceinline__ void fwd_bf16_body(const FwdParams &p) {
    const int cols = PAD ? p.cols : D;
    constexpr int RG = NW / KS, BM = 32 * RB * RG;   // the NW waves of the block share every K / V tile
    constexpr int NB = BN / 32, BNT = BN * KS;       // BN keys per wave, BNT per tile
    constexpr int CPR = D / 8;   // 16-byte chunks per row
    constexpr int RPI = 64 / CPR;            // rows filled by one wave-wide 16-byte-per-lane LDS-direct load (1 KB)
    constexpr int NI = BNT / (RPI * NW);      // such loads per wave, per tensor and per tile
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // two K tiles, two V tiles,
    constexpr int TILE = BNT * D;            // rows unpadded, 16-byte chunks XOR-swizzled (lds_swz)
    constexpr int BUF_ELEMS = 2 * TILE;

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = w / KS, ks = w % KS;      // row group and key share of the wave
    const bool causal = p.flags & LTR_CAUSAL;

    // block -> (batch, kv head, q head of the group, q tile); late (heavier under a causal mask) q tiles first
    const BlockItem item = block_item(p.map, p.B * p.Hkv);
    const int pair = item.pair, rep = item.sub, slot = item.item;
    if (pair >= p.B * p.Hkv) return;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv, h = hkv * p.n_rep + rep;
    // A slot is one q tile (late, heavier tiles first) or, when the host paired them, a late tile and its early
    // counterpart: under a causal mask every block then has the same amount of work.
    const bool paired = p.n_slots != p.n_qtiles;
    // every other block (of an XCD) takes the early tile first: the blocks of a round then change tiles at different times
    const bool two = paired && slot < p.n_qtiles - 1 - slot, early_first = two && (item.order & 1);
#pragma nounroll
    for (int part = 0; part < 2; part++) {
    const int qt = (part == 0) != early_first ? p.n_qtiles - 1 - slot : slot;
    if (part == 1 && !two) break;
    if (part == 1) __syncthreads();   // the first tile's epilogue used the LDS buffers as staging areas
    // the lane index is made opaque per tile: everything derived from it (LDS addresses of the tile loop ...) is then
    // computed inside the tile's own scope instead of being hoisted out of this loop and kept alive across the epilogue
    int lane_of_part = threadIdx.x & 63;
    asm volatile("" : "+v"(lane_of_part));
    const int lane = lane_of_part, l32 = lane & 31, hh = lane >> 5;

    const int row0 = qt * BM;
    int my_row[RB], my_pos[RB];   // row block rb of row group rg: rows row0 + 32 * (RB * rg + rb) ..
    bool row_ok[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        my_row[rb] = row0 + (rg * RB + rb) * 32 + l32;
        row_ok[rb] = my_row[rb] < p.Sq;
        my_pos[rb] = q_position(my_row[rb], p.q_split, p.q_pos0[0], p.q_pos0[1]);
    }
    int blk_lo, blk_hi, w_lo, w_hi;
    q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);
    {
        int wr0 = row0 + rg * 32 * RB, wr1 = min(wr0 + 32 * RB, p.Sq) - 1;
        if (wr1 >= wr0) q_pos_range(wr0, wr1, p.q_split, p.q_pos0[0], p.q_pos0[1], w_lo, w_hi);
        else { w_lo = 0x7fffffff; w_hi = -0x7fffffff; }  // wave has no valid row
    }

    // Q operand (B of S^T = K Q^T): lane (query l32, half hh) holds d = 16*kb + 8*hh .. +7
    bf16x8 qreg[RB][D / 16];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        const __bf16 *qp = (const __bf16 *)p.q + b * p.qs[0] + (long long)my_row[rb] * p.qs[1] + h * p.qs[2];
#pragma unroll
        for (int kb = 0; kb < DC / 16; kb++) {
            uint4 x = make_uint4(0, 0, 0, 0);
            if (row_ok[rb] && (!PAD || kb * 16 + 8 * hh < cols)) x = *(const uint4 *)(qp + kb * 16 + 8 * hh);
            qreg[rb][kb] = as_bf16x8(x);
        }
        // fused RoPE prologue: q arrives un-rotated and is rotated here, in the registers that hold it as the MFMA operand,
        // by the angles of the row's global position; the rotated row can be stored for the backward
        if ((p.flags & LTR_ROPE_Q) && row_ok[rb]) {
            const float *fr = p.rope + (long long)(my_pos[rb] - p.rope_pos0) * cols + 8 * hh;
            __bf16 *qr = p.q_rot && ks == 0 ? (__bf16 *)p.q_rot + b * p.qrs[0] + (long long)my_row[rb] * p.qrs[1] + h * p.qrs[2] + 8 * hh : nullptr;
#pragma unroll
            for (int kb = 0; kb < DC / 16; kb++) {
                if (PAD && kb * 16 + 8 * hh >= cols) continue;
                qreg[rb][kb] = rope_rotate8(qreg[rb][kb], *(const f32x4 *)(fr + 16 * kb), *(const f32x4 *)(fr + 16 * kb + 4));
                if (qr) *(bf16x8 *)(qr + 16 * kb) = qreg[rb][kb];
            }
        }
    }

    f32x16 zero16;
#pragma unroll
    for (int r = 0; r < 16; r++) zero16[r] = 0.f;
    f32x16 oacc[RB][D / 32];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int i = 0; i < D / 32; i++) oacc[rb][i] = zero16;
    // Online softmax state of this lane's query row.  mc is the reference point of the exponent (exp2 domain:
    // m * scale * log2(e)).  It does not follow the running max: P = exp2(s*c2 - mc) keeps its relative precision
    // whatever mc is, l and O accumulate in fp32 and LSE = mc*ln2 + log(l) is unaffected, so mc only has to keep
    // the row sum inside [TINY, BIG] where neither overflow nor flushed small terms matter.  That is checked on
    // the row sum of each tile (two compares), and the row max is only computed on the rare tile that fails the
    // check: the common tile has no max reduction and no rescale of the O accumulator.
    float mc[RB], l_run[RB];  // l_run: this lane's partial row sum (its half of the keys of every tile)
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        mc[rb] = 0.f;
        l_run[rb] = 0.f;
    }
    const float c2 = p.scale * LTR_LOG2E;
    constexpr float BIG = 1.152921504606846976e18f, TINY = 8.673617379884035472e-19f;   // 2^60, 2^-60

    // tile iterator over (chunk, key tile)
    // The fields of the chunk being loaded live in scalar registers and are re-read from the argument
    // table only when the chunk changes (a scalar load per tile would share the LDS wait counter).
    int c = -1, t = 0, nt = 0;
    int ld_sk = 0, ld_pos0 = 0;
    const __bf16 *ld_kb = nullptr, *ld_vb = nullptr;
    auto settle = [&]() {
        while (c < p.n_chunks && t >= nt) {
            c++;
            t = 0;
            if (c < p.n_chunks) {
                ld_sk = p.chunk[c].sk;
                ld_pos0 = p.chunk[c].pos0;
                ld_kb = (const __bf16 *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
                ld_vb = (const __bf16 *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
                const int nvis = causal ? max(0, min(ld_sk, blk_hi - ld_pos0 + 1)) : ld_sk;
                nt = (nvis + BNT - 1) / BNT;
            }
        }
    };
    settle();

    // Tiles go from global memory straight into LDS (global_load_lds, 16 bytes per lane, no staging
    // registers): wave w fills rows RPI*(NI*w + i) .. of the tile with its i-th load, lane l the chunk
    // position l % CPR of row l / CPR, fetching the logical chunk that the swizzle places there.  Rows past
    // the end of a chunk are fetched from its last row; their keys are masked.
    const int st_row = lane / CPR, st_pc = lane % CPR;
    int nx_sk = 0, nx_pos0 = 0, nx_key0 = 0;   // the tile in flight: becomes the tile computed next
    // transfer j of the tile in flight (ti, into buffer buf): j < NI are this wave's K rows, the rest its V rows
    auto gload_one = [&](int j, int ti, int buf) {
        const int i = j % NI;
        const unsigned dst = lds_address(smem) + buf * TILE * 2 + (j / NI) * BUF_ELEMS * 2 + RPI * (NI * w + i) * D * 2;
        const int row = RPI * (NI * w + i) + st_row;
        const int key = min(ti * BNT + row, ld_sk - 1);
        const int chunk = st_pc ^ lds_swz<D>(row);
        const __bf16 *src = j < NI ? ld_kb + (long long)(key * (int)p.ks[1] + chunk * 8)
                                   : ld_vb + (long long)(key * (int)p.vs[1] + chunk * 8);
        if (!PAD || chunk * 8 < cols) global_to_lds_b128(src, dst);
    };
    auto gload_begin = [&](int ti) {   // scalar state of the tile whose transfers are issued next
        nx_sk = ld_sk;
        nx_pos0 = ld_pos0;
        nx_key0 = ti * BNT;
    };

    // Double-buffered LDS, one barrier per tile: tile t+1 streams into the other buffer (whose readers all
    // passed the previous barrier) while tile t is computed; the barrier also waits for those loads.
    bool have = c < p.n_chunks;
    // Merging an empty partial result leaves (O, LSE) as they are: a block that sees no key of this launch's chunks (the
    // early rows of a causal ring step) skips the read-modify-write of its rows altogether.
    if (!have && (p.flags & LTR_MERGE)) continue;
    if constexpr (PAD) clear_lds<2 * BUF_ELEMS * 2>(smem);
    if (have) {
        gload_begin(t);
#pragma unroll
        for (int j = 0; j < 2 * NI; j++) gload_one(j, t, 0);
    }
    tile_barrier();
    // One tile; the loop below is unrolled over the two LDS buffers so that every LDS address is a loop-invariant
    // per-lane register plus an immediate offset (no address arithmetic between the MFMAs).  The registers are spelled out and opaque:
    // the K tiles and the V tiles each lie in one window of 64 KB, which the offsets reach, and 16 registers address all of it.
    static_assert(2 * TILE * 2 <= 65536, "offsets of an LDS read end at 65535");
    unsigned ka[D / 16], va[D / 32][2];
    if constexpr (RB == 1) {
        const unsigned lds0 = lds_address(smem) + (KS > 1 ? ks * BN * D * 2 : 0);
        const int sw = lds_swz<D>(l32) ^ hh;        // rows l32 + 32 n share the swizzle word of row l32
#pragma unroll
        for (int kb = 0; kb < DC / 16; kb++) {
            ka[kb] = lds0 + ((l32 * D + (((2 * kb) ^ sw) << 3)) << 1);
            asm volatile("" : "+v"(ka[kb]));
        }
        const int li = lane & 15, g = lane >> 4;
#pragma unroll
        for (int i = 0; i < DC / 32; i++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int col = i * 32 + ((g & 1) << 4) + ((li & 3) << 2), row = 4 * (g >> 1) + (li >> 2) + 8 * e;
                va[i][e] = lds0 + 2 * TILE * 2 + ((lds_swz_off<D>(row, col >> 3) + (col & 7)) << 1);
                asm volatile("" : "+v"(va[i][e]));
            }
    }
    auto tile_step = [&](auto par_tag) {
        constexpr int par = decltype(par_tag)::value;
        const int sk = nx_sk, pos0 = nx_pos0, key0 = nx_key0 + (KS > 1 ? ks * BN : 0);
        constexpr int at = par * TILE * 2;                                                        // RB == 1: offset of ka, va
        const __bf16 *const Ks = (const __bf16 *)smem + par * TILE, *const Vs = Ks + BUF_ELEMS;   // RB == 2
        t++;
        settle();
        const bool have_next = c < p.n_chunks;
        // All transfers of the next tile are issued here, right after the barrier: the memory pipe takes them
        // at 64 bytes per clock and a wave waits at the issue port meanwhile; issued between MFMAs instead
        // (measured) the same waits cost more, because they then stall waves that are feeding the matrix pipe.
        if (have_next) {
            gload_begin(t);
#pragma unroll
            for (int j = 0; j < 2 * NI; j++) gload_one(j, t, par ^ 1);
        }

        // A wave whose 32 rows all precede the tile's first key (upper part of a diagonal tile, rows past the end) has
        // nothing to add: it only takes part in the transfers and the barrier.
        if ((!causal || pos0 + key0 <= w_hi) && (KS == 1 || key0 < sk)) {
        // S^T of the two 32-key blocks of the tile.  The wave raises its priority while it issues MFMAs: the
        // other wave of the SIMD then fills the gaps with its softmax arithmetic instead of delaying them.
        __builtin_amdgcn_s_setprio(1);
        f32x16 s[NB][RB];
        if constexpr (RB == 1) {
#pragma unroll
            for (int nb = 0; nb + 1 < NB; nb += 2) {
                s[nb][0] = zero16;
                s[nb + 1][0] = zero16;
                lds_gemm_pair_at<D, DC>(ka, at + nb * 32 * D * 2, at + (nb + 1) * 32 * D * 2, qreg[0], qreg[0], s[nb][0], s[nb + 1][0]);
            }
            if constexpr (NB == 1) {
                s[0][0] = zero16;
                lds_gemm_chain_at<D, DC>(ka, at, qreg[0], s[0][0]);
            }
        } else {
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
#pragma unroll
                for (int rb = 0; rb < RB; rb++) s[nb][rb] = zero16;
                lds_gemm_chain_kw<D, RB>(Ks + (nb * 32 + l32) * D, lds_swz<D>(nb * 32 + l32) ^ hh, qreg, s[nb]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        // mask fix-up (tail of the chunk, diagonal tiles): wave-uniform branch touching S only
        const bool need_mask = (key0 + BN > sk) || (causal && (pos0 + key0 + BN - 1 > w_lo));
        if (need_mask) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int nb = 0; nb < NB; nb++) {
                    const unsigned bits = visible_bits(causal, my_pos[rb], pos0, sk, key0 + nb * 32 + 4 * hh);
#pragma unroll
                    for (int r = 0; r < 16; r++) s[nb][rb][r] = visible_score(bits, 8 * (r / 4) + r % 4, s[nb][rb][r]);
                }
        }
        // t = s*c2 - reference (exp2 domain), P = exp2(t) rounded to bf16, row sum of the rounded P (what PV uses)
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
#pragma unroll
                for (int r = 0; r < 16; r++) s[nb][rb][r] = s[nb][rb][r] * c2 - mc[rb];
        PackedTile pt[RB][NB];
        bf16x2 ones;
        ones[0] = (__bf16)1.0f;
        ones[1] = (__bf16)1.0f;
        float l_tile[RB];
        auto exponentials = [&](int rb) {
            l_tile[rb] = 0.f;
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    bf16x2 pr;
                    pr[0] = (__bf16)__builtin_amdgcn_exp2f(s[nb][rb][2 * j]);
                    pr[1] = (__bf16)__builtin_amdgcn_exp2f(s[nb][rb][2 * j + 1]);
                    l_tile[rb] = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, l_tile[rb], false);
                    pt[rb][nb].u[j] = __builtin_bit_cast(unsigned, pr);
                }
        };
        bool out_of_range = false;
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            exponentials(rb);
            // in range: the tile's sum did not overflow and the row has a healthy sum by now (a lane sees half of the
            // row's keys, so its partial sum can lag behind the row's: that only costs a visit of the branch below)
            out_of_range = out_of_range || !(l_tile[rb] < BIG) || !(l_run[rb] + l_tile[rb] >= TINY);
        }
        if (__builtin_amdgcn_ballot_w64(out_of_range) != 0) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                float mx = -INFINITY;
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
#pragma unroll
                    for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[nb][rb][r]);
                mx = xhalf_max(mx);                       // row max of t over the tile (-inf: no visible key)
                const float l_row = xhalf_sum(l_run[rb]), lt_row = xhalf_sum(l_tile[rb]);   // whole-row sums: both halves agree
                const bool row_bad = !(lt_row < BIG) || !(l_row + lt_row >= TINY);
                // New reference for a row that is out of range: the larger of the tile's max and the magnitude of the
                // history (log2 of its sum), so that neither overflows after the move; with a history never below -126, so
                // that the factor applied to it stays finite.  Rows that are in range, and rows that have seen no key at
                // all, keep theirs.
                const float hist = l_row > 0.f ? __log2f(l_row) : -INFINITY;
                const float target = fmaxf(mx, hist);
                const float shift = (row_bad && target > -INFINITY) ? (l_row > 0.f ? fmaxf(target, -126.f) : target) : 0.f;
                const float alpha = l_row > 0.f ? __builtin_amdgcn_exp2f(-shift) : 1.f;
                l_run[rb] *= alpha;
#pragma unroll
                for (int i = 0; i < DC / 32; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) oacc[rb][i][r] *= alpha;
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
#pragma unroll
                    for (int r = 0; r < 16; r++) s[nb][rb][r] -= shift;
                mc[rb] += shift;
                exponentials(rb);
            }
        }
#pragma unroll
        for (int rb = 0; rb < RB; rb++) l_run[rb] += l_tile[rb];
        __builtin_amdgcn_s_setprio(1);
        if constexpr (RB == 1) {
            bf16x8 pb[2 * NB];
#pragma unroll
            for (int kb = 0; kb < 2 * NB; kb++) pb[kb] = operand_of(pt[0][kb >> 1], kb & 1);
            lds_tr_gemm_at<D, 2 * NB, DC>(va, at, pb, oacc[0]);   // 16 keys per MFMA
        } else {
            bf16x8 pb[RB][2 * NB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int kb = 0; kb < 2 * NB; kb++) pb[rb][kb] = operand_of(pt[rb][kb >> 1], kb & 1);
            lds_tr_gemm_kw<D, 2 * NB, RB>(Vs, 0, lane, pb, oacc);   // 16 keys per MFMA, one V operand read for both row blocks
        }
        __builtin_amdgcn_s_setprio(0);
        }
        tile_barrier();
        have = have_next;
    };
    while (have) {
        tile_step(std::integral_constant<int, 0>{});
        if (!have) break;
        tile_step(std::integral_constant<int, 1>{});
    }

    // The KS partial results of a row group: the waves agree on a reference (the largest share's log2 of its own sum), scale their O to
    // it, and each collects CW of the D columns from the others.  The tile buffers are no longer read: the last barrier is
    // behind us.
    constexpr int CW = KeyShares<D, KS>::CW;   // columns a wave writes, from column col0 on
    const int col0 = KS > 1 ? ks * CW : 0;
    f32x16 own[CW / 32];                       // KS > 1: those columns of O
    float l_shared = 0.f, lse_before = 0.f;
    if constexpr (KS > 1) {
        static_assert(RB == 1, "key shares are built for one row block per wave");
        if ((p.flags & LTR_MERGE) && row_ok[0]) lse_before = p.lse[((long long)b * p.Hq + h) * p.Sq + my_row[0]];   // before any wave writes it
        float *const ml = (float *)smem + w * 64;   // [wave][32 references | 32 sums]
        const float l_own = xhalf_sum(l_run[0]), ref_own = l_own > 0.f ? mc[0] + __log2f(l_own) : -INFINITY;
        if (hh == 0) ml[l32] = ref_own;
        __syncthreads();
        float ref = -INFINITY;
#pragma unroll
        for (int k = 0; k < KS; k++) ref = fmaxf(ref, ml[(k - ks) * 64 + l32]);
        const float f_own = l_own > 0.f ? __builtin_amdgcn_exp2f(mc[0] - ref) : 0.f;
        if (hh == 0) ml[32 + l32] = l_own * f_own;
        collect_shares<D, KS>(smem, w, ks, lane, oacc[0], f_own, own);
#pragma unroll
        for (int k = 0; k < KS; k++) l_shared += ml[32 + (k - ks) * 64 + l32];
        mc[0] = ref == -INFINITY ? 0.f : ref;
        __syncthreads();                            // the partials are read: their memory becomes the staging areas
        if (col0 >= D) continue;                    // more shares than 32-column groups: nothing left to write
    }
    // epilogue: normalise, optional merge with the partial result already in (o, lse); one row block after the other
    // through the same staging area
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
    const float l_tot = KS > 1 ? l_shared : xhalf_sum(l_run[rb]);
    float lse_new = (l_tot > 0.f) ? mc[rb] * LTR_LN2 + logf(l_tot) : -INFINITY;
    float w_cur = (l_tot > 0.f) ? 1.f / l_tot : 0.f;
    float w_old = 0.f;
    float *lse_p = p.lse + ((long long)b * p.Hq + h) * p.Sq + my_row[rb];
    if ((p.flags & LTR_MERGE) && row_ok[rb]) {
        const float lse_old = KS > 1 ? lse_before : *lse_p;
        const float mxl = fmaxf(lse_old, lse_new);
        if (mxl == -INFINITY) {
            w_cur = 0.f;
        } else {
            const float e_old = expf(lse_old - mxl), e_new = expf(lse_new - mxl);
            const float tot = e_old + e_new;
            w_old = e_old / tot;
            w_cur *= e_new / tot;
            lse_new = mxl + logf(tot);
        }
    }
    if (row_ok[rb] && hh == 0 && col0 == 0) *lse_p = lse_new;
    // O through the wave's LDS staging area (the tiles are no longer read: the last barrier is behind us)
    unsigned char *stage = smem + w * WaveStage<CW>::BYTES;
    float *row_w_old = (float *)(stage + 32 * WaveStage<CW>::ROW_BYTES);
    if (hh == 0) row_w_old[l32] = w_old;
    constexpr int LPR = CW / 4, ROWS_PER_IT = 64 / LPR;      // see wave_tile_rowmajor
    const int Sq_u = uniform32(p.Sq), wave_row0 = uniform32(row0 + (rg * RB + rb) * 32);
    const bool merge = uniform32(p.flags & LTR_MERGE) != 0, o_f32 = uniform32(p.o_f32) != 0;
    const long long os1 = uniform64(p.os[1]);
    const long long off0 = uniform64(b * p.os[0] + h * p.os[2] + col0) + (wave_row0 + lane / LPR) * os1 + 4 * (lane % LPR);
    // merging: all reads of the earlier partial result first (independent loads in flight together), then the writes
    constexpr int NIT = 32 / ROWS_PER_IT;
    f32x4 old[NIT];
#pragma unroll
    for (int it = 0; it < NIT; it++) {
        old[it] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (merge && wave_row0 + it * ROWS_PER_IT + lane / LPR < Sq_u && (!PAD || col0 + 4 * (lane % LPR) < cols)) {
            if (o_f32) {
                old[it] = *(const f32x4 *)((const float *)p.o + off0 + it * ROWS_PER_IT * os1);
            } else {
                const bf16x4 x = *(const bf16x4 *)((const __bf16 *)p.o + off0 + it * ROWS_PER_IT * os1);
#pragma unroll
                for (int e = 0; e < 4; e++) old[it][e] = (float)x[e];
            }
        }
    }
    int it = 0;
    auto &result = [&]() -> f32x16(&)[CW / 32] {
        if constexpr (KS > 1) return own;
        else return oacc[rb];
    }();
    if (o_f32) {
        float *op = (float *)p.o + off0;
        wave_tile_rowmajor<CW>(stage, lane, result, w_cur, [&](int row, int col, f32x4 val) {
            if (wave_row0 + row < Sq_u && (!PAD || col0 + col < cols)) {
                if (merge) {
                    const float wo = row_w_old[row];
#pragma unroll
                    for (int e = 0; e < 4; e++) val[e] += old[it][e] * wo;
                }
                *(f32x4 *)op = val;
            }
            op += ROWS_PER_IT * os1;
            it++;
        });
    } else {
        __bf16 *op = (__bf16 *)p.o + off0;
        wave_tile_rowmajor<CW>(stage, lane, result, w_cur, [&](int row, int col, f32x4 val) {
            if (wave_row0 + row < Sq_u && (!PAD || col0 + col < cols)) {
                if (merge) {
                    const float wo = row_w_old[row];
#pragma unroll
                    for (int e = 0; e < 4; e++) val[e] += old[it][e] * wo;
                }
                bf16x4 ob;
#pragma unroll
                for (int e = 0; e < 4; e++) ob[e] = (__bf16)val[e];
                *(bf16x4 *)op = ob;
            }
            op += ROWS_PER_IT * os1;
            it++;
        });
    }
    }   // row block
    }   // part
}

// Blocks of four waves and 128 rows: three share a CU at head dim 64 (168 registers, 35 KB of LDS), two at 128.  A block's start (its Q
// rows and first tile from memory), its barriers and its O stores, 7 - 9 us that an eight-wave block alone on its CU waits for, then
// run under the other blocks' arithmetic; 128-row blocks also leave less of a diagonal tile masked and a shorter tail.  The price is a K / V
// tile per four waves.  Kernel us, best of the eight-wave blocks -> this one, forward / dQ, causal:
//   16 x 12 heads D=64 S=1024   56 / 65 -> 43 / 58       7 x 32 heads D=64 S=2214  210 / 273 -> 185 / 251
//   4 x 16 heads D=128 S=1024   35 / 46 -> 32 / 42      13 x 16 heads D=128 S=1800  241 / 317 -> 229 / 308
//   4 x 32 heads D=128 S=8192 2046 / 2844 -> 2173 / 2925 (long blocks: the tile traffic shows)
// Bound at head dim 64 by vector instructions: 13.6 / 10.2 per MFMA in the first of these launches, the vector pipe active 59 / 52 % and the
// matrix pipe 30 / 36 % of a SIMD's time.
template <int D>
struct FourWaves {
    static constexpr int BN = 64, PER_CU = D == 64 ? 3 : 2;
    static constexpr int TILES = 2 * 2 * BN * D * 2, LDS = TILES > 4 * WaveStage<D>::BYTES ? TILES : 4 * WaveStage<D>::BYTES;
    static_assert(PER_CU * LDS <= 160 * 1024, "LDS of one CU");
};
template <int D>
__global__ __launch_bounds__(256, FourWaves<D>::PER_CU) void fwd_bf16_w4_kernel(const FwdParams p) {
    fwd_bf16_body<D, 1, 1, false, 4, FourWaves<D>::BN>(p);
}
template <int D, int RB>
__global__ __launch_bounds__(512) void fwd_bf16_kernel(const FwdParams p) {
    fwd_bf16_body<D, RB, 1, false>(p);
}
template <int D, int KS>
__global__ __launch_bounds__(512) void fwd_bf16_shares_kernel(const FwdParams p) {
    fwd_bf16_body<D, 1, KS, false>(p);
}
template <int D, int KS>   // head dims below D
__global__ __launch_bounds__(512) void fwd_bf16_pad_kernel(const FwdParams p) {
    fwd_bf16_body<D, 1, KS, true>(p);
}
template <int D, int KS>
__global__ __launch_bounds__(512) void fwd_bf16_pad_kernel(const Columns96<FwdParams> p) {
    static_assert(D == 128);
    fwd_bf16_body<D, 1, KS, true, 8, FwdTile<D, 1, KS>::BN, 96>(p);
}

// ------------------------------------------------------------------------------ forward, fp32
// One lane per query row, 64 rows per block, K/V tiles of 32 keys broadcast from LDS.
template <int D>
__global__ __launch_bounds__(64) void fwd_f32_kernel(const FwdParams p) {
    constexpr int BN = 32;
    __shared__ __attribute__((aligned(16))) float Ks[BN * D];
    __shared__ __attribute__((aligned(16))) float Vs[BN * D];
    const int tid = threadIdx.x;
    const bool causal = p.flags & LTR_CAUSAL;
    int idx = blockIdx.x;
    const int qt = p.n_qtiles - 1 - idx / (p.B * p.Hq);
    const int bh = idx % (p.B * p.Hq);
    const int b = bh / p.Hq, h = bh % p.Hq, hkv = h / p.n_rep;
    const int row0 = qt * 64, my_row = row0 + tid;
    const bool row_ok = my_row < p.Sq;
    const int my_pos = q_position(my_row, p.q_split, p.q_pos0[0], p.q_pos0[1]);
    int blk_lo, blk_hi;
    q_pos_range(row0, min(row0 + 64, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);

    float q[D], o[D];
    {
        const float *qp = (const float *)p.q + b * p.qs[0] + (long long)my_row * p.qs[1] + h * p.qs[2];
#pragma unroll
        for (int d = 0; d < D; d++) {
            q[d] = row_ok ? qp[d] : 0.f;
            o[d] = 0.f;
        }
    }
    float m_run = -INFINITY, l_run = 0.f;
    for (int c = 0; c < p.n_chunks; c++) {
        const int sk = p.chunk[c].sk, pos0 = p.chunk[c].pos0;
        const int nvis = causal ? max(0, min(sk, blk_hi - pos0 + 1)) : sk;
        const float *kp = (const float *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
        const float *vp = (const float *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
        for (int key0 = 0; key0 < nvis; key0 += BN) {
            __syncthreads();
            for (int i = tid; i < BN * D / 4; i += 64) {
                int key = key0 + i / (D / 4), dc = i % (D / 4);
                f32x4 kv = {0.f, 0.f, 0.f, 0.f}, vv = {0.f, 0.f, 0.f, 0.f};
                if (key < sk) {
                    kv = *(const f32x4 *)(kp + (long long)key * p.ks[1] + dc * 4);
                    vv = *(const f32x4 *)(vp + (long long)key * p.vs[1] + dc * 4);
                }
                *(f32x4 *)(Ks + i * 4) = kv;
                *(f32x4 *)(Vs + i * 4) = vv;
            }
            __syncthreads();
            float s[BN];
            float mx = -INFINITY;
#pragma unroll
            for (int j = 0; j < BN; j++) {
                float acc = 0.f;
#pragma unroll
                for (int d = 0; d < D; d++) acc = fmaf(q[d], Ks[j * D + d], acc);
                acc *= p.scale;
                const int key = key0 + j;
                const bool vis = key < sk && (!causal || pos0 + key <= my_pos);
                s[j] = vis ? acc : -INFINITY;
                mx = fmaxf(mx, s[j]);
            }
            const float m_new = fmaxf(m_run, mx);
            const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
            const float alpha = expf(m_run - m_use);
            l_run *= alpha;
#pragma unroll
            for (int d = 0; d < D; d++) o[d] *= alpha;
#pragma unroll
            for (int j = 0; j < BN; j++) {
                const float pj = expf(s[j] - m_use);
                l_run += pj;
#pragma unroll
                for (int d = 0; d < D; d++) o[d] = fmaf(pj, Vs[j * D + d], o[d]);
            }
            m_run = m_new;
        }
    }
    if (!row_ok) return;
    float lse_new = (l_run > 0.f) ? m_run + logf(l_run) : -INFINITY;
    float w_cur = (l_run > 0.f) ? 1.f / l_run : 0.f, w_old = 0.f;
    float *lse_p = p.lse + ((long long)b * p.Hq + h) * p.Sq + my_row;
    if (p.flags & LTR_MERGE) {
        const float lse_old = *lse_p;
        const float mxl = fmaxf(lse_old, lse_new);
        if (mxl == -INFINITY) {
            w_cur = 0.f;
        } else {
            const float e_old = expf(lse_old - mxl), e_new = expf(lse_new - mxl);
            const float tot = e_old + e_new;
            w_old = e_old / tot;
            w_cur *= e_new / tot;
            lse_new = mxl + logf(tot);
        }
    }
    *lse_p = lse_new;
    float *op = (float *)p.o + b * p.os[0] + (long long)my_row * p.os[1] + h * p.os[2];
#pragma unroll
    for (int d = 0; d < D; d++) {
        float val = o[d] * w_cur;
        if (p.flags & LTR_MERGE) val += op[d] * w_old;
        op[d] = val;
    }
}

// ------------------------------------------------------------------------------ forward, fp32 on the matrix pipe
// v_mfma_f32_32x32x2_f32 (lane l, i = l % 32, h = l / 32: A[i][h], B[h][i], C as for the bf16 shape): fp32 operands and
// fp32 accumulation, so the 1e-4 cases run on the matrix pipe at full precision.  A block has 4 waves; a wave owns 32 query
// rows (a lane = one query, as in the bf16 kernel) and one of KS interleaved shares of the keys: the RG = 4 / KS waves with
// different rows share every K / V tile, the KS waves with the same rows take the sub-tiles ks, ks + KS, ... of 32 keys and
// their partial (m, l, O) are merged at the end.  KS > 1 is for launches with too few query rows to fill the device (the
// reference's acceptance shapes).  Both contractions pick their own order of the contraction index so that no operand moves:
//   S^T = K Q^T   step 4g + j contracts d = 8g + 4h + j: the K operand of four steps is one 128-bit LDS read, Q stays in
//                 registers in that order;
//   O^T += V^T P^T  step r contracts the key of accumulator register r (8 (r / 4) + 4h + r % 4): P^T is used where it is.
// K / V tiles of 32 * KS keys go global -> LDS directly, double buffered, 16-byte chunks XOR-swizzled (f32_swz) so that the
// 128-bit K reads (16 rows, same chunk) and the 32-bit V reads (one row per half-wave, rows 4 apart) touch every bank once.
__device__ __forceinline__ int f32_swz(int row) {   // bits 2 and 3 of the row swapped: rows 4 apart land 32 banks apart
    return (row & 3) | (((row >> 2) & 1) << 3) | (((row >> 3) & 1) << 2);
}

template <int D, int KS>
struct F32Mfma {
    static constexpr int NW = 4, RG = NW / KS;          // waves; row groups of 32 rows
    static constexpr int BM = 32 * RG, BN = 32 * KS;    // rows per block, keys per step
    static constexpr int TILE = BN * D;                 // floats per K (or V) tile
    static constexpr int BUF_BYTES = 2 * TILE * 4;      // {K tile, V tile}
    static constexpr int ML_OFF = 0, ML_BYTES = NW * 64 * 4;                        // per wave: m[32], l[32]
    static constexpr int PART_OFF = ML_BYTES, PART_BYTES = (D / 32) * 16 * 64 * 4;  // one wave's O^T accumulators, lane-major
    static constexpr int MERGE_BYTES = PART_OFF + (KS - 1) * RG * PART_BYTES;
    static constexpr int STAGE_OFF = MERGE_BYTES;       // row-major staging of the RG writing waves, after the merge area
    static constexpr int EPI_BYTES = STAGE_OFF + RG * WaveStage<D>::BYTES;
    static constexpr int LDS = 2 * BUF_BYTES > EPI_BYTES ? 2 * BUF_BYTES : EPI_BYTES;
    static_assert(LDS <= 160 * 1024, "LDS of one CU");
};

template <int D, int KS>
__device__ __forceinline__ void fwd_f32_body(const FwdParams &p) {
    using L = F32Mfma<D, KS>;
    constexpr int NW = L::NW, RG = L::RG, BM = L::BM, BN = L::BN, TILE = L::TILE;
    constexpr int CPR = D / 4;               // 16-byte chunks per row
    constexpr int RPI = 64 / CPR;            // rows filled by one wave-wide LDS-direct load (1 KB)
    constexpr int NI = BN / (RPI * NW);      // such loads per wave, per tensor and per step
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = w / KS, ks = w % KS;
    const bool causal = p.flags & LTR_CAUSAL;
    int idx = blockIdx.x;
    const int qt = p.n_qtiles - 1 - idx / (p.B * p.Hq);     // late (heavier under a causal mask) q tiles first
    const int bh = idx % (p.B * p.Hq);
    const int b = bh / p.Hq, h = bh % p.Hq, hkv = h / p.n_rep;
    const int row0 = qt * BM, my_row = row0 + rg * 32 + l32;
    const bool row_ok = my_row < p.Sq;
    const int my_pos = q_position(my_row, p.q_split, p.q_pos0[0], p.q_pos0[1]);
    int blk_lo, blk_hi, w_lo, w_hi;
    q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);
    {
        const int wr0 = row0 + rg * 32, wr1 = min(wr0 + 32, p.Sq) - 1;
        if (wr1 >= wr0) q_pos_range(wr0, wr1, p.q_split, p.q_pos0[0], p.q_pos0[1], w_lo, w_hi);
        else { w_lo = 0x7fffffff; w_hi = -0x7fffffff; }   // wave has no valid row
    }

    // Q operand: qreg[4g + j] = Q[row][8g + 4h + j]
    float qreg[D / 2];
    {
        const float *qp = (const float *)p.q + b * p.qs[0] + (long long)min(my_row, p.Sq - 1) * p.qs[1] + h * p.qs[2];
#pragma unroll
        for (int g = 0; g < D / 8; g++) {
            f32x4 x = *(const f32x4 *)(qp + 8 * g + 4 * hh);
            if (!row_ok) x = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) qreg[4 * g + j] = x[j];
        }
    }
    f32x16 oacc[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[i][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;   // exp2 domain; l_run: this lane's half of the keys
    const float c2 = p.scale * LTR_LOG2E;

    // step iterator over (chunk, BN keys); chunk fields live in scalar registers (see the bf16 kernel)
    int c = -1, t = 0, nt = 0;
    int ld_sk = 0, ld_pos0 = 0;
    const float *ld_kb = nullptr, *ld_vb = nullptr;
    auto settle = [&]() {
        while (c < p.n_chunks && t >= nt) {
            c++;
            t = 0;
            if (c < p.n_chunks) {
                ld_sk = p.chunk[c].sk;
                ld_pos0 = p.chunk[c].pos0;
                ld_kb = (const float *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
                ld_vb = (const float *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
                const int nvis = causal ? max(0, min(ld_sk, blk_hi - ld_pos0 + 1)) : ld_sk;
                nt = (nvis + BN - 1) / BN;
            }
        }
    };
    settle();
    const int st_row = lane / CPR, st_pc = lane % CPR;
    int nx_sk = 0, nx_pos0 = 0, nx_key0 = 0;
    auto gload = [&](int ti, int buf) {
        nx_sk = ld_sk;
        nx_pos0 = ld_pos0;
        nx_key0 = ti * BN;
        const unsigned Kd = lds_address(smem) + buf * L::BUF_BYTES, Vd = Kd + TILE * 4;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int row = RPI * (NI * w + i) + st_row;
            const int key = min(ti * BN + row, ld_sk - 1);       // rows past the end repeat the last row; they are masked
            const int chunk = st_pc ^ f32_swz(row);
            global_to_lds_b128(ld_kb + ((long long)key * p.ks[1] + chunk * 4), Kd + RPI * (NI * w + i) * D * 4);
            global_to_lds_b128(ld_vb + ((long long)key * p.vs[1] + chunk * 4), Vd + RPI * (NI * w + i) * D * 4);
        }
    };
    bool have = c < p.n_chunks;
    if (!have && (p.flags & LTR_MERGE)) return;   // merging an empty partial result changes nothing (block-uniform)
    if (have) gload(t, 0);
    tile_barrier();
    int par = 0;
    while (have) {
        const int sk = nx_sk, pos0 = nx_pos0, key0 = nx_key0 + 32 * ks;   // this wave's 32 keys of the step
        const float *Ks = (const float *)(smem + par * L::BUF_BYTES) + 32 * ks * D, *Vs = Ks + TILE;
        t++;
        settle();
        const bool have_next = c < p.n_chunks;
        if (have_next) gload(t, par ^ 1);
        // nothing to add: the sub-tile starts past the chunk's end, or every row of the wave precedes its first key
        if (key0 < sk && (!causal || pos0 + key0 <= w_hi)) {
            f32x16 s;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.f;
            const float *krow = Ks + l32 * D;
            const int ksw = f32_swz(l32);
#pragma unroll
            for (int g = 0; g < D / 8; g++) {
                const f32x4 kx = *(const f32x4 *)(krow + (((2 * g + hh) ^ ksw) << 2));
#pragma unroll
                for (int j = 0; j < 4; j++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[j], qreg[4 * g + j], s, 0, 0, 0);
            }
            const bool need_mask = (key0 + 32 > sk) || (causal && (pos0 + key0 + 31 > w_lo));
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                float tv = s[r] * c2;
                if (need_mask) {
                    const int key = key0 + 8 * (r / 4) + 4 * hh + (r % 4);
                    const bool vis = key < sk && (!causal || pos0 + key <= my_pos);
                    tv = vis ? tv : -INFINITY;
                }
                s[r] = tv;
                mx = fmaxf(mx, tv);
            }
            mx = xhalf_max(mx);                                   // row max over the 32 keys (both halves agree)
            const float m_new = fmaxf(m_run, mx);
            const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);   // m_run = -inf: 0 (nothing accumulated yet)
            float l_tile = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s[r] = __builtin_amdgcn_exp2f(s[r] - m_use);
                l_tile += s[r];
            }
            l_run = l_run * alpha + l_tile;
            m_run = m_new;
#pragma unroll
            for (int i = 0; i < D / 32; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
            // O^T += V^T P^T: step r contracts key 8 (r / 4) + 4h + r % 4; lane (d = 32 db + l32, h) reads V[key][d]
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int vrow = 8 * (r / 4) + 4 * hh + (r % 4);
                const float *vr = Vs + vrow * D + (l32 & 3);
                const int vsw = f32_swz(vrow);
#pragma unroll
                for (int db = 0; db < D / 32; db++) {
                    const float vx = vr[((8 * db + (l32 >> 2)) ^ vsw) << 2];
                    oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vx, s[r], oacc[db], 0, 0, 0);
                }
            }
        }
        tile_barrier();
        par ^= 1;
        have = have_next;
    }

    // merge of the KS partial results of a row group (the tile buffers are no longer read: the last barrier is behind us)
    float l_tot = xhalf_sum(l_run);
    if constexpr (KS > 1) {
        float *ml = (float *)(smem + L::ML_OFF);
        if (hh == 0) {
            ml[w * 64 + l32] = m_run;
            ml[w * 64 + 32 + l32] = l_tot;
        }
        __syncthreads();
        float m_all = -INFINITY;
#pragma unroll
        for (int k2 = 0; k2 < KS; k2++) m_all = fmaxf(m_all, ml[(rg * KS + k2) * 64 + l32]);
        const float m_ref = m_all == -INFINITY ? 0.f : m_all;
        float l_sum = 0.f;
#pragma unroll
        for (int k2 = 0; k2 < KS; k2++)
            l_sum += ml[(rg * KS + k2) * 64 + 32 + l32] * __builtin_amdgcn_exp2f(ml[(rg * KS + k2) * 64 + l32] - m_ref);
        const float f_own = __builtin_amdgcn_exp2f(m_run - m_ref);
        float *part = (float *)(smem + L::PART_OFF);
        if (ks > 0) {
            float *mine = part + (size_t)(rg * (KS - 1) + ks - 1) * (L::PART_BYTES / 4);
#pragma unroll
            for (int i = 0; i < D / 32; i++)
#pragma unroll
                for (int r4 = 0; r4 < 4; r4++) {
                    f32x4 x;
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] = oacc[i][4 * r4 + e] * f_own;
                    *(f32x4 *)(mine + ((i * 4 + r4) * 64 + lane) * 4) = x;
                }
        }
        __syncthreads();
        if (ks == 0) {
#pragma unroll
            for (int i = 0; i < D / 32; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) oacc[i][r] *= f_own;
            for (int k2 = 1; k2 < KS; k2++) {
                const float *other = part + (size_t)(rg * (KS - 1) + k2 - 1) * (L::PART_BYTES / 4);
#pragma unroll
                for (int i = 0; i < D / 32; i++)
#pragma unroll
                    for (int r4 = 0; r4 < 4; r4++) {
                        const f32x4 x = *(const f32x4 *)(other + ((i * 4 + r4) * 64 + lane) * 4);
#pragma unroll
                        for (int e = 0; e < 4; e++) oacc[i][4 * r4 + e] += x[e];
                    }
            }
        }
        m_run = m_all;
        l_tot = l_sum;
        if (ks > 0) return;    // no barrier follows
    }

    // epilogue of the wave that holds the row group's result: normalise, optional merge with (o, lse), whole rows out
    float lse_new = (l_tot > 0.f) ? m_run * LTR_LN2 + logf(l_tot) : -INFINITY;
    float w_cur = (l_tot > 0.f) ? 1.f / l_tot : 0.f, w_old = 0.f;
    float *lse_p = p.lse + ((long long)b * p.Hq + h) * p.Sq + my_row;
    if ((p.flags & LTR_MERGE) && row_ok) {
        const float lse_old = *lse_p;
        const float mxl = fmaxf(lse_old, lse_new);
        if (mxl == -INFINITY) {
            w_cur = 0.f;
        } else {
            const float e_old = expf(lse_old - mxl), e_new = expf(lse_new - mxl);
            const float tot = e_old + e_new;
            w_old = e_old / tot;
            w_cur *= e_new / tot;
            lse_new = mxl + logf(tot);
        }
    }
    if (row_ok && hh == 0) *lse_p = lse_new;
    unsigned char *stage = smem + L::STAGE_OFF + rg * WaveStage<D>::BYTES;
    float *row_w_old = (float *)(stage + 32 * WaveStage<D>::ROW_BYTES);
    if (hh == 0) row_w_old[l32] = w_old;
    constexpr int LPR = D / 4, ROWS_PER_IT = 64 / LPR;
    const int wave_row0 = row0 + rg * 32;
    const bool merge = (p.flags & LTR_MERGE) != 0;
    float *op = (float *)p.o + b * p.os[0] + h * p.os[2] + (long long)(wave_row0 + lane / LPR) * p.os[1] + 4 * (lane % LPR);
    const long long os1 = p.os[1];
    const int Sq = p.Sq;
    wave_tile_rowmajor<D>(stage, lane, oacc, w_cur, [&](int row, int, f32x4 val) {
        if (wave_row0 + row < Sq) {
            if (merge) {
                const f32x4 old = *(const f32x4 *)op;
                const float wo = row_w_old[row];
#pragma unroll
                for (int e = 0; e < 4; e++) val[e] += old[e] * wo;
            }
            *(f32x4 *)op = val;
        }
        op += ROWS_PER_IT * os1;
    });
}


// Four key shares per row group (head dim 64), for launches with the fewest rows: groups of 16 rows on v_mfma_f32_16x16x4_f32 (the rate of
// 32x32x2), so that a launch has twice the blocks of 32-row groups: 2 x 8 heads of 256 rows give every CU one instead of every other.
// A wave's 32 keys of a step are two sub-tiles whose chains alternate.  Operand layout (lane l, i = l % 16, g = l / 16): A[i][g], B[g][i],
// C[4g + r][i] for accumulator register r.  As in the 32-row kernels both contractions choose their order: step 4s + j of S^T contracts d = 16s + 4g + j (K: one 128-bit read for four steps), step r of O^T / dQ^T the keys 4g + r of a
// sub-tile, whose P^T / dS^T is the accumulator register r as it is.  f32_swz serves both reads (rows 4 apart land 4 chunks apart).
// Each wave ends up with 16 of the 64 columns of all shares and writes 16 bytes per lane.  Bound by latency, one wave per SIMD (one block per
// CU): forward / dQ wait 35 / 43 % of the time for data and barriers, matrix pipe 29 / 33 % busy, vector 21 / 15, LDS 10 / 9 (a third of it bank
// conflicts).  Kernel us, 32 -> 16 rows, forward and dQ, 2 x 8 heads of 256 rows against 256, 768, 1024 keys:
// 10.8 -> 7.5, 22.0 -> 14.6, 27.7 -> 18.1 and 15.0 -> 9.4, 29.9 -> 18.7, 37.3 -> 23.3; one head of 8 rows and 64 keys 7.1 -> 5.0, 9.2 -> 6.2.
struct F32Rows16 {
    static constexpr int D = 64, KS = 4, BM = 16;
    static constexpr int PART = 16 * 64 * 4;             // one wave's D x 16 partial result
    static constexpr int PART_OFF = 4 * 32 * 4;          // after the waves' references and sums (forward)
    static constexpr int BYTES = PART_OFF + KS * PART;
    static_assert(BYTES <= F32Mfma<D, KS>::LDS, "reuses the tile buffers");
};
__device__ __forceinline__ float quarter_max(float x) {   // over the four lanes of a row (16 apart)
    const unsigned u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return xhalf_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float quarter_sum(float x) {
    const unsigned u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return xhalf_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}
// The row-group operand Q (or dO) of lane (row i, g): reg[4s + j] = X[row][16s + 4g + j]
__device__ __forceinline__ void rows16_operand(const float *row, int g, float (&reg)[16]) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const f32x4 x = *(const f32x4 *)(row + 16 * s + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; j++) reg[4 * s + j] = x[j];
    }
}
// acc[kb] += (rows 16 kb .. of the 32-row tile T) x reg^T, both sub-tiles' chains in turn
__device__ __forceinline__ void rows16_scores(const float *T, int i, int g, const float (&reg)[16], f32x4 (&acc)[2]) {
    const int sw = f32_swz(i);   // rows 16 apart share it
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const f32x4 a = *(const f32x4 *)(T + i * 64 + (((4 * s + g) ^ sw) << 2)), b = *(const f32x4 *)(T + (16 + i) * 64 + (((4 * s + g) ^ sw) << 2));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], reg[4 * s + j], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j], reg[4 * s + j], acc[1], 0, 0, 0);
        }
    }
}
// out[db] += T^T x w over the 32 keys: w[kb][r] belongs to key 16 kb + 4g + r of the lane's row
__device__ __forceinline__ void rows16_weighted(const float *T, int i, int g, const f32x4 (&w)[2], f32x4 (&out)[4]) {
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int key = 16 * kb + 4 * g + r, sw = f32_swz(key);
            const float *row = T + key * 64 + (i & 3);
#pragma unroll
            for (int db = 0; db < 4; db++)
                out[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(row[((4 * db + (i >> 2)) ^ sw) << 2], w[kb][r], out[db], 0, 0, 0);
        }
}
// Wave ks collects columns 16 ks .. +15 of all shares (times their factors): lane (row i, g) gets columns 16 ks + 4g .. +3.  The tile
// buffers are no longer read.
__device__ __forceinline__ f32x4 rows16_collect(unsigned char *smem, int ks, int lane, const f32x4 (&part)[4], float mul) {
    float *const parts = (float *)(smem + F32Rows16::PART_OFF);
#pragma unroll
    for (int db = 0; db < 4; db++) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = part[db][e] * mul;
        *(f32x4 *)(parts + ((ks * 4 + db) * 64 + lane) * 4) = x;
    }
    __syncthreads();
    f32x4 own = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const f32x4 x = *(const f32x4 *)(parts + ((k * 4 + ks) * 64 + lane) * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) own[e] += x[e];
    }
    return own;
}

template <int D, int KS>   // one key share at head dim 64: 36 KB of LDS; three blocks per CU (168 registers)
__global__ __launch_bounds__(256, D == 64 && KS == 1 ? 3 : 1) void fwd_f32_mfma_kernel(const FwdParams p) {
    fwd_f32_body<D, KS>(p);
}
template <int D, int KS>
__global__ __launch_bounds__(256) void fwd_f32_rows32_kernel(const FwdParams p) {
    fwd_f32_body<D, KS>(p);
}
template <>
__global__ __launch_bounds__(256) void fwd_f32_mfma_kernel<64, 4>(const FwdParams p) {   // see F32Rows16
    using L = F32Mfma<64, 4>;
    constexpr int D = 64, BM = F32Rows16::BM, BN = L::BN, TILE = L::TILE;
    constexpr int CPR = D / 4, RPI = 64 / CPR, NI = BN / (RPI * L::NW);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
    const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool causal = p.flags & LTR_CAUSAL;
    const int qt = p.n_qtiles - 1 - blockIdx.x / (p.B * p.Hq);     // late (heavier under a causal mask) q tiles first
    const int bh = blockIdx.x % (p.B * p.Hq);
    const int b = bh / p.Hq, h = bh % p.Hq, hkv = h / p.n_rep;
    const int row0 = qt * BM, my_row = row0 + i;
    const bool row_ok = my_row < p.Sq;
    const int my_pos = q_position(my_row, p.q_split, p.q_pos0[0], p.q_pos0[1]);
    int blk_lo, blk_hi;
    q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);

    float qreg[16];
    rows16_operand((const float *)p.q + b * p.qs[0] + (long long)min(my_row, p.Sq - 1) * p.qs[1] + h * p.qs[2], g, qreg);
    f32x4 oacc[4];
#pragma unroll
    for (int db = 0; db < 4; db++) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;   // exp2 domain; l_run: this lane's quarter of the keys
    const float c2 = p.scale * LTR_LOG2E;

    // step iterator and tile transfers: as in the kernels of 32-row groups
    int c = -1, t = 0, nt = 0;
    int ld_sk = 0, ld_pos0 = 0;
    const float *ld_kb = nullptr, *ld_vb = nullptr;
    auto settle = [&]() {
        while (c < p.n_chunks && t >= nt) {
            c++;
            t = 0;
            if (c < p.n_chunks) {
                ld_sk = p.chunk[c].sk;
                ld_pos0 = p.chunk[c].pos0;
                ld_kb = (const float *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
                ld_vb = (const float *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
                const int nvis = causal ? max(0, min(ld_sk, blk_hi - ld_pos0 + 1)) : ld_sk;
                nt = (nvis + BN - 1) / BN;
            }
        }
    };
    settle();
    const int st_row = lane / CPR, st_pc = lane % CPR;
    int nx_sk = 0, nx_pos0 = 0, nx_key0 = 0;
    auto gload = [&](int ti, int buf) {
        nx_sk = ld_sk;
        nx_pos0 = ld_pos0;
        nx_key0 = ti * BN;
        const unsigned Kd = lds_address(smem) + buf * L::BUF_BYTES, Vd = Kd + TILE * 4;
#pragma unroll
        for (int n = 0; n < NI; n++) {
            const int row = RPI * (NI * ks + n) + st_row;
            const int key = min(ti * BN + row, ld_sk - 1);       // rows past the end repeat the last row; they are masked
            const int chunk = st_pc ^ f32_swz(row);
            global_to_lds_b128(ld_kb + ((long long)key * p.ks[1] + chunk * 4), Kd + RPI * (NI * ks + n) * D * 4);
            global_to_lds_b128(ld_vb + ((long long)key * p.vs[1] + chunk * 4), Vd + RPI * (NI * ks + n) * D * 4);
        }
    };
    bool have = c < p.n_chunks;
    if (!have && (p.flags & LTR_MERGE)) return;   // merging an empty partial result changes nothing (block-uniform)
    if (have) gload(t, 0);
    tile_barrier();
    int par = 0;
    while (have) {
        const int sk = nx_sk, pos0 = nx_pos0, key0 = nx_key0 + 32 * ks;   // this wave's 32 keys of the step
        const float *Ks = (const float *)(smem + par * L::BUF_BYTES) + 32 * ks * D, *Vs = Ks + TILE;
        t++;
        settle();
        const bool have_next = c < p.n_chunks;
        if (have_next) gload(t, par ^ 1);
        // nothing to add: the sub-tile starts past the chunk's end, or every row precedes its first key
        if (key0 < sk && (!causal || pos0 + key0 <= blk_hi)) {
            f32x4 s[2];
            s[0] = s[1] = f32x4{0.f, 0.f, 0.f, 0.f};
            rows16_scores(Ks, i, g, qreg, s);
            const bool need_mask = (key0 + 32 > sk) || (causal && (pos0 + key0 + 31 > blk_lo));
            float mx = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float tv = s[kb][r] * c2;
                    if (need_mask) {
                        const int key = key0 + 16 * kb + 4 * g + r;
                        const bool vis = key < sk && (!causal || pos0 + key <= my_pos);
                        tv = vis ? tv : -INFINITY;
                    }
                    s[kb][r] = tv;
                    mx = fmaxf(mx, tv);
                }
            mx = quarter_max(mx);
            const float m_new = fmaxf(m_run, mx);
            const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);   // m_run = -inf: 0 (nothing accumulated yet)
            float l_tile = 0.f;
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[kb][r] = __builtin_amdgcn_exp2f(s[kb][r] - m_use);
                    l_tile += s[kb][r];
                }
            l_run = l_run * alpha + l_tile;
            m_run = m_new;
#pragma unroll
            for (int db = 0; db < 4; db++)
#pragma unroll
                for (int r = 0; r < 4; r++) oacc[db][r] *= alpha;
            rows16_weighted(Vs, i, g, s, oacc);
        }
        tile_barrier();
        par ^= 1;
        have = have_next;
    }

    // the shares agree on a reference, scale to it and exchange columns
    float *const ml = (float *)smem + ks * 32;   // [wave][16 references | 16 sums]
    const float l_own = quarter_sum(l_run);
    float *lse_p = p.lse + ((long long)b * p.Hq + h) * p.Sq + my_row;
    float lse_old = 0.f;
    if ((p.flags & LTR_MERGE) && row_ok) lse_old = *lse_p;   // before any wave writes it
    if (g == 0) {
        ml[i] = m_run;
        ml[16 + i] = l_own;
    }
    __syncthreads();
    float m_all = -INFINITY;
#pragma unroll
    for (int k = 0; k < 4; k++) m_all = fmaxf(m_all, ml[(k - ks) * 32 + i]);
    const float m_ref = m_all == -INFINITY ? 0.f : m_all;
    float l_tot = 0.f;
#pragma unroll
    for (int k = 0; k < 4; k++) l_tot += ml[(k - ks) * 32 + 16 + i] * __builtin_amdgcn_exp2f(ml[(k - ks) * 32 + i] - m_ref);
    const f32x4 own = rows16_collect(smem, ks, lane, oacc, __builtin_amdgcn_exp2f(m_run - m_ref));
    float lse_new = (l_tot > 0.f) ? m_all * LTR_LN2 + logf(l_tot) : -INFINITY;
    float w_cur = (l_tot > 0.f) ? 1.f / l_tot : 0.f, w_old = 0.f;
    if ((p.flags & LTR_MERGE) && row_ok) {
        const float mxl = fmaxf(lse_old, lse_new);
        if (mxl == -INFINITY) {
            w_cur = 0.f;
        } else {
            const float e_old = expf(lse_old - mxl), e_new = expf(lse_new - mxl);
            const float tot = e_old + e_new;
            w_old = e_old / tot;
            w_cur *= e_new / tot;
            lse_new = mxl + logf(tot);
        }
    }
    if (!row_ok) return;
    if (ks == 0 && g == 0) *lse_p = lse_new;
    float *op = (float *)p.o + b * p.os[0] + h * p.os[2] + (long long)my_row * p.os[1] + 16 * ks + 4 * g;
    f32x4 val;
#pragma unroll
    for (int e = 0; e < 4; e++) val[e] = own[e] * w_cur;
    if (p.flags & LTR_MERGE) {
        const f32x4 old = *(const f32x4 *)op;
#pragma unroll
        for (int e = 0; e < 4; e++) val[e] += old[e] * w_old;
    }
    *(f32x4 *)op = val;
}

// ------------------------------------------------------------------------------ delta
// 16 lanes per (b, row, h), 8 elements per lane in two sums of four: rows of one sequence index are read head after head, as they
// lie in memory.
__global__ __launch_bounds__(256) void delta_kernel(const DeltaParams p) {
    const long long rowid = ((long long)blockIdx.x * 256 + threadIdx.x) >> 4;
    const int d = 8 * (threadIdx.x & 15);
    const long long nrows = (long long)p.B * p.Hq * p.Sq;
    float acc = 0.f, acc_hi = 0.f;
    int i = 0, h = 0, b = 0;
    if (rowid < nrows) {
        const long long bi = rowid / p.Hq;   // b * Sq + i
        h = (int)(rowid - bi * p.Hq);
        if (p.rows32) {   // the usual case spares the 64-bit division
            b = (int)((unsigned)bi / (unsigned)p.Sq);
            i = (int)((unsigned)bi - (unsigned)b * (unsigned)p.Sq);
        } else {
            b = (int)(bi / p.Sq);
            i = (int)(bi - (long long)b * p.Sq);
        }
        if (d < p.D) {
            const long long oo = b * p.os[0] + (long long)i * p.os[1] + h * p.os[2] + d;
            const long long od = b * p.dos[0] + (long long)i * p.dos[1] + h * p.dos[2] + d;
            float ov[8], dv[8];
            auto load8 = [&](const void *base, long long off, bool f32, float (&v)[8]) {
                if (!p.vec) {
                    for (int e = 0; e < 8; e++) v[e] = f32 ? ((const float *)base)[off + e] : (float)((const __bf16 *)base)[off + e];
                } else if (f32) {
                    const f32x4 x = *(const f32x4 *)((const float *)base + off), y = *(const f32x4 *)((const float *)base + off + 4);
                    for (int e = 0; e < 4; e++) v[e] = x[e], v[4 + e] = y[e];
                } else {
                    const bf16x8 x = *(const bf16x8 *)((const __bf16 *)base + off);
                    for (int e = 0; e < 8; e++) v[e] = (float)x[e];
                }
            };
            load8(p.o, oo, p.o_f32, ov);
            load8(p.d_o, od, p.do_f32, dv);
#pragma unroll
            for (int e = 0; e < 4; e++) acc = fmaf(ov[e], dv[e], acc), acc_hi = fmaf(ov[4 + e], dv[4 + e], acc_hi);
            acc += acc_hi;
        }
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 16);
    if (rowid < nrows && d == 0) p.delta[((long long)b * p.Hq + h) * p.Sq + i] = acc;
}

// The same sums for bf16 in 16-byte loads and less than 2^31 rows, the DELTA launch of a joint backward: LANES lanes per row (8 where the columns end
// by 64: the halves that they leave out added zeros), FLIGHT rows per lane with their loads issued together, 32-bit row numbers.  Bound by latency: a
// launch of few microseconds is one load and its address; the general kernel (a 64-bit division, one row per lane, always 16 lanes) takes
// 6.9 us for 1237 x 32 rows of 128 (5.7 here), 4.7 for 2 x 777 x 16 of 96 (4.0).
template <int LANES>
__global__ __launch_bounds__(256) void delta_bf16_kernel(const DeltaParams p) {
    constexpr unsigned ROWS = 256 / LANES, FLIGHT = 2;
    const int d = 8 * (threadIdx.x % LANES);
    const unsigned first = blockIdx.x * (ROWS * FLIGHT) + threadIdx.x / LANES, n = (unsigned)p.B * p.Hq * p.Sq;
    bf16x8 o[FLIGHT], g[FLIGHT];
    unsigned at[FLIGHT];
#pragma unroll
    for (unsigned k = 0; k < FLIGHT; k++) {
        const unsigned row = first + k * ROWS, bi = row / (unsigned)p.Hq, h = row - bi * p.Hq, b = bi / (unsigned)p.Sq, i = bi - b * p.Sq;
        at[k] = (b * p.Hq + h) * p.Sq + i;
        o[k] = g[k] = as_bf16x8(make_uint4(0, 0, 0, 0));
        if (row < n && d < p.D) {
            o[k] = as_bf16x8(*(const uint4 *)((const __bf16 *)p.o + b * p.os[0] + i * p.os[1] + h * p.os[2] + d));
            g[k] = as_bf16x8(*(const uint4 *)((const __bf16 *)p.d_o + b * p.dos[0] + i * p.dos[1] + h * p.dos[2] + d));
        }
    }
#pragma unroll
    for (unsigned k = 0; k < FLIGHT; k++) {
        float acc = 0.f, acc_hi = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            acc = fmaf((float)o[k][e], (float)g[k][e], acc);
            acc_hi = fmaf((float)o[k][4 + e], (float)g[k][4 + e], acc_hi);
        }
        acc += acc_hi;
#pragma unroll
        for (int off = LANES / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, LANES);
        if (first + k * ROWS < n && d == 0) p.delta[at[k]] = acc;
    }
}

__global__ __launch_bounds__(256) void cast_kernel(const float *src, __bf16 *dst, long long n) {
    long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i + 3 < n) {
        f32x4 x = *(const f32x4 *)(src + i);
        bf16x4 y;
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = (__bf16)x[e];
        *(bf16x4 *)(dst + i) = y;
    } else {
        for (; i < n; i++) dst[i] = (__bf16)src[i];
    }
}

// ------------------------------------------------------------------------------ backward, bf16
// Two kernels, no atomics, bitwise reproducible:
//   bwd_dkdv_kernel  a block owns 128 keys of one kv head and runs 8 waves, two per SIMD: for each of
//                    the four 32-key slices one "P wave" (S = Q K^T, P, dV^T += dO^T P; K operand in
//                    registers) and one "dS wave" (dP = dO V^T, dS = P*(dP - DELTA), dK^T += Q^T dS;
//                    V operand in registers).  The P wave hands P (bf16, accumulator layout) to its
//                    partner through a 2 KB LDS slot; the dS wave runs one tile behind, so one block
//                    barrier per tile is enough.  The block loops over the query heads of the GQA
//                    group and over 64-row Q / dO tiles in triple-buffered LDS; dK^T and dV^T stay
//                    in registers for the whole loop.
//   bwd_dq_kernel    a block owns 256 query rows of one query head (32 per wave; Q and dO
//                    operands in registers), loops over 64-key K/V tiles like the forward;
//                    dQ^T accumulates in registers.
// LDS of bwd_dkdv_kernel (dynamic): three buffers of {Q tile, dO tile, -LSE/scale, -DELTA, row positions}, the P slots,
// the tile lists.
template <int D, int KW>
struct BwdLds {
    static constexpr int BN = 128 * KW; // keys per block, 32 * KW per wave pair
    static constexpr int BM = 64;       // query rows per tile (two 32-row MFMA sub-tiles)
    static constexpr int NT = 512;      // threads per block
    static constexpr int TILE = BM * D;                                  // elements; rows unpadded, chunks swizzled
    static constexpr int BUF_BYTES = 2 * TILE * 2 + 3 * BM * 4;          // Q, dO, -LSE/scale, -DELTA, row positions (masked tiles)
    static constexpr int P_SLOT = 64 * 32;                               // one lane = 16 bf16 = 32 bytes
    static constexpr int NBUF = 3;                                       // tile t (P waves), t-1 (dS waves), t+1 (in flight)
    static constexpr int P_OFF = NBUF * BUF_BYTES;
    static constexpr int MAX_QTILES = 4096;                              // Sq <= 262144 per launch
    static constexpr int LIST_OFF = P_OFF + 4 * 4 * KW * P_SLOT;         // 4 slices x 2 parities x 2 sub-tiles x KW halves of P slots
    static constexpr int TOTAL = LIST_OFF + 2 * MAX_QTILES * 2 + 16;     // two tile lists (ushort) + counts
    static_assert(TOTAL >= 8 * WaveStage<D>::BYTES, "the epilogue's staging areas reuse this memory");
    static_assert(TOTAL <= 160 * 1024, "LDS of one CU");
};

// Masked tiles: the visibility of (row, key) is kpos <= qpos[row], with the rows' positions staged in LDS beside LSE and
// DELTA (INT_MIN for a row past the end; INT_MAX - 1 for every row when there is no causal mask) and kpos = INT_MAX for
// a key past the end of its chunk: one compare and one select per element, whatever the position map of the rows is.
constexpr int BWD_QPOS_NONE = (int)0x80000000, BWD_QPOS_ALL = 0x7ffffffe, BWD_KPOS_NONE = 0x7fffffff;

// P wave, accumulator registers 2j and 2j+1 of a 32x32 sub-tile: sm = S - LSE / scale (the accumulator started at
// -LSE / scale), P = exp2(sm * c2) -> one packed bf16 pair in accumulator layout; qpos = positions of the sub-tile's 16
// rows in accumulator-register order
template <bool MASK>
__device__ __forceinline__ unsigned bwd_p_pair(const f32x16 &sm, int j, float c2, int kpos, const int (&qpos)[16]) {
    float p0 = __builtin_amdgcn_exp2f(sm[2 * j] * c2), p1 = __builtin_amdgcn_exp2f(sm[2 * j + 1] * c2);
    if (MASK) {
        p0 = kpos <= qpos[2 * j] ? p0 : 0.f;
        p1 = kpos <= qpos[2 * j + 1] ? p1 : 0.f;
    }
    return pack2_bf16(p0, p1);
}

// dS wave, the same pair: dS = P * (dP - DELTA), pu = packed P pair from the partner's LDS slot (masked entries
// are 0), dpm = dP - DELTA (the accumulator started at -DELTA)
__device__ __forceinline__ unsigned bwd_ds_pair(unsigned pu, const f32x16 &dpm, int j) {
    const float p0 = __uint_as_float(pu << 16), p1 = __uint_as_float(pu & 0xffff0000u);
    return pack2_bf16(p0 * dpm[2 * j], p1 * dpm[2 * j + 1]);
}

// A wave's D x 32 accumulator tile as it lies in its registers: 16 bytes per lane and instruction, 1 KB runs.
template <int D>
__device__ __forceinline__ void store_partial(float *dst, int lane, const f32x16 (&acc)[D / 32], float mul) {
#pragma unroll
    for (int i = 0; i < D / 32; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = acc[i][4 * g + e] * mul;
            *(f32x4 *)(dst + ((i * 4 + g) * 64 + lane) * 4) = v;
        }
}

// Key tiles of a chunk that have blocks: those up to position q_last.  Blocks that share a tile leave partial sums, so a tile that no
// query sees gets neither blocks nor a place in the workspace (the reduction kernel alone visits it); q_last is the largest
// int where every tile has its one block.
__host__ __device__ __forceinline__ int seen_tiles(int sk, int pos0, int q_last, int keys) {
    const long long seen = (long long)q_last - pos0 + 1;
    return seen <= 0 ? 0 : ((int)(seen < sk ? seen : sk) + keys - 1) / keys;
}

// The q tiles (BM rows) of a dK/dV block, listed once per block by one wave (ballot compaction: the order, and with it the rounding of
// the accumulation, is fixed), so that the main loops carry no classification arithmetic.  A tile's class depends on its rows
// only: 0 = no row sees any key of the block (skipped); 1 = every (row, key) pair is visible (list 0); 2 = needs the mask
// (diagonal, tails: list 1).  kpos_lo, kpos_hi: positions of the block's first and last key; split: which of the blocks that share the
// keys this is.
template <int BM, int MAX_QTILES>
__device__ __forceinline__ void list_q_tiles(const BwdParams &p, int lane, int split, int kpos_lo, int kpos_hi, bool key_tail,
                                             unsigned short *tlist, int *tcount) {
    const bool causal = p.flags & LTR_CAUSAL;
    auto tile_class = [&](int qt) {
        const int row0 = qt * BM;
        const bool edge = key_tail || row0 + BM > p.Sq;
        if (!causal) return edge ? 2 : 1;
        int lo, hi;
        q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], lo, hi);
        if (hi < kpos_lo) return 0;
        return (edge || kpos_hi > lo) ? 2 : 1;
    };
    // a block that shares its keys lists every n_share-th visible tile, counted from its own offset
    const int n_share = 1 << p.share_log2;
    int n1 = 0, n2 = 0;
    int skip = split & (n_share - 1);   // visible tiles to pass over before the next one of this block
    for (int base = 0; base < p.n_qtiles; base += 64) {
        const int qt = base + lane;
        int cls = qt < p.n_qtiles ? tile_class(qt) : 0;
        if (n_share > 1) {
            const unsigned long long vis = __builtin_amdgcn_ballot_w64(cls != 0);
            const int rank = __builtin_popcountll(vis & ((1ull << lane) - 1ull)), n = __builtin_popcountll(vis);
            if (((rank - skip) & (n_share - 1)) != 0 || rank < skip) cls = 0;
            skip = (skip - n) & (n_share - 1);
        }
        const unsigned long long m1 = __builtin_amdgcn_ballot_w64(cls == 1), m2 = __builtin_amdgcn_ballot_w64(cls == 2);
        const unsigned long long below = (1ull << lane) - 1ull;
        if (cls == 1) tlist[n1 + __builtin_popcountll(m1 & below)] = (unsigned short)qt;
        if (cls == 2) tlist[MAX_QTILES + n2 + __builtin_popcountll(m2 & below)] = (unsigned short)qt;
        n1 += __builtin_popcountll(m1);
        n2 += __builtin_popcountll(m2);
    }
    if (lane == 0) {
        tcount[0] = n1;
        tcount[1] = n2;
    }
}

// A wave's dK^T or dV^T tile of 32 keys (times mul) through its LDS staging area: stored as bf16 rows (LTR_DKDV_BF16: every query that
// sees these keys was in this launch) or added to the fp32 accumulator in whole rows.  base + off: key 0, column 0.
template <int D, bool PAD>
__device__ __forceinline__ void write_key_rows(unsigned char *stage, int lane, const f32x16 (&acc)[D / 32], float mul, bool as_bf16,
                                               void *base, long long off, long long row_stride, int first_key, int n_keys, int cols) {
    constexpr int LPR = D / 4, ROWS_PER_IT = 64 / LPR;      // see wave_tile_rowmajor
    const long long stride = uniform64(row_stride);
    const int key_base = uniform32(first_key), sk = uniform32(n_keys);
    const long long goff = off + (key_base + lane / LPR) * stride + 4 * (lane % LPR);
    if (as_bf16) {
        __bf16 *gb = (__bf16 *)base + goff;
        wave_tile_rowmajor<D>(stage, lane, acc, mul, [&](int row, int col, f32x4 val) {
            if (key_base + row < sk && (!PAD || col < cols)) {
                bf16x4 y;
#pragma unroll
                for (int e = 0; e < 4; e++) y[e] = (__bf16)val[e];
                *(bf16x4 *)gb = y;
            }
            gb += ROWS_PER_IT * stride;
        });
        return;
    }
    float *gp = (float *)base + goff;
    // all reads of the accumulator first (independent loads in flight together), then the adds and the writes
    constexpr int NIT = 32 / ROWS_PER_IT;
    f32x4 old[NIT];
#pragma unroll
    for (int it = 0; it < NIT; it++) {
        old[it] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (key_base + it * ROWS_PER_IT + lane / LPR < sk && (!PAD || 4 * (lane % LPR) < cols)) old[it] = *(const f32x4 *)(gp + it * ROWS_PER_IT * stride);
    }
    int it = 0;
    wave_tile_rowmajor<D>(stage, lane, acc, mul, [&](int row, int col, f32x4 val) {
        if (key_base + row < sk && (!PAD || col < cols)) {
#pragma unroll
            for (int e = 0; e < 4; e++) val[e] += old[it][e];
            *(f32x4 *)gp = val;
        }
        gp += ROWS_PER_IT * stride;
        it++;
    });
}

// DELTA = rowsum(dO * O) of every row of the q heads that a dK/dV block walks, by the block itself (into LDS: [head][row]), for launches of few rows:
// the additions are delta_kernel's, whose launch costs more than these rows' bytes.
template <int D, bool PAD>
__device__ __forceinline__ void own_delta(const BwdParams &p, int b, int h_first, float *out) {
    constexpr int LANES = D / 8, ROWS = 512 / LANES, FLIGHT = 4;   // lanes per row, rows per pass, passes in flight
    const int d = 8 * (threadIdx.x % LANES), first = threadIdx.x / LANES, n = p.n_reps * p.Sq;
    const bool in = !PAD || d < p.cols;
    for (int base = first; base < n; base += FLIGHT * ROWS) {
        bf16x8 o[FLIGHT], g[FLIGHT];
#pragma unroll
        for (int i = 0; i < FLIGHT; i++) {
            const int idx = base + i * ROWS, rep = idx / p.Sq, row = idx - rep * p.Sq;
            o[i] = g[i] = as_bf16x8(make_uint4(0, 0, 0, 0));
            if (idx < n && in) {
                o[i] = as_bf16x8(*(const uint4 *)((const __bf16 *)p.o + b * p.os_[0] + (long long)row * p.os_[1] + (h_first + rep) * p.os_[2] + d));
                g[i] = as_bf16x8(*(const uint4 *)((const __bf16 *)p.d_o + b * p.dos[0] + (long long)row * p.dos[1] + (h_first + rep) * p.dos[2] + d));
            }
        }
#pragma unroll
        for (int i = 0; i < FLIGHT; i++) {
            float acc = 0.f, acc_hi = 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                acc = fmaf((float)o[i][e], (float)g[i][e], acc);
                acc_hi = fmaf((float)o[i][4 + e], (float)g[i][4 + e], acc_hi);
            }
            acc += acc_hi;
#pragma unroll
            for (int off = LANES / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, LANES);
            if (base + i * ROWS < n && d == 0) out[base + i * ROWS] = acc;
        }
    }
}

template <int D, int KW, bool PAD, bool OWN_DELTA = false, int DC = D>
__device__ __forceinline__ void bwd_dkdv_body(const BwdParams &p, const BlockItem item) {
    const int cols = PAD ? p.cols : D;
    using L = BwdLds<D, KW>;   // KW = 32-key halves per wave
    constexpr int BN = L::BN, BM = L::BM;
    constexpr int CPR = D / 8;
    constexpr int RPI = 64 / CPR;        // rows filled by one wave-wide LDS-direct load (1 KB)
    constexpr int NI = BM / (RPI * 8);   // such loads per wave, per tensor and per tile
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slice = w & 3;             // slice of 32 * KW keys; waves w and w+4 (same SIMD) are partners
    const bool p_role = w < 4;           // P wave (S, P, dV) or dS wave (dP, dS, dK)
    const int l32 = lane & 31, hh = lane >> 5;
    const bool causal = p.flags & LTR_CAUSAL;

    // block -> (batch, kv head, chunk, key tile); same XCD grouping as the forward.  Blocks that share a key tile follow each
    // other: each takes n_reps of the q heads and, of a head's visible q tiles, every 2^share_log2-th
    const int pair = item.pair, split = item.sub, tile = item.item;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv;
    int c = 0, kt = tile;
    for (; c < p.n_chunks; c++) {
        const int n = seen_tiles(p.chunk[c].sk, p.chunk[c].pos0, p.q_last, BN);
        if (kt < n) break;
        kt -= n;
    }
    if (c >= p.n_chunks) return;
    const int sk = p.chunk[c].sk, pos0 = p.chunk[c].pos0;
    const int key0 = kt * BN;
    int my_key[KW];   // this lane's keys in the S / dP / dK^T / dV^T tiles of the wave's two halves
    bool key_ok[KW];
#pragma unroll
    for (int k = 0; k < KW; k++) {
        my_key[k] = key0 + slice * 32 * KW + 32 * k + l32;
        key_ok[k] = my_key[k] < sk;
    }
    const int tile_kpos_lo = pos0 + key0;
    const int tile_kpos_hi = pos0 + min(key0 + BN, sk) - 1;
    const bool key_tail = key0 + BN > sk;
    if (causal) {   // no query of this launch sees the block (a later chunk of the ring): nothing to add, nothing to load
        int q_lo, q_hi;
        q_pos_range(0, (int)p.Sq - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], q_lo, q_hi);
        if (q_hi < tile_kpos_lo) {
            for (int k = 0; k < KW; k++)
            if ((p.flags & LTR_DKDV_BF16) && key_ok[k]) {   // results, not accumulators: these keys get zeros
                __bf16 *gz = p_role ? (__bf16 *)p.chunk[c].dv + b * p.dvs[0] + (long long)my_key[k] * p.dvs[1] + hkv * p.dvs[2]
                                    : (__bf16 *)p.chunk[c].dk + b * p.dks[0] + (long long)my_key[k] * p.dks[1] + hkv * p.dks[2];
                for (int d = 8 * hh; d < cols; d += 16) *(uint4 *)(gz + d) = make_uint4(0, 0, 0, 0);
            }
            return;
        }
    }

    // resident B operand: K rows for a P wave, V rows for a dS wave; lane (key l32, half hh) holds
    // d = 16*kb + 8*hh .. +7
    bf16x8 kvreg[KW][D / 16];
    {
        const __bf16 *base = p_role ? (const __bf16 *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2]
                                    : (const __bf16 *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
        const long long rs = p_role ? p.ks[1] : p.vs[1];
#pragma unroll
        for (int k = 0; k < KW; k++) {
            const int ksafe = min(my_key[k], sk - 1);
#pragma unroll
            for (int kb = 0; kb < DC / 16; kb++) {
                uint4 x = make_uint4(0, 0, 0, 0);
                if (!PAD || kb * 16 + 8 * hh < cols) x = *(const uint4 *)(base + (long long)ksafe * rs + kb * 16 + 8 * hh);
                if (!key_ok[k]) x = make_uint4(0, 0, 0, 0);
                kvreg[k][kb] = as_bf16x8(x);
            }
        }
    }

    f32x16 zero16;
#pragma unroll
    for (int r = 0; r < 16; r++) zero16[r] = 0.f;
    f32x16 acc[KW][D / 32];              // dV^T (P wave) or dK^T (dS wave) of the two halves
#pragma unroll
    for (int k = 0; k < KW; k++)
#pragma unroll
        for (int i = 0; i < D / 32; i++) acc[k][i] = zero16;
    const float c2 = p.scale * LTR_LOG2E;

    unsigned short *const tlist = (unsigned short *)(smem + L::LIST_OFF);     // [2][MAX_QTILES]
    int *const tcount = (int *)(smem + L::LIST_OFF + 2 * L::MAX_QTILES * 2);
    const int h_first = hkv * p.n_rep + (split >> p.share_log2) * p.n_reps;   // first of the n_reps q heads this block walks
    float *const dlt = (float *)(smem + L::TOTAL);                            // OWN_DELTA: [n_reps][Sq]
    if (w == 0) list_q_tiles<BM, L::MAX_QTILES>(p, lane, split, tile_kpos_lo, tile_kpos_hi, key_tail, tlist, tcount);
    if constexpr (OWN_DELTA) own_delta<D, PAD>(p, b, h_first, dlt);
    __syncthreads();

    const int st_row = lane / CPR, st_pc = lane % CPR;   // this lane's place inside a 1 KB LDS-direct load
    // Per-lane element offsets of this lane's pieces of a Q / dO tile (unmasked tiles: row and chunk do not depend on the
    // tile) and the bases of the current q head: a step then adds one scalar product per tensor instead of redoing the
    // 64-bit address arithmetic of (batch, head, row).
    unsigned offq[NI], offdo[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int row = RPI * (NI * w + i) + st_row;
        const int chunk = st_pc ^ lds_swz<D>(row);
        offq[i] = (unsigned)(row * (int)p.qs[1] + chunk * 8);
        offdo[i] = (unsigned)(row * (int)p.dos[1] + chunk * 8);
    }
    const __bf16 *qp_head = nullptr, *dop_head = nullptr;
    const float *sp_head = nullptr;   // LSE (wave 0) or DELTA - BM (wave 1) of the head's rows, indexed by row0 + tid
    auto set_head = [&](int rep) __attribute__((always_inline)) {
        const int h = h_first + rep;
        qp_head = (const __bf16 *)p.q + b * p.qs[0] + h * p.qs[2];
        dop_head = (const __bf16 *)p.d_o + b * p.dos[0] + h * p.dos[2];
        const long long so = ((long long)b * p.Hq + h) * p.Sq;
        sp_head = w == 0 ? p.lse + so : p.delta + so - BM;
    };
    const float st_mul = tid < BM ? -1.f / p.scale : -1.f;  // threads 0..63 stage -LSE/scale, 64..127 stage -DELTA
    float sld = 0.f;      // raw LSE / DELTA value in flight; scaled when it is written to LDS
    bool sld_ok = true;
    int sld_row0 = 0;     // first row of the tile in flight
    unsigned *const pslot_base = (unsigned *)(smem + L::P_OFF) + slice * 4 * KW * (L::P_SLOT / 4);   // [parity][sub-tile][half]

    // two passes, each a loop of its own (unmasked tiles, then masked ones), so the accumulators
    // live in straight-line loop bodies and the unmasked pass carries no bounds checks at all
    auto run_pass = [&](auto mask_tag) {
        constexpr bool MASK = decltype(mask_tag)::value;
        constexpr int cls = MASK ? 2 : 1;
        const int cnt = __builtin_amdgcn_readfirstlane(tcount[cls - 1]);
        const unsigned short *const list = tlist + (cls - 1) * L::MAX_QTILES;
        int li_ = -1;                                 // index into the list
        // the list entry of the next call is read from LDS one call ahead, so its latency is never waited for
        unsigned short pre = list[0];
        auto advance = [&](int &rep, int &qt) {   // next tile of this class after (rep, qt); false when done
            if (++li_ >= cnt) {
                li_ = 0;
                if (++rep >= p.n_reps) return false;
                set_head(rep);
            }
            qt = __builtin_amdgcn_readfirstlane((int)pre);
            pre = list[li_ + 1 < cnt ? li_ + 1 : 0];
            return true;
        };
        // Q and dO tiles go from global memory straight into LDS (global_load_lds, 16 bytes per lane): wave w
        // fills rows RPI*(NI*w + i) .. of both tiles with its i-th pair of loads, lane l the chunk position
        // l % CPR of row l / CPR, fetching the logical chunk the swizzle places there.  Rows past the end of Q
        // repeat its last row (they are masked).  LSE and DELTA go through a register of threads 0..127.
        auto gload = [&](int rep, int qt, int buf) {
            const int row0 = qt * BM;
            sld_row0 = row0;
            const unsigned Qd = lds_address(smem) + buf * L::BUF_BYTES, dOd = Qd + L::TILE * 2;   // LDS byte addresses
            if (!MASK) {
                const unsigned tq = (unsigned)(row0 * (int)p.qs[1]), tdo = (unsigned)(row0 * (int)p.dos[1]);
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    if (PAD && (st_pc ^ lds_swz<D>(RPI * (NI * w + i) + st_row)) * 8 >= cols) continue;
                    global_to_lds_b128(qp_head + (unsigned long long)(tq + offq[i]), Qd + RPI * (NI * w + i) * D * 2);
                    global_to_lds_b128(dop_head + (unsigned long long)(tdo + offdo[i]), dOd + RPI * (NI * w + i) * D * 2);
                }
            } else {
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    const int row = RPI * (NI * w + i) + st_row;
                    const int grow = min(row0 + row, p.Sq - 1);
                    const int chunk = st_pc ^ lds_swz<D>(row);
                    if (PAD && chunk * 8 >= cols) continue;
                    global_to_lds_b128(qp_head + (long long)(grow * (int)p.qs[1] + chunk * 8), Qd + RPI * (NI * w + i) * D * 2);
                    global_to_lds_b128(dop_head + (long long)(grow * (int)p.dos[1] + chunk * 8), dOd + RPI * (NI * w + i) * D * 2);
                }
            }
            if (tid < 2 * BM) {
                const float *sp = sp_head + row0;
                const int r = tid < BM ? tid : tid - BM;
                if (MASK) sld_ok = row0 + r < p.Sq;
                if (OWN_DELTA && w == 1) sld = dlt[rep * p.Sq + (!MASK || sld_ok ? row0 + r : 0)];
                else if (!MASK) sld = sp[tid];
                else sld = sp[sld_ok ? tid : (tid < BM ? 0 : BM)];
            }
        };
        auto lds_store = [&](int buf) {   // the LSE / DELTA values fetched by gload
            float *st = (float *)(smem + buf * L::BUF_BYTES) + L::TILE;   // after the two bf16 tiles
            if (tid < 2 * BM) {
                float x = sld * st_mul;
                // rows past the end: -LSE/scale = -inf makes P = 0 (they are masked as well)
                if (MASK) x = sld_ok ? x : (tid < BM ? -INFINITY : 0.f);
                st[tid] = x;
            } else if (MASK && tid < 3 * BM) {   // positions of the tile's rows (third wave)
                const int row = sld_row0 + tid - 2 * BM;
                ((int *)st)[tid] = row >= p.Sq ? BWD_QPOS_NONE
                                   : causal ? q_position(row, p.q_split, p.q_pos0[0], p.q_pos0[1]) : BWD_QPOS_ALL;
            }
        };

        int kpos[KW];
#pragma unroll
        for (int k = 0; k < KW; k++) kpos[k] = key_ok[k] ? pos0 + my_key[k] : BWD_KPOS_NONE;
        if (cnt == 0) return;
        int rep = 0, qt = 0;
        set_head(0);
        advance(rep, qt);
        __syncthreads();   // the previous pass has finished reading LDS
        gload(rep, qt, 0);
        lds_store(0);
        tile_barrier();
        // One LDS barrier per 64-row tile.  In step t the P wave does all its work on tile t (S of both
        // sub-tiles, P -> slots of parity t & 1, dV) and the dS wave all its work on tile t-1 (dP, dS with P
        // from the slots filled one step earlier, dK): inside a step the two waves of a SIMD are independent,
        // so one wave's softmax arithmetic runs under the other's MFMAs.  Slots of parity (t & 1) are
        // rewritten in step t+2, after the barrier that ends step t+1 in which they were read.  Tile t+1 is
        // fetched into registers at the start of step t and stored at its end into buffer (t+1) % 3, which
        // held tile t-2, last read in step t-1.  Both roles execute T + 1 barriers.
        auto put_slot = [&](unsigned *slot, const PackedTile &t) {
            // two 16-byte halves per lane, each half contiguous over the lanes (no bank conflicts)
            *(uint4 *)(slot + lane * 4) = make_uint4(t.u[0], t.u[1], t.u[2], t.u[3]);
            *(uint4 *)(slot + 256 + lane * 4) = make_uint4(t.u[4], t.u[5], t.u[6], t.u[7]);
        };
        int par = 0;
        // In the pass over unmasked tiles both loops are unrolled over the three Q / dO buffers (buf is a compile-time
        // constant inside a step), so that LDS addresses are loop-invariant per-lane registers plus immediate offsets;
        // the pass over masked tiles (few steps, more live registers) keeps one loop body with buf in a register.
        if (p_role) {
            bool more = true;
            auto p_step = [&](auto buf_tag) {
                const int buf = buf_tag;
                more = advance(rep, qt);
                const int nbuf = buf == L::NBUF - 1 ? 0 : buf + 1;
                if (more) gload(rep, qt, nbuf);
                const __bf16 *Qs = (const __bf16 *)(smem + buf * L::BUF_BYTES);
                const __bf16 *dOs = Qs + L::TILE;
                const float *st_s = (const float *)(dOs + L::TILE);   // -LSE/scale of the tile's rows
                unsigned *slots = pslot_base + par * 2 * KW * (L::P_SLOT / 4);
                // Accumulator register r of a sub-tile <-> tile row 8*(r/4) + 4*hh + r%4: both S accumulators start at
                // -LSE/scale of their rows.  Order of the step: S of sub-tile a; S of sub-tile b with the
                // exponentials of a issued under its MFMAs; first half of dV (rows of a) with the exponentials of b
                // under its MFMAs; second half of dV.
                f32x16 sa[KW], sb[KW];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 la = *(const f32x4 *)(st_s + 8 * g + 4 * hh), lb = *(const f32x4 *)(st_s + 32 + 8 * g + 4 * hh);
#pragma unroll
                    for (int k = 0; k < KW; k++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            sa[k][4 * g + e] = la[e];
                            sb[k][4 * g + e] = lb[e];
                        }
                }
                int qa[16], qb[16];   // positions of the rows (masked tiles only)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int *st_q = (const int *)st_s + 2 * BM;
                    const i32x4 xa = MASK ? *(const i32x4 *)(st_q + 8 * g + 4 * hh) : i32x4{0, 0, 0, 0};
                    const i32x4 xb = MASK ? *(const i32x4 *)(st_q + 32 + 8 * g + 4 * hh) : i32x4{0, 0, 0, 0};
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        qa[4 * g + e] = xa[e];
                        qb[4 * g + e] = xb[e];
                    }
                }
                PackedTile ppa[KW], ppb[KW];
                constexpr int NK = DC / 16, NS = 2 * (DC / 32);   // MFMAs of a chain, of a half of dV / dK
                __builtin_amdgcn_s_setprio(1);
                // every Q / dO operand read from LDS feeds the MFMAs of both halves
                lds_gemm_chain_kw<D, KW, DC>(Qs + l32 * D, lds_swz<D>(l32) ^ hh, kvreg, sa);
                lds_gemm_chain_kw<D, KW, DC>(Qs + (32 + l32) * D, lds_swz<D>(32 + l32) ^ hh, kvreg, sb, [&](int kb) {
#pragma unroll
                    for (int k = 0; k < KW; k++)
#pragma unroll
                        for (int j = kb * 8 / NK; j < (kb + 1) * 8 / NK; j++) ppa[k].u[j] = bwd_p_pair<MASK>(sa[k], j, c2, kpos[k], qa);
                });
                bf16x8 pba[KW][2], pbb[KW][2];
#pragma unroll
                for (int k = 0; k < KW; k++) {
                    put_slot(slots + k * (L::P_SLOT / 4), ppa[k]);
                    pba[k][0] = operand_of(ppa[k], 0);
                    pba[k][1] = operand_of(ppa[k], 1);
                }
                lds_tr_gemm_kw<D, 2, KW, DC>(dOs, 0, lane, pba, acc, [&](int step) {
#pragma unroll
                    for (int k = 0; k < KW; k++)
#pragma unroll
                        for (int j = step * 8 / NS; j < (step + 1) * 8 / NS; j++) ppb[k].u[j] = bwd_p_pair<MASK>(sb[k], j, c2, kpos[k], qb);
                });
#pragma unroll
                for (int k = 0; k < KW; k++) {
                    put_slot(slots + (KW + k) * (L::P_SLOT / 4), ppb[k]);
                    pbb[k][0] = operand_of(ppb[k], 0);
                    pbb[k][1] = operand_of(ppb[k], 1);
                }
                lds_tr_gemm_kw<D, 2, KW, DC>(dOs, 32, lane, pbb, acc);
                __builtin_amdgcn_s_setprio(0);
                if (more) lds_store(nbuf);
                tile_barrier();
                par ^= 1;
            };
            static_assert(L::NBUF == 3, "unrolled over three buffers");
            if (MASK) {
                int buf = 0;
                while (more) {
                    p_step(buf);
                    buf = buf == L::NBUF - 1 ? 0 : buf + 1;
                }
            } else {
                for (;;) {
                    p_step(std::integral_constant<int, 0>{});
                    if (!more) break;
                    p_step(std::integral_constant<int, 1>{});
                    if (!more) break;
                    p_step(std::integral_constant<int, 2>{});
                    if (!more) break;
                }
            }
            tile_barrier();                        // step T: only the dS waves have work
        } else {
            bool more = advance(rep, qt);          // step 0: staging duties only
            if (more) gload(rep, qt, 1);
            tile_barrier();
            bool had_next = true;
            auto ds_step = [&](auto buf_tag) {
                const int buf = buf_tag;
                had_next = more;
                if (more) {
                    more = advance(rep, qt);
                    if (more) gload(rep, qt, buf + 2 >= L::NBUF ? buf + 2 - L::NBUF : buf + 2);
                }
                const __bf16 *Qs = (const __bf16 *)(smem + buf * L::BUF_BYTES);
                const __bf16 *dOs = Qs + L::TILE;
                const float *dlt_s = (const float *)(dOs + L::TILE) + BM;
                const unsigned *slots = pslot_base + par * 2 * KW * (L::P_SLOT / 4);
                // the dP accumulators start at -DELTA of their rows (register r <-> tile row 8*(r/4) + 4*hh + r%4);
                // same order as the P wave: dP of a; dP of b with dS of a under its MFMAs; first half of dK with dS of
                // b under its MFMAs; second half of dK
                f32x16 dpa[KW], dpb[KW];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 da = *(const f32x4 *)(dlt_s + 8 * g + 4 * hh), db4 = *(const f32x4 *)(dlt_s + 32 + 8 * g + 4 * hh);
#pragma unroll
                    for (int k = 0; k < KW; k++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            dpa[k][4 * g + e] = da[e];
                            dpb[k][4 * g + e] = db4[e];
                        }
                }
                PackedTile dsa[KW], dsb[KW];
                constexpr int NK = DC / 16, NS = 2 * (DC / 32);   // MFMAs of a chain, of a half of dV / dK
                __builtin_amdgcn_s_setprio(1);
                lds_gemm_chain_kw<D, KW, DC>(dOs + l32 * D, lds_swz<D>(l32) ^ hh, kvreg, dpa);
                unsigned pua[KW][8], pub[KW][8];
#pragma unroll
                for (int k = 0; k < KW; k++) {
                    const unsigned *sl = slots + k * (L::P_SLOT / 4);
                    const uint4 pa0 = *(const uint4 *)(sl + lane * 4), pa1 = *(const uint4 *)(sl + 256 + lane * 4);
                    pua[k][0] = pa0.x; pua[k][1] = pa0.y; pua[k][2] = pa0.z; pua[k][3] = pa0.w;
                    pua[k][4] = pa1.x; pua[k][5] = pa1.y; pua[k][6] = pa1.z; pua[k][7] = pa1.w;
                }
                lds_gemm_chain_kw<D, KW, DC>(dOs + (32 + l32) * D, lds_swz<D>(32 + l32) ^ hh, kvreg, dpb, [&](int kb) {
#pragma unroll
                    for (int k = 0; k < KW; k++)
#pragma unroll
                        for (int j = kb * 8 / NK; j < (kb + 1) * 8 / NK; j++) dsa[k].u[j] = bwd_ds_pair(pua[k][j], dpa[k], j);
                });
                bf16x8 dba[KW][2], dbb[KW][2];
#pragma unroll
                for (int k = 0; k < KW; k++) {
                    const unsigned *sl = slots + (KW + k) * (L::P_SLOT / 4);
                    const uint4 pb0 = *(const uint4 *)(sl + lane * 4), pb1 = *(const uint4 *)(sl + 256 + lane * 4);
                    pub[k][0] = pb0.x; pub[k][1] = pb0.y; pub[k][2] = pb0.z; pub[k][3] = pb0.w;
                    pub[k][4] = pb1.x; pub[k][5] = pb1.y; pub[k][6] = pb1.z; pub[k][7] = pb1.w;
                    dba[k][0] = operand_of(dsa[k], 0);
                    dba[k][1] = operand_of(dsa[k], 1);
                }
                lds_tr_gemm_kw<D, 2, KW, DC>(Qs, 0, lane, dba, acc, [&](int step) {
#pragma unroll
                    for (int k = 0; k < KW; k++)
#pragma unroll
                        for (int j = step * 8 / NS; j < (step + 1) * 8 / NS; j++) dsb[k].u[j] = bwd_ds_pair(pub[k][j], dpb[k], j);
                });
#pragma unroll
                for (int k = 0; k < KW; k++) {
                    dbb[k][0] = operand_of(dsb[k], 0);
                    dbb[k][1] = operand_of(dsb[k], 1);
                }
                lds_tr_gemm_kw<D, 2, KW, DC>(Qs, 32, lane, dbb, acc);
                __builtin_amdgcn_s_setprio(0);
                tile_barrier();
                par ^= 1;
            };
            if (MASK) {
                int buf = 0;
                while (had_next) {
                    ds_step(buf);
                    buf = buf == L::NBUF - 1 ? 0 : buf + 1;
                }
            } else {
                for (;;) {
                    ds_step(std::integral_constant<int, 0>{});
                    if (!had_next) break;
                    ds_step(std::integral_constant<int, 1>{});
                    if (!had_next) break;
                    ds_step(std::integral_constant<int, 2>{});
                    if (!had_next) break;
                }
            }
        }
    };
    if constexpr (PAD) clear_lds<L::P_OFF>(smem);
    run_pass(std::false_type{});
    run_pass(std::true_type{});

    if (p.split_log2) {   // a share of the keys' gradients: stored as it lies in registers, summed by the reduction kernel
        float *const part = p.part + (((((long long)pair * p.tiles_seen + tile) << p.split_log2) + split) * 8 + w) * (KW * 32 * D);
        const float mul = p_role ? 1.f : p.scale;
#pragma unroll
        for (int k = 0; k < KW; k++) store_partial<D>(part + k * 32 * D, lane, acc[k], mul);
        return;
    }
    // dV^T (P wave) / dK^T (dS wave); every wave is past the last barrier: tiles, slots and lists are no longer read
#pragma unroll
    for (int k = 0; k < KW; k++)
        write_key_rows<D, PAD>(smem + w * WaveStage<D>::BYTES, lane, acc[k], p_role ? 1.f : p.scale, uniform32(p.flags & LTR_DKDV_BF16),
                               p_role ? p.chunk[c].dv : p.chunk[c].dk,
                               p_role ? b * p.dvs[0] + hkv * p.dvs[2] : b * p.dks[0] + hkv * p.dks[2], p_role ? p.dvs[1] : p.dks[1],
                               key0 + slice * 32 * KW + 32 * k, sk, cols);
}

template <int D, int KW>
__global__ __launch_bounds__(512) void bwd_dkdv_kernel(const BwdParams p) {
    const int P = p.B * p.Hkv;
    BlockItem item;
    if constexpr (KW == 1) {
        item = block_item(p.kv_map, P);
        if (item.pair >= P) return;
    } else {   // pair after pair on a linear grid: this kernel runs without a mask, and has no scalar registers left for a map (6 % slower)
        int idx = blockIdx.x, rest;
        if ((P & 7) == 0) {
            const int n = p.tiles_seen << p.split_log2;
            item.pair = (idx >> 3) / n * 8 + (idx & 7);
            rest = (idx >> 3) % n;
        } else {
            item.pair = idx % P;
            rest = idx / P;
        }
        item.sub = rest & ((1 << p.split_log2) - 1);
        item.item = rest >> p.split_log2;
    }
    bwd_dkdv_body<D, KW, false>(p, item);
}
template <int D>   // head dims below D
__global__ __launch_bounds__(512) void bwd_dkdv_pad_kernel(const BwdParams p) {
    const BlockItem item = block_item(p.kv_map, p.B * p.Hkv);
    if (item.pair < p.B * p.Hkv) bwd_dkdv_body<D, 1, true>(p, item);
}
template <int D>
__global__ __launch_bounds__(512) void bwd_dkdv_pad_kernel(const Columns96<BwdParams> p) {
    static_assert(D == 128);
    const BlockItem item = block_item(p.kv_map, p.B * p.Hkv);
    if (item.pair < p.B * p.Hkv) bwd_dkdv_body<D, 1, true, false, 96>(p, item);
}

// dK/dV at head dim 64, one wave per 32-key slice: K and V operands (32 registers) and both accumulators (64) fit one wave, so nothing is
// handed over between waves, a block of four waves owns 128 keys in 51 KB of LDS, and two blocks share a CU: one's start, end and barriers run
// under the other's matrix work, which is what bounds bwd_dkdv_kernel<64, 1> on short rows of blocks (16 x 12 heads, causal S=1024:
// 115 us there, 97 here, 82 with the blocks longest first; 32 x 4 heads S=4096: 680 -> 579; the same sums in the same order, bit for
// bit).  1.06 PFLOP/s without a mask at S=4096.  Bound by two waves per SIMD that fill neither pipe: vector active 40 %, matrix 31 % of a
// SIMD's time at S=1024, a wave waits a third of its time for data and barriers and a third for issue.  Three blocks per CU would need 168 registers:
// 21 and more spill, 83 -> 88 us.  Every (row, key) sub-tile of 32 x 32: S and dP in two alternating chains, P and dS in registers,
// dV^T += dO^T P, dK^T += Q^T dS.
template <int D>
struct KeyWaveLds {
    static constexpr int NW = 4, BN = 32 * NW, BM = 64, NT = 64 * NW;
    static constexpr int TILE = BM * D;                                  // elements; rows unpadded, chunks swizzled
    static constexpr int BUF_BYTES = 2 * TILE * 2 + 3 * BM * 4;          // Q, dO, -LSE/scale, -DELTA, row positions (masked tiles)
    static constexpr int MAX_QTILES = BwdLds<D, 1>::MAX_QTILES;
    static constexpr int LIST_OFF = 2 * BUF_BYTES;
    static constexpr int TOTAL = LIST_OFF + 2 * MAX_QTILES * 2 + 16;     // two tile lists (ushort) + counts
    static_assert(TOTAL >= NW * WaveStage<D>::BYTES, "the epilogue's staging areas reuse this memory");
    static_assert(2 * TOTAL <= 160 * 1024, "two blocks per CU");
};
template <int D>
__global__ __launch_bounds__(256, 2) void bwd_dkdv_keywave_kernel(const BwdParams p) {
    using L = KeyWaveLds<D>;
    constexpr int BN = L::BN, BM = L::BM;
    constexpr int CPR = D / 8;
    constexpr int RPI = 64 / CPR;            // rows filled by one wave-wide LDS-direct load (1 KB)
    constexpr int NI = BM / (RPI * L::NW);   // such loads per wave, per tensor and per tile
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool causal = p.flags & LTR_CAUSAL;
    // block -> (batch, kv head, chunk, key tile), shares of a key tile: as in bwd_dkdv_body
    const BlockItem item = block_item(p.kv_map, p.B * p.Hkv);
    const int pair = item.pair, split = item.sub, tile = item.item;
    if (pair >= p.B * p.Hkv) return;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv;
    int c = 0, kt = tile;
    for (; c < p.n_chunks; c++) {
        const int n = seen_tiles(p.chunk[c].sk, p.chunk[c].pos0, p.q_last, BN);
        if (kt < n) break;
        kt -= n;
    }
    if (c >= p.n_chunks) return;
    const int sk = p.chunk[c].sk, pos0 = p.chunk[c].pos0;
    const int key0 = kt * BN, my_key = key0 + 32 * w + l32;
    const bool key_ok = my_key < sk;
    const int kpos = key_ok ? pos0 + my_key : BWD_KPOS_NONE;
    const int tile_kpos_lo = pos0 + key0, w_kpos_lo = tile_kpos_lo + 32 * w;
    const int tile_kpos_hi = pos0 + min(key0 + BN, sk) - 1;
    if (causal) {   // no query of this launch sees the block: nothing to add; results are zero
        int q_lo, q_hi;
        q_pos_range(0, (int)p.Sq - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], q_lo, q_hi);
        if (q_hi < tile_kpos_lo) {
            if ((p.flags & LTR_DKDV_BF16) && key_ok) {
                __bf16 *gv = (__bf16 *)p.chunk[c].dv + b * p.dvs[0] + (long long)my_key * p.dvs[1] + hkv * p.dvs[2];
                __bf16 *gk = (__bf16 *)p.chunk[c].dk + b * p.dks[0] + (long long)my_key * p.dks[1] + hkv * p.dks[2];
                for (int d = 8 * hh; d < D; d += 16) *(uint4 *)(gv + d) = *(uint4 *)(gk + d) = make_uint4(0, 0, 0, 0);
            }
            return;
        }
    }

    // resident B operands: the lane's K and V row, d = 16*kb + 8*hh .. +7
    bf16x8 kreg[D / 16], vreg[D / 16];
    {
        const int ksafe = min(my_key, sk - 1);
        const __bf16 *kp = (const __bf16 *)p.chunk[c].k + b * p.ks[0] + (long long)ksafe * p.ks[1] + hkv * p.ks[2];
        const __bf16 *vp = (const __bf16 *)p.chunk[c].v + b * p.vs[0] + (long long)ksafe * p.vs[1] + hkv * p.vs[2];
#pragma unroll
        for (int kb = 0; kb < D / 16; kb++) {
            uint4 x = *(const uint4 *)(kp + kb * 16 + 8 * hh), y = *(const uint4 *)(vp + kb * 16 + 8 * hh);
            if (!key_ok) x = y = make_uint4(0, 0, 0, 0);
            kreg[kb] = as_bf16x8(x);
            vreg[kb] = as_bf16x8(y);
        }
    }
    f32x16 dkacc[D / 32], dvacc[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) dkacc[i][r] = dvacc[i][r] = 0.f;
    const float c2 = p.scale * LTR_LOG2E;

    unsigned short *const tlist = (unsigned short *)(smem + L::LIST_OFF);     // [2][MAX_QTILES]
    int *const tcount = (int *)(smem + L::LIST_OFF + 2 * L::MAX_QTILES * 2);
    if (w == 0) list_q_tiles<BM, L::MAX_QTILES>(p, lane, split, tile_kpos_lo, tile_kpos_hi, key0 + BN > sk, tlist, tcount);
    __syncthreads();

    // tile transfers and the rows' scalars: see bwd_dkdv_body
    const int st_row = lane / CPR, st_pc = lane % CPR;
    unsigned offq[NI], offdo[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int row = RPI * (NI * w + i) + st_row;
        const int chunk = st_pc ^ lds_swz<D>(row);
        offq[i] = (unsigned)(row * (int)p.qs[1] + chunk * 8);
        offdo[i] = (unsigned)(row * (int)p.dos[1] + chunk * 8);
    }
    const __bf16 *qp_head = nullptr, *dop_head = nullptr;
    const float *sp_head = nullptr;   // LSE (wave 0) or DELTA - BM (wave 1) of the head's rows, indexed by row0 + tid
    const int h_first = hkv * p.n_rep + (split >> p.share_log2) * p.n_reps;   // first of the n_reps q heads this block walks
    auto set_head = [&](int rep) __attribute__((always_inline)) {
        const int h = h_first + rep;
        qp_head = (const __bf16 *)p.q + b * p.qs[0] + h * p.qs[2];
        dop_head = (const __bf16 *)p.d_o + b * p.dos[0] + h * p.dos[2];
        const long long so = ((long long)b * p.Hq + h) * p.Sq;
        sp_head = w == 0 ? p.lse + so : p.delta + so - BM;
    };
    const float st_mul = tid < BM ? -1.f / p.scale : -1.f;   // threads 0..63 stage -LSE/scale, 64..127 -DELTA, 128..191 positions
    float sld = 0.f;      // raw LSE / DELTA value in flight
    bool sld_ok = true;
    int sld_row0 = 0;     // first row of the tile in flight
    // LDS byte addresses of this lane's operands in the first buffer's Q tile and of its scalars; all else is an immediate
    unsigned pa[D / 16], ta[D / 32][2];
    const unsigned lds0 = lds_address(smem), sa = lds0 + 16 * hh;
    {
        const int sw = lds_swz<D>(l32) ^ hh;        // rows l32 + 32 n share the swizzle word of row l32
#pragma unroll
        for (int kb = 0; kb < D / 16; kb++) pa[kb] = lds0 + ((l32 * D + (((2 * kb) ^ sw) << 3)) << 1);
        const int li = lane & 15, g = lane >> 4;
#pragma unroll
        for (int j = 0; j < D / 32; j++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int col = j * 32 + ((g & 1) << 4) + ((li & 3) << 2), row = 4 * (g >> 1) + (li >> 2) + 8 * e;
                ta[j][e] = lds0 + ((lds_swz_off<D>(row, col >> 3) + (col & 7)) << 1);
            }
    }

    auto run_pass = [&](auto mask_tag) {   // unmasked tiles, then masked ones
        constexpr bool MASK = decltype(mask_tag)::value;
        constexpr int list_of = MASK ? 1 : 0;
        const int cnt = __builtin_amdgcn_readfirstlane(tcount[list_of]);
        const unsigned short *const list = tlist + list_of * L::MAX_QTILES;
        int li_ = -1;
        unsigned short pre = list[0];   // the next call's entry, read one call ahead
        auto advance = [&](int &rep, int &qt) {   // next tile of this class after (rep, qt); false when done
            if (++li_ >= cnt) {
                li_ = 0;
                if (++rep >= p.n_reps) return false;
                set_head(rep);
            }
            qt = __builtin_amdgcn_readfirstlane((int)pre);
            pre = list[li_ + 1 < cnt ? li_ + 1 : 0];
            return true;
        };
        auto gload = [&](int qt, int buf) {
            const int row0 = qt * BM;
            sld_row0 = row0;
            const unsigned Qd = lds0 + buf * L::BUF_BYTES, dOd = Qd + L::TILE * 2;
            if (!MASK) {
                const unsigned tq = (unsigned)(row0 * (int)p.qs[1]), tdo = (unsigned)(row0 * (int)p.dos[1]);
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    global_to_lds_b128(qp_head + (unsigned long long)(tq + offq[i]), Qd + RPI * (NI * w + i) * D * 2);
                    global_to_lds_b128(dop_head + (unsigned long long)(tdo + offdo[i]), dOd + RPI * (NI * w + i) * D * 2);
                }
            } else {   // rows past the end repeat the last row (they are masked)
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    const int row = RPI * (NI * w + i) + st_row;
                    const int grow = min(row0 + row, p.Sq - 1);
                    const int chunk = st_pc ^ lds_swz<D>(row);
                    global_to_lds_b128(qp_head + (long long)(grow * (int)p.qs[1] + chunk * 8), Qd + RPI * (NI * w + i) * D * 2);
                    global_to_lds_b128(dop_head + (long long)(grow * (int)p.dos[1] + chunk * 8), dOd + RPI * (NI * w + i) * D * 2);
                }
            }
            if (tid < 2 * BM) {
                const float *sp = sp_head + row0;
                if (!MASK) {
                    sld = sp[tid];
                } else {
                    const int r = tid < BM ? tid : tid - BM;
                    sld_ok = row0 + r < p.Sq;
                    sld = sp[sld_ok ? tid : (tid < BM ? 0 : BM)];
                }
            }
        };
        auto lds_store = [&](int buf) {   // the scalars of the tile that gload fetched last
            float *st = (float *)(smem + buf * L::BUF_BYTES) + L::TILE;
            if (tid < 2 * BM) {
                float x = sld * st_mul;
                if (MASK) x = sld_ok ? x : (tid < BM ? -INFINITY : 0.f);
                st[tid] = x;
            } else if (MASK && tid < 3 * BM) {
                const int row = sld_row0 + tid - 2 * BM;
                ((int *)st)[tid] = row >= p.Sq ? BWD_QPOS_NONE
                                   : causal ? q_position(row, p.q_split, p.q_pos0[0], p.q_pos0[1]) : BWD_QPOS_ALL;
            }
        };
        if (cnt == 0) return;
        int rep = 0, qt = 0;
        set_head(0);
        advance(rep, qt);
        __syncthreads();   // the previous pass has finished reading LDS
        gload(qt, 0);
        lds_store(0);
        tile_barrier();
        // one barrier per tile: tile t+1 streams into the other buffer, whose readers all passed the previous barrier
        bool more = true;
        auto step = [&](auto buf_tag) {
            constexpr int buf = decltype(buf_tag)::value;
            const int row0 = sld_row0;
            more = advance(rep, qt);
            if (more) gload(qt, buf ^ 1);
#pragma unroll
            for (int half = 0; half < 2; half++) {
                if (MASK && causal) {   // no row of the sub-tile sees a key of this wave
                    const int r0 = row0 + 32 * half;
                    if (r0 >= p.Sq) continue;
                    int lo, hi;
                    q_pos_range(r0, min(r0 + 32, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], lo, hi);
                    if (hi < w_kpos_lo) continue;
                }
                constexpr int Q0 = buf * L::BUF_BYTES, DO0 = Q0 + L::TILE * 2;
                const int rows = 32 * half, at = DO0 + L::TILE * 2 + rows * 4;
                // both accumulators start at their rows' scalars (register r <-> row 8*(r/4) + 4*hh + r%4)
                f32x16 s, dp;
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 a = *(lds_f32x4_ptr)(uintptr_t)(sa + at + 32 * g), d4 = *(lds_f32x4_ptr)(uintptr_t)(sa + at + BM * 4 + 32 * g);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        s[4 * g + e] = a[e];
                        dp[4 * g + e] = d4[e];
                    }
                }
                __builtin_amdgcn_s_setprio(1);
                lds_gemm_pair_at<D>(pa, Q0 + rows * D * 2, DO0 + rows * D * 2, kreg, vreg, s, dp);
                __builtin_amdgcn_s_setprio(0);
                PackedTile pt, ds;
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    int qpos[4] = {0, 0, 0, 0};
                    if (MASK) {
                        const i32x4 q4 = *(lds_i32x4_ptr)(uintptr_t)(sa + at + 2 * BM * 4 + 32 * g);
#pragma unroll
                        for (int e = 0; e < 4; e++) qpos[e] = q4[e];
                    }
#pragma unroll
                    for (int j = 2 * g; j < 2 * g + 2; j++) {
                        float p0 = __builtin_amdgcn_exp2f(s[2 * j] * c2), p1 = __builtin_amdgcn_exp2f(s[2 * j + 1] * c2);
                        if (MASK) {
                            p0 = kpos <= qpos[2 * (j & 1)] ? p0 : 0.f;
                            p1 = kpos <= qpos[2 * (j & 1) + 1] ? p1 : 0.f;
                        }
                        pt.u[j] = pack2_bf16(p0, p1);
                        asm("" : "+v"(pt.u[j]));   // or one half of the pair is rounded a second time for dS
                        ds.u[j] = bwd_ds_pair(pt.u[j], dp, j);
                    }
                }
                const bf16x8 pb[2] = {operand_of(pt, 0), operand_of(pt, 1)}, db[2] = {operand_of(ds, 0), operand_of(ds, 1)};
                __builtin_amdgcn_s_setprio(1);
                lds_tr_gemm_at<D, 2>(ta, DO0 + rows * D * 2, pb, dvacc);
                lds_tr_gemm_at<D, 2>(ta, Q0 + rows * D * 2, db, dkacc);
                __builtin_amdgcn_s_setprio(0);
            }
            if (more) lds_store(buf ^ 1);
            tile_barrier();
        };
        for (;;) {
            step(std::integral_constant<int, 0>{});
            if (!more) break;
            step(std::integral_constant<int, 1>{});
            if (!more) break;
        }
    };
    run_pass(std::false_type{});
    run_pass(std::true_type{});

    if (p.split_log2) {   // a share of the keys' gradients, in the layout of bwd_dkdv_body's partials
        float *const part = p.part + (((((long long)pair * p.tiles_seen + tile) << p.split_log2) + split) * 8 + w) * (32 * D);
        store_partial<D>(part, lane, dvacc, 1.f);
        store_partial<D>(part + 4 * 32 * D, lane, dkacc, p.scale);
        return;
    }
    unsigned char *const stage = smem + w * WaveStage<D>::BYTES;   // every wave is past the last barrier
    const bool as_bf16 = uniform32(p.flags & LTR_DKDV_BF16);
    write_key_rows<D, false>(stage, lane, dvacc, 1.f, as_bf16, p.chunk[c].dv, b * p.dvs[0] + hkv * p.dvs[2], p.dvs[1], key0 + 32 * w, sk, D);
    write_key_rows<D, false>(stage, lane, dkacc, p.scale, as_bf16, p.chunk[c].dk, b * p.dks[0] + hkv * p.dks[2], p.dks[1], key0 + 32 * w, sk, D);
}

// Sum of the partial dK / dV that the blocks sharing a key tile left in p.part (bf16 and fp32 kernels alike), in the order of
// the shares: results do not depend on which block finished first.  A wave takes 64 columns of one 32-key slice of dK or dV
// (slots 0-3 of a tile's partials are dV of its four slices, 4-7 dK) and writes them the way the dK/dV kernels do.  Bound:
// the partials' traffic, which was written just before and mostly still lies in L2 / the memory-side cache.
template <int D, int KW>
__global__ __launch_bounds__(256) void bwd_dkdv_reduce_kernel(const BwdParams p) {
    __shared__ __attribute__((aligned(16))) unsigned char stage_mem[4 * WaveStage<64>::BYTES];
    constexpr int BN = 128 * KW, WPT = 8 * KW * (D / 64), BPT = WPT / 4;   // waves and blocks per key tile
    const int lane = threadIdx.x & 63, w4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int idx = blockIdx.x, pair, rest;
    const int P = p.B * p.Hkv;
    if ((P & 7) == 0) {   // the XCD that wrote the partials reads them
        const int j = idx >> 3, n = p.tiles_total * BPT;
        pair = (j / n) * 8 + (idx & 7);
        rest = j % n;
    } else {
        pair = idx % P;
        rest = idx / P;
    }
    const int tile = rest / BPT, item = (rest % BPT) * 4 + w4;
    const int half = item % (D / 64), k = (item / (D / 64)) % KW, slot = item / (D / 64 * KW);
    const bool is_dv = slot < 4;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv;
    int c = 0, kt = tile, first = 0;   // first: tiles with partials in the chunks before
    for (; c < p.n_chunks; c++) {
        const int n = (p.chunk[c].sk + BN - 1) / BN;
        if (kt < n) break;
        kt -= n;
        first += seen_tiles(p.chunk[c].sk, p.chunk[c].pos0, p.q_last, BN);
    }
    if (c >= p.n_chunks) return;
    const int sk = p.chunk[c].sk, key_base = kt * BN + (slot & 3) * 32 * KW + 32 * k;
    const bool out_bf16 = (p.flags & LTR_DKDV_BF16) != 0;
    const bool seen = kt < seen_tiles(sk, p.chunk[c].pos0, p.q_last, BN);   // else: a tile without blocks, nothing but zeros to store
    if (key_base >= sk || (!seen && !out_bf16)) return;
    f32x16 acc[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.f;
    if (seen) {
        const float *src = p.part + ((((long long)pair * p.tiles_seen + first + kt) << p.split_log2) * 8 + slot) * (KW * 32 * D) + k * 32 * D + half * 2048;
        for (int s = 0; s < 1 << p.split_log2; s++, src += 8 * KW * 32 * D)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const f32x4 v = *(const f32x4 *)(src + (i * 64 + lane) * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[i / 4][4 * (i % 4) + e] += v[e];
            }
    }
    const long long stride = is_dv ? p.dvs[1] : p.dks[1];
    const long long off = (is_dv ? b * p.dvs[0] + hkv * p.dvs[2] : b * p.dks[0] + hkv * p.dks[2]) + (key_base + lane / 16) * stride +
                          64 * half + 4 * (lane % 16);
    unsigned char *const stage = stage_mem + w4 * WaveStage<64>::BYTES;
    float *gp = (is_dv ? p.chunk[c].dv : p.chunk[c].dk) + (out_bf16 ? 0 : off);
    __bf16 *gb = (__bf16 *)(is_dv ? p.chunk[c].dv : p.chunk[c].dk) + (out_bf16 ? off : 0);
    wave_tile_rowmajor<64>(stage, lane, acc, 1.f, [&](int row, int col, f32x4 val) {
        if (key_base + row < sk && 64 * half + col < p.cols) {
            if (out_bf16) {
                bf16x4 y;
#pragma unroll
                for (int e = 0; e < 4; e++) y[e] = (__bf16)val[e];
                *(bf16x4 *)gb = y;
            } else {
                const f32x4 old = *(const f32x4 *)gp;
#pragma unroll
                for (int e = 0; e < 4; e++) val[e] += old[e];
                *(f32x4 *)gp = val;
            }
        }
        gp += 4 * stride;
        gb += 4 * stride;
    });
}

// dQ: same block / wave / lane roles as the forward (a lane owns one query row), so LSE and DELTA are
// per-lane scalars.  S^T = K Q^T and dP^T = V dO^T with K, V tiles natural in LDS; dS^T leaves the
// registers as the B operand of dQ^T += K^T dS^T, whose A operand is the K tile read by transpose loads.
// lds_gemm_pair_at / lds_tr_gemm_at for a wave that owns RB 32-row blocks: every operand read from LDS feeds one MFMA per row
// block (ba[rb], bb[rb], ra[rb], rb_[rb] / b[rb], acc[rb] belong to row block rb).
template <int D, int RB, int DC>
__device__ __forceinline__ void lds_gemm_pair_at_rb(const unsigned (&addr)[D / 16], int imm_a, int imm_b, const bf16x8 (&ba)[RB][D / 16],
                                                    const bf16x8 (&bb)[RB][D / 16], f32x16 (&ra)[RB], f32x16 (&rb_)[RB]) {
    constexpr int NK = DC / 16, PF = 2;
    bf16x8 xa[PF + 1], xb[PF + 1];
#pragma unroll
    for (int i = 0; i < PF; i++) {
        xa[i] = *(lds_bf16x8_ptr)(uintptr_t)(addr[i] + imm_a);
        xb[i] = *(lds_bf16x8_ptr)(uintptr_t)(addr[i] + imm_b);
    }
#pragma unroll
    for (int kb = 0; kb < NK; kb++) {
        if (kb + PF < NK) {
            xa[(kb + PF) % (PF + 1)] = *(lds_bf16x8_ptr)(uintptr_t)(addr[kb + PF] + imm_a);
            xb[(kb + PF) % (PF + 1)] = *(lds_bf16x8_ptr)(uintptr_t)(addr[kb + PF] + imm_b);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RB; r++) {
            ra[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[kb % (PF + 1)], ba[r][kb], ra[r], 0, 0, 0);
            rb_[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xb[kb % (PF + 1)], bb[r][kb], rb_[r], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <int D, int NKB, int RB, int DC>
__device__ __forceinline__ void lds_tr_gemm_at_rb(const unsigned (&addr)[D / 32][2], int imm, const bf16x8 (&b)[RB][NKB],
                                                  f32x16 (&acc)[RB][D / 32]) {
    constexpr int ND = DC / 32, N = NKB * ND, PF = 3;
    auto operand = [&](int i) {
        const int off = imm + (i / ND) * 16 * D * 2;
        union {
            struct { i16x4 a, b; } s;
            bf16x8 v;
        } u;
        u.s.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(uintptr_t)(addr[i % ND][0] + off));
        u.s.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(uintptr_t)(addr[i % ND][1] + off));
        return u.v;
    };
    bf16x8 a[PF + 1];
#pragma unroll
    for (int i = 0; i < PF && i < N; i++) a[i] = operand(i);
#pragma unroll
    for (int step = 0; step < N; step++) {
        if (step + PF < N) a[(step + PF) % (PF + 1)] = operand(step + PF);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RB; r++)
            acc[r][step % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[step % (PF + 1)], b[r][step / ND], acc[r][step % ND], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// RB = 32-row blocks per wave: a lane owns RB query rows, a block 256 * RB / KS; KS = key shares per row group as in the forward
template <int D, int RB, int KS, bool PAD, int NW = 8, int BN = FwdTile<D, 1, KS>::BN, int DC = D>
__device__ __forceinline__ void bwd_dq_body(const BwdParams &p, const BlockItem item) {
    const int cols = PAD ? p.cols : D;
    constexpr int RG = NW / KS, BM = 32 * RB * RG;   // the NW waves of the block share every K / V tile
    constexpr int BNT = BN * KS;                     // BN keys per wave, BNT per tile
    constexpr int CPR = D / 8;
    constexpr int RPI = 64 / CPR;            // rows filled by one wave-wide 16-byte-per-lane LDS-direct load (1 KB)
    constexpr int NI = BNT / (RPI * NW);      // such loads per wave, per tensor and per tile
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // two {K tile, V tile} buffers,
    constexpr int TILE = BNT * D;            // rows unpadded, 16-byte chunks XOR-swizzled (lds_swz)
    constexpr int BUF_ELEMS = 2 * TILE;

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = w / KS, ks = w % KS;      // row group and key share of the wave
    const bool causal = p.flags & LTR_CAUSAL;

    const int pair = item.pair, rep = item.sub, slot = item.item;
    if (pair >= p.B * p.Hkv) return;
    const int n_qt = (p.Sq + BM - 1) / BM;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv, h = hkv * p.n_rep + rep;
    // one q tile per block (late tiles first) or a late tile and its early counterpart (see q_tile_slots)
    const bool paired = p.n_slots != n_qt;
    const bool two = paired && slot < n_qt - 1 - slot, early_first = two && (item.order & 1);   // as in the forward kernel
#pragma nounroll
    for (int part = 0; part < 2; part++) {
    const int qt = (part == 0) != early_first ? n_qt - 1 - slot : slot;
    if (part == 1 && !two) break;
    if (part == 1) __syncthreads();   // the first tile's epilogue used the LDS buffers as staging areas
    int lane_of_part = threadIdx.x & 63;   // opaque per tile, see the forward kernel
    asm volatile("" : "+v"(lane_of_part));
    const int lane = lane_of_part, l32 = lane & 31, hh = lane >> 5;

    const int row0 = qt * BM;
    int my_row[RB], my_pos[RB];
    bool row_ok[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        my_row[rb] = row0 + rg * 32 * RB + 32 * rb + l32;
        row_ok[rb] = my_row[rb] < p.Sq;
        my_pos[rb] = q_position(my_row[rb], p.q_split, p.q_pos0[0], p.q_pos0[1]);
    }
    int blk_lo, blk_hi, w_lo, w_hi;
    q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);
    {
        int wr0 = row0 + rg * 32 * RB, wr1 = min(wr0 + 32 * RB, p.Sq) - 1;
        if (wr1 >= wr0) q_pos_range(wr0, wr1, p.q_split, p.q_pos0[0], p.q_pos0[1], w_lo, w_hi);
        else { w_lo = -0x7fffffff; w_hi = -0x7fffffff; }  // wave has no valid row: everything masked
    }

    bf16x8 qreg[RB][D / 16], doreg[RB][D / 16];
    float lse2[RB], dlt[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        lse2[rb] = INFINITY;
        dlt[rb] = 0.f;
        const int rsafe = min(my_row[rb], p.Sq - 1);
        const __bf16 *qp = (const __bf16 *)p.q + b * p.qs[0] + (long long)rsafe * p.qs[1] + h * p.qs[2];
        const __bf16 *dop = (const __bf16 *)p.d_o + b * p.dos[0] + (long long)rsafe * p.dos[1] + h * p.dos[2];
#pragma unroll
        for (int kb = 0; kb < DC / 16; kb++) {
            if (PAD && kb * 16 + 8 * hh >= cols) {
                qreg[rb][kb] = doreg[rb][kb] = as_bf16x8(make_uint4(0, 0, 0, 0));
                continue;
            }
            qreg[rb][kb] = as_bf16x8(*(const uint4 *)(qp + kb * 16 + 8 * hh));
            doreg[rb][kb] = as_bf16x8(*(const uint4 *)(dop + kb * 16 + 8 * hh));
        }
        if (p.flags & LTR_DELTA_FROM_O) {
            // DELTA = rowsum(dO * O) of this lane's row: its half of every 16-element block, then the other half's
            const __bf16 *op = (const __bf16 *)p.o + b * p.os_[0] + (long long)rsafe * p.os_[1] + h * p.os_[2];
            float part = 0.f;
#pragma unroll
            for (int kb = 0; kb < DC / 16; kb++) {
                if (PAD && kb * 16 + 8 * hh >= cols) continue;
                const bf16x8 ov = as_bf16x8(*(const uint4 *)(op + kb * 16 + 8 * hh));
#pragma unroll
                for (int e = 0; e < 8; e++) part += (float)ov[e] * (float)doreg[rb][kb][e];
            }
            dlt[rb] = xhalf_sum(part);
            if (row_ok[rb] && hh == 0 && ks == 0) p.delta[((long long)b * p.Hq + h) * p.Sq + my_row[rb]] = dlt[rb];
        }
        if (row_ok[rb]) {
            // a row that saw no key has LSE = -inf: give it +inf like a row past the end, so that P = exp2(-inf) = 0
            // whatever S is (S = -inf after the mask fix-up would otherwise meet -(-inf))
            const float lse_row = p.lse[((long long)b * p.Hq + h) * p.Sq + my_row[rb]];
            lse2[rb] = lse_row == -INFINITY ? INFINITY : lse_row * LTR_LOG2E;
            if (!(p.flags & LTR_DELTA_FROM_O)) dlt[rb] = p.delta[((long long)b * p.Hq + h) * p.Sq + my_row[rb]];
        }
    }
    f32x16 zero16;
#pragma unroll
    for (int r = 0; r < 16; r++) zero16[r] = 0.f;
    f32x16 dqacc[RB][D / 32];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int i = 0; i < D / 32; i++) dqacc[rb][i] = zero16;
    // the dP^T accumulators start at -DELTA of the lane's row (the first MFMA of the chain takes this as its addend), so
    // dS = P * (dP - DELTA) needs no subtraction per element (one row block per wave only: with two the 16 registers per
    // row block are not there)
    constexpr bool DLT_INIT = RB == 1;
    f32x16 ndlt[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int r = 0; r < 16; r++) ndlt[rb][r] = DLT_INIT ? -dlt[rb] : 0.f;
    const float c2 = p.scale * LTR_LOG2E;

    // The fields of the chunk being loaded live in scalar registers and are re-read from the argument
    // table only when the chunk changes (a scalar load per tile would share the LDS wait counter).
    int c = -1, t = 0, nt = 0;
    int ld_sk = 0, ld_pos0 = 0;
    const __bf16 *ld_kb = nullptr, *ld_vb = nullptr;
    auto settle = [&]() {
        while (c < p.n_chunks && t >= nt) {
            c++;
            t = 0;
            if (c < p.n_chunks) {
                ld_sk = p.chunk[c].sk;
                ld_pos0 = p.chunk[c].pos0;
                ld_kb = (const __bf16 *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
                ld_vb = (const __bf16 *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
                const int nvis = causal ? max(0, min(ld_sk, blk_hi - ld_pos0 + 1)) : ld_sk;
                nt = (nvis + BNT - 1) / BNT;
            }
        }
    };
    settle();

    // Tiles go from global memory straight into LDS (see the forward kernel): wave w fills rows
    // RPI*(NI*w + i) .. with its i-th load; rows past the end of a chunk repeat its last row and are masked.
    const int st_row = lane / CPR, st_pc = lane % CPR;
    int nx_sk = 0, nx_pos0 = 0, nx_key0 = 0;   // the tile in flight: becomes the tile computed next
    auto gload = [&](int ti, int buf) {
        nx_sk = ld_sk;
        nx_pos0 = ld_pos0;
        nx_key0 = ti * BNT;
        const unsigned Kd = lds_address(smem) + buf * BUF_ELEMS * 2, Vd = Kd + TILE * 2;   // LDS byte addresses
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int row = RPI * (NI * w + i) + st_row;
            const int key = min(ti * BNT + row, ld_sk - 1);
            const int chunk = st_pc ^ lds_swz<D>(row);
            if (PAD && chunk * 8 >= cols) continue;
            global_to_lds_b128(ld_kb + (long long)(key * (int)p.ks[1] + chunk * 8), Kd + RPI * (NI * w + i) * D * 2);
            global_to_lds_b128(ld_vb + (long long)(key * (int)p.vs[1] + chunk * 8), Vd + RPI * (NI * w + i) * D * 2);
        }
    };

    bool have = c < p.n_chunks;
    // a block that sees no key of this launch's chunks adds nothing to an fp32 dQ accumulator: no read-modify-write
    if (!have && !(p.flags & LTR_DQ_BF16)) continue;
    if constexpr (PAD) clear_lds<2 * BUF_ELEMS * 2>(smem);
    if (have) gload(t, 0);
    tile_barrier();
    // LDS byte addresses of this lane's operands in the K tile of the current buffer (the V tile and the other 32-key
    // blocks are immediates away): kept in registers and flipped to the other buffer with one XOR each per tile
    static_assert((BUF_ELEMS * 2 & (BUF_ELEMS * 2 - 1)) == 0, "buffer size must be a power of two for the XOR flip");
    unsigned pa[D / 16], ta[D / 32][2];
    {
        const unsigned lds0 = lds_address(smem) + (KS > 1 ? ks * BN * D * 2 : 0);   // the only LDS object of the kernel: aligned far beyond the buffer size
        const int sw = lds_swz<D>(l32) ^ hh;        // rows l32 + 32 n share the swizzle word of row l32
#pragma unroll
        for (int kb = 0; kb < DC / 16; kb++) pa[kb] = lds0 + ((l32 * D + (((2 * kb) ^ sw) << 3)) << 1);
        const int li = lane & 15, g = lane >> 4;
#pragma unroll
        for (int j = 0; j < DC / 32; j++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int col = j * 32 + ((g & 1) << 4) + ((li & 3) << 2), row = 4 * (g >> 1) + (li >> 2) + 8 * e;
                ta[j][e] = lds0 + ((lds_swz_off<D>(row, col >> 3) + (col & 7)) << 1);
            }
    }
    int par = 0;
    while (have) {
        const int sk = nx_sk, pos0 = nx_pos0, key0 = nx_key0 + (KS > 1 ? ks * BN : 0);
        t++;
        settle();
        const bool have_next = c < p.n_chunks;
        if (have_next) gload(t, par ^ 1);

        // 32 keys at a time, one block after the other: one live (S^T, dP^T) tile pair keeps the kernel at two
        // waves per SIMD, and the other wave's MFMAs cover this wave's softmax arithmetic.  A wave whose rows all
        // precede the tile's first key has nothing to add (see the forward kernel).
        if ((!causal || pos0 + key0 <= w_hi) && (KS == 1 || key0 < sk)) {
#pragma unroll
        for (int nb = 0; nb < BN / 32; nb++) {
            // with two row blocks per wave (64 rows) the rest of a diagonal or last tile is left out and whole blocks of one go without a mask: 4 x 16
            // heads of 64, causal S=4096 211 -> 198 us; with one it is 1 - 3 % slower
            if (RB == 2 && nb > 0 && ((causal && pos0 + key0 + nb * 32 > w_hi) || key0 + nb * 32 >= sk)) break;
            const int mask_end = key0 + (RB == 2 ? nb * 32 + 32 : BN);
            const bool need_mask = mask_end > sk || (causal && pos0 + mask_end - 1 > w_lo);
            f32x16 s[RB], dp[RB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                s[rb] = zero16;
                dp[rb] = ndlt[rb];
            }
            __builtin_amdgcn_s_setprio(1);   // MFMA sections run at raised priority, see the forward kernel
            lds_gemm_pair_at_rb<D, RB, DC>(pa, nb * 32 * D * 2, TILE * 2 + nb * 32 * D * 2, qreg, doreg, s, dp);
            __builtin_amdgcn_s_setprio(0);
            // mask fix-up (tail of the chunk, diagonal tiles, rows past the end): wave-uniform branch touching S only;
            // an invisible entry gets S = -inf, so P = 0 and dS = 0
            if (need_mask) {
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    const unsigned bits = row_ok[rb] ? visible_bits(causal, my_pos[rb], pos0, sk, key0 + nb * 32 + 4 * hh) : 0u;
#pragma unroll
                    for (int r = 0; r < 16; r++) s[rb][r] = visible_score(bits, 8 * (r / 4) + r % 4, s[rb][r]);
                }
            }
            bf16x8 dsb[RB][2];
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                PackedTile ds;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    float dsv[2];
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const int r = 2 * j + e;
                        const float pv = __builtin_amdgcn_exp2f(s[rb][r] * c2 - lse2[rb]);
                        dsv[e] = DLT_INIT ? pv * dp[rb][r] : pv * (dp[rb][r] - dlt[rb]);
                    }
                    ds.u[j] = pack2_bf16(dsv[0], dsv[1]);
                }
                dsb[rb][0] = operand_of(ds, 0);
                dsb[rb][1] = operand_of(ds, 1);
            }
            __builtin_amdgcn_s_setprio(1);
            lds_tr_gemm_at_rb<D, 2, RB, DC>(ta, nb * 32 * D * 2, dsb, dqacc);   // every K^T operand feeds one MFMA per row block
            __builtin_amdgcn_s_setprio(0);
        }
        }
        tile_barrier();
#pragma unroll
        for (int kb = 0; kb < DC / 16; kb++) pa[kb] ^= BUF_ELEMS * 2;
#pragma unroll
        for (int j = 0; j < DC / 32; j++) {
            ta[j][0] ^= BUF_ELEMS * 2;
            ta[j][1] ^= BUF_ELEMS * 2;
        }
        par ^= 1;
        have = have_next;
    }

    constexpr int CW = KeyShares<D, KS>::CW;   // columns a wave writes, from column col0 on
    const int col0 = KS > 1 ? ks * CW : 0;
    f32x16 own[CW / 32];                       // KS > 1: those columns, summed over the shares
    if constexpr (KS > 1) {
        static_assert(RB == 1, "key shares are built for one row block per wave");
        collect_shares<D, KS>(smem, w, ks, lane, dqacc[0], 1.f, own);
        __syncthreads();                        // the partials are read: their memory becomes the staging areas
        if (col0 >= D) continue;                // more shares than 32-column groups: nothing left to write
    }
    // dQ in whole rows through the wave's LDS staging area (the tiles are no longer read: the last barrier is behind us)
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        constexpr int LPR = CW / 4, ROWS_PER_IT = 64 / LPR;      // see wave_tile_rowmajor
        unsigned char *stage = smem + w * WaveStage<CW>::BYTES;
        const int Sq_u = uniform32(p.Sq), wave_row0 = uniform32(row0 + rg * 32 * RB + 32 * rb);
        const long long dqs1 = uniform64(p.dqs[1]);
        const long long off0 = uniform64(b * p.dqs[0] + h * p.dqs[2] + col0) + (wave_row0 + lane / LPR) * dqs1 + 4 * (lane % LPR);
        // LTR_ROPE_DQ: q was rotated by the forward's prologue, so the gradient of the caller's un-rotated q is dQ rotated by
        // the conjugate angles of its row's position (the rotation is linear: it commutes with the accumulation over calls)
        const bool rope = uniform32(p.flags & LTR_ROPE_DQ) != 0;
        const float *const rope_tab = p.rope;
        const int rope_p0 = uniform32(p.rope_pos0), split_u = uniform32(p.q_split), qp0 = uniform32(p.q_pos0[0]), qp1 = uniform32(p.q_pos0[1]);
        auto unrotate = [&](int row, int col, f32x4 val) {
            if (!rope) return val;
            const int pos = q_position(wave_row0 + row, split_u, qp0, qp1);
            return rope_conj4(val, *(const f32x4 *)(rope_tab + (long long)(pos - rope_p0) * cols + col0 + col));
        };
        auto &result = [&]() -> f32x16(&)[CW / 32] {
            if constexpr (KS > 1) return own;
            else return dqacc[rb];
        }();
        if (uniform32(p.flags & LTR_DQ_BF16)) {   // this call saw every key of these rows: store the result, no accumulator
            __bf16 *dqp = (__bf16 *)p.dq + off0;
            wave_tile_rowmajor<CW>(stage, lane, result, p.scale, [&](int row, int col, f32x4 val) {
                if (wave_row0 + row < Sq_u && (!PAD || col0 + col < cols)) {
                    val = unrotate(row, col, val);
                    bf16x4 y;
#pragma unroll
                    for (int e = 0; e < 4; e++) y[e] = (__bf16)val[e];
                    *(bf16x4 *)dqp = y;
                }
                dqp += ROWS_PER_IT * dqs1;
            });
        } else {
            float *dqp = (float *)p.dq + off0;
            constexpr int NIT = 32 / ROWS_PER_IT;
            f32x4 old[NIT];   // all reads of the accumulator first, then the adds and the writes
#pragma unroll
            for (int it = 0; it < NIT; it++) {
                old[it] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (wave_row0 + it * ROWS_PER_IT + lane / LPR < Sq_u && (!PAD || col0 + 4 * (lane % LPR) < cols))
                    old[it] = *(const f32x4 *)(dqp + it * ROWS_PER_IT * dqs1);
            }
            int it = 0;
            wave_tile_rowmajor<CW>(stage, lane, result, p.scale, [&](int row, int col, f32x4 val) {
                if (wave_row0 + row < Sq_u && (!PAD || col0 + col < cols)) {
                    val = unrotate(row, col, val);
#pragma unroll
                    for (int e = 0; e < 4; e++) val[e] += old[it][e];
                    *(f32x4 *)dqp = val;
                }
                dqp += ROWS_PER_IT * dqs1;
                it++;
            });
        }
    }
    }   // part
}

template <int D>   // see FourWaves
__global__ __launch_bounds__(256, FourWaves<D>::PER_CU) void bwd_dq_w4_kernel(const BwdParams p) {
    bwd_dq_body<D, 1, 1, false, 4, FourWaves<D>::BN>(p, block_item(p.q_map, p.B * p.Hkv));
}
template <int D, int RB>
__global__ __launch_bounds__(512) void bwd_dq_kernel(const BwdParams p) {
    bwd_dq_body<D, RB, 1, false>(p, block_item(p.q_map, p.B * p.Hkv));
}
template <int D, int KS>
__global__ __launch_bounds__(512) void bwd_dq_shares_kernel(const BwdParams p) {
    bwd_dq_body<D, 1, KS, false>(p, block_item(p.q_map, p.B * p.Hkv));
}
template <int D, int KS>   // head dims below D
__global__ __launch_bounds__(512) void bwd_dq_pad_kernel(const BwdParams p) {
    bwd_dq_body<D, 1, KS, true>(p, block_item(p.q_map, p.B * p.Hkv));
}
template <int D, int KS>
__global__ __launch_bounds__(512) void bwd_dq_pad_kernel(const Columns96<BwdParams> p) {
    static_assert(D == 128);
    bwd_dq_body<D, 1, KS, true, 8, FwdTile<D, 1, KS>::BN, 96>(p, block_item(p.q_map, p.B * p.Hkv));
}

// dQ and dK/dV blocks in one launch (LTR_BWD_JOINT).  Given DELTA, neither kind needs anything of the other; in launches of their own each ends with
// CUs idle and the next begins with all of them waiting for their first tiles, which is what a pass of few blocks spends its time on.  DELTA
// comes from ltr_attn_bwd_delta's launch then (delta_bf16_kernel).  Taken where the modelled time is shorter (joint_launch).  us of the backward, apart -> joint:
//   4 x 12 heads D=64 S=128   17.2 -> 12.0       2 x 16 heads D=96 S=777   57.8 -> 42.5       1 x 32 heads on 8 D=128 S=1237   94.8 -> 78
//   1 x 16 heads D=128 S=4096  257 -> 242        1 x 12 heads D=128 S=3418  181 -> 145        3 x 8 heads D=128 S=926   61 -> 42
// Registers are those of the dK/dV kernel, LDS the larger of both: one block per CU, as for either kind alone.
template <int D, int KS, bool PAD, bool OWN_DELTA = false, int DC = D>
__device__ __forceinline__ void bwd_joint_body(const BwdParams &p) {
    const int P = p.B * p.Hkv;
    const JointItem j = joint_item_at(p.joint, p.q_map, p.kv_map, P, blockIdx.x);
    if (j.item.pair >= P) return;
    if (j.keys) bwd_dkdv_body<D, 1, PAD, OWN_DELTA, DC>(p, j.item);
    else bwd_dq_body<D, 1, KS, PAD, 8, FwdTile<D, 1, KS>::BN, DC>(p, j.item);
}
template <int D, int KS>
__global__ __launch_bounds__(512) void bwd_joint_kernel(const BwdParams p) {
    bwd_joint_body<D, KS, false>(p);
}
template <int D, int KS>   // head dims below D
__global__ __launch_bounds__(512) void bwd_joint_pad_kernel(const BwdParams p) {
    bwd_joint_body<D, KS, true>(p);
}
template <int D, int KS>
__global__ __launch_bounds__(512) void bwd_joint_pad_kernel(const Columns96<BwdParams> p) {
    static_assert(D == 128);
    bwd_joint_body<D, KS, true, false, 96>(p);
}

// the same with DELTA computed by the dK/dV blocks for themselves (own_delta), as the dQ blocks compute theirs: launches of few rows (own_delta_rows)
template <int D>
__global__ __launch_bounds__(512) void bwd_joint_delta_kernel(const BwdParams p) {
    bwd_joint_body<D, 2, false, true>(p);
}
template <int D>
__global__ __launch_bounds__(512) void bwd_joint_delta_pad_kernel(const BwdParams p) {
    bwd_joint_body<D, 2, true, true>(p);
}
template <int D>
__global__ __launch_bounds__(512) void bwd_joint_delta_pad_kernel(const Columns96<BwdParams> p) {
    static_assert(D == 128);
    bwd_joint_body<D, 2, true, true, 96>(p);
}

// ------------------------------------------------------------------------------ backward, fp32
// The fp32 path (1e-4 parity cases, not a performance path): scalar FMAs like fwd_f32_kernel, no atomics.
//   bwd_dq_f32_kernel    one query row per lane (q, dO, dQ in registers), K/V tiles of 32 keys broadcast from LDS
//   bwd_dkdv_f32_kernel  one key per lane, Q/dO tiles of 32 rows (+ LSE, DELTA) broadcast from LDS; two passes so that
//                        the per-lane state fits the register file: DV = false keeps K, V, dK; DV = true keeps K, dV
template <int D>
__global__ __launch_bounds__(64) void bwd_dq_f32_kernel(const BwdParams p) {
    constexpr int BN = 32;
    __shared__ __attribute__((aligned(16))) float Ks[BN * D];
    __shared__ __attribute__((aligned(16))) float Vs[BN * D];
    const int tid = threadIdx.x;
    const bool causal = p.flags & LTR_CAUSAL;
    const int n_qt = (p.Sq + 63) / 64;
    const int qt = n_qt - 1 - (int)(blockIdx.x % n_qt), bh = blockIdx.x / n_qt;
    const int b = bh / p.Hq, h = bh % p.Hq, hkv = h / p.n_rep;
    const int row0 = qt * 64, my_row = row0 + tid;
    const bool row_ok = my_row < p.Sq;
    const int my_pos = q_position(my_row, p.q_split, p.q_pos0[0], p.q_pos0[1]);
    int blk_lo, blk_hi;
    q_pos_range(row0, min(row0 + 64, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);

    // the accumulator covers 64 (D = 128: 32) elements of the head dimension at a time, one pass over the keys each, so that the
    // per-lane state stays inside the register file
    constexpr int DP = D == 128 ? 32 : 64;
    float q[D], dO[D], dq[DP];
    float lse = INFINITY, dlt = 0.f;   // +inf: P = exp(s - inf) = 0 for rows past the end and rows that saw no key
    {
        const int rs = min(my_row, p.Sq - 1);
        const float *qp = (const float *)p.q + b * p.qs[0] + (long long)rs * p.qs[1] + h * p.qs[2];
        const float *dop = (const float *)p.d_o + b * p.dos[0] + (long long)rs * p.dos[1] + h * p.dos[2];
#pragma unroll
        for (int d = 0; d < D; d++) {
            q[d] = qp[d];
            dO[d] = dop[d];
        }
        if (row_ok) {
            const float l = p.lse[((long long)b * p.Hq + h) * p.Sq + my_row];
            lse = l == -INFINITY ? INFINITY : l;
            dlt = p.delta[((long long)b * p.Hq + h) * p.Sq + my_row];
        }
    }
    for (int part = 0; part < D / DP; part++) {
#pragma unroll
    for (int d = 0; d < DP; d++) dq[d] = 0.f;
    for (int c = 0; c < p.n_chunks; c++) {
        const int sk = p.chunk[c].sk, pos0 = p.chunk[c].pos0;
        const int nvis = causal ? max(0, min(sk, blk_hi - pos0 + 1)) : sk;
        const float *kp = (const float *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
        const float *vp = (const float *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
        for (int key0 = 0; key0 < nvis; key0 += BN) {
            __syncthreads();
            for (int i = tid; i < BN * D / 4; i += 64) {
                const int key = key0 + i / (D / 4), dc = i % (D / 4);
                f32x4 kv = {0.f, 0.f, 0.f, 0.f}, vv = {0.f, 0.f, 0.f, 0.f};
                if (key < sk) {
                    kv = *(const f32x4 *)(kp + (long long)key * p.ks[1] + dc * 4);
                    vv = *(const f32x4 *)(vp + (long long)key * p.vs[1] + dc * 4);
                }
                *(f32x4 *)(Ks + i * 4) = kv;
                *(f32x4 *)(Vs + i * 4) = vv;
            }
            __syncthreads();
#pragma unroll 1
            for (int j = 0; j < BN; j++) {
                float s = 0.f, dp = 0.f;
#pragma unroll
                for (int d4 = 0; d4 < D / 4; d4++) {
                    const f32x4 kq = *(const f32x4 *)(Ks + j * D + 4 * d4), vq = *(const f32x4 *)(Vs + j * D + 4 * d4);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        s = fmaf(q[4 * d4 + e], kq[e], s);
                        dp = fmaf(dO[4 * d4 + e], vq[e], dp);
                    }
                    if ((d4 & 7) == 7) asm volatile("" ::: "memory");   // bounds the LDS reads in flight (registers)
                }
                const int key = key0 + j;
                const bool vis = key < sk && (!causal || pos0 + key <= my_pos);
                const float pj = vis ? expf(s * p.scale - lse) : 0.f;
                const float ds = pj * (dp - dlt);
#pragma unroll
                for (int d = 0; d < DP; d++) dq[d] = fmaf(ds, Ks[j * D + part * DP + d], dq[d]);
            }
        }
    }
    if (row_ok) {
        float *dqp = (float *)p.dq + b * p.dqs[0] + (long long)my_row * p.dqs[1] + h * p.dqs[2] + part * DP;
#pragma unroll
        for (int d = 0; d < DP; d++) dqp[d] += dq[d] * p.scale;
    }
    }
}

template <int D, bool DV>
__global__ __launch_bounds__(64) void bwd_dkdv_f32_kernel(const BwdParams p) {
    constexpr int BM = 32;
    __shared__ __attribute__((aligned(16))) float Qs[BM * D];
    __shared__ __attribute__((aligned(16))) float dOs[BM * D];
    __shared__ float lse_s[BM], dlt_s[BM];
    const int tid = threadIdx.x;
    const bool causal = p.flags & LTR_CAUSAL;
    // block -> (batch, kv head, chunk, 64-key tile)
    const int P = p.B * p.Hkv;
    const int pair = blockIdx.x % P;
    int kt = blockIdx.x / P;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv;
    int c = 0;
    for (; c < p.n_chunks; c++) {
        const int n = (p.chunk[c].sk + 63) / 64;
        if (kt < n) break;
        kt -= n;
    }
    if (c >= p.n_chunks) return;
    const int sk = p.chunk[c].sk, pos0 = p.chunk[c].pos0;
    const int my_key = kt * 64 + tid;
    const bool key_ok = my_key < sk;
    const int my_kpos = pos0 + my_key, tile_kpos_lo = pos0 + kt * 64;

    constexpr int DP = D == 128 ? 32 : 64;   // see bwd_dq_f32_kernel
    float k[D], v[DV ? 1 : D], acc[DP];
    {
        const int ks_ = min(my_key, sk - 1);
        const float *kp = (const float *)p.chunk[c].k + b * p.ks[0] + (long long)ks_ * p.ks[1] + hkv * p.ks[2];
        const float *vp = (const float *)p.chunk[c].v + b * p.vs[0] + (long long)ks_ * p.vs[1] + hkv * p.vs[2];
#pragma unroll
        for (int d = 0; d < D; d++) {
            k[d] = kp[d];
            if (!DV) v[d] = vp[d];
        }
    }
    for (int part = 0; part < D / DP; part++) {
#pragma unroll
    for (int d = 0; d < DP; d++) acc[d] = 0.f;
    for (int rep = 0; rep < p.n_rep; rep++) {
        const int h = hkv * p.n_rep + rep;
        const float *qp = (const float *)p.q + b * p.qs[0] + h * p.qs[2];
        const float *dop = (const float *)p.d_o + b * p.dos[0] + h * p.dos[2];
        const long long so = ((long long)b * p.Hq + h) * p.Sq;
        for (int row0 = 0; row0 < p.Sq; row0 += BM) {
            if (causal) {   // no row of the tile sees any key of the block
                int lo, hi;
                q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], lo, hi);
                if (hi < tile_kpos_lo) continue;
            }
            __syncthreads();
            for (int i = tid; i < BM * D / 4; i += 64) {
                const int row = row0 + i / (D / 4), dc = i % (D / 4);
                f32x4 qv = {0.f, 0.f, 0.f, 0.f}, dv = {0.f, 0.f, 0.f, 0.f};
                if (row < p.Sq) {
                    qv = *(const f32x4 *)(qp + (long long)row * p.qs[1] + dc * 4);
                    dv = *(const f32x4 *)(dop + (long long)row * p.dos[1] + dc * 4);
                }
                *(f32x4 *)(Qs + i * 4) = qv;
                *(f32x4 *)(dOs + i * 4) = dv;
            }
            if (tid < BM) {
                const int row = row0 + tid;
                const float l = row < p.Sq ? p.lse[so + row] : INFINITY;
                lse_s[tid] = l == -INFINITY ? INFINITY : l;     // +inf: P = 0
                dlt_s[tid] = row < p.Sq ? p.delta[so + row] : 0.f;
            }
            __syncthreads();
#pragma unroll 1
            for (int i = 0; i < BM; i++) {
                float s = 0.f, dp = 0.f;
#pragma unroll
                for (int d4 = 0; d4 < D / 4; d4++) {
                    const f32x4 qq = *(const f32x4 *)(Qs + i * D + 4 * d4);
                    f32x4 oq = {0.f, 0.f, 0.f, 0.f};
                    if (!DV) oq = *(const f32x4 *)(dOs + i * D + 4 * d4);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        s = fmaf(k[4 * d4 + e], qq[e], s);
                        if (!DV) dp = fmaf(v[4 * d4 + e], oq[e], dp);
                    }
                    if ((d4 & 7) == 7) asm volatile("" ::: "memory");   // bounds the LDS reads in flight (registers)
                }
                const int qpos = q_position(row0 + i, p.q_split, p.q_pos0[0], p.q_pos0[1]);
                const bool vis = key_ok && (!causal || my_kpos <= qpos);
                const float pi = vis ? expf(s * p.scale - lse_s[i]) : 0.f;
                if (DV) {
#pragma unroll
                    for (int d = 0; d < DP; d++) acc[d] = fmaf(pi, dOs[i * D + part * DP + d], acc[d]);
                } else {
                    const float ds = pi * (dp - dlt_s[i]);
#pragma unroll
                    for (int d = 0; d < DP; d++) acc[d] = fmaf(ds, Qs[i * D + part * DP + d], acc[d]);
                }
            }
        }
    }
    if (key_ok) {
        float *gp = (DV ? p.chunk[c].dv + b * p.dvs[0] + (long long)my_key * p.dvs[1] + hkv * p.dvs[2]
                        : p.chunk[c].dk + b * p.dks[0] + (long long)my_key * p.dks[1] + hkv * p.dks[2]) + part * DP;
        const float mul = DV ? 1.f : p.scale;
#pragma unroll
        for (int d = 0; d < DP; d++) gp[d] += acc[d] * mul;
    }
    }
}

// ------------------------------------------------------------------------------ backward, fp32 on the matrix pipe
// The recompute backward of the fp32 path on v_mfma_f32_32x32x2_f32, in the shapes of fwd_f32_mfma_kernel (same LDS-direct
// swizzled fp32 tiles, same choice of contraction order so that no operand moves), no atomics:
//   bwd_dq_f32_mfma_kernel<D, KS>   4 waves, a wave owns 32 query rows (lane = row; Q, dO operands in registers) and one of
//                        KS key shares: S^T = K Q^T and dP^T = V dO^T (accumulators start at -DELTA), dS^T = P (dP - DELTA)
//                        in registers, dQ^T += K^T dS^T with the accumulator register as the step's operand; the KS partial
//                        dQ of a row group are summed through LDS; dQ is added to the fp32 accumulator in whole rows, or, with
//                        LTR_DQ_F32_RESULT, stored, and DELTA of the block's rows is computed from O in the prologue and left for the
//                        dK/dV kernel: no DELTA launch, no fill of dQ (B=2, 8 heads of 64, 256 rows: launches of 3 us each).
//   bwd_dkdv_f32_mfma_kernel<D>     4 waves, a wave owns 32 keys (lane = key; K, V operands and the dK^T, dV^T accumulators
//                        in registers: one wave per SIMD), the block loops over the group's query heads and over 32-row
//                        Q / dO tiles in double-buffered LDS: S = Q K^T, dP = dO V^T (accumulators start at -DELTA of
//                        their rows), P and dS in registers, dV^T += dO^T P, dK^T += Q^T dS.
template <int D, int KS>
__device__ __forceinline__ void bwd_dq_f32_body(const BwdParams &p) {
    using L = F32Mfma<D, KS>;
    constexpr int NW = L::NW, RG = L::RG, BM = L::BM, BN = L::BN, TILE = L::TILE;
    constexpr int CPR = D / 4, RPI = 64 / CPR, NI = BN / (RPI * NW);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = w / KS, ks = w % KS;
    const bool causal = p.flags & LTR_CAUSAL, result = p.flags & LTR_DQ_F32_RESULT;
    const int n_qt = (p.Sq + BM - 1) / BM;
    const int idx = blockIdx.x;
    const int qt = n_qt - 1 - idx / (p.B * p.Hq);
    const int bh = idx % (p.B * p.Hq);
    const int b = bh / p.Hq, h = bh % p.Hq, hkv = h / p.n_rep;
    const int row0 = qt * BM, my_row = row0 + rg * 32 + l32;
    const bool row_ok = my_row < p.Sq;
    const int my_pos = q_position(my_row, p.q_split, p.q_pos0[0], p.q_pos0[1]);
    int blk_lo, blk_hi, w_lo, w_hi;
    q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);
    {
        const int wr0 = row0 + rg * 32, wr1 = min(wr0 + 32, p.Sq) - 1;
        if (wr1 >= wr0) q_pos_range(wr0, wr1, p.q_split, p.q_pos0[0], p.q_pos0[1], w_lo, w_hi);
        else { w_lo = 0x7fffffff; w_hi = -0x7fffffff; }
    }
    // operands of the lane's row: qreg[4g + j] = Q[row][8g + 4h + j], doreg likewise
    float qreg[D / 2], doreg[D / 2];
    float lse2 = INFINITY, dlt = 0.f;   // +inf: P = exp2(s - inf) = 0 for rows past the end and rows that saw no key
    {
        const int rs = min(my_row, p.Sq - 1);
        const float *qp = (const float *)p.q + b * p.qs[0] + (long long)rs * p.qs[1] + h * p.qs[2];
        const float *dop = (const float *)p.d_o + b * p.dos[0] + (long long)rs * p.dos[1] + h * p.dos[2];
#pragma unroll
        for (int g = 0; g < D / 8; g++) {
            const f32x4 x = *(const f32x4 *)(qp + 8 * g + 4 * hh), y = *(const f32x4 *)(dop + 8 * g + 4 * hh);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                qreg[4 * g + j] = x[j];
                doreg[4 * g + j] = y[j];
            }
        }
        if (row_ok) {
            const float lse_row = p.lse[((long long)b * p.Hq + h) * p.Sq + my_row];
            lse2 = lse_row == -INFINITY ? INFINITY : lse_row * LTR_LOG2E;
            if (!result) dlt = p.delta[((long long)b * p.Hq + h) * p.Sq + my_row];
        }
        if (result) {   // the two lanes of a row hold its column groups in turn: 16 sums of D / 16 terms in all, as in delta_kernel
            const float *op = (const float *)p.o + b * p.os_[0] + (long long)rs * p.os_[1] + h * p.os_[2];
            float sum[8];
#pragma unroll
            for (int i = 0; i < 8; i++) sum[i] = 0.f;
#pragma unroll
            for (int g = 0; g < D / 8; g++) {
                const f32x4 x = *(const f32x4 *)(op + 8 * g + 4 * hh);
#pragma unroll
                for (int j = 0; j < 4; j++) sum[(g & 1) * 4 + j] = fmaf(x[j], doreg[4 * g + j], sum[(g & 1) * 4 + j]);
            }
            const float part = xhalf_sum(((sum[0] + sum[1]) + (sum[2] + sum[3])) + ((sum[4] + sum[5]) + (sum[6] + sum[7])));
            if (row_ok) dlt = part;
            if (row_ok && hh == 0 && ks == 0) p.delta[((long long)b * p.Hq + h) * p.Sq + my_row] = part;
        }
    }
    f32x16 dqacc[D / 32], ndlt;
#pragma unroll
    for (int r = 0; r < 16; r++) ndlt[r] = -dlt;
#pragma unroll
    for (int i = 0; i < D / 32; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) dqacc[i][r] = 0.f;
    const float c2 = p.scale * LTR_LOG2E;

    int c = -1, t = 0, nt = 0;
    int ld_sk = 0, ld_pos0 = 0;
    const float *ld_kb = nullptr, *ld_vb = nullptr;
    auto settle = [&]() {
        while (c < p.n_chunks && t >= nt) {
            c++;
            t = 0;
            if (c < p.n_chunks) {
                ld_sk = p.chunk[c].sk;
                ld_pos0 = p.chunk[c].pos0;
                ld_kb = (const float *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
                ld_vb = (const float *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
                const int nvis = causal ? max(0, min(ld_sk, blk_hi - ld_pos0 + 1)) : ld_sk;
                nt = (nvis + BN - 1) / BN;
            }
        }
    };
    settle();
    const int st_row = lane / CPR, st_pc = lane % CPR;
    int nx_sk = 0, nx_pos0 = 0, nx_key0 = 0;
    auto gload = [&](int ti, int buf) {
        nx_sk = ld_sk;
        nx_pos0 = ld_pos0;
        nx_key0 = ti * BN;
        const unsigned Kd = lds_address(smem) + buf * L::BUF_BYTES, Vd = Kd + TILE * 4;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int row = RPI * (NI * w + i) + st_row;
            const int key = min(ti * BN + row, ld_sk - 1);
            const int chunk = st_pc ^ f32_swz(row);
            global_to_lds_b128(ld_kb + ((long long)key * p.ks[1] + chunk * 4), Kd + RPI * (NI * w + i) * D * 4);
            global_to_lds_b128(ld_vb + ((long long)key * p.vs[1] + chunk * 4), Vd + RPI * (NI * w + i) * D * 4);
        }
    };
    bool have = c < p.n_chunks;
    if (!have && !result) return;   // no visible key: nothing to add to the accumulator (block-uniform)
    if (have) gload(t, 0);
    tile_barrier();
    int par = 0;
    while (have) {
        const int sk = nx_sk, pos0 = nx_pos0, key0 = nx_key0 + 32 * ks;
        const float *Ks = (const float *)(smem + par * L::BUF_BYTES) + 32 * ks * D, *Vs = Ks + TILE;
        t++;
        settle();
        const bool have_next = c < p.n_chunks;
        if (have_next) gload(t, par ^ 1);
        if (key0 < sk && (!causal || pos0 + key0 <= w_hi)) {
            f32x16 s, dp = ndlt;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.f;
            const float *krow = Ks + l32 * D, *vrow_ = Vs + l32 * D;
            const int ksw = f32_swz(l32);
#pragma unroll
            for (int g = 0; g < D / 8; g++) {
                const f32x4 kx = *(const f32x4 *)(krow + (((2 * g + hh) ^ ksw) << 2));
                const f32x4 vx = *(const f32x4 *)(vrow_ + (((2 * g + hh) ^ ksw) << 2));
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[j], qreg[4 * g + j], s, 0, 0, 0);
                    dp = __builtin_amdgcn_mfma_f32_32x32x2f32(vx[j], doreg[4 * g + j], dp, 0, 0, 0);
                }
            }
            const bool need_mask = (key0 + 32 > sk) || (causal && (pos0 + key0 + 31 > w_lo));
#pragma unroll
            for (int r = 0; r < 16; r++) {
                float pv = __builtin_amdgcn_exp2f(s[r] * c2 - lse2);
                if (need_mask) {
                    const int key = key0 + 8 * (r / 4) + 4 * hh + (r % 4);
                    const bool vis = key < sk && row_ok && (!causal || pos0 + key <= my_pos);
                    pv = vis ? pv : 0.f;
                }
                s[r] = pv * dp[r];          // dS^T, key 8 (r / 4) + 4h + r % 4 of the sub-tile
            }
            // dQ^T += K^T dS^T: step r contracts the key of accumulator register r; lane (d = 32 db + l32, h) reads K[key][d]
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int krow_i = 8 * (r / 4) + 4 * hh + (r % 4);
                const float *kr = Ks + krow_i * D + (l32 & 3);
                const int sw = f32_swz(krow_i);
#pragma unroll
                for (int db = 0; db < D / 32; db++) {
                    const float kx = kr[((8 * db + (l32 >> 2)) ^ sw) << 2];
                    dqacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx, s[r], dqacc[db], 0, 0, 0);
                }
            }
        }
        tile_barrier();
        par ^= 1;
        have = have_next;
    }
    // sum of the KS partial dQ of a row group
    if constexpr (KS > 1) {
        float *part = (float *)(smem + L::PART_OFF);
        if (ks > 0) {
            float *mine = part + (size_t)(rg * (KS - 1) + ks - 1) * (L::PART_BYTES / 4);
#pragma unroll
            for (int i = 0; i < D / 32; i++)
#pragma unroll
                for (int r4 = 0; r4 < 4; r4++) {
                    f32x4 x;
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] = dqacc[i][4 * r4 + e];
                    *(f32x4 *)(mine + ((i * 4 + r4) * 64 + lane) * 4) = x;
                }
        }
        __syncthreads();
        if (ks > 0) return;
        for (int k2 = 1; k2 < KS; k2++) {
            const float *other = part + (size_t)(rg * (KS - 1) + k2 - 1) * (L::PART_BYTES / 4);
#pragma unroll
            for (int i = 0; i < D / 32; i++)
#pragma unroll
                for (int r4 = 0; r4 < 4; r4++) {
                    const f32x4 x = *(const f32x4 *)(other + ((i * 4 + r4) * 64 + lane) * 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) dqacc[i][4 * r4 + e] += x[e];
                }
        }
    }
    unsigned char *stage = smem + L::STAGE_OFF + rg * WaveStage<D>::BYTES;
    constexpr int LPR = D / 4, ROWS_PER_IT = 64 / LPR;
    const int wave_row0 = row0 + rg * 32, Sq = p.Sq;
    const long long dqs1 = p.dqs[1];
    float *dqp = (float *)p.dq + b * p.dqs[0] + h * p.dqs[2] + (long long)(wave_row0 + lane / LPR) * dqs1 + 4 * (lane % LPR);
    wave_tile_rowmajor<D>(stage, lane, dqacc, p.scale, [&](int row, int, f32x4 val) {
        if (wave_row0 + row < Sq) {
            if (!result) {
                const f32x4 old = *(const f32x4 *)dqp;
#pragma unroll
                for (int e = 0; e < 4; e++) val[e] += old[e];
            }
            *(f32x4 *)dqp = val;
        }
        dqp += ROWS_PER_IT * dqs1;
    });
}

template <int D, int KS>
__global__ __launch_bounds__(256) void bwd_dq_f32_mfma_kernel(const BwdParams p) {
    bwd_dq_f32_body<D, KS>(p);
}
template <int D, int KS>
__global__ __launch_bounds__(256) void bwd_dq_f32_rows32_kernel(const BwdParams p) {
    bwd_dq_f32_body<D, KS>(p);
}
template <>
__global__ __launch_bounds__(256) void bwd_dq_f32_mfma_kernel<64, 4>(const BwdParams p) {   // see F32Rows16
    using L = F32Mfma<64, 4>;
    constexpr int D = 64, BM = F32Rows16::BM, BN = L::BN, TILE = L::TILE;
    constexpr int CPR = D / 4, RPI = 64 / CPR, NI = BN / (RPI * L::NW);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
    const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool causal = p.flags & LTR_CAUSAL, result = p.flags & LTR_DQ_F32_RESULT;
    const int n_qt = (p.Sq + BM - 1) / BM;
    const int qt = n_qt - 1 - blockIdx.x / (p.B * p.Hq);
    const int bh = blockIdx.x % (p.B * p.Hq);
    const int b = bh / p.Hq, h = bh % p.Hq, hkv = h / p.n_rep;
    const int row0 = qt * BM, my_row = row0 + i;
    const bool row_ok = my_row < p.Sq;
    const int my_pos = q_position(my_row, p.q_split, p.q_pos0[0], p.q_pos0[1]);
    int blk_lo, blk_hi;
    q_pos_range(row0, min(row0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], blk_lo, blk_hi);
    float qreg[16], doreg[16];
    float lse2 = INFINITY, dlt = 0.f;   // +inf: P = exp2(s - inf) = 0 for rows past the end and rows that saw no key
    {
        const int rs = min(my_row, p.Sq - 1);
        const long long so = ((long long)b * p.Hq + h) * p.Sq + my_row;
        rows16_operand((const float *)p.q + b * p.qs[0] + (long long)rs * p.qs[1] + h * p.qs[2], g, qreg);
        rows16_operand((const float *)p.d_o + b * p.dos[0] + (long long)rs * p.dos[1] + h * p.dos[2], g, doreg);
        if (row_ok) {
            const float lse_row = p.lse[so];
            lse2 = lse_row == -INFINITY ? INFINITY : lse_row * LTR_LOG2E;
            if (!result) dlt = p.delta[so];
        }
        if (result) {   // the four lanes of a row: 16 sums of D / 16 terms in all, as in delta_kernel
            float oreg[16], sum[4];
            rows16_operand((const float *)p.o + b * p.os_[0] + (long long)rs * p.os_[1] + h * p.os_[2], g, oreg);
#pragma unroll
            for (int j = 0; j < 4; j++) sum[j] = 0.f;
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int j = 0; j < 4; j++) sum[j] = fmaf(oreg[4 * s + j], doreg[4 * s + j], sum[j]);
            const float part = quarter_sum((sum[0] + sum[1]) + (sum[2] + sum[3]));
            if (row_ok) dlt = part;
            if (row_ok && g == 0 && ks == 0) p.delta[so] = part;
        }
    }
    f32x4 dqacc[4];
#pragma unroll
    for (int db = 0; db < 4; db++) dqacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float c2 = p.scale * LTR_LOG2E;

    int c = -1, t = 0, nt = 0;
    int ld_sk = 0, ld_pos0 = 0;
    const float *ld_kb = nullptr, *ld_vb = nullptr;
    auto settle = [&]() {
        while (c < p.n_chunks && t >= nt) {
            c++;
            t = 0;
            if (c < p.n_chunks) {
                ld_sk = p.chunk[c].sk;
                ld_pos0 = p.chunk[c].pos0;
                ld_kb = (const float *)p.chunk[c].k + b * p.ks[0] + hkv * p.ks[2];
                ld_vb = (const float *)p.chunk[c].v + b * p.vs[0] + hkv * p.vs[2];
                const int nvis = causal ? max(0, min(ld_sk, blk_hi - ld_pos0 + 1)) : ld_sk;
                nt = (nvis + BN - 1) / BN;
            }
        }
    };
    settle();
    const int st_row = lane / CPR, st_pc = lane % CPR;
    int nx_sk = 0, nx_pos0 = 0, nx_key0 = 0;
    auto gload = [&](int ti, int buf) {
        nx_sk = ld_sk;
        nx_pos0 = ld_pos0;
        nx_key0 = ti * BN;
        const unsigned Kd = lds_address(smem) + buf * L::BUF_BYTES, Vd = Kd + TILE * 4;
#pragma unroll
        for (int n = 0; n < NI; n++) {
            const int row = RPI * (NI * ks + n) + st_row;
            const int key = min(ti * BN + row, ld_sk - 1);
            const int chunk = st_pc ^ f32_swz(row);
            global_to_lds_b128(ld_kb + ((long long)key * p.ks[1] + chunk * 4), Kd + RPI * (NI * ks + n) * D * 4);
            global_to_lds_b128(ld_vb + ((long long)key * p.vs[1] + chunk * 4), Vd + RPI * (NI * ks + n) * D * 4);
        }
    };
    bool have = c < p.n_chunks;
    if (!have && !result) return;   // no visible key: nothing to add to the accumulator (block-uniform)
    if (have) gload(t, 0);
    tile_barrier();
    int par = 0;
    while (have) {
        const int sk = nx_sk, pos0 = nx_pos0, key0 = nx_key0 + 32 * ks;
        const float *Ks = (const float *)(smem + par * L::BUF_BYTES) + 32 * ks * D, *Vs = Ks + TILE;
        t++;
        settle();
        const bool have_next = c < p.n_chunks;
        if (have_next) gload(t, par ^ 1);
        if (key0 < sk && (!causal || pos0 + key0 <= blk_hi)) {
            f32x4 s[2], dp[2];
            s[0] = s[1] = f32x4{0.f, 0.f, 0.f, 0.f};
            dp[0] = dp[1] = f32x4{-dlt, -dlt, -dlt, -dlt};
            rows16_scores(Ks, i, g, qreg, s);
            rows16_scores(Vs, i, g, doreg, dp);
            const bool need_mask = (key0 + 32 > sk) || (causal && (pos0 + key0 + 31 > blk_lo));
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float pv = __builtin_amdgcn_exp2f(s[kb][r] * c2 - lse2);
                    if (need_mask) {
                        const int key = key0 + 16 * kb + 4 * g + r;
                        const bool vis = key < sk && row_ok && (!causal || pos0 + key <= my_pos);
                        pv = vis ? pv : 0.f;
                    }
                    s[kb][r] = pv * dp[kb][r];
                }
            rows16_weighted(Ks, i, g, s, dqacc);
        }
        tile_barrier();
        par ^= 1;
        have = have_next;
    }
    const f32x4 own = rows16_collect(smem, ks, lane, dqacc, 1.f);
    if (!row_ok) return;
    float *dqp = (float *)p.dq + b * p.dqs[0] + h * p.dqs[2] + (long long)my_row * p.dqs[1] + 16 * ks + 4 * g;
    f32x4 val;
#pragma unroll
    for (int e = 0; e < 4; e++) val[e] = own[e] * p.scale;
    if (!result) {
        const f32x4 old = *(const f32x4 *)dqp;
#pragma unroll
        for (int e = 0; e < 4; e++) val[e] += old[e];
    }
    *(f32x4 *)dqp = val;
}

template <int D>
struct F32DkdvLds {
    static constexpr int TILE = 32 * D;                          // floats per Q (or dO) tile of 32 rows
    static constexpr int BUF_BYTES = 2 * TILE * 4 + 3 * 32 * 4;  // Q, dO, LSE * log2(e), -DELTA, row positions
    static constexpr int STAGE_BYTES = 4 * WaveStage<D>::BYTES;
    static constexpr int LDS = 2 * BUF_BYTES > STAGE_BYTES ? 2 * BUF_BYTES : STAGE_BYTES;
};

template <int D>
__global__ __launch_bounds__(256) void bwd_dkdv_f32_mfma_kernel(const BwdParams p) {
    using L = F32DkdvLds<D>;
    constexpr int BN = 128, BM = 32, TILE = L::TILE;
    constexpr int CPR = D / 4, RPI = 64 / CPR, NI = BM / (RPI * 4);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool causal = p.flags & LTR_CAUSAL;
    // block -> (batch, kv head, chunk, 128-key tile)
    const int P = p.B * p.Hkv;
    const int pair = blockIdx.x % P, rest = blockIdx.x / P;
    const int step = 1 << p.split_log2;                            // blocks that share a key tile take every step-th q tile
    const int split = rest & (step - 1), tile = rest >> p.split_log2;
    int c = 0, kt = tile;
    for (; c < p.n_chunks; c++) {
        const int n = seen_tiles(p.chunk[c].sk, p.chunk[c].pos0, p.q_last, BN);
        if (kt < n) break;
        kt -= n;
    }
    if (c >= p.n_chunks) return;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv;
    const int sk = p.chunk[c].sk, pos0 = p.chunk[c].pos0;
    const int key0 = kt * BN, my_key = key0 + 32 * w + l32;
    const bool key_ok = my_key < sk;
    const int kpos = key_ok ? pos0 + my_key : BWD_KPOS_NONE;
    const int blk_kpos_lo = pos0 + key0, w_kpos_lo = pos0 + key0 + 32 * w;
    if (causal) {   // no query of this launch sees the block
        int q_lo, q_hi;
        q_pos_range(0, (int)p.Sq - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], q_lo, q_hi);
        if (q_hi < blk_kpos_lo) return;
    }
    // operands of the lane's key: kreg[4g + j] = K[key][8g + 4h + j], vreg likewise
    float kreg[D / 2], vreg[D / 2];
    {
        const int ksafe = min(my_key, sk - 1);
        const float *kp = (const float *)p.chunk[c].k + b * p.ks[0] + (long long)ksafe * p.ks[1] + hkv * p.ks[2];
        const float *vp = (const float *)p.chunk[c].v + b * p.vs[0] + (long long)ksafe * p.vs[1] + hkv * p.vs[2];
#pragma unroll
        for (int g = 0; g < D / 8; g++) {
            f32x4 x = *(const f32x4 *)(kp + 8 * g + 4 * hh), y = *(const f32x4 *)(vp + 8 * g + 4 * hh);
            if (!key_ok) x = y = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                kreg[4 * g + j] = x[j];
                vreg[4 * g + j] = y[j];
            }
        }
    }
    f32x16 dkacc[D / 32], dvacc[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) dkacc[i][r] = dvacc[i][r] = 0.f;
    const float c2 = p.scale * LTR_LOG2E;

    // walk over (query head of the group, 32-row q tile); tiles none of whose rows sees a key of the block are skipped
    const int n_qt = (p.Sq + BM - 1) / BM, total = p.n_rep * n_qt;
    auto visible = [&](int it) {
        if (!causal) return true;
        const int r0 = (it % n_qt) * BM;
        int lo, hi;
        q_pos_range(r0, min(r0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], lo, hi);
        return hi >= blk_kpos_lo;
    };
    auto next_visible = [&](int it) {
        while (it < total && !visible(it)) it += step;
        return it;
    };
    const int st_row = lane / CPR, st_pc = lane % CPR;
    auto gload = [&](int it, int buf) {
        const int rep = it / n_qt, r0 = (it % n_qt) * BM, h = hkv * p.n_rep + rep;
        const float *qp = (const float *)p.q + b * p.qs[0] + h * p.qs[2];
        const float *dop = (const float *)p.d_o + b * p.dos[0] + h * p.dos[2];
        const unsigned Qd = lds_address(smem) + buf * L::BUF_BYTES, dOd = Qd + TILE * 4;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int row = RPI * (NI * w + i) + st_row;
            const int grow = min(r0 + row, p.Sq - 1);
            const int chunk = st_pc ^ f32_swz(row);
            global_to_lds_b128(qp + ((long long)grow * p.qs[1] + chunk * 4), Qd + RPI * (NI * w + i) * D * 4);
            global_to_lds_b128(dop + ((long long)grow * p.dos[1] + chunk * 4), dOd + RPI * (NI * w + i) * D * 4);
        }
        // per-row scalars of the tile: LSE * log2(e) (+inf for rows past the end or without a visible key), -DELTA, position
        float *st = (float *)(smem + buf * L::BUF_BYTES) + 2 * TILE;
        if (tid < 96) {
            const int r = tid & 31, row = r0 + r;
            const bool ok = row < p.Sq;
            const long long so = ((long long)b * p.Hq + h) * p.Sq + min(row, p.Sq - 1);
            if (tid < 32) {
                const float l = p.lse[so];
                st[r] = (!ok || l == -INFINITY) ? INFINITY : l * LTR_LOG2E;
            } else if (tid < 64) {
                st[32 + r] = ok ? -p.delta[so] : 0.f;
            } else {
                ((int *)st)[64 + r] = !ok ? BWD_QPOS_NONE : causal ? q_position(row, p.q_split, p.q_pos0[0], p.q_pos0[1]) : BWD_QPOS_ALL;
            }
        }
    };
    int it = next_visible(split);
    if (it < total) gload(it, 0);
    tile_barrier();
    int par = 0;
    while (it < total) {
        const int nxt = next_visible(it + step);
        if (nxt < total) gload(nxt, par ^ 1);
        const float *Qs = (const float *)(smem + par * L::BUF_BYTES), *dOs = Qs + TILE;
        const float *st = dOs + TILE;
        // a wave whose 32 keys no row of the tile sees has nothing to add
        int lo, hi;
        {
            const int r0 = (it % n_qt) * BM;
            q_pos_range(r0, min(r0 + BM, p.Sq) - 1, p.q_split, p.q_pos0[0], p.q_pos0[1], lo, hi);
        }
        if (!causal || hi >= w_kpos_lo) {
            f32x16 s, dp;
            float lse2[16];
            int qpos[16];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const f32x4 a = *(const f32x4 *)(st + 8 * g + 4 * hh), d4 = *(const f32x4 *)(st + 32 + 8 * g + 4 * hh);
                const i32x4 q4 = *(const i32x4 *)((const int *)st + 64 + 8 * g + 4 * hh);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    lse2[4 * g + e] = a[e];
                    dp[4 * g + e] = d4[e];      // the dP accumulator starts at -DELTA of its row
                    qpos[4 * g + e] = q4[e];
                    s[4 * g + e] = 0.f;
                }
            }
            const float *qrow = Qs + l32 * D, *dorow = dOs + l32 * D;
            const int rsw = f32_swz(l32);
#pragma unroll
            for (int g = 0; g < D / 8; g++) {
                const f32x4 qx = *(const f32x4 *)(qrow + (((2 * g + hh) ^ rsw) << 2));
                const f32x4 dx = *(const f32x4 *)(dorow + (((2 * g + hh) ^ rsw) << 2));
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(qx[j], kreg[4 * g + j], s, 0, 0, 0);
                    dp = __builtin_amdgcn_mfma_f32_32x32x2f32(dx[j], vreg[4 * g + j], dp, 0, 0, 0);
                }
            }
            // register r <-> tile row 8 (r / 4) + 4h + r % 4, lane <-> key: P and dS of the (row, key) pair
#pragma unroll
            for (int r = 0; r < 16; r++) {
                float pv = __builtin_amdgcn_exp2f(s[r] * c2 - lse2[r]);
                pv = kpos <= qpos[r] ? pv : 0.f;
                s[r] = pv;
                dp[r] = pv * dp[r];
            }
            // dV^T += dO^T P and dK^T += Q^T dS: step r contracts the row of accumulator register r; lane (d = 32 db + l32, h)
            // reads dO[row][d] / Q[row][d]
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int trow = 8 * (r / 4) + 4 * hh + (r % 4);
                const int sw = f32_swz(trow);
                const float *dor = dOs + trow * D + (l32 & 3), *qr = Qs + trow * D + (l32 & 3);
#pragma unroll
                for (int db = 0; db < D / 32; db++) {
                    const int off = ((8 * db + (l32 >> 2)) ^ sw) << 2;
                    dvacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(dor[off], s[r], dvacc[db], 0, 0, 0);
                    dkacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(qr[off], dp[r], dkacc[db], 0, 0, 0);
                }
            }
        }
        tile_barrier();
        par ^= 1;
        it = nxt;
    }
    if (p.split_log2) {   // a share of the keys' gradients, summed by the reduction kernel
        float *const part = p.part + (((((long long)pair * p.tiles_seen + tile) << p.split_log2) + split) * 8 + w) * (32 * D);
        store_partial<D>(part, lane, dvacc, 1.f);
        store_partial<D>(part + 4 * 32 * D, lane, dkacc, p.scale);
        return;
    }
    // dK^T / dV^T of the wave's 32 keys: added to the fp32 accumulators in whole rows through the wave's staging area
    unsigned char *stage = smem + w * WaveStage<D>::BYTES;
    constexpr int LPR = D / 4, ROWS_PER_IT = 64 / LPR;
    const int key_base = key0 + 32 * w;
    auto add_rows = [&](const f32x16 (&acc)[D / 32], float mul, float *base, long long stride) {
        float *gp = base + (long long)(key_base + lane / LPR) * stride + 4 * (lane % LPR);
        wave_tile_rowmajor<D>(stage, lane, acc, mul, [&](int row, int, f32x4 val) {
            if (key_base + row < sk) {
                const f32x4 old = *(const f32x4 *)gp;
#pragma unroll
                for (int e = 0; e < 4; e++) val[e] += old[e];
                *(f32x4 *)gp = val;
            }
            gp += ROWS_PER_IT * stride;
        });
    };
    add_rows(dkacc, p.scale, p.chunk[c].dk + b * p.dks[0] + hkv * p.dks[2], p.dks[1]);
    add_rows(dvacc, 1.f, p.chunk[c].dv + b * p.dvs[0] + hkv * p.dvs[2], p.dvs[1]);
}

// ------------------------------------------------------------------------------ host side
bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// Per-device facts, found out on the first call on each device and read-only afterwards.  The fields are atomics: two host
// threads that make their first call at the same time both do the (idempotent) work and store the same answer.  A failed
// query or opt-in is not remembered: the next call tries again.
constexpr int LTR_MAX_DEVICES = 64;
struct DeviceState {
    std::atomic<int> arch{0};          // 0 unknown, 1 gfx950, -1 something else
    std::atomic<int> large_lds{0};     // 1: the kernels of this device may use more than 64 KB of dynamic LDS
    std::atomic<int> cus{0};           // compute units (0: not asked yet)
    std::atomic<float *> scratch{nullptr};   // device address of this device's copy of `scratch`
};
DeviceState g_dev[LTR_MAX_DEVICES];

int current_device(int *dev) {
    if (hipGetDevice(dev) != hipSuccess || *dev < 0 || *dev >= LTR_MAX_DEVICES) return LTR_EDEVICE;
    return LTR_OK;
}

int check_device() {   // gfx950 only
    int dev = 0;
    if (current_device(&dev)) return LTR_EDEVICE;
    int arch = g_dev[dev].arch.load(std::memory_order_acquire);
    if (arch == 0) {
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return LTR_EDEVICE;
        const char *a = prop.gcnArchName;
        arch = (a[0] == 'g' && a[1] == 'f' && a[2] == 'x' && a[3] == '9' && a[4] == '5' && a[5] == '0') ? 1 : -1;
        g_dev[dev].arch.store(arch, std::memory_order_release);
    }
    return arch == 1 ? LTR_OK : LTR_EDEVICE;
}

// kernels that need more than 64 KB of dynamic LDS must opt in once per device
template <int D, int RB = 1>
constexpr int fwd_lds_bytes() {   // the K / V tile buffers, reused by the epilogue's staging areas (one per wave)
    return 2 * 2 * FwdTile<D, RB>::BN * D * 2 > 8 * WaveStage<D>::BYTES ? 2 * 2 * FwdTile<D, RB>::BN * D * 2 : 8 * WaveStage<D>::BYTES;
}
template <int D>
constexpr int dq_lds_bytes() { return fwd_lds_bytes<D>(); }   // same tile buffers and staging areas as the forward
template <int D, int KS>
constexpr int shares_lds_bytes() {   // forward and dQ kernels with key shares: tile buffers, then the shares' partial results
    return 2 * 2 * FwdTile<D, 1, KS>::BN * KS * D * 2 > KeyShares<D, KS>::BYTES ? 2 * 2 * FwdTile<D, 1, KS>::BN * KS * D * 2 : KeyShares<D, KS>::BYTES;
}
static_assert(shares_lds_bytes<128, 2>() <= 160 * 1024 && shares_lds_bytes<128, 4>() <= 160 * 1024 && shares_lds_bytes<64, 4>() <= 160 * 1024, "LDS of one CU");
static_assert(8 * WaveStage<64>::BYTES <= shares_lds_bytes<128, 2>() && 8 * WaveStage<32>::BYTES <= shares_lds_bytes<64, 2>(), "staging areas");

template <int D, int KS>
constexpr int joint_lds_bytes() {
    constexpr int dq = KS == 1 ? dq_lds_bytes<D>() : shares_lds_bytes<D, KS>();
    return dq > BwdLds<D, 1>::TOTAL ? dq : BwdLds<D, 1>::TOTAL;
}

// Rows (q heads x rows) of a dK/dV block that computes DELTA itself: what they cost a block against delta_kernel's launch.  Backward in a graph, faster
// than with that launch, one round of blocks (means of 10000 random launches; a launch by the host less besides):
//   head dims up to 64    up to 128 rows 1.08 - 1.14     256 rows 1.05 - 1.09     384 rows 1.01     512 rows 0.99 - 1.01     768 rows 0.96
//   up to 128             up to 128 rows 1.05 - 1.07     256 rows 0.99 - 1.00     384 rows 0.94     more than a round of blocks: 0.94 and less
constexpr int own_delta_rows(int D) { return D == 64 ? 320 : 144; }
template <int D>
constexpr int joint_delta_lds_bytes() {
    constexpr int kv = BwdLds<D, 1>::TOTAL + own_delta_rows(D) * 4;
    return joint_lds_bytes<D, 2>() > kv ? joint_lds_bytes<D, 2>() : kv;
}
static_assert(joint_delta_lds_bytes<128>() <= 160 * 1024, "LDS of one CU");

// address of a kernel that takes this argument (the padded kernels of width 128 exist for two)
template <class Params>
const void *kernel_of(void (*kernel)(Params)) { return (const void *)kernel; }

int enable_large_lds() {
    int dev = 0;
    if (current_device(&dev)) return LTR_EDEVICE;
    if (g_dev[dev].large_lds.load(std::memory_order_acquire) == 1) return LTR_OK;
    const struct { const void *kernel; int bytes; } large[] = {
        {(const void *)bwd_dkdv_kernel<128, 1>, BwdLds<128, 1>::TOTAL},
        {(const void *)bwd_dkdv_kernel<64, 1>, BwdLds<64, 1>::TOTAL},
        {(const void *)bwd_dkdv_kernel<64, 2>, BwdLds<64, 2>::TOTAL},
        {(const void *)bwd_dkdv_keywave_kernel<64>, KeyWaveLds<64>::TOTAL},
        {(const void *)fwd_bf16_w4_kernel<128>, FourWaves<128>::LDS},
        {(const void *)fwd_bf16_w4_kernel<64>, FourWaves<64>::LDS},
        {(const void *)bwd_dq_w4_kernel<128>, FourWaves<128>::LDS},
        {(const void *)bwd_dq_w4_kernel<64>, FourWaves<64>::LDS},
        {(const void *)fwd_bf16_kernel<128, 1>, fwd_lds_bytes<128>()},
        {(const void *)fwd_bf16_kernel<64, 1>, fwd_lds_bytes<64>()},
        {(const void *)fwd_bf16_kernel<64, 2>, fwd_lds_bytes<64, 2>()},
        {(const void *)bwd_dq_kernel<128, 1>, dq_lds_bytes<128>()},
        {(const void *)bwd_dq_kernel<64, 1>, dq_lds_bytes<64>()},
        {(const void *)bwd_dq_kernel<64, 2>, dq_lds_bytes<64>()},
        {(const void *)fwd_f32_mfma_kernel<128, 1>, F32Mfma<128, 1>::LDS},
        {(const void *)fwd_f32_mfma_kernel<128, 2>, F32Mfma<128, 2>::LDS},
        {(const void *)fwd_f32_mfma_kernel<64, 1>, F32Mfma<64, 1>::LDS},
        {(const void *)fwd_f32_mfma_kernel<64, 2>, F32Mfma<64, 2>::LDS},
        {(const void *)fwd_f32_mfma_kernel<64, 4>, F32Mfma<64, 4>::LDS},
        {(const void *)fwd_f32_rows32_kernel<64, 4>, F32Mfma<64, 4>::LDS},
        {(const void *)bwd_dq_f32_mfma_kernel<128, 1>, F32Mfma<128, 1>::LDS},
        {(const void *)bwd_dq_f32_mfma_kernel<128, 2>, F32Mfma<128, 2>::LDS},
        {(const void *)bwd_dq_f32_mfma_kernel<64, 1>, F32Mfma<64, 1>::LDS},
        {(const void *)bwd_dq_f32_mfma_kernel<64, 2>, F32Mfma<64, 2>::LDS},
        {(const void *)bwd_dq_f32_mfma_kernel<64, 4>, F32Mfma<64, 4>::LDS},
        {(const void *)bwd_dq_f32_rows32_kernel<64, 4>, F32Mfma<64, 4>::LDS},
        {(const void *)bwd_dkdv_f32_mfma_kernel<128>, F32DkdvLds<128>::LDS},
        {(const void *)bwd_dkdv_f32_mfma_kernel<64>, F32DkdvLds<64>::LDS},
        {kernel_of<BwdParams>(bwd_dkdv_pad_kernel<128>), BwdLds<128, 1>::TOTAL},
        {kernel_of<Columns96<BwdParams>>(bwd_dkdv_pad_kernel<128>), BwdLds<128, 1>::TOTAL},
        {kernel_of<FwdParams>(fwd_bf16_pad_kernel<128, 1>), fwd_lds_bytes<128>()},
        {kernel_of<Columns96<FwdParams>>(fwd_bf16_pad_kernel<128, 1>), fwd_lds_bytes<128>()},
        {kernel_of<FwdParams>(fwd_bf16_pad_kernel<128, 2>), shares_lds_bytes<128, 2>()},
        {kernel_of<Columns96<FwdParams>>(fwd_bf16_pad_kernel<128, 2>), shares_lds_bytes<128, 2>()},
        {kernel_of<FwdParams>(fwd_bf16_pad_kernel<128, 4>), shares_lds_bytes<128, 4>()},
        {kernel_of<Columns96<FwdParams>>(fwd_bf16_pad_kernel<128, 4>), shares_lds_bytes<128, 4>()},
        {kernel_of<BwdParams>(bwd_dq_pad_kernel<128, 1>), dq_lds_bytes<128>()},
        {kernel_of<Columns96<BwdParams>>(bwd_dq_pad_kernel<128, 1>), dq_lds_bytes<128>()},
        {kernel_of<BwdParams>(bwd_dq_pad_kernel<128, 2>), shares_lds_bytes<128, 2>()},
        {kernel_of<Columns96<BwdParams>>(bwd_dq_pad_kernel<128, 2>), shares_lds_bytes<128, 2>()},
        {kernel_of<BwdParams>(bwd_dq_pad_kernel<128, 4>), shares_lds_bytes<128, 4>()},
        {kernel_of<Columns96<BwdParams>>(bwd_dq_pad_kernel<128, 4>), shares_lds_bytes<128, 4>()},
        {kernel_of<BwdParams>(bwd_dkdv_pad_kernel<64>), BwdLds<64, 1>::TOTAL},
        {kernel_of<FwdParams>(fwd_bf16_pad_kernel<64, 1>), fwd_lds_bytes<64>()},
        {kernel_of<FwdParams>(fwd_bf16_pad_kernel<64, 2>), shares_lds_bytes<64, 2>()},
        {kernel_of<FwdParams>(fwd_bf16_pad_kernel<64, 4>), shares_lds_bytes<64, 4>()},
        {kernel_of<BwdParams>(bwd_dq_pad_kernel<64, 1>), dq_lds_bytes<64>()},
        {kernel_of<BwdParams>(bwd_dq_pad_kernel<64, 2>), shares_lds_bytes<64, 2>()},
        {kernel_of<BwdParams>(bwd_dq_pad_kernel<64, 4>), shares_lds_bytes<64, 4>()},
        {(const void *)fwd_bf16_shares_kernel<128, 2>, shares_lds_bytes<128, 2>()},
        {(const void *)fwd_bf16_shares_kernel<128, 4>, shares_lds_bytes<128, 4>()},
        {(const void *)fwd_bf16_shares_kernel<64, 2>, shares_lds_bytes<64, 2>()},
        {(const void *)fwd_bf16_shares_kernel<64, 4>, shares_lds_bytes<64, 4>()},
        {(const void *)bwd_dq_shares_kernel<128, 2>, shares_lds_bytes<128, 2>()},
        {(const void *)bwd_dq_shares_kernel<128, 4>, shares_lds_bytes<128, 4>()},
        {(const void *)bwd_dq_shares_kernel<64, 2>, shares_lds_bytes<64, 2>()},
        {(const void *)bwd_dq_shares_kernel<64, 4>, shares_lds_bytes<64, 4>()},
        {(const void *)bwd_joint_delta_kernel<64>, joint_delta_lds_bytes<64>()},
        {kernel_of<BwdParams>(bwd_joint_delta_pad_kernel<64>), joint_delta_lds_bytes<64>()},
        {(const void *)bwd_joint_delta_kernel<128>, joint_delta_lds_bytes<128>()},
        {kernel_of<BwdParams>(bwd_joint_delta_pad_kernel<128>), joint_delta_lds_bytes<128>()},
        {kernel_of<Columns96<BwdParams>>(bwd_joint_delta_pad_kernel<128>), joint_delta_lds_bytes<128>()},
        {(const void *)bwd_joint_kernel<64, 1>, joint_lds_bytes<64, 1>()},
        {(const void *)bwd_joint_kernel<64, 2>, joint_lds_bytes<64, 2>()},
        {kernel_of<BwdParams>(bwd_joint_pad_kernel<64, 1>), joint_lds_bytes<64, 1>()},
        {kernel_of<BwdParams>(bwd_joint_pad_kernel<64, 2>), joint_lds_bytes<64, 2>()},
        {(const void *)bwd_joint_kernel<128, 1>, joint_lds_bytes<128, 1>()},
        {(const void *)bwd_joint_kernel<128, 2>, joint_lds_bytes<128, 2>()},
        {kernel_of<BwdParams>(bwd_joint_pad_kernel<128, 1>), joint_lds_bytes<128, 1>()},
        {kernel_of<Columns96<BwdParams>>(bwd_joint_pad_kernel<128, 1>), joint_lds_bytes<128, 1>()},
        {kernel_of<BwdParams>(bwd_joint_pad_kernel<128, 2>), joint_lds_bytes<128, 2>()},
        {kernel_of<Columns96<BwdParams>>(bwd_joint_pad_kernel<128, 2>), joint_lds_bytes<128, 2>()},
    };
    bool ok = true;
    for (const auto &k : large) ok = ok && hipFuncSetAttribute(k.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, k.bytes) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        return LTR_ELAUNCH;
    }
    g_dev[dev].large_lds.store(1, std::memory_order_release);
    return LTR_OK;
}

bool strides_ok(const int64_t *s, int elem_bytes) {
    const int per16 = 16 / elem_bytes;
    for (int i = 0; i < 3; i++)
        if (s[i] < 0 || (s[i] % per16) != 0) return false;
    return true;
}

// Width of the kernels that serve head dim D: D itself where they are instantiated, the next width with LTR_HEAD_COLS, 0 = none.
int head_width(int D, unsigned flags) {
    if (D == 64 || D == 128) return D;
    if (!(flags & LTR_HEAD_COLS) || D <= 0 || D > 128 || D % 8) return 0;
    return D < 64 ? 64 : 128;
}

int fits_i32(int64_t x) { return x >= 0 && x < (int64_t)0x7fffffff; }

// How evenly `blocks` equal blocks, one per CU at a time, fill the CUs: blocks / (rounds x CUs), 1 = no idle CU in any round.
double cu_fill(long long blocks, int cus) {
    const long long rounds = (blocks + cus - 1) / cus;
    return rounds > 0 ? (double)blocks / (double)(rounds * cus) : 0.0;
}

// compute units of the current device (the launch heuristics below count rounds of blocks over them); asked once per
// device.  Without a device (a host-only ltr_attn_plan call) the answer is that of the part this library is written for.
int device_cus() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= LTR_MAX_DEVICES) {
        (void)hipGetLastError();   // "no device" is an answer here, not an error to leave behind
        return 256;
    }
    int cus = g_dev[dev].cus.load(std::memory_order_acquire);
    if (cus <= 0) {
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 256;
        g_dev[dev].cus.store(cus, std::memory_order_release);
    }
    return cus;
}

// One kernel launch whose own status is what is returned: hipLaunchKernel reports the submission of THIS launch, so an
// error that unrelated earlier work left in the thread's last-error slot is neither reported as ours nor cleared.
dim3 dims(const BlockGrid &g) { return dim3(g.x, g.y, g.z); }
template <class Params>
int launch(const void *kernel, dim3 grid, int threads, size_t lds_bytes, hipStream_t st, const Params &p) {
    void *args[] = {(void *)&p};
    return hipLaunchKernel(kernel, grid, dim3((unsigned)threads), args, lds_bytes, st) == hipSuccess ? LTR_OK : LTR_ELAUNCH;
}
template <class Params>
int launch(const void *kernel, long long blocks, int threads, size_t lds_bytes, hipStream_t st, const Params &p) {
    return launch(kernel, dim3((unsigned)blocks), threads, lds_bytes, st, p);
}

// Keys that the q rows [r0, r1] walk through under the causal mask: per chunk, those up to the rows' last position.
long long visible_keys(int r0, int r1, int q_split, const int *q_pos0, const ChunkDev *chunk, int n_chunks) {
    auto pos = [&](int row) { return row < q_split ? q_pos0[0] + row : q_pos0[1] + (row - q_split); };
    int hi = pos(r1);
    if (r0 < q_split && r1 >= q_split) hi = std::max(hi, pos(q_split - 1));
    long long keys = 0;
    for (int c = 0; c < n_chunks; c++) keys += std::min<long long>(std::max<long long>((long long)hi - chunk[c].pos0 + 1, 0), chunk[c].sk);
    return keys;
}

// Under a causal mask, do the q tiles of `rows` rows differ in work?  Compared are the first and the last tile: a late
// chunk of a long ring sees nearly all keys from every tile (nothing to balance), a single causal chunk 1 / n of them
// from its first tile.
bool q_tiles_uneven(int Sq, int rows, int q_split, const int *q_pos0, const ChunkDev *chunk, int n_chunks) {
    const int n = (Sq + rows - 1) / rows;
    if (n < 2) return false;
    const long long first = visible_keys(0, rows - 1, q_split, q_pos0, chunk, n_chunks);
    const long long last = visible_keys((n - 1) * rows, Sq - 1, q_split, q_pos0, chunk, n_chunks);
    return std::min(first, last) * 4 < std::max(first, last) * 3;
}

// The same for the key tiles of the dK/dV kernel: the rows that see the first and the last tile's first key.
bool key_tiles_uneven(int Sq, int keys, int q_split, const int *q_pos0, const ChunkDev *chunk, int n_chunks) {
    long long lo = 0x7fffffff, hi = 0;
    for (int c = 0; c < n_chunks; c++)
        for (const int kpos : {chunk[c].pos0, chunk[c].pos0 + (chunk[c].sk - 1) / keys * keys}) {
            const long long rows = std::min<long long>(std::max<long long>(q_pos0[0] + (long long)q_split - kpos, 0), q_split) +
                                   std::min<long long>(std::max<long long>(q_pos0[1] + (long long)(Sq - q_split) - kpos, 0), Sq - q_split);
            lo = std::min(lo, rows);
            hi = std::max(hi, rows);
        }
    return lo * 4 < hi * 3;
}

// Slots of q tiles handed to the blocks of the forward and dQ kernels.  Under a causal mask a tile's work grows with its
// rows' positions; pairing tile t with tile n - 1 - t in one block gives every block the same work (no long blocks left
// over at the end of the launch) and halves the number of blocks to start.  Only done when the tiles do differ (see
// q_tiles_uneven: paired tiles run one after the other, so fewer blocks walk through the same K / V rows at the same time)
// and while the equal blocks still fill the device's CUs evenly; otherwise one tile per slot, heaviest first, and the
// hardware's in-order dispatch balances.
int q_tile_slots(int n_qtiles, long long blocks_per_tile, bool uneven, int cus) {
    if (!uneven || n_qtiles < 2) return n_qtiles;
    const int n_slots = (n_qtiles + 1) / 2;
    const long long n = n_slots * blocks_per_tile, rounds = (n + cus - 1) / cus;
    return n * 10 >= rounds * cus * 9 ? n_slots : n_qtiles;
}

// Waves that share a row group's keys in the bf16 forward and dQ kernels.  Blocks of 256 rows leave CUs idle when a launch has few
// rows (a short or single sequence, few heads), and the longest block of a causal launch then decides its time; with 2 or 4
// waves per row group a block has 128 or 64 rows and each wave walks half or a quarter of the keys.  The price is more K / V
// traffic per row and the merge at the end.  The choice compares launch times: a q tile costs its K / V tiles times step_us plus
// fixed_us, blocks run longest first, one per CU.  Constants fitted to 24 shapes with every size forced; forward / dQ
// kernel in us, shares 1, 2, 4 (with the launch gap):
//   B=1 32 heads D=128 causal S=1237   38.1 / 48.1    26.7 / 32.9    36.3 / 43.3
//   B=1  8 heads D=128 causal S=4096   99.0 / 128.7   64.8 / 81.3    52.7 / 66.1
//   B=1  8 heads D=64  causal S=4096   64.9 / 72.8    40.4 / 46.6    34.5 / 40.8
//   B=1 32 heads D=128 causal S=4096  135.1 / 183.9  158.5 / 204.6  203.2 / 256.8   (256-row blocks fill the device)
//
// Under a causal mask two shares may also take their q tiles in pairs (late + early, see q_tile_slots): where 256-row tiles give every
// CU one block of its own length and the longest decides, 128-row tiles pair to one equal block per CU.  Only for a round that is
// (nearly) full: with fewer blocks idle CUs cost more than the balance gives.  Kernel us unpaired -> paired, forward / dQ:
//   B=1 16 heads D=128 S=4096   115 / 128 -> 97 / 123 (256 paired blocks)    B=1 16 heads D=64 S=4096    72 / 86 -> 58 / 70 (256)
//   B=2 16 heads D=128 S=2048    64 / 86  -> 59 / 74 (256)                   B=4 16 heads D=128 S=1024   39 / 51 -> 40 / 50 (256)
//   B=1 16 heads D=128 S=3500    79 / 101 -> 83 / 107 (224)                  B=2  8 heads D=128 S=3000   64 / 82 -> 70 / 90 (192)
//   B=1 12 heads D=64 S=3333     38 / 46  -> 44 / 54 (168)                   B=1 32 heads D=128 S=1237   31 / 39 -> 39 / 50 (160)
// Four shares in pairs were slower than two at all nine shapes tried.
struct ShareCost {
    double step_us[3], fixed_us[3];   // per step (one K / V tile) and per block, for 1, 2 and 4 shares
    double paired_us;                 // per step of two shares in pairs (a block on every CU)
};
struct ShareChoice {
    int ks;
    bool paired;
    double us;   // the launch, by these constants
};
ShareChoice key_shares(const ShareCost &cost, int D, bool causal, long long BH, long long kv_heads, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk, int n_chunks, int cus) {
    if (BH * ((Sq + 255) / 256) >= 4LL * cus) return {1, false, 0};   // several rounds of 256-row blocks: they balance by themselves
    ShareChoice best{1, false, 0};
    double best_us = 0;
    for (int i = 0; i < 3; i++) {
        const int ks = 1 << i, rows = 256 >> i, key_log2 = i + (D == 64 ? (ks == 1 ? 7 : 6) : (ks == 4 ? 5 : 6));
        const int n = (Sq + rows - 1) / rows;
        // more than one kv head per XCD and every CU busy: the extra K / V traffic of the shares shows (B=1, 32 kv heads, D=128,
        // S=2048: 57 us with one share, 67 with two; with 8 kv heads 57 and 49)
        const double step_us = cost.step_us[i] * (ks > 1 && BH * n > cus && kv_heads > 8 ? 1.25 : 1.0);
        auto steps = [&](int t) {
            double sum = 0;
            const int r0 = t * rows, r1 = std::min(Sq, r0 + rows) - 1;
            int hi = r1 < q_split ? q_pos0[0] + r1 : q_pos0[1] + (r1 - q_split);
            if (r0 < q_split && r1 >= q_split) hi = std::max(hi, q_pos0[0] + q_split - 1);
            for (int c = 0; c < n_chunks; c++) {
                const long long seen = causal ? std::min<long long>(std::max<long long>((long long)hi - chunk[c].pos0 + 1, 0), chunk[c].sk) : chunk[c].sk;
                sum += (double)((seen + (1 << key_log2) - 1) >> key_log2);
            }
            return sum;
        };
        double sum = 0, most = 0;
        for (int t = 0; t < n; t++) {
            const double us = steps(t) * step_us + cost.fixed_us[i];
            sum += us;
            most = std::max(most, us);
        }
        const double us = BH * n <= cus ? most : std::max(most, sum * BH / cus + 0.25 * sum / n);
        if (i == 0 || us < 0.97 * best_us) {
            best_us = us;
            best = {ks, false, us};
        }
        const int slots = (n + 1) / 2;
        if (ks == 2 && causal && BH * slots <= cus && BH * slots * 10 >= cus * 9 && q_tiles_uneven(Sq, rows, q_split, q_pos0, chunk, n_chunks)) {
            double pair_us = 0;
            for (int t = 0; t < slots; t++) {
                const bool two = t < n - 1 - t;
                pair_us = std::max(pair_us, (steps(t) + (two ? steps(n - 1 - t) : 0)) * cost.paired_us + (two ? 2 : 1) * cost.fixed_us[i]);
            }
            if (pair_us < 0.97 * best_us) {
                best_us = pair_us;
                best = {ks, true, pair_us};
            }
        }
    }
    return best;
}
constexpr ShareCost FWD_SHARES_128{{1.45, 1.8, 1.05}, {9.0, 8.0, 10.0}, 2.2}, FWD_SHARES_64{{1.7, 0.95, 1.0}, {9.0, 8.0, 6.0}, 1.09};
constexpr ShareCost DQ_SHARES_128{{1.85, 2.2, 1.4}, {11.0, 10.0, 10.0}, 2.7}, DQ_SHARES_64{{1.95, 1.15, 1.35}, {10.0, 9.0, 6.0}, 1.3};

// Blocks of the bf16 forward and dQ kernels: which of the kernels below a launch takes.
//   256 rows, 8 waves                long blocks: a K / V tile serves eight waves
//   512 rows, 8 waves (head dim 64)  longer ones: every operand read serves two row blocks
//   128 / 64 rows, 8 waves           2 / 4 waves share a row group's keys: launches with few rows (key_shares)
//   128 rows, 4 waves                several blocks per CU (FourWaves): launches of many blocks that are not long
// The choice compares launch times.  A block of n K / V tiles takes n alone_us + alone_fixed_us on a CU of its own and costs the CU
// n step_us + fixed_us when there are enough of them; blocks run longest first, so a launch of unequal ones takes their sum over
// the CUs plus `tail` of the shortest, a launch of equal ones its largest number of blocks on a CU.  Constants fitted to 120 random
// launches (8 - 32 heads, 64 - 7900 rows, 4 in 5 causal) of every kernel: rms error 4 - 7 %; the steps of four waves are those of long equal
// blocks (1024 rows against 8192 and 16384 keys), 2 - 8 % above the fit.  256-row blocks are replaced where
// another kernel is 1.5 % faster (more: complete rounds of pairs), shares where four waves are 12 % faster, and what key_shares says about
// shares, with coarser rounds, where other shares are 20 % faster (280 blocks of four shares on 256 CUs: 16.4 us for 9.0 of two).
struct TileCost {
    double alone_us, alone_fixed_us, step_us, fixed_us, tail;
};
enum { ROWS_256, SHARES_2, SHARES_4, FOUR_WAVES, ROWS_512, N_ROW_KERNELS };
struct RowCosts {
    ShareCost shares;
    TileCost kernel[N_ROW_KERNELS];
};
struct RowChoice {
    int kernel;
    bool paired;   // SHARES_2: q tiles in pairs
};
struct RowKernel {
    int rows, key_log2;   // query rows per block, log2 of the keys per K / V tile
};
RowKernel row_kernel(int kernel, int D) {
    switch (kernel) {
        case ROWS_512: return {512, 6};
        case SHARES_2: return {128, 7};
        case SHARES_4: return {64, D == 64 ? 8 : 7};
        case FOUR_WAVES: return {128, 6};
        default: return {256, D == 64 ? 7 : 6};
    }
}
// allowed: bit per kernel
RowChoice choose_rows(const RowCosts &costs, unsigned allowed, int D, bool causal, long long BH, long long kv_heads, int Sq, int q_split,
                      const int *q_pos0, const ChunkDev *chunk, int n_chunks, int cus) {
    if ((allowed & (allowed - 1)) == 0) return {__builtin_ctz(allowed), false};   // a hint
    RowChoice first{ROWS_256, false};
    double first_us = 0;
    if (allowed >> SHARES_2 & 1) {
        const ShareChoice sc = key_shares(costs.shares, D, causal, BH, kv_heads, Sq, q_split, q_pos0, chunk, n_chunks, cus);
        first = {sc.ks == 4 ? SHARES_4 : sc.ks == 2 ? SHARES_2 : ROWS_256, sc.paired};
        if (sc.paired) first_us = sc.us;
    }
    const bool shared = first.kernel != ROWS_256;
    double four_waves = 0.985;
    if (!shared && causal) {
        // 256-row tiles whose pairs come out in complete rounds of equal blocks: nothing of a CU is idle.  At head dim 128 four waves are then
        // not faster (us forward / dQ, pairs / four waves: 4 x 32 heads S=1024 51 / 71 - 52 / 70, 8 x 32 heads S=512 41 / 52 - 40 / 51,
        // 8 x 32 heads S=2048 324 / 448 - 340 / 458).  At head dim 64 they are, in chunk tables as well (37 launches 1.03 - 1.72 times; forward:
        // 8 x 32 heads, 1100 rows against 1000 + 400 keys 140 - 93, 16 x 16 heads S=1024 72 - 57), but the model makes them too short in one full
        // round of pairs, four of their blocks on a CU that runs three (4 x 16 heads S=2048 forward 50.0 - 52.7, modelled 0.98 of the pairs), and
        // for zig-zag shares with long blocks, where some CUs get one more of the late segment's than others (4 x 8 heads, 3612 rows of 7224
        // 138 - 160, 0.91; 2 x 32 heads, 3618 of 28944 1043 - 1122, 0.98).  Padded heads have no four-wave form and take two shares for some
        // zig-zag shares (heads of 40, forward / forward and backward: 4 x 128 heads S=820 of 1640 278 / 913 - 246 / 824, 8 x 24 heads 4028 of 8056
        // 1082 / 4257 - 1104 / 4239, 8 x 64 heads 3934 of 15736 5508 / 22407 - 5551 / 21818)
        const int n = (Sq + 255) / 256, slots = (n + 1) / 2;
        if (n > 1 && BH * slots % cus == 0 && q_tiles_uneven(Sq, 256, q_split, q_pos0, chunk, n_chunks)) {
            if (D == 128) return first;
            const bool two_segments = q_split > 0 && q_split < Sq;
            if (two_segments && visible_keys(Sq - 256, Sq - 1, q_split, q_pos0, chunk, n_chunks) > 4096) four_waves = 0.88;
            else if (BH * slots == cus && n % 2 == 0) four_waves = 0.95;
        }
    }
    double us[N_ROW_KERNELS];
    for (int i = 0; i < N_ROW_KERNELS; i++) {
        us[i] = 0;
        const RowKernel k = row_kernel(i, D);
        const int n = (Sq + k.rows - 1) / k.rows;
        if (!(allowed >> i & 1) || (i == FOUR_WAVES && BH * n <= cus)) continue;   // four waves alone on a CU: no
        // the constants of 512 rows are those of blocks without a diagonal (8 of 34 launches): 384 heads causal S=1496, dQ 251 us with 256 rows, 267
        if (i == ROWS_512 && causal && Sq < 4096) continue;
        const TileCost &c = costs.kernel[i];
        // of many q tiles, 16 evenly spaced ones stand for all
        const int m = causal ? std::min(n, 16) : 1;
        double sum = 0, most = 0, least = 1e30, at[16];
        for (int j = 0; j < m; j++) {
            const int t = m > 1 ? (int)((long long)j * (n - 1) / (m - 1)) : n - 1;
            const int r0 = t * k.rows, r1 = std::min(Sq, r0 + k.rows) - 1;
            int hi = r1 < q_split ? q_pos0[0] + r1 : q_pos0[1] + (r1 - q_split);
            if (r0 < q_split && r1 >= q_split) hi = std::max(hi, q_pos0[0] + q_split - 1);
            long long tiles = 0;
            for (int ch = 0; ch < n_chunks; ch++) {
                const long long seen = causal ? std::min<long long>(std::max<long long>((long long)hi - chunk[ch].pos0 + 1, 0), chunk[ch].sk) : chunk[ch].sk;
                tiles += (seen + (1 << k.key_log2) - 1) >> k.key_log2;
            }
            at[j] = (double)tiles;
            sum += at[j] / m;
            most = std::max(most, at[j]);
            least = std::min(least, at[j]);
        }
        // head dim 128: past 8192 keys the tile traffic of four waves outweighs the fixed cost they hide (4 x 32 heads S=8192 forward / dQ
        // 2046 / 2844 us with eight, 2173 / 2925 with four; zig-zag share of 32768 tokens, 32 heads, dQ 1295 / 1360)
        if (i == FOUR_WAVES && D == 128 && most * (1 << k.key_log2) > 8192) continue;
        const double blocks = (double)BH * n, on_a_cu = std::ceil(blocks / cus);
        // one round of the shares that key_shares chose ends with its longest block.  With a tail on top, 8 x 16 heads of 128 with 200 rows went
        // from 256 blocks of two shares to 128 of 256 rows (forward / dQ 12.1 / 14.5 us - 16.1 / 19.4), 84 of 18000 launches likewise (1.08 - 1.35
        // times).  At head dim 64 key_shares takes four shares for two too early, which the tail mends (8 x 8 heads, 216 rows of a zig-zag
        // share 12.8 / 14.3 - 11.3 / 13.1)
        if (D == 128 && shared && i == first.kernel && blocks <= cus) {
            us[i] = std::max(most * c.alone_us + c.alone_fixed_us, most * c.step_us + c.fixed_us);
            continue;
        }
        if (least >= 0.9 * most) {
            us[i] = std::max(most * c.alone_us + c.alone_fixed_us, on_a_cu * (most * c.step_us + c.fixed_us));
            continue;
        }
        // the long blocks (all of the late segment of zig-zag rows are) come in whole numbers per CU as well
        double longs = 0, long_sum = 0;
        for (int j = 0; j < m; j++)
            if (at[j] >= 0.75 * most) longs += 1, long_sum += at[j];
        const double long_us = std::ceil(blocks * longs / m / cus) * (long_sum / longs * c.step_us + c.fixed_us);
        us[i] = std::max(std::max(most * c.alone_us + c.alone_fixed_us, std::max(long_us, on_a_cu * (least * c.step_us + c.fixed_us))),
                         blocks * (sum * c.step_us + c.fixed_us) / cus + c.tail * (least * c.step_us + c.fixed_us));
        if ((i == ROWS_256 || i == ROWS_512) && q_tile_slots(n, BH, q_tiles_uneven(Sq, k.rows, q_split, q_pos0, chunk, n_chunks), cus) != n) {   // in pairs
            double pair = 0;
            for (int j = 0; 2 * j < m; j++) pair = std::max(pair, at[j] + (2 * j < m - 1 ? at[m - 1 - j] : 0));
            // the middle one of an odd number is a block by itself, of half the work: it can fill half a round (384 heads, 13 tiles of 512 rows:
            // 9.75 pairs per CU; taken for 11 whole rounds the launch went to 256 rows, dQ 3007 us for 2900)
            const double halves = n % 2 ? std::ceil((double)BH * n / cus) : 2 * std::ceil((double)BH * (n / 2) / cus);
            us[i] = halves / 2 * (pair * c.step_us + 2 * c.fixed_us);
        }
    }
    RowChoice best = first;
    const double from = first_us > 0 ? first_us : us[first.kernel];
    double best_us = from;
    for (int i = 0; i < N_ROW_KERNELS; i++) {
        const bool to_shares = i == SHARES_2 || i == SHARES_4;
        if (us[i] > 0 && us[i] < best_us && us[i] < from * (to_shares || first.paired ? 0.8 : shared ? 0.88 : i == FOUR_WAVES ? four_waves : 0.985)) {
            best_us = us[i];
            best = {i, false};
        }
    }
    return best;
}
constexpr RowCosts FWD_ROWS_64{FWD_SHARES_64, {{1.83, 6.9, 2.01, 7.2, 0.16}, {0.98, 7.0, 1.15, 5.0, 0.64}, {0.94, 8.3, 1.22, 6.5, 0.49}, {0.76, 6.8, 0.55, 2.1, 1.22}, {1.70, 11.1, 1.94, 4.7, 0.56}}};
constexpr RowCosts FWD_ROWS_128{FWD_SHARES_128, {{1.52, 7.3, 1.70, 7.5, 0.26}, {1.77, 8.6, 1.98, 6.9, 0.72}, {1.03, 8.5, 1.18, 6.8, 0.44}, {1.16, 7.8, 0.92, 4.5, 0.57}, {}}};
constexpr RowCosts DQ_ROWS_64{DQ_SHARES_64, {{2.17, 7.7, 2.61, 7.2, 0.43}, {1.26, 7.9, 1.43, 6.3, 0.54}, {1.33, 8.9, 1.69, 6.7, 0.57}, {1.04, 6.9, 0.75, 3.5, 0.59}, {1.93, 15.4, 2.51, 6.5, 0.48}}};
constexpr RowCosts DQ_ROWS_128{DQ_SHARES_128, {{2.02, 9.5, 2.45, 6.7, 0.52}, {2.32, 10.4, 2.65, 8.5, 0.69}, {1.33, 11.3, 1.51, 9.1, 0.44}, {1.63, 8.3, 1.30, 5.4, 0.56}, {}}};
// The blocks of a launch as classes for launch_us: neighbours that differ by less than 3 % are one class.
struct BlockList {
    static constexpr int MOST = 64;   // tiles looked at: all of up to 64, else 64 evenly spaced ones
    BlockClass c[MOST];
    int k = 0;
    long long n = 0;
    void add(double us, long long blocks) {
        n += blocks;
        if (k > 0 && std::abs(c[k - 1].us - us) < 0.03 * us) {
            c[k - 1].us = (c[k - 1].us * c[k - 1].n + us * blocks) / (double)(c[k - 1].n + blocks);
            c[k - 1].n += blocks;
        } else {
            c[k++] = {us, blocks};
        }
    }
    // the least that the launch can take: its blocks spread evenly, or the longest of them
    double least_us(int slots) const { return std::max(total_us() / slots, longest_us()); }
    double total_us() const {
        double t = 0;
        for (int i = 0; i < k; i++) t += c[i].us * c[i].n;
        return t;
    }
    double longest_us() const {
        double t = 0;
        for (int i = 0; i < k; i++) t = std::max(t, c[i].us);
        return t;
    }
};
// 0, then n / d more each time, in whole numbers: floor(j n / d) for j = 0, 1, 2 ... with one division in all
struct EvenSteps {
    long long at = 0, whole, rest, d, over = 0;
    EvenSteps(long long n, long long d_) : whole(d_ > 0 ? n / d_ : 0), rest(d_ > 0 ? n - whole * d_ : 0), d(d_) {}
    long long next() {   // by how much it grew
        over += rest;
        const long long grew = whole + (over >= d);
        if (over >= d) over -= d;
        at += grew;
        return grew;
    }
};
// Blocks of a forward or dQ launch, late tiles first: a block takes step_us per K / V tile and fixed_us besides, one that sees nothing 1 us.
BlockList q_tile_blocks(RowKernel kernel, double step_us, double fixed_us, bool paired, bool causal, long long BH, int Sq, int q_split, const int *q_pos0,
                        const ChunkDev *chunk, int n_chunks) {
    BlockList l;
    const int n = (Sq + kernel.rows - 1) / kernel.rows, slots = paired ? (n + 1) / 2 : n, k = causal ? std::min(slots, BlockList::MOST) : 1;
    auto us = [&](int t) {
        long long tiles = 0;
        const int r0 = t * kernel.rows, r1 = std::min(Sq, r0 + kernel.rows) - 1;
        int hi = r1 < q_split ? q_pos0[0] + r1 : q_pos0[1] + (r1 - q_split);
        if (r0 < q_split && r1 >= q_split) hi = std::max(hi, q_pos0[0] + q_split - 1);
        for (int c = 0; c < n_chunks; c++) {
            const long long seen = causal ? std::min<long long>(std::max<long long>((long long)hi - chunk[c].pos0 + 1, 0), chunk[c].sk) : chunk[c].sk;
            tiles += (seen + (1 << kernel.key_log2) - 1) >> kernel.key_log2;
        }
        return tiles ? tiles * step_us + fixed_us : 1.0;
    };
    EvenSteps blocks(BH * slots, k), tile(slots - 1, k - 1);
    for (int j = 0; j < k; j++, tile.next()) {
        const int slot = (int)tile.at, late = n - 1 - slot;
        l.add(us(late) + (paired && slot < late ? us(slot) : 0), blocks.next());
    }
    return l;
}

// A second look at the choice of a forward launch, by launch_us: choose_rows knows a launch by its longest and average block, which is wrong by up to 40 %
// where whole rounds decide (a zig-zag share whose late half is one round of two shares, taken for a round and a half: 1 x 32 heads,
// 1194 rows of 9552, D=128 194 us with four shares, 140 with two).  Constants fitted to 5500 random launches of every kernel (rms 6 - 10 %).
// How much shorter another kernel has to be by them depends on what changes (needed_share).
struct LaunchCost {
    double step_us[N_ROW_KERNELS], fixed_us[N_ROW_KERNELS];   // four waves: of a block among others, as a share of its CU
    double alone_us, alone_fixed_us;                          // four waves, alone on a CU
    double paired_us, paired_fixed_us;                        // two shares in pairs
};
constexpr LaunchCost FWD_LAUNCH_64{{1.92, 1.125, 1.35, 0.447, 1.76}, {4.8, 5.1, 5.45, 2.5, 6.2}, 0.78, 4.7, 1.09, 4.8},
    FWD_LAUNCH_128{{1.565, 1.84, 1.2, 0.816, 0}, {5.8, 6.5, 6.6, 4.0, 0}, 1.09, 6.2, 1.76, 6.1};
// The share of the present launch's time that another kernel may take at most, 0: never.  rounds: of 256-row blocks.  From 15085 random launches that
// changed with one share of 0.94 (four waves 0.9) for all, one in 13 of those looked at (calls, ring and zig-zag ranks, single steps; 90 - 8190 rows,
// 8 - 256 heads): 1.127 times as fast in the mean, but 746 more than 2 % slower, 487 more than 5 %, the worst 1.7 times (8 x 32 heads of 128, 192 rows
// of a zig-zag share 99 us with 256 rows, 170 with four shares).  With these and four_waves_us, chosen on those launches, 15323 of 253436 others
// change: 1.150 times as fast in the mean, 151 more than 2 % slower, 49 more than 5 %, the worst 1.20 times.
double needed_share(int D, double now, double rounds, int from, bool from_paired, int to, bool to_paired) {
    switch (to) {
        case SHARES_4: return from == ROWS_256 ? 0.0 : D == 64 ? 0.94 : now < 20.5 ? 0.75 : 0.89;
        case SHARES_2: return D == 64 || from == SHARES_4 ? 0.94 : from_paired || rounds > 2 ? 0.88 : now < 20.5 ? 0.85 : 0.92;
        case FOUR_WAVES: return from == SHARES_4 ? 0.85 : 0.9;
        case ROWS_512: return to_paired ? 0.0 : from_paired ? 0.91 : 0.94;
        default: return 0.94;
    }
}
RowChoice faster_rows(const LaunchCost &cost, RowChoice chosen, unsigned allowed, int D, bool causal, long long BH, int Sq, int q_split, const int *q_pos0,
                      const ChunkDev *chunk, int n_chunks, int cus) {
    // a hint; four waves; past 32 rounds nothing decides but the step
    if ((allowed & (allowed - 1)) == 0 || chosen.kernel == FOUR_WAVES || BH * ((Sq + 255) / 256) > 32LL * cus) return chosen;
    // Four waves: the long blocks (0.75 of the longest and more) come in whole numbers per CU and take the step of long equal blocks, which the fitted
    // one is 11 - 19 % below; at head dim 128 with up to 1.6 of them per CU they are slower still (4 x 16 heads on 4, 1284 rows of a zig-zag
    // share of 20544 479 us with 256 rows, 556 with four waves; modelled 568 and 504).
    auto four_waves_us = [&](const BlockList &l, double end, double step, double fixed) {
        double longs = 0, tiles = 0;
        const double least = 0.75 * (l.longest_us() - fixed);
        for (int i = 0; i < l.k; i++)
            if (l.c[i].us - fixed >= least) longs += l.c[i].n, tiles += (l.c[i].us - fixed) / step * l.c[i].n;
        const TileCost &tile = (D == 128 ? FWD_ROWS_128 : FWD_ROWS_64).kernel[FOUR_WAVES];
        return std::max(end, std::ceil(longs / cus) * (tiles / longs * tile.step_us + tile.fixed_us)) * (D == 128 && longs <= 1.6 * cus ? 1.06 : 1.0);
    };
    auto in_pairs = [&](int i) {   // q tiles of 256 or 512 rows
        const int rows = row_kernel(i, D).rows, n = (Sq + rows - 1) / rows;
        return (i == ROWS_256 || i == ROWS_512) && q_tile_slots(n, BH, causal && q_tiles_uneven(Sq, rows, q_split, q_pos0, chunk, n_chunks), cus) != n;
    };
    auto launch = [&](int i, bool paired, double most) {   // `most` or more is not worth a closer look
        const RowKernel k = row_kernel(i, D);
        int per_cu = 1;
        double step = i == SHARES_2 && paired ? cost.paired_us : cost.step_us[i], fixed = i == SHARES_2 && paired ? cost.paired_fixed_us : cost.fixed_us[i];
        if (i == FOUR_WAVES) {
            per_cu = (int)std::min<long long>(D == 64 ? FourWaves<64>::PER_CU : FourWaves<128>::PER_CU, (BH * ((Sq + k.rows - 1) / k.rows) + cus - 1) / cus);
            step = per_cu == 1 ? cost.alone_us : per_cu * step;
            fixed = per_cu == 1 ? cost.alone_fixed_us : per_cu * fixed;
        }
        const BlockList l = q_tile_blocks(k, step, fixed, paired, causal, BH, Sq, q_split, q_pos0, chunk, n_chunks);
        if (l.least_us(per_cu * cus) >= most) return most;
        Dispatch d(per_cu * cus);
        if (!d.add(l.c, l.k, most)) return most;
        return i == FOUR_WAVES && chosen.kernel != SHARES_4 ? four_waves_us(l, d.end, step, fixed) : d.end;
    };
    const bool now_paired = chosen.paired || in_pairs(chosen.kernel);
    const double now = launch(chosen.kernel, now_paired, 1e30);
    if (now < 14) return chosen;   // a call of that length waits for its host side
    RowChoice better = chosen;
    double best = now;
    for (int i = 0; i < N_ROW_KERNELS; i++) {
        if (!(allowed >> i & 1) || i == chosen.kernel) continue;
        // four waves: not alone on a CU, and not for 256 rows without a mask (11 of 22 such launches 3 - 13 % slower)
        if (i == FOUR_WAVES && (BH * ((Sq + 127) / 128) <= cus || (!causal && chosen.kernel == ROWS_256))) continue;
        const bool paired = in_pairs(i);
        const double most = std::min(best, needed_share(D, now, (double)(BH * ((Sq + 255) / 256)) / cus, chosen.kernel, now_paired, i, paired) * now);
        if (most <= 0) continue;
        const double us = launch(i, paired, most);
        if (us < most) {
            best = us;
            better = {i, false};
        }
    }
    return better;
}

// rows_256, rows_512: the caller's hints; shares: a row group's keys may be shared
unsigned allowed_rows(bool rows_256, bool rows_512, bool shares, bool pad, int D) {
    if (rows_512) return 1u << ROWS_512;
    if (rows_256) return 1u << ROWS_256;
    return 1u << ROWS_256 | (shares ? 1u << SHARES_2 | 1u << SHARES_4 : 0u) | (pad ? 0u : 1u << FOUR_WAVES | (D == 64 ? 1u << ROWS_512 : 0u));
}

// What a forward launch looks like: rows per block, q tiles, slots (see q_tile_slots), blocks.  One function decides for
// ltr_attn_fwd and for ltr_attn_plan, so the plan a caller is shown is the launch it gets.
struct FwdPlan {
    bool wide;          // 512-row blocks (two 32-row blocks per wave, head dim 64)
    bool four_waves;    // 128-row blocks of four waves (FourWaves)
    int ks;             // bf16: key shares per row group (1, or 2 / 4 with blocks of 256 / ks rows; see choose_rows)
    int f32_ks;         // fp32: 0 = scalar kernel, else the key shares per row group of fwd_f32_mfma_kernel
    int rows, n_qtiles, n_slots, group;
    long long blocks;
};
// Rows per block and key shares of the fp32 forward and dQ kernels: 128 rows, or fewer and the keys split over 2 / 4 waves of a row group
// when the launch has too few rows to give every CU a block (4 key shares need the LDS that only head dim 64 leaves); with 4 shares groups
// of 16 rows where the launch still fits the chip in one round.  Kernel us with 32 and 16 rows, 1024 keys at head dim 64, forward / dQ:
// 256 blocks of 16 rows 27.7 / 37.3 and 18.1 / 23.3; 336 blocks, a second round, 27.7 / 37.0 and 34.4 / 44.8; 864 blocks 53.7 / 72.7 and
// 67.0 / 87.8.
int f32_rows(int D, long long pairs, int Sq, int cus, int &ks) {
    const int max_ks = D == 64 ? 4 : 2;
    auto blocks = [&](int rows) { return (long long)((Sq + rows - 1) / rows) * pairs; };
    ks = 1;
    while (ks < max_ks && blocks(128 / ks) < cus) ks *= 2;
    return ks == F32Rows16::KS && blocks(F32Rows16::BM) <= cus ? F32Rows16::BM : 128 / ks;
}
// The kernels of these choices, for the launches and for the plans: a plan's name is that of the kernel a launch takes.
struct KernelChoice {
    const void *fn;
    const char *name;
    int lds;
};
#define LTR_KERNEL(...) (const void *)__VA_ARGS__, #__VA_ARGS__
KernelChoice f32_fwd_kernel(int D, int ks, int rows) {
    if (D == 128) return ks == 1 ? KernelChoice{LTR_KERNEL(fwd_f32_mfma_kernel<128, 1>), F32Mfma<128, 1>::LDS} : KernelChoice{LTR_KERNEL(fwd_f32_mfma_kernel<128, 2>), F32Mfma<128, 2>::LDS};
    if (ks == 1) return {LTR_KERNEL(fwd_f32_mfma_kernel<64, 1>), F32Mfma<64, 1>::LDS};
    if (ks == 2) return {LTR_KERNEL(fwd_f32_mfma_kernel<64, 2>), F32Mfma<64, 2>::LDS};
    return rows == F32Rows16::BM ? KernelChoice{LTR_KERNEL(fwd_f32_mfma_kernel<64, 4>), F32Mfma<64, 4>::LDS} : KernelChoice{LTR_KERNEL(fwd_f32_rows32_kernel<64, 4>), F32Mfma<64, 4>::LDS};
}
KernelChoice f32_dq_kernel(int D, int ks, int rows) {
    if (D == 128) return ks == 1 ? KernelChoice{LTR_KERNEL(bwd_dq_f32_mfma_kernel<128, 1>), F32Mfma<128, 1>::LDS} : KernelChoice{LTR_KERNEL(bwd_dq_f32_mfma_kernel<128, 2>), F32Mfma<128, 2>::LDS};
    if (ks == 1) return {LTR_KERNEL(bwd_dq_f32_mfma_kernel<64, 1>), F32Mfma<64, 1>::LDS};
    if (ks == 2) return {LTR_KERNEL(bwd_dq_f32_mfma_kernel<64, 2>), F32Mfma<64, 2>::LDS};
    return rows == F32Rows16::BM ? KernelChoice{LTR_KERNEL(bwd_dq_f32_mfma_kernel<64, 4>), F32Mfma<64, 4>::LDS} : KernelChoice{LTR_KERNEL(bwd_dq_f32_rows32_kernel<64, 4>), F32Mfma<64, 4>::LDS};
}
#define LTR_PAD_KERNEL(params, ...) kernel_of<params>(__VA_ARGS__), #__VA_ARGS__
KernelChoice joint_kernel(int D, bool pad, int ks, bool own_delta, int cols) {
    const bool three = cols <= 96;   // blocks of 32 columns, width 128
    if (own_delta) {
        if (pad && D == 128)
            return three ? KernelChoice{LTR_PAD_KERNEL(Columns96<BwdParams>, bwd_joint_delta_pad_kernel<128>), joint_delta_lds_bytes<128>()} : KernelChoice{LTR_PAD_KERNEL(BwdParams, bwd_joint_delta_pad_kernel<128>), joint_delta_lds_bytes<128>()};
        if (pad) return {LTR_PAD_KERNEL(BwdParams, bwd_joint_delta_pad_kernel<64>), joint_delta_lds_bytes<64>()};
        return D == 128 ? KernelChoice{LTR_KERNEL(bwd_joint_delta_kernel<128>), joint_delta_lds_bytes<128>()} : KernelChoice{LTR_KERNEL(bwd_joint_delta_kernel<64>), joint_delta_lds_bytes<64>()};
    }
    if (pad) {
        if (D == 128 && three) return ks == 1 ? KernelChoice{LTR_PAD_KERNEL(Columns96<BwdParams>, bwd_joint_pad_kernel<128, 1>), joint_lds_bytes<128, 1>()} : KernelChoice{LTR_PAD_KERNEL(Columns96<BwdParams>, bwd_joint_pad_kernel<128, 2>), joint_lds_bytes<128, 2>()};
        if (D == 128) return ks == 1 ? KernelChoice{LTR_PAD_KERNEL(BwdParams, bwd_joint_pad_kernel<128, 1>), joint_lds_bytes<128, 1>()} : KernelChoice{LTR_PAD_KERNEL(BwdParams, bwd_joint_pad_kernel<128, 2>), joint_lds_bytes<128, 2>()};
        return ks == 1 ? KernelChoice{LTR_PAD_KERNEL(BwdParams, bwd_joint_pad_kernel<64, 1>), joint_lds_bytes<64, 1>()} : KernelChoice{LTR_PAD_KERNEL(BwdParams, bwd_joint_pad_kernel<64, 2>), joint_lds_bytes<64, 2>()};
    }
    if (D == 128) return ks == 1 ? KernelChoice{LTR_KERNEL(bwd_joint_kernel<128, 1>), joint_lds_bytes<128, 1>()} : KernelChoice{LTR_KERNEL(bwd_joint_kernel<128, 2>), joint_lds_bytes<128, 2>()};
    return ks == 1 ? KernelChoice{LTR_KERNEL(bwd_joint_kernel<64, 1>), joint_lds_bytes<64, 1>()} : KernelChoice{LTR_KERNEL(bwd_joint_kernel<64, 2>), joint_lds_bytes<64, 2>()};
}
#undef LTR_PAD_KERNEL
#undef LTR_KERNEL

// What a bf16 plan depends on, and the plans that a thread keeps: pricing launches takes 1 - 11 us, as long as queueing them, and a program asks for the
// same few problems again and again (layers, steps, the ranks of a ring).  32 pairs of places by a hash of the sizes, nothing of a tensor among them;
// a new problem takes the place of its pair that was not used last.
struct Problem {
    int head[12];
    int keys[LTR_MAX_CHUNKS][2];
    size_t used;   // bytes of the above
    Problem() : head{}, used(0) {}   // no problem has 0 chunks
    Problem(int D, unsigned flags, int B, int Hq, int Hkv, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk, int n_chunks, bool may)
        : head{n_chunks, D, (int)flags, B, Hq, Hkv, Sq, q_split, q_pos0[0], q_pos0[1], may, device_cus()}, used(sizeof(head) + n_chunks * sizeof(keys[0])) {
        for (int c = 0; c < n_chunks; c++) {
            keys[c][0] = chunk[c].sk;
            keys[c][1] = chunk[c].pos0;
        }
    }
    bool operator==(const Problem &o) const { return head[0] == o.head[0] && memcmp(this, &o, used) == 0; }
    unsigned hash() const {
        uint64_t h = 0;
        for (int i : head) h = (h ^ (unsigned)i) * 0x9e3779b97f4a7c15ull, h ^= h >> 29;
        for (int c = 0; c < head[0]; c++)
            for (int i : keys[c]) h = (h ^ (unsigned)i) * 0x9e3779b97f4a7c15ull, h ^= h >> 29;
        return (unsigned)(h >> 32) % 32;
    }
};
template <class Plan>
struct KeptPlans {
    Problem problem[32][2];
    Plan plan[32][2];
    unsigned char used_last[32] = {};
    template <class Make>
    Plan get(const Problem &now, Make make) {
        const unsigned h = now.hash();
        unsigned i = used_last[h];
        if (!(problem[h][i] == now)) {
            i ^= 1;
            if (!(problem[h][i] == now)) {
                plan[h][i] = make();
                problem[h][i] = now;
            }
            used_last[h] = i;
        }
        return plan[h][i];
    }
};

FwdPlan make_fwd_plan(int D, bool f32, unsigned flags, int B, int Hq, int Hkv, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk,
                      int n_chunks, bool may_share) {
    FwdPlan pl;
    pl.f32_ks = 0;
    pl.ks = 1;
    pl.group = 1;
    pl.four_waves = false;
    if (f32) {
        pl.wide = false;
        if (flags & LTR_FWD_F32_SCALAR) {
            pl.rows = 64;
        } else {
            // matrix-pipe kernel
            pl.rows = f32_rows(D, (long long)B * Hq, Sq, device_cus(), pl.f32_ks);
        }
        pl.n_qtiles = pl.n_slots = (Sq + pl.rows - 1) / pl.rows;
        pl.blocks = (long long)pl.n_qtiles * B * Hq;
        return pl;
    }
    const bool causal_ = (flags & LTR_CAUSAL) != 0;
    const int cus = device_cus();
    const unsigned allowed = allowed_rows(flags & LTR_FWD_ROWS_256, flags & LTR_FWD_ROWS_512, may_share, flags & LTR_HEAD_COLS, D);
    const RowChoice first = choose_rows(D == 128 ? FWD_ROWS_128 : FWD_ROWS_64, allowed, D, causal_, (long long)B * Hq, (long long)B * Hkv, Sq, q_split, q_pos0, chunk,
                                        n_chunks, cus);
    const RowChoice choice = faster_rows(D == 128 ? FWD_LAUNCH_128 : FWD_LAUNCH_64, first, allowed, D, causal_, (long long)B * Hq, Sq, q_split, q_pos0, chunk, n_chunks, cus);
    pl.wide = choice.kernel == ROWS_512;
    pl.four_waves = choice.kernel == FOUR_WAVES;
    pl.ks = choice.kernel == SHARES_2 ? 2 : choice.kernel == SHARES_4 ? 4 : 1;
    pl.rows = row_kernel(choice.kernel, D).rows;
    pl.n_qtiles = (Sq + pl.rows - 1) / pl.rows;
    const bool uneven = causal_ && q_tiles_uneven(Sq, pl.rows, q_split, q_pos0, chunk, n_chunks);
    pl.n_slots = choice.paired ? (pl.n_qtiles + 1) / 2 : pl.ks > 1 || pl.four_waves ? pl.n_qtiles : q_tile_slots(pl.n_qtiles, (long long)B * Hq, uneven, cus);
    pl.blocks = (long long)pl.n_slots * B * Hq;
    pl.group = pair_group((long long)B * Hkv, (long long)pl.n_slots * (Hq / Hkv), cus / 8 * (pl.four_waves ? D == 64 ? FourWaves<64>::PER_CU : FourWaves<128>::PER_CU : 1),
                          uneven && pl.n_slots == pl.n_qtiles);   // paired tiles are equal blocks
    return pl;
}
FwdPlan plan_fwd(int D, bool f32, unsigned flags, int B, int Hq, int Hkv, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk,
                 int n_chunks, bool may_share = true) {
    auto make = [&] { return make_fwd_plan(D, f32, flags, B, Hq, Hkv, Sq, q_split, q_pos0, chunk, n_chunks, may_share); };
    if (f32) return make();
    static thread_local KeptPlans<FwdPlan> kept;
    return kept.get(Problem(D, flags, B, Hq, Hkv, Sq, q_split, q_pos0, chunk, n_chunks, may_share), make);
}

// Blocks that share one key tile of the dK/dV kernel.  A launch with fewer key tiles than the device has CUs (few kv heads, a
// short or single sequence, one ring step's half-chunk) leaves CUs idle while each block walks all q heads of its group and
// all q tiles; n blocks per tile then take a share of the (q head, q tile) steps each and leave partial sums in a workspace,
// which bwd_dkdv_reduce_kernel adds up.  The choice compares launch times of n = 1, 2, 4 ...: a block costs its steps plus a fixed
// part worth `fixed` steps, the blocks run longest first, one per CU, and the partials are written and read once.  The
// constants are fitted to measured launches of 22 shapes with every n forced (each choice within 3 % of the best n):
// B=1, 32/8 heads, D=128, causal S=1237: n=1 123 us, 2 75, 4 52, 8 67; S=4096: 374, 262, 281, 360; the half-filled ring
// step of 2048 keys x 4096 rows: 184, 129, 138, 158; enough key tiles (B=1, 32 heads, S=2048, 512 tiles): 100, 115, 197, 344;
// fp32, 4/16 heads, D=128, S=700: 870, 445, 233, 128, 83 (n=16).
struct KvSplit {
    int n, reps;      // blocks per key tile; how many of them share out the q heads (the largest power of two that divides both)
    int q_last;       // n > 1: the tiles that have blocks, see seen_tiles
    long long tiles;  // and how many of them there are for one (batch, kv head)
    double us;        // the launch by the model below
};
constexpr double MAX_PART_BYTES = 512e6;   // of partial sums
struct KvSplitCost {
    int rows;                           // q rows per step
    double alone_us, alone_fixed_us;    // a block that has its CU to itself: per step, and its fixed part
    double step_us, fixed_us;           // what a block costs its CU when there are enough of them
    double tail;                        // of an average block, at the end of such a launch
    double reduce_us;                   // the reduction's launch
    double part_bytes_per_us;           // rate at which partials move (each is written and read)
};
KvSplit kv_split(const KvSplitCost &cost, int max_n, int D, int keys, bool causal, int B, int Hkv, int n_rep, int Sq, int q_split, const int *q_pos0,
                 const ChunkDev *chunk, int n_chunks, int n_cus) {
    auto steps_at = [&](long long kpos) -> long long {   // steps of one q head that see the key at position kpos
        long long rows = Sq;
        if (causal)
            rows = std::min<long long>(std::max<long long>(q_pos0[0] + (long long)q_split - kpos, 0), q_split) +
                   std::min<long long>(std::max<long long>(q_pos0[1] + (long long)(Sq - q_split) - kpos, 0), Sq - q_split);
        return (rows + cost.rows - 1) / cost.rows;
    };
    int q_last = 0x7fffffff;
    if (causal)
        q_last = std::max(q_split > 0 ? q_pos0[0] + q_split - 1 : (int)0x80000000, Sq > q_split ? q_pos0[1] + (Sq - q_split) - 1 : (int)0x80000000);
    long long tiles = 0, longest = 0, shortest = 0x7fffffff;
    double total = 0;
    for (int c = 0; c < n_chunks; c++) {
        const long long n = seen_tiles(chunk[c].sk, chunk[c].pos0, q_last, keys);
        if (n == 0) continue;
        const long long first = steps_at(chunk[c].pos0), last = steps_at(chunk[c].pos0 + (n - 1) * keys);
        tiles += n;
        total += 0.5 * n * (first + last);
        longest = std::max(longest, first);
        shortest = std::min(shortest, last);
    }
    KvSplit best{1, 1, q_last, tiles, 0};
    if (tiles == 0) return best;
    const double cus = n_cus, blocks = (double)tiles * B * Hkv, avg = total / tiles * n_rep, most = (double)longest * n_rep;
    for (int n = 1; n <= max_n && n <= std::max(most, 1.0); n *= 2) {
        const double one = avg / n * cost.step_us + cost.fixed_us, longest_us = (double)(((long long)most + n - 1) / n) * cost.alone_us + cost.alone_fixed_us;
        const double bytes = blocks * n * keys * D * 8.0;
        // equal blocks: the largest number on a CU (2 x 8 pairs of 64, 514 rows and keys, no mask inside: 160 blocks 32.6 us, 320 blocks 37.1)
        const bool equal = shortest * 10 >= longest * 9;
        double us = std::max(std::max(longest_us, equal ? std::ceil(blocks * n / cus) * one : 0.0), blocks * n * one / cus + cost.tail * one);
        if (n > 1) us += cost.reduce_us + 2.0 * bytes / cost.part_bytes_per_us;
        if (n == 1 || (us < best.us && bytes <= MAX_PART_BYTES)) {
            best.us = us;
            best.n = n;
        }
    }
    while (best.reps * 2 <= best.n && n_rep % (best.reps * 2) == 0) best.reps *= 2;
    return best;
}

// The same for the two backward kernels.
struct BwdPlan {
    int f32_ks;         // fp32: 0 = scalar kernels, else the key shares per row group of bwd_dq_f32_mfma_kernel
    bool wide_kv;       // dK/dV kernel: 256 keys per block (two 32-key halves per wave, head dim 64)
    bool key_waves;     // dK/dV kernel: bwd_dkdv_keywave_kernel (head dim 64)
    int keys_per_block;
    long long kv_tiles; // key blocks over all chunks of one (batch, kv head)
    long long kv_blocks;
    KvSplit split;      // blocks per key tile (1 unless the caller brought a workspace for their partial sums)
    int64_t part_bytes; // workspace they need
    bool wide_q;        // dQ kernel: 512 rows per block
    bool dq_four_waves; // dQ kernel: blocks of four waves (FourWaves)
    int dq_ks;          // bf16 dQ kernel: key shares per row group, as in the forward
    int dq_rows, dq_qtiles, dq_slots;
    int dq_group, kv_group;   // see pair_group
    long long dq_blocks;
    bool joint, keys_first;   // one launch for both kinds of blocks (bwd_joint_kernel), and which of them go first
    bool own_delta;           // and its dK/dV blocks compute DELTA for themselves (own_delta)
};
// Does a bf16 backward run its dQ and dK/dV blocks in one launch, with how many key shares per row group and blocks per key tile, and which kind
// first?  Both ways are priced by launch_us over classes of blocks (BlockList): the plan as it is, one launch after
// the other, and every joint one.  Constants fitted to random problems (calls, ring and zig-zag ranks, single ring steps; 4 - 32 heads, 45 - 5800
// rows; rms error 9 - 12 %).  Of 40405 others (8 - 256 heads, 90 - 8190 rows) 25360 are joined, 1 / 1.314 of the time apart in the geometric mean:
// 1.54 times as fast where that was up to 25 us, 1.38 up to 50, 1.27 up to 100, 1.19 up to 200, 1.08 past 1600.  75 are more than 2 % slower, 16
// more than 5 %, the worst 1.095 times.
struct JointCost {
    double q_step_us[2], q_fixed_us[2];   // dQ blocks of one and two key shares: per K / V tile and per block
    double shares4_step_us, shares4_fixed_us;
    double kv_step_us, kv_fixed_us;       // dK/dV blocks: per 64 q rows of a head and per block
    double q_acc_us, kv_acc_us;           // more per block where the results are added to fp32 accumulators
    double launch_us, delta_us, delta_bytes_per_us, reduce_us, reduce_bytes_per_us;
};
constexpr JointCost JOINT_128{{2.13, 2.56}, {8.1, 8.5}, 1.33, 8.5, 1.68, 8.9, 2.8, 2.4, 1.4, 2.0, 3.3e6, 5.2, 18e6},
    JOINT_64{{2.90, 1.35}, {4.6, 5.7}, 1.33, 6.5, 0.99, 5.8, 1.0, 2.3, 3.3, 1.8, 2.7e6, 4.6, 23e6};
constexpr KvSplitCost KEY_WAVES_64{64, 1.43, 6.7, 0.82, 3.4, 1.35, 3.5, 19e6};
// pl: the launches apart; alone: those that share no key tiles, which a joint launch that shares none has to be faster than as well (it is also the plan
// of a call without a workspace)
void joint_launch(BwdPlan &pl, const BwdPlan &alone, int D, unsigned flags, int B, int Hq, int Hkv, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk,
                  int n_chunks, bool may_split, int cus) {
    const JointCost &cost = D == 128 ? JOINT_128 : JOINT_64;
    const bool causal = (flags & LTR_CAUSAL) != 0;
    const long long pairs = (long long)B * Hkv, q_pairs = (long long)B * Hq;
    const int n_rep = Hq / Hkv;
    // key tiles by position, as the launch sorts them
    int order[LTR_MAX_CHUNKS];
    for (int i = 0; i < n_chunks; i++) {
        int k = i;
        for (; causal && k > 0 && chunk[order[k - 1]].pos0 > chunk[i].pos0; k--) order[k] = order[k - 1];
        order[k] = i;
    }
    const int q_last = !causal ? 0x7fffffff
                               : std::max(q_split > 0 ? q_pos0[0] + q_split - 1 : (int)0x80000000, Sq > q_split ? q_pos0[1] + (Sq - q_split) - 1 : (int)0x80000000);
    long long tiles_seen = 0;
    for (int i = 0; i < n_chunks; i++) tiles_seen += seen_tiles(chunk[i].sk, chunk[i].pos0, q_last, 128);
    // few blocks only: past some hundred rounds nothing is left to gain
    if (tiles_seen == 0 || pl.kv_tiles > GRID_YZ_MAX || pairs > 8LL * GRID_YZ_MAX || pl.dq_blocks + pl.kv_blocks > 1 << 18) return;
    using List = BlockList;
    auto dq_blocks = [&](int rows, int key_log2, double step_us, double fixed_us, bool paired) {
        return q_tile_blocks({rows, key_log2}, step_us, fixed_us + (flags & LTR_DQ_BF16 ? 0 : cost.q_acc_us), paired, causal, q_pairs, Sq, q_split, q_pos0, chunk, n_chunks);
    };
    // rows that see each of the key tiles looked at, tiles by position: of all tiles, and of those that some row sees (the launches that share)
    struct KeyTiles {
        long long n = 0;
        int k = 0;
        int rows[List::MOST];
    } key_tiles[2];
    auto look_at = [&](KeyTiles &t, long long n, int last) {
        t.n = n;
        t.k = causal ? (int)std::min<long long>(n, List::MOST) : 1;
        EvenSteps tile(n - 1, t.k - 1);
        long long before = 0;   // tiles of the chunks before chunk i
        int i = 0, in_chunk = seen_tiles(chunk[order[0]].sk, chunk[order[0]].pos0, last, 128);
        for (int j = 0; j < t.k; j++, tile.next()) {
            while (i < n_chunks - 1 && tile.at - before >= in_chunk) {
                before += in_chunk;
                i++;
                in_chunk = seen_tiles(chunk[order[i]].sk, chunk[order[i]].pos0, last, 128);
            }
            long long rows = Sq;
            const long long kpos = chunk[order[i]].pos0 + (tile.at - before) * 128;
            if (causal)
                rows = std::min<long long>(std::max<long long>(q_pos0[0] + (long long)q_split - kpos, 0), q_split) +
                       std::min<long long>(std::max<long long>(q_pos0[1] + (long long)(Sq - q_split) - kpos, 0), Sq - q_split);
            t.rows[j] = (int)rows;
        }
    };
    auto kv_blocks = [&](int n_split, double step_us, double fixed_us) {   // n_split: a power of two
        KeyTiles &t = key_tiles[n_split > 1];
        if (t.k == 0) look_at(t, n_split > 1 ? tiles_seen : pl.kv_tiles, n_split > 1 ? q_last : 0x7fffffff);
        List l;
        const double acc_us = n_split > 1 || (flags & LTR_DKDV_BF16) ? 0 : cost.kv_acc_us;
        EvenSteps blocks(pairs * t.n * n_split, t.k);
        for (int j = 0; j < t.k; j++) {
            const long long steps = ((t.rows[j] + 63LL) / 64 * n_rep + n_split - 1) >> __builtin_ctz(n_split);
            l.add(t.rows[j] > 0 ? steps * step_us + fixed_us + acc_us : 1.0, blocks.next());
        }
        return l;
    };
    auto reduce_us = [&](int n_split) { return n_split > 1 ? cost.reduce_us + (double)pl.kv_tiles * pairs * n_split * 128 * D * 8 / cost.reduce_bytes_per_us : 0.0; };

    // the launches of a plan one after the other, and what a joint one has to be shorter than
    auto apart_us = [&](const BwdPlan &x) {
        double us = 2 * cost.launch_us + reduce_us(x.split.n);
        if (x.dq_four_waves) {
            const TileCost &c = (D == 128 ? DQ_ROWS_128 : DQ_ROWS_64).kernel[FOUR_WAVES];
            const int per_cu = (int)std::min<long long>(D == 128 ? FourWaves<128>::PER_CU : FourWaves<64>::PER_CU, (x.dq_blocks + cus - 1) / cus);
            const List l = dq_blocks(128, 6, per_cu == 1 ? c.alone_us : per_cu * c.step_us, per_cu == 1 ? c.alone_fixed_us : per_cu * c.fixed_us, false);
            us += launch_us(l.c, l.k, per_cu * cus);
        } else {
            const int i = x.dq_ks == 4 ? SHARES_4 : x.dq_ks == 2 ? SHARES_2 : ROWS_256;
            const RowKernel k = row_kernel(i, D);
            const List l = dq_blocks(k.rows, k.key_log2, i == SHARES_4 ? cost.shares4_step_us : cost.q_step_us[i == SHARES_2], i == SHARES_4 ? cost.shares4_fixed_us : cost.q_fixed_us[i == SHARES_2],
                                     x.dq_slots != x.dq_qtiles);
            us += launch_us(l.c, l.k, cus);
        }
        if (x.key_waves) {
            const int per_cu = pairs * x.kv_tiles * x.split.n > cus ? 2 : 1;
            const List l = kv_blocks(x.split.n, per_cu == 1 ? KEY_WAVES_64.alone_us : 2 * KEY_WAVES_64.step_us, per_cu == 1 ? KEY_WAVES_64.alone_fixed_us : 2 * KEY_WAVES_64.fixed_us);
            us += launch_us(l.c, l.k, per_cu * cus);
        } else {
            const List l = kv_blocks(x.split.n, cost.kv_step_us, cost.kv_fixed_us);
            us += launch_us(l.c, l.k, cus);
        }
        // where the plan has several blocks on a CU the model takes it for slower than it is, most of all at head dim 64 with both kernels of that
        // kind.  Of those joined with these factors, by the kernels apart: four-wave dQ at head dim 128 1455, 1.100 times as fast, 41 more than 2 %
        // slower (at 0.86 none of 984, 1.123 times); both of that kind at 64 245, 1.078 times, 12 (at 0.74 none of 162); all others 23660, 22
        return us * (D == 128 ? x.dq_four_waves ? 0.92 : 0.98
                              : x.key_waves && x.dq_four_waves ? 0.78 : x.key_waves || x.dq_four_waves || x.dq_blocks + x.kv_blocks > 8 * cus ? 0.88 : 0.96);
    };
    double best = apart_us(pl);
    const double delta_us = flags & LTR_DELTA_FROM_O ? cost.delta_us + (double)q_pairs * Sq * D * 4 / cost.delta_bytes_per_us : 0.0;
    int best_ks = 0, best_n = 1;
    bool keys_first = false;
    // dQ blocks of one and two shares; the blocks of both kinds are looked at in both orders, unless all run at once or even spread evenly over
    // the CUs they take longer than the best so far.  The kind that goes first is dispatched once, for all that may follow
    List q[2];
    double q_total[2], q_longest[2];
    std::optional<Dispatch> after_q[2];
    for (int ks = 1; ks <= 2; ks++) {
        const RowKernel k = row_kernel(ks == 2 ? SHARES_2 : ROWS_256, D);
        q[ks - 1] = dq_blocks(k.rows, k.key_log2, cost.q_step_us[ks - 1], cost.q_fixed_us[ks - 1], false);
        q_total[ks - 1] = q[ks - 1].total_us();
        q_longest[ks - 1] = q[ks - 1].longest_us();
    }
    for (int n = 1; n <= 16; n *= 2) {
        if (n > 1 && (!may_split || pairs * tiles_seen * n > 5LL * cus || (double)pairs * tiles_seen * n * 128 * D * 8 > MAX_PART_BYTES)) break;
        if (n > 1 && n > (long long)(Sq + 63) / 64 * n_rep) break;
        const List kv = kv_blocks(n, cost.kv_step_us, cost.kv_fixed_us);
        const double kv_total = kv.total_us(), kv_longest = kv.longest_us();
        std::optional<Dispatch> after_kv;
        int reps = 1;
        while (reps * 2 <= n && n_rep % (reps * 2) == 0) reps *= 2;
        for (int ks = 1; ks <= 2; ks++) {
            const bool one_round = q[ks - 1].n + kv.n <= cus;
            const bool own = ks == 2 && one_round && (flags & LTR_DELTA_FROM_O) && (long long)n_rep / reps * Sq <= own_delta_rows(D);
            const double rest = cost.launch_us + (own ? 0.5 : delta_us) + reduce_us(n);
            if (rest + std::max((q_total[ks - 1] + kv_total) / cus, std::max(q_longest[ks - 1], kv_longest)) >= best) continue;
            for (int first = 0; first < (one_round ? 1 : 2); first++) {
                const List &one = first ? kv : q[ks - 1], &other = first ? q[ks - 1] : kv;
                std::optional<Dispatch> &after_one = first ? after_kv : after_q[ks - 1];
                if (!after_one) after_one.emplace(cus).add(one.c, one.k);
                Dispatch both(*after_one);
                if (!both.add(other.c, other.k, best - rest)) continue;
                const double us = rest + both.end;
                if (us < best) {
                    best = us;
                    best_ks = ks;
                    best_n = n;
                    keys_first = first;
                    pl.own_delta = own;
                }
            }
        }
    }
    if (!best_ks) return;
    if (best_n == 1 && pl.split.n > 1 && best >= apart_us(alone)) {
        pl = alone;
        return;
    }
    pl.joint = true;
    pl.keys_first = keys_first;
    pl.key_waves = pl.dq_four_waves = false;
    pl.dq_ks = best_ks;
    pl.dq_rows = 256 / best_ks;
    pl.dq_qtiles = pl.dq_slots = (Sq + pl.dq_rows - 1) / pl.dq_rows;
    pl.dq_blocks = (long long)pl.dq_slots * B * Hq;
    pl.split = {best_n, 1, best_n > 1 ? q_last : 0x7fffffff, best_n > 1 ? tiles_seen : pl.kv_tiles, 0};
    while (pl.split.reps * 2 <= best_n && Hq / Hkv % (pl.split.reps * 2) == 0) pl.split.reps *= 2;
}
BwdPlan make_bwd_plan(int D, bool f32, unsigned flags, int B, int Hq, int Hkv, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk,
                      int n_chunks, bool may_split) {
    BwdPlan pl;
    pl.f32_ks = 0;
    pl.split = KvSplit{1, 1, 0x7fffffff, 0, 0};
    pl.part_bytes = 0;
    pl.dq_ks = 1;
    pl.dq_group = pl.kv_group = 1;
    pl.dq_four_waves = pl.joint = pl.keys_first = pl.own_delta = false;
    may_split = may_split && !(flags & (LTR_NO_DKDV | LTR_BWD_F32_SCALAR));
    pl.key_waves = false;
    const int cus = device_cus();
    auto split_keys = [&](const KvSplitCost &cost, int max_n) {
        return kv_split(cost, max_n, D, pl.keys_per_block, (flags & LTR_CAUSAL) != 0, B, Hkv, Hq / Hkv, Sq, q_split, q_pos0, chunk, n_chunks, cus);
    };
    auto size_parts = [&]() {
        if (pl.split.n > 1) pl.part_bytes = (int64_t)pl.split.tiles * B * Hkv * pl.split.n * pl.keys_per_block * D * 2 * 4;
    };
    if (f32) {
        pl.wide_kv = pl.wide_q = false;
        if (flags & LTR_BWD_F32_SCALAR) {
            pl.keys_per_block = 64;
            pl.dq_rows = 64;
        } else {
            // matrix-pipe kernels: 128 keys per dK/dV block; the dQ kernel sized like the fp32 forward (see plan_fwd)
            pl.keys_per_block = 128;
            pl.dq_rows = f32_rows(D, (long long)B * Hq, Sq, cus, pl.f32_ks);
        }
        pl.kv_tiles = 0;
        for (int c = 0; c < n_chunks; c++) pl.kv_tiles += (chunk[c].sk + pl.keys_per_block - 1) / pl.keys_per_block;
        pl.kv_blocks = pl.kv_tiles * B * Hkv;
        // fp32 sums of more than 4096 rows keep their one serial order, and with it their rounding: shared sums are nearer to fp64
        // (4 q heads on one kv head, D=128, causal, error of dK relative to its norm, whole / shared: 4096 rows 1.3e-6 / 5.3e-7, 27064 rows
        // 3.1e-6 / 9.6e-7; largest single error in units of the rms 4e-5 / 1e-5 and 2.5e-4 / 5e-5) and faster (8513 / 1081 us at
        // 27064), but they would move single elements by the whole sum's error, which from about here on exceeds 1e-4 of them:
        // the tolerance to which results of this path are to stay the same
        may_split = may_split && (long long)(Hq / Hkv) * Sq <= 4096;
        pl.split = split_keys(D == 128 ? KvSplitCost{32, 9.0, 18.0, 9.0, 18.0, 0.25, 2.0, 6e6} : KvSplitCost{32, 4.5, 6.75, 4.5, 6.75, 0.25, 2.0, 6e6},
                              may_split ? 32 : 1);
        size_parts();
        pl.dq_qtiles = pl.dq_slots = (Sq + pl.dq_rows - 1) / pl.dq_rows;
        pl.dq_blocks = (long long)pl.dq_qtiles * B * Hq;
        return pl;
    }
    const bool causal_ = (flags & LTR_CAUSAL) != 0;
    // keys per block of the dK/dV kernel: 256 (two 32-key halves per wave) pays at head dim 64 for long equal blocks without any masked
    // tile, against bwd_dkdv_keywave_kernel (us, 256 keys / one wave per 32 keys, no mask): 128 heads S=4096 1000 / 1060, 128 heads S=2048 263 / 276,
    // 192 heads S=1024 116 / 115; with tails 160 heads S=1231 562 / 443 (its masked pass spills), causal 30 heads S=2571 315 / 235
    bool wide = (flags & LTR_DKDV_KEYS_256) != 0;
    if (!wide && !(flags & LTR_DKDV_KEYS_128) && D == 64 && !(flags & (LTR_NO_DKDV | LTR_HEAD_COLS))) {
        long long blocks256 = 0, blocks128 = 0;
        bool tails = Sq % 64 != 0;
        for (int c = 0; c < n_chunks; c++) {
            blocks256 += (chunk[c].sk + 255) / 256;
            blocks128 += (chunk[c].sk + 127) / 128;
            tails = tails || chunk[c].sk % 256 != 0;
        }
        blocks256 *= (long long)B * Hkv;
        blocks128 *= (long long)B * Hkv;
        const long long q_tiles = (long long)(Hq / Hkv) * (Sq / 64);
        wide = !causal_ && !tails && q_tiles >= 32 && cu_fill(blocks256, cus) * 1.12 >= cu_fill(blocks128, cus);
    }
    pl.wide_kv = wide;
    pl.keys_per_block = wide ? BwdLds<64, 2>::BN : BwdLds<64, 1>::BN;
    pl.kv_tiles = 0;
    for (int c = 0; c < n_chunks; c++) pl.kv_tiles += (chunk[c].sk + pl.keys_per_block - 1) / pl.keys_per_block;
    pl.kv_blocks = pl.kv_tiles * B * Hkv;
    auto choose_kv = [&](BwdPlan &x, int max_n) {   // the kernel of whole or shared key tiles
        x.key_waves = false;
        if (D == 128 || (flags & LTR_HEAD_COLS) || wide) {
            x.split = split_keys(D == 128 ? KvSplitCost{64, 1.4, 11.2, 1.4, 11.2, 0.25, 2.0, 8e6}
                                          : wide ? KvSplitCost{64, 1.9, 11.4, 1.9, 11.4, 0.25, 2.0, 6e6} : KvSplitCost{64, 1.0, 8.0, 1.0, 8.0, 0.25, 2.0, 6e6}, max_n);
            return;
        }
        // head dim 64: one wave per 32 keys (two blocks per CU) or two (one block).  A block alone on its CU is faster with eight
        // waves, a CU is faster with two blocks of four.  Constants fitted to 195 launches each (60 shapes, n = 1 .. 32; rms 7 %)
        const KvSplit one_wave = split_keys(KEY_WAVES_64, max_n);
        x.split = split_keys(KvSplitCost{64, 1.14, 7.0, 1.01, 5.8, 0.6, 4.0, 17e6}, max_n);
        x.key_waves = one_wave.us < 0.96 * x.split.us;
        if (x.key_waves) x.split = one_wave;
    };
    choose_kv(pl, may_split ? 32 : 1);
    const RowChoice choice = flags & LTR_NO_DQ
                                 ? RowChoice{flags & LTR_DQ_ROWS_512 ? ROWS_512 : ROWS_256, false}
                                 : choose_rows(D == 128 ? DQ_ROWS_128 : DQ_ROWS_64,
                                               allowed_rows(flags & LTR_DQ_ROWS_256, flags & LTR_DQ_ROWS_512, true, flags & LTR_HEAD_COLS, D), D, causal_,
                                               (long long)B * Hq, (long long)B * Hkv, Sq, q_split, q_pos0, chunk, n_chunks, cus);
    pl.wide_q = choice.kernel == ROWS_512;
    pl.dq_four_waves = choice.kernel == FOUR_WAVES;
    pl.dq_ks = choice.kernel == SHARES_2 ? 2 : choice.kernel == SHARES_4 ? 4 : 1;
    pl.dq_rows = row_kernel(choice.kernel, D).rows;
    pl.dq_qtiles = (Sq + pl.dq_rows - 1) / pl.dq_rows;
    bool uneven = causal_ && q_tiles_uneven(Sq, pl.dq_rows, q_split, q_pos0, chunk, n_chunks);
    pl.dq_slots = choice.paired ? (pl.dq_qtiles + 1) / 2 : pl.dq_ks > 1 || pl.dq_four_waves ? pl.dq_qtiles : q_tile_slots(pl.dq_qtiles, (long long)B * Hq, uneven, cus);
    pl.dq_blocks = (long long)pl.dq_slots * B * Hq;
    constexpr unsigned NOT_JOINT = LTR_NO_DQ | LTR_NO_DKDV | LTR_DQ_ROWS_256 | LTR_DQ_ROWS_512 | LTR_DKDV_KEYS_128 | LTR_DKDV_KEYS_256;
    if ((flags & LTR_BWD_JOINT) && !(flags & NOT_JOINT) && !pl.wide_q && !pl.wide_kv) {
        BwdPlan alone = pl;
        if (pl.split.n > 1) choose_kv(alone, 1);
        joint_launch(pl, alone, D, flags, B, Hq, Hkv, Sq, q_split, q_pos0, chunk, n_chunks, may_split, cus);
        if (pl.joint) uneven = causal_ && q_tiles_uneven(Sq, pl.dq_rows, q_split, q_pos0, chunk, n_chunks);
    }
    size_parts();
    const long long pairs = (long long)B * Hkv;
    const int slots = cus / 8;
    pl.dq_group = pair_group(pairs, (long long)pl.dq_slots * (Hq / Hkv), slots * (pl.dq_four_waves ? D == 64 ? FourWaves<64>::PER_CU : FourWaves<128>::PER_CU : 1),
                             uneven && pl.dq_slots == pl.dq_qtiles);
    pl.kv_group = pair_group(pairs, (pl.split.n > 1 ? pl.split.tiles : pl.kv_tiles) * pl.split.n, pl.key_waves ? 2 * slots : slots,
                             causal_ && key_tiles_uneven(Sq, pl.keys_per_block, q_split, q_pos0, chunk, n_chunks));
    return pl;
}
// The plan of a problem.  One with LTR_BWD_JOINT prices up to 20 launches (1 - 11 us: 4 x 12 heads of 64, S=100 1.5, 8 heads of 64, S=4000 7.6,
// a zig-zag rank of 8 with 8000 rows 10.6), and a backward asks twice, for the workspace and for the launch.
BwdPlan plan_bwd(int D, bool f32, unsigned flags, int B, int Hq, int Hkv, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk,
                 int n_chunks, bool may_split = false) {
    auto make = [&] { return make_bwd_plan(D, f32, flags, B, Hq, Hkv, Sq, q_split, q_pos0, chunk, n_chunks, may_split); };
    if (!(flags & LTR_BWD_JOINT) || f32) return make();
    static thread_local KeptPlans<BwdPlan> kept;
    return kept.get(Problem(D, flags, B, Hq, Hkv, Sq, q_split, q_pos0, chunk, n_chunks, may_split), make);
}
// The plan with a workspace of that many bytes: shared key tiles if their partial sums fit, else the launch without a workspace (whose kernel
// and block order are other ones than those chosen for sharing).  A joint plan that shares no tiles fits no workspace as well: it is not priced again.
BwdPlan plan_bwd_ws(int D, bool f32, unsigned flags, int B, int Hq, int Hkv, int Sq, int q_split, const int *q_pos0, const ChunkDev *chunk, int n_chunks,
                    int64_t work_bytes) {
    if (work_bytes > 0 || (flags & LTR_BWD_JOINT)) {
        const BwdPlan pl = plan_bwd(D, f32, flags, B, Hq, Hkv, Sq, q_split, q_pos0, chunk, n_chunks, true);
        if (pl.part_bytes <= work_bytes) return pl;
    }
    return plan_bwd(D, f32, flags, B, Hq, Hkv, Sq, q_split, q_pos0, chunk, n_chunks);
}
// blocks of bwd_dkdv_reduce_kernel: four waves each, one per 64 columns of a 32-key slice of dK or dV
long long reduce_blocks(const BwdPlan &pl, int D) { return pl.kv_blocks * (pl.keys_per_block / 128) * (D / 32); }

// every position of the local rows lies inside the rows [pos0, pos0 + len) of a RoPE table
bool rope_table_covers(const int64_t *q_pos0, int64_t q_split, int64_t Sq, int64_t pos0, int64_t len) {
    if (len <= 0 || !fits_i32(pos0)) return false;
    if (q_split > 0 && (q_pos0[0] < pos0 || q_pos0[0] + q_split > pos0 + len)) return false;
    if (Sq > q_split && (q_pos0[1] < pos0 || q_pos0[1] + (Sq - q_split) > pos0 + len)) return false;
    return true;
}

// ------------------------------------------------------------------------------ fixed scratch
// DELTA workspace of ltr_attn_bwd_noalloc: a fixed array in device memory that belongs to the library (every device the
// library runs on holds its own copy until the process ends).  Host code never uses the array's name as an address: the
// device address of the current device's copy is looked up once per device (scratch_address) and passed to the kernels
// like any caller-owned workspace.
}  // namespace
static __device__ __align__(256) float scratch[LTR_NOALLOC_MAX_ROWS];
namespace {

int scratch_address(float **out) {
    int dev = 0;
    if (current_device(&dev)) return LTR_EDEVICE;
    float *ptr = g_dev[dev].scratch.load(std::memory_order_acquire);
    if (!ptr) {
        void *sym = nullptr;
        if (hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)) != hipSuccess || !sym) {
            (void)hipGetLastError();
            return LTR_ELAUNCH;
        }
        ptr = (float *)sym;
        g_dev[dev].scratch.store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return LTR_OK;
}

}  // namespace

extern "C" int ltr_abi_version(void) { return LTR_ABI_VERSION; }

extern "C" const char *ltr_strerror(int code) {
    switch (code) {
        case LTR_OK: return "ok";
        case LTR_EINVAL: return "invalid argument (null pointer, bad size or flag)";
        case LTR_EUNSUP: return "unsupported head dim / dtype combination";
        case LTR_EALIGN: return "pointer or stride not 16-byte aligned";
        case LTR_ELAUNCH: return "HIP launch error";
        case LTR_EDEVICE: return "current device is not gfx950";
        case LTR_ETOOBIG: return "size beyond the fixed scratch of the no-allocation entry point";
        default: return "unknown error";
    }
}

extern "C" int ltr_attn_fwd(const ltr_attn_fwd_args *a, void *stream) {
    if (!a || !a->q || !a->o || !a->lse) return LTR_EINVAL;
    if (a->B <= 0 || a->Hq <= 0 || a->Hkv <= 0 || a->Sq <= 0 || a->Hq % a->Hkv) return LTR_EINVAL;
    if (a->n_chunks < 1 || a->n_chunks > LTR_MAX_CHUNKS) return LTR_EINVAL;
    if (a->flags & ~(LTR_CAUSAL | LTR_MERGE | LTR_ROPE_Q | LTR_FWD_ROWS_256 | LTR_FWD_ROWS_512 | LTR_FWD_F32_SCALAR | LTR_HEAD_COLS))
        return LTR_EINVAL;
    if ((a->flags & LTR_FWD_F32_SCALAR) && a->io_dtype != LTR_F32) return LTR_EUNSUP;
    if ((a->flags & LTR_FWD_ROWS_256) && (a->flags & LTR_FWD_ROWS_512)) return LTR_EINVAL;
    const int D = head_width(a->D, a->flags);
    const bool pad = D != a->D;
    if (!D) return LTR_EUNSUP;
    if (a->io_dtype != LTR_BF16 && a->io_dtype != LTR_F32) return LTR_EUNSUP;
    if (pad && a->io_dtype != LTR_BF16) return LTR_EUNSUP;
    if (a->o_dtype != LTR_BF16 && a->o_dtype != LTR_F32) return LTR_EUNSUP;
    if (a->io_dtype == LTR_F32 && a->o_dtype != LTR_F32) return LTR_EUNSUP;
    if (!fits_i32(a->Sq) || a->q_split < 0 || a->q_split > a->Sq) return LTR_EINVAL;
    if (!fits_i32(a->q_pos0[0] + a->Sq) || !fits_i32(a->q_pos0[1] + a->Sq)) return LTR_EINVAL;
    const int eb = a->io_dtype == LTR_BF16 ? 2 : 4, ob = a->o_dtype == LTR_BF16 ? 2 : 4;
    if (!aligned16(a->q) || !aligned16(a->o) || !aligned16(a->lse)) return LTR_EALIGN;
    if (!strides_ok(a->q_stride, eb) || !strides_ok(a->k_stride, eb) || !strides_ok(a->v_stride, eb)) return LTR_EALIGN;
    // o rows are written in 4-element groups
    for (int i = 0; i < 3; i++)
        if (a->o_stride[i] < 0 || (a->o_stride[i] * ob) % 8) return LTR_EALIGN;
    FwdParams p;
    p.rope = nullptr;
    p.rope_pos0 = 0;
    p.q_rot = nullptr;
    for (int i = 0; i < 3; i++) p.qrs[i] = 0;
    if (a->flags & LTR_ROPE_Q) {
        if (a->io_dtype != LTR_BF16) return LTR_EUNSUP;
        if (!a->rope_freqs) return LTR_EINVAL;
        if (!rope_table_covers(a->q_pos0, a->q_split, a->Sq, a->rope_pos0, a->rope_len)) return LTR_EINVAL;
        if (!aligned16(a->rope_freqs) || (a->q_rot && (!aligned16(a->q_rot) || !strides_ok(a->q_rot_stride, 2)))) return LTR_EALIGN;
        p.rope = a->rope_freqs;
        p.rope_pos0 = (int)a->rope_pos0;
        p.q_rot = a->q_rot;
        for (int i = 0; i < 3; i++) p.qrs[i] = a->q_rot ? a->q_rot_stride[i] : 0;
    }
    for (int c = 0; c < a->n_chunks; c++) {
        const ltr_kv_chunk &ch = a->chunk[c];
        if (!ch.k || !ch.v || ch.sk <= 0 || !fits_i32(ch.sk) || !fits_i32(ch.pos0 + ch.sk)) return LTR_EINVAL;
        if (!aligned16(ch.k) || !aligned16(ch.v)) return LTR_EALIGN;
        // tile offsets inside a chunk are 32-bit element counts
        if ((ch.sk + 64) * a->k_stride[1] >= 0x7fffffffLL || (ch.sk + 64) * a->v_stride[1] >= 0x7fffffffLL) return LTR_EUNSUP;
        p.chunk[c].k = ch.k;
        p.chunk[c].v = ch.v;
        p.chunk[c].dk = nullptr;
        p.chunk[c].dv = nullptr;
        p.chunk[c].sk = (int)ch.sk;
        p.chunk[c].pos0 = (int)ch.pos0;
    }
    int rc = check_device();
    if (rc) return rc;
    p.q = a->q;
    p.o = a->o;
    p.lse = a->lse;
    p.B = a->B;
    p.Hq = a->Hq;
    p.Hkv = a->Hkv;
    p.n_rep = a->Hq / a->Hkv;
    p.Sq = (int)a->Sq;
    for (int i = 0; i < 3; i++) {
        p.qs[i] = a->q_stride[i];
        p.os[i] = a->o_stride[i];
        p.ks[i] = a->k_stride[i];
        p.vs[i] = a->v_stride[i];
    }
    p.q_pos0[0] = (int)a->q_pos0[0];
    p.q_pos0[1] = (int)a->q_pos0[1];
    p.q_split = (int)a->q_split;
    p.scale = a->scale;
    p.flags = a->flags & (LTR_CAUSAL | LTR_MERGE | LTR_ROPE_Q);
    p.o_f32 = a->o_dtype == LTR_F32;
    p.n_chunks = a->n_chunks;
    hipStream_t st = (hipStream_t)stream;
    if ((a->flags & LTR_FWD_ROWS_512) && (a->D != 64 || a->io_dtype != LTR_BF16)) return LTR_EUNSUP;
    p.cols = a->D;
    const FwdPlan pl = plan_fwd(D, a->io_dtype == LTR_F32, pad ? a->flags : a->flags & ~LTR_HEAD_COLS, p.B, p.Hq, p.Hkv, p.Sq, p.q_split, p.q_pos0, p.chunk, p.n_chunks,
                                // q rotated in place: a row is read and written by one wave only without key shares
                                !p.q_rot || p.q_rot != p.q);
    if (pl.blocks > 0x7fffffffLL) return LTR_EINVAL;
    p.n_qtiles = pl.n_qtiles;
    p.n_slots = pl.n_slots;
    const BlockGrid grid = block_grid((long long)p.B * p.Hkv, pl.n_slots, p.n_rep, pl.group);
    p.map = grid.map;
    if (a->io_dtype == LTR_BF16) {
        rc = enable_large_lds();
        if (rc) return rc;
        if (pad) {
            const int i = pl.ks >> 1;
            using Three = Columns96<FwdParams>;
            const void *const kernels[3][3] = {
                {kernel_of<FwdParams>(fwd_bf16_pad_kernel<64, 1>), kernel_of<FwdParams>(fwd_bf16_pad_kernel<64, 2>), kernel_of<FwdParams>(fwd_bf16_pad_kernel<64, 4>)},
                {kernel_of<FwdParams>(fwd_bf16_pad_kernel<128, 1>), kernel_of<FwdParams>(fwd_bf16_pad_kernel<128, 2>), kernel_of<FwdParams>(fwd_bf16_pad_kernel<128, 4>)},
                {kernel_of<Three>(fwd_bf16_pad_kernel<128, 1>), kernel_of<Three>(fwd_bf16_pad_kernel<128, 2>), kernel_of<Three>(fwd_bf16_pad_kernel<128, 4>)}};
            const int lds[2][3] = {{fwd_lds_bytes<64>(), shares_lds_bytes<64, 2>(), shares_lds_bytes<64, 4>()},
                                   {fwd_lds_bytes<128>(), shares_lds_bytes<128, 2>(), shares_lds_bytes<128, 4>()}};
            return launch(kernels[D == 64 ? 0 : a->D > 96 ? 1 : 2][i], dims(grid), 512, lds[D == 128][i], st, p);
        }
        if (pl.four_waves)
            return a->D == 128 ? launch((const void *)fwd_bf16_w4_kernel<128>, dims(grid), 256, FourWaves<128>::LDS, st, p)
                               : launch((const void *)fwd_bf16_w4_kernel<64>, dims(grid), 256, FourWaves<64>::LDS, st, p);
        if (pl.ks == 2)
            return a->D == 128 ? launch((const void *)fwd_bf16_shares_kernel<128, 2>, dims(grid), 512, shares_lds_bytes<128, 2>(), st, p)
                               : launch((const void *)fwd_bf16_shares_kernel<64, 2>, dims(grid), 512, shares_lds_bytes<64, 2>(), st, p);
        if (pl.ks == 4)
            return a->D == 128 ? launch((const void *)fwd_bf16_shares_kernel<128, 4>, dims(grid), 512, shares_lds_bytes<128, 4>(), st, p)
                               : launch((const void *)fwd_bf16_shares_kernel<64, 4>, dims(grid), 512, shares_lds_bytes<64, 4>(), st, p);
        if (a->D == 128) return launch((const void *)fwd_bf16_kernel<128, 1>, dims(grid), 512, fwd_lds_bytes<128>(), st, p);
        if (pl.wide) return launch((const void *)fwd_bf16_kernel<64, 2>, dims(grid), 512, fwd_lds_bytes<64, 2>(), st, p);
        return launch((const void *)fwd_bf16_kernel<64, 1>, dims(grid), 512, fwd_lds_bytes<64>(), st, p);
    }
    if (pl.f32_ks) {   // fp32 on the matrix pipe; the chunk offsets of its LDS-direct loads are 64-bit, nothing more to check
        rc = enable_large_lds();
        if (rc) return rc;
        const KernelChoice k = f32_fwd_kernel(a->D, pl.f32_ks, pl.rows);
        return launch(k.fn, pl.blocks, 256, k.lds, st, p);
    }
    if (a->D == 128) return launch((const void *)fwd_f32_kernel<128>, pl.blocks, 64, 0, st, p);
    return launch((const void *)fwd_f32_kernel<64>, pl.blocks, 64, 0, st, p);
}

extern "C" int ltr_attn_bwd_delta(const ltr_attn_delta_args *a, void *stream) {
    if (!a || !a->o || !a->d_o || !a->delta) return LTR_EINVAL;
    if (a->B <= 0 || a->Hq <= 0 || a->Sq <= 0 || !fits_i32(a->Sq)) return LTR_EINVAL;
    if (a->D <= 0 || a->D > 128 || a->D % 8) return LTR_EUNSUP;
    if ((a->o_dtype != LTR_BF16 && a->o_dtype != LTR_F32) || (a->do_dtype != LTR_BF16 && a->do_dtype != LTR_F32))
        return LTR_EUNSUP;
    for (int i = 0; i < 3; i++)
        if (a->o_stride[i] < 0 || a->do_stride[i] < 0) return LTR_EINVAL;
    int rc = check_device();
    if (rc) return rc;
    DeltaParams p;
    p.o = a->o;
    p.d_o = a->d_o;
    p.delta = a->delta;
    p.B = a->B;
    p.Hq = a->Hq;
    p.D = a->D;
    p.Sq = (int)a->Sq;
    for (int i = 0; i < 3; i++) {
        p.os[i] = a->o_stride[i];
        p.dos[i] = a->do_stride[i];
    }
    p.o_f32 = a->o_dtype == LTR_F32;
    p.do_f32 = a->do_dtype == LTR_F32;
    p.rows32 = fits_i32((int64_t)a->B * a->Sq);
    p.vec = aligned16(a->o) && aligned16(a->d_o) && strides_ok(a->o_stride, p.o_f32 ? 4 : 2) && strides_ok(a->do_stride, p.do_f32 ? 4 : 2);
    const long long rows = (long long)p.B * p.Hq * p.Sq;
    if (p.vec && !p.o_f32 && !p.do_f32 && rows <= 0x7fffffffLL)
        return p.D <= 64 ? launch((const void *)delta_bf16_kernel<8>, (rows + 63) / 64, 256, 0, (hipStream_t)stream, p)
                         : launch((const void *)delta_bf16_kernel<16>, (rows + 31) / 32, 256, 0, (hipStream_t)stream, p);
    const long long nthreads = rows * 16;
    const long long nblk = (nthreads + 255) / 256;
    if (nblk > 0x7fffffffLL) return LTR_EINVAL;
    return launch((const void *)delta_kernel, nblk, 256, 0, (hipStream_t)stream, p);
}

namespace {
// ltr_attn_bwd (DELTA is the caller's buffer) and ltr_attn_bwd_noalloc (use_scratch: DELTA lives in the library's fixed
// scratch array; flags already carry LTR_DELTA_FROM_O); work: the caller's workspace for partial dK / dV, or nullptr
int bwd_launch(const ltr_attn_bwd_args *a, unsigned flags, bool use_scratch, void *stream, void *work = nullptr, int64_t work_bytes = 0) {
    float *delta = use_scratch ? nullptr : a->delta;
    if (!a->q || !a->d_o || !a->lse || (!use_scratch && !delta)) return LTR_EINVAL;
    const bool do_dq = !(flags & LTR_NO_DQ), do_dkdv = !(flags & LTR_NO_DKDV);
    if (do_dq && !a->dq) return LTR_EINVAL;
    if (a->B <= 0 || a->Hq <= 0 || a->Hkv <= 0 || a->Sq <= 0 || a->Hq % a->Hkv) return LTR_EINVAL;
    if (a->n_chunks < 1 || a->n_chunks > LTR_MAX_CHUNKS) return LTR_EINVAL;
    if (flags & ~(LTR_CAUSAL | LTR_NO_DQ | LTR_NO_DKDV | LTR_DQ_BF16 | LTR_DELTA_FROM_O | LTR_DKDV_BF16 | LTR_ROPE_DQ | LTR_DKDV_KEYS_128 |
                  LTR_DKDV_KEYS_256 | LTR_DQ_ROWS_256 | LTR_DQ_ROWS_512 | LTR_BWD_F32_SCALAR | LTR_HEAD_COLS | LTR_DQ_F32_RESULT | LTR_BWD_JOINT))
        return LTR_EINVAL;
    if ((flags & LTR_BWD_F32_SCALAR) && a->io_dtype != LTR_F32) return LTR_EUNSUP;
    if ((flags & LTR_DQ_F32_RESULT) && (a->io_dtype != LTR_F32 || (flags & LTR_BWD_F32_SCALAR))) return LTR_EUNSUP;
    if ((flags & LTR_DKDV_KEYS_128) && (flags & LTR_DKDV_KEYS_256)) return LTR_EINVAL;
    if ((flags & LTR_DQ_ROWS_256) && (flags & LTR_DQ_ROWS_512)) return LTR_EINVAL;
    const bool fused_delta = flags & (LTR_DELTA_FROM_O | LTR_DQ_F32_RESULT);
    if (fused_delta && (!do_dq || !a->o)) return LTR_EINVAL;
    const int D = head_width(a->D, flags);
    const bool pad = D != a->D;
    if (!D) return LTR_EUNSUP;
    if (a->io_dtype != LTR_BF16 && a->io_dtype != LTR_F32) return LTR_EUNSUP;
    const bool f32 = a->io_dtype == LTR_F32;
    if (pad && f32) return LTR_EUNSUP;
    if (!pad) flags &= ~LTR_HEAD_COLS;
    if (f32 && (flags & (LTR_DQ_BF16 | LTR_DELTA_FROM_O | LTR_DKDV_BF16 | LTR_ROPE_DQ | LTR_DKDV_KEYS_256 | LTR_DQ_ROWS_512)))
        return LTR_EUNSUP;   // bf16 conveniences and kernels only
    const int gb = (flags & LTR_DKDV_BF16) ? 2 : 4;   // bytes per dK / dV element
    const int eb = f32 ? 4 : 2;
    if (!fits_i32(a->Sq) || a->q_split < 0 || a->q_split > a->Sq) return LTR_EINVAL;
    if (!fits_i32(a->q_pos0[0] + a->Sq) || !fits_i32(a->q_pos0[1] + a->Sq)) return LTR_EINVAL;
    if (!aligned16(a->q) || !aligned16(a->d_o) || (do_dq && !aligned16(a->dq))) return LTR_EALIGN;
    if (!strides_ok(a->q_stride, eb) || !strides_ok(a->do_stride, eb) || !strides_ok(a->k_stride, eb) ||
        !strides_ok(a->v_stride, eb) || !strides_ok(a->dk_stride, gb) || !strides_ok(a->dv_stride, gb))
        return LTR_EALIGN;
    for (int i = 0; i < 3; i++)
        if (a->dq_stride[i] < 0) return LTR_EINVAL;
    if (do_dq && !strides_ok(a->dq_stride, (flags & LTR_DQ_BF16) ? 2 : 4)) return LTR_EALIGN;
    if (fused_delta && (!aligned16(a->o) || !strides_ok(a->o_stride, eb))) return LTR_EALIGN;
    if (fused_delta && !f32 && (a->Sq + 64) * a->o_stride[1] >= 0x7fffffffLL) return LTR_EUNSUP;
    if ((a->Sq + 63) / 64 > BwdLds<128, 1>::MAX_QTILES) return LTR_EUNSUP;       // q tile lists live in LDS
    if ((a->Sq + 64) * a->q_stride[1] >= 0x7fffffffLL || (a->Sq + 64) * a->do_stride[1] >= 0x7fffffffLL) return LTR_EUNSUP;
    BwdParams p;
    p.rope = nullptr;
    p.rope_pos0 = 0;
    if (flags & LTR_ROPE_DQ) {
        if (!do_dq || !a->rope_freqs) return LTR_EINVAL;
        if (!rope_table_covers(a->q_pos0, a->q_split, a->Sq, a->rope_pos0, a->rope_len)) return LTR_EINVAL;
        if (!aligned16(a->rope_freqs)) return LTR_EALIGN;
        p.rope = a->rope_freqs;
        p.rope_pos0 = (int)a->rope_pos0;
    }
    if ((flags & LTR_DKDV_KEYS_256) && (a->D != 64 || f32)) return LTR_EUNSUP;
    if ((flags & LTR_DQ_ROWS_512) && a->D != 64) return LTR_EUNSUP;
    for (int c = 0; c < a->n_chunks; c++) {
        const ltr_kv_chunk &ch = a->chunk[c];
        if (!ch.k || !ch.v || ch.sk <= 0 || !fits_i32(ch.sk) || !fits_i32(ch.pos0 + ch.sk)) return LTR_EINVAL;
        if (do_dkdv && (!ch.dk || !ch.dv)) return LTR_EINVAL;
        if ((ch.sk + 64) * a->k_stride[1] >= 0x7fffffffLL || (ch.sk + 64) * a->v_stride[1] >= 0x7fffffffLL) return LTR_EUNSUP;
        if (!aligned16(ch.k) || !aligned16(ch.v)) return LTR_EALIGN;
        if (do_dkdv && (!aligned16(ch.dk) || !aligned16(ch.dv))) return LTR_EALIGN;
        p.chunk[c].k = ch.k;
        p.chunk[c].v = ch.v;
        p.chunk[c].dk = (float *)ch.dk;
        p.chunk[c].dv = (float *)ch.dv;
        p.chunk[c].sk = (int)ch.sk;
        p.chunk[c].pos0 = (int)ch.pos0;
    }
    int rc = check_device();
    if (rc) return rc;
    if (use_scratch) {
        rc = scratch_address(&delta);
        if (rc) return rc;
    }
    p.q = a->q;
    p.d_o = a->d_o;
    p.lse = a->lse;
    p.delta = delta;
    p.o = a->o;
    for (int i = 0; i < 3; i++) p.os_[i] = fused_delta ? a->o_stride[i] : 0;
    p.dq = a->dq;
    p.B = a->B;
    p.Hq = a->Hq;
    p.Hkv = a->Hkv;
    p.n_rep = a->Hq / a->Hkv;
    p.Sq = (int)a->Sq;
    p.n_qtiles = (p.Sq + 63) / 64;
    for (int i = 0; i < 3; i++) {
        p.qs[i] = a->q_stride[i];
        p.dos[i] = a->do_stride[i];
        p.dqs[i] = a->dq_stride[i];
        p.ks[i] = a->k_stride[i];
        p.vs[i] = a->v_stride[i];
        p.dks[i] = a->dk_stride[i];
        p.dvs[i] = a->dv_stride[i];
    }
    p.q_pos0[0] = (int)a->q_pos0[0];
    p.q_pos0[1] = (int)a->q_pos0[1];
    p.q_split = (int)a->q_split;
    p.scale = a->scale;
    p.flags = flags;
    p.n_chunks = a->n_chunks;
    p.cols = a->D;
    const BwdPlan pl = plan_bwd_ws(D, f32, flags, p.B, p.Hq, p.Hkv, p.Sq, p.q_split, p.q_pos0, p.chunk, p.n_chunks, work ? work_bytes : 0);
    p.q_last = pl.split.n > 1 ? pl.split.q_last : 0x7fffffff;
    const long long tiles_seen = pl.split.n > 1 ? pl.split.tiles : pl.kv_tiles;
    const long long kv_grid = tiles_seen * p.B * p.Hkv * pl.split.n, reduce_grid = reduce_blocks(pl, D);
    if (kv_grid > 0x7fffffffLL || reduce_grid > 0x7fffffffLL || pl.dq_blocks > 0x7fffffffLL) return LTR_EINVAL;
    p.tiles_total = (int)pl.kv_tiles;
    p.tiles_seen = (int)tiles_seen;
    p.split_log2 = __builtin_ctz(pl.split.n);
    p.share_log2 = __builtin_ctz(pl.split.n / pl.split.reps);
    p.n_reps = p.n_rep / pl.split.reps;
    p.part = (float *)work;
    p.n_slots = pl.dq_slots;
    const BlockGrid q_grid = block_grid((long long)p.B * p.Hkv, pl.dq_slots, p.n_rep, pl.dq_group);
    const BlockGrid key_grid = block_grid((long long)p.B * p.Hkv, tiles_seen, pl.split.n, pl.kv_group);
    p.q_map = q_grid.map;
    p.kv_map = key_grid.map;
    hipStream_t st = (hipStream_t)stream;
    if (f32 && pl.f32_ks) {   // fp32 on the matrix pipe
        rc = enable_large_lds();
        if (rc) return rc;
        if (do_dq) {
            const KernelChoice k = f32_dq_kernel(a->D, pl.f32_ks, pl.dq_rows);
            rc = launch(k.fn, pl.dq_blocks, 256, k.lds, st, p);
            if (rc) return rc;
        }
        if (do_dkdv) {
            rc = a->D == 128 ? launch((const void *)bwd_dkdv_f32_mfma_kernel<128>, kv_grid, 256, F32DkdvLds<128>::LDS, st, p)
                             : launch((const void *)bwd_dkdv_f32_mfma_kernel<64>, kv_grid, 256, F32DkdvLds<64>::LDS, st, p);
            if (rc || pl.split.n == 1) return rc;
            rc = a->D == 128 ? launch((const void *)bwd_dkdv_reduce_kernel<128, 1>, reduce_grid, 256, 0, st, p)
                             : launch((const void *)bwd_dkdv_reduce_kernel<64, 1>, reduce_grid, 256, 0, st, p);
        }
        return rc;
    }
    if (f32) {
        if (do_dq) {
            rc = a->D == 128 ? launch((const void *)bwd_dq_f32_kernel<128>, pl.dq_blocks, 64, 0, st, p)
                             : launch((const void *)bwd_dq_f32_kernel<64>, pl.dq_blocks, 64, 0, st, p);
            if (rc) return rc;
        }
        if (do_dkdv) {
            rc = a->D == 128 ? launch((const void *)bwd_dkdv_f32_kernel<128, false>, pl.kv_blocks, 64, 0, st, p)
                             : launch((const void *)bwd_dkdv_f32_kernel<64, false>, pl.kv_blocks, 64, 0, st, p);
            if (rc) return rc;
            rc = a->D == 128 ? launch((const void *)bwd_dkdv_f32_kernel<128, true>, pl.kv_blocks, 64, 0, st, p)
                             : launch((const void *)bwd_dkdv_f32_kernel<64, true>, pl.kv_blocks, 64, 0, st, p);
        }
        return rc;
    }
    rc = enable_large_lds();
    if (rc) return rc;
    if (pl.joint) {
        if (fused_delta && !pl.own_delta) {
            ltr_attn_delta_args d{};
            d.o = a->o;
            d.d_o = a->d_o;
            d.delta = delta;
            d.B = a->B;
            d.Hq = a->Hq;
            d.D = a->D;
            d.Sq = a->Sq;
            for (int i = 0; i < 3; i++) {
                d.o_stride[i] = a->o_stride[i];
                d.do_stride[i] = a->do_stride[i];
            }
            d.o_dtype = d.do_dtype = LTR_BF16;
            rc = ltr_attn_bwd_delta(&d, stream);
            if (rc) return rc;
            p.flags &= ~LTR_DELTA_FROM_O;
        }
        if (flags & LTR_CAUSAL)   // longest dK/dV blocks first, as below
            std::stable_sort(p.chunk, p.chunk + p.n_chunks, [](const ChunkDev &x, const ChunkDev &y) { return x.pos0 < y.pos0; });
        const unsigned n_q = map_blocks(p.q_map, p.B * p.Hkv), n_kv = map_blocks(p.kv_map, p.B * p.Hkv);
        p.joint = {pl.keys_first ? n_kv : n_q, pl.keys_first};
        const KernelChoice k = joint_kernel(D, pad, pl.dq_ks, pl.own_delta, a->D);
        rc = launch(k.fn, (long long)n_q + n_kv, 512, k.lds, st, p);
        return rc || pl.split.n == 1 ? rc
               : D == 128            ? launch((const void *)bwd_dkdv_reduce_kernel<128, 1>, reduce_grid, 256, 0, st, p)
                                     : launch((const void *)bwd_dkdv_reduce_kernel<64, 1>, reduce_grid, 256, 0, st, p);
    }
    // the dQ kernel goes first: with LTR_DELTA_FROM_O it produces the DELTA that the dK/dV kernel reads
    if (do_dq) {
        if (pad) {
            const int i = pl.dq_ks >> 1;
            using Three = Columns96<BwdParams>;
            const void *const kernels[3][3] = {
                {kernel_of<BwdParams>(bwd_dq_pad_kernel<64, 1>), kernel_of<BwdParams>(bwd_dq_pad_kernel<64, 2>), kernel_of<BwdParams>(bwd_dq_pad_kernel<64, 4>)},
                {kernel_of<BwdParams>(bwd_dq_pad_kernel<128, 1>), kernel_of<BwdParams>(bwd_dq_pad_kernel<128, 2>), kernel_of<BwdParams>(bwd_dq_pad_kernel<128, 4>)},
                {kernel_of<Three>(bwd_dq_pad_kernel<128, 1>), kernel_of<Three>(bwd_dq_pad_kernel<128, 2>), kernel_of<Three>(bwd_dq_pad_kernel<128, 4>)}};
            const int lds[2][3] = {{dq_lds_bytes<64>(), shares_lds_bytes<64, 2>(), shares_lds_bytes<64, 4>()},
                                   {dq_lds_bytes<128>(), shares_lds_bytes<128, 2>(), shares_lds_bytes<128, 4>()}};
            rc = launch(kernels[D == 64 ? 0 : a->D > 96 ? 1 : 2][i], dims(q_grid), 512, lds[D == 128][i], st, p);
        } else if (pl.dq_four_waves)
            rc = a->D == 128 ? launch((const void *)bwd_dq_w4_kernel<128>, dims(q_grid), 256, FourWaves<128>::LDS, st, p)
                             : launch((const void *)bwd_dq_w4_kernel<64>, dims(q_grid), 256, FourWaves<64>::LDS, st, p);
        else if (pl.dq_ks == 2)
            rc = a->D == 128 ? launch((const void *)bwd_dq_shares_kernel<128, 2>, dims(q_grid), 512, shares_lds_bytes<128, 2>(), st, p)
                             : launch((const void *)bwd_dq_shares_kernel<64, 2>, dims(q_grid), 512, shares_lds_bytes<64, 2>(), st, p);
        else if (pl.dq_ks == 4)
            rc = a->D == 128 ? launch((const void *)bwd_dq_shares_kernel<128, 4>, dims(q_grid), 512, shares_lds_bytes<128, 4>(), st, p)
                             : launch((const void *)bwd_dq_shares_kernel<64, 4>, dims(q_grid), 512, shares_lds_bytes<64, 4>(), st, p);
        else if (a->D == 128) rc = launch((const void *)bwd_dq_kernel<128, 1>, dims(q_grid), 512, dq_lds_bytes<128>(), st, p);
        else if (pl.wide_q) rc = launch((const void *)bwd_dq_kernel<64, 2>, dims(q_grid), 512, dq_lds_bytes<64>(), st, p);
        else rc = launch((const void *)bwd_dq_kernel<64, 1>, dims(q_grid), 512, dq_lds_bytes<64>(), st, p);
        if (rc) return rc;
    }
    if (do_dkdv) {
        // A block of the dK/dV kernel owns 128 keys and loops over the query tiles that see them: under a causal mask its
        // work falls with the keys' position.  The blocks of one (batch, kv head) are handed out in the order of the chunk
        // table, so the table of THIS kernel is sorted by position: the longest blocks start first and the short ones fill
        // the tail (the sums inside a block do not depend on the table's order).
        if (flags & LTR_CAUSAL)
            std::stable_sort(p.chunk, p.chunk + p.n_chunks, [](const ChunkDev &x, const ChunkDev &y) { return x.pos0 < y.pos0; });
        if (pad) rc = D == 64     ? launch(kernel_of<BwdParams>(bwd_dkdv_pad_kernel<64>), dims(key_grid), BwdLds<64, 1>::NT, BwdLds<64, 1>::TOTAL, st, p)
                      : a->D > 96 ? launch(kernel_of<BwdParams>(bwd_dkdv_pad_kernel<128>), dims(key_grid), BwdLds<128, 1>::NT, BwdLds<128, 1>::TOTAL, st, p)
                                  : launch(kernel_of<Columns96<BwdParams>>(bwd_dkdv_pad_kernel<128>), dims(key_grid), BwdLds<128, 1>::NT, BwdLds<128, 1>::TOTAL, st, p);
        else if (a->D == 128) rc = launch((const void *)bwd_dkdv_kernel<128, 1>, dims(key_grid), BwdLds<128, 1>::NT, BwdLds<128, 1>::TOTAL, st, p);
        else if (pl.wide_kv) rc = launch((const void *)bwd_dkdv_kernel<64, 2>, kv_grid, BwdLds<64, 2>::NT, BwdLds<64, 2>::TOTAL, st, p);
        else if (pl.key_waves) rc = launch((const void *)bwd_dkdv_keywave_kernel<64>, dims(key_grid), KeyWaveLds<64>::NT, KeyWaveLds<64>::TOTAL, st, p);
        else rc = launch((const void *)bwd_dkdv_kernel<64, 1>, dims(key_grid), BwdLds<64, 1>::NT, BwdLds<64, 1>::TOTAL, st, p);
        if (rc || pl.split.n == 1) return rc;
        rc = D == 128 ? launch((const void *)bwd_dkdv_reduce_kernel<128, 1>, reduce_grid, 256, 0, st, p)
             : pl.wide_kv ? launch((const void *)bwd_dkdv_reduce_kernel<64, 2>, reduce_grid, 256, 0, st, p)
                          : launch((const void *)bwd_dkdv_reduce_kernel<64, 1>, reduce_grid, 256, 0, st, p);
    }
    return rc;
}
}  // namespace

extern "C" int ltr_attn_bwd(const ltr_attn_bwd_args *a, void *stream) {
    if (!a) return LTR_EINVAL;
    return bwd_launch(a, a->flags, false, stream);
}

extern "C" int ltr_attn_bwd_ws(const ltr_attn_bwd_args *a, void *workspace, int64_t workspace_bytes, void *stream) {
    if (!a || workspace_bytes < 0) return LTR_EINVAL;
    if (workspace && !aligned16(workspace)) return LTR_EALIGN;
    return bwd_launch(a, a->flags, false, stream, workspace, workspace_bytes);
}

// Host-only: sizes, positions and flags are read, no pointer.
extern "C" int ltr_attn_bwd_workspace(const ltr_attn_bwd_args *a, int64_t *bytes) {
    if (!a || !bytes) return LTR_EINVAL;
    *bytes = 0;
    if (a->B <= 0 || a->Hq <= 0 || a->Hkv <= 0 || a->Sq <= 0 || a->Hq % a->Hkv || a->n_chunks < 1 || a->n_chunks > LTR_MAX_CHUNKS) return LTR_EINVAL;
    const int D = head_width(a->D, a->flags);
    if (!D) return LTR_EUNSUP;
    if (!fits_i32(a->Sq) || a->q_split < 0 || a->q_split > a->Sq) return LTR_EINVAL;
    if (!fits_i32(a->q_pos0[0] + a->Sq) || !fits_i32(a->q_pos0[1] + a->Sq)) return LTR_EINVAL;
    ChunkDev chunk[LTR_MAX_CHUNKS];
    for (int c = 0; c < a->n_chunks; c++) {
        if (a->chunk[c].sk <= 0 || !fits_i32(a->chunk[c].sk) || !fits_i32(a->chunk[c].pos0 + a->chunk[c].sk)) return LTR_EINVAL;
        chunk[c].sk = (int)a->chunk[c].sk;
        chunk[c].pos0 = (int)a->chunk[c].pos0;
    }
    const int q_pos0[2] = {(int)a->q_pos0[0], (int)a->q_pos0[1]};
    *bytes = plan_bwd(D, a->io_dtype == LTR_F32, D != a->D ? a->flags : a->flags & ~LTR_HEAD_COLS, a->B, a->Hq, a->Hkv, (int)a->Sq, (int)a->q_split, q_pos0, chunk, a->n_chunks, true).part_bytes;
    return LTR_OK;
}

namespace {
// ltr_attn_plan and ltr_attn_plan_ws; ws: the plan of ltr_attn_bwd_ws with a workspace of that many bytes, or nullptr
int describe_plan(const ltr_attn_bwd_args *a, ltr_attn_plan_t *out, int64_t work_bytes, ltr_attn_plan_ws_t *ws) {
    if (a->B <= 0 || a->Hq <= 0 || a->Hkv <= 0 || a->Sq <= 0 || a->Hq % a->Hkv) return LTR_EINVAL;
    if (a->n_chunks < 1 || a->n_chunks > LTR_MAX_CHUNKS) return LTR_EINVAL;
    const int D = head_width(a->D, a->flags);
    const bool pad = D != a->D;
    if (!D) return LTR_EUNSUP;
    if (a->io_dtype != LTR_BF16 && a->io_dtype != LTR_F32) return LTR_EUNSUP;
    if (!fits_i32(a->Sq) || a->q_split < 0 || a->q_split > a->Sq) return LTR_EINVAL;
    if (!fits_i32(a->q_pos0[0] + a->Sq) || !fits_i32(a->q_pos0[1] + a->Sq)) return LTR_EINVAL;
    const unsigned flags = pad ? a->flags : a->flags & ~LTR_HEAD_COLS;
    if ((flags & LTR_DKDV_KEYS_128) && (flags & LTR_DKDV_KEYS_256)) return LTR_EINVAL;
    if ((flags & LTR_DQ_ROWS_256) && (flags & LTR_DQ_ROWS_512)) return LTR_EINVAL;
    if ((flags & LTR_FWD_ROWS_256) && (flags & LTR_FWD_ROWS_512)) return LTR_EINVAL;
    const bool f32 = a->io_dtype == LTR_F32;
    if (pad && f32) return LTR_EUNSUP;
    if ((flags & (LTR_DKDV_KEYS_256 | LTR_DQ_ROWS_512 | LTR_FWD_ROWS_512)) && (a->D != 64 || f32)) return LTR_EUNSUP;
    if ((flags & (LTR_FWD_F32_SCALAR | LTR_BWD_F32_SCALAR)) && !f32) return LTR_EUNSUP;
    ChunkDev chunk[LTR_MAX_CHUNKS];
    for (int c = 0; c < a->n_chunks; c++) {
        const ltr_kv_chunk &ch = a->chunk[c];
        if (ch.sk <= 0 || !fits_i32(ch.sk) || !fits_i32(ch.pos0 + ch.sk)) return LTR_EINVAL;
        chunk[c].k = chunk[c].v = nullptr;
        chunk[c].dk = chunk[c].dv = nullptr;
        chunk[c].sk = (int)ch.sk;
        chunk[c].pos0 = (int)ch.pos0;
    }
    const int q_pos0[2] = {(int)a->q_pos0[0], (int)a->q_pos0[1]};
    const FwdPlan f = plan_fwd(D, f32, flags, a->B, a->Hq, a->Hkv, (int)a->Sq, (int)a->q_split, q_pos0, chunk, a->n_chunks);
    const BwdPlan b = plan_bwd_ws(D, f32, flags, a->B, a->Hq, a->Hkv, (int)a->Sq, (int)a->q_split, q_pos0, chunk, a->n_chunks, work_bytes);
    const bool shared = b.split.n > 1;
    out->compute_units = device_cus();
    out->fwd_rows = f.rows;
    out->fwd_paired = f.n_slots != f.n_qtiles;
    out->fwd_blocks = f.blocks;
    out->dq_rows = b.dq_rows;
    out->dq_paired = b.dq_slots != b.dq_qtiles;
    out->dq_blocks = b.dq_blocks;
    out->dkdv_keys = b.keys_per_block;
    out->dkdv_blocks = shared ? b.split.tiles * a->B * a->Hkv * b.split.n : b.kv_blocks;
    if (f32) {
        if (f.f32_ks) snprintf(out->fwd_kernel, sizeof(out->fwd_kernel), "%s", f32_fwd_kernel(D, f.f32_ks, f.rows).name);
        else snprintf(out->fwd_kernel, sizeof(out->fwd_kernel), "fwd_f32_kernel<%d>", D);
        if (b.f32_ks) {
            snprintf(out->dq_kernel, sizeof(out->dq_kernel), "%s", f32_dq_kernel(D, b.f32_ks, b.dq_rows).name);
            snprintf(out->dkdv_kernel, sizeof(out->dkdv_kernel), "bwd_dkdv_f32_mfma_kernel<%d>", D);
        } else {
            snprintf(out->dq_kernel, sizeof(out->dq_kernel), "bwd_dq_f32_kernel<%d>", D);
            snprintf(out->dkdv_kernel, sizeof(out->dkdv_kernel), "bwd_dkdv_f32_kernel<%d, *>", D);
        }
    } else if (pad) {
        snprintf(out->fwd_kernel, sizeof(out->fwd_kernel), "fwd_bf16_pad_kernel<%d, %d>", D, f.ks);
        snprintf(out->dq_kernel, sizeof(out->dq_kernel), "bwd_dq_pad_kernel<%d, %d>", D, b.dq_ks);
        snprintf(out->dkdv_kernel, sizeof(out->dkdv_kernel), "bwd_dkdv_pad_kernel<%d>", D);
    } else {
        if (f.ks > 1) snprintf(out->fwd_kernel, sizeof(out->fwd_kernel), "fwd_bf16_shares_kernel<%d, %d>", D, f.ks);
        else if (f.four_waves) snprintf(out->fwd_kernel, sizeof(out->fwd_kernel), "fwd_bf16_w4_kernel<%d>", D);
        else snprintf(out->fwd_kernel, sizeof(out->fwd_kernel), "fwd_bf16_kernel<%d, %d>", D, f.wide ? 2 : 1);
        if (b.dq_ks > 1) snprintf(out->dq_kernel, sizeof(out->dq_kernel), "bwd_dq_shares_kernel<%d, %d>", D, b.dq_ks);
        else if (b.dq_four_waves) snprintf(out->dq_kernel, sizeof(out->dq_kernel), "bwd_dq_w4_kernel<%d>", D);
        else snprintf(out->dq_kernel, sizeof(out->dq_kernel), "bwd_dq_kernel<%d, %d>", D, b.wide_q ? 2 : 1);
        if (b.key_waves) snprintf(out->dkdv_kernel, sizeof(out->dkdv_kernel), "bwd_dkdv_keywave_kernel<%d>", D);
        else snprintf(out->dkdv_kernel, sizeof(out->dkdv_kernel), "bwd_dkdv_kernel<%d, %d>", D, b.wide_kv ? 2 : 1);
    }
    if (b.joint) {   // one kernel for both
        const char *name = joint_kernel(D, pad, b.dq_ks, b.own_delta, a->D).name;
        snprintf(out->dq_kernel, sizeof(out->dq_kernel), "%s", name);
        snprintf(out->dkdv_kernel, sizeof(out->dkdv_kernel), "%s", name);
    }
    if (ws) {
        ws->blocks_per_tile = shared ? b.split.n : 1;
        ws->keys_first = b.joint && b.keys_first;
        ws->reduce_blocks = shared ? reduce_blocks(b, D) : 0;
        ws->reduce_kernel[0] = 0;
        if (shared) snprintf(ws->reduce_kernel, sizeof(ws->reduce_kernel), "bwd_dkdv_reduce_kernel<%d, %d>", D, b.wide_kv ? 2 : 1);
    }
    return LTR_OK;
}
}  // namespace

// Host-only: nothing is enqueued, no pointer is read.
extern "C" int ltr_attn_plan(const ltr_attn_bwd_args *a, ltr_attn_plan_t *out) { return a && out ? describe_plan(a, out, 0, nullptr) : LTR_EINVAL; }

extern "C" int ltr_attn_plan_ws(const ltr_attn_bwd_args *a, int64_t workspace_bytes, ltr_attn_plan_ws_t *out) {
    return a && out && workspace_bytes >= 0 ? describe_plan(a, &out->plan, workspace_bytes, out) : LTR_EINVAL;
}

extern "C" int ltr_attn_bwd_noalloc(const ltr_attn_bwd_args *a, void *stream) {
    if (!a) return LTR_EINVAL;
    if (a->io_dtype != LTR_BF16) return LTR_EUNSUP;                 // DELTA comes from the bf16 forward output
    if (a->flags & LTR_NO_DQ) return LTR_EINVAL;                    // the dQ kernel is the one that fills DELTA
    if (a->B <= 0 || a->Hq <= 0 || a->Sq <= 0) return LTR_EINVAL;
    if (a->Sq > LTR_NOALLOC_MAX_ROWS || (long long)a->B * a->Hq > LTR_NOALLOC_MAX_ROWS ||
        (long long)a->B * a->Hq * a->Sq > LTR_NOALLOC_MAX_ROWS)
        return LTR_ETOOBIG;
    return bwd_launch(a, (a->flags | LTR_DELTA_FROM_O) & ~LTR_BWD_JOINT, true, stream);
}

extern "C" int ltr_cast_f32_to_bf16(const float *src, void *dst, int64_t n, void *stream) {
    if (!src || !dst || n < 0) return LTR_EINVAL;
    if (n == 0) return LTR_OK;
    if (!aligned16(src) || ((uintptr_t)dst & 7)) return LTR_EALIGN;
    int rc = check_device();
    if (rc) return rc;
    const long long nblk = (n / 4 + 256) / 256;
    if (nblk > 0x7fffffffLL) return LTR_EINVAL;
    __bf16 *dst16 = (__bf16 *)dst;
    long long n64 = n;
    void *args[] = {(void *)&src, (void *)&dst16, (void *)&n64};
    return hipLaunchKernel((const void *)cast_kernel, dim3((unsigned)nblk), dim3(256), args, 0, (hipStream_t)stream) == hipSuccess
               ? LTR_OK
               : LTR_ELAUNCH;
}
