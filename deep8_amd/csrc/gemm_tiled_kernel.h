// Tiled GEMM for gfx950, fp16 (v_mfma_f32_32x32x16_f16, fp32 accumulation) and fp32
// (v_mfma_f32_32x32x2_f32, true fp32 operands).
//
// A workgroup owns a BM x BN tile of C and walks K in steps of 128 bytes of a row (64 halfs or
// 32 floats).  While step t is multiplied out of one half of a double-buffered LDS area, the A
// and B tiles of step t+1 are written from registers into the other half and the tiles of step
// t+2 are fetched from global memory into those registers with 16-byte buffer loads (uniform
// address part in scalar registers, one offset VGPR per operand).  The loop body is written, and
// pinned with scheduling barriers, in issue order: every MFMA is followed by at most one LDS
// write, one global load and a couple of LDS reads, so the matrix pipe never waits behind a burst
// of memory instructions.  The one workgroup barrier per step sits before the last quarter of the
// step's MFMAs, which then cover the latency of the first operand reads of the next step.
//
// Both tiles keep in LDS the layout they have in memory; the transposed-operand products differ
// only in how the tiles are read back:
//   * an operand contiguous along K is stored [row][k]; one 16-byte LDS read gives a lane the 8
//     halfs (4 floats) of its row that it feeds to the next MFMA(s);
//   * an operand contiguous along M (A of a TN product) or N (B of an NN / TN product) is stored
//     [k][row]; fp16 reads it back with ds_read_b64_tr_b16, the transposing LDS read, which hands
//     each lane four consecutive-k values of its row; fp32 reads one float per k, consecutive
//     lanes reading consecutive addresses.  No transpose is ever materialised.
// Any pairing of k values with lanes works as long as A and B use the same one, because the MFMA
// sums over k; both element types pair lanes 0-31 with the first half of a k group and lanes
// 32-63 with the second half.
//
// Workgroup ids are remapped so that the workgroups one XCD receives (ids congruent mod 8) cover
// a compact block of tiles and share A / B panels in that XCD's L2.  The epilogue turns each
// 32 x 32 accumulator block around through LDS so that C is read and written 16 bytes per lane.
//
// That is Tile: fp32, half products on 256 x 256 tiles and half operands whose rows start anywhere.  Half operands that can be
// moved in 16-byte pieces go straight into LDS (DmaTile, dma_loop); everything around the K loop is shared.
//
// An operand may be a patch matrix that is never written out (GemmArgs::virt): its loader turns
// row / column numbers into image offsets, and an offset outside the image makes the buffer load
// return zeros, which is the padding.  That carries the convolutions: Conv2d forward and its two
// gradients, DeConv2d's gradient of x and of the filter, and -- one residue class of output
// pixels per grid layer (OutClass) -- DeConv2d forward and Conv2d's gradient of x for strides
// above 1, whose rows of C are then pixels of the output image rather than consecutive rows.
//
// The same device covers ragged reductions and skinny matrices: in a last K step that is
// partly past K the pieces beyond K are fetched at an offset outside the buffer (zeros), and a matrix with
// fewer rows or columns than the tile is covered by a tile that starts at 0 and reaches past it -- what
// its loads bring in from there only enters results that are not stored.
#ifndef DEEP8_AMD_GEMM_TILED_KERNEL_H
#define DEEP8_AMD_GEMM_TILED_KERNEL_H

#include <type_traits>

#include "gemm_args.h"

namespace d8 {

typedef __fp16 f16x4v __attribute__((ext_vector_type(4)));
typedef __fp16 f16x8v __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T *)(p))

// instruction classes of __builtin_amdgcn_sched_group_barrier
#define SG_MFMA 0x008
#define SG_VMEM_READ 0x020
#define SG_DS_READ 0x100
#define SG_DS_WRITE 0x200

// What a product's operands look like at their edges (a template argument of the kernels):
//   EDGE_NONE    K is a multiple of the K step
//   EDGE_PIECES  a last, partial K step; a 16-byte piece of an operand lies on one side of K
//   EDGE_ANY     rows that start anywhere: any leading dimension, any K, any element-aligned pointer.  A piece is fetched
//                from a 4-byte aligned address (which is all a buffer load needs), for half from the one at or before it,
//                with one more dword where the row starts in the middle of a dword, and shifted into place on its way to
//                LDS; what a piece of a row stored along K brings in from past K is cut off there as well.  Rows
//                keep their parity from step to step (K steps and passes are even numbers of rows), so shift and extra
//                dword are constants of a thread.  Half 4096 x 1024 by 1024 x 1001, which a kernel that moved single elements
//                served before: product with bias and ReLu 68 -> 24 us, its gradients 50 and 68 -> 21 and 22 us.  Bound by
//                the K loop's latency as the other variants, plus 60 vector instructions a step.
//                A DmaTile cannot shift its pieces: it takes copies of such operands (GemmArgs::packed), and EDGE_ANY there means
//                a partial last step and a C whose rows start anywhere.
enum { EDGE_NONE = 0, EDGE_PIECES = 1, EDGE_ANY = 2 };

// ---- per element type: operand fragments and how to multiply one k group --------------------
template <typename E>
struct Elem;

template <>
struct Elem<f16> {
    typedef f16x8 Frag;                      // 8 k values of one row
    static constexpr int KG = 16;            // k values one fragment pair covers (2 lane halves x 8)
    static constexpr int MFMA_PER_FRAG = 1;  // MFMAs that consume one fragment pair
    static constexpr int TR_READS = 2;       // LDS instructions per fragment in the [k][row] layout
    static constexpr int TR_PAD = 64;        // bytes added to a [k][row] row: its 4 k-rows x 64 B hit different banks
    static constexpr int KC_HALF = 8;        // [row][k] tile: elements between what the two lane halves read
    // ... and inside a [k][row] tile: the lane whose index within its group of 16 is i addresses
    // k-row (i / 4), columns 4 * (i % 4) .. + 3 of its 16-column group, and receives column i
    __device__ static int tr_offset(int lane, int ld, int row0) {
        return ((lane >> 5) * 8 + ((lane & 15) >> 2)) * ld + row0 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    }
    __device__ static Frag read_kc(const f16 *p) { return *(const f16x8 *)p; }
    __device__ static Frag read_tr(const f16 *p, int ld) {
        const f16x4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16(LDS_PTR(f16x4v, p));
        const f16x4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16(LDS_PTR(f16x4v, p + 4 * ld));
        const f16x8v both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(f16x8, both);
    }
    __device__ static f32x16 mfma(const Frag &a, const Frag &b, const f32x16 &c, int) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

template <>
struct Elem<float> {
    typedef f32x4 Frag;  // lanes 0-31: k 0..3 of the group of 8, lanes 32-63: k 4..7
    static constexpr int KG = 8;
    static constexpr int MFMA_PER_FRAG = 4;  // MFMA e pairs k = e with k = 4 + e
    static constexpr int TR_READS = 4;
    static constexpr int TR_PAD = 32;  // k-rows 4 apart (the two lane halves) land in different bank halves
    static constexpr int KC_HALF = 4;
    __device__ static int tr_offset(int lane, int ld, int row0) { return (lane >> 5) * 4 * ld + row0 + (lane & 31); }
    __device__ static Frag read_kc(const float *p) { return *(const f32x4 *)p; }
    __device__ static Frag read_tr(const float *p, int ld) {
        Frag v;
        v[0] = p[0];
        v[1] = p[ld];
        v[2] = p[2 * ld];
        v[3] = p[3 * ld];
        return v;
    }
    __device__ static f32x16 mfma(const Frag &a, const Frag &b, const f32x16 &c, int e) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
    }
};

template <typename E_, int BM_, int BN_, int WGM_, int WGN_, bool A_KC_, bool B_KC_, int VIRT_ = VIRT_NONE>
struct Tile {
    typedef E_ E;
    typedef Elem<E> EL;
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_;
    static constexpr bool A_KC = A_KC_, B_KC = B_KC_;
    static constexpr int VIRT = VIRT_;  // which operand, if any, is a patch matrix read from its image
    static constexpr bool TWO_FIT = false;  // (the compiler is not told to make room for two workgroups per compute unit)
    static constexpr bool DMA = false;  // pieces go through registers (DmaTile: straight into LDS)
    static_assert((VIRT != VIRT_A_ROWS && VIRT != VIRT_A_CLASSES) || A_KC, "patch rows are K-contiguous");
    static_assert(VIRT != VIRT_B_KROWS || !B_KC, "patch k-rows are N-contiguous");
    static constexpr int ES = sizeof(E), EPV = 16 / ES;  // element size, elements per 16-byte piece
    static constexpr int BK = 128 / ES;                  // K step: 128 bytes of a row
    static constexpr int QUARTERS = 4, KQ = BK / QUARTERS;
    static_assert(KQ == EL::KG, "a quarter step is one k group");
    static constexpr int NT = WGM * WGN * 64;
    static constexpr int TM = BM / WGM / 32, TN = BN / WGN / 32;
    static constexpr int MQ = TM * TN * EL::MFMA_PER_FRAG;  // MFMAs per quarter step
    // A [row][k] tile keeps its rows (128 bytes each) in order with 16 bytes of padding after every
    // second row: the 16 rows that one cycle of a 16-byte LDS read touches then start in 16 different
    // groups of four banks, and two workgroup tiles of the 64-wide shapes stay under a third of the
    // CU's LDS.  A [k][row] tile has a leading dimension (A_LD / B_LD) with TR_PAD bytes of padding.
    __device__ __host__ static constexpr int kc_row(int r) { return r * BK + (r >> 1) * EPV; }
    static constexpr int KC_BLK = kc_row(32);  // elements between rows 32 apart (from an even row)
    static constexpr int A_LD = BM + EL::TR_PAD / ES, B_LD = BN + EL::TR_PAD / ES;
    static constexpr int A_TILE = A_KC ? kc_row(BM) : BK * A_LD, PATCHES = NT / 128 * 32 * 36 * 4 / ES;  // (patches: the epilogue's, see below)
    static constexpr int A_SZ = A_TILE > PATCHES ? A_TILE : PATCHES;
    static constexpr int B_SZ = B_KC ? kc_row(BN) : BK * B_LD;
    // 16-byte pieces each thread moves per K step, and the rows one pass of all threads covers
    static constexpr int A_IT = BM * 8 / NT, B_IT = BN * 8 / NT, NP = A_IT + B_IT;
    static constexpr int A_ROWS = A_KC ? NT / 8 : NT / (BM / EPV);
    // Patch k-rows as B, fp32: the threads' passes walk the tile's columns instead of its rows -- a pass is all BK k-rows
    // x 32 columns, so a thread keeps ONE patch row per K step, decoded once, and its pieces differ by tap and channel
    // (an add and a bounds check each).  Decoding a row per piece cost Conv2d C4's filter gradient 11 of its 74 us.
    static constexpr bool B_COLS = VIRT == VIRT_B_KROWS && ES == 4 && NT / 8 == BK;
    static constexpr int B_ROWS = B_COLS ? BK : B_KC ? NT / 8 : NT / (BN / EPV);
    static_assert(A_ROWS % 2 == 0 && B_ROWS % 2 == 0, "a pass of all threads starts on an even row");
    // elements between the pieces two consecutive passes write, and between a wave's 32-row blocks
    static constexpr int A_PASS = A_KC ? kc_row(A_ROWS) : A_ROWS * A_LD, B_PASS = B_COLS ? 8 * EPV : B_KC ? kc_row(B_ROWS) : B_ROWS * B_LD;
    static constexpr int A_BLK = A_KC ? KC_BLK : 32, B_BLK = B_KC ? KC_BLK : 32;
    static constexpr int A_RD = A_KC ? 1 : EL::TR_READS, B_RD = B_KC ? 1 : EL::TR_READS;
    // the epilogue's transposing patches reuse the two halves of the larger operand area: the first
    // half of the waves turn their blocks around in one, the rest in the other
    static constexpr bool PATCH_IN_A = A_SZ >= B_SZ;
    static constexpr int PATCH_SZ = PATCH_IN_A ? A_SZ : B_SZ;
};

// fp16 tile whose operand pieces go from global memory straight into LDS (buffer_load_dwordx4 ... lds), STAGES K steps ahead: no
// registers between the two, no LDS writes, and operands that have to come from memory are asked for early enough.  Against
// tiles that pass through registers, one step ahead: 1024^3 8.4 -> 7.4 us and, with operands that no cache holds, 12.6 -> 8.2;
// 6272 x 256 x 2304 19.8 -> 16.0, cold 32.3 -> 24.  (A product by itself.  Of a layer with its gate and gradients, whose operands the
// call before has left in a cache or not, less is left: 1024^3 with new inputs each time 4.5 %, the same ones 18 %.)
//
// A lane's 16 bytes land at a wave-uniform base + 16 x lane, so rows cannot be padded; bank conflicts are avoided by choosing
// WHICH 16 bytes a lane fetches.  The LDS reads serve 256 bytes (64 banks) at a time:
//   * [row][64 k], 128 bytes a row: chunk c of row r lies at position c ^ (r >> 1 & 7), so that the 16 rows of a 16-byte read
//     cover all banks;
//   * [k][row], 2 * BM (2 * BN) bytes a k-row: 32 lanes of a transposing read touch 64 bytes of each of 4 k-rows.  Rows of 256
//     bytes keep their 64-byte groups at g ^ (k & 3), rows of 128 bytes at g ^ (k >> 1 & 1).
template <int BM_, int BN_, int WGM_, int WGN_, int STAGES_, bool A_KC_, bool B_KC_, int VIRT_ = VIRT_NONE>
struct DmaTile {
    typedef f16 E;
    typedef Elem<f16> EL;
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, STAGES = STAGES_;
    static constexpr bool A_KC = A_KC_, B_KC = B_KC_;
    static constexpr int VIRT = VIRT_;
    static constexpr bool DMA = true, B_COLS = false;
    static constexpr int ES = 2, EPV = 8, BK = 64, QUARTERS = 4, KQ = 16;
    static constexpr int NT = WGM * WGN * 64;
    static constexpr int TM = BM / WGM / 32, TN = BN / WGN / 32;
    static constexpr int A_IT = BM * 8 / NT, B_IT = BN * 8 / NT, NP = A_IT + B_IT;
    static_assert(A_IT * NT == BM * 8 && B_IT * NT == BN * 8, "every thread moves whole pieces of either operand");
    static constexpr int A_ROWS = A_KC ? NT / 8 : NT / (BM / EPV), B_ROWS = B_KC ? NT / 8 : NT / (BN / EPV);
    static_assert(A_ROWS % 16 == 0 && B_ROWS % 16 == 0, "a thread's swizzle is the same in every pass");
    __device__ __host__ static constexpr int kc_row(int r) { return r * BK; }
    static constexpr int A_LD = BM, B_LD = BN;
    static constexpr int A_BYTES = BM * 128, STAGE_BYTES = (BM + BN) * 128, LDS_BYTES = STAGES * STAGE_BYTES;
    static constexpr int HALF_PATCHES = NT / 128 * 32 * 36;  // floats: the epilogue's patches, in the stages
    static constexpr int PATCH_SZ = HALF_PATCHES * 4 / ES;
    static constexpr bool TWO_FIT = LDS_BYTES <= 80 * 1024;  // two workgroups per compute unit
    static_assert(LDS_BYTES >= 2 * HALF_PATCHES * 4, "the patches fit the stages");
    static constexpr bool PATCH_IN_A = true;
    // position of a thread's piece in its row -> which piece of the row it fetches
    template <bool KC, int SIDE>
    __device__ __forceinline__ static int chunk_of(int row, int pos) {
        if (KC) return pos ^ ((row >> 1) & 7);
        return SIDE == 128 ? pos ^ ((row & 3) << 2) : pos ^ (((row >> 1) & 1) << 2);
    }
    // byte offset in an operand area of what this lane reads of 32-row block `blk` at k group 0
    template <bool KC, int SIDE>
    __device__ __forceinline__ static int frag_of(int lane, int blk) {
        if (KC) return (blk * 32 + (lane & 31)) * 128 + (((lane >> 5) ^ ((lane >> 1) & 7)) << 4);
        const int k = (lane >> 5) * 8 + ((lane & 15) >> 2), s = SIDE == 128 ? k & 3 : (k >> 1) & 1;
        return k * SIDE * 2 + ((blk ^ s) << 6) + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
    }
    template <bool KC, int SIDE>
    __device__ __forceinline__ static f16x8 read(const char *area, int frag, int kg) {
        if (KC) return *(const f16x8 *)(area + (frag ^ (kg << 5)));
        const char *p = area + frag + kg * 16 * SIDE * 2;
        const f16x4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16(LDS_PTR(f16x4v, p));
        const f16x4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16(LDS_PTR(f16x4v, p + 4 * SIDE * 2));
        const f16x8v both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(f16x8, both);
    }
};

// One 16-byte piece per lane from global memory into LDS: lane i's lands at `target` + 16 * i (target, soffset and the descriptor
// are uniform).  Written as asm so that the compiler does not hold every later LDS read until the load has landed; the waits and
// the barrier of each K step order the two.  (m0 is written a wait state before the load that uses it.)
__device__ __forceinline__ void dma_piece(unsigned target, const u32x4 &desc, unsigned voffset, unsigned soffset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 : : "s"(target), "v"(voffset), "s"(desc), "s"(soffset) : "memory");
}
// s_waitcnt vmcnt(n) lgkmcnt(0): the builtin, so that the compiler knows that its own LDS reads have arrived
template <int N>
__device__ __forceinline__ void wait_loads_and_lds() {
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | 0x70 | ((N >> 4) << 14));
}

// Pieces [lo(q), lo(q+1)) are written to LDS during quarter q = 0, 1, 2 of a step and re-fetched
// from global memory during quarter q + 1.
template <int NP>
__device__ __host__ constexpr int piece_lo(int q) { return q * NP / 3; }
// The t-th of n events of a quarter goes right after MFMA number (t * MQ) / n.
__device__ __host__ constexpr int slot_of(int t, int n, int MQ) { return t * MQ / n; }

// EDGE_ANY: what a thread needs to put its pieces into place
template <typename T, int EDGE>
struct Loose {
    static constexpr bool ANY = EDGE == EDGE_ANY && !T::DMA, ODD = ANY && T::ES == 2;
    unsigned X[ODD ? T::NP : 1];  // the dword after each piece
    unsigned shift[2], next[2];   // per operand: bits to shift by, byte offset of that dword (outside the buffer where it is not needed)
    u32x4 keep[2];                // ... and which bits of a piece are within K (operands stored along K)
    __device__ __forceinline__ u32x4 place(int p, u32x4 v) const {
        if constexpr (ANY) {
            const int o = p < T::A_IT ? 0 : 1;
            if constexpr (ODD) {
                u32x4 w;
#pragma unroll
                for (int d = 0; d < 4; ++d) w[d] = __builtin_amdgcn_alignbit(d < 3 ? v[d < 3 ? d + 1 : 3] : X[p], v[d], shift[o]);
                v = w;
            }
            if (o == 0 ? T::A_KC : T::B_KC) v &= keep[o];
        }
        return v;
    }
    __device__ __forceinline__ void fetch(int p, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
        if constexpr (ODD) X[p] = __builtin_amdgcn_raw_buffer_load_b32(r, v + next[p < T::A_IT ? 0 : 1], s, 0);
    }
    // the pieces of operand o written next have `left` elements of K from this thread's first on
    __device__ __forceinline__ void keep_first(int o, int left) {
        if constexpr (ANY) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                if constexpr (T::ES == 2) keep[o][d] = left > 2 * d + 1 ? 0xffffffffu : left > 2 * d ? 0xffffu : 0u;
                else keep[o][d] = left > d ? 0xffffffffu : 0u;
            }
        }
    }
};

// One K step.  Ar/Br: this lane's operand addresses in the LDS half being multiplied; An/Bn: the
// same in the other half (next step); Aw/Bw: where this thread's pieces of the next step go;
// ra/rb: buffer descriptors of the A and B matrices; ga/gb: wave-uniform byte offset (tile origin +
// K step) of the pieces of the step after that, av/bv: this thread's byte offset for each piece.
template <typename T, int EDGE>
__device__ __forceinline__ void k_step(const typename T::E *Ar, const typename T::E *Br, const typename T::E *An,
                                       const typename T::E *Bn, typename T::E *Aw, typename T::E *Bw,
                                       __amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rb, unsigned ga, unsigned gb,
                                       unsigned a_pass, unsigned b_pass, const unsigned (&av)[T::A_IT],
                                       const unsigned (&bv)[T::B_IT], u32x4 (&R)[T::NP], Loose<T, EDGE> &L, typename T::EL::Frag (&fa)[2][T::TM],
                                       typename T::EL::Frag (&fb)[2][T::TN], f32x16 (&acc)[T::TM][T::TN]) {
    typedef typename T::E E;
    typedef typename T::EL EL;
    constexpr int TM = T::TM, TN = T::TN, MQ = T::MQ, NP = T::NP, A_IT = T::A_IT, NF = TM + TN;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (q == 3) __syncthreads();  // every wave has written its pieces and finished reading this half
        const int w_lo = q < 3 ? piece_lo<NP>(q) : 0, w_n = q < 3 ? piece_lo<NP>(q + 1) - w_lo : 0;
        const int g_lo = q > 0 ? piece_lo<NP>(q - 1) : 0, g_n = q > 0 ? piece_lo<NP>(q) - g_lo : 0;
#pragma unroll
        for (int m = 0; m < MQ; ++m) {
            {
                const int e = m / (TM * TN), ij = m % (TM * TN), i = ij / TN, j = ij % TN;
                acc[i][j] = EL::mfma(fa[q & 1][i], fb[q & 1][j], acc[i][j], e);
            }
#pragma unroll
            for (int t = 0; t < w_n; ++t)
                if (slot_of(t, w_n, MQ) == m) {
                    const int p = w_lo + t;
                    E *dst = p < A_IT ? Aw + p * T::A_PASS : Bw + (p - A_IT) * T::B_PASS;
                    *(u32x4 *)dst = L.place(p, R[p]);
                }
#pragma unroll
            for (int t = 0; t < g_n; ++t)
                if (slot_of(t, g_n, MQ) == m) {
                    const int p = g_lo + t;
                    R[p] = p < A_IT ? __builtin_amdgcn_raw_buffer_load_b128(ra, av[p < A_IT ? p : 0], ga + p * a_pass, 0)
                                    : __builtin_amdgcn_raw_buffer_load_b128(rb, bv[p < A_IT ? 0 : p - A_IT], gb + (p - A_IT) * b_pass, 0);
                    L.fetch(p, p < A_IT ? ra : rb, p < A_IT ? av[p < A_IT ? p : 0] : bv[p < A_IT ? 0 : p - A_IT], p < A_IT ? ga + p * a_pass : gb + (p - A_IT) * b_pass);
                }
            // operands of the next quarter (of the next step's first quarter when q == 3)
#pragma unroll
            for (int f = 0; f < NF; ++f)
                if (slot_of(f, NF, MQ) == m) {
                    const int kk = q < 3 ? (q + 1) * T::KQ : 0;
                    const E *a_base = q < 3 ? Ar : An, *b_base = q < 3 ? Br : Bn;
                    if (f < TM)
                        fa[(q + 1) & 1][f] = T::A_KC ? EL::read_kc(a_base + f * T::A_BLK + kk)
                                                     : EL::read_tr(a_base + kk * T::A_LD + f * 32, T::A_LD);
                    else
                        fb[(q + 1) & 1][f - TM] = T::B_KC ? EL::read_kc(b_base + (f - TM) * T::B_BLK + kk)
                                                          : EL::read_tr(b_base + kk * T::B_LD + (f - TM) * 32, T::B_LD);
                }
        }
        // pin the issue order to the program order above
#pragma unroll
        for (int m = 0; m < MQ; ++m) {
            __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
#pragma unroll
            for (int t = 0; t < w_n; ++t)
                if (slot_of(t, w_n, MQ) == m) __builtin_amdgcn_sched_group_barrier(SG_DS_WRITE, 1, 0);
#pragma unroll
            for (int t = 0; t < g_n; ++t)
                if (slot_of(t, g_n, MQ) == m) __builtin_amdgcn_sched_group_barrier(SG_VMEM_READ, Loose<T, EDGE>::ODD ? 2 : 1, 0);
#pragma unroll
            for (int f = 0; f < NF; ++f)
                if (slot_of(f, NF, MQ) == m) {
                    if (f < TM) __builtin_amdgcn_sched_group_barrier(SG_DS_READ, T::A_RD, 0);
                    else __builtin_amdgcn_sched_group_barrier(SG_DS_READ, T::B_RD, 0);
                }
        }
    }
}

__device__ inline float as_f32(float v) { return v; }
__device__ inline float as_f32(f16 v) { return (float)v; }

struct Origin {
    int m0, n0;        // where the computed tile starts (moved inside the matrix)
    int m_own, n_own;  // rows / columns from here on are this workgroup's to store
    int m_end, n_end;  // ... up to the matrix's own (a tile may be larger than a matrix with fewer than BM rows or BN columns)
    int wm0, wn0;      // this wave's offset inside the tile
};

// Store a wave's accumulators.  Lane holds column lane%32 of rows 8*(r/4) + 4*(lane/32) + r%4 of
// each 32x32 block.  Where rows of C can be moved 16 bytes at a time, each block is turned around
// through the wave's own 32 x 36 float patch of LDS, so that a lane ends up with 8 consecutive
// columns of one row: 16-byte loads of the old C and 16-byte stores.
// C row of tile row m: m itself, or the output pixel of row (b, y', x') of a class of a transposed convolution
struct RowMap {
    int plane, OW;                           // 0: identity
    int out_H, out_W, out_sy, out_sx, py, px;
    int perm_T, perm_OC;                     // perm_OC > 0: stored transposed per tap (GemmArgs::perm_OC)
    unsigned by_plane, by_ow, by_perm;       // reciprocals of plane, OW, perm_OC
    __device__ long operator()(int m) const {
        if (!plane) return m;
        int rem, x;
        const int img = Divisor(plane, by_plane).div(m, rem), y = Divisor(OW, by_ow).div(rem, x);
        return ((long)img * out_H + out_sy * y + py) * out_W + out_sx * x + px;
    }
    __device__ long at(int m, int n, int ldc) const {
        if (perm_OC) {
            int oc;
            const int t = Divisor(perm_OC, by_perm).div(n, oc);
            return ((long)oc * perm_T + t) * ldc + m;
        }
        return (*this)(m) * ldc + n;
    }
};

// LOOSE (the kernels for rows that start anywhere): the same with 16-byte accesses at the alignment of an element, and
// element by element only where the eight columns of a lane cross the edge of what is this workgroup's.  Half 4096 x 1024 by
// 1024 x 1001 with bias and ReLu: 28.2 -> 23.8 us; the element-wise store below asks for beta, bias and ReLu at
// every one of its 64 elements a thread.
template <typename T, typename O, bool LOOSE = false>
__device__ __forceinline__ void store_tile(f32x16 (&acc)[T::TM][T::TN], float *lds0, float *lds1, O *C, int ldc, float beta,
                                           bool aligned, int N, const Origin &o, const RowMap &crow,
                                           const O *bias = nullptr, bool relu = false, bool round_first = false) {
    constexpr int TM = T::TM, TN = T::TN, OPV = 16 / sizeof(O);
    typedef O OV __attribute__((ext_vector_type(OPV)));
    typedef OV MV __attribute__((aligned(LOOSE ? sizeof(O) : sizeof(OV))));  // as it lies in memory
    constexpr int HALF_WAVES = T::NT / 128;
    static_assert((size_t)T::PATCH_SZ * T::ES >= (size_t)HALF_WAVES * 32 * 36 * sizeof(float), "patch space");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, lhi = lane >> 5;
    if (!crow.perm_OC && (LOOSE || (aligned && N % 8 == 0 && ((size_t)bias & 15) == 0))) {
        float *patch = (wave < HALF_WAVES ? lds0 + wave * (32 * 36) : lds1 + (wave - HALF_WAVES) * (32 * 36));
        // fp32: the bias of a lane's columns before the first store, because a load that is waited for behind a store waits for
        // the store's acknowledgement too (51 drawn layers with bias and ReLu 1.7 % faster at the mean, Conv2d 13 x 10x9x64 -> 128
        // 1x1 stride 2 11.4 -> 9.7 us; half, with half as many stores, 0.4 % slower)
        constexpr bool BIAS_FIRST = sizeof(O) == 4;
        OV bias_v[BIAS_FIRST ? TN : 1][8 / OPV];
        if constexpr (BIAS_FIRST)
            if (bias)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int n = o.n0 + o.wn0 + j * 32 + (lane & 3) * 8;
                    if (n + 8 <= N)
#pragma unroll
                        for (int h = 0; h < 8 / OPV; ++h) bias_v[j][h] = *(const MV *)(bias + n + h * OPV);
                }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
#pragma unroll
                for (int r = 0; r < 16; ++r) patch[((r >> 2) * 8 + lhi * 4 + (r & 3)) * 36 + l32] = acc[i][j][r];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int q = lane + 64 * t, row = q >> 2, cc = (q & 3) * 8;
                    const int m = o.m0 + o.wm0 + i * 32 + row, n = o.n0 + o.wn0 + j * 32 + cc;
                    float v[8];
                    *(f32x4 *)&v[0] = *(const f32x4 *)(patch + row * 36 + cc);
                    *(f32x4 *)&v[4] = *(const f32x4 *)(patch + row * 36 + cc + 4);
                    const bool in_m = m >= o.m_own && m < o.m_end, whole = !LOOSE || n + 8 <= o.n_end;
                    if (in_m && n >= o.n_own && n < o.n_end && whole) {
                        O *c = C + crow(m) * ldc + n;
#pragma unroll
                        for (int h = 0; h < 8 / OPV; ++h) {
                            OV out;
                            if (beta != 0.f) {
                                const OV old = *(const MV *)(c + h * OPV);
#pragma unroll
                                for (int e = 0; e < OPV; ++e) v[h * OPV + e] += as_f32(old[e]);
                            }
                            if (bias) {
                                OV bv;
                                if constexpr (BIAS_FIRST) bv = bias_v[j][h];
                                else bv = *(const MV *)(bias + n + h * OPV);
#pragma unroll
                                for (int e = 0; e < OPV; ++e) v[h * OPV + e] = (round_first ? as_f32((O)v[h * OPV + e]) : v[h * OPV + e]) + as_f32(bv[e]);
                            }
#pragma unroll
                            for (int e = 0; e < OPV; ++e) out[e] = (O)(relu && !(v[h * OPV + e] > 0.f) ? 0.f : v[h * OPV + e]);
                            *(MV *)(c + h * OPV) = out;
                        }
                    } else if (LOOSE && in_m) {
                        O *c = C + crow(m) * ldc + n;
                        for (int e = 0; e < 8; ++e)
                            if (n + e >= o.n_own && n + e < o.n_end) {
                                float w = patch[row * 36 + cc + e];
                                if (beta != 0.f) w += as_f32(c[e]);
                                if (bias) w = (round_first ? as_f32((O)w) : w) + as_f32(bias[n + e]);
                                c[e] = (O)(relu && !(w > 0.f) ? 0.f : w);
                            }
                    }
                }
            }
        return;
    }
    // element by element: 32 lanes store 32 consecutive columns of a row.  The outer loop runs over a thread's columns, the
    // bias of a column being read once; an element of it lies at a start of the column plus a step per row of the tile, but
    // for the pixels of a class, whose rows are looked up one by one.  (Divided out at every element, a filter gradient
    // stored transposed per tap lost some 5 us to divisions: half DeConv2d 33 x 4x4x320 -> 64, 3x3 stride 2, forward and
    // both gradients 41.5 -> 37.1 us.)
    const bool lines = !crow.plane || crow.perm_OC;
    const long step = crow.perm_OC ? 1 : ldc;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = o.n0 + o.wn0 + j * 32 + l32;
        const bool in_n = n >= o.n_own && n < o.n_end;
        const float bias_n = bias && in_n ? as_f32(bias[n]) : 0.f;
        O *const start = C + (crow.perm_OC ? crow.at(0, n, ldc) : n);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = o.m0 + o.wm0 + i * 32 + (r >> 2) * 8 + lhi * 4 + (r & 3);
                if (in_n && m >= o.m_own && m < o.m_end) {
                    O *c = lines ? start + m * step : C + crow.at(m, n, ldc);
                    float v = acc[i][j][r];
                    if (beta != 0.f) v += as_f32(*c);
                    if (bias) v = (round_first ? as_f32((O)v) : v) + bias_n;
                    *c = (O)(relu && !(v > 0.f) ? 0.f : v);
                }
            }
    }
}

// body(std::integral_constant<int, 0>) ... body(std::integral_constant<int, N - 1>), in order
template <int N, int I = 0, class F>
__device__ __forceinline__ void each(F &&body) {
    if constexpr (I < N) {
        body(std::integral_constant<int, I>());
        each<N, I + 1>(body);
    }
}

// The K loop of a DmaTile.  In step t a wave's fragments of the whole step are in registers: the stage they came from is free,
// and the fragments of step t + 1 are read while step t is multiplied, so neither the way from memory (STAGES - 1 steps) nor
// that from LDS (one step) is waited for, and a step needs one barrier.
// A load into LDS holds its wave until the address path (16 cycles a load, one path a compute unit) has taken it: issued in one
// go behind the barrier the loads of all waves keep every matrix instruction waiting for 256 to 512 cycles (a 64 x 128 step
// then takes 836 cycles instead of 620).  They are issued one at a time between the matrix instructions.
// Bound by the loads: without them a 64 x 64 / 64 x 128 step takes 245 / 369 cycles, the loads alone 326 / 606, both 454 / 620 (about
// 40 bytes a cycle and compute unit; free-running waves reach 64, waves that meet at a barrier do not, whatever the number of
// stages, the pitch of the rows or the order of the steps).
// Nothing is fetched past the last step: such loads bring zeros, but take the address path as long as others, a stage's worth each
// for S steps of every tile.  With few steps a tile that was most of them.  100 drawn half Conv2d of 8 to 100 channels,
// forward: 1363 us with them, 1286 without (1357 on tiles that pass through registers); 14 x 75x75x8 -> 89 1x1 22.9 -> 20.6.
//   aim()                   turns to the next step; fetch(piece, target) puts a piece of it on its way
//   started()               is called when the first operands have arrived
template <typename T, class Aim, class Fetch, class Started>
__device__ __forceinline__ void dma_loop(f16 *lds, int wave, int lane, int wm, int wn, int nsteps, f32x16 (&acc)[T::TM][T::TN],
                                         Aim &&aim, Fetch &&fetch, Started &&started) {
    constexpr int TM = T::TM, TN = T::TN, KG = T::QUARTERS, S = T::STAGES, NP = T::NP, NF = KG * (TM + TN), NM = KG * TM * TN;
    const char *const base = (const char *)lds;
    const unsigned wave_base = (unsigned)(unsigned long)LDS_PTR(char, lds) + (unsigned)wave * 1024u;
    f16x8 fa[2][KG][TM], fb[2][KG][TN];
    int a_at[TM], b_at[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_at[i] = T::template frag_of<T::A_KC, T::BM>(lane, wm * TM + i);
#pragma unroll
    for (int j = 0; j < TN; ++j) b_at[j] = T::template frag_of<T::B_KC, T::BN>(lane, wn * TN + j);
    // fragment f of a step: k group by k group, in the order of their first use
    auto read = [&](auto f, int set, int stage) {
        constexpr int q = decltype(f)::value / (TM + TN), e = decltype(f)::value % (TM + TN);
        const char *const as = base + stage * T::STAGE_BYTES, *const bs = as + T::A_BYTES;
        if constexpr (e < TN) fb[set][q][e] = T::template read<T::B_KC, T::BN>(bs, b_at[e], q);
        else fa[set][q][e - TN] = T::template read<T::A_KC, T::BM>(as, a_at[e - TN], q);
    };
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (s > 0 && s >= nsteps) break;
        aim();
        each<NP>([&](auto p) { fetch(p, wave_base + s * T::STAGE_BYTES); });
    }
    if (nsteps < S) wait_loads_and_lds<0>();
    else wait_loads_and_lds<(S - 1) * NP>();
    __syncthreads();
    each<NF>([&](auto f) { read(f, 0, 0); });
    started();
    int stage = 0;  // of step t
    auto step = [&](auto set_tag, auto fetches) {
        constexpr int set = decltype(set_tag)::value;
        constexpr bool FETCH = decltype(fetches)::value;
        const int next = stage + 1 == S ? 0 : stage + 1;
        const unsigned target = wave_base + stage * T::STAGE_BYTES;
        if constexpr (FETCH) aim();
        // this wave's fragments of step t have been read and its pieces of step t + 1 have landed (with nothing to follow: all
        // of them); behind the barrier that holds for all waves
        wait_loads_and_lds<FETCH ? (S - 2) * NP : 0>();
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        each<NM>([&](auto m_tag) {
            constexpr int m = decltype(m_tag)::value, q = m / (TM * TN), i = m % (TM * TN) / TN, j = m % TN;
            each<NF>([&](auto f) { if constexpr (slot_of(decltype(f)::value, NF, NM) == m) read(f, set ^ 1, next); });
            acc[i][j] = Elem<f16>::mfma(fa[set][q][i], fb[set][q][j], acc[i][j], 0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (FETCH) each<NP>([&](auto p) { if constexpr (slot_of(decltype(p)::value, NP, NM) == m) fetch(p, target); });
            __builtin_amdgcn_sched_barrier(0);
        });
        stage = next;
    };
    // steps that fetch one further on, an even number of them (one of the loads may lie past the last step), then the rest
    const int fetching = nsteps > S ? (nsteps - S + 1) & ~1 : 0;
    int t = 0;
    for (; t < fetching; t += 2) {
        step(std::integral_constant<int, 0>(), std::true_type());
        step(std::integral_constant<int, 1>(), std::true_type());
    }
    for (; t < nsteps; t += 2) {
        step(std::integral_constant<int, 0>(), std::false_type());
        if (t + 1 < nsteps) step(std::integral_constant<int, 1>(), std::false_type());
    }
    wait_loads_and_lds<0>();  // (nothing lands in LDS any more: the epilogue uses it)
}

// A value that is the same for all lanes, in a scalar register (DmaTile).  The compiler keeps the quotients of integer divisions
// and what it computes from them in vector registers, and would read a load's offset from there right before dma_piece: a load wants
// five wait states behind a vector instruction that writes a scalar it takes, which the compiler keeps before loads of its own
// only.  Whatever an offset is made of is therefore made scalar well before the loads (tests/test_kernel_wait_states.py looks
// for any that is not).  Five wait states before every step's loads instead: a dense layer of 4096 x 1024 x 1024 with its gradients
// 23.0 -> 23.8 us; so, 23.2, and Conv2d 32 x 14x14x256 3x3 with its 56.5 -> 56.9.
template <typename T>
__device__ __forceinline__ int uniform(int v) {
    if constexpr (T::DMA) return __builtin_amdgcn_readfirstlane(v);
    else return v;
}

// The work of one workgroup: workgroup (bx, bz) of a grid of nbx x layers (the launch's own blockIdx / gridDim, or what a
// launch of two products makes of them).  As0 .. Bs1: the two halves of both operand areas in LDS.
template <typename T, int EDGE>
__device__ __forceinline__ void gemm_tiled_body(const GemmArgs &g, int tilesM, const int tilesN, const int bx, const int bz, const int nbx,
                                                typename T::E *As0, typename T::E *As1, typename T::E *Bs0, typename T::E *Bs1) {
    typedef typename T::E E;
    typedef typename T::EL EL;
    typedef E EV __attribute__((ext_vector_type(T::EPV)));
    constexpr int BM = T::BM, BN = T::BN, BK = T::BK, TM = T::TM, TN = T::TN, A_LD = T::A_LD, B_LD = T::B_LD;
    constexpr int A_IT = T::A_IT, NP = T::NP, ES = T::ES, EPV = T::EPV;
    constexpr bool A_KC = T::A_KC, B_KC = T::B_KC;

    const int tid = threadIdx.x, lane = tid & 63, wave = T::DMA ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6;
    const int wm = wave / T::WGN, wn = wave % T::WGN;
    unsigned long long st_w[4] = {0, 0, 0, 0}, st_c[2] = {0, 0};  // phase record (GemmArgs::phase_rec), a measurement aid
    if (g.phase_rec) st_w[0] = wall_clock64();

    // ---- which tile: ids of one XCD (same id mod 8) form a contiguous run, runs are laid out in
    // bands of GM tile rows walked column by column
    // blockIdx.z = output batch index * splits + piece of the reduction.  The reduction runs over
    // `red` products (1 unless the whole batch is summed into one C) times K, cut into `splits`.
    // The tiles of one piece read the same rows of A and B, so they should meet in one L2: the
    // launch's workgroups (x fastest, then z) go to the XCDs in turn, and the ids one XCD receives
    // are therefore dealt out piece by piece, all tiles of a piece before the next.
    constexpr int VIRT = T::VIRT, B_IT = T::B_IT;
    constexpr bool VA = VIRT == VIRT_A_ROWS || VIRT == VIRT_A_CLASSES;  // A's rows are patch rows
    PatchGeom pg = g.pg;
    int M = g.M, red = g.red;
    unsigned b_cls = 0;
    RowMap crow = {0, 0, 0, 0, 0, 0, 0, 0, g.perm_T, g.perm_OC, 0, 0, g.by.perm_OC};
    const RowMap plain = {};
    unsigned by_plane = g.by.plane, by_ow = g.by.ow;
    if constexpr (VIRT == VIRT_A_CLASSES) {
        const OutClass &c = g.cls[bz];
        M = c.M, red = c.red, b_cls = c.b_off;
        pg.OH = c.OH, pg.OW = c.OW, pg.FW = c.taps_w, pg.pt = c.pt, pg.pl = c.pl;
        by_plane = c.by_plane, by_ow = c.by_ow;
        crow = {c.OH * c.OW, c.OW, g.out_H, g.out_W, g.out_sy, g.out_sx, c.py, c.px, 0, 0, by_plane, by_ow, 0};
        tilesM = (M + BM - 1) / BM;
        if (bx >= tilesM * tilesN) return;  // the grid is sized for the largest class
    }
    int id = bx;
    const int total = tilesM * tilesN;
    int b = 0, split = 0;
    if constexpr (VIRT != VIRT_A_CLASSES) b = Divisor(g.splits, g.by.layers).div(bz, split);
    // a workgroup past the product's own tiles works on the remainder band (GemmArgs::tail_m0)
    const bool in_tail = VIRT != VIRT_A_CLASSES && g.tail_splits > 0 && id >= total;
    int tps = g.tiles_per_split;
    if (in_tail) {
        id = Divisor(g.tail_splits, g.by.tail_splits).div(id - total, split);  // tile of the band, column by column
        tps = g.tail_tps;
    } else if constexpr (VIRT == VIRT_A_CLASSES) {
        if (T::DMA || (total & 7) == 0) id = (id & 7) * (total >> 3) + min(id & 7, total & 7) + (id >> 3);
    } else {
        // an unsplit batched product is dealt out the same way over its batch index: one XCD takes all
        // tiles of a batch element, whose A and B it then reads once
        const bool by_batch = g.splits == 1;
        int layer = by_batch ? b : split;
        const int layers = by_batch ? g.batch : g.splits;
        const int linear = id + total * layer, whole = total * (layers & ~7);
        if (linear < whole) {
            const int piece = Divisor(total, g.by.tiles).div(linear >> 3, id);
            layer = (piece << 3) + (linear & 7);
        } else if (T::DMA || (total & 7) == 0) {  // (the first total % 8 runs are one tile longer)
            id = (id & 7) * (total >> 3) + min(id & 7, total & 7) + (id >> 3);
        }
        if (by_batch) b = layer;
        else split = layer;
    }
    constexpr int GM = 4;
    int tm, tn;
    if (in_tail) {
        tn = Divisor((M - g.tail_m0 + BM - 1) / BM, g.by.tail_tilesM).div(id, tm);
    } else {
        int in_band;
        const int first = Divisor(GM * tilesN, g.by.band).div(id, in_band) * GM, rows_in_band = max(1, min(GM, tilesM - first));
        tn = rows_in_band == 3 ? (int)__umulhi((unsigned)in_band, 0x55555556u) : in_band >> (rows_in_band >> 1);  // (four, two or one: a shift)
        tm = first + in_band - tn * rows_in_band;
    }
    // A tile that would stick out of the matrix is moved back inside; the rows / columns it then
    // shares with its neighbour are computed twice but stored only by the neighbour.
    const int m_own = uniform<T>((in_tail ? g.tail_m0 : 0) + tm * BM), n_own = uniform<T>(tn * BN);
    // (a matrix with fewer rows or columns than the tile: the tile starts at 0 and reaches past it; what the loads
    // bring in from there -- zeros past the end of the buffer, otherwise whatever follows -- only ever enters
    // results of rows / columns past the matrix, which are not stored)
    // (copies in whole pieces, GemmArgs::packed: the tile is moved back by whole pieces)
    const int M_in = T::DMA && EDGE == EDGE_ANY && !A_KC ? g.padM : M, N_in = T::DMA && EDGE == EDGE_ANY && !B_KC ? g.padN : g.N;
    const int m0 = max(0, min(m_own, M_in - BM)), n0 = max(0, min(n_own, N_in - BN));

    // ---- the 16-byte pieces this thread moves each K step: piece `it` of an operand lies a fixed
    // number of rows below piece 0, in global memory and in LDS alike.  Global memory is read
    // through buffer descriptors: byte offset = uniform part (tile origin, K step, piece; scalar
    // registers) + per-thread part (one VGPR per operand).
    // EDGE_ANY: the buffers start at the dword that holds the operand's first element and end with the one that holds its
    // last (a dword at a multiple of 4 never reaches into another page); at the elements before and after sit no results.
    constexpr bool ANY = Loose<T, EDGE>::ANY, ODD = Loose<T, EDGE>::ODD;
    b = uniform<T>(b);
    const long a_rows = A_KC ? g.M : g.K, b_rows = B_KC ? g.N : g.K;
    const E *Ab = (const E *)g.A + (long)b * g.sA, *Bb = (const E *)g.B + (long)b * g.sB;
    const unsigned a_odd = ODD ? (unsigned)((size_t)Ab & 2) >> 1 : 0u, b_odd = ODD ? (unsigned)((size_t)Bb & 2) >> 1 : 0u;
    const long a_len = ANY ? (g.red - 1) * g.sA + (a_rows - 1) * g.lda + (A_KC ? g.K : g.M) + a_odd : (g.red - 1) * g.sA + a_rows * g.lda;
    // (the taps of a filter interleave inside its rows: the filter ends with its last row)
    const long b_len = ANY ? (g.red - 1) * g.sB + (b_rows - 1) * g.ldb + (B_KC ? g.K : g.N) + b_odd : (VA ? 0 : (g.red - 1) * g.sB) + b_rows * g.ldb;
    const int a_bytes = VA ? (int)pg.bytes : (int)((ES * a_len + 3) & ~3L), b_bytes = VIRT == VIRT_B_KROWS ? (int)pg.bytes : (int)((ES * b_len + 3) & ~3L);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(Ab - a_odd), 0, a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)(Bb - b_odd), 0, b_bytes, 0x00020000);
    // where the tile starts, in elements: uniform, but for half rows at any element only the dword part of it is
    const unsigned a_tile = (A_KC ? (unsigned)m0 * g.lda : (unsigned)m0) + a_odd, b_tile = (B_KC ? (unsigned)n0 * g.ldb : (unsigned)n0) + b_odd;
    const unsigned Au = (unsigned)ES * (ODD ? a_tile & ~1u : a_tile), Bu = (unsigned)ES * (ODD ? b_tile & ~1u : b_tile);
    const int a_r = A_KC ? tid >> 3 : tid / (BM / EPV), b_r = (B_KC || T::B_COLS) ? tid >> 3 : tid / (BN / EPV);
    int a_c = A_KC ? tid & 7 : tid % (BM / EPV), b_c = (B_KC || T::B_COLS) ? tid & 7 : tid % (BN / EPV);
    if constexpr (T::DMA) a_c = T::template chunk_of<A_KC, BM>(a_r, a_c), b_c = T::template chunk_of<B_KC, BN>(b_r, b_c);
    const int a_dst = (A_KC ? T::kc_row(a_r) : a_r * A_LD) + a_c * EPV, b_dst = (B_KC ? T::kc_row(b_r) : b_r * B_LD) + b_c * EPV;
    const unsigned a_pass = VA ? 0u : (unsigned)ES * T::A_ROWS * g.lda;  // bytes
    const unsigned b_pass = VIRT == VIRT_B_KROWS ? 0u : (unsigned)ES * T::B_ROWS * g.ldb;
    const unsigned a_step = A_KC ? 128u : (unsigned)ES * BK * g.lda;
    const unsigned b_step = B_KC ? 128u : (unsigned)ES * BK * g.ldb;
    // per-thread byte offset of each piece: one value for a real matrix, recomputed every step
    // for a patch matrix (an offset beyond the image makes the buffer load return zeros)
    constexpr unsigned OUTSIDE = 0x80000000u;
    const unsigned a_first = (unsigned)a_r * (unsigned)g.lda + a_c * EPV + (ODD ? a_tile & 1u : 0u);
    const unsigned b_first_el = (unsigned)b_r * (unsigned)g.ldb + b_c * EPV + (ODD ? b_tile & 1u : 0u);
    const unsigned av_plain = (unsigned)ES * (ODD ? a_first & ~1u : a_first), bv_plain = (unsigned)ES * (ODD ? b_first_el & ~1u : b_first_el);
    unsigned av[A_IT], bv[B_IT];
#pragma unroll
    for (int p = 0; p < A_IT; ++p) av[p] = av_plain;
#pragma unroll
    for (int p = 0; p < B_IT; ++p) bv[p] = bv_plain;
    Loose<T, EDGE> L;
    if constexpr (ODD) {
        L.shift[0] = (a_first & 1u) * 16, L.shift[1] = (b_first_el & 1u) * 16;
        L.next[0] = a_first & 1u ? 16u : OUTSIDE, L.next[1] = b_first_el & 1u ? 16u : OUTSIDE;
    }
    // patch rows as A: this thread's rows never change; a step selects the tap
    int va_base[A_IT], va_iy[A_IT], va_ix[A_IT];
    if constexpr (VA) {
        const Divisor plane(pg.OH * pg.OW, by_plane), width(pg.OW, by_ow);
#pragma unroll
        for (int p = 0; p < A_IT; ++p) {
            int rem, ox;
            const int m = g.m_base + m0 + a_r + p * T::A_ROWS, img = plane.div(m, rem), oy = width.div(rem, ox);
            va_iy[p] = oy * pg.sy - pg.pt;
            va_ix[p] = ox * pg.sx - pg.pl;
            va_base[p] = (((img * pg.H + va_iy[p]) * pg.W + va_ix[p]) * pg.C + a_c * EPV) * ES;
        }
    }
    // patch k-rows as B: this thread's taps and channels never change; a step selects the rows.  A row is one output
    // pixel, and each of the rows a thread fetches moves on by BK pixels per step: its source coordinates and byte
    // offset are kept and advanced by uniform amounts with a carry per axis, so a step costs a dozen additions and
    // selects per row instead of two divisions by multiplication and four further multiplications (a quarter of
    // the vector rate each).  A row past the last is in an image past the last, i.e. outside the buffer: zeros.
    // (with column passes, Tile::B_COLS: one row per thread and step, and piece p has its own tap and channel)
    constexpr int VB_N = VIRT == VIRT_B_KROWS ? (T::B_COLS ? 1 : B_IT) : 1;
    int vb_y[VB_N], vb_x[VB_N], vb_off[VB_N];  // source row, column and byte offset of this thread's rows
    int vb_ty[B_IT], vb_tx[B_IT], vb_toff[B_IT];  // column passes: tap displacement and byte offset of each piece
    int vb_y_end = 0, vb_x_end = 0;
    if constexpr (VIRT == VIRT_B_KROWS) {
        int cy = -pg.pt, cx = -pg.pl, cc = 0;  // what the tap and channel add to an output pixel's source coordinates
        if constexpr (T::B_COLS) {
            const Divisor channels(pg.C, g.by.channels), taps(pg.FW, g.by.taps_w);
#pragma unroll
            for (int p = 0; p < B_IT; ++p) {
                int c, fx;
                const int t = channels.div(n0 + p * T::B_PASS + b_c * EPV, c), fy = taps.div(t, fx);
                vb_ty[p] = fy * pg.dy;
                vb_tx[p] = fx * pg.dx;
                vb_toff[p] = ((vb_ty[p] * pg.W + vb_tx[p]) * pg.C + c) * ES;
            }
        } else {
            int fx;
            const int t = Divisor(pg.C, g.by.channels).div(n0 + b_c * EPV, cc), fy = Divisor(pg.FW, g.by.taps_w).div(t, fx);
            cy += fy * pg.dy;
            cx += fx * pg.dx;
        }
        vb_y_end = pg.OH * pg.sy + cy, vb_x_end = pg.OW * pg.sx + cx;
        const Divisor plane(pg.OH * pg.OW, by_plane), width(pg.OW, by_ow);
#pragma unroll
        for (int p = 0; p < VB_N; ++p) {
            int rem, ox;
            const int m = split * tps * BK + b_r + p * T::B_ROWS, img = plane.div(m, rem), oy = width.div(rem, ox);
            vb_y[p] = oy * pg.sy + cy;
            vb_x[p] = ox * pg.sx + cx;
            vb_off[p] = (((img * pg.H + vb_y[p]) * pg.W + vb_x[p]) * pg.C + cc) * ES;
        }
    }

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // ---- per-lane LDS offsets of its MFMA operands
    const int a_frag = A_KC ? T::kc_row(wm * TM * 32 + (lane & 31)) + (lane >> 5) * EL::KC_HALF : EL::tr_offset(lane, A_LD, wm * TM * 32);
    const int b_frag = B_KC ? T::kc_row(wn * TN * 32 + (lane & 31)) + (lane >> 5) * EL::KC_HALF : EL::tr_offset(lane, B_LD, wn * TN * 32);

    // ---- this workgroup's steps x0 .. x0 + nsteps - 1 of the extended reduction; step x reads
    // product x / ktiles at K offset (x % ktiles) * BK (all uniform: scalar arithmetic, counted on from step to step)
    // K need not be a multiple of the K step: the last step of a product (of a filter tap, where K is its channels) is then
    // partly past K, and the pieces that lie past it are fetched at an offset beyond the buffer, i.e. as zeros.  Where the
    // reduction runs over patch rows or over the rows of a real matrix, rows past the last lie outside the buffer anyway.
    const int ktiles = (g.K + BK - 1) / BK, last_len = g.K - (ktiles - 1) * BK;
    const int x0 = uniform<T>(split * tps), nsteps = min(red * ktiles, x0 + tps) - x0;
    const unsigned a_prod = (unsigned)ES * (unsigned)g.sA, b_prod = (unsigned)ES * (unsigned)g.sB;
    const unsigned b_prod_row = (unsigned)ES * (unsigned)g.sB_row, b_first = (unsigned)ES * b_cls;
    // The step that is fetched next: its product, K step and filter tap are counted on from step to step (every step is
    // fetched once, in order), because four divisions by runtime numbers at the head of each step -- some 35 dependent
    // scalar instructions that no matrix instruction covers -- were a fifth of a short half step's time.
    int ld_i = 0, ld_r = 0, ld_kx = 0, ld_fy = 0, ld_fx = 0;
    if constexpr (VIRT != VIRT_A_CLASSES) ld_r = uniform<T>(Divisor(ktiles, g.by.ktiles).div(x0, ld_kx));
    if constexpr (VIRT == VIRT_A_ROWS) ld_fy = uniform<T>(Divisor(pg.FW, g.by.taps_w).div(ld_r, ld_fx));
    // patch k-rows: what BK more pixels add, and the corrections when a row or an image is complete
    int vb_dy = 0, vb_dx = 0, vb_d = 0, vb_d_row = 0, vb_d_img = 0;
    if constexpr (VIRT == VIRT_B_KROWS) {
        int rem, ox;
        const int img = Divisor(pg.OH * pg.OW, by_plane).div(BK, rem), oy = Divisor(pg.OW, by_ow).div(rem, ox);
        vb_dy = oy * pg.sy, vb_dx = ox * pg.sx;
        vb_d = ((img * pg.H + vb_dy) * pg.W + vb_dx) * pg.C * ES;
        vb_d_row = (pg.sy * pg.W - pg.OW * pg.sx) * pg.C * ES;
        vb_d_img = (pg.H - pg.OH * pg.sy) * pg.W * pg.C * ES;
    }
    // How much of the step that is fetched lies within K: all of it, or what is left of K in a product's last step.  (Where
    // K is a multiple of the K step -- EDGE_NONE -- nothing asks: on patch rows in fp32 the
    // comparisons alone cost 2 % of a launch.)
    constexpr bool PARTIAL = EDGE != EDGE_NONE && VIRT != VIRT_B_KROWS;
    auto k_left = [&]() -> int { return ld_kx == ktiles - 1 ? last_len : BK; };
    auto step_a = [&]() -> unsigned {
        if constexpr (VA) {
            const int tdy = ld_fy * pg.dy, tdx = ld_fx * pg.dx;
            const int toff = ((tdy * pg.W + tdx) * pg.C + ld_kx * BK) * ES;
            const bool live = !PARTIAL || a_c * EPV < k_left();
#pragma unroll
            for (int p = 0; p < A_IT; ++p) {
                const bool inside = (unsigned)(va_iy[p] + tdy) < (unsigned)pg.H && (unsigned)(va_ix[p] + tdx) < (unsigned)pg.W;
                av[p] = inside && live ? (unsigned)(va_base[p] + toff) : OUTSIDE;
            }
            return 0u;
        } else {
            if constexpr (PARTIAL) {
                const int left = k_left();
#pragma unroll
                for (int p = 0; p < A_IT; ++p) av[p] = (A_KC ? a_c * EPV : a_r + p * T::A_ROWS) < left ? av_plain : OUTSIDE;
            }
            return Au + ld_r * a_prod + ld_kx * a_step;
        }
    };
    auto step_b = [&]() -> unsigned {
        if constexpr (VIRT == VIRT_B_KROWS) {
#pragma unroll
            for (int p = 0; p < B_IT; ++p) {
                const int q = T::B_COLS ? 0 : p;
                const int iy = vb_y[q] + (T::B_COLS ? vb_ty[p] : 0), ix = vb_x[q] + (T::B_COLS ? vb_tx[p] : 0);
                const bool inside = (unsigned)iy < (unsigned)pg.H && (unsigned)ix < (unsigned)pg.W;
                bv[p] = inside ? (unsigned)(vb_off[q] + (T::B_COLS ? vb_toff[p] : 0)) : OUTSIDE;
            }
            return 0u;
        }
        if constexpr (PARTIAL) {
            const int left = k_left();
#pragma unroll
            for (int p = 0; p < B_IT; ++p) bv[p] = (B_KC ? b_c * EPV : b_r + p * T::B_ROWS) < left ? bv_plain : OUTSIDE;
        }
        if constexpr (VIRT == VIRT_A_CLASSES) return Bu + b_first + ld_fy * b_prod_row + ld_fx * b_prod + ld_kx * b_step;
        return Bu + ld_r * b_prod + ld_kx * b_step;
    };
    // (selects, no branches: around a branch the compiler moves all accumulators out of the AGPRs and back.  Past the end
    // the last step is fetched again, or zeros where patch k-rows move on past it; never used)
    auto step_on = [&]() {
        ld_kx += ++ld_i < nsteps ? 1 : 0;
        const int done = ld_kx == ktiles ? 1 : 0;
        ld_kx = uniform<T>(done ? 0 : ld_kx);
        ld_r = uniform<T>(ld_r + done);
        if constexpr (VA) {
            ld_fx += done;
            const int row = ld_fx == pg.FW ? 1 : 0;
            ld_fx = uniform<T>(row ? 0 : ld_fx);
            ld_fy = uniform<T>(ld_fy + row);
        }
        if constexpr (VIRT == VIRT_B_KROWS) {
#pragma unroll
            for (int q = 0; q < VB_N; ++q) {
                vb_x[q] += vb_dx;
                const bool row = vb_x[q] >= vb_x_end;
                vb_x[q] -= row ? pg.OW * pg.sx : 0;
                vb_y[q] += vb_dy + (row ? pg.sy : 0);
                const bool img = vb_y[q] >= vb_y_end;
                vb_y[q] -= img ? pg.OH * pg.sy : 0;
                vb_off[q] += vb_d + (row ? vb_d_row : 0) + (img ? vb_d_img : 0);
            }
        }
    };

    // EDGE_ANY: the pieces that are written next are those of the step before the one fetched next
    int written_left = BK;
    auto next_step = [&](unsigned &pa, unsigned &pb) {
        if constexpr (ANY) {
            L.keep_first(0, written_left - a_c * EPV);
            L.keep_first(1, written_left - b_c * EPV);
            written_left = k_left();
        }
        pa = step_a(), pb = step_b();
        step_on();
    };
    unsigned pa, pb;
    if constexpr (T::DMA) {
        // the next step: where it lies (past the last one nothing is fetched), then its pieces one by one
        u32x4 da, db;
        unsigned sa, sb;
        auto aim = [&]() {
            const bool live = ld_i < nsteps;
            next_step(pa, pb);
            sa = __builtin_amdgcn_readfirstlane(pa), sb = __builtin_amdgcn_readfirstlane(pb);  // (scalars already: see uniform)
            const unsigned long at_a = (unsigned long)Ab, at_b = (unsigned long)Bb;
            da = (u32x4){(unsigned)at_a, (unsigned)(at_a >> 32) & 0xffffu, live ? (unsigned)a_bytes : 0u, 0x00020000u};
            db = (u32x4){(unsigned)at_b, (unsigned)(at_b >> 32) & 0xffffu, live ? (unsigned)b_bytes : 0u, 0x00020000u};
        };
        auto fetch = [&](auto piece, unsigned target) {
            constexpr int p = decltype(piece)::value;
            if constexpr (p < A_IT) dma_piece(target + p * T::NT * 16, da, av[p], sa + p * a_pass);
            else dma_piece(target + T::A_BYTES + (p - A_IT) * T::NT * 16, db, bv[p - A_IT], sb + (p - A_IT) * b_pass);
        };
        dma_loop<T>(As0, wave, lane, wm, wn, nsteps, acc, aim, fetch, [&]() { if (g.phase_rec) st_w[1] = wall_clock64(), st_c[0] = __builtin_readcyclecounter(); });
    } else {
        u32x4 R[NP];
        typename EL::Frag fa[2][TM], fb[2][TN];
        auto fetch_all = [&](unsigned pa, unsigned pb) {
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                R[p] = p < A_IT ? __builtin_amdgcn_raw_buffer_load_b128(ra, av[p < A_IT ? p : 0], pa + p * a_pass, 0)
                                : __builtin_amdgcn_raw_buffer_load_b128(rb, bv[p < A_IT ? 0 : p - A_IT], pb + (p - A_IT) * b_pass, 0);
                L.fetch(p, p < A_IT ? ra : rb, p < A_IT ? av[p < A_IT ? p : 0] : bv[p < A_IT ? 0 : p - A_IT], p < A_IT ? pa + p * a_pass : pb + (p - A_IT) * b_pass);
            }
        };

        // ---- prologue: step 0 into LDS half 0, step 1 into registers, first operands of step 0
        next_step(pa, pb);
        fetch_all(pa, pb);
        next_step(pa, pb);
#pragma unroll
        for (int p = 0; p < NP; ++p)
            *(u32x4 *)(p < A_IT ? As0 + a_dst + p * T::A_PASS : Bs0 + b_dst + (p - A_IT) * T::B_PASS) = L.place(p, R[p]);
        fetch_all(pa, pb);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TM; ++i)
            fa[0][i] = A_KC ? EL::read_kc(As0 + a_frag + i * T::A_BLK) : EL::read_tr(As0 + a_frag + i * 32, A_LD);
#pragma unroll
        for (int j = 0; j < TN; ++j)
            fb[0][j] = B_KC ? EL::read_kc(Bs0 + b_frag + j * T::B_BLK) : EL::read_tr(Bs0 + b_frag + j * 32, B_LD);

        if (g.phase_rec) st_w[1] = wall_clock64(), st_c[0] = __builtin_readcyclecounter();
        // ---- main loop, two steps per trip so that the LDS half of every access is known statically;
        for (int i = 0; i < nsteps; i += 2) {
            next_step(pa, pb);
            k_step<T, EDGE>(As0 + a_frag, Bs0 + b_frag, As1 + a_frag, Bs1 + b_frag, As1 + a_dst, Bs1 + b_dst, ra, rb, pa, pb,
                            a_pass, b_pass, av, bv, R, L, fa, fb, acc);
            if (i + 1 < nsteps) {
                next_step(pa, pb);
                k_step<T, EDGE>(As1 + a_frag, Bs1 + b_frag, As0 + a_frag, Bs0 + b_frag, As0 + a_dst, Bs0 + b_dst, ra, rb, pa, pb,
                                a_pass, b_pass, av, bv, R, L, fa, fb, acc);
            }
        }
    }

    if (g.phase_rec) st_w[2] = wall_clock64(), st_c[1] = __builtin_readcyclecounter();
    // ---- epilogue: the result itself, or this piece's fp32 partial sums when the reduction is split
    __syncthreads();  // every wave is past the last step: the operand areas are free
    const Origin o = {m0, n0, m_own, n_own, M, g.N, (wm * TM) * 32, (wn * TN) * 32};
    float *patches = (float *)(T::PATCH_IN_A ? As0 : Bs0), *patches1 = (float *)(T::PATCH_IN_A ? As1 : Bs1);
    if constexpr (T::DMA) patches1 = patches + T::HALF_PATCHES;
    if (in_tail) {  // partial sums of the band, rows counted from its first
        const int tail_M = M - g.tail_m0;
        const Origin ot = {m0 - g.tail_m0, n0, m_own - g.tail_m0, n_own, tail_M, g.N, (wm * TM) * 32, (wn * TN) * 32};
        store_tile<T, float, EDGE == EDGE_ANY>(acc, patches, patches1, g.ws + ((long)split * tail_M) * g.N, g.N, 0.f, true, g.N, ot, plain);
    } else if (g.splits > 1)
        store_tile<T, float, EDGE == EDGE_ANY>(acc, patches, patches1, g.ws + ((long)(b * g.splits + split) * g.M) * g.N, g.N, 0.f, true, g.N, o, plain);
    else
        store_tile<T, E, EDGE == EDGE_ANY>(acc, patches, patches1, (E *)g.C + (long)b * g.sC, g.ldc, g.beta,
                         g.ldc % EPV == 0 && g.sC % EPV == 0 && ((size_t)g.C & 15) == 0, g.N, o, crow, (const E *)g.bias, g.relu != 0,
                         ES == 2 && g.round_first != 0);
    if (g.phase_rec) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's stores have been acknowledged
        st_w[3] = wall_clock64();
        if (tid == 0) {
            unsigned long long *rec = g.phase_rec + 8 * (bx + (unsigned long long)nbx * bz);
            rec[0] = st_w[0], rec[1] = st_w[1], rec[2] = st_w[2], rec[3] = st_w[3], rec[4] = st_c[0], rec[5] = st_c[1];
            // s_getreg_b32 of all 32 bits of hardware registers 20 (XCC_ID) and 4 (HW_ID: wave, SIMD, CU, SH, SE)
            rec[6] = ((unsigned long long)__builtin_amdgcn_s_getreg((31 << 11) | 20) << 32) | __builtin_amdgcn_s_getreg((31 << 11) | 4);
            rec[7] = (in_tail ? 1 : 0) | (g.stamps << 1);  // (stamps: which product of a launch of two)
        }
    }
}

// (EDGE: instantiations of their own, so that the per-piece offsets of the ordinary case stay constants; patch k-rows as B
// need none)
// (classes on 128 x 128 tiles: left to itself the compiler takes 280 registers for the addresses of the element-wise store,
// which leaves room for one workgroup per compute unit; told to make room for two it takes 186 and spills none.  Half DeConv2d
// 32 x 20x20x128 -> 128, 2x2 stride 2, 15.7 -> 11.0 us; 24 x 26x26x448 -> 288, 4x4 stride 2, 150 -> 119 us)
template <typename T, int EDGE = EDGE_NONE>
__global__ __launch_bounds__(T::NT, T::VIRT == VIRT_A_CLASSES && T::BN == 128 || T::TWO_FIT ? 2 : 1) void gemm_tiled_kernel(GemmArgs g, int tilesM, int tilesN) {
    typedef typename T::E E;
    if constexpr (T::DMA) {
        __shared__ __attribute__((aligned(1024))) E stages[T::LDS_BYTES / T::ES];
        gemm_tiled_body<T, EDGE>(g, tilesM, tilesN, (int)blockIdx.x, (int)blockIdx.z, (int)gridDim.x, stages, nullptr, nullptr, nullptr);
    } else {
        // four separate arrays, so that reads of one half are known not to touch the other
        __shared__ __attribute__((aligned(16))) E As0[T::A_SZ];
        __shared__ __attribute__((aligned(16))) E As1[T::A_SZ];
        __shared__ __attribute__((aligned(16))) E Bs0[T::B_SZ];
        __shared__ __attribute__((aligned(16))) E Bs1[T::B_SZ];
        gemm_tiled_body<T, EDGE>(g, tilesM, tilesN, (int)blockIdx.x, (int)blockIdx.z, (int)gridDim.x, As0, As1, Bs0, Bs1);
    }
}

// Two products in one launch: the first nx0 * nz0 workgroups are the first product's grid (x fastest), the rest the
// second's.  Built for the two gradients of a convolution on a small layer, which are independent of each other and
// each leave the chip half empty: their workgroups are short (a dozen K steps between a prologue and an epilogue
// that nothing hides when a compute unit holds one workgroup), and side by side on a compute unit one's waits are
// the other's issue slots.  The operand areas are as large as the larger tile needs.
template <typename T0, typename T1, int EDGE = EDGE_NONE>
__global__ __launch_bounds__(T0::NT, T0::TWO_FIT && T1::TWO_FIT ? 2 : 1) void gemm_tiled_pair_kernel(int ahead, int nx0, int nz0, int nx1, int tilesM0, int tilesN0,
                                                                 int tilesM1, int tilesN1, GemmArgs g0, GemmArgs g1) {
    typedef typename T0::E E;
    static_assert(T0::NT == T1::NT && sizeof(typename T0::E) == sizeof(typename T1::E) && T0::DMA == T1::DMA, "one workgroup shape, one element type");
    if constexpr (T0::DMA) {
        __shared__ __attribute__((aligned(1024))) E stages[(T0::LDS_BYTES > T1::LDS_BYTES ? T0::LDS_BYTES : T1::LDS_BYTES) / T0::ES];
        const int at = (int)blockIdx.x, first = nx0 * nz0, id = at < ahead ? at + first : at - ahead, j = id - first;
        int bx;
        if (id < first) {
            const int bz = Divisor(nx0, g0.by.nbx).div(id, bx);
            gemm_tiled_body<T0, EDGE>(g0, tilesM0, tilesN0, bx, bz, nx0, stages, nullptr, nullptr, nullptr);
        } else {
            const int bz = Divisor(nx1, g1.by.nbx).div(j, bx);
            gemm_tiled_body<T1, EDGE>(g1, tilesM1, tilesN1, bx, bz, nx1, stages, nullptr, nullptr, nullptr);
        }
    } else {
        constexpr int A_SZ = T0::A_SZ > T1::A_SZ ? T0::A_SZ : T1::A_SZ, B_SZ = T0::B_SZ > T1::B_SZ ? T0::B_SZ : T1::B_SZ;
        __shared__ __attribute__((aligned(16))) E As0[A_SZ];
        __shared__ __attribute__((aligned(16))) E As1[A_SZ];
        __shared__ __attribute__((aligned(16))) E Bs0[B_SZ];
        __shared__ __attribute__((aligned(16))) E Bs1[B_SZ];
        const int at = (int)blockIdx.x, first = nx0 * nz0, id = at < ahead ? at + first : at - ahead;
        int bx;
        if (id < first) {
            const int bz = Divisor(nx0, g0.by.nbx).div(id, bx);
            gemm_tiled_body<T0, EDGE>(g0, tilesM0, tilesN0, bx, bz, nx0, As0, As1, Bs0, Bs1);
        } else {
            const int bz = Divisor(nx1, g1.by.nbx).div(id - first, bx);
            gemm_tiled_body<T1, EDGE>(g1, tilesM1, tilesN1, bx, bz, nx1, As0, As1, Bs0, Bs1);
        }
    }
}

// The kernel tile of a BM x BN output tile: in half, operands in whole pieces go straight into LDS, on four waves and as many
// stages as let FIT workgroups share a compute unit.
// FIT 1: 128 x 128 tiles of a launch of at most one workgroup per compute unit,
// which may have all of its LDS: two stages fetch one step ahead, less than the way from memory takes (2048^3, a K step of 128 x
// 128: 1270 cycles with two stages, 825 - 870 with four; with five the same), and eight waves share out the addresses of
// patch rows (Conv2d 16 x 57x57x96 -> 160, 3x3 stride 2, forward 17.1 us with four waves, 15.3 with eight).  More stages or
// eight waves on the smaller tiles gave nothing (64 x 64 with 4, 6, 8 stages 454, 516, 522 cycles a step, with eight waves 520).
// FIT 3: smaller tiles of a launch of more than two workgroups per compute unit.  Two stages let three in (64 x 64: four), which
// hide each other's prologue and store and need no further
// round.  100 drawn half Conv2d of 8 to 100 channels, forward, 1286 -> 1244 us (1360 on tiles that pass through registers, of which
// none is lost by 3 % any more): 29 x 55x55x16 -> 42 1x1 12.1 -> 9.3, DeConv2d 23 x 18x18x8 -> 72 4x4 stride 2 12.4 -> 9.8.
template <typename E, int BM, int BN, bool A_KC, bool B_KC, int VIRT = VIRT_NONE, int FIT = 2>
struct TileOf {
    typedef Tile<E, BM, BN, BM == 256 || BN == 32 ? 4 : 2, BN == 32 ? 1 : 2, A_KC, B_KC, VIRT> type;
};
template <bool A_KC, bool B_KC, int VIRT, int FIT>
struct TileOf<f16, 64, 64, A_KC, B_KC, VIRT, FIT> {
    typedef DmaTile<64, 64, 2, 2, FIT == 3 ? 2 : 4, A_KC, B_KC, VIRT> type;
};
template <bool A_KC, bool B_KC, int VIRT, int FIT>
struct TileOf<f16, 64, 128, A_KC, B_KC, VIRT, FIT> {
    typedef DmaTile<64, 128, 2, 2, FIT == 3 ? 2 : 3, A_KC, B_KC, VIRT> type;
};
template <bool A_KC, bool B_KC, int VIRT, int FIT>
struct TileOf<f16, 128, 64, A_KC, B_KC, VIRT, FIT> {
    typedef DmaTile<128, 64, 2, 2, FIT == 3 ? 2 : 3, A_KC, B_KC, VIRT> type;
};
template <bool A_KC, bool B_KC, int VIRT, int FIT>
struct TileOf<f16, 128, 128, A_KC, B_KC, VIRT, FIT> {
    typedef DmaTile<128, 128, 2, FIT == 1 ? 4 : 2, FIT == 1 ? 4 : 2, A_KC, B_KC, VIRT> type;
};

// where d8_gemm_phase_record asked the next launches to write their records (process-wide; null: no records; defined in
// gemm_tiled.hip)
extern unsigned long long *phase_rec_buf;
extern size_t phase_rec_bytes;

// What the kernel divides by (GemmArgs::by) for a grid of tilesM x tilesN tiles of BM rows and nbx workgroups a layer.
static inline void set_reciprocals(GemmArgs &g, int tilesM, int tilesN, int BM, int BK, int nbx) {
    TiledReciprocals &by = g.by;
    by.layers = reciprocal_of(g.splits), by.tiles = reciprocal_of(tilesM * tilesN), by.band = reciprocal_of(4 * tilesN);
    by.ktiles = reciprocal_of(ceil_div(g.K, BK)), by.nbx = reciprocal_of(nbx), by.perm_OC = reciprocal_of(g.perm_OC);
    by.taps_w = reciprocal_of(g.pg.FW), by.channels = reciprocal_of(g.pg.C);
    by.plane = reciprocal_of(g.pg.OH * g.pg.OW), by.ow = reciprocal_of(g.pg.OW);
    by.tail_splits = reciprocal_of(g.tail_splits), by.tail_tilesM = reciprocal_of(ceil_div(g.M - g.tail_m0, BM));
    if (g.virt == VIRT_A_CLASSES)
        for (int i = 0; i < g.ncls; ++i) g.cls[i].by_plane = reciprocal_of(g.cls[i].OH * g.cls[i].OW), g.cls[i].by_ow = reciprocal_of(g.cls[i].OW);
}

// Launches of one product, one translation unit each (gemm_tiled_launch.h)
int gemm_tiled_plain_f16(const GemmArgs &g, int transA, int transB, hipStream_t stream);
int gemm_tiled_plain_f32(const GemmArgs &g, int transA, int transB, hipStream_t stream);
int gemm_tiled_patch_f16(const GemmArgs &g, int transB, hipStream_t stream);
int gemm_tiled_patch_f32(const GemmArgs &g, int transB, hipStream_t stream);

// Which tile a product runs on.
enum TileId { TILE_WIDE, TILE_256, TILE_128x64, TILE_64x64, TILE_64x128, TILE_128x128, TILE_128x32 };

// Whether both operands of a product of real matrices can be moved in 16-byte pieces that K does not cut (else EDGE_ANY).
template <typename E>
static bool in_pieces(const GemmArgs &g, bool a_kc, bool b_kc) {
    constexpr int EPV = 16 / (int)sizeof(E), BK = 128 / (int)sizeof(E);
    if (g.packed) return true;
    if ((g.lda | g.ldb) % EPV || (g.sA | g.sB) % EPV || (((size_t)g.A | (size_t)g.B) & 15)) return false;
    if ((a_kc || b_kc) && g.K % BK && g.K % EPV) return false;
    return (a_kc || g.M % EPV == 0) && (b_kc || g.N % EPV == 0);
}

template <typename E, bool A_KC, bool B_KC, int VIRT = VIRT_NONE>
static TileId choose_tile(const GemmArgs &g, bool any = false) {
    static const char *force = getenv("D8_GEMM_TILE");  // tuning aid
    if (g.tile_hint) return g.tile_hint == HINT_128x32 ? TILE_128x32 : TILE_64x64;
    const long big_tiles = (long)ceil_div(g.M, 256) * ceil_div(g.N, 256) * g.batch * g.splits;
    bool big = g.M >= 256 && g.N >= 256 && big_tiles >= (long)cu_count() * 3 / 4;
    if (force && g.M >= 256 && g.N >= 256) big = atoi(force) != 128;
    // fp32 runs 64-cycle MFMAs on a quarter of the bytes per flop: the 128 x 128 tile already
    // keeps the matrix pipe fed, and the compiler cannot hold the 256 x 256 variant in registers
    if (any || g.packed) big = false;  // (and rows that start anywhere have no kernel of 256 x 256 tiles)
    if constexpr (sizeof(E) == 2) {
        static const char *wide = getenv("D8_GEMM_WIDE");  // tuning aid: 0 keeps the 32x32x16 kernel
        if (big && VIRT == VIRT_NONE && !(wide && atoi(wide) == 0) && gemm_wide_eligible(g, !A_KC, B_KC)) return TILE_WIDE;
        if (big) return TILE_256;
    }
    // an output smaller than a tile both ways (a filter gradient of few channels and taps)
    if ((VIRT == VIRT_B_KROWS || any) && g.M < 128 && g.N < 128) return TILE_64x64;
    // a 64-wide side gets a tile of that width (im2col products with 64 output channels)
    if (g.N < 128) return TILE_128x64;
    // a patch-matrix product whose last 128-column tile would be at most half full: 64 x 64 tiles, no padding
    // multiplied (C4's filter gradient, N = 576: 83.7 -> 73.8 us)
    if (gemm_tiled_krows_64(VIRT, g.M, g.N)) return TILE_64x64;
    if (g.M < 128) return TILE_64x128;
    if (g.splits == 1 && gemm_tiled_half_tiles(g.M, g.N, g.batch, (long)g.red * ceil_div(g.K, 128 / (int)sizeof(E)), 128 / (int)sizeof(E)))
        return TILE_64x128;
    return TILE_128x128;
}

// ---- two products in one launch (gemm_tiled_pair_kernel): the tile grid of a product, and the launch of gy's workgroups
// followed by gx's
static void grid_of(TileId t, const GemmArgs &g, int &tilesM, int &tilesN) {
    const int bm = (t == TILE_64x64 || t == TILE_64x128) ? 64 : 128, bn = (t == TILE_64x64 || t == TILE_128x64) ? 64 : 128;
    tilesM = ceil_div(g.M, bm), tilesN = ceil_div(g.N, bn);
}

template <typename TX, typename TY, int EDGE = EDGE_NONE>
static int launch_pair_tiles(const GemmArgs &gx0, const GemmArgs &gy0, hipStream_t stream) {
    GemmArgs gx = gx0, gy = gy0;
    // (gx may carry its remainder band as pieces of the same launch: GemmArgs::tail_m0; then it has one layer)
    const bool tail = gx.tail_splits > 0;
    const int tMx = ceil_div(tail ? gx.tail_m0 : gx.M, TX::BM), tNx = ceil_div(gx.N, TX::BN), tMy = ceil_div(gy.M, TY::BM), tNy = ceil_div(gy.N, TY::BN);
    const int extra = tail ? ceil_div(gx.M - gx.tail_m0, TX::BM) * tNx * gx.tail_splits : 0;
    const int ny = tMy * tNy, nzy = gy.batch * gy.splits, nx = tMx * tNx + extra;
    const int nzx = TX::VIRT == VIRT_A_CLASSES ? gx.ncls : tail ? 1 : gx.batch * gx.splits;
    // phase records (a measurement aid): gy's workgroups first, then gx's, tagged 0 and 1
    const bool rec = (size_t)(ny * nzy + nx * nzx) * 64 <= phase_rec_bytes;
    gy.phase_rec = rec ? phase_rec_buf : nullptr, gy.stamps = 0;
    gx.phase_rec = rec && phase_rec_buf ? phase_rec_buf + 8L * ny * nzy : nullptr, gx.stamps = 1;
    // (at most two workgroups per compute unit: none takes a third, as in launch_edge)
    constexpr long third = 160 * 1024 / 3;
    long lds;
    if constexpr (TX::DMA) lds = TX::LDS_BYTES > TY::LDS_BYTES ? TX::LDS_BYTES : TY::LDS_BYTES;
    else lds = 2L * ((TX::A_SZ > TY::A_SZ ? TX::A_SZ : TY::A_SZ) + (TX::B_SZ > TY::B_SZ ? TX::B_SZ : TY::B_SZ)) * TX::ES;
    const long wgs = (long)ny * nzy + (long)nx * nzx, cus = cu_count();
    const unsigned pad = lds <= third && wgs > cus && wgs <= 2 * cus ? (unsigned)(third + 512 - lds) : 0u;
    // Of more workgroups than compute units the longer ones first, gx's (`ahead` of them) or gy's: what starts last runs alone at the end.
    // fp32 classes, whose longest run up to twice their mean, only where the chip cannot hold all workgroups at once: two of them on a compute
    // unit end later than one beside a shorter one of gy's (Conv2d, both gradients, gx's first / gy's: 31 x 15x15x64 -> 320 5x5 stride 2 120 /
    // 101 us, 27 x 24x18x120 -> 128 3x3 stride 2 34.5 / 29.0; of more, 26 x 28x28x256 -> 96 61 / 77; in half either may be first).
    auto time = [](const GemmArgs &g, int bm, int bn, int bk, double red) {
        const double steps = g.splits > 1 ? g.tiles_per_split : red * ceil_div(g.K, bk);
        return steps * (TX::DMA ? bm + bn : bm * bn);  // (half waits for its loads, fp32 for its matrix instructions)
    };
    double red = gx.red;
    if constexpr (TX::VIRT == VIRT_A_CLASSES) {  // (at the mean)
        red = 0;
        for (int i = 0; i < gx.ncls; ++i) red += (double)gx.cls[i].red / gx.ncls;
    }
    const bool crowded = wgs > (TX::VIRT == VIRT_A_CLASSES && !TX::DMA ? 2 * cus : cus);
    const int ahead = crowded && time(gx, TX::BM, TX::BN, TX::BK, red) > time(gy, TY::BM, TY::BN, TY::BK, gy.red) ? nx * nzx : 0;
    set_reciprocals(gy, tMy, tNy, TY::BM, TY::BK, ny);
    set_reciprocals(gx, tMx, tNx, TX::BM, TX::BK, nx);
    hipLaunchKernelGGL((gemm_tiled_pair_kernel<TY, TX, EDGE>), dim3(ny * nzy + nx * nzx), dim3(TX::NT), pad, stream, ahead, ny, nzy, nx, tMy, tNy, tMx, tNx, gy, gx);
    D8_LAUNCH_CHECK();
    return 0;
}

}  // namespace d8

#endif
