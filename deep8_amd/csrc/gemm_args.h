// Argument block shared by the GEMM kernels and their host-side dispatcher.
#ifndef DEEP8_AMD_GEMM_ARGS_H
#define DEEP8_AMD_GEMM_ARGS_H

#include "common.h"

namespace d8 {

// A patch matrix that is never written out: row m = (b, oy, ox) enumerates an OH x OW grid per
// image, column (t, c) is channel c of filter tap t = fy * FW + fx, and the element is
//   image[b][oy * sy + fy * dy - pt][ox * sx + fx * dx - pl][c]      (0 outside the image).
// dy, dx, pt, pl may be negative, which expresses the gradient-side gather of a stride-1
// convolution (source row = iy + pt - fy * dy) with the same formula.
struct PatchGeom {
    int H, W, C;    // the image [B][H][W][C] the patches are cut from
    int OH, OW;     // the grid the rows enumerate
    int FW;         // taps per filter row
    int sy, sx, dy, dx, pt, pl;
    unsigned mg_plane, mg_ow;  // floor(2^32 / (OH * OW)), floor(2^32 / OW): division by multiplication
    unsigned bytes;            // size of the image
};

enum { VIRT_NONE = 0, VIRT_A_ROWS = 1, VIRT_B_KROWS = 2, VIRT_A_CLASSES = 3 };

// A strided transposed convolution, output pixel by output pixel: the output pixels whose
// coordinates have one residue (py, px) modulo the stride form a class; a class is an ordinary
// stride-1 patch product over the taps fy = f0y + sy * j, fx = f0x + sx * i that reach it:
//   z[b][sy * y' + py][sx * x' + px][:] = sum over (j, i) of x[b][y' + j - pt][x' + i - pl][:] . w[:][fy][fx][:]
// VIRT_A_CLASSES runs all classes in one launch (blockIdx.z = class): the patch grid, the taps, the
// filter slice and the rows of C a class writes come from its OutClass, everything else from GemmArgs.
struct OutClass {
    int M;             // rows (b, y', x') of the class
    int OH, OW;        // its grid of (y', x')
    int taps_w, red;   // taps per filter row that reach it, and in all
    int pt, pl;        // patch origin (may be negative)
    int py, px;        // residue: output pixel = (sy * y' + py, sx * x' + px)
    unsigned b_off;    // element offset of the filter slice of its first tap (f0y, f0x)
    unsigned by_plane, by_ow;  // reciprocal_of(OH * OW), reciprocal_of(OW), set at the launch of a tiled kernel
};
enum { MAX_CLASSES = 16 };

// Division of 0 <= n < 2^31 by a d > 0 that the host knows: n times reciprocal_of(d) over 2^32 is the quotient or one less.  Half a
// dozen instructions, scalar ones where n is uniform, instead of some 25 in a row.  The tiled kernels had 7 to 15 of those, one
// after the other, before their first load (550 - 790 instructions, now 200 - 500): DeConv2d forward, half 4 x 23x23x104 -> 448
// 2x2 stride 2 9.9 -> 9.0 us, fp32 25 x 37x37x64 -> 51 3x3 stride 2 49.6 -> 44.3; Conv2d 16 x 57x57x96 -> 160 3x3 stride 2,
// forward and gradients, 53.0 -> 47.4; 42 drawn DeConv2d forward calls 6 % faster at the mean, none more than 1 % slower.
inline unsigned reciprocal_of(int d) { return 0xffffffffu / (unsigned)(d < 1 ? 1 : d); }
struct Divisor {
    int d;
    unsigned m;
    __device__ __forceinline__ Divisor(int by, unsigned reciprocal) : d(by), m(reciprocal) {}
    __device__ __forceinline__ int div(int n, int &rem) const {
        int q = (int)__umulhi((unsigned)n, m);
        rem = n - q * d;
        const bool more = rem >= d;
        rem -= more ? d : 0;
        return q + (more ? 1 : 0);
    }
};
// What the tiled kernels divide by before their first load, set at the launch.
struct TiledReciprocals {
    unsigned layers, tiles, band;         // splits; tiles of the grid; tiles of a band of four tile rows
    unsigned ktiles, taps_w;              // K steps of a product, taps per filter row
    unsigned plane, ow, channels;         // of the patch geometry
    unsigned tail_splits, tail_tilesM;    // of the remainder band
    unsigned perm_OC;
    unsigned nbx;                         // a launch of two products: workgroups of a layer of the grid
    unsigned row, groups;                 // the pass over partial sums: N; groups of four outputs
};

struct GemmArgs {
    const void *A;
    const void *B;
    void *C;
    float *ws;
    int M, N, K;
    int lda, ldb, ldc;
    long sA, sB, sC;
    int batch;            // independent outputs
    int red;              // products summed into each output (1 unless strideC == 0)
    int splits;           // pieces the extended reduction (red x K tiles) is cut into
    int tiles_per_split;  // K tiles per piece
    float beta;
    // Implicit convolution: one operand is a patch matrix read straight from the image.
    //   VIRT_A_ROWS   A is the image; product r of the `red` summed products is filter tap r, its
    //                 A[m][k] = channel k of tap r of patch row m (K = channels per tap)
    //   VIRT_B_KROWS  B is the image; B[k][n] = column n of patch row k (N = taps x channels)
    int virt;
    PatchGeom pg;
    int m_base;  // VIRT_A_ROWS: row 0 of this product is patch row m_base (a product over a band of rows)
    // VIRT_A_CLASSES: product (j, i) of a class reads B at b_off + j * sB_row + i * sB; row (b, y', x') of
    // the class is row ((b * out_H + out_sy * y' + py) * out_W + out_sx * x' + px) of C
    long sB_row;
    int out_H, out_W, out_sy, out_sx;
    int ncls;
    // perm_OC > 0: the result is stored transposed per filter tap: element (m, n = t * perm_OC + oc) of the
    // product goes to C[(oc * perm_T + t) * ldc + m] (a filter gradient [OC][taps][IC] computed as [IC][taps x OC])
    int perm_T, perm_OC;
    // measurement aid (gemm_wide only, set by its launcher when the environment asks for it and a workspace
    // is given): every workgroup records when its prologue, K loop and epilogue ended into ws
    int stamps;
    size_t ws_bytes;  // size of ws as d8_gemm received it (0 where a planner filled the block in)
    // Fused store (the tiled kernels, the large-output fp16 kernel, the small-product kernel and the split reduction): after the product
    // (and beta * C), column n of the result gets bias[n] added (bias: N elements of C's type, may be null),
    // then negative values become 0 when relu is set.  What Add (a per-column bias broadcast over the rows) and
    // ReLu do as separate passes over C in the reference (deep8/src/math/Add.cu:21-52, ReLu.cu:20-59).
    const void *bias;
    int relu;
    // Half: the product is rounded to half before the bias is added, as a separate pass over it would find it.  Set where
    // product and bias + ReLu used to be two passes: a gate decided by the sum that is rounded once opens for other
    // elements (about one in five thousand), and a layer keeps the gates it had.
    int round_first;
    // Half, rows that started anywhere, copied to rows of whole 16-byte pieces (gemm_pack): the operands may be moved in pieces
    // though M, N or K is no multiple of one; what the loads may reach along M and N (operands not stored along K) is padM,
    // padN; what follows K in a row is zero.  C is stored at the alignment of an element.
    int packed, padM, padN;
    // a smaller tile than the shape's own (128 x 32: fp32 only), chosen by gemm_tiled_run and gemm_tiled_run_plain_pair
    // (few_tiles_small, narrow_output)
    int tile_hint;
    // half: which estimate plans the pieces (few_tiles_small).  Of two gradients that share a launch, or would, the one that suits
    // the two of them (half_pair_plan)
    int pieces_by;
    // Remainder band in the same launch (tail_splits > 0; unsplit, unbatched products only): rows tail_m0 .. M - 1
    // are not tiled by the launch's first tiles(tail_m0) x tiles(N) workgroups but by further ones, tail_splits per
    // tile, each walking tail_tps K steps and writing fp32 partial sums to ws[piece][row - tail_m0][n].  They start
    // as the first workgroups retire, so the band costs a fraction of a tile's time instead of a launch of its own.
    int tail_m0, tail_splits, tail_tps;
    // measurement aid of the tiled kernels (d8_gemm_phase_record): when set, every workgroup writes eight 64-bit words
    // at index blockIdx.x + gridDim.x * blockIdx.z -- the chip's 100 MHz wall clock at its start, after its prologue,
    // after its K loop and after its last store was acknowledged, the shader clock at both ends of the loop, its
    // placement (XCC_ID << 32 | HW_ID) and, in the last word, whether it worked on the remainder band (bit 0) and which
    // product of a launch of two it belongs to (bit 1: gemm_tiled_pair_launch's gx)
    unsigned long long *phase_rec;
    TiledReciprocals by;
    OutClass cls[MAX_CLASSES];  // (last: a kernel reads one of them, and the rest of its arguments from lines that follow each other)
};

enum { HINT_NONE = 0, HINT_64x64 = 1, HINT_128x32 = 2 };  // GemmArgs::tile_hint
enum { BY_TILE_TIMES = 0, BY_STEPS = 1, BY_SHARED_TIMES = 2 };  // GemmArgs::pieces_by

// Whether two gradients have run as one launch.  Of a MatrixMultiply: SHARED if their reductions are whole K steps (or both are small, or
// copies) and all their workgroups fit the chip at once, else SHARED_KEPT.  Of a convolution, tiled and cut as alone: SHARED_KEPT if in fp32
// both have 128 x 128 tiles or there are more workgroups than run at once, else SHARED.  The two are counted apart
// (d8_matmul_grad_pair_launches, ..._kept_pair_launches; d8_conv_grad_kept_pair_launches, ..._crowded_pair_launches).
enum SharedLaunch { APART = 0, SHARED, SHARED_KEPT };
enum TiledRule { TILED_ANY, TILED_PIECES, TILED_WHOLE };  // see gemm_tiled_eligible

// Whether a product with these arguments would run on a kernel that applies GemmArgs::bias / relu in its store
// (else the caller runs the plain product and launch_bias_relu).
bool gemm_fuses_store(int dtype, const GemmArgs &g, int transA, int transB, TiledRule rule = TILED_ANY);
// The product of d8_gemm (beta = 0, no summed batch) with the fused store; the shape must pass gemm_fuses_store.
int gemm_run_fused(int dtype, GemmArgs &g, int transA, int transB, void *workspace, size_t workspace_bytes, hipStream_t stream);
// z[r][c] = relu?(z[r][c] + bias[c]) in place, one pass (bias may be null): the fallback for shapes the fused store does not take.
int launch_bias_relu(int dtype, void *z, const void *bias, long rows, int cols, int relu, hipStream_t stream);

// Tiled kernels (fp16 and fp32): operands that can be moved in 16-byte pieces, and real matrices whose rows start at any element.
int gemm_tiled_k_step(int dtype);  // K elements per step: 64 (fp16) or 32 (fp32)
// Whether the shape qualifies (g.splits / g.tiles_per_split need not be set yet).
//   TILED_ANY     whatever a single launch takes: real matrices of any shape and alignment (but sums of half matrices an odd
//                 number of elements apart, and short reductions over many tiles of rows that start anywhere, which the
//                 any-shape kernel has), patch matrices whose channels can be moved in 16-byte pieces
//   TILED_PIECES  ... real matrices too only in 16-byte pieces, and at least one side of the output as long as a tile (what
//                 a launch of two products takes)
//   TILED_WHOLE   ... and patch matrices only where all K steps are whole and the output is no smaller than a tile (what
//                 a launch of a convolution's two gradients takes, and what the scratch queries plan without an interim
//                 matrix)
bool gemm_tiled_eligible(int dtype, const GemmArgs &g, int transA, int transB, TiledRule rule = TILED_ANY);
// Launch; with g.splits > 1 the fp32 partial sums go to g.ws for the caller to reduce.
int gemm_tiled_launch(int dtype, const GemmArgs &g, int transA, int transB, hipStream_t stream);
bool gemm_tiled_loose(int dtype, const GemmArgs &g, int transA, int transB);  // runs on the variant for rows that start anywhere
// Two patch-matrix products as ONE launch: gx with patch rows as A (NN: a convolution's gradient of its input), gy with
// patch k-rows as B (TN: its filter gradient; g.splits / tiles_per_split set, the caller reduces).  Workgroups of
// both are resident side by side.  gemm_tiled_pair_workgroups: how many workgroups the launch would have, 0 when the
// pair cannot run this way (the tiles the two products would choose have no common kernel, or one is cut into a band).
long gemm_tiled_pair_workgroups(int dtype, const GemmArgs &gx, const GemmArgs &gy);
int gemm_tiled_pair_launch(int dtype, const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream);
// The same with both products tiled and cut as they would be alone, also where K cuts the last step of gx short and where
// gx runs over classes of output pixels (VIRT_A_CLASSES: strides above 1).  _plan decides and sets how the reductions are
// cut; _run launches and reduces.
bool gemm_tiled_kept_pair_plan(int dtype, GemmArgs &gx, GemmArgs &gy, void *workspace, size_t workspace_bytes);
int gemm_tiled_kept_pair_run(int dtype, const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream);
SharedLaunch gemm_tiled_kept_pair_tiles_f16(const GemmArgs &gx, const GemmArgs &gy);
SharedLaunch gemm_tiled_kept_pair_tiles_f32(const GemmArgs &gx, const GemmArgs &gy);
int gemm_tiled_pair_rows_f16(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream);
int gemm_tiled_pair_rows_f32(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream);
int gemm_tiled_pair_classes_f16(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream);
int gemm_tiled_pair_classes_f32(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream);
// The same for two real products: g0 NT, g1 TN (the two gradients of a MatrixMultiply), each batched or split as planned
// (g.splits / tiles_per_split / ws set; the caller reduces).
long gemm_tiled_plain_pair_workgroups(int dtype, const GemmArgs &g0, const GemmArgs &g1);
int gemm_tiled_plain_pair_launch(int dtype, const GemmArgs &g0, const GemmArgs &g1, hipStream_t stream);
int gemm_tiled_plain_pair_pieces_f16(const GemmArgs &g0, const GemmArgs &g1, hipStream_t stream);
int gemm_tiled_plain_pair_pieces_f32(const GemmArgs &g0, const GemmArgs &g1, hipStream_t stream);
// Where the next launches write their per-workgroup phase records (GemmArgs::phase_rec); null switches them off.
void gemm_tiled_phase_record(void *records, size_t bytes);

// fp16 kernel for large outputs (256 x 256 tiles, v_mfma_f32_16x16x32_f16, loads straight into
// LDS): unsplit, unsummed products of real matrices with M, N >= 256 and K a multiple of 64.
bool gemm_wide_eligible(const GemmArgs &g, int transA, int transB);
int gemm_wide_launch(const GemmArgs &g, int transA, int transB, hipStream_t stream);
// Two such products (each eligible) as ONE launch: a workgroup that has finished a tile of the first goes on to a
// tile of the second without the kernel boundary in between (the end of one launch -- the write of the whole of
// C, the wait for its acknowledgement, the gap -- and the start of the next, whose first operand bytes come from
// memory).  Built for the two gradients of a MatrixMultiply, which are independent of each other.
int gemm_wide_pair_launch(const GemmArgs &g0, int transA0, int transB0, const GemmArgs &g1, int transA1, int transB1,
                          hipStream_t stream);

// Whether the two gradients of a MatrixMultiply (NT, TN) run on the small-product kernel, and one of them on it.
bool gemm_gradients_are_small(int dtype, const GemmArgs &g0, int ta0, int tb0, const GemmArgs &g1, int ta1, int tb1);
int gemm_small_run(int dtype, const GemmArgs &g, int transA, int transB, hipStream_t stream);
// Whether the two by their shapes share a launch of the tiled kernels, given aligned tensors and scratch enough; their pieces_by is set if so.
bool gemm_gradients_share(int dtype, GemmArgs &g0, int ta0, int tb0, GemmArgs &g1, int ta1, int tb1);
// The pieces_by of a convolution's gradient of x on patch rows, beside the filter's gradient gy (half; else nothing is set).
void gemm_conv_pieces(int dtype, GemmArgs &gx, const GemmArgs &gy);
// Both as ONE launch; APART, with nothing launched, when they do not qualify.
SharedLaunch gemm_small_pair_run(int dtype, const GemmArgs &g0, int ta0, int tb0, const GemmArgs &g1, int ta1, int tb1, hipStream_t stream, int *rc);

// fp64 kernel (64 x 64 or 128 x 128 tiles, v_mfma_f64_16x16x4_f64): any shape; plans its own split of the
// reduction from g.ws / g.ws_bytes (double partial sums) and reduces.
int gemm_f64_launch(const GemmArgs &g, int transA, int transB, hipStream_t stream);
// Pieces it would cut the reduction into given that much workspace.
int gemm_f64_splits(int M, int N, int K, int batch, int red, size_t workspace_bytes, int *tiles_per_split);

// Whether an unsplit product of this shape should run on 64 x 128 tiles: too few 128 x 128 tiles
// for the chip, enough half-height ones, and a reduction (k_steps K steps in all) too short to
// be worth splitting.
bool gemm_tiled_half_tiles(int M, int N, int batch, long k_steps, int BK);

// The two gradients of a MatrixMultiply in half whose rows start anywhere: the operands that cannot be moved in 16-byte pieces are
// copied to rows that can, into the workspace, where that is expected to pay (one launch, a matrix that both read once), and
// the products run on the copies, in one launch (*shared) or one after the other.  False, with nothing launched, where it does not
// pay or the copies do not fit beside the partial sums.
struct PackedProduct {
    GemmArgs *g;
    int ta, tb;
};
bool gemm_pack_run(int dtype, const PackedProduct (&p)[2], void *workspace, size_t workspace_bytes, hipStream_t stream, SharedLaunch *shared, int *rc);
size_t gemm_pack_bytes(int dtype, const PackedProduct (&p)[2]);  // what it takes of the workspace (0: it does not pay)
// The same for a forward product by itself (bias and ReLu included: the caller has checked gemm_fuses_store).
bool gemm_pack_run_one(int dtype, const PackedProduct &p, void *workspace, size_t workspace_bytes, hipStream_t stream, int *rc);
size_t gemm_pack_one_bytes(int dtype, const PackedProduct &p);

// Plan the split of the reduction, launch the tiled kernel (which must be eligible) and reduce.
int gemm_tiled_run(int dtype, GemmArgs &g, int transA, int transB, void *workspace, size_t workspace_bytes,
                   hipStream_t stream);
// The two gradients of a convolution (gx: patch rows as A, NN, into the input's gradient; gy: patch k-rows as B, TN,
// into the filter's) as one launch where that pays; false, with nothing launched, where it does not (the caller then
// runs them one after the other).  The workspace is gy's.
bool gemm_tiled_run_pair(int dtype, GemmArgs &gx, GemmArgs &gy, void *workspace, size_t workspace_bytes, hipStream_t stream, int *rc);
// The two gradients of a MatrixMultiply (g0 = dZ . Y^T, NT; g1 = X^T . dZ, TN; both on the tiled kernels, their operands in whole pieces or
// copies) as one launch plus their split reductions, whatever K leaves of a last step and, but for pairs that leave a tail
// behind, however many workgroups there are; APART, with nothing launched, otherwise.  The workspace holds both products' partial
// sums side by side.
SharedLaunch gemm_tiled_run_plain_pair(int dtype, GemmArgs &g0, int ta0, int tb0, GemmArgs &g1, int ta1, int tb1, void *workspace,
                               size_t workspace_bytes, hipStream_t stream, int *rc);
// Microseconds that a product is expected to take with all the workspace it asks for (which of two ways a convolution goes).
double gemm_estimate_us(int dtype, const GemmArgs &g, int transA, int transB);
// Workspace gemm_tiled_run may use for this shape.
size_t gemm_tiled_workspace(int dtype, int M, int N, int K, int red, int virt = VIRT_NONE);
// Whether a product whose B is a patch matrix (VIRT_B_KROWS) runs on 64 x 64 tiles: fewer than 128 rows, and the last
// 128-column tile would be half empty or emptier (a 3 x 3 x 64 filter gradient: N = 576 = 4.5 x 128).
inline bool gemm_tiled_krows_64(int virt, int M, int N) { return virt == VIRT_B_KROWS && M < 128 && N % 128 != 0 && N % 128 <= 64; }

}  // namespace d8

#endif
