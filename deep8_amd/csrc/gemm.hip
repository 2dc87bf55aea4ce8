// Row-major GEMM for gfx950 on MFMA: C_b = op(A_b) op(B_b) + beta C_b, fp32 and fp16 (fp32
// accumulate), NN / NT / TN, strided batch with broadcast operands, optional summation of the
// whole batch into one C, and a deterministic split of the reduction through a workspace.
//
// Replaces the cuBLAS calls of deep8/src/math/MatrixMultiply.cu, Conv2d.cu and DeConv2d.cu
// (call sites listed in include/deep8_hip.h).
//
// MFMA operand layouts used throughout (wave64):
//   v_mfma_f32_32x32x16_f16 : lane l supplies A[row l%32][8 consecutive k of group l/32] and
//                             B[8 consecutive k of group l/32][col l%32]
//   v_mfma_f32_32x32x2_f32  : lane l supplies A[row l%32][k = l/32], B[k = l/32][col l%32]
//   accumulator register r of lane l is C[8*(r/4) + 4*(l/32) + r%4][l%32]
// Both LDS tiles are kept K-contiguous ([row][k]), so one 16-byte LDS read feeds an MFMA
// operand; the transposed-operand cases differ only in how the tile loader walks global memory.
#include <atomic>
#include <cmath>
#include <type_traits>

#include "gemm_args.h"

namespace d8 {

template <typename T>
struct Tile;
template <>
struct Tile<f16> {
    static constexpr int BK = 32, LD = 40;
};
template <>
struct Tile<float> {
    static constexpr int BK = 16, LD = 20;
};

__device__ inline float to_f32(float v) { return v; }
__device__ inline float to_f32(f16 v) { return (float)v; }

// One wave multiplies its (TM*32) x (TN*32) sub-tile over one K tile held in LDS.
template <int TM, int TN, int LD, int BK>
__device__ inline void wave_mma(const f16 *As, const f16 *Bs, int arow, int brow, int lane,
                                f32x16 (&acc)[TM][TN]) {
    const int l32 = lane & 31, kg = (lane >> 5) * 8;
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
        f16x8 a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = *(const f16x8 *)&As[(arow + i * 32 + l32) * LD + kk + kg];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = *(const f16x8 *)&Bs[(brow + j * 32 + l32) * LD + kk + kg];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
}

// fp32: an 8-wide K chunk is read as two float4 per operand row (lanes 0-31 take k 0..3,
// lanes 32-63 take k 4..7); MFMA q of the chunk then pairs k = q with k = 4 + q.  A and B use
// the same assignment, so every k is multiplied exactly once.
template <int TM, int TN, int LD, int BK>
__device__ inline void wave_mma(const float *As, const float *Bs, int arow, int brow, int lane,
                                f32x16 (&acc)[TM][TN]) {
    const int l32 = lane & 31, kg = (lane >> 5) * 4;
#pragma unroll
    for (int kk = 0; kk < BK; kk += 8) {
        f32x4 a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = *(const f32x4 *)&As[(arow + i * 32 + l32) * LD + kk + kg];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = *(const f32x4 *)&Bs[(brow + j * 32 + l32) * LD + kk + kg];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][q], b[j][q], acc[i][j], 0, 0, 0);
    }
}

// ------------------------------------------------------------------------------------------
// General kernel: what the tiled kernels refuse -- operands of 2 GiB and more, sums over half matrices that lie an odd
// number of elements apart, short reductions over many tiles of rows that start anywhere (see gemm_tiled.hip).  128 x 128 tile, 4 waves in a
// 2 x 2 arrangement, 64 x 64 per wave; element-wise, bounds-checked tile loads.
// ------------------------------------------------------------------------------------------
template <typename T, bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm_general_kernel(GemmArgs g) {
    constexpr int BM = 128, BN = 128, BK = Tile<T>::BK, LD = Tile<T>::LD;
    __shared__ __attribute__((aligned(16))) T As[2][BM * LD];
    __shared__ __attribute__((aligned(16))) T Bs[2][BN * LD];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int b = blockIdx.z / g.splits, s = blockIdx.z % g.splits;

    const int ktiles = (g.K + BK - 1) / BK;
    const int total = g.red * ktiles;
    const int t0 = s * g.tiles_per_split;
    const int t1 = min(total, t0 + g.tiles_per_split);

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // A thread moves NE elements of each operand per K step; element u is tile element tid + 256 u.  Stored
    // along K (A not transposed, B transposed): k = tid % BK for every u, row tid / BK + u * (256 / BK); stored
    // K-row-major: row or column tid % 128, k = tid / 128 + 2 u.  The next step's elements are fetched into
    // registers before the current step is multiplied and written to the other LDS half after it.
    constexpr int NE = BM * BK / 256;
    static_assert(BM == BN && 256 % BK == 0 && BM == 128, "element map");
    const int kc_k = tid % BK, kc_row = tid / BK, tr_col = tid % 128, tr_k = tid / 128;
    const bool a_in = TA ? m0 + tr_col < g.M : true, b_in = TB ? true : n0 + tr_col < g.N;
    T pa[NE], pb[NE];
    auto fetch = [&](int t) {
        const int r = t / ktiles, k0 = (t - r * ktiles) * BK;
        const T *Ap = (const T *)g.A + (long)(b + r) * g.sA;
        const T *Bp = (const T *)g.B + (long)(b + r) * g.sB;
#pragma unroll
        for (int u = 0; u < NE; ++u) {
            pa[u] = (T)0;
            if (TA) {
                const int gk = k0 + tr_k + 2 * u;
                if (a_in && gk < g.K) pa[u] = Ap[(long)gk * g.lda + m0 + tr_col];
            } else {
                const int gm = m0 + kc_row + u * (256 / BK);
                if (gm < g.M && k0 + kc_k < g.K) pa[u] = Ap[(long)gm * g.lda + k0 + kc_k];
            }
        }
#pragma unroll
        for (int u = 0; u < NE; ++u) {
            pb[u] = (T)0;
            if (TB) {
                const int gn = n0 + kc_row + u * (256 / BK);
                if (gn < g.N && k0 + kc_k < g.K) pb[u] = Bp[(long)gn * g.ldb + k0 + kc_k];
            } else {
                const int gk = k0 + tr_k + 2 * u;
                if (b_in && gk < g.K) pb[u] = Bp[(long)gk * g.ldb + n0 + tr_col];
            }
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int u = 0; u < NE; ++u) {
            if (TA) As[buf][tr_col * LD + tr_k + 2 * u] = pa[u];
            else As[buf][(kc_row + u * (256 / BK)) * LD + kc_k] = pa[u];
            if (TB) Bs[buf][(kc_row + u * (256 / BK)) * LD + kc_k] = pb[u];
            else Bs[buf][tr_col * LD + tr_k + 2 * u] = pb[u];
        }
    };

    if (t0 < t1) {
        fetch(t0);
        stage(0);
    }
    __syncthreads();
    for (int t = t0; t < t1; ++t) {
        const int cur = (t - t0) & 1;
        const bool more = t + 1 < t1;
        if (more) fetch(t + 1);
        wave_mma<2, 2, LD, BK>(As[cur], Bs[cur], wm * 64, wn * 64, lane, acc);
        if (more) stage(cur ^ 1);  // nobody reads that half before the barrier below
        __syncthreads();
    }

    const int l32 = lane & 31, lhi = lane >> 5;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn * 64 + j * 32 + l32;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm * 64 + i * 32 + (r >> 2) * 8 + lhi * 4 + (r & 3);
                if (m < g.M && n < g.N) {
                    if (g.splits == 1) {
                        T *c = (T *)g.C + (long)b * g.sC + (long)m * g.ldc + n;
                        float v = acc[i][j][r];
                        if (g.beta != 0.f) v += to_f32(*c);
                        *c = (T)v;
                    } else {
                        g.ws[((long)(b * g.splits + s) * g.M + m) * g.N + n] = acc[i][j][r];
                    }
                }
            }
        }
}

// Where element (m, n) of an output lives (GemmArgs::perm_OC: a filter gradient stored transposed per tap).
__device__ inline long c_index(const GemmArgs &g, int m, int n) {
    if (g.perm_OC) {
        const int t = n / g.perm_OC, oc = n - t * g.perm_OC;
        return ((long)oc * g.perm_T + t) * g.ldc + m;
    }
    return (long)m * g.ldc + n;
}

// ------------------------------------------------------------------------------------------
// Small products: a handful of 128 x 128 tiles would leave the chip to a few workgroups, each
// walking its whole reduction at one MFMA per 64 (fp32) cycles behind one load latency per K step.
// Here a workgroup owns a 32 x 32 tile of C and its eight waves take every eighth chunk of the
// reduction each (8 k values for fp32, 16 for fp16: one MFMA operand per lane).  A lane fetches
// its operand values of ALL its chunks straight from global memory into registers before the
// first MFMA, so the whole product costs one load latency: no branch lies between the loads (an
// index past the matrix is clamped and the value replaced by zero) and no division (unless products
// are summed).  The eight partial tiles meet in LDS in wave order, every wave adding up and storing
// an eighth, so the result does not depend on scheduling.  Any M, N, K, leading dimension and alignment.
// fp32 64 x 128 x 256: forward 6.3 -> 3.8 us, both gradients 7.4 -> 5.4 us (four waves, each value behind a bounds check of its
// own before); an empty kernel takes 1.3 us.
// ------------------------------------------------------------------------------------------
template <typename T>
struct SmallOp;
template <>
struct SmallOp<float> {
    static constexpr int PER = 4, KG = 8;  // values per lane and chunk, k per chunk
    typedef f32x4 Frag;
    __device__ static void mma(const Frag &a, const Frag &b, f32x16 &acc) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], acc, 0, 0, 0);
    }
};
template <>
struct SmallOp<f16> {
    static constexpr int PER = 8, KG = 16;
    typedef f16x8 Frag;
    __device__ static void mma(const Frag &a, const Frag &b, f32x16 &acc) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
    }
};
enum { SMALL_WAVES = 8, SMALL_MAXC = 8 };  // chunks per wave: gemm_is_small admits 64 in all
typedef float SmallParts[SMALL_WAVES][32 * 32];

// One operand's values of a chunk, PER consecutive k of row (column) `line`, as they lie in memory (VEC: in one load; K and
// with it every piece are then multiples of PER) ...
template <typename T, bool KC, bool VEC, typename Index>
__device__ __forceinline__ void small_fetch(T (&v)[SmallOp<T>::PER], const T *p, int ld, int line, int k0, int K) {
    constexpr int PER = SmallOp<T>::PER;
    if constexpr (VEC) {
        *(typename SmallOp<T>::Frag *)v = *(const typename SmallOp<T>::Frag *)(p + (Index)line * (Index)ld + (Index)min(k0, K - PER));
    } else {
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int k = min(k0 + e, K - 1);
            v[e] = p[KC ? (Index)line * (Index)ld + (Index)k : (Index)k * (Index)ld + (Index)line];
        }
    }
}
// ... and with zeros past K, once all loads are under way
template <typename T>
__device__ __forceinline__ typename SmallOp<T>::Frag small_cut(const T (&v)[SmallOp<T>::PER], int k0, int K) {
    typename SmallOp<T>::Frag f;
#pragma unroll
    for (int e = 0; e < SmallOp<T>::PER; ++e) f[e] = k0 + e < K ? v[e] : (T)0;
    return f;
}

template <typename T, bool TA, bool TB, bool VECA, bool VECB, typename Index>
__device__ __forceinline__ void small_multiply(const GemmArgs &g, int gm, int gn, int b, int wave, int lhi, f32x16 &acc) {
    typedef SmallOp<T> OP;
    constexpr int PER = OP::PER, KG = OP::KG;
    const int kchunks = (g.K + KG - 1) / KG, total = g.red * kchunks;
    const int lm = min(gm, g.M - 1), ln = min(gn, g.N - 1);  // (rows and columns past the matrix: results that are not stored)
    T va[SMALL_MAXC][PER], vb[SMALL_MAXC][PER];
    int k0[SMALL_MAXC];
#pragma unroll
    for (int c = 0; c < SMALL_MAXC; ++c) {
        const int t = wave + SMALL_WAVES * c;
        k0[c] = 0;
        if (t < total) {
            const int r = g.red == 1 ? 0 : t / kchunks;
            k0[c] = (t - r * kchunks) * KG + lhi * PER;
            small_fetch<T, !TA, VECA, Index>(va[c], (const T *)g.A + (long)(b + r) * g.sA, g.lda, lm, k0[c], g.K);
            small_fetch<T, TB, VECB, Index>(vb[c], (const T *)g.B + (long)(b + r) * g.sB, g.ldb, ln, k0[c], g.K);
        }
    }
#pragma unroll
    for (int c = 0; c < SMALL_MAXC; ++c)
        if (wave + SMALL_WAVES * c < total) OP::mma(small_cut<T>(va[c], k0[c], g.K), small_cut<T>(vb[c], k0[c], g.K), acc);
}

// (the work of workgroup (bx, by) of output b)
template <typename T, bool TA, bool TB>
__device__ __forceinline__ void gemm_small_body(const GemmArgs &g, const int bx, const int by, const int b, SmallParts &part) {
    constexpr int BT = 32;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lhi = lane >> 5;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const int gm = by * BT + l32, gn = bx * BT + l32;
    constexpr int PER = SmallOp<T>::PER;
    const bool vec_a = !TA && g.lda % PER == 0 && g.sA % PER == 0 && g.K % PER == 0 && ((size_t)g.A & 15) == 0;
    const bool vec_b = TB && g.ldb % PER == 0 && g.sB % PER == 0 && g.K % PER == 0 && ((size_t)g.B & 15) == 0;
    // (32-bit offsets where both operands allow them)
    if ((long)(TA ? g.K : g.M) * g.lda * (long)sizeof(T) >= (1L << 31) || (long)(TB ? g.N : g.K) * g.ldb * (long)sizeof(T) >= (1L << 31))
        small_multiply<T, TA, TB, false, false, long>(g, gm, gn, b, wave, lhi, acc);
    else if ((TA || vec_a) && (!TB || vec_b))
        small_multiply<T, TA, TB, !TA, TB, unsigned>(g, gm, gn, b, wave, lhi, acc);
    else
        small_multiply<T, TA, TB, false, false, unsigned>(g, gm, gn, b, wave, lhi, acc);
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][((r >> 2) * 8 + lhi * 4 + (r & 3)) * BT + l32] = acc[r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < BT * BT / (SMALL_WAVES * 64); ++i) {
        const int e = tid + i * (SMALL_WAVES * 64), m = by * BT + e / BT, gn = bx * BT + e % BT;
        float v = part[0][e];
#pragma unroll
        for (int w = 1; w < SMALL_WAVES; ++w) v += part[w][e];
        if (m < g.M && gn < g.N) {
            T *c = (T *)g.C + (long)b * g.sC + (long)m * g.ldc + gn;
            if (g.beta != 0.f) v += to_f32(*c);
            if (g.bias) v = (g.round_first ? to_f32((T)v) : v) + to_f32(((const T *)g.bias)[gn]);
            *c = (T)(g.relu && !(v > 0.f) ? 0.f : v);
        }
    }
}

template <typename T, bool TA, bool TB>
__global__ __launch_bounds__(SMALL_WAVES * 64) void gemm_small_kernel(GemmArgs g) {
    __shared__ SmallParts part;
    gemm_small_body<T, TA, TB>(g, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, part);
}

// Two small products in one launch: the first n0 = nx0 * ny0 * batch workgroups are g0's grid (NT: the gradient of
// a MatrixMultiply's first input), the rest g1's (TN: the gradient of its second).  Each of them is one load
// latency and a few matrix instructions long; what a launch of its own costs on top is most of its time.
template <typename T>
__global__ __launch_bounds__(SMALL_WAVES * 64) void gemm_small_pair_kernel(GemmArgs g0, GemmArgs g1, int nx0, int ny0, int n0, int nx1, int ny1) {
    __shared__ SmallParts part;
    const bool first = (int)blockIdx.x < n0;
    const GemmArgs &g = first ? g0 : g1;
    const int nx = first ? nx0 : nx1, ny = first ? ny0 : ny1;
    int tile, bx;
    const int b = Divisor(nx * ny, g.by.tiles).div((int)blockIdx.x - (first ? 0 : n0), tile), by = Divisor(nx, g.by.nbx).div(tile, bx);
    if (first) gemm_small_body<T, false, true>(g0, bx, by, b, part);
    else gemm_small_body<T, true, false>(g1, bx, by, b, part);
}

// Whether a product is small in the sense above: at most four 128 x 128 tiles of output and a reduction of
// at most 512 (summed products included) in at most 64 chunks of 8.
static bool gemm_is_small(int M, int N, int K, int batch, int red) {
    return (long)ceil_div(M, 128) * ceil_div(N, 128) * batch <= 4 && (long)K * red <= 512 && (long)red * ceil_div(K, 8) <= 64 &&
           batch * 1L < 65536;
}

// Larger outputs of as short a reduction: what the kernel can hold, on as many workgroups as run at once, and no longer reductions on many of
// them than 400 elements a compute unit.  Beyond that the loads of a 32 x 32 tile, which a larger one would share, take longer than the
// way from memory that all of them wait for once.  In half up to 128 rows of a wider output have 240: the second operand is most of what is read,
// in half cache lines that no other row of tiles asks for meanwhile.  And rows that start anywhere have no line, because the larger tiles
// have no whole pieces to load there.  us, tiled / so, by workgroups; 570 drawn forward products, three sets of tensors in turn:
// fp32 64 x 200 x 640 (40) 7.8 / 4.5, 2824 x 272 x 64 (178) 9.0 / 5.2, 3 x 192 x 192 x 704 (396) 7.2 / 6.3, 13 x 112 x 496 x 152 (260) 11.4 / 12.9, 11 x
// 128 x 352 x 208 (308) 9.0 / 10.1, 28 x 225 x 192 x 128 (896) 7.8 / 10.7; half 64 x 352 x 896 (56) 5.1 / 4.2, 3520 x 576 x 46 (220) 11.8 / 5.3, 10 x 104 x
// 736 x 176 (240) 6.1 / 7.9, 720 x 896 x 304 (230) 6.1 / 7.0, 3 x 968 x 200 x 72 (279) 4.5 / 5.6.  Workgroups times elements: up to 60000 all faster,
// 1.3 to 1.6 times at the mean; up to 100000 half 1.3, fp32 1.4; up to 120000 half 1.10; beyond half 0.92 to 1.01, fp32 on more workgroups than
// compute units 1.02 (on at most as many 1.3).  Replayed from a graph, where launches do not count, up to 60000 and 102000: fp32 1.25 and 1.13, half 1.07 and
// 1.03, half rows that start anywhere 1.5 and 1.4.  Half, up to 128 rows, 61000 to 102000: 41 of them 0.98 (64 x 832 x 1920 6.4 / 7.5, 64 x 488 x 3176 5.7 /
// 6.7), other shapes 1.05.  Half rows that start anywhere, from 102000 on: 19 of them 1.14 (43 x 64 x 704 x 34 9.0 / 5.2).
static bool gemm_fits_small(int dtype, const GemmArgs &g) {
    const int KG = dtype == D8_FLOAT16 ? SmallOp<f16>::KG : SmallOp<float>::KG;
    return dtype != D8_FLOAT64 && g.virt == VIRT_NONE && !g.packed && !g.perm_OC && g.K >= 1 && (long)g.red * ceil_div(g.K, KG) <= SMALL_WAVES * SMALL_MAXC;
}
static long small_workgroups(const GemmArgs &g) { return (long)ceil_div(g.M, 32) * ceil_div(g.N, 32) * g.batch; }
// (products of rows by rows only: a gradient, which may share a launch, has a rule for the two of them, gemm_gradients_are_small)
static bool gemm_is_short(int dtype, const GemmArgs &g) {
    if (!gemm_fits_small(dtype, g)) return false;
    const long cus = cu_count(), n = small_workgroups(g), most = 400 * cus / ((long)g.red * g.K);
    if (dtype == D8_FLOAT32) return n <= cus || (n <= cus * 3 / 2 && n <= most);
    return n <= cus && (n <= (g.M <= 128 && g.N > 64 ? most * 3 / 5 : most) || !gemm_tiled_eligible(dtype, g, 0, 0, TILED_PIECES));
}

// C[b][m][n] = beta * C + sum_s ws[b][s][m][n].  A workgroup covers groups of 4 consecutive outputs.
// Few pieces of many groups (LANES = 1): 256 groups, a thread adds all pieces of its group in order.  Else (LANES = 8): 32 groups, 8 thread rows each add every 8th piece, and the 8 sums meet in
// LDS in a fixed order.  Either way the result does not depend on scheduling, and up to 8 pieces
// it is the same.  Five pieces of 12544 x 32: 4.9 -> 4.0 us, four of 1024 x 1001 in half: 7.1 -> 5.4 us (3 us of which is
// what any launch behind one that wrote a lot takes).  The groups count through an output's elements
// whatever the length of its rows: with rows of an odd length a group starts at any 4-byte aligned address (which is what
// a 16-byte load needs) and may go on in the next row.  An output a thread, as rows of an odd length had it first, took
// 17.3 us for four partial sums of 1024 x 1001, this takes 8.0 us.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// Which of the two: a thread per group only where that alone gives three of four compute units a workgroup, and never where the
// output is stored transposed per tap (four scattered stores a thread).  Whole calls, a thread per group and eight, two to
// eight pieces: up to 147456 outputs level with two or four pieces and 0.1 - 0.8 us slower with others, 235520 level,
// 327680 0.3 - 0.5 us faster, 512512 up to 1.5; transposed 0 - 2.6 us slower from 65536 outputs to 1048576 (filter gradient of
// half DeConv2d 32 x 7x7x256 -> 64, 4x4 stride 2 15.4 and 12.9, of fp32 16 x 8x8x256 -> 64, 4x4 23.5 and 21.3).
__host__ __device__ static inline int reduce_lanes(const GemmArgs &g) {
    return g.splits <= 8 && !g.perm_OC && (long)g.M * g.N * g.batch > 3 * 256 * 256L ? 1 : 8;
}

// (ROWS: the rows are multiples of 4, so a group lies in one row and may be stored at once)
//
// Bound by latencies: the way of its loads from memory, and what is computed before them.  Up to eight pieces of a thread are in
// flight at once, with the old C and the bias beside them, and an output is found by 32-bit multiplications (a product that is
// cut has fewer tiles than the chip has compute units, so outputs and bytes of all pieces are far below 2^31).  Four in flight,
// the rest one by one, and 64-bit divisions before: filter gradient of half Conv2d 32 x 14x14x256 3x3 5.1 -> 4.1 us, of 16 x
// 57x57x96 -> 160 4.7 -> 4.1.  The loads are buffer loads because pieces past the last are zeros then without a branch: behind
// branches of their own they took 88 registers instead of 58 where two products share the pass, and 8.7 us became 23.
template <typename T, bool ROWS, int LANES>
__device__ __forceinline__ void gemm_split_reduce_body(const GemmArgs &g, const int block, f32x4 (*part)[32]) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    const int mn = g.M * g.N, groups = ROWS ? mn / 4 : (mn + 3) / 4;
    constexpr int GROUPS = 256 / LANES;
    const int lane = threadIdx.x % GROUPS, row = threadIdx.x / GROUPS;
    const int id = block * GROUPS + lane;  // this thread's group of 4 outputs
    const bool live = id < groups * g.batch;
    int b = 0, n, r = id;
    if (g.batch > 1) b = Divisor(groups, g.by.groups).div(id, r);
    r *= 4;
    int m = Divisor(g.N, g.by.row).div(r, n);
    const int n_out = ROWS || mn - r >= 4 ? 4 : mn - r;
    T *const c0 = (T *)g.C + (long)b * g.sC;
    const bool whole = ROWS && !g.perm_OC && g.ldc % 4 == 0 && (((size_t)c0 | (size_t)g.bias) & (4 * sizeof(T) - 1)) == 0;
    T4 *const c = (T4 *)(c0 + (long)m * g.ldc + n);
    T4 old = {}, bias = {};
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    const bool tiny = !ROWS && mn < 4;
    if (live && whole && row == 0) {
        if (g.beta != 0.f) old = *c;
        if (g.bias) bias = *(const T4 *)((const T *)g.bias + n);
    }
    if (!tiny) {
        // (a last group of fewer than 4 is loaded with the outputs before it and moved down.  Pieces past the last and groups past
        // the last are fetched at an offset outside the buffer, as zeros: no load lies behind a branch)
        const int back = ROWS || !live ? 0 : 4 - n_out;
        const unsigned bytes = (unsigned)(g.splits * g.batch) * (unsigned)mn * 4u, step = (unsigned)(LANES * mn) * 4u;
        const __amdgpu_buffer_rsrc_t ws = __builtin_amdgcn_make_buffer_rsrc(g.ws, 0, (int)bytes, 0x00020000);
        const unsigned at = live ? (unsigned)((b * g.splits + row) * mn + r - back) * 4u : 0x80000000u;
        auto add = [&](auto in_flight, int s) {  // pieces s + row, s + row + LANES ...
            constexpr int N = decltype(in_flight)::value;
            u32x4 t[N];
#pragma unroll
            for (int u = 0; u < N; ++u)
                t[u] = __builtin_amdgcn_raw_buffer_load_b128(ws, row + s + u * LANES < g.splits ? at : 0x80000000u, (s / LANES + u) * step, 0);
#pragma unroll
            for (int u = 0; u < N; ++u) v += __builtin_bit_cast(f32x4, t[u]);
        };
        int s = 0;
        for (; g.splits - s > 4 * LANES; s += 8 * LANES) add(std::integral_constant<int, 8>(), s);
        if (g.splits - s > 2 * LANES) add(std::integral_constant<int, 4>(), s);
        else if (g.splits - s > 0) add(std::integral_constant<int, 2>(), s);
        if constexpr (!ROWS)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (k < back) v = (f32x4){v[1], v[2], v[3], 0.f};
    } else if (live) {  // an output of fewer than 4 in all
        const float *p = g.ws + (long)b * g.splits * mn;
        for (int s = row; s < g.splits; s += LANES)
            for (int k = 0; k < n_out; ++k) v[k] += p[(long)s * mn + k];
    }
    if constexpr (LANES > 1) {
        part[row][lane] = v;
        __syncthreads();
    }
    if (row == 0 && live) {
        if constexpr (LANES > 1)
#pragma unroll
            for (int k = 1; k < LANES; ++k) v += part[k][lane];
        auto finish = [&](float o, float old, float bias) {
            if (g.beta != 0.f) o += old;
            if (g.bias) o = (g.round_first ? to_f32((T)o) : o) + bias;
            return (T)(g.relu && !(o > 0.f) ? 0.f : o);
        };
        if (whole) {
            T4 out;
#pragma unroll
            for (int k = 0; k < 4; ++k) out[k] = finish(v[k], to_f32(old[k]), to_f32(bias[k]));
            *c = out;
            return;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (ROWS || k < n_out) {
                T *c = c0 + c_index(g, m, n);
                *c = finish(v[k], g.beta != 0.f ? to_f32(*c) : 0.f, g.bias ? to_f32(((const T *)g.bias)[n]) : 0.f);
            }
            if (++n == g.N && !ROWS) n = 0, ++m;
        }
    }
}

template <typename T, bool ROWS, int LANES>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(GemmArgs g) {
    __shared__ f32x4 part[8][32];
    gemm_split_reduce_body<T, ROWS, LANES>(g, (int)blockIdx.x, part);
}

// The reductions of two products in one launch: the first blocks0 workgroups are g0's, the rest g1's.
template <typename T>
__global__ __launch_bounds__(256) void gemm_split_reduce_pair_kernel(GemmArgs g0, GemmArgs g1, unsigned blocks0) {
    __shared__ f32x4 part[8][32];
    const bool first = blockIdx.x < blocks0;
    const GemmArgs &g = first ? g0 : g1;
    const int block = (int)(first ? blockIdx.x : blockIdx.x - blocks0);
    if (reduce_lanes(g) == 1) gemm_split_reduce_body<T, true, 1>(g, block, part);
    else gemm_split_reduce_body<T, true, 8>(g, block, part);
}

// ---- planning a product whose 128 x 128 tiles are fewer than the CUs -----------------------------------------
// Three ways to spread it: cut the reduction into s pieces per tile (a second pass adds them up), run it whole on
// 64 x 128 tiles (twice as many workgroups, no second pass), or leave it.  Rules of thumb give a first choice --
// a workgroup or two per CU, pieces of at least 8 K steps -- and a count of steps per CU decides among the
// admitted alternatives, because how the workgroups fall into rounds matters as much as how many there are: a
// CU's share is ceil(workgroups / CUs) pieces of ceil(total / s) steps plus a prologue and an epilogue each, a
// workgroup alone on its CU walks its steps about a tenth slower than two that share one, a half tile's step is
// half a step (0.65 in half precision), and the second pass costs a launch plus the s partial sums read back (at
// some 4 TB/s).  In units of a K step (about 2 us of a CU's time in fp32, 0.5 us in half): prologue + epilogue
// 2.5 / 7, second pass 2 / 14.
// Measured against it: Conv2d 14 x 14 x 256 fp32, 98 tiles over 72 steps, 36 / 48 / 36 / 30 / 36 steps per CU for
// s = 2 .. 6, ran 83.9 / 103.3 / 82.9 / 72.8 / 86.9 us; 7 x 7 x 512, 52 tiles over 144 steps, 146 / 102 / 80.7 / 116 /
// 100 us for s = 2 .. 6; 1024 x 2048 x 2048 fp32 64.9 us on half tiles against 77.4 in two pieces, 1024 x 1024 x 2048
// 63.4 us on (128) half tiles against 43.9 in four pieces.
struct FewTiles {
    long splits;         // pieces per tile (1: unsplit)
    bool half;           // unsplit on 64 x 128 tiles
    bool half_if_whole;  // were it to run unsplit (no workspace for the pieces, say): on 64 x 128 tiles rather than 128 x 128
};

static long piece_limit(long tiles, long total, int cus) {
    // Every piece costs a tile's prologue, a tile of fp32 partial sums written and read back: at least 8 K steps
    // per piece, or 4 where 8 would leave more than half of the CUs without a workgroup.
    long most = total / 8;
    if (most * tiles < cus / 2) most = total / 4;
    if (most > 512) most = 512;
    return most < 1 ? 1 : most;
}

static FewTiles plan_few_tiles(int BK, int M, int N, int batch, long total) {
    const long tiles = (long)ceil_div(M, 128) * ceil_div(N, 128) * batch, cus = cu_count();
    // the rules' choice: at most two workgroups per CU (a third one would run alone, after the rest) ...
    long rule = 2L * cus / tiles;
    // ... one per CU where its pieces are then still 32 K steps or longer: as fast, and half the partial sums (C2b's
    // dY, 512 x 512 over 16 384: 72.8 -> 70.6 us)
    if (M >= 128 && N >= 128 && total / (cus / tiles) >= 32) rule = cus / tiles;
    // (never more than two pieces per CU in all: a long reduction would otherwise be cut ever finer for an ever
    // smaller gain, and the partial sums -- at most 2 x CUs tiles of fp32, 32 MiB -- would grow with it)
    long most = piece_limit(tiles, total, (int)cus);
    if (most > 2 * cus / tiles) most = 2 * cus / tiles;
    if (rule > most) rule = most;
    if (rule < 1) rule = 1;
    const bool half_elems = BK == 64;
    const double ends = half_elems ? 7.0 : 2.5, second = half_elems ? 14.0 : 2.0;
    const double per_split = (double)M * N * batch / (half_elems ? 0.5e6 : 2e6);
    auto cost = [&](long s) {
        const long rounds = (tiles * s + cus - 1) / cus, len = (total + s - 1) / s;
        return rounds * (len * (rounds == 1 ? 1.1 : 1.0) + ends) + (s > 1 ? second + s * per_split : 0.0);
    };
    FewTiles best = {rule, false, false};
    double best_cost = cost(rule) * 0.97;  // the rules' own choice on a tie
    for (long c = 1; c <= most; ++c)
        if (cost(c) < best_cost) best.splits = c, best_cost = cost(c);
    // half tiles: a short reduction over an output that they spread over most of the chip saves the fp32 partial
    // sums, their round trip through memory and the second launch (C5's dX, 98 tiles over 16 steps: 16.8 + 10.9 us
    // in four pieces, 11.3 us whole on 196 half tiles)
    if (M >= 128 && N >= 128 && 4 * tiles >= cus) {
        const long rounds = (2 * tiles + cus - 1) / cus;
        // (a 64 x 128 tile's step against a 128 x 128 tile's: half the MFMAs; 0.65 in half, where the rest of the step weighs more)
        const double c = rounds * ((half_elems ? 0.65 : 0.5) * total * (rounds == 1 ? 1.1 : 1.0) + ends);
        best.half_if_whole = c < cost(1);
        if (c < best_cost) best.splits = 1, best.half = true;
    }
    return best;
}

bool gemm_tiled_half_tiles(int M, int N, int batch, long k_steps, int BK) {
    if (M < 128 || N < 128) return false;
    const long tiles = (long)ceil_div(M, 128) * ceil_div(N, 128) * batch;
    return tiles < cu_count() && plan_few_tiles(BK, M, N, batch, k_steps).half_if_whole;  // (asked of an unsplit product)
}

// How many pieces to cut the reduction into, for a kernel whose K step is BK.  Splitting is only
// worth a second pass when the output alone gives the 256 CUs too few tiles; the long reductions
// this catches are also the ones whose single fp32 accumulation chain would be longest.
static int plan_splits(int BK, int M, int N, int K, int batch, int red, size_t workspace_bytes, int *tiles_per_split, int virt = VIRT_NONE) {
    const bool t64 = gemm_tiled_krows_64(virt, M, N);  // 64 x 64 tiles, 37 KB of LDS each
    const long tiles = t64 ? (long)ceil_div(M, 64) * ceil_div(N, 64) * batch : (long)ceil_div(M, 128) * ceil_div(N, 128) * batch;
    const long total = (long)red * ceil_div(K, BK);
    if (gemm_is_small(M, N, K, batch, red)) {  // runs whole on gemm_small_kernel
        *tiles_per_split = (int)total;
        return 1;
    }
    const int cus = cu_count();
    long splits = 1;
    if (tiles < cus) {
        if (t64) {
            // three of the small tiles per CU (56 / 85 / 113 / 140 pieces on C4's dW: 75.6 / 73.8 / 75.0 / 78.5 us)
            splits = 3L * cus / tiles;
            const long most = piece_limit(tiles, total, cus);
            if (splits > most) splits = most;
        } else {
            const FewTiles plan = plan_few_tiles(BK, M, N, batch, total);
            splits = plan.half ? 1 : plan.splits;  // (half: the tiled kernel asks gemm_tiled_half_tiles itself)
        }
        static const char *force = getenv("D8_GEMM_SPLITS");  // tuning aid
        if (force && splits > 1) splits = atoi(force);
    }
    // no more pieces than the caller's workspace holds
    const size_t per_split = (size_t)batch * M * N * sizeof(float);
    const long fit = (long)(workspace_bytes / per_split);
    if (splits > fit) splits = fit;
    if (splits < 2) splits = 1;
    const long tps = (total + splits - 1) / splits;
    *tiles_per_split = (int)tps;
    return tps > 0 ? (int)((total + tps - 1) / tps) : 1;
}

// ---- rows that start anywhere, copied to rows of whole pieces -------------------------------------------------
struct PackArgs {
    const f16 *src;
    f16 *dst;
    int rows, cols, ld, pitch;  // rows of all matrices that follow each other, `per` of them `stride` elements from the next
    int per;
    unsigned by_per;  // reciprocal_of(per)
    long stride;
    int across;  // as a power of two
    unsigned first;  // workgroup
};
struct PackList {
    PackArgs m[3];
    int n;
};

// Bound by the way to memory and back.  2^across threads (at most 256) lie along a row, a thread copies 16 bytes of ROWS rows before
// it goes on along them, read at the alignment of an element.  A row's last piece is read where it ends with the row and shifted
// into place: element by element it kept the whole workgroup waiting for up to seven loads in a row (4096 x 1001 and 1024 x 1001
// 8.4 -> 6.0 us, 1024 x 1001 alone 6.9 -> 4.5, 888 x 1255 6.7 -> 2.8).  Copied rows start at multiples of 128 bytes, as the K steps of
// the product want them (pitch 1008 instead of 1024: 4096 x 1001 x 1024 loop of the product 9.7 us instead of 8.3).
template <int ROWS>
__global__ __launch_bounds__(256) void pack_rows_kernel(PackList L) {
    typedef f16x8 f16x8_any __attribute__((aligned(2)));
    const int i = L.n > 2 && blockIdx.x >= L.m[2].first ? 2 : L.n > 1 && blockIdx.x >= L.m[1].first ? 1 : 0;
    const PackArgs a = L.m[i];
    const int down = 256 >> a.across, row0 = (int)(blockIdx.x - a.first) * ROWS * down + ((int)threadIdx.x >> a.across);
    const f16 *src[ROWS];
    f16 *const dst = a.dst + (long)row0 * a.pitch;
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
        const int row = min(row0 + u * down, a.rows - 1);  // (rows past the last are read there and not written)
        int m = 0, r = row;
        if (a.per < a.rows) m = Divisor(a.per, a.by_per).div(row, r);
        src[u] = a.src + (long)m * a.stride + (long)r * a.ld;
    }
    const int step = 8 << a.across;
    for (int c = ((int)threadIdx.x & ((1 << a.across) - 1)) * 8; c < a.pitch; c += step) {
        u32x4 v[ROWS];
        const int from = max(min(c, a.cols - 8), 0), left = a.cols - c, shift = c - from;  // elements of the piece that are the row's
#pragma unroll
        for (int u = 0; u < ROWS; ++u) v[u] = __builtin_bit_cast(u32x4, (f16x8)*(const f16x8_any *)(src[u] + from));
        if (left < 8) {
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                u32x4 w = v[u];
                if (shift & 4) w = (u32x4){w[2], w[3], 0u, 0u};
                if (shift & 2) w = (u32x4){w[1], w[2], w[3], 0u};
                if (shift & 1) w = (u32x4){w[0] >> 16 | w[1] << 16, w[1] >> 16 | w[2] << 16, w[2] >> 16 | w[3] << 16, w[3] >> 16};
                v[u] = left > 0 ? w : (u32x4){0u, 0u, 0u, 0u};
            }
        }
#pragma unroll
        for (int u = 0; u < ROWS; ++u)
            if (row0 + u * down < a.rows) *(u32x4 *)(dst + (long)u * down * a.pitch + c) = v[u];
    }
}

// Which operands of a product have to be copied (bit 0: A, bit 1: B): those that cannot be moved in whole pieces, and if K is no
// multiple of a piece all that are stored along K, whose copies end in zeros.
static int pack_operands(const GemmArgs &g, int ta, int tb) {
    auto odd = [](const void *p, int ld, long s, int extent) { return (((size_t)p & 15) || ld % 8 || s % 8 || extent % 8) ? 1 : 0; };
    return odd(g.A, g.lda, g.sA, ta ? g.M : g.K) | odd(g.B, g.ldb, g.sB, tb ? g.K : g.N) << 1;
}

struct PackShape {
    const void *p;
    long rows;
    int cols, ld, per;
    long stride;
};
static PackShape pack_shape(const GemmArgs &g, int ta, int tb, int op) {
    const int count = (op ? g.sB : g.sA) ? g.batch * g.red : 1;
    PackShape s;
    s.p = op ? g.B : g.A;
    s.per = op ? (tb ? g.N : g.K) : (ta ? g.K : g.M), s.cols = op ? (tb ? g.K : g.N) : (ta ? g.M : g.K);
    s.rows = (long)s.per * count, s.ld = op ? g.ldb : g.lda, s.stride = op ? g.sB : g.sA;
    return s;
}
static int pack_pitch(const PackShape &s) { return (s.cols + 63) & ~63; }
static size_t pack_bytes(const PackShape &s) { return (size_t)s.rows * pack_pitch(s) * 2; }  // (a multiple of 128)

// What is to be copied for one product or two: a matrix that is read twice is copied once.
struct PackPlan {
    PackShape shapes[4];
    int n, slot[2][2];
    size_t bytes;
};

// Whether copies pay.  Both gradients: a product saves 0.5 us for each K step that a compute unit walks (0.3 on tiles of 64 columns or rows), or
// 0.25 where both of its operands are odd, and a MB of copies takes 0.2; on copies the two mostly share a launch, which they would not without.  A forward
// product by itself: 0.2 and 0.25 us a step, 0.3 a MB, and a launch for the copies; an output narrower than a tile is bound by its operands' way
// from memory, and a product that fills the chip with tiles of few steps has them hide each other's ways.
// Drawn calls with odd sizes, a third of them batched, three sets of tensors in turn, us on the kernels for rows that start anywhere /
// on copies always / by this rule / with the better of the two, and how many lose more than 3 % to the better one by the rule:
//   691 calls of both gradients   19571 / 15311 / 15516 / 15220, 69 (4 of them to the way without copies, at most 12 %; 0.5 us a step for narrow
//                                 tiles too: 12)
//   330 forward products           5774 / 5491 / 5351 / 5183, 85 (6 lose more than 3 % to the way without copies, at most 10 %)
// Gradients of 3039 x 376 x 2289 52.7 -> 34.8, 6 x 1005 x 368 x 1211 45.1 -> 33.0; forward 4096 x 1024 x 1001 with bias and ReLu 21.1 -> 20.2, 883 x 624 x 334
// 17.1 -> 10.7, 107 x 1440 x 3121 36.2 -> 15.8.
static bool pack_pays(const PackedProduct *p, int products, const PackPlan &plan) {
    const char *force = getenv("D8_GEMM_PACK");  // tuning and test aid (read at every call): 0 never, 1 always
    if (force) return atoi(force) != 0;
    const double cus = cu_count();
    const bool both = products == 2;
    double saved = 0.0, least = both && (plan.slot[0][0] >= 0 || plan.slot[0][1] >= 0) ? 0.2 : 1.0;
    for (int i = 0; i < products; ++i) {
        const GemmArgs &g = *p[i].g;
        const int odd = (plan.slot[i][0] >= 0) + (plan.slot[i][1] >= 0);
        const long tiles = (long)ceil_div(g.M, 128) * ceil_div(g.N, 128) * g.batch, total = (long)g.red * ceil_div(g.K, 64);
        const double share = tiles * total / cus, alone = total < 8 ? total : 8.0;
        const double one = !both ? 0.2 : g.M <= 64 || g.N <= 64 ? 0.3 : 0.5;
        saved += (odd == 2 ? 0.25 : odd == 1 ? one : 0.0) * (share > alone ? share : alone);
        if (!both) {
            if (g.M < 128 || g.N < 128 || (gemm_is_short(D8_FLOAT16, g) && (long)g.red * g.K <= 512)) return false;
            least = 4 * tiles >= cus && total <= 32 ? 1.7 : 0.2;
        }
    }
    return saved > least + (both ? 0.2e-6 : 0.3e-6) * plan.bytes;
}

// (products on the tiled kernels; false: nothing to copy, or not with these)
static bool pack_plan(int dtype, const PackedProduct *p, int products, PackPlan &plan) {
    plan.n = 0, plan.bytes = 0;
    if (dtype != D8_FLOAT16) return false;
    for (int i = 0; i < products; ++i) {
        const GemmArgs &g = *p[i].g;
        if (g.virt != VIRT_NONE || g.K < 1 || g.batch > 448 || g.M > 65535 * 128 || gemm_is_small(g.M, g.N, g.K, g.batch, g.red) ||
            !gemm_tiled_eligible(dtype, g, p[i].ta, p[i].tb)) return false;
        const int ops = pack_operands(g, p[i].ta, p[i].tb);
        for (int op = 0; op < 2; ++op) {
            plan.slot[i][op] = -1;
            if (!(ops >> op & 1)) continue;
            const PackShape s = pack_shape(g, p[i].ta, p[i].tb, op);
            if (pack_bytes(s) >= (1u << 31) || s.cols < 8) return false;  // (byte offsets inside an operand are 32-bit; a row has a piece)
            int k = 0;
            while (k < plan.n && !(plan.shapes[k].p == s.p && plan.shapes[k].rows == s.rows && plan.shapes[k].cols == s.cols &&
                                   plan.shapes[k].ld == s.ld && plan.shapes[k].per == s.per && plan.shapes[k].stride == s.stride)) ++k;
            if (k == plan.n) plan.shapes[plan.n++] = s, plan.bytes += pack_bytes(s);
            plan.slot[i][op] = k;
        }
    }
    return plan.n > 0 && plan.n <= 3;
}

// C = beta * C + the g.splits partial sums in g.ws (+ bias, ReLu)
static long reduce_blocks(const GemmArgs &g, int lanes) {
    const int groups = 256 / lanes;
    return (((long)g.M * g.N + 3) / 4 * g.batch + groups - 1) / groups;
}

static void set_reduce_reciprocals(GemmArgs &g) { g.by.row = reciprocal_of(g.N), g.by.groups = reciprocal_of((g.M * g.N + 3) / 4); }

template <typename T>
static int launch_reduce(const GemmArgs &g0, hipStream_t stream) {
    GemmArgs g = g0;
    set_reduce_reciprocals(g);
    const int lanes = reduce_lanes(g);
    const dim3 grid((unsigned)reduce_blocks(g, lanes));
    if (g.N % 4 == 0 && lanes == 1) hipLaunchKernelGGL((gemm_split_reduce_kernel<T, true, 1>), grid, dim3(256), 0, stream, g);
    else if (g.N % 4 == 0) hipLaunchKernelGGL((gemm_split_reduce_kernel<T, true, 8>), grid, dim3(256), 0, stream, g);
    else if (lanes == 1) hipLaunchKernelGGL((gemm_split_reduce_kernel<T, false, 1>), grid, dim3(256), 0, stream, g);
    else hipLaunchKernelGGL((gemm_split_reduce_kernel<T, false, 8>), grid, dim3(256), 0, stream, g);
    D8_LAUNCH_CHECK();
    return 0;
}

// The reductions that follow a launch of two products (either may be unsplit): one launch for both (whose rows are
// multiples of 4, or they would not have shared the first).
static int launch_reduce_pair(int dtype, const GemmArgs &p0, const GemmArgs &p1, hipStream_t stream) {
    GemmArgs g0 = p0, g1 = p1;
    set_reduce_reciprocals(g0), set_reduce_reciprocals(g1);
    const bool r0 = g0.splits > 1, r1 = g1.splits > 1;
    const long b0 = reduce_blocks(g0, reduce_lanes(g0)), b1 = reduce_blocks(g1, reduce_lanes(g1));
    if (r0 && r1 && g0.N % 4 == 0 && g1.N % 4 == 0 && b0 + b1 < 0x7fffffffL) {
        if (dtype == D8_FLOAT16)
            hipLaunchKernelGGL(gemm_split_reduce_pair_kernel<f16>, dim3((unsigned)(b0 + b1)), dim3(256), 0, stream, g0, g1, (unsigned)b0);
        else
            hipLaunchKernelGGL(gemm_split_reduce_pair_kernel<float>, dim3((unsigned)(b0 + b1)), dim3(256), 0, stream, g0, g1, (unsigned)b0);
        D8_LAUNCH_CHECK();
        return 0;
    }
    if (r0)
        if (int rc = dtype == D8_FLOAT16 ? launch_reduce<f16>(g0, stream) : launch_reduce<float>(g0, stream)) return rc;
    if (r1)
        if (int rc = dtype == D8_FLOAT16 ? launch_reduce<f16>(g1, stream) : launch_reduce<float>(g1, stream)) return rc;
    return 0;
}

template <typename T>
static int launch_small(const GemmArgs &g, int transA, int transB, hipStream_t stream) {
    dim3 grid(ceil_div(g.N, 32), ceil_div(g.M, 32), g.batch);
    if (!transA && !transB)
        hipLaunchKernelGGL((gemm_small_kernel<T, false, false>), grid, dim3(SMALL_WAVES * 64), 0, stream, g);
    else if (!transA && transB)
        hipLaunchKernelGGL((gemm_small_kernel<T, false, true>), grid, dim3(SMALL_WAVES * 64), 0, stream, g);
    else
        hipLaunchKernelGGL((gemm_small_kernel<T, true, false>), grid, dim3(SMALL_WAVES * 64), 0, stream, g);
    D8_LAUNCH_CHECK();
    return 0;
}

template <typename T>
static int launch(GemmArgs &g, int transA, int transB, bool tiled, hipStream_t stream) {
    if (g.virt == VIRT_NONE && g.splits == 1 && gemm_is_small(g.M, g.N, g.K, g.batch, g.red)) return launch_small<T>(g, transA, transB, stream);
    if (tiled) {
        if (int rc = gemm_tiled_launch(sizeof(T) == 2 ? D8_FLOAT16 : D8_FLOAT32, g, transA, transB, stream)) return rc;
    } else {
        dim3 grid(ceil_div(g.N, 128), ceil_div(g.M, 128), g.batch * g.splits);
        if (!transA && !transB)
            hipLaunchKernelGGL((gemm_general_kernel<T, false, false>), grid, dim3(256), 0, stream, g);
        else if (!transA && transB)
            hipLaunchKernelGGL((gemm_general_kernel<T, false, true>), grid, dim3(256), 0, stream, g);
        else
            hipLaunchKernelGGL((gemm_general_kernel<T, true, false>), grid, dim3(256), 0, stream, g);
        D8_LAUNCH_CHECK();
    }
    return g.splits > 1 ? launch_reduce<T>(g, stream) : 0;
}

// A tall product whose output is one column of 128-row tiles (a convolution with up to 127 output
// channels: M = images x pixels) rarely gives every CU the same number of tiles: 784 tiles on 256
// CUs run as long as 1024 would.  Such a product is cut in two along M: the rows that fill whole
// rounds of the chip run unsplit, the remaining band of rows runs as a second product whose
// reduction is split so that it, too, occupies the whole chip for a fraction of a tile's time.
// Returns the rows of the first part (0: do not cut).
static int balanced_rows(const GemmArgs &g) {
    if (g.batch != 1 || g.N >= 128 || g.M < 128 || g.virt == VIRT_B_KROWS) return 0;
    const long tiles = ceil_div(g.M, 128), cus = cu_count();
    const long rest = tiles % cus;
    if (tiles < cus || rest == 0 || rest * 2 > cus) return 0;
    return (int)((tiles - rest) * 128);
}

// Pieces of a remainder band whose workgroups ride in the launch of the rows before it: they start as that launch's
// first tiles retire and cost neither a launch nor a tile's prologue on an idle chip, so they may be short -- about one
// piece per CU, two K steps at least (C4's band of 16 tiles over 18 steps: 4 / 6 / 9 pieces per tile gave
// 0.2105 / 0.2065 / 0.2060 ms per Conv2d step, 18 pieces 0.2147).  0: the band does not ride along.
static int plan_band_pieces(int BK, int rows, int N, int K, int red, size_t workspace_bytes, int *tiles_per_split) {
    if (rows < 128) return 0;
    const long total = (long)red * ceil_div(K, BK), tiles = (long)ceil_div(rows, 128) * ceil_div(N, 128);
    long tps = ceil_div(total, (long)ceil_div((long)cu_count(), tiles));
    if (tps < 2) tps = 2;
    long splits = ceil_div(total, tps);
    const long fit = (long)(workspace_bytes / ((size_t)rows * N * sizeof(float)));
    if (splits > fit) splits = fit;
    if (splits < 2) return 0;
    tps = ceil_div(total, splits);
    *tiles_per_split = (int)tps;
    return (int)ceil_div(total, tps);
}

size_t gemm_tiled_workspace(int dtype, int M, int N, int K, int red, int virt) {
    int tps = 0;
    GemmArgs probe;
    memset(&probe, 0, sizeof(probe));
    probe.M = M, probe.N = N, probe.K = K, probe.batch = 1, probe.red = red;
    const int head = balanced_rows(probe);
    const int rows = head ? M - head : M;  // with a cut, only the second part is split
    int splits = plan_splits(gemm_tiled_k_step(dtype), rows, N, K, 1, red, (size_t)-1, &tps, virt);
    if (head) {  // (the band may run either way: as pieces of the first part's launch or as a launch of its own)
        const int riding = plan_band_pieces(gemm_tiled_k_step(dtype), rows, N, K, red, (size_t)-1, &tps);
        if (riding > splits) splits = riding;
    }
    return splits > 1 ? (size_t)splits * rows * N * sizeof(float) : 0;
}

// 64 x 64 tiles where the 128-wide ones leave compute units idle.  In fp32, whose K step is bound by the matrix pipe, a step of
// theirs is a quarter of the work; in half, whose step waits longer than it multiplies, half of it (through registers 0.25 us against
// 0.38 for a 64 x 128 tile and 0.46 for 128 x 128).  The same pieces -- or none, and no second pass -- spread over four times as many
// workgroups.  The estimate counts steps of a 128 x 128 tile (about 2 us of a CU in fp32, 0.5 us in half), for the plan that g
// holds (splits set) and for 64 x 64 tiles in 1 .. as many pieces as that plan; 7 % or more decide.  In half it was fitted to tiles
// that pass through registers; most products are decided by half_tile_us.  A 64 x 128 half step is 0.76
// here and 0.65 in plan_few_tiles, a half product's second pass 6.5 steps + 1 per 0.25e6 outputs and piece here, 14 + 1 per 0.5e6
// there, which only chooses among 128-wide tiles.
// A narrow output (128 x 32 tiles, below) counts its pieces the same way.
// NN, us before and after (M x K x N; NT and TN alike): fp32 512 x 512 x 512 16.4 -> 10.2, 784 x 1152 x 128 16.0 -> 10.3,
// 1024 x 1024 x 1024 33.6 -> 23.5, 12544 x 800 x 64 24.0 -> 17.0, 3136 x 576 x 256 24.5 -> 12.7, 1536 x 1536 x 1536
// 76.8 -> 72.5; half 512 x 512 x 512 8.6 -> 5.5, 256 x 1024 x 1024 11.8 -> 7.5, 1024 x 1024 x 1024 9.6 -> 8.2,
// 1600 x 2304 x 256 18.2 -> 12.6 (in pieces 18.7), 300 x 3136 x 256 10.6 -> 9.1 (whole 15.7); left alone, and slower if not:
// 1536 x 1536 x 1536 16.5 (19.8), 1024 x 2048 x 2048 18.2 (19.3).
static double tile_cost(bool half_elems, int bm, int bn, const GemmArgs &g, long total, long s) {
    const long cus = cu_count(), n = (ceil_div(g.M, bm) * (long)ceil_div(g.N, bn) * g.batch * s + cus - 1) / cus, len = (total + s - 1) / s;
    const double area = bm * bn / 16384.0, mn = (double)g.M * g.N * g.batch;
    // (a 64 x 64 half step takes 0.25 us on operands that its XCD's L2 holds and 0.41 on others; of products of 4 MB none had the
    // longer step, of 7 MB half of them, from 14 MB on all.  The longer one counts as 0.36, because the larger tiles' steps take
    // longer as well.  3264 x 4416 x 256 NT 31.4 us whole on 64 x 64 tiles, 22.6 in four pieces on 128 x 128; 256 x 3136 x 2200 TN
    // 25.3 and 18.9; 1472 x 3368 x 416 25.3 and 19.1.  700 drawn products, the same operands again / others each time: 9964 / 10556 us
    // with 0.3 from 16 MB on, 9900 / 10494 so, 9702 / 10290 at best.)
    const double far = (2.0 * g.red * g.K * g.batch * ((double)g.M + g.N) - 4e6) / 8e6;
    if (half_elems) return n * len * (area < 0.3 ? 0.5 + 0.22 * (far < 0.0 ? 0.0 : far > 1.0 ? 1.0 : far) : area < 0.6 ? 0.76 : 1.0) + 7.0 + 0.5 * (n - 1) + (s > 1 ? 6.5 + s * (mn / 0.25e6) : 0.0);
    return n * len * area * (n == 1 ? 1.1 : area < 0.3 ? 1.08 : 1.0) + 0.5 + 2.0 * sqrt(area) + 0.3 * (n - 1) + (s > 1 ? 2.0 + s * (mn / 2e6) : 0.0);
}

// ... in half, in microseconds, of tiles whose operands go straight into LDS: a workgroup's ends, its steps, a further round, what
// patch rows take longer, and a second pass.  Fitted to 80 drawn forward products and convolutions of at most 255 128 x 128 tiles, each on three
// tiles in 1 to 12 pieces; 5 % or more decide.  (The estimate above, which 7 % had to decide, counts the same ends for all
// tiles, and for products of few steps those are most of the time.)  110 drawn half products and convolutions forward 1384 ->
// 1358 us, 3.4 % at the mean: 218 x 64 x 1328 5.6 -> 4.0, 1504 x 3648 x 128 14.6 -> 10.8, Conv2d 37 x 8x8x64 -> 368 1x1 6.2 -> 4.7.
// What a workgroup takes besides its steps, and a step (128 x 128 and 64 x 64 tiles, and the two between).
static double half_ends_us(int bm, int bn) { return bm * bn == 64 * 64 ? 3.6 : 4.1; }
// (operands of more than 4 MB are farther away, for two products at once more so: 4352 x 1152 x 192 8.1 us on 64 x 64 tiles, 10.0 on those that 0.11 chooses,
// 2304 x 2560 x 320 12.1 and 17.0; 1828 drawn forward products and convolutions 18821 -> 18716 us.  43 x 64 x 248 x 512, both gradients, by 0.06 10.1 -> 12.4)
static double half_step_us(int bm, int bn, const GemmArgs &g, bool shared) {
    const double far = bm * bn == 64 * 64 ? (2.0 * g.red * g.K * g.batch * ((double)g.M + g.N) - 4e6) / 8e6 : 0.0;  // (see above)
    return (bm * bn == 128 * 128 ? 0.47 : bm * bn == 64 * 64 ? 0.23 : 0.31) + (shared ? 0.11 : 0.06) * (far < 0.0 ? 0.0 : far > 1.0 ? 1.0 : far);
}
static double half_rows_us(int bm, int bn) { return bm * bn == 128 * 128 ? 1.65 : bm * bn == 64 * 64 ? 0.95 : 1.25; }
static double half_tile_us(int bm, int bn, const GemmArgs &g, long total, long s) {
    const long cus = cu_count(), n = (ceil_div(g.M, bm) * (long)ceil_div(g.N, bn) * g.batch * s + cus - 1) / cus, len = (total + s - 1) / s;
    return half_ends_us(bm, bn) + n * len * half_step_us(bm, bn, g, g.pieces_by == BY_SHARED_TIMES) + 0.2 * (n - 1) + (g.virt == VIRT_A_ROWS ? half_rows_us(bm, bn) : 0.0) +
           (s > 1 ? 2.6 + 1.85e-6 * s * g.M * (double)g.N * g.batch : 0.0);
}

static void few_tiles_small(int dtype, GemmArgs &g, int transA, int transB, size_t usable) {
    // (a filter gradient's pieces stay those of the launch it may share with the input's: one sum, one result)
    if (g.virt == VIRT_A_CLASSES || g.virt == VIRT_B_KROWS || gemm_is_small(g.M, g.N, g.K, g.batch, g.red)) return;
    if ((long)ceil_div(g.M, 128) * ceil_div(g.N, 128) * g.batch >= cu_count()) return;
    const bool half_elems = dtype == D8_FLOAT16;
    // (half rows that start anywhere: a 64 x 64 tile's step takes 0.6 us of the 0.9 of a 128 x 128 one's, so the pieces stay:
    // 1024 x 4096 x 1001 TN 38.9 us whole on small tiles, 21.7 + 5.4 in four pieces)
    if (half_elems && gemm_tiled_loose(dtype, g, transA, transB)) return;
    const int BK = gemm_tiled_k_step(dtype);
    const long total = (long)g.red * ceil_div(g.K, BK);
    const bool half = g.splits == 1 && gemm_tiled_half_tiles(g.M, g.N, g.batch, total, BK);
    const bool narrow = g.tile_hint == HINT_128x32;
    const bool by_time = half_elems && g.pieces_by != BY_STEPS;
    auto cost = [&](int bm, int bn, long pieces) { return by_time ? half_tile_us(bm, bn, g, total, pieces) : tile_cost(half_elems, bm, bn, g, total, pieces); };
    const double now = narrow ? 1e30 : g.N < 128 ? cost(128, 64, g.splits) : cost(g.M < 128 || half ? 64 : 128, 128, g.splits);
    long most = (long)(usable / ((size_t)g.batch * g.M * g.N * sizeof(float)));
    int tps;  // (no more pieces than the 128-wide plan would have: what the scratch queries provide for, whatever is passed)
    const long planned = plan_splits(BK, g.M, g.N, g.K, g.batch, g.red, (size_t)-1, &tps, g.virt);
    if (most > planned) most = planned;
    if (most > total / 2) most = total / 2;
    double best = (by_time ? 0.95 : 0.93) * now;
    long pieces = 0;
    for (long s = 1; s == 1 || s <= most; ++s)
        if (const double c = narrow ? cost(128, 32, s) : cost(64, 64, s); c < best) best = c, pieces = s;
    if (!pieces) return;
    if (!narrow) g.tile_hint = HINT_64x64;
    g.tiles_per_split = (int)((total + pieces - 1) / pieces);
    g.splits = (int)((total + g.tiles_per_split - 1) / g.tiles_per_split);
}

// fp32 outputs of at most 32 columns (an input gradient of few channels): 128 x 32 tiles, because half of a 128 x 64 tile's
// matrix instructions would multiply columns that are not there.  50000 x 288 x 32: 22.0 -> 14.3 us.
static bool narrow_output(int dtype, const GemmArgs &g) {
    return dtype == D8_FLOAT32 && g.N <= 32 && g.M >= 128 && (g.virt == VIRT_NONE || g.virt == VIRT_A_ROWS);
}

static void plan_pieces(int dtype, GemmArgs &g, int ta, int tb, size_t usable) {
    g.splits = plan_splits(gemm_tiled_k_step(dtype), g.M, g.N, g.K, g.batch, g.red, usable, &g.tiles_per_split, g.virt);
    few_tiles_small(dtype, g, ta, tb, usable);
}

// A planned half product as one of two that share a launch.  One that runs whole may take larger tiles than alone, which sum in the same
// order: fewer steps for the chip, where the smaller ones make shorter workgroups.
struct HalfShare {
    // us of a workgroup and of its steps, workgroups, and a compute unit's share of all steps; on its tiles and on larger ones
    double longest[2], steps[2], workgroups[2], share[2];
    double pass;                  // over its partial sums, the launch left out
    bool larger;                  // whether there is the choice
};
static HalfShare half_share(const GemmArgs &g) {
    const long total = (long)g.red * ceil_div(g.K, 64), len = g.splits > 1 ? g.tiles_per_split : total;
    const bool small = g.tile_hint == HINT_64x64 || (g.virt == VIRT_B_KROWS && ((g.M < 128 && g.N < 128) || gemm_tiled_krows_64(g.virt, g.M, g.N)));
    HalfShare h;
    h.larger = g.virt == VIRT_NONE && g.splits == 1 && g.tile_hint == HINT_64x64;
    h.pass = g.splits > 1 ? 1.85e-6 * g.splits * g.M * (double)g.N * g.batch : 0.0;
    for (int i = 0; i < (h.larger ? 2 : 1); ++i) {
        const bool t64 = small && i == 0;
        const int bn = t64 || g.N < 128 ? 64 : 128;
        const int bm = t64 || (bn == 128 && (g.M < 128 || (g.splits == 1 && gemm_tiled_half_tiles(g.M, g.N, g.batch, total, 64)))) ? 64 : 128;
        const double steps = len * half_step_us(bm, bn, g, true);
        const double slow = bm * bn == 128 * 128 ? 1.4 : bm * bn == 64 * 64 ? 1.0 : 1.3;  // (four waves and fewer stages than in a launch alone)
        h.longest[i] = half_ends_us(bm, bn) + slow * steps + (g.virt != VIRT_NONE ? half_rows_us(bm, bn) : 0.0);
        h.steps[i] = steps, h.workgroups[i] = (double)ceil_div(g.M, bm) * ceil_div(g.N, bn) * g.batch * g.splits;
        h.share[i] = h.workgroups[i] * steps / cu_count();
    }
    return h;
}
// What the launch takes with the pass after it: its longest workgroup or a compute unit's share, whichever is more; bit i of tiles: product i on
// larger ones.  Some more workgroups than compute units lie beside a longest one (3 x 2600 x 128 x 2176 29.1 us on 63 + 204 workgroups, 21.7 on 246 + 204).
static double half_pair_us(const HalfShare &a, const HalfShare &b, int &tiles) {
    double best = INFINITY;
    for (int t = 0; t < 4; ++t) {
        const int i = t & 1, j = t >> 1;
        if (i > a.larger || j > b.larger) continue;
        const double rounds = (a.workgroups[i] + b.workgroups[j]) / cu_count(), shorter = a.steps[i] < b.steps[j] ? a.steps[i] : b.steps[j];
        const double longest = (a.longest[i] > b.longest[j] ? a.longest[i] : b.longest[j]) + (rounds > 1.0 && rounds <= 1.5 ? 0.75 * shorter : 0.0);
        const double share = 4.0 + a.share[i] + b.share[j];
        if (const double us = longest > share ? longest : share; us < best) best = us, tiles = t;
    }
    return best + (a.pass + b.pass > 0.0 ? 3.5 + a.pass + b.pass : 0.0);
}

// Plans the two half gradients of a MatrixMultiply for a launch that they share.  Which estimate plans the pieces of each (and of each alone, for
// the same bits: by the shapes only): by its tiles' times a product is cut where that pays in a launch of its own; beside another one that runs
// as long anyway, a second pass comes on top.  Both by the tiles' times and on larger tiles where they run whole, as it was, / so, us: 4 x 320 x
// 128 x 1408 12.6 / 9.0, 960 x 128 x 1872 18.4 / 11.4 (apart 15.2), 3 x 384 x 768 x 264 16.2 / 9.7 (12.8), 4 x 832 x 448 x 160 14.2 / 8.8 (12.1), 1216 x
// 128 x 256 10.3 / 7.7, 1856 x 128 x 3200 14.9 / 14.5 (by its steps 18.4); 500 drawn calls of both gradients 6083 / 5739.
// Within 5 % of each other the tiles' times decide: without that line 34 of 378 drawn calls whose plans differ were more than 3 % slower than by the
// tiles' times alone (more pieces of larger tiles, whose pass takes longer: 4560 x 1216 x 64 15.3 / 16.6, 4056 x 1416 x 64 15.9 / 17.2), with it 16.
static void half_pair_plan(GemmArgs &g0, GemmArgs &g1, size_t usable) {
    GemmArgs *const g[2] = {&g0, &g1};
    HalfShare plan[2][2];
    const int ways[2] = {BY_SHARED_TIMES, BY_STEPS};
    int tiles = 0, choice = 0;
    for (int i = 0; i < 2; ++i)
        for (int k = 0; k < 2; ++k) {
            GemmArgs p = *g[i];
            p.pieces_by = ways[k];
            plan_pieces(D8_FLOAT16, p, i, !i, (size_t)-1);
            plan[i][k] = half_share(p);
        }
    double best = INFINITY;
    for (int c = 0; c < 4; ++c)
        if (const double us = half_pair_us(plan[0][c & 1], plan[1][c >> 1], tiles) * (c ? 1.05 : 1.0); us < best) best = us, choice = c;
    g0.pieces_by = ways[choice & 1], g1.pieces_by = ways[choice >> 1];
    plan_pieces(D8_FLOAT16, g0, 0, 1, usable), plan_pieces(D8_FLOAT16, g1, 1, 0, usable);
    half_pair_us(half_share(g0), half_share(g1), tiles);
    for (int i = 0; i < 2; ++i)
        if (tiles >> i & 1) g[i]->tile_hint = HINT_NONE;
}

// (Conv2d 2 x 19x19x64 -> 128 3x3, both gradients, by its tiles' times 14.8 us, so 12.7; 217 drawn layers level)
void gemm_conv_pieces(int dtype, GemmArgs &gx, const GemmArgs &gy) {
    if (dtype != D8_FLOAT16 || gx.virt != VIRT_A_ROWS || gy.virt != VIRT_B_KROWS) return;
    GemmArgs y = gy;
    y.splits = plan_splits(gemm_tiled_k_step(dtype), y.M, y.N, y.K, 1, y.red, (size_t)-1, &y.tiles_per_split, y.virt);
    const HalfShare other = half_share(y);
    const int ways[2] = {BY_SHARED_TIMES, BY_STEPS};
    double us[2];
    for (int k = 0; k < 2; ++k) {
        GemmArgs x = gx;
        int tiles;
        x.pieces_by = ways[k];
        plan_pieces(dtype, x, 0, 0, (size_t)-1);
        us[k] = half_pair_us(half_share(x), other, tiles);
    }
    gx.pieces_by = ways[us[1] < us[0]];
}

// Microseconds of a product in steps of its tiles, for the choice between two ways of a convolution (products and patch products alike,
// so what counts is their ratio).  Over 3100 calls on drawn layers the time measured was 1.0 - 1.2 of this at the median in fp32, 1.1 - 1.5
// in half, before half tiles went straight into LDS.  Later kernels are not in it: a half plan may have been made by half_tile_us and is priced in
// steps all the same, and a product that gemm_is_short takes is counted as a tiled one.  Of 5440 drawn half layers one goes the wrong way for that
// (both gradients of DeConv2d 2 x 7x7x64 -> 448 5x5 stride 2, 9.9 us through the loader, 18.7 on an interim matrix) and several go the right way (Conv2d
// 1 x 50x50x80 -> 136 5x5 34 and 21.9).  Plans in steps here, for either kind of product or both, or the lower of the two prices, were no better.
double gemm_estimate_us(int dtype, const GemmArgs &g0, int transA, int transB) {
    const bool half_elems = dtype == D8_FLOAT16;
    const int BK = gemm_tiled_k_step(dtype);
    const double unit = half_elems ? 0.5 : 2.0;
    const double patch = !half_elems && (g0.virt == VIRT_A_ROWS || g0.virt == VIRT_A_CLASSES) ? 1.1 : 1.0;  // (offsets per step)
    if (g0.virt == VIRT_A_CLASSES) {  // one launch, no class cut: its longest workgroup or a compute unit's share of all of them
        const int bn = !half_elems && g0.N <= 32 ? 32 : g0.N < 128 ? 64 : 128;
        const double area = bn / 128.0, step = half_elems ? (area < 0.6 ? 0.76 : 1.0) : area * 1.08;
        const long cus = cu_count(), tilesN = ceil_div(g0.N, bn), k = ceil_div(g0.K, BK);
        long wgs = 0, steps = 0, longest = 0;
        for (int i = 0; i < g0.ncls; ++i) {
            const long t = ceil_div(g0.cls[i].M, 128) * tilesN, n = g0.cls[i].red * k;
            wgs += t, steps += t * n;
            if (n > longest) longest = n;
        }
        const double share = (double)steps / (wgs < cus ? wgs : cus), alone = longest * (half_elems ? 1.0 : 1.02);
        return ((share > alone ? share : alone) * step + (half_elems ? 7.0 : 0.5 + 2.0 * sqrt(area)) + (half_elems ? 0.5 : 0.3) * ((wgs + cus - 1) / cus - 1)) *
               unit * patch;
    }
    if (g0.virt == VIRT_NONE && gemm_is_small(g0.M, g0.N, g0.K, g0.batch, g0.red)) return 4.0;
    GemmArgs g = g0;
    g.tile_hint = narrow_output(dtype, g) ? HINT_128x32 : HINT_NONE;
    plan_pieces(dtype, g, transA, transB, (size_t)-1);
    const long total = (long)g.red * ceil_div(g.K, BK);
    int bm = 128, bn = 128;
    if (g.tile_hint) bm = g.tile_hint == HINT_64x64 ? 64 : 128, bn = g.tile_hint == HINT_64x64 ? 64 : 32;
    else if (g.virt == VIRT_B_KROWS && ((g.M < 128 && g.N < 128) || gemm_tiled_krows_64(g.virt, g.M, g.N))) bm = bn = 64;
    else if (g.N < 128) bn = 64;
    else if (g.M < 128 || (g.splits == 1 && gemm_tiled_half_tiles(g.M, g.N, g.batch, total, BK))) bm = 64;
    // (a filter gradient that is stored transposed per tap straight from its tiles, two bytes at a time: 4 - 6 us)
    return tile_cost(half_elems, bm, bn, g, total, g.splits) * unit * patch + (half_elems && g.perm_OC && g.splits == 1 ? 4.0 : 0.0);
}

static int gemm_tiled_run_whole(int dtype, GemmArgs &g, int transA, int transB, void *workspace, size_t workspace_bytes,
                                hipStream_t stream) {
    g.ws = (float *)workspace;
    const size_t usable = (workspace && ((size_t)workspace & 15) == 0) ? workspace_bytes : 0;
    plan_pieces(dtype, g, transA, transB, usable);
    return dtype == D8_FLOAT16 ? launch<f16>(g, transA, transB, true, stream) : launch<float>(g, transA, transB, true, stream);
}

int gemm_small_run(int dtype, const GemmArgs &g, int transA, int transB, hipStream_t stream) {
    return dtype == D8_FLOAT16 ? launch_small<f16>(g, transA, transB, stream) : launch_small<float>(g, transA, transB, stream);
}

int gemm_tiled_run(int dtype, GemmArgs &g, int transA, int transB, void *workspace, size_t workspace_bytes,
                   hipStream_t stream) {
    if (!transA && !transB && gemm_is_short(dtype, g)) return gemm_small_run(dtype, g, transA, transB, stream);
    if (narrow_output(dtype, g)) g.tile_hint = HINT_128x32;
    static const bool no_cut = getenv("D8_GEMM_NO_ROW_CUT") != nullptr;  // tuning and test aid
    const int head = (no_cut || transA) ? 0 : balanced_rows(g);
    if (!head) return gemm_tiled_run_whole(dtype, g, transA, transB, workspace, workspace_bytes, stream);
    const size_t es = dtype_bytes(dtype);
    GemmArgs first = g, second = g;
    first.M = head;
    second.M = g.M - head;
    second.C = (char *)g.C + (size_t)head * g.ldc * es;
    if (g.virt == VIRT_A_ROWS) second.m_base = g.m_base + head;
    else second.A = (const char *)g.A + (size_t)head * g.lda * es;
    if (!gemm_tiled_eligible(dtype, second, transA, transB))
        return gemm_tiled_run_whole(dtype, g, transA, transB, workspace, workspace_bytes, stream);
    // The band's pieces ride in the first part's launch (GemmArgs::tail_m0) when it is split at all and is at least
    // one tile high; only its reduction is a launch of its own.
    const bool two_launches = getenv("D8_GEMM_BAND_LAUNCH") != nullptr;  // tuning and test aid (read at every call)
    second.ws = (float *)workspace;
    second.splits = (two_launches || g.splits != 1 || g.perm_OC != 0) ? 0
                    : plan_band_pieces(gemm_tiled_k_step(dtype), second.M, second.N, second.K, second.red,
                                       (workspace && ((size_t)workspace & 15) == 0) ? workspace_bytes : 0, &second.tiles_per_split);
    if (second.splits > 1) {
        GemmArgs both = g;
        both.ws = second.ws;
        both.splits = 1;
        both.tiles_per_split = g.red * ceil_div(g.K, gemm_tiled_k_step(dtype));
        both.tail_m0 = head, both.tail_splits = second.splits, both.tail_tps = second.tiles_per_split;
        if (int rc = gemm_tiled_launch(dtype, both, transA, transB, stream)) return rc;
        return dtype == D8_FLOAT16 ? launch_reduce<f16>(second, stream) : launch_reduce<float>(second, stream);
    }
    if (int rc = gemm_tiled_run_whole(dtype, first, transA, transB, nullptr, 0, stream)) return rc;
    return gemm_tiled_run_whole(dtype, second, transA, transB, workspace, workspace_bytes, stream);
}

static bool grads_apart() { return getenv("D8_MATMUL_GRADS_APART") != nullptr; }  // tuning and test aid (read at every call)

// Whether the two gradients of a MatrixMultiply (g0 = dZ . Y^T, NT; g1 = X^T . dZ, TN) run on the kernel for small products, in
// one launch where one call asks for both, and so that a call for one leaves the same bits: both small in the sense of
// gemm_is_small, or both short and with no more workgroups than run at once.  us, as they ran before (two launches, or one of tiles
// and a pass over partial sums) / so, by workgroups; 70 drawn calls: fp32 280 x 192 x 64 (66) 9.8 / 5.3, 64 x 704 x 336 (286)
// 10.4 / 6.5, 64 x 2525 x 120 (474) 13.3 / 5.1, 128 x 3200 x 64 (600) 6.6 / 7.1; half 336 x 320 x 14 (120) 11.7 / 4.5, 640 x 320 x 128 (240)
// 9.4 / 5.8, 384 x 832 x 64 (364) 6.2 / 6.6, 3 x 64 x 832 x 640 (676) 9.3 / 10.2.
bool gemm_gradients_are_small(int dtype, const GemmArgs &g0, int ta0, int tb0, const GemmArgs &g1, int ta1, int tb1) {
    if (dtype == D8_FLOAT64 || ta0 || !tb0 || !ta1 || tb1) return false;
    if (g0.virt != VIRT_NONE || g1.virt != VIRT_NONE || g0.K < 1 || g1.K < 1) return false;
    const long n = small_workgroups(g0) + small_workgroups(g1);
    if (gemm_is_small(g0.M, g0.N, g0.K, g0.batch, g0.red) && gemm_is_small(g1.M, g1.N, g1.K, g1.batch, g1.red)) return n <= 0x7fffffffL;
    const char *copies = getenv("D8_GEMM_PACK");  // (see pack_pays; both are tuning and test aids, read at every call)
    if (grads_apart() || (copies && atoi(copies) != 0)) return false;
    return gemm_fits_small(dtype, g0) && gemm_fits_small(dtype, g1) && n <= (dtype == D8_FLOAT16 ? 1L : 2L) * cu_count();
}

static bool whole_steps(int dtype, const GemmArgs &g0, const GemmArgs &g1) {
    const int BK = gemm_tiled_k_step(dtype);
    return g0.K % BK == 0 && g1.K % BK == 0;
}

SharedLaunch gemm_small_pair_run(int dtype, const GemmArgs &g0, int ta0, int tb0, const GemmArgs &g1, int ta1, int tb1, hipStream_t stream, int *rc) {
    if (!gemm_gradients_are_small(dtype, g0, ta0, tb0, g1, ta1, tb1)) return APART;
    const int nx0 = ceil_div(g0.N, 32), ny0 = ceil_div(g0.M, 32), nx1 = ceil_div(g1.N, 32), ny1 = ceil_div(g1.M, 32);
    const long n0 = small_workgroups(g0), n1 = small_workgroups(g1);
    GemmArgs a = g0, b = g1;
    a.splits = b.splits = 1;
    a.by.nbx = reciprocal_of(nx0), a.by.tiles = reciprocal_of(nx0 * ny0), b.by.nbx = reciprocal_of(nx1), b.by.tiles = reciprocal_of(nx1 * ny1);
    if (dtype == D8_FLOAT16)
        hipLaunchKernelGGL((gemm_small_pair_kernel<f16>), dim3((unsigned)(n0 + n1)), dim3(SMALL_WAVES * 64), 0, stream, a, b, nx0, ny0, (int)n0, nx1, ny1);
    else
        hipLaunchKernelGGL((gemm_small_pair_kernel<float>), dim3((unsigned)(n0 + n1)), dim3(SMALL_WAVES * 64), 0, stream, a, b, nx0, ny0, (int)n0, nx1, ny1);
    const hipError_t e = hipGetLastError();
    *rc = e == hipSuccess ? 0 : fail((int)e, "kernel launch: %s", hipGetErrorString(e));
    const bool small = gemm_is_small(g0.M, g0.N, g0.K, g0.batch, g0.red) && gemm_is_small(g1.M, g1.N, g1.K, g1.batch, g1.red);
    return small || whole_steps(dtype, g0, g1) ? SHARED : SHARED_KEPT;
}

// d8_conv_grad_pair_launches, d8_conv_grad_kept_pair_launches, d8_conv_grad_crowded_pair_launches
static std::atomic<unsigned long> pair_launches{0}, kept_pair_launches{0}, crowded_pair_launches{0};

// Both gradients of a convolution as one launch (gemm_tiled_pair_launch) when that fills compute units the two
// products would each leave idle: gx is not cut into a band and not split, the workgroups of both fit the chip
// side by side (two per compute unit).  gy's reduction is split as it would be alone and reduced afterwards.
// Returns false, with nothing launched, when the pair does not qualify; *rc is the launches' status otherwise.
bool gemm_tiled_run_pair(int dtype, GemmArgs &gx, GemmArgs &gy, void *workspace, size_t workspace_bytes, hipStream_t stream, int *rc) {
    const bool off = getenv("D8_CONV_GRADS_APART") != nullptr;  // tuning and test aid (read at every call)
    if (off || dtype == D8_FLOAT64) return false;
    if (gx.virt != VIRT_A_ROWS || gy.virt != VIRT_B_KROWS || gx.batch != 1 || gy.batch != 1) return false;
    if (!gemm_tiled_eligible(dtype, gx, 0, 0, TILED_WHOLE) || !gemm_tiled_eligible(dtype, gy, 1, 0, TILED_WHOLE)) return false;
    // More workgroups than the chip holds at once (two per compute unit): in half the shared launch still gains
    // (3x3 Conv2d, B32: 56x56x64 49.9 -> 47.0 us, 14x14x256 46.0 -> 34.9, 56x56x64->128 74.2 -> 65.0; DeConv2d 4x4 s2
    // B64 14x14x256 60.7 -> 47.9), gx's remainder band riding along as it does alone.  In fp32, bound by the matrix
    // pipe, it gains 2-4 % where gx's output is narrow (fewer than 128 input channels: three workgroups of either
    // product fit a compute unit; B32 56x56x64 135.4 -> 129.7 us) and loses 8-21 % on 3x3 layers of 128 channels at
    // 28x28 (128 x 128 tiles in both products): there only a gx with a remainder band, i.e. a narrow one, pairs.
    const int head = balanced_rows(gx);
    const bool big = dtype == D8_FLOAT16 || head != 0;
    const size_t usable = (workspace && ((size_t)workspace & 15) == 0) ? workspace_bytes : 0;
    const int BK = gemm_tiled_k_step(dtype);
    int tps = 0;
    // Alone, a gx of few tiles would be cut into pieces to fill the chip; beside gy's workgroups it runs whole when
    // its reduction is short: up to 40 K steps in half, where a step waits longer than it multiplies (B16 14x14x256
    // 4x4 s2 DeConv2d: 43.3 -> 30.1 us, 3x3 Conv2d of 256 channels at B16 14x14: 45.5 -> 37.4 us); never in fp32,
    // whose steps are bound by the matrix pipe (36 steps whole: 49 -> 80 us).
    const char *lim = getenv("D8_CONV_PAIR_STEPS");  // tuning and test aid (read at every call)
    const long whole_steps = lim ? atol(lim) : (dtype == D8_FLOAT16 ? 40 : 0);
    if (plan_splits(BK, gx.M, gx.N, gx.K, 1, gx.red, usable, &tps, gx.virt) != 1 && (long)gx.red * ceil_div(gx.K, BK) > whole_steps) return false;
    gx.splits = 1, gx.tiles_per_split = gx.red * ceil_div(gx.K, BK);
    gx.ws = nullptr, gx.tail_splits = 0;
    gy.ws = (float *)workspace, gy.tail_splits = 0;
    gy.splits = plan_splits(BK, gy.M, gy.N, gy.K, 1, gy.red, usable, &gy.tiles_per_split, gy.virt);
    GemmArgs band = gx;
    if (head) {  // the band's pieces behind gy's partial sums in the workspace (the scratch query's which = 3 has room for both)
        const size_t gy_bytes = gy.splits > 1 ? ((size_t)gy.splits * gy.M * gy.N * sizeof(float) + 255) & ~(size_t)255 : 0;
        if (usable <= gy_bytes) return false;
        band.M = gx.M - head;
        band.C = (char *)gx.C + (size_t)head * gx.ldc * dtype_bytes(dtype);
        band.m_base = gx.m_base + head;
        band.ws = (float *)((char *)workspace + gy_bytes);
        band.splits = plan_band_pieces(BK, band.M, band.N, band.K, band.red, usable - gy_bytes, &band.tiles_per_split);
        if (band.splits < 2) return false;
        gx.ws = band.ws;
        gx.tail_m0 = head, gx.tail_splits = band.splits, gx.tail_tps = band.tiles_per_split;
    }
    const long wgs = gemm_tiled_pair_workgroups(dtype, gx, gy);
    if (wgs <= 0 || (wgs > 2L * cu_count() && !big)) return false;
    ++pair_launches;
    *rc = gemm_tiled_pair_launch(dtype, gx, gy, stream);
    if (!head) band.splits = 1;  // (no band: nothing of gx's to reduce)
    if (*rc == 0) *rc = launch_reduce_pair(dtype, band, gy, stream);
    return true;
}

// Both gradients of a convolution in one launch, in half and fp32, on classes of output pixels or on patch rows.
// A Conv2d with a stride in half: the classes' workgroups are short (1 to 4 taps of a 3 x 3 filter) and rarely a
// whole number of rounds, and the filter gradient's fill the last one.
// 16 x 57x57x96 -> 160, 3x3 stride 2: both gradients 38.4 -> 31.8 us; 60 drawn layers 1810 -> 1539 us, none slower.
// Patch rows whose last K step is cut short, or that are cut into pieces: a launch or two fewer, and no half empty chip behind the
// pieces of either.  98 drawn layers 3642 -> 3312 us, 9 x 33x33x64 -> 64 3x3 18.5 -> 12.4, 15 x 18x18x192 -> 272 5x5 67.1 -> 49.7,
// DeConv2d 1 x 33x33x56 -> 320 2x2 stride 2 19.2 -> 11.7; none slower by more than 1 %.  fp32
// (where kept_tiles takes it): 340 drawn layers 15179 -> 14044 us, 6 x 8x8x64 -> 64 3x3 17.8 -> 9.9.
bool gemm_tiled_kept_pair_plan(int dtype, GemmArgs &gx, GemmArgs &gy, void *workspace, size_t workspace_bytes) {
    if (getenv("D8_CONV_GRADS_APART") != nullptr || dtype == D8_FLOAT64) return false;
    const size_t usable = (workspace && ((size_t)workspace & 15) == 0) ? workspace_bytes : 0;
    const int BK = gemm_tiled_k_step(dtype);
    if (!gemm_tiled_eligible(dtype, gy, 1, 0) || gemm_is_small(gy.M, gy.N, gy.K, gy.batch, gy.red)) return false;
    gy.ws = (float *)workspace;
    gy.splits = plan_splits(BK, gy.M, gy.N, gy.K, 1, gy.red, usable, &gy.tiles_per_split, gy.virt);
    const auto tiles = dtype == D8_FLOAT16 ? gemm_tiled_kept_pair_tiles_f16 : gemm_tiled_kept_pair_tiles_f32;
    if (gx.virt == VIRT_A_CLASSES) return tiles(gx, gy) != APART;
    if (narrow_output(dtype, gx)) gx.tile_hint = HINT_128x32;
    if (gx.virt != VIRT_A_ROWS || balanced_rows(gx) || !gemm_tiled_eligible(dtype, gx, 0, 0) || gemm_is_small(gx.M, gx.N, gx.K, gx.batch, gx.red)) return false;
    gemm_conv_pieces(dtype, gx, gy);
    plan_pieces(dtype, gx, 0, 0, usable);
    // the partial sums side by side
    const size_t gy_bytes = gy.splits > 1 ? ((size_t)gy.splits * gy.M * gy.N * sizeof(float) + 255) & ~(size_t)255 : 0;
    const size_t gx_bytes = gx.splits > 1 ? (size_t)gx.splits * gx.M * gx.N * sizeof(float) : 0;
    if (gy_bytes + gx_bytes > usable) return false;
    gx.ws = (float *)((char *)workspace + gy_bytes);
    return tiles(gx, gy) != APART;
}

int gemm_tiled_kept_pair_run(int dtype, const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    const bool classes = gx.virt == VIRT_A_CLASSES;
    const auto pair = dtype == D8_FLOAT16 ? (classes ? gemm_tiled_pair_classes_f16 : gemm_tiled_pair_rows_f16) : (classes ? gemm_tiled_pair_classes_f32 : gemm_tiled_pair_rows_f32);
    const SharedLaunch shared = dtype == D8_FLOAT16 ? gemm_tiled_kept_pair_tiles_f16(gx, gy) : gemm_tiled_kept_pair_tiles_f32(gx, gy);
    ++(shared == SHARED ? kept_pair_launches : crowded_pair_launches);
    if (int rc = pair(gx, gy, stream)) return rc;
    return launch_reduce_pair(dtype, gx, gy, stream);
}

// Both gradients of a MatrixMultiply in one launch, each cut as it would be alone, whatever K leaves of a last step and however
// many workgroups there are: a launch or two fewer, and one last round instead of two.  us apart / so: a K step cut short, of 90
// drawn calls the 25 that are, 1.29 times as fast at the mean: fp32 448 x 304 x 152 15.8 / 10.2, 648 x 1128 x 64 15.4 / 11.5; half 368 x 824 x
// 64 8.8 / 6.8, 5864 x 568 x 576 27.6 / 22.1.  More workgroups than the chip holds, longer ones first, 58 drawn calls in fp32 3750 / 3331:
// 608 x 2816 x 768 61.5 / 46.4, 4096 x 2112 x 480 179 / 143, and apart where one launch leaves a tail behind (leaves_a_tail, leaves_a_half_tail); in half 4 x 3072 x
// 680 x 1152 70.9 / 54.1, 3072 x 3584 x 744 59.0 / 48.4.
static SharedLaunch plain_pair_plan(int dtype, GemmArgs &g0, int ta0, int tb0, GemmArgs &g1, int ta1, int tb1, void *workspace, size_t workspace_bytes) {
    if (dtype == D8_FLOAT64 || ta0 || !tb0 || !ta1 || tb1) return APART;
    if (g0.virt != VIRT_NONE || g1.virt != VIRT_NONE || g0.K < 1 || g1.K < 1) return APART;
    for (const GemmArgs *g : {&g0, &g1})
        if (g->batch > 448 || g->M > 65535 * 128) return APART;  // (beyond one launch's limits: d8_gemm cuts it into several)
    if (!g0.packed && !g1.packed && (!gemm_tiled_eligible(dtype, g0, ta0, tb0, TILED_PIECES) || !gemm_tiled_eligible(dtype, g1, ta1, tb1, TILED_PIECES))) return APART;
    if (gemm_is_small(g0.M, g0.N, g0.K, g0.batch, g0.red) || gemm_is_small(g1.M, g1.N, g1.K, g1.batch, g1.red)) return APART;
    if (balanced_rows(g0) || balanced_rows(g1)) return APART;
    const size_t usable = (workspace && ((size_t)workspace & 15) == 0) ? workspace_bytes : 0;
    // each split as it would be alone, the partial sums of the two side by side in the workspace
    if (dtype == D8_FLOAT16) half_pair_plan(g0, g1, usable);
    else plan_pieces(dtype, g0, 0, 1, usable), plan_pieces(dtype, g1, 1, 0, usable);
    const size_t need0 = g0.splits > 1 ? ((size_t)g0.splits * g0.batch * g0.M * g0.N * sizeof(float) + 255) & ~(size_t)255 : 0;
    const size_t need1 = g1.splits > 1 ? (size_t)g1.splits * g1.batch * g1.M * g1.N * sizeof(float) : 0;
    if (need0 + need1 > usable) return APART;
    g0.ws = (float *)workspace, g1.ws = (float *)((char *)workspace + need0);
    g0.tail_splits = g1.tail_splits = 0;
    const long wgs = gemm_tiled_plain_pair_workgroups(dtype, g0, g1);
    if (wgs <= 0 || wgs > 0x7fffffffL) return APART;
    return wgs <= 2L * cu_count() && (g0.packed || whole_steps(dtype, g0, g1)) ? SHARED : SHARED_KEPT;
}

bool gemm_gradients_share(int dtype, GemmArgs &g0, int ta0, int tb0, GemmArgs &g1, int ta1, int tb1) {
    GemmArgs a = g0, b = g1;
    for (GemmArgs *g : {&a, &b}) g->A = g->B = nullptr, g->C = nullptr;
    if (plain_pair_plan(dtype, a, ta0, tb0, b, ta1, tb1, (void *)4096, (size_t)1 << 62) == APART) return false;
    g0.pieces_by = a.pieces_by, g1.pieces_by = b.pieces_by;
    return true;
}

static int plain_pair_run(int dtype, const GemmArgs &g0, const GemmArgs &g1, hipStream_t stream) {
    if (int rc = gemm_tiled_plain_pair_launch(dtype, g0, g1, stream)) return rc;
    return launch_reduce_pair(dtype, g0, g1, stream);
}

SharedLaunch gemm_tiled_run_plain_pair(int dtype, GemmArgs &g0, int ta0, int tb0, GemmArgs &g1, int ta1, int tb1, void *workspace,
                                       size_t workspace_bytes, hipStream_t stream, int *rc) {
    if (grads_apart()) return APART;
    const SharedLaunch shared = plain_pair_plan(dtype, g0, ta0, tb0, g1, ta1, tb1, workspace, workspace_bytes);
    if (shared) *rc = plain_pair_run(dtype, g0, g1, stream);
    return shared;
}

// Where the copies go, one behind the other.  A thread copies a piece of four rows, or of one where that leaves compute units without
// two workgroups.
struct PackLaunch {
    PackList list;
    unsigned blocks;
    bool single;
};
static void pack_list(const PackPlan &plan, void *workspace, PackLaunch &p) {
    auto lay_out = [&](int rows) {
        p.blocks = 0;
        char *to = (char *)workspace;
        p.list.n = plan.n;
        for (int k = 0; k < plan.n; ++k) {
            const PackShape &s = plan.shapes[k];
            int across = 3;
            while (across < 8 && (8 << across) < pack_pitch(s)) ++across;
            p.list.m[k] = {(const f16 *)s.p, (f16 *)to, (int)s.rows, s.cols, s.ld, pack_pitch(s), s.per, reciprocal_of(s.per), s.stride, across, p.blocks};
            p.blocks += (unsigned)ceil_div(s.rows, rows * (256 >> across));
            to += pack_bytes(s);
        }
    };
    lay_out(4);
    p.single = p.blocks < 2u * cu_count();
    if (p.single) lay_out(1);
}
// The two products on copies, and how: whether they share a launch is known before anything is copied, because of products that run
// one after the other only those read copies that have something to copy.
struct PackRun {
    PackPlan plan;
    PackLaunch copies;
    GemmArgs g[2];
    SharedLaunch shared;
};
// The product on its copies.
static GemmArgs packed_args(GemmArgs g, const int (&slot)[2], const PackList &list) {
    if (slot[0] >= 0) {
        const PackArgs &a = list.m[slot[0]];
        g.A = a.dst, g.lda = a.pitch, g.sA = g.sA ? (long)a.per * a.pitch : 0;
    }
    if (slot[1] >= 0) {
        const PackArgs &b = list.m[slot[1]];
        g.B = b.dst, g.ldb = b.pitch, g.sB = g.sB ? (long)b.per * b.pitch : 0;
    }
    g.packed = 1, g.padM = (g.M + 7) & ~7, g.padN = (g.N + 7) & ~7;
    return g;
}
static int launch_pack(const PackLaunch &p, hipStream_t stream) {
    if (p.single) hipLaunchKernelGGL(pack_rows_kernel<1>, dim3(p.blocks), dim3(256), 0, stream, p.list);
    else hipLaunchKernelGGL(pack_rows_kernel<4>, dim3(p.blocks), dim3(256), 0, stream, p.list);
    D8_LAUNCH_CHECK();
    return 0;
}
static bool pack_run_plan(int dtype, const PackedProduct (&p)[2], void *workspace, size_t workspace_bytes, PackRun &r) {
    if (!workspace || ((size_t)workspace & 15) || !pack_plan(dtype, p, 2, r.plan) || r.plan.bytes > workspace_bytes) return false;
    char *const to = (char *)workspace + r.plan.bytes;
    pack_list(r.plan, workspace, r.copies);
    auto packed = [&](int i) { return packed_args(*p[i].g, r.plan.slot[i], r.copies.list); };
    r.g[0] = packed(0), r.g[1] = packed(1);
    const size_t rest = workspace_bytes - r.plan.bytes;
    r.shared = grads_apart() ? APART : plain_pair_plan(dtype, r.g[0], p[0].ta, p[0].tb, r.g[1], p[1].ta, p[1].tb, to, rest);
    if (!pack_pays(p, 2, r.plan)) return false;
    for (int i = 0; i < 2; ++i) {
        const GemmArgs &g = *p[i].g;  // (not at the cost of the pieces that it would run in without copies)
        if (d8_gemm_workspace_bytes(dtype, p[i].ta, p[i].tb, g.M, g.N, g.K, g.red > 1 ? g.red : g.batch, g.red > 1 ? 0 : 1) > rest) return false;
        if (!r.shared) r.g[i] = r.plan.slot[i][0] >= 0 || r.plan.slot[i][1] >= 0 ? packed(i) : g;
    }
    return true;
}

size_t gemm_pack_bytes(int dtype, const PackedProduct (&p)[2]) {
    PackRun r;
    return pack_run_plan(dtype, p, (void *)4096, (size_t)1 << 62, r) ? r.plan.bytes : 0;
}

bool gemm_pack_run(int dtype, const PackedProduct (&p)[2], void *workspace, size_t workspace_bytes, hipStream_t stream, SharedLaunch *shared, int *rc) {
    PackRun r;
    if (!pack_run_plan(dtype, p, workspace, workspace_bytes, r)) return false;
    *shared = r.shared;
    *rc = launch_pack(r.copies, stream);
    if (*rc == 0 && r.shared) *rc = plain_pair_run(dtype, r.g[0], r.g[1], stream);
    for (int i = 0; i < 2 && !r.shared && *rc == 0; ++i)
        *rc = gemm_tiled_run(dtype, r.g[i], p[i].ta, p[i].tb, (char *)workspace + r.plan.bytes, workspace_bytes - r.plan.bytes, stream);
    return true;
}

// A forward product by itself.
static bool pack_one_plan(int dtype, const PackedProduct &p, size_t workspace_bytes, PackPlan &plan) {
    if (!pack_plan(dtype, &p, 1, plan) || plan.bytes > workspace_bytes || !pack_pays(&p, 1, plan)) return false;
    const GemmArgs &g = *p.g;  // (not at the cost of the pieces that it would run in without copies)
    return d8_gemm_workspace_bytes(dtype, p.ta, p.tb, g.M, g.N, g.K, g.red > 1 ? g.red : g.batch, g.red > 1 ? 0 : 1) <= workspace_bytes - plan.bytes;
}

size_t gemm_pack_one_bytes(int dtype, const PackedProduct &p) {
    PackPlan plan;
    return pack_one_plan(dtype, p, (size_t)1 << 62, plan) ? plan.bytes : 0;
}

bool gemm_pack_run_one(int dtype, const PackedProduct &p, void *workspace, size_t workspace_bytes, hipStream_t stream, int *rc) {
    PackPlan plan;
    if (!workspace || ((size_t)workspace & 15) || !pack_one_plan(dtype, p, workspace_bytes, plan)) return false;
    PackLaunch copies;
    pack_list(plan, workspace, copies);
    GemmArgs g = packed_args(*p.g, plan.slot[0], copies.list);
    if ((*rc = launch_pack(copies, stream)) == 0)
        *rc = gemm_tiled_run(dtype, g, p.ta, p.tb, (char *)workspace + plan.bytes, workspace_bytes - plan.bytes, stream);
    return true;
}

bool gemm_fuses_store(int dtype, const GemmArgs &g, int transA, int transB, TiledRule rule) {
    // (a product beyond one launch's limits -- more than 448 outputs, more than 65535 * 128 rows -- is cut into several
    // by d8_gemm; the fused store stays out of that: the caller runs the product and one pass over its result)
    if (dtype == D8_FLOAT64 || g.K < 1 || g.beta != 0.f || g.red != 1 || g.batch > 448 || g.M > 65535 * 128) return false;
    // (gemm_small_kernel had no fused store: asked by the other rules, which say where two passes used to round twice, it has none)
    if (rule != TILED_ANY && g.virt == VIRT_NONE && gemm_is_small(g.M, g.N, g.K, g.batch, g.red)) return false;
    return gemm_tiled_eligible(dtype, g, transA, transB, rule);
}

int gemm_run_fused(int dtype, GemmArgs &g, int transA, int transB, void *workspace, size_t workspace_bytes, hipStream_t stream) {
    return gemm_tiled_run(dtype, g, transA, transB, workspace, workspace_bytes, stream);
}

}  // namespace d8

using namespace d8;

extern "C" {

size_t d8_gemm_workspace_bytes(int dtype, int transA, int transB, int M, int N, int K,
                               int batch, long strideC) {
    (void)transA;
    (void)transB;
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return 0;
    const int red = (strideC == 0 && batch > 1) ? batch : 1;
    const int outs = red > 1 ? 1 : batch;
    if (dtype == D8_FLOAT64) {
        int tps64 = 0;
        const int pieces = gemm_f64_splits(M, N, K, outs, red, (size_t)-1, &tps64);
        return pieces > 1 ? (size_t)pieces * outs * M * N * sizeof(double) : 0;
    }
    // whichever kernel ends up running, the larger of the two plans fits
    int tps = 0;
    const int a = plan_splits(gemm_tiled_k_step(dtype), M, N, K, outs, red, (size_t)-1, &tps);
    const int b = plan_splits(dtype == D8_FLOAT16 ? Tile<f16>::BK : Tile<float>::BK, M, N, K, outs, red, (size_t)-1, &tps);
    const int splits = a > b ? a : b;
    const size_t whole = splits > 1 ? (size_t)splits * outs * M * N * sizeof(float) : 0;
    const size_t band = outs == 1 ? gemm_tiled_workspace(dtype, M, N, K, red) : 0;  // a tall product's remainder band, split
    return whole > band ? whole : band;
}

// One product whose grid fits the launch limits (at most MAX_BATCH independent outputs, at most MAX_ROWS rows).
static int gemm_one(int dtype, int transA, int transB, int M, int N, int K,
                    const void *A, int lda, long strideA, const void *B, int ldb, long strideB,
                    float beta, void *C, int ldc, long strideC, int batch,
                    void *workspace, size_t workspace_bytes, void *stream) {
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.A = A;
    g.B = B;
    g.C = C;
    g.ws = (float *)workspace;
    g.ws_bytes = workspace_bytes;
    g.M = M;
    g.N = N;
    g.K = K;
    g.lda = lda;
    g.ldb = ldb;
    g.ldc = ldc;
    g.sA = strideA;
    g.sB = strideB;
    g.sC = strideC;
    g.beta = beta;
    g.red = (strideC == 0 && batch > 1) ? batch : 1;
    g.batch = g.red > 1 ? 1 : batch;
    g.splits = 1;
    g.tiles_per_split = 0;
    g.virt = VIRT_NONE;
    g.m_base = 0;
    memset(&g.pg, 0, sizeof(g.pg));
    if (dtype == D8_FLOAT64) return gemm_f64_launch(g, transA, transB, as_stream(stream));
    const bool tiled = K > 0 && gemm_tiled_eligible(dtype, g, transA, transB);
    // the tiled kernels' own driver plans the split and cuts a tall product's remainder band
    if (tiled && !gemm_is_small(M, N, K, g.batch, g.red)) return gemm_tiled_run(dtype, g, transA, transB, workspace, workspace_bytes, as_stream(stream));
    if (K > 0) {  // K == 0 is the empty reduction: C = beta * C
        const int BK = tiled ? gemm_tiled_k_step(dtype) : (dtype == D8_FLOAT16 ? Tile<f16>::BK : Tile<float>::BK);
        g.splits = plan_splits(BK, M, N, K, g.batch, g.red, (workspace && ((size_t)workspace & 15) == 0) ? workspace_bytes : 0, &g.tiles_per_split);
    }
    return dtype == D8_FLOAT16 ? launch<f16>(g, transA, transB, tiled, as_stream(stream))
                               : launch<float>(g, transA, transB, tiled, as_stream(stream));
}

unsigned long d8_conv_grad_pair_launches(void) { return pair_launches.load(); }
unsigned long d8_conv_grad_kept_pair_launches(void) { return kept_pair_launches.load(); }
unsigned long d8_conv_grad_crowded_pair_launches(void) { return crowded_pair_launches.load(); }

int d8_gemm_phase_record(void *records, size_t bytes) {
    D8_REQUIRE(((size_t)records & 7) == 0, "d8_gemm_phase_record: the record buffer is not 8-byte aligned");
    gemm_tiled_phase_record(records, bytes);
    return 0;
}

int d8_gemm(int dtype, int transA, int transB, int M, int N, int K,
            const void *A, int lda, long strideA,
            const void *B, int ldb, long strideB,
            float beta, void *C, int ldc, long strideC, int batch,
            void *workspace, size_t workspace_bytes, void *stream) {
    if (dtype != D8_FLOAT16 && dtype != D8_FLOAT32 && dtype != D8_FLOAT64)
        return fail(D8_ERR_DTYPE, "d8_gemm: element type %d is not supported", dtype);
    D8_REQUIRE(!(transA && transB), "d8_gemm: transA and transB together are not supported");
    D8_REQUIRE(M >= 0 && N >= 0 && K >= 0 && batch >= 0, "d8_gemm: negative size");
    D8_REQUIRE(beta == 0.f || beta == 1.f, "d8_gemm: beta must be 0 or 1");
    if (M == 0 || N == 0 || batch == 0) return 0;
    D8_REQUIRE(A && B && C, "d8_gemm: null operand");
    D8_REQUIRE(lda >= (transA ? M : K), "d8_gemm: lda %d too small", lda);
    D8_REQUIRE(ldb >= (transB ? K : N), "d8_gemm: ldb %d too small", ldb);
    D8_REQUIRE(ldc >= N, "d8_gemm: ldc %d too small", ldc);
    D8_REQUIRE(strideA >= 0 && strideB >= 0 && strideC >= 0, "d8_gemm: negative stride");
    D8_REQUIRE(dtype != D8_FLOAT64 || (long)ceil_div(N, 64) < 65536, "d8_gemm: N = %d is beyond the %d columns a Float64 launch covers", N, 65535 * 64);

    // A launch covers at most 65535 workgroups along its second and third axes.  A longer batch of independent
    // products and a taller matrix are walked in slices, each an ordinary product on advanced pointers (the
    // slices run one after the other on the stream, so they may share the workspace).
    constexpr int MAX_BATCH = 448;            // independent outputs per launch (the tiled kernels take fewer than 512)
    constexpr int MAX_ROWS = 65535 * 128;     // rows of C per launch
    const size_t es = dtype_bytes(dtype);
    const bool summed = strideC == 0 && batch > 1;
    const int nb = summed ? 1 : ceil_div(batch, MAX_BATCH), per_b = summed ? batch : ceil_div(batch, nb);
    const int nm = ceil_div(M, MAX_ROWS);
    const int per_m = nm > 1 ? (ceil_div(ceil_div(M, nm), 128) * 128) : M;
    for (int b0 = 0; b0 < batch; b0 += per_b) {
        const int bn = batch - b0 < per_b ? batch - b0 : per_b;
        for (int m0 = 0; m0 < M; m0 += per_m) {
            const int mn = M - m0 < per_m ? M - m0 : per_m;
            const char *a = (const char *)A + ((size_t)b0 * strideA + (transA ? (size_t)m0 : (size_t)m0 * lda)) * es;
            const char *b = (const char *)B + (size_t)b0 * strideB * es;
            char *c = (char *)C + ((size_t)b0 * strideC + (size_t)m0 * ldc) * es;
            if (int rc = gemm_one(dtype, transA, transB, mn, N, K, a, lda, strideA, b, ldb, strideB, beta, c, ldc, strideC, bn,
                                  workspace, workspace_bytes, stream))
                return rc;
        }
    }
    return 0;
}

}  // extern "C"
