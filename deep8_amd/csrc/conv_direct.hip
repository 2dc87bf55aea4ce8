// Conv2d on an image of few channels (a network's first layer: 1 or 3 channels), forward and filter gradient.
//
// The patch rows of such an image (25, 27, 75, 147 elements) cannot be cut into 16-byte pieces of one tap's channels, which is
// what the tiled GEMM's patch loader fetches, and writing the patch matrix out moves the image FH * FW / stride^2 times.
// What a filter row covers is contiguous, though: FW * C elements of one image row.  A workgroup therefore keeps the image
// rows under a TR x TC block of output pixels in LDS, with zeros where they leave the image, and the matrix instructions'
// operands are read straight from there:
//   forward   D[oc][pixel] = w[oc][k] . patch[k][pixel]: k runs over FH runs of FW * C elements, each filled up to P pieces of
//             16 bytes.  The filter stays in registers (one fragment per pair of pieces), a patch fragment is 16 bytes at
//             pixel + run + piece, and what a run's last piece brings in from behind the run is cut off (not merely met by a
//             zero weight: it may be an infinity).  Channels are D's rows, so a lane holds four consecutive channels of a
//             pixel; in half two lanes exchange halves and store 16 bytes each.
//   gradient  D[oc][n] = dz^T[oc][pixel] . patch[pixel][n], n = (fy, fx, c) unpadded: a wave owns 32 n, a lane one n and 8 (4
//             in fp32) consecutive pixels of a row, i.e. strided single elements; dz is staged beside the image and read
//             transposed.  Waves beyond the n blocks take every other group of pixels and meet in LDS, workgroups leave
//             partial sums that conv_direct_reduce_kernel adds in a fixed order.
#include <cmath>

#include "conv_direct.h"
#include "gemm_tiled_kernel.h"

namespace d8 {

namespace {

struct DirectArgs {
    DirectShape s;
    const void *x, *w, *bias;
    void *z;
    float *ws;
    int relu, round_first;
    int K, run, P;              // FH * FW * C; FW * C; 16-byte pieces of a run
    int TR, TC, TCp;            // tile of output pixels; TC rounded up to what a lane's fragment covers
    int tiles_y, tiles_x, ntiles;
    int rows, pitch;            // image rows of a tile, and elements an image row takes in LDS
    int vec_x, vec_z;           // elements a staging access of the image / of z moves
    unsigned mg_chunks, mg_tc;  // ceil(2^32 / (pitch / vec_x)), ceil(2^32 / TC or TCp)
    unsigned mg_pieces;         // ceil(2^32 / P)
    int zeros;                  // forward: element of LDS from which 32 bytes may be zeros
    int kb, pixels_p;           // gradient: blocks of 32 n; pixels of a tile with its rows filled up, a multiple of a k group
};

// quotient by multiplication: exact for n, d < 2^16
__device__ __forceinline__ int quotient(int n, unsigned magic, int d) { return d == 1 ? n : (int)__umulhi((unsigned)n, magic); }

struct TileAt {
    int b, oy0, ox0, first, skip;  // first: image column (in elements) LDS column 0 holds; skip: LDS column of the tile's first patch
};

__device__ __forceinline__ TileAt tile_at(const DirectArgs &a, int t) {
    TileAt r;
    const int plane = a.tiles_y * a.tiles_x;
    r.b = t / plane;
    t -= r.b * plane;
    r.oy0 = t / a.tiles_x;
    r.ox0 = (t - r.oy0 * a.tiles_x) * a.TC;
    r.oy0 *= a.TR;
    const int lead = (r.ox0 * a.s.sx - a.s.pl) * a.s.C;
    r.skip = lead & (a.vec_x - 1);  // (vec_x is a power of two)
    r.first = lead - r.skip;
    return r;
}

// Piece `idx` of the tile's image rows: where it lies in LDS, and its elements (zeros outside the image: a piece lies
// inside or outside as a whole, because a row's length and `first` are multiples of it)
template <typename E, typename V>
__device__ __forceinline__ V image_piece(const DirectArgs &a, const TileAt &t, int idx, int total, int &dst) {
    constexpr int N = sizeof(V) / sizeof(E);
    const int per_row = a.pitch / N, r = quotient(idx, a.mg_chunks, per_row), col = (idx - r * per_row) * N;
    dst = r * a.pitch + col;
    const int iy = t.oy0 * a.s.sy - a.s.pt + r, el = t.first + col, row = a.s.IW * a.s.C;
    V v = {};
    if (idx < total && (unsigned)iy < (unsigned)a.s.IH && el >= 0 && el < row)
        v = *(const V *)((const E *)a.x + ((long)t.b * a.s.IH + iy) * row + el);
    return v;
}

template <typename E, typename V>
__device__ __forceinline__ void stage_image_as(const DirectArgs &a, const TileAt &t, E *img) {
    constexpr int N = sizeof(V) / sizeof(E), AHEAD = 4;
    const int total = a.rows * (a.pitch / N);
    for (int i = threadIdx.x; i < total; i += AHEAD * blockDim.x) {
        V v[AHEAD];
        int dst[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) v[u] = image_piece<E, V>(a, t, i + u * blockDim.x, total, dst[u]);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (i + u * (int)blockDim.x < total) *(V *)(img + dst[u]) = v[u];
    }
}

template <typename E>
__device__ __forceinline__ void stage_image(const DirectArgs &a, const TileAt &t, E *img) {
    if (a.vec_x * sizeof(E) == 16) stage_image_as<E, u32x4>(a, t, img);
    else if (sizeof(E) == 4 || a.vec_x == 2) stage_image_as<E, unsigned>(a, t, img);
    else stage_image_as<E, E>(a, t, img);
}

// 16 bytes from any element of LDS
template <typename E, bool ODD>
__device__ __forceinline__ u32x4 piece_at(const E *lds, int el) {
    u32x4 v;
    if constexpr (sizeof(E) == 4) {
        const unsigned *p = (const unsigned *)lds + el;
        v[0] = p[0], v[1] = p[1], v[2] = p[2], v[3] = p[3];
    } else {
        const unsigned *p = (const unsigned *)lds + (el >> 1);
        v[0] = p[0], v[1] = p[1], v[2] = p[2], v[3] = p[3];
        if constexpr (ODD) {
            const unsigned x = p[4], shift = (el & 1) * 16;
            v[0] = __builtin_amdgcn_alignbit(v[1], v[0], shift), v[1] = __builtin_amdgcn_alignbit(v[2], v[1], shift);
            v[2] = __builtin_amdgcn_alignbit(v[3], v[2], shift), v[3] = __builtin_amdgcn_alignbit(x, v[3], shift);
        }
    }
    return v;
}

// the bits of dword d of a piece whose first n elements count
template <typename E>
__device__ __forceinline__ unsigned first_mask(int n, int d) {
    if constexpr (sizeof(E) == 4) return n > d ? 0xffffffffu : 0u;
    else return n > 2 * d + 1 ? 0xffffffffu : n > 2 * d ? 0xffffu : 0u;
}

}  // namespace

// G: k groups (pairs of pieces) a wave keeps of the filter; NB: blocks of 32 channels per workgroup; ODD: half patches may
// start in the middle of a dword.  A workgroup walks every gridDim.x-th tile, its four waves every fourth block of 32 pixels.
// Bound by the store of z and the latency of a tile's image rows, which two workgroups and more per compute unit hide from each
// other; figures at conv_direct_forward.
template <typename E, int G, int NB, bool ODD, int RESIDENT = 2>
__global__ __launch_bounds__(256, RESIDENT) void conv_direct_forward_kernel(DirectArgs a) {
    typedef Elem<E> EL;
    typedef typename EL::Frag Frag;
    constexpr int EPV = 16 / sizeof(E), PITCH = 32 * EPV + EPV;  // a piece of 32 channels in LDS, and one to keep pieces in different banks
    constexpr bool LONG = sizeof(E) == 2 && G * NB > 11;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    __shared__ __attribute__((aligned(16))) float bias_s[NB * 32];
    __shared__ __attribute__((aligned(16))) E bias_e[NB * 32];
    E *lds = (E *)lds_bytes;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, half = lane >> 5;
    const int oc0 = blockIdx.y * (NB * 32), ocs = min(NB * 32, a.s.OC - oc0);

    const int pieces = a.s.FH * a.P, tail = a.run - (a.P - 1) * EPV;  // elements of a run's last piece
    unsigned tail_mask[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) tail_mask[d] = first_mask<E>(tail, d);
    // ---- the filter.  Half: piece by piece from memory, with zeros behind the last run and behind each run's end, into LDS in the
    // order of the fragments, and from there into registers (picked out of rows in LDS, five dwords and a shift each, they took
    // 4.7 us of a 7x7x3 stem's 15.5, so 3.8).  fp32: through LDS as rows of K elements, as they lie in memory.
    if constexpr (sizeof(E) == 2) {
        typedef E EVec __attribute__((ext_vector_type(EPV)));
        typedef EVec EVec_any __attribute__((aligned(sizeof(E))));
        constexpr int N = NB * 32 * 2 * G, IT = (N + 255) / 256;
        const E *const w = (const E *)a.w;
        const int total = a.s.OC * a.K;
        u32x4 v[IT];
        int moved[IT];  // elements that a piece was read before its place (the last ones of the filter, which nothing follows)
#pragma unroll
        for (int u = 0; u < IT; ++u) {
            moved[u] = 0;
            const int i = u * 256 + threadIdx.x, ch = i / (2 * G), p = i - ch * (2 * G), fy = quotient(p, a.mg_pieces, a.P), j = p - fy * a.P;
            // (channels past OC repeat the last: their results are not stored)
            const int at = (oc0 + min(ch, ocs - 1)) * a.K + fy * a.run + j * EPV;
            v[u] = (u32x4){0u, 0u, 0u, 0u};
            if (p < pieces && ch < NB * 32) {
                if (total >= EPV) {
                    const int from = min(at, total - EPV), shift = at - from;
                    u32x4 t = __builtin_bit_cast(u32x4, (EVec)*(const EVec_any *)(w + from));
                    v[u] = t, moved[u] = shift;
                } else {
                    E t[EPV] = {};
                    for (int e = 0; e < EPV; ++e)
                        if (at + e < total) t[e] = w[at + e];
                    v[u] = *(u32x4 *)t;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < IT; ++u) {
            const int i = u * 256 + threadIdx.x, ch = i / (2 * G), p = i - ch * (2 * G);
            if (moved[u]) {
                u32x4 t = v[u];
                const int dwords = moved[u] * (int)sizeof(E) / 4;
                if (dwords & 2) t = (u32x4){t[2], t[3], 0u, 0u};
                if (dwords & 1) t = (u32x4){t[1], t[2], t[3], 0u};
                if (sizeof(E) == 2 && (moved[u] & 1)) t = (u32x4){t[0] >> 16 | t[1] << 16, t[1] >> 16 | t[2] << 16, t[2] >> 16 | t[3] << 16, t[3] >> 16};
                v[u] = t;
            }
            const unsigned all = (p + 1) - quotient(p + 1, a.mg_pieces, a.P) * a.P ? 0xffffffffu : 0u;  // (not a run's last piece)
#pragma unroll
            for (int d = 0; d < 4; ++d) v[u][d] &= tail_mask[d] | all;
            if (ch < NB * 32) *(u32x4 *)(lds + ((ch >> 5) * (2 * G) + p) * PITCH + (ch & 31) * EPV) = v[u];
        }
    } else {
        const E *w = (const E *)a.w + (long)oc0 * a.K;
        const int n = ocs * a.K;
        if (((size_t)w & 15) == 0) {
            constexpr int LOADS = 5;  // in flight at a time
            for (int i = threadIdx.x * EPV; i + EPV <= n; i += LOADS * 256 * EPV) {
                u32x4 v[LOADS];
#pragma unroll
                for (int u = 0; u < LOADS; ++u)
                    if (i + u * 256 * EPV + EPV <= n) v[u] = *(const u32x4 *)(w + i + u * 256 * EPV);
#pragma unroll
                for (int u = 0; u < LOADS; ++u)
                    if (i + u * 256 * EPV + EPV <= n) *(u32x4 *)(lds + i + u * 256 * EPV) = v[u];
            }
            for (int i = n / EPV * EPV + threadIdx.x; i < n; i += 256) lds[i] = w[i];
        } else {
            for (int i = threadIdx.x; i < n; i += 256) lds[i] = w[i];
        }
    }
    if (threadIdx.x < NB * 32) {
        const E b = a.bias && (int)threadIdx.x < ocs ? ((const E *)a.bias)[oc0 + threadIdx.x] : (E)0.f;
        bias_e[threadIdx.x] = b, bias_s[threadIdx.x] = (float)b;
    }
    __syncthreads();
    Frag wf[NB][G];
    int koff[G];              // element offset of this lane's piece of each group from its pixel's first element
    unsigned some = 0, all = 0;  // bit g: the piece has elements of the patch (may be a run's last one) / only such
    auto piece_mask = [&](int d, int g) -> unsigned {
        return (tail_mask[d] & (unsigned)((int)(some << (31 - g)) >> 31)) | (unsigned)((int)(all << (31 - g)) >> 31);
    };
    int fy = half >= a.P ? 1 : 0, j = half - fy * a.P;  // piece 2 g + half is piece j of run fy
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const bool in = fy < a.s.FH, last = j == a.P - 1;
        koff[g] = in ? fy * a.s.dy * a.pitch + j * EPV : 0;
        const int woff = in ? fy * a.run + j * EPV : 0;
        some |= in ? 1u << g : 0u;
        all |= in && !last ? 1u << g : 0u;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if constexpr (sizeof(E) == 2) {
                wf[nb][g] = *(const Frag *)(lds + (nb * (2 * G) + 2 * g + half) * PITCH + l32 * EPV);
            } else {
                // (channels past OC repeat the last: their results are not stored)
                u32x4 v = piece_at<E, true>(lds, min(nb * 32 + l32, ocs - 1) * a.K + woff);
#pragma unroll
                for (int d = 0; d < 4; ++d) v[d] &= piece_mask(d, g);
                wf[nb][g] = __builtin_bit_cast(Frag, v);
            }
        }
        if (sizeof(E) == 4 && g % 3 == 2) __builtin_amdgcn_sched_barrier(0);  // (all reads at once would not fit the registers)
        j += 2;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (j >= a.P) j -= a.P, ++fy;
    }
    const int mine = pieces - half, zeros = a.zeros;
    const int blocks = (a.TR * a.TC + 31) / 32;
    const bool vec = a.s.OC % EPV == 0 && ((size_t)a.z & 15) == 0;
    for (int t = blockIdx.x; t < a.ntiles; t += gridDim.x) {
        const TileAt at = tile_at(a, t);
        __syncthreads();  // the filter's fragments have been read; every wave is done with the tile before
        stage_image<E>(a, at, lds);
        if (LONG && threadIdx.x < 8) ((unsigned *)(lds + zeros))[threadIdx.x] = 0u;
        __syncthreads();
        E *const z0 = (E *)a.z + (((long)at.b * a.s.OH + at.oy0) * a.s.OW + at.ox0) * a.s.OC + oc0;
        const int rows_here = min(a.TR, a.s.OH - at.oy0), cols_here = min(a.TC, a.s.OW - at.ox0);
        for (int blk = wave; blk < blocks; blk += 4) {
            const int q = blk * 32 + l32, qc = min(q, a.TR * a.TC - 1), r = quotient(qc, a.mg_tc, a.TC), c = qc - r * a.TC;
            const int base = r * a.s.sy * a.pitch + c * a.s.sx * a.s.C + at.skip;
            f32x16 acc[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[nb][i] = 0.f;
            // (masks built again for every block: hoisted, the four of each group take more registers than a long filter leaves)
            if constexpr (G * NB > 11) asm volatile("" : "+v"(some), "+v"(all));
#pragma unroll
            for (int g = 0; g < G; ++g) {
                u32x4 v;
                if constexpr (LONG) {  // (pieces past the last are read where zeros lie: one instruction a dword is left of the masks)
                    v = piece_at<E, ODD>(lds, 2 * g >= mine ? zeros : base + koff[g]);
                    const unsigned whole = (unsigned)((int)(all << (31 - g)) >> 31);
#pragma unroll
                    for (int d = 0; d < 4; ++d) v[d] &= tail_mask[d] | whole;
                } else {
                    v = piece_at<E, ODD>(lds, base + koff[g]);
#pragma unroll
                    for (int d = 0; d < 4; ++d) v[d] &= piece_mask(d, g);
                }
                const Frag f = __builtin_bit_cast(Frag, v);
#pragma unroll
                for (int e = 0; e < EL::MFMA_PER_FRAG; ++e)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) acc[nb] = EL::mfma(wf[nb][g], f, acc[nb], e);
            }
            // this lane's pixel, counted from the tile's first; -1: not one of z
            const int px = q < a.TR * a.TC && r < rows_here && c < cols_here ? r * a.s.OW + c : -1;
            E *const z = z0 + (long)px * a.s.OC;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                // register i of the block is channel 8 * (i / 4) + 4 * half + i % 4 of this lane's pixel
                typedef E E2 __attribute__((ext_vector_type(2)));
                E2 o[8];
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const int at_bias = nb * 32 + 8 * q4 + 4 * half;
                    f32x4 v = {acc[nb][4 * q4], acc[nb][4 * q4 + 1], acc[nb][4 * q4 + 2], acc[nb][4 * q4 + 3]};
                    if (sizeof(E) == 2 && a.round_first) {  // (the half sum of two halfs is their fp32 sum rounded to half)
                        o[2 * q4] = __builtin_convertvector(v.xy, E2), o[2 * q4 + 1] = __builtin_convertvector(v.zw, E2);
                        if (a.bias) {
                            typedef E E4 __attribute__((ext_vector_type(4)));
                            const E4 add = *(const E4 *)(bias_e + at_bias);
                            o[2 * q4] += add.xy, o[2 * q4 + 1] += add.zw;
                        }
                    } else {
                        if (a.bias) v += *(const f32x4 *)(bias_s + at_bias);
                        if (sizeof(E) == 4 && a.relu)
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[e] = !(v[e] > 0.f) ? 0.f : v[e];
                        o[2 * q4] = __builtin_convertvector(v.xy, E2), o[2 * q4 + 1] = __builtin_convertvector(v.zw, E2);
                    }
                    if (sizeof(E) == 2 && a.relu)
#pragma unroll
                        for (int e = 0; e < 2; ++e) o[2 * q4 + e] = __builtin_elementwise_max(o[2 * q4 + e], (E2){(E)0.f, (E)0.f});
                }
                if (vec) {
                    if constexpr (sizeof(E) == 4) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int n = nb * 32 + 8 * i + 4 * half;
                            if (px >= 0 && n < ocs) *(f32x4 *)(z + n) = (f32x4){(float)o[2 * i][0], (float)o[2 * i][1], (float)o[2 * i + 1][0], (float)o[2 * i + 1][1]};
                        }
                    } else {
                        // the lower half of the wave takes channels 16 i .. + 7 of its pixel, the upper 16 i + 8 .. + 15
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            u32x4 out;
#pragma unroll
                            for (int d = 0; d < 2; ++d) {
                                const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, o[4 * i + d]), __builtin_bit_cast(unsigned, o[4 * i + 2 + d]), false, false);
                                out[d] = s[0], out[d + 2] = s[1];
                            }
                            const int n = nb * 32 + 16 * i + 8 * half;
                            if (px >= 0 && n < ocs) *(u32x4 *)(z + n) = out;
                        }
                    }
                } else if (px >= 0) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int n = nb * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
                        if (n < ocs) z[n] = o[i >> 1][i & 1];
                    }
                }
            }
        }
    }
}

// Filter gradient.  blockDim = 64 * kb * (a power of two of waves that share the pixels of a tile).  The next tile's image
// rows and dz are fetched into registers while the present one is multiplied (where both move in 16-byte pieces and fit).
// What bounds it, by the counters of 16 x 224x224x3 -> 64, 7x7 stride 2 in half (25 us, of which the bytes would take 5 and the matrix
// instructions 2): 47 % of the waves' time are waits, for memory, LDS and the two barriers of a tile; 23 % vector instructions, 54 for a
// matrix instruction, which put patch elements that are read one by one (8 per 32 x 32 x 16 block) into fragments.  The LDS is busy 19 % of the
// time, the matrix pipe 7 %.
template <typename E, int NB>
__global__ __launch_bounds__(768) void conv_direct_grad_kernel(DirectArgs a) {
    typedef Elem<E> EL;
    typedef typename EL::Frag Frag;
    constexpr int EPV = 16 / sizeof(E);
    constexpr int LD = NB * 32 + (sizeof(E) == 4 ? 8 : NB == 2 ? 32 : 16);  // elements a pixel's channels take in LDS
    constexpr int PARTS = NB * 32 / EPV, IMG_AHEAD = 3, DZ_AHEAD = 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    E *dzs = (E *)lds_bytes, *img = dzs + a.pixels_p * LD;
    const int nt = blockDim.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5;
    const int sharers = (nt >> 6) / a.kb, kb = wave % a.kb, ps = wave / a.kb;
    const int oc0 = blockIdx.y * (NB * 32), ocs = min(NB * 32, a.s.OC - oc0);
    const int n = kb * 32 + l32, fy = n / a.run;
    const int noff = n < a.K ? fy * a.s.dy * a.pitch + (n - fy * a.run) : 0;
    const int step = a.s.sx * a.s.C;
    const E *gz = (const E *)a.w;
    const int img_total = a.rows * (a.pitch / EPV), dz_total = a.pixels_p * PARTS;
    const bool ahead = a.vec_x == EPV && a.vec_z == EPV && img_total <= IMG_AHEAD * nt && dz_total <= DZ_AHEAD * nt;

    // piece idx of dz: PARTS pieces per pixel, zeros for the pixels that fill a row up or lie outside z
    auto dz_at = [&](const TileAt &t, int px, int ch, const E *&src) -> bool {
        const int r = quotient(px, a.mg_tc, a.TCp), c = px - r * a.TCp, oy = t.oy0 + r, ox = t.ox0 + c;
        src = gz + (((long)t.b * a.s.OH + oy) * a.s.OW + ox) * a.s.OC + oc0 + ch;
        return r < a.TR && c < a.TC && oy < a.s.OH && ox < a.s.OW && ch < ocs;
    };
    u32x4 ri[IMG_AHEAD], rd[DZ_AHEAD];
    auto fetch = [&](const TileAt &t) {
#pragma unroll
        for (int u = 0; u < IMG_AHEAD; ++u) {
            int dst;
            ri[u] = image_piece<E, u32x4>(a, t, tid + u * nt, img_total, dst);
        }
#pragma unroll
        for (int u = 0; u < DZ_AHEAD; ++u) {
            const int i = tid + u * nt;
            const E *src;
            rd[u] = (u32x4){0, 0, 0, 0};
            if (i < dz_total && dz_at(t, i / PARTS, i % PARTS * EPV, src)) rd[u] = *(const u32x4 *)src;
        }
    };
    auto put = [&](const TileAt &t) {
#pragma unroll
        for (int u = 0; u < IMG_AHEAD; ++u) {
            const int i = tid + u * nt, per_row = a.pitch / EPV, r = quotient(i, a.mg_chunks, per_row);
            if (i < img_total) *(u32x4 *)(img + r * a.pitch + (i - r * per_row) * EPV) = ri[u];
        }
#pragma unroll
        for (int u = 0; u < DZ_AHEAD; ++u) {
            const int i = tid + u * nt;
            if (i < dz_total) *(u32x4 *)(dzs + i / PARTS * LD + i % PARTS * EPV) = rd[u];
        }
    };

    f32x16 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[nb][i] = 0.f;

    TileAt at = tile_at(a, blockIdx.x);  // (the grid has no more workgroups than there are tiles)
    if (ahead) fetch(at);
    for (int t = blockIdx.x; t < a.ntiles; t += gridDim.x) {
        __syncthreads();
        if (ahead) {
            put(at);
        } else {
            stage_image<E>(a, at, img);
            if (a.vec_z == EPV) {
                for (int i = tid; i < dz_total; i += nt) {
                    const E *src;
                    u32x4 v = {0, 0, 0, 0};
                    if (dz_at(at, i / PARTS, i % PARTS * EPV, src)) v = *(const u32x4 *)src;
                    *(u32x4 *)(dzs + i / PARTS * LD + i % PARTS * EPV) = v;
                }
            } else {
                for (int i = tid; i < a.pixels_p * (NB * 32); i += nt) {
                    const E *src;
                    const int px = i / (NB * 32), ch = i % (NB * 32);
                    dzs[px * LD + ch] = dz_at(at, px, ch, src) ? *src : (E)0.f;
                }
            }
        }
        __syncthreads();
        const int skip = at.skip, rows_here = min(a.TR, a.s.OH - at.oy0), cols_here = min(a.TC, a.s.OW - at.ox0);
        if (t + (int)gridDim.x < a.ntiles) {
            at = tile_at(a, t + gridDim.x);
            if (ahead) fetch(at);
        }
        for (int g = ps; g < a.pixels_p / (2 * EPV); g += sharers) {
            // this lane's EPV pixels: consecutive ones of a tile row (rows are filled up to a multiple of EPV)
            const int q = (2 * g + half) * EPV, r = quotient(q, a.mg_tc, a.TCp), c = q - r * a.TCp;
            const int valid = r < rows_here ? cols_here - c : 0;
            const E *p = img + (r < a.TR ? r * a.s.sy * a.pitch + c * step + skip : 0) + noff;
            Frag b;
            if constexpr (sizeof(E) == 4) {
#pragma unroll
                for (int e = 0; e < 4; ++e) b[e] = p[r < a.TR ? e * step : 0];
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) b[e] = p[r < a.TR ? e * step : 0];
            }
            u32x4 v = __builtin_bit_cast(u32x4, b);
#pragma unroll
            for (int d = 0; d < 4; ++d) v[d] &= first_mask<E>(valid, d);
            b = __builtin_bit_cast(Frag, v);
            Frag fa[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) fa[nb] = EL::read_tr(dzs + 2 * g * EPV * LD + EL::tr_offset(lane, LD, nb * 32), LD);
#pragma unroll
            for (int e = 0; e < EL::MFMA_PER_FRAG; ++e)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[nb] = EL::mfma(fa[nb], b, acc[nb], e);
        }
    }

    // ---- the waves that shared the pixels of an n block meet: the upper half hands its sums to the lower until one is left
    float *meet = (float *)lds_bytes;
    for (int s = sharers >> 1; s >= 1; s >>= 1) {
        __syncthreads();
        if (ps >= s && ps < 2 * s) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i = 0; i < 16; ++i) meet[(((ps - s) * a.kb + kb) * (NB * 16) + nb * 16 + i) * 64 + lane] = acc[nb][i];
        }
        __syncthreads();
        if (ps < s) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[nb][i] += meet[((ps * a.kb + kb) * (NB * 16) + nb * 16 + i) * 64 + lane];
        }
    }
    if (ps == 0 && n < a.K) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int oc = nb * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
                if (oc < ocs) a.ws[((long)blockIdx.x * a.s.OC + oc0 + oc) * a.K + n] = acc[nb][i];
            }
    }
}

// gw[i] = beta * gw[i] + the sum of `parts` partial sums ws[.][i]: 64 outputs per workgroup, 16 waves that take every
// sixteenth part each (sixteen loads in flight) and meet in LDS in wave order.
template <typename E>
__global__ __launch_bounds__(1024) void conv_direct_reduce_kernel(const float *ws, E *gw, int n, int parts, float beta) {
    __shared__ float met[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
    if (i < n) {
        for (int p = wave; p < parts; p += 256) {
            float t[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) t[u] = p + 16 * u < parts ? ws[(long)(p + 16 * u) * n + i] : 0.f;
#pragma unroll
            for (int u = 0; u < 16; ++u) sum[u & 3] += t[u];
        }
    }
    met[wave][lane] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    __syncthreads();
    if (wave == 0 && i < n) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < 16; ++w) v += met[w][lane];
        if (beta != 0.f) v += (float)gw[i];
        gw[i] = (E)v;
    }
}

// ---- host ------------------------------------------------------------------------------------------------------------
namespace {

constexpr int LDS_LIMIT = 64 * 1024;

unsigned magic_up(int d) { return d == 1 ? 0u : (unsigned)(((1UL << 32) + d - 1) / d); }

int pieces_of(int dtype, const DirectShape &s) {
    const int epv = 16 / (int)dtype_bytes(dtype);
    return s.FH * ceil_div((long)s.FW * s.C, epv);
}
int most_groups(int dtype) { return dtype == D8_FLOAT16 ? 11 : 21; }

// Everything of a launch but the pointers.  `grain`: pixels a tile row is filled up to (1 forward, a fragment's for the
// gradient); `pixels`: how many a tile may have; `px_bytes`: LDS of a pixel besides the image.  False where no tile fits.
bool plan_tiles(int dtype, const DirectShape &s, const void *x, int grain, int pixels, int px_bytes, int min_bytes, DirectArgs &a, size_t &lds) {
    const int es = (int)dtype_bytes(dtype), epv = 16 / es;
    memset(&a, 0, sizeof(a));
    a.s = s, a.x = x;
    a.run = s.FW * s.C, a.K = s.FH * a.run, a.P = ceil_div(a.run, epv);
    const long row = (long)s.IW * s.C;
    a.vec_x = row % epv == 0 && ((size_t)x & 15) == 0 ? epv : es == 2 && row % 2 == 0 && ((size_t)x & 3) == 0 ? 2 : 1;
    a.TC = ceil_div(s.OW, ceil_div(s.OW, pixels));
    a.TR = 1;
    auto fits = [&](int TR, int TC) {
        const int TCp = ceil_div(TC, grain) * grain, k_group = grain > 1 ? 2 * grain : 1;
        const long px = (long)ceil_div((long)TR * TCp, k_group) * k_group;
        const long rows = (long)(TR - 1) * s.sy + (long)(s.FH - 1) * s.dy + 1;
        // the last pixel's pieces, the part of a staging access before the first, and a dword for the odd start
        long pitch = (long)(TCp - 1) * s.sx * s.C + (long)a.P * epv + (a.vec_x - 1) + 2;
        const int unit = a.vec_x > 2 / es ? a.vec_x : 2;
        pitch = (pitch + unit - 1) / unit * unit;
        const long image = ((rows * pitch * es + 15) & ~15L) + 16, bytes = image + (grain > 1 ? px * px_bytes : 32);
        if (px > pixels + k_group || rows * pitch >= (1 << 15) || bytes > LDS_LIMIT) return false;
        a.TR = TR, a.TC = TC, a.TCp = TCp, a.pixels_p = (int)px, a.rows = (int)rows, a.pitch = (int)pitch, a.zeros = (int)(image / es), lds = (size_t)bytes;
        return true;
    };
    int TC = a.TC;
    while (!fits(1, TC)) {
        if (TC == 1) return false;
        TC = (TC + 1) / 2;
    }
    TC = ceil_div(s.OW, ceil_div(s.OW, TC));
    int TR = pixels / a.TCp;
    TR = TR < 1 ? 1 : TR > s.OH ? s.OH : TR;
    while (TR > 1 && !fits(TR, TC)) --TR;
    if (!fits(ceil_div(s.OH, ceil_div(s.OH, TR)), TC)) return false;
    a.tiles_y = ceil_div(s.OH, a.TR), a.tiles_x = ceil_div(s.OW, a.TC);
    const long tiles = (long)s.B * a.tiles_y * a.tiles_x;
    if (tiles >= (1L << 30)) return false;
    a.ntiles = (int)tiles;
    a.mg_chunks = magic_up(a.pitch / a.vec_x);
    a.mg_pieces = magic_up(a.P);
    a.mg_tc = magic_up(grain > 1 ? a.TCp : a.TC);
    if (lds < (size_t)min_bytes) lds = min_bytes;
    return lds <= (size_t)LDS_LIMIT;
}

template <typename E, int G, int NB>
int launch_forward(const DirectArgs &a, size_t lds, bool odd, hipStream_t stream) {
    const dim3 grid((unsigned)(a.ntiles < 2 * cu_count() ? a.ntiles : 2 * cu_count()), (unsigned)ceil_div(a.s.OC, NB * 32));
    // (fp32, ten groups: 135 registers let three workgroups share a compute unit; where there are more than that, the variant of 128
    // takes all of a fourth round off, 43 x 133x133x1 -> 64 7x7 166 -> 119 us; where not, the other one is up to 3 % faster)
    const bool many = sizeof(E) == 4 && G == 10 && (long)grid.x * grid.y > 3L * cu_count();
    if (sizeof(E) == 2 && odd) hipLaunchKernelGGL((conv_direct_forward_kernel<E, G, NB, sizeof(E) == 2>), grid, dim3(256), lds, stream, a);
    else if (many) hipLaunchKernelGGL((conv_direct_forward_kernel<E, G, NB, false, sizeof(E) == 4 && G == 10 ? 4 : 2>), grid, dim3(256), lds, stream, a);
    else hipLaunchKernelGGL((conv_direct_forward_kernel<E, G, NB, false>), grid, dim3(256), lds, stream, a);
    D8_LAUNCH_CHECK();
    return 0;
}

// channels per workgroup: the filter's fragments are what fills the registers (8 dwords a group for 64 channels)
int forward_channels(int dtype, const DirectShape &s) { return dtype == D8_FLOAT16 && s.OC > 32 ? 64 : 32; }

// k groups that the kernel keeps of them
int forward_groups(int dtype, const DirectShape &s) {
    const int groups = ceil_div(pieces_of(dtype, s), 2);
    return dtype == D8_FLOAT16 ? (groups <= 3 ? 3 : groups <= 5 ? 5 : 11) : (groups <= 5 ? 5 : groups <= 10 ? 10 : 21);
}

bool plan_forward(int dtype, const DirectShape &s, const void *x, DirectArgs &a, size_t &lds) {
    const int ch = forward_channels(dtype, s), filter = dtype == D8_FLOAT16 ? ch / 32 * 2 * forward_groups(dtype, s) * 33 * 16 : (ch * s.FH * s.FW * s.C + 8) * 4 + 16;
    return plan_tiles(dtype, s, x, 1, 256, 0, filter, a, lds);
}

int grad_waves(int kb) { return kb == 1 ? 8 : kb == 2 ? 8 : kb == 3 ? 6 : 2 * kb; }

bool plan_grad(int dtype, const DirectShape &s, const void *x, const void *gz, DirectArgs &a, size_t &lds) {
    const int es = (int)dtype_bytes(dtype), epv = 16 / es, nb = s.OC > 32 ? 2 : 1, kb = ceil_div((long)s.FH * s.FW * s.C, 32);
    if (kb > 6) return false;
    const int ld = nb * 32 + (es == 4 ? 8 : nb == 2 ? 32 : 16), meet = grad_waves(kb) / 2 * nb * 16 * 64 * 4;
    if (!plan_tiles(dtype, s, x, epv, es == 2 ? 224 : 128, ld * es, meet, a, lds)) return false;
    a.kb = kb;
    a.vec_z = s.OC % epv == 0 && ((size_t)gz & 15) == 0 ? epv : 1;
    return true;
}

}  // namespace

bool conv_direct_eligible(int dtype, const DirectShape &s) {
    if (dtype != D8_FLOAT16 && dtype != D8_FLOAT32) return false;
    // (the groups of output channels are the grid's second dimension)
    if (ceil_div(s.OC, 32) > 65535 || (long)s.OC * s.FH * s.FW * s.C > 0x7fffffffL) return false;
    if (s.dx != 1 || (long)s.FH * s.FW * s.C >= 4096 || pieces_of(dtype, s) > 2 * most_groups(dtype)) return false;
    DirectArgs a;
    size_t lds;
    return plan_forward(dtype, s, nullptr, a, lds) && plan_grad(dtype, s, nullptr, nullptr, a, lds);
}

// What the kernels take, fitted to 4776 calls on 2500 drawn layers (1 - 170 channels to 8 - 512, both types; half of the calls
// within 7 % of the estimate, nine tenths of the forward ones within 20 %), before the forward kernel's last changes, which
// took 4 % off it, 13 % with a bias: the patch matrix keeps a few layers that it would now be faster on.  Forward: the filter's way into registers, a
// tile's accesses to the image, a wave's blocks of 32 pixels (products and stores); the image's fragments are built again for
// every 64 (fp32: 32) output channels.
double conv_direct_forward_us(int dtype, const DirectShape &s, const void *x) {
    DirectArgs a;
    size_t lds;
    if (!plan_forward(dtype, s, x, a, lds)) return INFINITY;
    const bool half = dtype == D8_FLOAT16;
    const int es = half ? 2 : 4, ch = forward_channels(dtype, s), kept = forward_groups(dtype, s), cus = cu_count();
    const long wide = a.ntiles < 2 * cus ? a.ntiles : 2 * cus, wgs = wide * ceil_div(s.OC, ch), per_cu = (wgs + cus - 1) / cus;
    const double rounds = (double)((wgs + 2 * cus - 1) / (2 * cus)), tiles = (double)((a.ntiles + wide - 1) / wide);
    const double blocks = per_cu * tiles * ceil_div(ceil_div(a.TR * a.TC, 32), 4), accesses = rounds * tiles * ceil_div(a.rows * (a.pitch / a.vec_x), 256);
    const double filter = rounds * ch * a.K / 1000.0, single = s.OC % (16 / es) ? blocks * (ch / 32) : 0.0;
    if (half) return 4.2 + 0.04 * blocks * kept + 0.57 * blocks * (ch / 32) + 0.55 * single + 0.14 * accesses + 0.31 * filter;
    return 4.4 + 0.185 * blocks * kept + 0.5 * single + 0.15 * accesses + 0.48 * filter + 0.105e-6 * es * s.B * s.OH * s.OW * (double)s.OC;
}

static long grad_workgroups(const DirectArgs &a, const DirectShape &s) {
    const int oc_tiles = ceil_div(s.OC, s.OC > 32 ? 64 : 32);
    const long most = oc_tiles < cu_count() ? cu_count() / oc_tiles : 1;
    return most < a.ntiles ? most : a.ntiles;
}

size_t conv_direct_grad_bytes(int dtype, const DirectShape &s) {
    DirectArgs a;
    size_t lds;
    return plan_grad(dtype, s, nullptr, nullptr, a, lds) ? (size_t)grad_workgroups(a, s) * s.OC * a.K * sizeof(float) : 0;
}

// Gradient: per tile a wave's groups of pixels, and the accesses to dz and the image (single ones where a row or a pixel's
// channels are no multiple of 16 bytes, which do not overlap the products); then the partial sums.
double conv_direct_grad_us(int dtype, const DirectShape &s, const void *x, const void *gz, size_t ws_bytes) {
    DirectArgs a;
    size_t lds;
    if (!plan_grad(dtype, s, x, gz, a, lds)) return INFINITY;
    const bool half = dtype == D8_FLOAT16;
    const int epv = half ? 8 : 4, nb = s.OC > 32 ? 2 : 1, waves = grad_waves(a.kb), nt = 64 * waves;
    const size_t one = (size_t)s.OC * a.K * sizeof(float);
    long wgs = grad_workgroups(a, s);
    if (wgs > (long)(ws_bytes / one)) wgs = (long)(ws_bytes / one);
    if (wgs < 1) return INFINITY;
    const double tiles = (double)((a.ntiles + wgs - 1) / wgs), groups = ceil_div(a.pixels_p / (2 * epv), waves / a.kb) * nb;
    const double image = ceil_div(a.rows * (a.pitch / a.vec_x), nt), dz = ceil_div((long)a.pixels_p * nb * 32 / a.vec_z, nt);
    const bool ahead = a.vec_x == epv && a.vec_z == epv && a.rows * (a.pitch / epv) <= 3 * nt && a.pixels_p * (nb * 32 / epv) <= 4 * nt;
    const double staging = ahead ? (half ? 0.04 : 0.15) * (image + dz) : 0.115 * image + 0.225 * dz + (half ? 0.0 : 0.45);
    return 6.7 + tiles * ((half ? 1.2 + 0.147 * groups : 0.44 + 0.33 * groups) + staging) + 0.77e-6 * wgs * one;
}

// Half 16 x
// 224x224x3 -> 64, 7x7 stride 2 (K = 147): patch matrix + padded filter + product 81 -> 23 us (26 MB are stored: 5 us at a
// copy's rate; what the rest goes on is the filter's fragments and a block's chain of LDS reads, products and stores); fp32 64 x 28x28x1 -> 32,
// 5x5: patch matrix + product 18 -> 11 us.
// Then 19.7 and 7.3 us: the bias is read four values at a time, the filter's loads are in flight together, and masks are not kept for
// every group where the filter is long (two workgroups per compute unit need at most 256 registers; 295 gave 29.8 us).  A
// block of z is stored from registers, 16 bytes a lane: turned around through LDS for whole lines it took 21.2 and 7.5 us, and the
// LDS (8 - 16 KB) and registers kept workgroups off the compute unit (fp32 32 x 311x311x4 -> 64, 5x5 stride 4, 113 us, now 88).  Image
// rows of the next tile fetched into registers gave nothing beside several workgroups.  248 drawn layers, all three against
// none: with bias and ReLu 3142 us, now 2901; without 3098 us (125 layers more than 3 % slower than when z was not
// turned around), then 2853 (one).
// Now 17.0 and 7.25 us: in half, filter fragments that are read from LDS whole, one mask instruction a dword where the filter is
// long, and bias and ReLu on packed halfs, the bias read four values at a time (two at a time it is 18.2): 50 drawn half layers 10 %
// faster at the mean, 40 in fp32 2 %, none more than 2 % slower.  Two blocks at a time for a wave gave nothing (the
// instructions count, not their latencies) and took registers that workgroups need (32 x 163x145x3 -> 80 3x3 64 -> 98).
int conv_direct_forward(int dtype, const DirectShape &s, const void *x, const void *w, void *z, const void *bias, int relu,
                        int round_first, hipStream_t stream) {
    DirectArgs a;
    size_t lds;
    D8_REQUIRE(conv_direct_eligible(dtype, s) && plan_forward(dtype, s, x, a, lds), "conv_direct_forward: the layer does not fit");
    a.w = w, a.z = z, a.bias = bias, a.relu = relu, a.round_first = round_first;
    const int groups = forward_groups(dtype, s);
    if (dtype == D8_FLOAT32) {
        if (groups == 5) return launch_forward<float, 5, 1>(a, lds, false, stream);
        if (groups == 10) return launch_forward<float, 10, 1>(a, lds, false, stream);
        return launch_forward<float, 21, 1>(a, lds, false, stream);
    }
    // every patch starts at an even element of an even pitch
    const bool odd = (s.sx * s.C) % 2 != 0 || (s.pl * s.C) % 2 != 0;
    if (s.OC > 32) {
        if (groups == 3) return launch_forward<f16, 3, 2>(a, lds, odd, stream);
        if (groups == 5) return launch_forward<f16, 5, 2>(a, lds, odd, stream);
        return launch_forward<f16, 11, 2>(a, lds, odd, stream);
    }
    if (groups == 3) return launch_forward<f16, 3, 1>(a, lds, odd, stream);
    if (groups == 5) return launch_forward<f16, 5, 1>(a, lds, odd, stream);
    return launch_forward<f16, 11, 1>(a, lds, odd, stream);
}

// One workgroup per compute unit (10 waves for 147 columns): the partial sums are OC * K floats each, and a second workgroup
// would double what is written and read again.  In all, rounded down: with one workgroup more a compute unit holds two, and the
// others wait for it (half 18 x 221x173x3 -> 192, 7x7, three groups of channels: 3 x 86 workgroups 486 us, 3 x 85 258).  The layers above: 82 -> 28 us, 29 -> 13 us, both with the reduction.
bool conv_direct_grad_y(int dtype, const DirectShape &s, const void *x, void *gw, const void *gz, float beta, void *ws,
                        size_t ws_bytes, hipStream_t stream, int *rc) {
    DirectArgs a;
    size_t lds;
    if (!plan_grad(dtype, s, x, gz, a, lds)) return false;
    const int nb = s.OC > 32 ? 2 : 1, oc_tiles = ceil_div(s.OC, nb * 32);
    const size_t one = (size_t)s.OC * a.K * sizeof(float);
    long wgs = grad_workgroups(a, s);
    if (wgs > (long)(ws_bytes / one)) wgs = (long)(ws_bytes / one);
    if (wgs < 1 || ((size_t)ws & 3)) return false;
    a.w = gz, a.ws = (float *)ws;
    const dim3 grid((unsigned)wgs, (unsigned)oc_tiles), block(64 * grad_waves(a.kb));
    if (dtype == D8_FLOAT32) {
        if (nb == 2) hipLaunchKernelGGL((conv_direct_grad_kernel<float, 2>), grid, block, lds, stream, a);
        else hipLaunchKernelGGL((conv_direct_grad_kernel<float, 1>), grid, block, lds, stream, a);
    } else {
        if (nb == 2) hipLaunchKernelGGL((conv_direct_grad_kernel<f16, 2>), grid, block, lds, stream, a);
        else hipLaunchKernelGGL((conv_direct_grad_kernel<f16, 1>), grid, block, lds, stream, a);
    }
    auto launched = [&]() -> int {
        D8_LAUNCH_CHECK();
        return 0;
    };
    if ((*rc = launched())) return true;
    const int n = s.OC * a.K;
    if (dtype == D8_FLOAT32) hipLaunchKernelGGL((conv_direct_reduce_kernel<float>), dim3(ceil_div(n, 64)), dim3(1024), 0, stream, (const float *)ws, (float *)gw, n, (int)wgs, beta);
    else hipLaunchKernelGGL((conv_direct_reduce_kernel<f16>), dim3(ceil_div(n, 64)), dim3(1024), 0, stream, (const float *)ws, (f16 *)gw, n, (int)wgs, beta);
    *rc = launched();
    return true;
}

}  // namespace d8
