// Host side of the tiled GEMM kernels (gemm_tiled_kernel.h): eligibility, the choice of the translation unit that carries a
// product, the phase-record switch.
#include "gemm_tiled_kernel.h"

namespace d8 {

unsigned long long *phase_rec_buf = nullptr;
size_t phase_rec_bytes = 0;

void gemm_tiled_phase_record(void *records, size_t bytes) {
    phase_rec_buf = (unsigned long long *)records;
    phase_rec_bytes = records ? bytes : 0;
}

template <typename E>
static bool eligible(const GemmArgs &g, int transA, int transB, TiledRule rule) {
    constexpr long ES = sizeof(E), EPV = 16 / ES, BK = 128 / ES;
    const bool va = g.virt == VIRT_A_ROWS || g.virt == VIRT_A_CLASSES, vb = g.virt == VIRT_B_KROWS;
    if (g.virt == VIRT_A_CLASSES && (g.splits > 1 || g.ncls < 1 || g.ncls > MAX_CLASSES)) return false;
    if (va && (transA || g.K != g.pg.C)) return false;                       // a K step stays inside one tap
    if (vb && (!transA || transB || g.red != 1 || g.pg.C % EPV || g.N % g.pg.C)) return false;  // a piece stays inside one tap
    if ((va || vb) && (g.pg.bytes >= (1u << 31) || g.batch != 1)) return false;
    // (pixels past the last, in a last partial step, are told from the image by their 32-bit byte offset, which must not come
    // round to its start: one output pixel per image of 64 MiB, say)
    if (vb && ((g.K + BK - 1) / BK * BK - 1) / ((long)g.pg.OH * g.pg.OW) + 1 > (1L << 32) / (ES * g.pg.H * g.pg.W * g.pg.C)) return false;
    // byte offsets inside one operand (all summed products of it included) are 32-bit
    if (!va && ((g.red - 1) * g.sA + (long)(transA ? g.K : g.M) * g.lda) * ES >= (1L << 31)) return false;
    if (!vb && ((g.red - 1) * g.sB + (long)(transB ? g.N : g.K) * g.ldb) * ES >= (1L << 31)) return false;
    if (g.K < 1) return false;  // (a K below one K step is a lone partial step)
    if ((long)ceil_div(g.M, 128) * ceil_div(g.N, 128) > 0x7fffffffL || (long)g.batch * 128 > 65535) return false;
    if (g.virt == VIRT_NONE && rule == TILED_ANY) {
        if (in_pieces<E>(g, !transA, transB)) return true;
        // Rows may start at any element (EDGE_ANY).  But short products over many tiles are left to the any-shape kernel.  Its K step
        // is half as long, so it has half of the padding of a reduction of at most half a step (fp32 4032 x 2 x 2672, 9 summed:
        // 43 us against 63, 2624 x 13 x 3207 14.5 against 21.8; with fewer tiles, 8583 x 8 x 296, 9.0 against 7.5); and four of its
        // workgroups fit a compute unit, where two of the tiled kernels' do, which a third of a tile's time away from the last round
        // shows (fp32 4141 x 35 x 2349, 627 tiles, 21.9 and 27.6; 15 products of K <= 32 and 513 to 768 tiles 0.78 to 0.98 of the
        // tiled time, 32 of K <= 80 0.79 to 1.04, with up to 512 or 769 to 1024 tiles 0.95 to 1.2 at the median).  In half, whose
        // steps wait longer than they multiply, only A^T . B, whose tiles are turned on the way to the matrix instructions
        // (57 x 1480 x 8 x 139 19.5 against 25.3; 6 of K <= 32 with more than 1024 tiles 0.90 to 0.95, 13 of K <= 64 with 513 to 768 0.78
        // to 0.94).  A product that adds a bias or cuts at zero stays: the any-shape kernel does neither, and a pass over that
        // much output takes longer than the difference.
        const long tiles = (long)ceil_div(g.M, 128) * ceil_div(g.N, 128) * g.batch, cus = cu_count();
        const bool third_round = tiles > 2 * cus && tiles <= 3 * cus;
        if (!g.bias && !g.relu && (ES == 4 ? g.M > 64 && g.N > 64 && ((g.K <= 16 && 4 * tiles >= 3 * cus) || (g.K <= 80 && third_round))
                                           : transA && ((g.K <= 32 && tiles >= 4 * cus) || (g.K <= 64 && third_round)))) return false;
        // a thread's shift must hold for all products of a sum
        return g.red == 1 || ((g.sA | g.sB) * ES) % 4 == 0;
    }
    // one side may be shorter than any tile (a few rows against a wide matrix: the 64 x 128 / 128 x 64 tile
    // then reaches past it) when the other side fills a tile; a patch-matrix product may have both short
    if (g.M < 128 && g.N < 128 && (g.virt == VIRT_NONE || rule == TILED_WHOLE)) return false;
    if (rule == TILED_WHOLE && g.virt != VIRT_NONE && (g.K % BK || g.M < (g.virt == VIRT_A_CLASSES ? 128 : 64) || (vb && g.N < 64))) return false;
    // a 16-byte piece of an operand stored along K must lie wholly on one side of K
    if (g.K % BK && (!transA || transB) && g.K % EPV) return false;
    if (!va && (g.lda % EPV || g.sA % EPV)) return false;
    if (!vb && (g.ldb % EPV || g.sB % EPV)) return false;
    if (((size_t)g.A | (size_t)g.B) & 15) return false;
    if (transA && g.M % EPV) return false;
    if (!transB && g.N % EPV) return false;
    return true;
}

int gemm_tiled_k_step(int dtype) { return dtype == D8_FLOAT16 ? 64 : 32; }

bool gemm_tiled_eligible(int dtype, const GemmArgs &g, int transA, int transB, TiledRule rule) {
    if (dtype == D8_FLOAT64) return false;
    return dtype == D8_FLOAT16 ? eligible<f16>(g, transA, transB, rule) : eligible<float>(g, transA, transB, rule);
}

bool gemm_tiled_loose(int dtype, const GemmArgs &g, int transA, int transB) {
    if (g.virt != VIRT_NONE) return false;
    return dtype == D8_FLOAT16 ? !in_pieces<f16>(g, !transA, transB) : !in_pieces<float>(g, !transA, transB);
}

int gemm_tiled_launch(int dtype, const GemmArgs &g, int transA, int transB, hipStream_t stream) {
    if (g.virt == VIRT_NONE)
        return dtype == D8_FLOAT16 ? gemm_tiled_plain_f16(g, transA, transB, stream) : gemm_tiled_plain_f32(g, transA, transB, stream);
    return dtype == D8_FLOAT16 ? gemm_tiled_patch_f16(g, transB, stream) : gemm_tiled_patch_f32(g, transB, stream);
}

}  // namespace d8
