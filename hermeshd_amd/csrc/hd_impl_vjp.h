// hd_impl_vjp.h -- the stage transpose of Impl, out of the class so that a
// unit can leave its instantiation to another (hd_k4_vjp.hip).
#pragma once
#include "hd_impl.h"

namespace hd {

template <int NB, int QP, int NQ, int RM>
void Impl<NB, QP, NQ, RM>::stage_vjp(hd_ctx* c, const double* q, const double* lam, double* lam_in,
                                     const adj::AdjParams& ap, hipStream_t s) {
    if constexpr (NQ == 13) {
        // periodic grids: the split transpose (a face point, then a volume
        // point a lane); bq2 exists only for those
        if (c->bq2[0]) {
            const Grid& g = c->grid;
            const unsigned nf = 3 * blocks_for(g.N, adj::face13_faces<QP>());
            hipLaunchKernelGGL((adj::k_face13_vjp<NB, QP, RM>), dim3((nf + 7) / 8 * 8), dim3(256), 0, s, q, lam,
                               c->fl[0], c->fl[1], c->fl[2], c->bq2[0], c->bq2[1], c->bq2[2], g, c->ph, ap);
            c->vjp_blocks = (int)blocks_for(c->N, adj::cell13_cells<QP>());
            hipLaunchKernelGGL((adj::k_cell13_vjp<NB, QP, RM>), dim3(c->vjp_blocks), dim3(adj::cell13_threads<QP>()),
                               0, s, q, lam, lam_in, c->fl[0], c->fl[1], c->fl[2], c->bq2[0], c->bq2[1], c->bq2[2],
                               c->dtab, g, c->ph, ap);
            return;
        }
    }
    if constexpr (QP == 2) {
        // A point a lane up to 7/8 of two rounds of the per-cell kernel's
        // workgroups (256 cells, one a CU); past that a lane that holds its
        // cell takes fewer steps in all.  nbasis 4, 11 fields: 21 us against
        // 41 (8,192 cells, the per-cell kernel split over four waves, which
        // this replaced), 133 against 133 (64,000, one round), 181 against 307
        // (92,160, split), but 585 against 469 (262,144).
        if (!c->fused_vjp && 4 * c->N <= 7 * 256L * c->num_cus) {
            c->vjp_blocks = (int)blocks_for(c->N, adj::kPointCells);
            hipLaunchKernelGGL((adj::k_points_vjp<NB, QP, NQ, RM>), dim3(c->vjp_blocks), dim3(512), 0, s, q, lam,
                               lam_in, c->dtab, c->grid, c->ph, ap);
            return;
        }
    } else {
        // small grids are latency-bound: spread each cell over four waves
        if constexpr (adj::split_fits<NB, NQ>()) {
            if (!c->fused_vjp && c->N <= adj::kSplitCells) {
                c->vjp_blocks = (int)blocks_for(c->N, 64);
                hipLaunchKernelGGL((adj::k_stage_vjp_split<NB, QP, NQ, RM>), dim3(c->vjp_blocks), dim3(256), 0,
                                   s, q, lam, lam_in, c->grid, c->ph, ap);
                return;
            }
        }
    }
    c->vjp_blocks = (int)blocks_for(c->N, 256);
    hipLaunchKernelGGL((adj::k_stage_vjp<NB, QP, NQ, RM>), dim3(c->vjp_blocks), dim3(256), 0, s, q, lam, lam_in,
                       c->grid, c->ph, ap);
}

}  // namespace hd
