// hd_impl.h -- launch wrappers of one (nbasis, iquad, nQ, Riemann solver)
// configuration; included by the instantiation units only.
#pragma once
#include "hd_ctx.h"
#include "hd_stage.h"

#include <algorithm>

namespace hd {

template <int NB, int QP, int NQ, int RM>
struct Impl {
    static void limiter(hd_ctx* c, double* q, hipStream_t s) {
        // compile-time face tables and an exact early-out for cells no floor
        // can reach; the table-driven k_limiter stays for HD_LIMITER=table
        if (c->generic && c->table_limiter)
            hipLaunchKernelGGL((k_limiter<NB, QP>), dim3(blocks_for(c->N, 256)), dim3(256), 0, s, q, c->dtab, c->grid, c->lp);
        else
            hipLaunchKernelGGL((fz::k_limit<NB, QP>), dim3(blocks_for(c->N, 256)), dim3(256), 0, s, q, c->grid, c->lp);
    }
    static void start(hd_ctx* c, double* q, const CflEos& eos, double* dt, double* t, hipStream_t s) {
        // one block, and no second launch, while its two cells a thread cost less
        // than that (512 cells 30.9 us a step, 513 in three blocks 32.0)
        const long nblk = c->N <= 512 ? 1 : (c->N + 255) / 256;
        hipLaunchKernelGGL((fz::k_start<NB, QP>), dim3((unsigned)nblk), dim3(256), 0, s, q, c->grid, c->lp, eos,
                           1.01 * c->cfg.rh_floor, c->cfg.cflm, c->partial, dt, t);
        if (nblk > 1)
            hipLaunchKernelGGL(k_dt_finish, dim3(1), dim3(256), 0, s, q, c->grid, eos, c->partial, (int)nblk,
                               c->partial + nblk, c->cfg.cflm, dt, t);
    }
    static void faces(hd_ctx* c, const double* q, hipStream_t s) {
        const Grid& g = c->grid;
        long nfx = (long)(g.nx + 1) * g.ny * g.nz, nfy = (long)g.nx * (g.ny + 1) * g.nz, nfz = (long)g.nx * g.ny * (g.nz + 1);
        hipLaunchKernelGGL((k_face_flux<NB, QP, NQ, RM, 0>), dim3(blocks_for(nfx, 128)), dim3(128), 0, s, q, c->fl[0], c->dtab, g, c->ph, c->inflow);
        hipLaunchKernelGGL((k_face_flux<NB, QP, NQ, RM, 1>), dim3(blocks_for(nfy, 128)), dim3(128), 0, s, q, c->fl[1], c->dtab, g, c->ph, c->inflow);
        hipLaunchKernelGGL((k_face_flux<NB, QP, NQ, RM, 2>), dim3(blocks_for(nfz, 128)), dim3(128), 0, s, q, c->fl[2], c->dtab, g, c->ph, c->inflow);
    }
    static void cell(hd_ctx* c, const double* qin, const double* qn, double* qout, const StageParams& sp, hipStream_t s) {
        if constexpr (NQ == 13) {
            // one field per wave, 64 cells per workgroup (every wave of a
            // workgroup reaches its barriers: the grid is padded, not clipped)
            hipLaunchKernelGGL((k_cell13<NB, QP>), dim3(blocks_for(c->N, 64)), dim3(CELL13_WAVES * 64), 0, s, qin, qn,
                               qout, c->fl[0], c->fl[1], c->fl[2], c->dtab, c->grid, c->ph, sp);
            return;
        }
        hipLaunchKernelGGL((k_cell<NB, QP, NQ>), dim3(blocks_for(c->N, 128)), dim3(128), 0, s, qin, qn, qout, c->fl[0],
                           c->fl[1], c->fl[2], c->dtab, c->grid, c->ph, sp);
    }
    static void fused(hd_ctx* c, const double* qin, const double* qn, double* qout, const StageParams& sp, hipStream_t s) {
        const Grid& g = c->grid;
        const int planes = c->stage_planes == STAGE_AUTO ? sg::stage_planes<NB, NQ>(g, c->num_cus) : c->stage_planes;
        if constexpr (!(NB == 10 && NQ >= 11)) {  // its five waves would not have the registers
            if (planes < 0) {
                const unsigned tiles = (unsigned)sg::plane_tiles(g), n = tiles * (unsigned)g.nz, grid = (n + 7) / 8 * 8;
                if constexpr (NQ == 11) {
                    if (sp.noise[0]) {
                        hipLaunchKernelGGL((sg::k_stage_wide<NB, QP, NQ, RM, true>), dim3(grid), dim3(320), 0, s, qin,
                                           qn, qout, g, c->ph, sp, tiles, n);
                        return;
                    }
                }
                hipLaunchKernelGGL((sg::k_stage_wide<NB, QP, NQ, RM, false>), dim3(grid), dim3(320), 0, s, qin, qn,
                                   qout, g, c->ph, sp, tiles, n);
                return;
            }
        }
        if (planes > 0 && sg::stage_folds(g)) {
            const int zc = std::min(planes, g.nz);
            const unsigned tiles = (unsigned)sg::fold_tiles(g, zc);
            march<true>(c, qin, qn, qout, sp, (tiles + 7) / 8 * 8, tiles, zc, s);
        } else {
            const int zc = planes > 0 ? planes : 0;
            const long tiles = sg::plane_tiles(g);
            const long n = zc ? tiles * ((g.nz + zc - 1) / zc)
                              : std::min(tiles * g.nz, (long)c->num_cus * sg::occupancy<NB, NQ>());
            march<false>(c, qin, qn, qout, sp, (unsigned)((n + 7) / 8 * 8), (unsigned)tiles, zc, s);
        }
    }
    template <bool FOLD>
    static void march(hd_ctx* c, const double* qin, const double* qn, double* qout, const StageParams& sp, unsigned grid,
                      unsigned tiles, int zc, hipStream_t s) {
        if constexpr (NQ == 11) {
            if (sp.noise[0]) {
                hipLaunchKernelGGL((sg::k_stage<NB, QP, NQ, RM, true, FOLD>), dim3(grid), dim3(256), 0, s, qin, qn,
                                   qout, c->grid, c->ph, sp, tiles, zc);
                return;
            }
        }
        hipLaunchKernelGGL((sg::k_stage<NB, QP, NQ, RM, false, FOLD>), dim3(grid), dim3(256), 0, s, qin, qn, qout,
                           c->grid, c->ph, sp, tiles, zc);
    }
    static void ens_limit(hd_ens* e, double* q, hipStream_t s) {
        // a cell a thread of the largest realization, in a bounded launch (one
        // box of 160^3 cells in 64 workgroups: 353 us, in 16,000: 108)
        const long ny = std::min(e->nreal, 65535);
        const long nx = std::min((e->max_cells + 255) / 256, std::max(64L, 65536 / ny));
        hipLaunchKernelGGL((ens::k_ens_limit<NB, QP>), dim3((unsigned)nx, (unsigned)ny), dim3(256), 0, s, q, e->dreal,
                           e->nreal, e->lp);
    }
    static void ens_stage(hd_ens* e, const double* qin, const double* qn, double* qout, const StageParams& sp,
                          hipStream_t s) {
        if (e->launch.fold) ens_march<true>(e, qin, qn, qout, sp, s);
        else ens_march<false>(e, qin, qn, qout, sp, s);
    }
    template <bool FOLD>
    static void ens_march(hd_ens* e, const double* qin, const double* qn, double* qout, const StageParams& sp,
                          hipStream_t s) {
        if constexpr (NQ >= 11) {
            if (e->base.noise) {
                hipLaunchKernelGGL((ens::k_ens_stage<NB, QP, NQ, RM, true, FOLD>), dim3(e->grid), dim3(256), 0, s, qin,
                                   qn, qout, e->dreal, e->dwork, e->launch, e->ph, sp, e->noise);
                return;
            }
        }
        hipLaunchKernelGGL((ens::k_ens_stage<NB, QP, NQ, RM, false, FOLD>), dim3(e->grid), dim3(256), 0, s, qin, qn,
                           qout, e->dreal, e->dwork, e->launch, e->ph, sp, e->noise);
    }
    // defined in hd_impl_vjp.h; the units that include it instantiate it
    // there, and hd_k4_vjp.hip holds the nbasis 4 instances, so that those
    // compile with the default scheduler while hd_k4.hip takes another
    static void stage_vjp(hd_ctx* c, const double* q, const double* lam, double* lam_in, const adj::AdjParams& ap,
                          hipStream_t s);
    static Ops ops() {
        // no ensembles of the 13-moment model; its transpose is split on periodic grids
        if constexpr (NQ == 13) return Ops{&limiter, &start, &faces, &cell, &fused, nullptr, nullptr, &stage_vjp};
        else return Ops{&limiter, &start, &faces, &cell, &fused, &ens_limit, &ens_stage, &stage_vjp};
    }
};

template <int NB, int QP, int NQ>
bool pick_rm(int rm, Ops* o) {
    switch (rm) {
        case RIEMANN_CENTRAL: *o = Impl<NB, QP, NQ, RIEMANN_CENTRAL>::ops(); return true;
        case RIEMANN_HLLC: *o = Impl<NB, QP, NQ, RIEMANN_HLLC>::ops(); return true;
        case RIEMANN_ROE: *o = Impl<NB, QP, NQ, RIEMANN_ROE>::ops(); return true;
    }
    return false;
}

}  // namespace hd
