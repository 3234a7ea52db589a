// hd_ensemble.h -- many independent realizations of one configuration, on
// boxes of different sizes, advanced by one launch per RK stage.
//
// The reference runs one realization per process (src/main.f90 time loop,
// src/random.f90 noise); here the realizations' states are packed back to
// back, each in the reference layout Q(nx,ny,nz,nQ,nbasis), and the marching
// stage kernel (hd_stage.h) takes a list of (realization, tile, planes) items,
// one a workgroup.  With `xcd_chunk` each XCD takes a contiguous eighth of the
// list, so that a realization's tiles share one L2 (workgroup b runs on XCD
// b mod 8).
// Noise is drawn per realization with the same counter layout as one
// context, keyed by the realization id, so results do not depend on the
// schedule.
#pragma once
#include "hd_noise.h"
#include "hd_stage.h"

namespace hd {
namespace ens {

struct EnsReal {
    Grid g;
    long qoff;     // offset of the realization's state in a packed array (doubles)
    long noff;     // offset of its noise block: 3 face families of 3*nface*nfb, then 6*npg*N volume
    long nfb;      // (nx+1)(ny+1)(nz+1)
    long cell0;    // first cell of the realization in the packed cell numbering
    int ntile;     // tiles of a plane
    unsigned int realization;
};

struct Launch {
    int zc;           // planes per item
    int fold;         // items are tiles of segments of zc planes (sg::Rows)
    int xcd_chunk;    // 1: XCD-contiguous chunks of the work list
    int nwork;
};

template <int NB, int QP, int NQ, int RM, bool NZ, bool FOLD>
__global__ __launch_bounds__(256, (sg::occupancy<NB, NQ>())) void k_ens_stage(
    const double* __restrict__ qin, const double* __restrict__ qn, double* __restrict__ qout,
    const EnsReal* __restrict__ reals, const int2* __restrict__ work, Launch L, Phys ph, StageParams sp,
    const float* __restrict__ noise) {
    constexpr int NF = QP * QP;
    __shared__ double lds[sg::lds_doubles<NB, NQ>()];
    __shared__ int flags[2];
    const int b = (int)(blockIdx.x >> 3);
    const int t = L.xcd_chunk ? (int)(blockIdx.x & 7u) * (int)(gridDim.x >> 3) + b : (int)blockIdx.x;
    if (t >= L.nwork) return;
    const sg::Shared sh = sg::share<NB, NQ>(lds, flags);
    const int2 wk = work[t];
    const EnsReal& R = reals[wk.x];
    const Grid g = R.g;
    if constexpr (NZ) {
        const long fsz = 3L * NF * R.nfb;
        const float* base = noise + R.noff;
        sp.noise[0] = base;
        sp.noise[1] = base + fsz;
        sp.noise[2] = base + 2 * fsz;
        sp.noise[3] = base + 3 * fsz;
        sp.nfb = R.nfb;
    }
    const int part = __builtin_amdgcn_readfirstlane(((int)(threadIdx.x >> 6) + b) & 3);
    if constexpr (FOLD) {
        const int zc = L.zc < g.nz ? L.zc : g.nz;
        sg::stage_march<NB, QP, NQ, RM, NZ, true>(qin + R.qoff, qn + R.qoff, qout + R.qoff, g, ph, sp, (unsigned)wk.y,
                                                  zc, 0, sg::fold_planes(g, (unsigned)wk.y, zc), 0, part, R.cell0, sh);
    } else {
        const int ch = wk.y / R.ntile, k0 = ch * L.zc, k1 = k0 + L.zc < g.nz ? k0 + L.zc : g.nz;
        sg::stage_march<NB, QP, NQ, RM, NZ, false>(qin + R.qoff, qn + R.qoff, qout + R.qoff, g, ph, sp,
                                                   (unsigned)(wk.y - ch * R.ntile), 0, k0, k1, 0, part, R.cell0, sh);
    }
}

// The limiter, a cell a thread: realizations along y of the grid.
template <int NB, int QP>
__global__ __launch_bounds__(256) void k_ens_limit(double* __restrict__ q, const EnsReal* __restrict__ reals, int nreal,
                                                   LimParams lp) {
    for (int r = blockIdx.y; r < nreal; r += gridDim.y) {
        const EnsReal& R = reals[r];
        double* qr = q + R.qoff;
        const long N = R.g.N;
        const int nQ = R.g.nQ;
        for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < N; c += (long)gridDim.x * blockDim.x) {
            double m[5][NB];
#pragma unroll
            for (int i = 0; i < NB; i++)
#pragma unroll
                for (int f = 0; f < 5; f++) m[f][i] = qr[((long)i * nQ + f) * N + c];
            if (fz::limit_cell<NB, QP, 5>(m, lp)) {
#pragma unroll
                for (int i = 0; i < NB; i++)
#pragma unroll
                    for (int f = 0; f < 5; f++) qr[((long)i * nQ + f) * N + c] = m[f][i];
            }
        }
    }
}

// Noise of every realization for the current step: flat over all points of
// the realizations' families (three of faces, nface*nfb points each, and
// npg*N volume points); `pts` holds the prefix sums of the families' counts,
// each rounded up to whole chunks of 256 points so that a chunk lies in one
// family (4*nreal+1 entries).
constexpr long NOISE_CHUNK = 256;
struct EnsNoise {
    unsigned long long seed;
    const unsigned long long* step;
    const double* dt;
    double eta_sd, zeta_sd, dVi, kap_f, kap_v;
    int nface, npg, nreal;
    const long* pts;
    const EnsReal* reals;
    float* out;
};

// Each block takes an equal run of chunks: the amplitude is worked out and the
// first family searched for once per block, not once per chunk.  The draw is
// bound by vector instructions, as the stages are, so it runs before them, on
// the whole device: beside them on a second stream, one block a CU, it slowed
// them by more than it saved (96 boxes of 16^3 cells, 96 of 24^3 and 64 of
// 32^3, one step: 5.7 ms beside the stages, 4.9 ms before them with the same
// draw, 4.7 ms with this one).
static __global__ __launch_bounds__(NOISE_CHUNK) void k_ens_noise(EnsNoise np) {
    const long nchunk = np.pts[4 * np.nreal] / NOISE_CHUNK;
    long b = nchunk * blockIdx.x / gridDim.x;
    const long b1 = nchunk * (blockIdx.x + 1) / gridDim.x;
    if (b >= b1) return;
    const double sq = sqrt(np.dVi / *np.dt);
    const double ef = np.eta_sd * sq * np.kap_f, zf = np.zeta_sd * sq * np.kap_f;
    const double ev = np.eta_sd * sq * np.kap_v, zv = np.zeta_sd * sq * np.kap_v;
    const unsigned long long st = *np.step;
    int s = 0, hi = 4 * np.nreal;  // pts[s] <= the chunk's first point < pts[hi]
    while (hi - s > 1) {
        const int mid = (s + hi) >> 1;
        if (np.pts[mid] <= b * NOISE_CHUNK) s = mid; else hi = mid;
    }
    while (b < b1) {
        const EnsReal& R = np.reals[s >> 2];
        const int fam = s & 3;
        const long nf = (long)np.nface * R.nfb, nv = (long)np.npg * R.g.N, count = fam < 3 ? nf : nv;
        const long p0 = np.pts[s], p1 = np.pts[s + 1];
        const long e = b1 < p1 / NOISE_CHUNK ? b1 : p1 / NOISE_CHUNK;
        float* const out = np.out + R.noff + (long)fam * 3 * nf;
        const double ae = fam < 3 ? ef : ev, az = fam < 3 ? zf : zv;
        const unsigned realization = R.realization;
        for (; b < e; b++) {
            const long id = b * NOISE_CHUNK - p0 + threadIdx.x;
            if (id < count) noise::draw(np.seed, realization, st, fam, id, count, ae, az, out);
        }
        s++;
    }
}

}  // namespace ens
}  // namespace hd
