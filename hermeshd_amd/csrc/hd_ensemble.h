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
    long noff;     // offset of its noise block: 3 face families of 6*nface*nfb, then 6*npg*N volume
    long nfb;      // (nx+1)(ny+1)(nz+1)
    long cell0;    // first cell of the realization in the packed cell numbering
    int ntile;     // tiles of a plane
    unsigned int realization;
};

struct Launch {
    int zc;           // planes per item
    int xcd_chunk;    // 1: XCD-contiguous chunks of the work list
    int nwork;
};

template <int NB, int QP, int NQ, int RM, bool NZ>
__global__ __launch_bounds__(256, (sg::occupancy<NB, NQ>())) void k_ens_stage(
    const double* __restrict__ qin, const double* __restrict__ qn, double* __restrict__ qout,
    const EnsReal* __restrict__ reals, const int2* __restrict__ work, Launch L, Phys ph, StageParams sp,
    const float* __restrict__ noise, const unsigned long long* __restrict__ step, long nfloats) {
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
        const long fsz = 6L * NF * R.nfb;
        // the field of the current step: buffer (step & 1)
        const float* base = noise + ((*step & 1ull) ? nfloats : 0L) + R.noff;
        sp.noise[0] = base;
        sp.noise[1] = base + fsz;
        sp.noise[2] = base + 2 * fsz;
        sp.noise[3] = base + 3 * fsz;
        sp.nfb = R.nfb;
    }
    const int ch = wk.y / R.ntile, k0 = ch * L.zc, k1 = k0 + L.zc < g.nz ? k0 + L.zc : g.nz;
    const int part = __builtin_amdgcn_readfirstlane(((int)(threadIdx.x >> 6) + b) & 3);
    sg::stage_march<NB, QP, NQ, RM, NZ>(qin + R.qoff, qn + R.qoff, qout + R.qoff, g, ph, sp,
                                        (unsigned)(wk.y - ch * R.ntile), k0, k1, 0, part, R.cell0, sh);
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

// Noise of every realization for the current step: flat over all points;
// `pts` holds the prefix sums of the per-realization point counts
// (3*nface*nfb + npg*N), each rounded up to a whole number of 256-thread
// blocks so that a block lies in one realization (nreal+1 entries).
constexpr long NOISE_BLOCK = 256;
struct EnsNoise {
    unsigned long long seed;
    const unsigned long long* step;
    int ahead;       // draws step *step + ahead
    long nfloats;    // floats of one step's field; step s lives in buffer s & 1
    const double* dt;
    double eta_sd, zeta_sd, dVi, kap_f, kap_v;
    int nface, npg, nreal;
    const long* pts;
    const EnsReal* reals;
    float* out;
};

// One chunk of NOISE_BLOCK points (chunk b covers points b*NOISE_BLOCK ...).
__device__ __forceinline__ void ens_noise_chunk(const EnsNoise& np, long b) {
    // the chunk's realization: a search on its first point, uniform over the
    // block
    const long t0 = b * NOISE_BLOCK;
    if (t0 >= np.pts[np.nreal]) return;
    int lo = 0, hi = np.nreal;  // pts[lo] <= t0 < pts[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (np.pts[mid] <= t0) lo = mid; else hi = mid;
    }
    const EnsReal& R = np.reals[lo];
    const long u = t0 - np.pts[lo] + threadIdx.x;
    const long nf = (long)np.nface * R.nfb, nv = (long)np.npg * R.g.N;
    if (u >= 3 * nf + nv) return;  // the padding of the last block
    const double sq = sqrt(np.dVi / *np.dt);
    const unsigned long long st = *np.step + (unsigned long long)np.ahead;
    long id, count;
    unsigned int stream;
    float* out = np.out + ((st & 1ull) ? np.nfloats : 0L) + R.noff;
    double kap;
    if (u < 3 * nf) {
        const int d = (u >= nf) + (u >= 2 * nf);
        id = u - (long)d * nf;
        count = nf;
        stream = (unsigned int)(d + 1);
        out += (long)d * 6 * nf;
        kap = np.kap_f;
    } else {
        id = u - 3 * nf;
        count = nv;
        stream = 4u;
        out += 3L * 6 * nf;
        kap = np.kap_v;
    }
    double S[6];
    noise::stress(np.seed, R.realization, st, stream, (unsigned long long)id, np.eta_sd * sq * kap,
                  np.zeta_sd * sq * kap, S);
#pragma unroll
    for (int e = 0; e < 6; e++) out[(long)e * count + id] = (float)S[e];  // single precision, as k_noise
}

// Blocks stride over the chunks: one chunk per block when the grid covers
// them all, or a small grid (one block per CU) that stays beside a running
// stage kernel and draws the next step's field in the stage's shadow.
static __global__ __launch_bounds__(NOISE_BLOCK) void k_ens_noise(EnsNoise np) {
    const long nchunk = np.pts[np.nreal] / NOISE_BLOCK;
    for (long b = blockIdx.x; b < nchunk; b += gridDim.x) ens_noise_chunk(np, b);
}

}  // namespace ens
}  // namespace hd
