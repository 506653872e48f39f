// svlg_explicit.hip -- CentralDifference with lumped mass, matrix-free, on the device.
//
// Replaces CentralDifference::Initialize / ComputeEffectiveForce / ComputeEffectiveStiffness
// / ComputeNewStep (RP/10-Integrators/02-CentralDifference/CentralDifference.cpp:36-71,
// 124-152, 206-231) driven by Linear::ComputeNewIncrement (RP/09-Algorithms/01-Linear/
// Linear.cpp:22-56) inside DynamicAnalysis::Analyze (RP/08-Analysis/02-Dynamic/
// DynamicAnalysis.cpp:25-64). With lumped mass and dashpot-only damping Keff is
// diagonal, so EigenSolver's LDL^T solve is the division dU_i = Feff_i / Keff_ii.
//
// Per step k (load sample k, displacements U_{k-1}, U_{k-2}):
//   Feff = (Fext(k) - Fint(U_{k-1})) + (M/dt^2 - C/2dt)(U_{k-1} - U_{k-2})
//   U_k  = U_{k-1} + Feff / (M/dt^2 + C/2dt)
// The three displacement vectors rotate through a ring so V and A (which need
// U_{k-2}) can be formed on demand with SVL's expressions.
#include <algorithm>
#include <cstring>
#include <iterator>
#include <memory>
#include <new>

#include "svlg_common.hpp"
#include "svlg_drm.hpp"
#include "svlg_support.hpp"
#include "svlg_elem.hpp"
#include "svlg_mfma.hpp"
#include "svlg_tiles.hpp"

namespace svlg {

int launch_fint_colored(Model &m, const double *U, double ftol, double *F);
int gather_free(Model &m, const double *dnode, double *dfree);
int record_positions(Model &m, int nrec, const int32_t *rec_dofs, std::vector<int32_t> &pos);
int scatter_free(Model &m, const double *dfree, double *dnode);

// keff = M/dt^2 + C/2dt, kforce = M/dt^2 - C/2dt per DOF (CentralDifference.cpp:64-70); dtv
// (per DOF, may be null) gives every DOF its own time step (independent batched meshes).
__global__ void k_cd_coeffs(int n, double dt0, const double *__restrict__ dtv, const double *__restrict__ M,
                            const double *__restrict__ C, const int32_t *__restrict__ fdof,
                            double *__restrict__ keff, double *__restrict__ kforce, double *__restrict__ kinv,
                            int *__restrict__ singular) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (fdof[i] < 0) {
        keff[i] = 0.0;
        kforce[i] = 0.0;
        kinv[i] = 0.0;
        return;
    }
    const double dt = dtv ? dtv[i] : dt0;
    double k = 1.0 / dt / dt * M[i] + 1.0 / 2.0 / dt * C[i];
    keff[i] = k;
    kforce[i] = 1.0 / dt / dt * M[i] - 1.0 / 2.0 / dt * C[i];
    kinv[i] = k != 0.0 ? 1.0 / k : 0.0;
    if (!(k != 0.0)) atomicOr(singular, 1);
}

// Fext(k) = sum_l factor_l * (amp_l[k] * dir_l) by assignment per load, then summed in
// load order (Assembler.cpp:334-350, 485). One thread keeps that order.
__global__ void k_loads(int k, int nload, int nt, int ndim, int nldofs, const int32_t *__restrict__ ldofs,
                        const int32_t *__restrict__ node, const double *__restrict__ dir,
                        const double *__restrict__ factor, const double *__restrict__ series,
                        double *__restrict__ Fext) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    for (int i = 0; i < nldofs; ++i) Fext[ldofs[i]] = 0.0;
    for (int l = 0; l < nload; ++l) {
        double amp = (k >= 0 && k < nt) ? series[size_t(l) * nt + k] : 0.0;
        for (int c = 0; c < ndim; ++c) Fext[size_t(node[l]) * ndim + c] += factor[l] * (amp * dir[size_t(l) * ndim + c]);
    }
}

// U_next = U + (((Fext - F) + kforce (U - Up)) / keff); resets F for the next step.
__global__ void k_cd_update(int n, const double *__restrict__ U, const double *__restrict__ Up,
                            double *__restrict__ Unext, double *__restrict__ F, const double *__restrict__ Fext,
                            const double *__restrict__ keff, const double *__restrict__ kforce) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double k = keff[i];
    double fi = F[i];
    F[i] = 0.0;
    if (k == 0.0) {
        Unext[i] = 0.0;
        return;
    }
    double u = U[i];
    double feff = (Fext[i] - fi) + kforce[i] * (u - Up[i]);
    Unext[i] = u + feff / k;
}

// Feff = (Fext - F) + kforce (U - Up) on every node DOF (0 where keff = 0, the restrained
// DOFs); resets F for the next step (CentralDifference::ComputeEffectiveForce, :206-221).
__global__ void k_cd_feff(int n, const double *__restrict__ U, const double *__restrict__ Up, double *__restrict__ F,
                          const double *__restrict__ Fext, const double *__restrict__ keff,
                          const double *__restrict__ kforce, double *__restrict__ out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double fi = F[i];
    F[i] = 0.0;
    out[i] = keff[i] == 0.0 ? 0.0 : (Fext[i] - fi) + kforce[i] * (U[i] - Up[i]);
}

// U_next = U + dU on the free DOFs, 0 on the restrained ones (CentralDifference::ComputeNewStep,
// :137-148, with the algorithm's increment; support motion is added by its own kernel).
__global__ void k_cd_increment(int n, const double *__restrict__ U, const double *__restrict__ dU,
                               const double *__restrict__ keff, double *__restrict__ Unext) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Unext[i] = keff[i] == 0.0 ? 0.0 : U[i] + dU[i];
}

__global__ void k_record(int nrec, const int32_t *__restrict__ rec, const double *__restrict__ U,
                         double *__restrict__ out) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nrec) out[r] = U[rec[r]];
}

// Recording inside the step kernels (map null: none): the owner of a recorded DOF writes its new
// value into the history row of the step. A launch of its own per step cost 3 us of latency beside
// steps of 3 to 5 us on small models.
struct RecRef {
    const int32_t *map;     // [ndofn] column or -1
    const int32_t *tile;    // [ntiles] 1: the tile owns a recorded DOF
    double *hist;           // row of the launch's first step
    int nrec;
};

// Data that no kernel in flight writes: constant address space, so that a uniform index is a scalar
// load whose wait joins the tile bounds' (as ordinary memory it is a vector load with a full wait).
using const_i32 = const __attribute__((address_space(4))) int32_t;

__device__ __forceinline__ bool tile_records(const RecRef &r, int tile) {
    return r.map && ((const_i32 *)r.tile)[tile] != 0;
}

__device__ __forceinline__ void record_dof(const RecRef &r, size_t g, int row, double u) {
    const int c = r.map[g];
    if (c >= 0) r.hist[size_t(row) * r.nrec + c] = u;
}

// Sets (on = 1) or clears the columns of the recorded DOFs and the flags of the tiles that own them.
__global__ void k_rec_map(int nrec, const int32_t *__restrict__ rec, int on, int dim, int ntiles,
                          const int32_t *__restrict__ own_ptr, int32_t *__restrict__ map,
                          int32_t *__restrict__ tile) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrec || rec[r] < 0) return;
    map[rec[r]] = on ? r : -1;
    const int node = rec[r] / dim;
    int lo = 0, hi = ntiles;  // own_ptr[lo] <= node < own_ptr[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (own_ptr[mid] <= node) lo = mid;
        else hi = mid;
    }
    tile[lo] = on;
}

// U, V, A of the free DOFs in free order (CentralDifference::ComputeNewStep, :141-145, with U =
// U_{k-1}, Up = U_{k-2}, dU = U_k - U_{k-1}); null outputs are left out. Bandwidth-bound: one
// pass over the three vectors, then one copy per field that the caller asks for. The host loop
// it replaces read all three vectors back for every field: beside 500 steps of the 1.56M-DOF
// half-space (12.3 ms) the three fields took 25 ms, now 3.
__global__ void k_cd_state(int n, double dt0, const double *__restrict__ dtv, int moved,
                           const int32_t *__restrict__ fdof, const double *__restrict__ u0,
                           const double *__restrict__ u1, const double *__restrict__ u2, double *__restrict__ U,
                           double *__restrict__ V, double *__restrict__ A) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int f = fdof[i];
    if (f < 0) return;
    const double dt = dtv ? dtv[i] : dt0;
    const double a = u0[i], b = u1[i], c = u2[i];
    if (U) U[f] = a;
    if (V) V[f] = moved ? 1.0 / 2.0 / dt * (a - c) : 0.0;
    if (A) A[f] = moved ? 1.0 / dt / dt * (((a - b) - b) + c) : 0.0;
}

// Arguments of the fused step kernel.
struct FusedArgs {
    const int32_t *own_ptr, *nplain, *halo_ptr, *halo_node, *elem_ptr, *color_ptr;
    const uint16_t *lconn;
    const double *elam, *emu;
    const uint16_t *egeo;
    const double *geo;
    const double *X, *Ucur, *Uprev;
    double *Unext;
    const double *keff, *kforce, *kinv;
    const int32_t *nl_ptr, *nl_idx;
    const double *load_dir, *load_factor, *load_series;
    int load_nt, k;
    double th, ftol;
    int ntiles, ncolors, max_stage, max_own;
    const float *kmat;  // PATH 4: K_lambda, K_mu of the single element geometry
    const int *kdev;    // non-null: load sample = *kdev + k (graph replays advance *kdev)
    DrmRef drm;         // domain reduction forces of every step (F null: none)
    // Corner-slot step: fixed-stride tile data (TileSet::hpad ...; hstride 0: not built).
    const int32_t *hpad;
    const uint16_t *lcpad, *geopad;
    const double *lampad, *mupad;
    int hstride, estride;
    RecRef rec;
};

// Workgroup barrier with its own wait for this wave's LDS accesses. hipcc (ROCm 7.2, gfx950)
// leaves out the wait of a __syncthreads() that heads a loop whose back edge ends in LDS
// stores: the wave then arrives with its last stores still under way, and another wave's
// read-modify-write of the same word loses one of the two sums.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0), the other counters untouched
    __syncthreads();
}

__device__ __forceinline__ int color_of(const int32_t *__restrict__ cp, int i) {
    int c = 0;
    while (cp[c + 1] <= i) ++c;
    return c;
}

// One CentralDifference step for one node tile (one workgroup per tile):
//  1. stage U_{k-1} and X of owned + halo nodes in LDS;
//  2. every element touching an owned node computes its internal force (affine modal
//     form or the Gauss-point loop) and adds the owned corners into LDS, one element
//     color at a time (no two elements of a color share a node: race-free and the
//     summation order is fixed);
//  3. owned DOFs: U_k = U_{k-1} + ((Fext - Fint) + kforce (U_{k-1} - U_{k-2})) / keff,
//     with kforce == keff and Fext == 0 for the plain nodes at the head of the range.
// Workgroups b and b+8 run on the same XCD; tiles are handed out so that each XCD
// works on a contiguous range of neighbouring tiles (shared halo lines in its L2).
template <int DIM, int PATH>
__global__ __launch_bounds__(512) void k_cd_fused(FusedArgs a) {
    constexpr int NEN = Elem<DIM>::nen;
    constexpr int NB = 4;  // loads kept in flight per thread in the staging and update loops
    extern __shared__ double smem[];
    __shared__ int32_t cps[65];
    const int nt = a.ntiles;
    const int kstep = a.kdev ? *a.kdev + a.k : a.k;
    const int b = blockIdx.x, xcd = b & 7, j = b >> 3;
    const int q = nt >> 3, r = nt & 7;
    const int tile = xcd * q + min(xcd, r) + j;
    const int o0 = a.own_ptr[tile], nown = a.own_ptr[tile + 1] - o0;
    const int h0 = a.halo_ptr[tile], nh = a.halo_ptr[tile + 1] - h0;
    const int e0 = a.elem_ptr[tile], ne = a.elem_ptr[tile + 1] - e0;
    constexpr bool STAGE_X = PATH < 2;
    double *sU = smem;
    double *sX = smem + size_t(a.max_stage) * DIM;
    double *sF = smem + size_t((STAGE_X ? 2 : 1) * a.max_stage) * DIM;
    const int tid = threadIdx.x, B = blockDim.x;
    const int nU = nown * DIM, nH = nh * DIM;
    for (int c = tid; c <= a.ncolors; c += B) cps[c] = a.color_ptr[size_t(tile) * (a.ncolors + 1) + c];
    // Stage owned (contiguous) and halo (gathered) U, and X when needed, NB loads in flight.
    {
        const double *Ug = a.Ucur + size_t(o0) * DIM;
        const double *Xg = a.X + size_t(o0) * DIM;
        for (int base = 0; base < nU; base += NB * B) {
            double v[NB], w[NB];
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int i = base + k * B + tid;
                v[k] = i < nU ? Ug[i] : 0.0;
                if constexpr (STAGE_X) w[k] = i < nU ? Xg[i] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int i = base + k * B + tid;
                if (i < nU) {
                    sU[i] = v[k];
                    if constexpr (STAGE_X) sX[i] = w[k];
                    sF[i] = 0.0;
                }
            }
        }
        // Halo: one index load per node, then its DIM components.
        for (int base = 0; base < nh; base += NB * B) {
            size_t n[NB];
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int sl = base + k * B + tid;
                n[k] = sl < nh ? size_t(a.halo_node[h0 + sl]) * DIM : 0;
            }
            double v[NB][DIM], w[NB][DIM];
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int sl = base + k * B + tid;
#pragma unroll
                for (int c = 0; c < DIM; ++c) {
                    v[k][c] = sl < nh ? a.Ucur[n[k] + c] : 0.0;
                    if constexpr (STAGE_X) w[k][c] = sl < nh ? a.X[n[k] + c] : 0.0;
                }
            }
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int sl = base + k * B + tid;
                if (sl < nh) {
#pragma unroll
                    for (int c = 0; c < DIM; ++c) {
                        sU[nU + sl * DIM + c] = v[k][c];
                        if constexpr (STAGE_X) sX[nU + sl * DIM + c] = w[k][c];
                    }
                }
            }
        }
    }
    __syncthreads();
    const int32_t *cp = cps;
    for (int base = 0; base < ne; base += B) {
        const int i = base + tid;
        const bool valid = i < ne;
        double f[NEN][DIM];
        int lc[NEN];
        int mycol = -1;
        if (valid) {
            // Corner slots in one 8- or 16-byte load.
            if constexpr (NEN == 8) {
                const uint4 pk = *reinterpret_cast<const uint4 *>(a.lconn + size_t(e0 + i) * 8);
                const uint32_t w4[4] = {pk.x, pk.y, pk.z, pk.w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    lc[2 * c] = int(w4[c] & 0xffffu);
                    lc[2 * c + 1] = int(w4[c] >> 16);
                }
            } else {
                const uint2 pk = *reinterpret_cast<const uint2 *>(a.lconn + size_t(e0 + i) * 4);
                lc[0] = int(pk.x & 0xffffu);
                lc[1] = int(pk.x >> 16);
                lc[2] = int(pk.y & 0xffffu);
                lc[3] = int(pk.y >> 16);
            }
            const double lam = a.elam[e0 + i], mu = a.emu[e0 + i];
            double u[NEN][DIM];
#pragma unroll
            for (int c = 0; c < NEN; ++c)
#pragma unroll
                for (int d = 0; d < DIM; ++d) u[c][d] = sU[lc[c] * DIM + d];
            if constexpr (PATH >= 2) {
                const double *g = a.geo + size_t(a.egeo[e0 + i]) * (DIM * DIM);
                double Lam[DIM][DIM];
#pragma unroll
                for (int r2 = 0; r2 < DIM; ++r2)
#pragma unroll
                    for (int c2 = 0; c2 < DIM; ++c2) Lam[r2][c2] = g[r2 * DIM + c2];
                if constexpr (DIM == 3)
                    hexa_modal_force<PATH == 3>(Lam, lam, mu, u, f);
                else
                    quad_modal_force<PATH == 3>(Lam, lam, mu, u, f);
            } else {
                double x[NEN][DIM];
#pragma unroll
                for (int c = 0; c < NEN; ++c)
#pragma unroll
                    for (int d = 0; d < DIM; ++d) x[c][d] = sX[lc[c] * DIM + d];
                if constexpr (DIM == 3) {
                    if constexpr (PATH == 1)
                        hexa_affine_fint(x, u, lam, mu, f);
                    else
                        hexa_fint(x, u, lam, mu, f);
                } else {
                    if constexpr (PATH == 1)
                        quad_affine_fint(x, u, lam, mu, a.th, f);
                    else
                        quad_fint(x, u, lam, mu, a.th, f);
                }
            }
            mycol = color_of(cp, i);
        }
        const int clo = color_of(cp, base);
        const int chi = color_of(cp, min(base + B, ne) - 1);
        for (int c = clo; c <= chi; ++c) {
            lds_barrier();
            if (mycol == c) {
#pragma unroll
                for (int q2 = 0; q2 < NEN; ++q2)
                    if (lc[q2] < nown) {
#pragma unroll
                        for (int d = 0; d < DIM; ++d) {
                            double v = f[q2][d];
                            if (fabs(v) > a.ftol) sF[lc[q2] * DIM + d] += v;
                        }
                    }
            }
        }
    }
    // Owned DOFs: load U_{k-2} and keff with NB loads in flight, then update.
    const int npl = a.nplain[tile];
    const bool has_rec = tile_records(a.rec, tile);
    const size_t g0 = size_t(o0) * DIM;
    for (int base = 0; base < nU; base += NB * B) {
        double up[NB], kd[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            const int i = base + k * B + tid;
            up[k] = i < nU ? a.Uprev[g0 + i] : 0.0;
            kd[k] = i < nU ? a.keff[g0 + i] : 0.0;
        }
        if (base == 0) __syncthreads();
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            const int i = base + k * B + tid;
            if (i >= nU) continue;
            const int sl = i / DIM;
            const double u = sU[i], fi = sF[i];
            double un = 0.0;
            if (sl < npl) {
                un = u + ((0.0 - fi) + kd[k] * (u - up[k])) / kd[k];
            } else if (kd[k] != 0.0) {
                const int c = i - sl * DIM, node = o0 + sl;
                double fe = 0.0;
                for (int q2 = a.nl_ptr[node]; q2 < a.nl_ptr[node + 1]; ++q2) {
                    const int l = a.nl_idx[q2];
                    const double amp =
                        (kstep >= 0 && kstep < a.load_nt) ? a.load_series[size_t(l) * a.load_nt + kstep] : 0.0;
                    fe += a.load_factor[l] * (amp * a.load_dir[size_t(l) * DIM + c]);
                }
                const int ds = drm_slot(a.drm, node);
                if (ds >= 0) fe += drm_force(a.drm, ds, kstep, DIM, c);
                un = u + ((fe - fi) + a.kforce[g0 + i] * (u - up[k])) / kd[k];
            }
            a.Unext[g0 + i] = un;
            if (has_rec) record_dof(a.rec, g0 + i, 0, un);
        }
    }
}

// Corner-slot variant for meshes in which every (node, corner position) pair belongs
// to at most one element (conforming structured meshes): one thread per tile element
// and one thread per owned node, all tile elements in a single round. Each element
// writes its corner forces to the unique LDS slot (corner a, component c, node); each
// owned node then adds its NEN slots in corner order. No color phases; the corners go
// through the slot planes in NP passes of NEN / NP corners (same summation order as one
// pass, 1/NP of the slot LDS, one barrier per pass).
// MOC > 0: every tile owns at most MOC nodes; the slot planes then have the compile-time
// stride MOC + 1 with column MOC as the trash column, so that every slot address is one
// per-corner base plus an immediate offset.
// LATE: the update operands of a node (U_{k-2}, 1/keff) are loaded after the element
// phase instead of before the first barrier: 14 fewer registers live through the element
// step, more resident waves (on the Hexa8 table path, 86 -> 72 VGPRs).
// The update multiplies by the stored 1/keff (kinv) instead of dividing by keff: the
// diagonal solve as Eigen's LDL^T applies it (the inverse of D times the vector).
template <int DIM, int PATH, int MOC, bool LATE, int NP, bool PAD>
__device__ __forceinline__ void cd_corner_body(const FusedArgs &a) {
    constexpr int NEN = Elem<DIM>::nen;
    // Corner-slot planes per pass: the MFMA element step writes all corners at once.
    constexpr int NPASS = PATH == 4 ? 1 : NP, NH = NEN / NPASS;
    extern __shared__ double smem[];
    const int nt = a.ntiles;
    const int kstep = a.kdev ? *a.kdev + a.k : a.k;
    const int b = blockIdx.x, xcd = b & 7, j = b >> 3;
    const int q = nt >> 3, r = nt & 7;
    const int tile = xcd * q + min(xcd, r) + j;
    constexpr bool STAGE_X = PATH < 2;
    const int tid = threadIdx.x, B = blockDim.x;
    // Fixed-stride tile data: the halo node indices and the element data are loaded with
    // the tile index alone, in the same round trip as the tile bounds below.
    constexpr int NS = 2;  // strides of the one-pass staging
    // PAD: the fixed-stride copies exist (the host selects this instantiation only then).
    constexpr bool pad = PAD && !STAGE_X && PATH != 4;
    int hn[NS];  // halo node indices (raw: the address is formed where it is used)
    int lc[NEN];
    double lam = 0.0, mu = 0.0;
    int gid = 0;
    // Unconditional, in-bounds loads (indices clamped to the last entry; what lies past the
    // tile's counts is not used), unpacked only after the staging loads are issued.
    uint32_t pkw[NEN / 2];
    if constexpr (pad) {
        const int32_t *hp = a.hpad + size_t(tile) * a.hstride;
#pragma unroll
        for (int k = 0; k < NS; ++k) hn[k] = hp[min(k * B + tid, a.hstride - 1)];
        const size_t ei = size_t(tile) * a.estride + min(tid, a.estride - 1);
        if constexpr (NEN == 8) {
            const uint4 pk = *reinterpret_cast<const uint4 *>(a.lcpad + ei * 8);
            pkw[0] = pk.x;
            pkw[1] = pk.y;
            pkw[2] = pk.z;
            pkw[3] = pk.w;
        } else {
            const uint2 pk = *reinterpret_cast<const uint2 *>(a.lcpad + ei * 4);
            pkw[0] = pk.x;
            pkw[1] = pk.y;
        }
        lam = a.lampad[ei];
        mu = a.mupad[ei];
        if constexpr (PATH >= 2) gid = a.geopad[ei];
    }
    const int o0 = a.own_ptr[tile], nown = a.own_ptr[tile + 1] - o0;
    const int h0 = a.halo_ptr[tile], nh = a.halo_ptr[tile + 1] - h0;
    const int e0 = a.elem_ptr[tile], ne = a.elem_ptr[tile + 1] - e0;
    const int npl = a.nplain[tile];  // read with the tile bounds (one scalar round trip)
    const bool has_rec = tile_records(a.rec, tile);
    const int MO = MOC > 0 ? MOC + 1 : a.max_own;
    double *sU = smem;
    double *sX = smem + size_t(a.max_stage) * DIM;
    double *sIn = smem + size_t((STAGE_X ? 2 : 1) * a.max_stage) * DIM;  // [NH*DIM][MO]
    const int nU = nown * DIM, nH = nh * DIM;
    const size_t g0 = size_t(o0) * DIM;
    // Prefetch: update operands of this thread's node, element data of this thread's element.
    const bool has_node = tid < nown;
    double up[DIM], kd[DIM];
    if constexpr (!LATE)
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
            up[c] = has_node ? a.Uprev[g0 + size_t(tid) * DIM + c] : 0.0;
            kd[c] = has_node ? a.kinv[g0 + size_t(tid) * DIM + c] : 0.0;
        }
    const bool has_elem = PATH != 4 && tid < ne;
    if constexpr (!pad) {
        // (with PAD the element data are in flight and unpacked after the staging loads)
        if (has_elem) {
            if constexpr (NEN == 8) {
                const uint4 pk = *reinterpret_cast<const uint4 *>(a.lconn + size_t(e0 + tid) * 8);
                const uint32_t w4[4] = {pk.x, pk.y, pk.z, pk.w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    lc[2 * c] = int(w4[c] & 0xffffu);
                    lc[2 * c + 1] = int(w4[c] >> 16);
                }
            } else {
                const uint2 pk = *reinterpret_cast<const uint2 *>(a.lconn + size_t(e0 + tid) * 4);
                lc[0] = int(pk.x & 0xffffu);
                lc[1] = int(pk.x >> 16);
                lc[2] = int(pk.y & 0xffffu);
                lc[3] = int(pk.y >> 16);
            }
            lam = a.elam[e0 + tid];
            mu = a.emu[e0 + tid];
            if constexpr (PATH >= 2) gid = a.egeo[e0 + tid];
        } else {
#pragma unroll
            for (int c = 0; c < NEN; ++c) lc[c] = 0;
        }
    }
    // Stage U (and X), zero the corner slots.
    {
        const double *Ug = a.Ucur + g0;
        if constexpr (pad) {
            // One pass (the host checked that two strides cover the owned DOFs and the
            // halo): owned loads with the halo loads through the prefetched indices.
            double v[NS], hv[NS][DIM];
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int i = k * B + tid;
                v[k] = i < nU ? Ug[i] : 0.0;
#pragma unroll
                for (int c = 0; c < DIM; ++c) hv[k][c] = i < nh ? a.Ucur[size_t(hn[k]) * DIM + c] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const int i = k * B + tid;
                if (i < nU) sU[i] = v[k];
                if (i < nh)
#pragma unroll
                    for (int c = 0; c < DIM; ++c) sU[nU + i * DIM + c] = hv[k][c];
            }
#pragma unroll
            for (int c = 0; c < NEN / 2; ++c) {
                lc[2 * c] = int(pkw[c] & 0xffffu);
                lc[2 * c + 1] = int(pkw[c] >> 16);
            }
        } else if constexpr (!STAGE_X) {
            // One loop covers the owned DOFs and the halo nodes: every pass issues the halo
            // index loads and the owned loads together, then the halo loads, then the stores —
            // two dependent global round trips per pass instead of three.
            const int nrange = nU > nh ? nU : nh;
            for (int base = 0; base < nrange; base += NS * B) {
                size_t n[NS];
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    const int sl = base + k * B + tid;
                    n[k] = sl < nh ? size_t(a.halo_node[h0 + sl]) * DIM : 0;
                }
                double v[NS];
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    const int i = base + k * B + tid;
                    v[k] = i < nU ? Ug[i] : 0.0;
                }
                double hv[NS][DIM];
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    const int sl = base + k * B + tid;
#pragma unroll
                    for (int c = 0; c < DIM; ++c) hv[k][c] = sl < nh ? a.Ucur[n[k] + c] : 0.0;
                }
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    const int i = base + k * B + tid;
                    if (i < nU) sU[i] = v[k];
                    if (i < nh)
#pragma unroll
                        for (int c = 0; c < DIM; ++c) sU[nU + i * DIM + c] = hv[k][c];
                }
            }
        } else {
            // Coordinates staged too (Gauss-point and affine paths): owned values, then the
            // halo (one index load per node, then its DIM components).
            constexpr int NB = 4;  // loads kept in flight per thread
            const double *Xg = a.X + g0;
            for (int base = 0; base < nU; base += NB * B) {
                double v[NB], w[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int i = base + k * B + tid;
                    v[k] = i < nU ? Ug[i] : 0.0;
                    w[k] = i < nU ? Xg[i] : 0.0;
                }
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int i = base + k * B + tid;
                    if (i < nU) {
                        sU[i] = v[k];
                        sX[i] = w[k];
                    }
                }
            }
            for (int base = 0; base < nh; base += NB * B) {
                size_t n[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int sl = base + k * B + tid;
                    n[k] = sl < nh ? size_t(a.halo_node[h0 + sl]) * DIM : 0;
                }
                double v[NB][DIM], w[NB][DIM];
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int sl = base + k * B + tid;
#pragma unroll
                    for (int c = 0; c < DIM; ++c) {
                        v[k][c] = sl < nh ? a.Ucur[n[k] + c] : 0.0;
                        w[k][c] = sl < nh ? a.X[n[k] + c] : 0.0;
                    }
                }
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const int sl = base + k * B + tid;
                    if (sl < nh) {
#pragma unroll
                        for (int c = 0; c < DIM; ++c) {
                            sU[nU + sl * DIM + c] = v[k][c];
                            sX[nU + sl * DIM + c] = w[k][c];
                        }
                    }
                }
            }
        }
        for (int i = tid; i < NH * DIM * MO; i += B) sIn[i] = 0.0;
    }
    __syncthreads();
    double fi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) fi[d] = 0.0;
    if constexpr (PATH == 4) {
        // BF16 MFMA element step (single element geometry), FP64 slots and update.
        bf16x8 Ak[3];
        mfma_load_kblocks(a.kmat, Ak);
        mfma_hexa_elements<double>(a.lconn, a.elam, a.emu, e0, ne, nown, sU, sIn, MO, Ak, a.ftol);
        __syncthreads();
        if (has_node)
#pragma unroll
            for (int d = 0; d < DIM; ++d)
#pragma unroll
                for (int c = 0; c < NEN; ++c) fi[d] += sIn[(c * DIM + d) * MO + tid];
    } else {
        double f[NEN][DIM];
        if (has_elem) {
            double u[NEN][DIM];
#pragma unroll
            for (int c = 0; c < NEN; ++c)
#pragma unroll
                for (int d = 0; d < DIM; ++d) u[c][d] = sU[lc[c] * DIM + d];
            if constexpr (PATH == 5) {
                // FP32 element step (axis-aligned bricks): the modal force in single precision
                // from the FP64 staged displacements; slots, sums and the update stay FP64.
                static_assert(DIM == 3, "the FP32 element step is a Hexa8 path");
                const double *g = a.geo + size_t(gid) * 9;
                float Lf[3][3], uf[8][3], ff[8][3];
#pragma unroll
                for (int r2 = 0; r2 < 3; ++r2)
#pragma unroll
                    for (int c2 = 0; c2 < 3; ++c2) Lf[r2][c2] = float(g[r2 * 3 + c2]);
#pragma unroll
                for (int c = 0; c < 8; ++c)
#pragma unroll
                    for (int d = 0; d < 3; ++d) uf[c][d] = float(u[c][d]);
                hexa_modal_force<true, float>(Lf, float(lam), float(mu), uf, ff);
#pragma unroll
                for (int c = 0; c < 8; ++c)
#pragma unroll
                    for (int d = 0; d < 3; ++d) f[c][d] = double(ff[c][d]);
            } else if constexpr (PATH >= 2) {
                const double *g = a.geo + size_t(gid) * (DIM * DIM);
                double Lam[DIM][DIM];
#pragma unroll
                for (int r2 = 0; r2 < DIM; ++r2)
#pragma unroll
                    for (int c2 = 0; c2 < DIM; ++c2) Lam[r2][c2] = g[r2 * DIM + c2];
                if constexpr (DIM == 3)
                    hexa_modal_force<PATH == 3>(Lam, lam, mu, u, f);
                else
                    quad_modal_force<PATH == 3>(Lam, lam, mu, u, f);
            } else {
                double x[NEN][DIM];
#pragma unroll
                for (int c = 0; c < NEN; ++c)
#pragma unroll
                    for (int d = 0; d < DIM; ++d) x[c][d] = sX[lc[c] * DIM + d];
                if constexpr (DIM == 3) {
                    if constexpr (PATH == 1)
                        hexa_affine_fint(x, u, lam, mu, f);
                    else
                        hexa_fint(x, u, lam, mu, f);
                } else {
                    if constexpr (PATH == 1)
                        quad_affine_fint(x, u, lam, mu, a.th, f);
                    else
                        quad_fint(x, u, lam, mu, a.th, f);
                }
            }
        }
        // NPASS passes of NH corners through NH slot planes: elements write corners
        // pass*NH .. pass*NH+NH-1 (branch-free: corners of nodes this tile does not own go to
        // the trash cell after the slots), then every owned node adds its planes in corner
        // order and clears them for the next pass. Same summation order as one pass over
        // all corners, 1/NPASS of the LDS.
        const int trash = NH * DIM * MO;
        // LATE: the owned node's update operands are loaded at the start of the middle pass,
        // once half of the element forces are written out (their registers are free), so
        // that they arrive during the remaining passes.
#pragma unroll
        for (int pass = 0; pass < NPASS; ++pass) {
            if (pass > 0) __syncthreads();
            if constexpr (LATE)
                if (pass == NPASS / 2 && has_node)
#pragma unroll
                    for (int c = 0; c < DIM; ++c) {
                        up[c] = a.Uprev[g0 + size_t(tid) * DIM + c];
                        kd[c] = a.kinv[g0 + size_t(tid) * DIM + c];
                    }
            if (has_elem)
#pragma unroll
                for (int c = 0; c < NH; ++c) {
                    const int cc = pass * NH + c;
                    const bool own = lc[cc] < nown;
                    const int col = own ? lc[cc] : MOC;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        const double v = f[cc][d];
                        const double fv = fabs(v) > a.ftol ? v : 0.0;
                        if constexpr (MOC > 0)
                            sIn[(c * DIM + d) * MO + col] = fv;
                        else
                            sIn[own ? (c * DIM + d) * MO + lc[cc] : trash] = fv;
                    }
                }
            __syncthreads();
            if (has_node)
#pragma unroll
                for (int d = 0; d < DIM; ++d)
#pragma unroll
                    for (int c = 0; c < NH; ++c) {
                        double &slot = sIn[(c * DIM + d) * MO + tid];
                        fi[d] += slot;
                        if (pass + 1 < NPASS) slot = 0.0;
                    }
        }
    }
    if (!has_node) return;
    if constexpr (LATE && PATH == 4)
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
            up[c] = a.Uprev[g0 + size_t(tid) * DIM + c];
            kd[c] = a.kinv[g0 + size_t(tid) * DIM + c];
        }
    const int ds = tid >= npl ? drm_slot(a.drm, o0 + tid) : -1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const double u = sU[tid * DIM + d];
        const size_t g = g0 + size_t(tid) * DIM + d;
        double un = 0.0;
        if (tid < npl) {
            // Plain nodes: kforce = keff (no damping), so Feff / keff = (u - up) - fi / keff.
            un = u + ((u - up[d]) - fi[d] * kd[d]);
        } else if (kd[d] != 0.0) {
            const int node = o0 + tid;
            double fe = 0.0;
            for (int q2 = a.nl_ptr[node]; q2 < a.nl_ptr[node + 1]; ++q2) {
                const int l = a.nl_idx[q2];
                const double amp =
                    (kstep >= 0 && kstep < a.load_nt) ? a.load_series[size_t(l) * a.load_nt + kstep] : 0.0;
                fe += a.load_factor[l] * (amp * a.load_dir[size_t(l) * DIM + d]);
            }
            if (ds >= 0) fe += drm_force(a.drm, ds, kstep, DIM, d);
            un = u + ((fe - fi[d]) + a.kforce[g] * (u - up[d])) * kd[d];
        }
        a.Unext[g] = un;
        if (has_rec) record_dof(a.rec, g, 0, un);
    }
}

template <int DIM, int PATH, int MOC = 0, bool LATE = false, int NP = 2, bool PAD = false>
__global__ __launch_bounds__(512) void k_cd_corner(FusedArgs a) {
    cd_corner_body<DIM, PATH, MOC, LATE, NP, PAD>(a);
}

// Arguments of the multi-step kernel.
struct MultiArgs {
    const int32_t *cnt, *node;
    const uint16_t *econn, *ncor, *egeo;
    const double *elam, *emu, *geo, *X, *Ucur, *Uprev;
    double *out0, *out1, *out2;   // U_k, U_{k-1}, U_{k-2} of the owned nodes (null: not written)
    const double *kforce, *kinv;
    const int32_t *nl_ptr, *nl_idx;
    const double *load_dir, *load_factor, *load_series;
    int load_nt, k, nsteps;
    double th, ftol;
    int ntiles, depth, ns, ne, nu;
    DrmRef drm;
    RecRef rec;
};

// nsteps CentralDifference steps k .. k + nsteps - 1 for one node tile per workgroup, from one
// staging of the tile's nodes and nsteps rings of neighbours: step t updates the nodes of the
// rings that the steps after it still need, so tiles recompute each other's border instead of
// meeting at a launch boundary (nsteps <= depth, or one tile that holds the whole mesh). Ring
// nodes are computed by several tiles, each with the same operations in the same order.
//
// Bound: models whose single step leaves the chip idle are bound by the launch and by the chain of
// dependent global round trips before the first element (4.3 us for 0.3 us of data on 40,602
// DOFs), models of many tiles by the bytes of the state; both are paid once per nsteps
// here, and what a step keeps is its own chain of two LDS round trips and two barriers.
// One thread is one element and one node of the tile, with the element's constants and the node's
// u, u_prev, 1/keff in registers over all the steps. Elements write their corner forces to
// planes indexed by the element (neighbouring lanes, neighbouring words: no bank conflicts, no
// slots to clear, no ownership test), and a node reads its at most one element per corner
// position through 16-bit indices, in corner order; column ne of the planes is zero.
template <int DIM, int PATH, int MAXB, int MAXE, bool WIDE>
__global__ __launch_bounds__(MAXB) __attribute__((amdgpu_waves_per_eu(WIDE ? 8 : 1))) void k_cd_multi(MultiArgs a) {
    constexpr int NEN = Elem<DIM>::nen;
    constexpr bool STAGE_X = PATH < 2;
    constexpr int MO = MAXE + 1;  // column MAXE: no element
    extern __shared__ double smem[];
    const int b = blockIdx.x, xcd = b & 7, j = b >> 3;
    const int q = a.ntiles >> 3, r8 = a.ntiles & 7;
    const int tile = xcd * q + min(xcd, r8) + j;
    const int tid = threadIdx.x, n = a.nsteps;
    // Scalar loads: as ordinary memory the counts cost a vector round trip at the head of every step.
    const_i32 *ncnt = (const_i32 *)(a.cnt + size_t(tile) * 2 * (a.depth + 1)), *ecnt = ncnt + a.depth + 1;
    double *sF = smem;  // [NEN * DIM][MO]
    double *sU = sF + NEN * DIM * MO;
    double *sX = sU + size_t(a.ns) * DIM;
    // Everything addressed by the tile index goes out first, with indices clamped into the tile's rows.
    const int32_t nraw = a.node[size_t(tile) * a.ns + min(tid, a.ns - 1)];
    const size_t er = size_t(tile) * a.ne + min(tid, a.ne - 1);
    const size_t cr = size_t(tile) * a.nu + min(tid, a.nu - 1);
    uint32_t lcw[NEN / 2], ncw[NEN / 2];
    if constexpr (NEN == 8) {
        const uint4 x = *reinterpret_cast<const uint4 *>(a.econn + er * 8);
        const uint4 y = *reinterpret_cast<const uint4 *>(a.ncor + cr * 8);
        lcw[0] = x.x, lcw[1] = x.y, lcw[2] = x.z, lcw[3] = x.w;
        ncw[0] = y.x, ncw[1] = y.y, ncw[2] = y.z, ncw[3] = y.w;
    } else {
        const uint2 x = *reinterpret_cast<const uint2 *>(a.econn + er * 4);
        const uint2 y = *reinterpret_cast<const uint2 *>(a.ncor + cr * 4);
        lcw[0] = x.x, lcw[1] = x.y;
        ncw[0] = y.x, ncw[1] = y.y;
    }
    const double lam = a.elam[er], mu = a.emu[er];
    const int gid = PATH >= 2 ? int(a.egeo[er]) : 0;
    const int nown = ncnt[0];
    const bool staged = tid < ncnt[min(n, a.depth)];
    const int node = nraw & INT32_MAX;
    const bool special = nraw < 0;
    const size_t g = size_t(node) * DIM;
    double u[DIM], up[DIM], kd[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        u[d] = staged ? a.Ucur[g + d] : 0.0;
        up[d] = staged ? a.Uprev[g + d] : 0.0;
        kd[d] = staged ? a.kinv[g + d] : 0.0;
    }
    int q0 = 0, q1 = 0, ds = -1;
    if (staged && special) {
        q0 = a.nl_ptr[node];
        q1 = a.nl_ptr[node + 1];
        ds = drm_slot(a.drm, node);
    }
    if (staged) {
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            sU[tid * DIM + d] = u[d];
            if constexpr (STAGE_X) sX[tid * DIM + d] = a.X[g + d];
        }
    }
    if (tid < NEN * DIM) sF[tid * MO + MAXE] = 0.0;
    // Few tiles: the node's first load stays in registers, so that a step waits for one load of
    // its sample, in flight during the element phase (further loads are read in the step).
    double f0 = 0.0, d0[DIM], kf[DIM];
    const double *ser = nullptr;
#pragma unroll
    for (int d = 0; d < DIM; ++d) d0[d] = 0.0;
    if constexpr (!WIDE)
#pragma unroll
        for (int d = 0; d < DIM; ++d) kf[d] = (staged && special) ? a.kforce[g + d] : 0.0;
    if constexpr (!WIDE)
        if (q1 > q0) {
            const int l = a.nl_idx[q0];
            f0 = a.load_factor[l];
            ser = a.load_series + size_t(l) * a.load_nt;
#pragma unroll
            for (int d = 0; d < DIM; ++d) d0[d] = a.load_dir[size_t(l) * DIM + d];
            ++q0;
        }
    int rc[DIM];
    if constexpr (!WIDE)
#pragma unroll
        for (int d = 0; d < DIM; ++d) rc[d] = (a.rec.map && tid < nown) ? a.rec.map[g + d] : -1;
    const bool rec = WIDE && tile_records(a.rec, tile) && tid < nown;
    int lc[NEN];
#pragma unroll
    for (int c = 0; c < NEN / 2; ++c) {
        lc[2 * c] = int(lcw[c] & 0xffffu) * DIM;
        lc[2 * c + 1] = int(lcw[c] >> 16) * DIM;
    }
    double Lam[DIM][DIM];
    if constexpr (PATH >= 2) {
        const double *gt = a.geo + size_t(gid) * (DIM * DIM);
#pragma unroll
        for (int x = 0; x < DIM; ++x)
#pragma unroll
            for (int y = 0; y < DIM; ++y) Lam[x][y] = gt[x * DIM + y];
    }
    int ee = ecnt[min(n - 1, a.depth - 1)], nn = ncnt[min(n - 1, a.depth)];
    // Every load above has arrived before the loop: a wait inside it would also wait for the
    // sample loads and history stores of the steps.
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    lds_barrier();
    for (int t = 0; t < n; ++t) {
        const int left = n - 1 - t, k = a.k + t;
        // The next step's counts, a step ahead.
        const int nl = max(left - 1, 0), een = ecnt[min(nl, a.depth - 1)], nnn = ncnt[min(nl, a.depth)];
        const bool live = k >= 0 && k < a.load_nt;
        double amp = 0.0, dr[DIM];
        if constexpr (!WIDE) {
            if (ser && live) amp = ser[k];
#pragma unroll
            for (int d = 0; d < DIM; ++d) dr[d] = ds >= 0 ? drm_force(a.drm, ds, k, DIM, d) : 0.0;
        }
        if (tid < ee) {
            double v[NEN][DIM], f[NEN][DIM];
#pragma unroll
            for (int c = 0; c < NEN; ++c) {
                if constexpr (DIM == 2) {
                    const double2 w = *reinterpret_cast<const double2 *>(sU + lc[c]);
                    v[c][0] = w.x;
                    v[c][1] = w.y;
                } else {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) v[c][d] = sU[lc[c] + d];
                }
            }
            if constexpr (PATH >= 2) {
                if constexpr (DIM == 3)
                    hexa_modal_force<PATH == 3>(Lam, lam, mu, v, f);
                else
                    quad_modal_force<PATH == 3>(Lam, lam, mu, v, f);
            } else {
                double x[NEN][DIM];
#pragma unroll
                for (int c = 0; c < NEN; ++c)
#pragma unroll
                    for (int d = 0; d < DIM; ++d) x[c][d] = sX[lc[c] + d];
                if constexpr (DIM == 3) {
                    if constexpr (PATH == 1)
                        hexa_affine_fint(x, v, lam, mu, f);
                    else
                        hexa_fint(x, v, lam, mu, f);
                } else {
                    if constexpr (PATH == 1)
                        quad_affine_fint(x, v, lam, mu, a.th, f);
                    else
                        quad_fint(x, v, lam, mu, a.th, f);
                }
            }
#pragma unroll
            for (int c = 0; c < NEN; ++c)
#pragma unroll
                for (int d = 0; d < DIM; ++d) sF[(c * DIM + d) * MO + tid] = fabs(f[c][d]) > a.ftol ? f[c][d] : 0.0;
        }
        lds_barrier();
        if (tid < nn) {
            double fi[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) fi[d] = 0.0;
#pragma unroll
            for (int c = 0; c < NEN; ++c) {
                const int e = (c & 1) ? int(ncw[c / 2] >> 16) : int(ncw[c / 2] & 0xffffu);
#pragma unroll
                for (int d = 0; d < DIM; ++d) fi[d] += sF[(c * DIM + d) * MO + e];
            }
            double un[DIM];
            if (!special) {
#pragma unroll
                for (int d = 0; d < DIM; ++d) un[d] = u[d] + ((u[d] - up[d]) - fi[d] * kd[d]);
            } else {
                double fe[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) fe[d] = f0 * (amp * d0[d]);
                for (int x = q0; x < q1; ++x) {
                    const int l = a.nl_idx[x];
                    const double am = live ? a.load_series[size_t(l) * a.load_nt + k] : 0.0;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) fe[d] += a.load_factor[l] * (am * a.load_dir[size_t(l) * DIM + d]);
                }
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    if constexpr (WIDE) {
                        dr[d] = ds >= 0 ? drm_force(a.drm, ds, k, DIM, d) : 0.0;
                        kf[d] = a.kforce[g + d];
                    }
                    un[d] = kd[d] == 0.0
                                ? 0.0
                                : u[d] + ((fe[d] + dr[d] - fi[d]) + kf[d] * (u[d] - up[d])) * kd[d];
                }
            }
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                up[d] = u[d];
                u[d] = un[d];
            }
            if constexpr (DIM == 2) {
                *reinterpret_cast<double2 *>(sU + tid * 2) = make_double2(un[0], un[1]);
            } else {
#pragma unroll
                for (int d = 0; d < DIM; ++d) sU[tid * DIM + d] = un[d];
            }
            // The last steps leave their displacements as they are made (left = 2: U_{k-2}, ...).
            double *out = left == 0 ? a.out0 : left == 1 ? a.out1 : left == 2 ? a.out2 : nullptr;
            if (out && tid < nown)
#pragma unroll
                for (int d = 0; d < DIM; ++d) out[g + d] = un[d];
            if constexpr (WIDE) {
                if (rec)
#pragma unroll
                    for (int d = 0; d < DIM; ++d) record_dof(a.rec, g + d, t, un[d]);
            } else {
#pragma unroll
                for (int d = 0; d < DIM; ++d)
                    if (rc[d] >= 0) a.rec.hist[size_t(t) * a.rec.nrec + rc[d]] = un[d];
            }
        }
        ee = een;
        nn = nnn;
        lds_barrier();
    }
}

template <int DIM, int PATH>
static const void *fused_fn(bool corner) {
    return corner ? reinterpret_cast<const void *>(&k_cd_corner<DIM, PATH>)
                  : reinterpret_cast<const void *>(&k_cd_fused<DIM, PATH>);
}

// Corner passes of the corner-slot step (the slot planes hold NEN / passes corners): four on
// the compile-time stride Hexa8 paths, two elsewhere (one for the MFMA element step).
static int use_moc(const Model &m);
static int cd_passes(const Model &m) {
    if (m.elem_bf16) return 1;
    return m.ndim == 3 && use_moc(m) ? 4 : 2;
}

// Owned-node bound of the compile-time slot stride of the corner-slot step on axis-aligned
// meshes (0: the stride read from the tile set): 160 (the large default 3D tiles) for Hexa8, for Quad4
// 192 (the default above a million nodes) and 448 (covers the 400-node default).
static int use_moc(const Model &m) {
    if (m.variant != 3 || m.elem_bf16 || m.elem_path != 3) return 0;
    if (m.elem_fp32) return m.tiles.max_own <= 160 ? 160 : 0;
    const int mo = m.tiles.max_own;
    if (m.ndim == 3) return mo <= 160 ? 160 : 0;
    return mo <= 192 ? 192 : mo <= 448 ? 448 : 0;
}

static const void *moc_kernel(const Model &m) {
    const bool pad = m.tiles.hstride > 0;  // fixed-stride tile data built
    if (m.elem_fp32)
        return pad ? reinterpret_cast<const void *>(&k_cd_corner<3, 5, 160, true, 4, true>)
                   : reinterpret_cast<const void *>(&k_cd_corner<3, 5, 160, true, 4>);
    switch (m.ndim * 1000 + use_moc(m)) {
        case 3160:
            return pad ? reinterpret_cast<const void *>(&k_cd_corner<3, 3, 160, true, 4, true>)
                       : reinterpret_cast<const void *>(&k_cd_corner<3, 3, 160, true, 4>);
        case 2192:
            return pad ? reinterpret_cast<const void *>(&k_cd_corner<2, 3, 192, false, 2, true>)
                       : reinterpret_cast<const void *>(&k_cd_corner<2, 3, 192>);
        case 2448:
            return pad ? reinterpret_cast<const void *>(&k_cd_corner<2, 3, 448, false, 2, true>)
                       : reinterpret_cast<const void *>(&k_cd_corner<2, 3, 448>);
        default: return nullptr;
    }
}

static const void *fused_kernel(const Model &m) {
    const bool cr = m.variant == 3;
    if (m.elem_bf16) return reinterpret_cast<const void *>(&k_cd_corner<3, 4>);
    if (use_moc(m)) return moc_kernel(m);
    if (m.elem_fp32) return reinterpret_cast<const void *>(&k_cd_corner<3, 5>);
    if (m.ndim == 3)
        switch (m.elem_path) {
            case 3: return fused_fn<3, 3>(cr);
            case 2: return fused_fn<3, 2>(cr);
            case 1: return fused_fn<3, 1>(cr);
            default: return fused_fn<3, 0>(cr);
        }
    switch (m.elem_path) {
        case 3: return fused_fn<2, 3>(cr);
        case 2: return fused_fn<2, 2>(cr);
        case 1: return fused_fn<2, 1>(cr);
        default: return fused_fn<2, 0>(cr);
    }
}

int prepare_fused(Model &m) {
    if (m.variant != 1 && m.variant != 3) return 0;
    if (m.variant == 3) {
        // Staged U (and X unless the geometry table is used), the corner-slot planes of one
        // pass (half the corners; all of them for the MFMA element step) and the trash cell.
        const int staged = m.elem_path >= 2 ? 1 : 2;
        const int planes = m.nen / cd_passes(m);
        m.tiles.lds_bytes =
            use_moc(m) ? (size_t(staged) * m.tiles.max_stage * m.ndim + size_t(planes) * m.ndim * (use_moc(m) + 1)) *
                             sizeof(double)
                       : (size_t(staged) * m.tiles.max_stage * m.ndim + size_t(planes) * m.ndim * m.tiles.max_own + 1) *
                             sizeof(double);
    }
    SVLG_CHECK(m.tiles.block <= 512, "fused kernel block must be at most 512 threads");
    SVLG_CHECK(m.tiles.lds_bytes <= 160 * 1024, "node tile needs more than 160 KB of LDS; use smaller tiles");
    if (m.tiles.lds_bytes > 64 * 1024)
        SVLG_HIP(hipFuncSetAttribute(fused_kernel(m), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     int(m.tiles.lds_bytes)));
    return 0;
}

static int launch_fused(Model &m, int k, const double *Ucur, const double *Uprev, double *Unext,
                        const int *kdev = nullptr, const RecRef *rec = nullptr) {
    const TileSet &t = m.tiles;
    FusedArgs a;
    a.rec = rec ? *rec : RecRef{nullptr, nullptr, nullptr, 0};
    a.kdev = kdev;
    a.own_ptr = t.own_ptr.p;
    a.nplain = t.nplain.p;
    a.halo_ptr = t.halo_ptr.p;
    a.halo_node = t.halo_node.p;
    a.elem_ptr = t.elem_ptr.p;
    a.color_ptr = t.color_ptr.p;
    a.lconn = t.elem_lconn.p;
    a.elam = t.elem_lam.p;
    a.emu = t.elem_mu.p;
    a.X = m.X.p;
    a.Ucur = Ucur;
    a.Uprev = Uprev;
    a.Unext = Unext;
    a.keff = m.keff.p;
    a.kforce = m.kforce.p;
    a.kinv = m.kinv.p;
    a.nl_ptr = m.nl_ptr.p;
    a.nl_idx = m.nl_idx.p;
    a.load_dir = m.load_dir.p;
    a.load_factor = m.load_factor.p;
    a.load_series = m.load_series.p;
    a.load_nt = m.load_nt;
    a.k = k;
    a.th = m.th;
    a.ftol = m.ftol;
    a.ntiles = t.ntiles;
    a.ncolors = t.ncolors;
    a.max_stage = t.max_stage;
    a.max_own = t.max_own;
    a.egeo = t.elem_geo.p;
    a.geo = m.geo.p;
    a.drm = drm_ref(m);
    a.hpad = t.hpad.p;
    a.lcpad = t.lcpad.p;
    a.geopad = t.geopad.p;
    a.lampad = t.lampad.p;
    a.mupad = t.mupad.p;
    a.hstride = t.hstride;
    a.estride = t.estride;
    dim3 grid(t.ntiles), block(t.block);
#define SVLG_LAUNCH_FUSED(D, P)                                                                        \
    do {                                                                                              \
        if (m.variant == 3)                                                                           \
            hipLaunchKernelGGL((k_cd_corner<D, P>), grid, block, t.lds_bytes, m.stream, a);          \
        else                                                                                          \
            hipLaunchKernelGGL((k_cd_fused<D, P>), grid, block, t.lds_bytes, m.stream, a);           \
    } while (0)
    a.kmat = m.cd_kmat.p;
    if (m.elem_bf16) {
        hipLaunchKernelGGL((k_cd_corner<3, 4>), grid, block, t.lds_bytes, m.stream, a);
    } else if (use_moc(m)) {
        void *args[] = {&a};
        SVLG_HIP(hipLaunchKernel(moc_kernel(m), grid, block, args, t.lds_bytes, m.stream));
    } else if (m.elem_fp32) {
        hipLaunchKernelGGL((k_cd_corner<3, 5>), grid, block, t.lds_bytes, m.stream, a);
    } else if (m.ndim == 3) {
        if (m.elem_path == 3) SVLG_LAUNCH_FUSED(3, 3);
        else if (m.elem_path == 2) SVLG_LAUNCH_FUSED(3, 2);
        else if (m.elem_path == 1) SVLG_LAUNCH_FUSED(3, 1);
        else SVLG_LAUNCH_FUSED(3, 0);
    } else {
        if (m.elem_path == 3) SVLG_LAUNCH_FUSED(2, 3);
        else if (m.elem_path == 2) SVLG_LAUNCH_FUSED(2, 2);
        else if (m.elem_path == 1) SVLG_LAUNCH_FUSED(2, 1);
        else SVLG_LAUNCH_FUSED(2, 0);
    }
#undef SVLG_LAUNCH_FUSED
    return 0;
}

// Block and element-plane sizes of the multi-step kernel: the plan takes the smallest class that
// holds its tiles (0: none does). Hexahedra need 142 to 194 registers, which 1,024 threads do not have: such
// a class spilled 34 to 91 of them and took 11.0 us per step on 8,125 sheared bricks' nodes, whose
// 40-node tiles are less compact and stage more than 512 nodes, against 6.9 for single steps.
struct MultiClass {
    int block, elems;
};
static constexpr MultiClass kMulti2[] = {{256, 256}, {512, 456}, {1024, 968}}, kMulti3[] = {{256, 256}, {512, 512}};

template <int DIM, int MAXB, int MAXE, bool WIDE>
static const void *multi_fn_t(int path) {
    switch (path) {
        case 3: return reinterpret_cast<const void *>(&k_cd_multi<DIM, 3, MAXB, MAXE, WIDE>);
        case 2: return reinterpret_cast<const void *>(&k_cd_multi<DIM, 2, MAXB, MAXE, WIDE>);
        case 1: return reinterpret_cast<const void *>(&k_cd_multi<DIM, 1, MAXB, MAXE, false>);
        default: return reinterpret_cast<const void *>(&k_cd_multi<DIM, 0, MAXB, MAXE, false>);
    }
}

static bool multi_wide(const Model &m) { return m.multi.ntiles > 1024 && m.ndim == 2 && m.elem_path >= 2; }

static const void *multi_fn(const Model &m) {
    const bool wide = multi_wide(m);
    if (m.ndim == 2) {
        switch (m.multi.block) {
            case 256: return wide ? multi_fn_t<2, 256, 256, true>(m.elem_path) : multi_fn_t<2, 256, 256, false>(m.elem_path);
            case 512: return wide ? multi_fn_t<2, 512, 456, true>(m.elem_path) : multi_fn_t<2, 512, 456, false>(m.elem_path);
            default: return wide ? multi_fn_t<2, 1024, 968, true>(m.elem_path) : multi_fn_t<2, 1024, 968, false>(m.elem_path);
        }
    }
    switch (m.multi.block) {
        case 256: return multi_fn_t<3, 256, 256, false>(m.elem_path);
        default: return multi_fn_t<3, 512, 512, false>(m.elem_path);
    }
}

// Steps per launch of the multi-step kernel for this model's tiles (0: single-step kernels).
// Measured, microseconds per step, single-step kernel against the multi-step kernel:
//   one tile (231 Quad4 nodes)            4.3 -> 0.80
//   Quad4, 5,151 nodes, 64-node tiles     5.0 -> 1.37 (depth 5)      20,301 nodes, 128-node tiles  4.4 -> 1.42 (7)
//   Quad4, 80,601 nodes, 400-node tiles   5.4 -> 2.24 (5)            0.55M nodes, 400-node tiles  13.5 -> 9.6 (4)
//   Quad4, 1.77M nodes, 400-node tiles   29.4 -> 31.4 (4)            0.55M nodes, 128-node tiles  13.6 -> 19.9 (4)
//   distorted Quad4, 100,651 / 114,091 nodes, 252 / 286 tiles  7.5 -> 5.9 / 9.5 -> 10.4 (4), 0.55M nodes  25 -> 31 (4)
//   Quad4 25 times as wide as high, 400-node tiles, 210,951 / 0.55M nodes  7.4 -> 7.8 / 14.3 -> 14.9 (2)
//   Hexa8, 1,183 / 8,125 nodes            5.6 -> 3.3 / 5.7 -> 3.6 (2)
//   Hexa8, 18,513 / 60,025 nodes          5.9 -> 6.3 / 7.0 -> 17 (2)
//   Hexa8, 288 to 384 tiles of 40 nodes   6.0 -> 6.1 (2)      flat elements (1 : 10)  6.1 -> 6.3 to 6.5 (2)
//   sheared Hexa8, 2,890 nodes            6.2 -> 4.7 (2)      8,125 nodes, 300 tiles of 32 nodes  6.4 -> 7.1 (2)
// Below a chip full of workgroups the launch is saved and the recomputed rings are free; above
// it they compete with the tiles: in 2D the state's bytes still pay for them while a tile is
// large against its rings (three steps fit a launch) and up to about a million nodes, in 3D (one workgroup
// per CU) and for Gauss-point quadrilaterals never. Gauss-point hexahedra (1,300 operations an element)
// recompute nothing.
static int multi_depth(const Model &m) {
    const int nt = m.tiles.ntiles, own = m.nnodes / nt;
    if (nt == 1) return 1;
    if (m.ndim == 3) return m.elem_path >= 2 && nt <= 256 && own <= 64 ? 2 : 0;
    if (m.elem_path == 0 && nt > 256) return 0;
    if (nt > 512) return own >= 256 && m.nnodes <= 1000000 ? 4 : 0;
    int d = 1;  // rings up to about six times the tile
    while (d < 8 && (2.0 * (d + 1)) * (2.0 * (d + 1)) <= 2.4 * own) ++d;
    return d;
}

// Whether the first CentralDifference initialisation looks for a plan: the library chose the kernels, and
// they are the FP64 step of a corner-unique mesh that this integrator takes.
bool multi_wanted(const Model &m) {
    return m.auto_variant && m.corner_unique && m.lumped && !m.has_ak && !m.has_j2 && m.sm_ndofs == 0 &&
           !m.elem_bf16 && !m.elem_fp32 && multi_depth(m) > 0;
}

// The plan is set-up: Initialize takes 1.3 ms with it on 20,301 Quad4 nodes (0.2 without), 11.6 ms on 0.55M (0.4), 1.2
// ms on 8,125 Hexa8 nodes (0.15), the gain of 300, 2,500 and 500 steps over single steps. Rings and arrays are made by a
// few threads, straight into the block that is copied to the device.
static int multi_build(Model &m) {
    MultiSet &t = m.multi;
    MultiInput in;
    std::swap(in, m.multi_in);  // used once
    if (in.conn.empty()) return 0;
    int depth = multi_depth(m);
    const MultiClass *classes = m.ndim == 2 ? kMulti2 : kMulti3;
    const size_t nclasses = m.ndim == 2 ? std::size(kMulti2) : std::size(kMulti3);
    // One step per launch is the single-step kernels'; many tiles need three to pay for their rings.
    const int least = m.tiles.ntiles == 1 ? 1 : m.tiles.ntiles <= 512 ? 2 : 3;
    HostMulti h;
    MultiClass cls{0, 0};
    size_t lds = 0;
    for (; depth >= least; --depth) {  // the deepest that fits a class and the LDS
        cls = MultiClass{0, 0};
        if (make_multi(in, m.nen, depth, 1024, h))
            for (const MultiClass *c = classes; c != classes + nclasses && cls.block == 0; ++c)
                if (h.ns <= c->block && h.ne <= c->elems) cls = *c;
        lds = (size_t(m.elem_path < 2 ? 2 : 1) * h.ns * m.ndim + size_t(m.nen) * m.ndim * (cls.elems + 1)) *
              sizeof(double);
        if (cls.block != 0 && lds <= 160 * 1024) break;
    }
    if (depth < least) return 0;
    hipStream_t s = m.stream;
    // One allocation and one copy for all of it (each costs tens of microseconds of set-up).
    size_t total = 0;
    auto room = [&](size_t bytes) {
        const size_t at = total;
        total += (bytes + 15) / 16 * 16;
        return at;
    };
    const size_t nt = h.tiles.size(), ne = nt * h.ne, o_cnt = room(nt * 2 * (depth + 1) * 4),
                 o_node = room(nt * h.ns * 4), o_econn = room(ne * m.nen * 2), o_ncor = room(nt * h.nu * m.nen * 2),
                 o_egeo = room(ne * 2), o_lam = room(ne * 8), o_mu = room(ne * 8);
    std::unique_ptr<uint8_t[]> slab(new uint8_t[total]);
    auto at = [&](uint8_t *base) {
        return MultiArrays{reinterpret_cast<int32_t *>(base + o_cnt), reinterpret_cast<int32_t *>(base + o_node),
                           reinterpret_cast<uint16_t *>(base + o_econn), reinterpret_cast<uint16_t *>(base + o_ncor),
                           reinterpret_cast<uint16_t *>(base + o_egeo), reinterpret_cast<double *>(base + o_lam),
                           reinterpret_cast<double *>(base + o_mu)};
    };
    fill_multi(h, in, cls.elems, at(slab.get()));  // (no element at a corner: the zero column of the class)
    if (t.slab.alloc(total) != hipSuccess || t.U[0].alloc(m.ndofn) != hipSuccess ||
        t.U[1].alloc(m.ndofn) != hipSuccess) {
        t.slab.release();
        t.U[0].release();
        t.U[1].release();
        return 0;
    }
    SVLG_HIP(hipMemcpyAsync(t.slab.p, slab.get(), total, hipMemcpyHostToDevice, s));
    SVLG_HIP(hipStreamSynchronize(s));
    t.a = at(t.slab.p);
    t.ntiles = int(nt);
    t.ns = h.ns;
    t.ne = h.ne;
    t.nu = h.nu;
    t.block = cls.block;
    t.lds_bytes = lds;
    if (lds > 64 * 1024)
        SVLG_HIP(hipFuncSetAttribute(multi_fn(m), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    t.depth = depth;
    return 0;
}

// The plan saves time only: where host or device memory does not hold it, the model steps singly.
static int multi_setup(Model &m) {
    try {
        return multi_build(m);
    } catch (const std::bad_alloc &) {
        return 0;
    }
}

// n steps from k in one launch (n <= depth, or one tile); last: the caller reads the state next,
// which takes U_{k-2} too. Tiles read U_{k0} and U_{k0-1} of their neighbours, so the results go
// to other buffers, which then take the place of those in the ring.
static int multi_launch(Model &m, int k, int n, bool last, const RecRef &rec) {
    MultiSet &t = m.multi;
    double *&cur = m.U[m.ring].p, *&prev = m.U[(m.ring + 2) % 3].p, *&old = m.U[(m.ring + 1) % 3].p;
    MultiArgs a;
    a.cnt = t.a.cnt;
    a.node = t.a.node;
    a.econn = t.a.econn;
    a.ncor = t.a.ncor;
    a.egeo = t.a.egeo;
    a.elam = t.a.elam;
    a.emu = t.a.emu;
    a.geo = m.geo.p;
    a.X = m.X.p;
    a.Ucur = cur;
    a.Uprev = prev;
    a.out0 = n == 1 ? old : t.U[0].p;
    a.out1 = n == 1 ? nullptr : n == 2 ? old : t.U[1].p;
    a.out2 = n >= 3 && last ? old : nullptr;
    a.kforce = m.kforce.p;
    a.kinv = m.kinv.p;
    a.nl_ptr = m.nl_ptr.p;
    a.nl_idx = m.nl_idx.p;
    a.load_dir = m.load_dir.p;
    a.load_factor = m.load_factor.p;
    a.load_series = m.load_series.p;
    a.load_nt = m.load_nt;
    a.k = k;
    a.nsteps = n;
    a.th = m.th;
    a.ftol = m.ftol;
    a.ntiles = t.ntiles;
    a.depth = t.depth;
    a.ns = t.ns;
    a.ne = t.ne;
    a.nu = t.nu;
    a.drm = drm_ref(m);
    a.rec = rec;
    void *args[] = {&a};
    SVLG_HIP(hipLaunchKernel(multi_fn(m), dim3(t.ntiles), dim3(t.block), args, t.lds_bytes, m.stream));
    if (n == 1) {
        m.ring = (m.ring + 1) % 3;
    } else if (n == 2) {
        double *free_buf = prev;  // U_{k0-1} is no longer part of the state
        prev = old;
        old = cur;
        cur = t.U[0].p;
        t.U[0].p = free_buf;
    } else {
        std::swap(cur, t.U[0].p);
        std::swap(prev, t.U[1].p);
    }
    m.steps_done += n;
    return 0;
}

static int cd_one_step(Model &m, int k, const RecRef *rec = nullptr) {
    double *Ucur = m.U[m.ring].p;
    double *Uprev = m.U[(m.ring + 2) % 3].p;
    double *Unext = m.U[(m.ring + 1) % 3].p;
    // Support motion: the internal force sees U_(k-2) at its DOFs (the strains lag one
    // increment); afterwards U_(k-1) returns and U_k = U_(k-1) + a_k there.
    if (int rc = sm_lag_in(m, Ucur, Uprev, nullptr)) return rc;
    if (m.variant == 1 || m.variant == 3) {
        if (int rc = launch_fused(m, k, Ucur, Uprev, Unext, nullptr, rec)) return rc;
        if (int rc = sm_finish(m, 1, k, Ucur, Unext)) return rc;
        m.ring = (m.ring + 1) % 3;
        m.steps_done++;
        return 0;
    }
    if (m.nload > 0)
        hipLaunchKernelGGL(k_loads, dim3(1), dim3(64), 0, m.stream, k, m.nload, m.load_nt, m.ndim,
                           (int)m.h_load_dofs.size(), m.load_dofs.p, m.load_node.p, m.load_dir.p, m.load_factor.p,
                           m.load_series.p, m.Fext.p);
    if (int rc = drm_add_fext(m, k, m.Fext.p)) return rc;
    if (int rc = launch_fint_colored(m, Ucur, m.ftol, m.F.p)) return rc;
    int nb = (m.ndofn + 255) / 256;
    hipLaunchKernelGGL(k_cd_update, dim3(nb), dim3(256), 0, m.stream, m.ndofn, Ucur, Uprev, Unext, m.F.p, m.Fext.p,
                       m.keff.p, m.kforce.p);
    if (int rc = sm_finish(m, 1, k, Ucur, Unext)) return rc;
    m.ring = (m.ring + 1) % 3;
    m.steps_done++;
    return 0;
}

static void rec_columns(Model &m, int nrec, int on) {
    hipLaunchKernelGGL(k_rec_map, dim3((nrec + 255) / 256), dim3(256), 0, m.stream, nrec, m.rec.p, on, m.ndim,
                       m.tiles.ntiles, m.tiles.own_ptr.p, m.recmap.p, m.rectile.p);
}

// Whether steps go through the multi-step kernel: a plan exists, and the caller has not captured steps
// since the last initialisation. Its launches exchange buffers with the state's ring, which a
// replay would not repeat, and a graph captured before would go on in buffers that are no longer the state:
// from the first capture on, every step is a single step inside the ring's three buffers.
static bool multi_ready(Model &m) {
    if (m.multi.depth == 0 || m.captured) return false;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(m.stream, &st) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    m.captured = st != hipStreamCaptureStatusNone;
    return !m.captured;
}

// Steps per launch of the multi-step kernel (one tile has no neighbours to recompute).
static int multi_steps(const Model &m) { return m.multi.ntiles == 1 ? 2048 : m.multi.depth; }

// nsteps steps from k0, recording into rec (map null: nothing).
static int cd_advance(Model &m, int k0, int nsteps, const RecRef &rec) {
    if (!multi_ready(m)) {
        RecRef r = rec;
        for (int s = 0; s < nsteps; ++s) {
            if (int rc = cd_one_step(m, k0 + s, rec.map ? &r : nullptr)) return rc;
            if (rec.map) r.hist += rec.nrec;
        }
        return 0;
    }
    const int most = multi_steps(m);
    RecRef r = rec;
    for (int s = 0; s < nsteps;) {
        const int n = std::min(most, nsteps - s);
        if (int rc = multi_launch(m, k0 + s, n, s + n == nsteps, r)) return rc;
        if (rec.map) r.hist += size_t(n) * rec.nrec;
        s += n;
    }
    return 0;
}

// CentralDifference::Initialize (CentralDifference.cpp:36-71) with the per-DOF time steps
// dtd (device DOF order) or one dt.
static int cd_init_impl(Model &m, double dt, const std::vector<double> *dtd, double ftol) {
    SVLG_CHECK(dt > 0.0, "dt must be positive");
    SVLG_CHECK(m.lumped, "CentralDifference on the device needs MassFormulation = LUMPED");
    SVLG_CHECK(!m.has_ak, "CentralDifference on the device needs a diagonal C (Rayleigh ak must be 0)");
    SVLG_CHECK(!m.has_j2, "the explicit kernels restate elastic materials only; J2 models use svlg_nl_steps");
    m.dt = dt;
    m.ftol = ftol;
    m.cd_ready = false;
    m.captured = false;  // the state's buffers are new: graphs of the caller end here
    if (int rc = multi_setup(m)) return rc;
    if (m.cd_graph) {
        (void)hipGraphExecDestroy(m.cd_graph);
        m.cd_graph = nullptr;
        m.cd_graph_steps = 0;
        m.cd_graph_ring = -1;
    }
    for (auto &b : m.U) {
        SVLG_HIP(b.alloc(m.ndofn));
        SVLG_HIP(hipMemsetAsync(b.p, 0, sizeof(double) * m.ndofn, m.stream));
    }
    SVLG_HIP(m.F.alloc(m.ndofn));
    SVLG_HIP(hipMemsetAsync(m.F.p, 0, sizeof(double) * m.ndofn, m.stream));
    SVLG_HIP(m.Fext.alloc(m.ndofn));
    SVLG_HIP(hipMemsetAsync(m.Fext.p, 0, sizeof(double) * m.ndofn, m.stream));
    SVLG_HIP(m.keff.alloc(m.ndofn));
    SVLG_HIP(m.kforce.alloc(m.ndofn));
    SVLG_HIP(m.kinv.alloc(m.ndofn));
    if (dtd) {
        m.h_dt_dof = *dtd;
        SVLG_HIP(m.dt_dof.upload(dtd->data(), dtd->size(), m.stream));
    } else {
        m.h_dt_dof.clear();
    }
    DevBuf<int> sing;
    SVLG_HIP(sing.alloc(1));
    SVLG_HIP(hipMemsetAsync(sing.p, 0, sizeof(int), m.stream));
    int nb = (m.ndofn + 255) / 256;
    hipLaunchKernelGGL(k_cd_coeffs, dim3(nb), dim3(256), 0, m.stream, m.ndofn, dt, dtd ? m.dt_dof.p : nullptr,
                       m.mdiag.p, m.cdiag.p, m.fdof.p, m.keff.p, m.kforce.p, m.kinv.p, sing.p);
    SVLG_HIP(hipGetLastError());
    int hs = 0;
    SVLG_HIP(hipMemcpyAsync(&hs, sing.p, sizeof(int), hipMemcpyDeviceToHost, m.stream));
    SVLG_HIP(hipStreamSynchronize(m.stream));
    // EigenSolver::SolveSystem reports failure when the factorization breaks down
    // (EigenSolver.cpp:52-55): a free DOF with no mass and no damping.
    SVLG_CHECK(hs == 0, "EigenSolver::SolveSystem() : Solution for the linear system failed (zero Keff diagonal)");
    m.ring = 0;
    m.steps_done = 0;
    m.cd_ready = true;
    m.active = 1;
    return 0;
}

__global__ void k_step_advance(int *kdev, int by) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *kdev += by;
}

__global__ void k_step_set(int *kdev, int k) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *kdev = k;
}

// Captures cd_graph_steps fused launches (load sample *kdev + s for launch s) and the advance
// of *kdev into one executable graph, starting from the current U ring slot.
static int cd_capture(Model &m, int steps) {
    if (m.cd_graph) {
        (void)hipGraphExecDestroy(m.cd_graph);
        m.cd_graph = nullptr;
    }
    if (!m.kdev.p) SVLG_HIP(m.kdev.alloc(1));
    SVLG_HIP(hipStreamSynchronize(m.stream));
    SVLG_HIP(hipStreamBeginCapture(m.stream, hipStreamCaptureModeThreadLocal));
    int ring = m.ring, rc = 0;
    for (int s = 0; s < steps && rc == 0; ++s) {
        double *Ucur = m.U[ring].p, *Uprev = m.U[(ring + 2) % 3].p, *Unext = m.U[(ring + 1) % 3].p;
        rc = sm_lag_in(m, Ucur, Uprev, nullptr);
        if (rc == 0) rc = launch_fused(m, s, Ucur, Uprev, Unext, m.kdev.p);
        if (rc == 0) rc = sm_finish(m, 1, s, Ucur, Unext, m.kdev.p);
        ring = (ring + 1) % 3;
    }
    if (rc == 0) hipLaunchKernelGGL(k_step_advance, dim3(1), dim3(64), 0, m.stream, m.kdev.p, steps);
    hipGraph_t g = nullptr;
    const hipError_t ec = hipStreamEndCapture(m.stream, &g);
    if (rc != 0) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    SVLG_HIP(ec);
    const hipError_t ei = hipGraphInstantiate(&m.cd_graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    SVLG_HIP(ei);
    m.cd_graph_steps = steps;
    m.cd_graph_ring = m.ring;
    return 0;
}

}  // namespace svlg

using namespace svlg;

extern "C" {

int svlg_cd_init(svlg_model *h, double dt, double ftol) {
    SVLG_CHECK(h, "null model");
    return cd_init_impl(h->m, dt, nullptr, ftol);
}

int svlg_cd_init_batch(svlg_model *h, int32_t nparts, const int32_t *part_node_ptr, const double *dts, double ftol) {
    SVLG_CHECK(h && part_node_ptr && dts, "null argument");
    Model &m = h->m;
    SVLG_CHECK(nparts >= 1, "nparts must be positive");
    SVLG_CHECK(part_node_ptr[0] == 0 && part_node_ptr[nparts] == m.nnodes, "part ranges must cover the nodes");
    for (int p = 0; p < nparts; ++p) {
        SVLG_CHECK(part_node_ptr[p + 1] >= part_node_ptr[p], "part ranges must be ascending");
        SVLG_CHECK(dts[p] > 0.0, "dt must be positive");
    }
    // Per device DOF: the time step of the part that holds the node (description order).
    std::vector<double> dtd(m.ndofn);
    int part = 0;
    std::vector<double> dt_node(m.nnodes);
    for (int n = 0; n < m.nnodes; ++n) {
        while (n >= part_node_ptr[part + 1]) ++part;
        dt_node[n] = dts[part];
    }
    for (int p = 0; p < m.nnodes; ++p)
        for (int c = 0; c < m.ndim; ++c) dtd[size_t(p) * m.ndim + c] = dt_node[m.perm[p]];
    return cd_init_impl(m, dts[0], &dtd, ftol);
}

int svlg_cd_plan(svlg_model *h, int64_t *plan) {
    SVLG_CHECK(h && plan, "null argument");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    const bool multi = m.multi.depth > 0 && !m.captured;
    plan[0] = multi ? multi_steps(m) : 1;
    plan[1] = m.tiles.ntiles;
    plan[2] = multi ? m.multi.block : m.tiles.block;
    plan[3] = multi && multi_wide(m) ? 1 : 0;
    return 0;
}

int svlg_cd_steps_async(svlg_model *h, int32_t k0, int32_t nsteps) {
    SVLG_CHECK(h, "null model");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    if (int rc = cd_advance(m, k0, nsteps, RecRef{nullptr, nullptr, nullptr, 0})) return rc;
    SVLG_HIP(hipGetLastError());
    return 0;
}

int svlg_cd_graph_steps(svlg_model *h, int32_t k0, int32_t nsteps, int32_t graph_steps) {
    SVLG_CHECK(h, "null model");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    SVLG_CHECK(nsteps >= 0, "negative count");
    SVLG_CHECK(m.variant == 1 || m.variant == 3, "graph stepping needs the fused kernel (variant 1 or 3)");
    SVLG_CHECK(graph_steps >= 3 && graph_steps % 3 == 0 && graph_steps <= 3000,
               "graph_steps must be a multiple of 3 in [3, 3000]");
    if (multi_ready(m)) {
        // A launch already covers several steps, with its step index and buffers as arguments:
        // nothing is left for a graph to save.
        if (int rc = cd_advance(m, k0, nsteps, RecRef{nullptr, nullptr, nullptr, 0})) return rc;
        SVLG_HIP(hipGetLastError());
        return 0;
    }
    int done = 0;
    if (nsteps >= graph_steps) {
        if (!m.cd_graph || m.cd_graph_steps != graph_steps || m.cd_graph_ring != m.ring)
            if (int rc = cd_capture(m, graph_steps)) return rc;
        hipLaunchKernelGGL(k_step_set, dim3(1), dim3(64), 0, m.stream, m.kdev.p, int(k0));
        for (; done + graph_steps <= nsteps; done += graph_steps) SVLG_HIP(hipGraphLaunch(m.cd_graph, m.stream));
        m.steps_done += done;  // the ring returns to its slot after every replay
    }
    for (; done < nsteps; ++done)
        if (int rc = cd_one_step(m, k0 + done)) return rc;
    SVLG_HIP(hipGetLastError());
    return 0;
}

int svlg_autotune_tiles(const svlg_mesh_desc *desc, const svlg_exec_opts *base, const int32_t *cand, int32_t ncand,
                        int32_t nparts, const int32_t *part_node_ptr, const double *dts, int32_t steps,
                        int32_t *best_tile_nodes, double *us_per_step) {
    SVLG_CHECK(desc && cand && dts && best_tile_nodes, "null argument");
    SVLG_CHECK(ncand >= 1 && steps >= 1 && nparts >= 1, "empty search");
    SVLG_CHECK(nparts == 1 || part_node_ptr, "part ranges missing");
    double best = -1.0;
    *best_tile_nodes = 0;
    for (int c = 0; c < ncand; ++c) {
        if (us_per_step) us_per_step[c] = -1.0;
        svlg_exec_opts o{};
        if (base) o = *base;
        o.tile_nodes = cand[c];
        svlg_model *h = nullptr;
        if (svlg_model_create_ex(desc, &o, &h) != 0) continue;  // e.g. the tile does not fit the LDS
        Model &m = h->m;
        int rc = nparts > 1 ? svlg_cd_init_batch(h, nparts, part_node_ptr, dts, 1e-12) : svlg_cd_init(h, dts[0], 1e-12);
        if (rc == 0 && (m.variant == 1 || m.variant == 3)) {
            hipEvent_t e0 = nullptr, e1 = nullptr;
            bool ok = hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess;
            const RecRef none{nullptr, nullptr, nullptr, 0};
            ok = ok && cd_advance(m, 1, 3, none) == 0;
            ok = ok && hipEventRecord(e0, m.stream) == hipSuccess;
            ok = ok && cd_advance(m, 4, steps, none) == 0;
            ok = ok && hipEventRecord(e1, m.stream) == hipSuccess && hipEventSynchronize(e1) == hipSuccess;
            float ms = 0.0f;
            if (ok && hipEventElapsedTime(&ms, e0, e1) == hipSuccess) {
                const double us = 1e3 * double(ms) / steps;
                if (us_per_step) us_per_step[c] = us;
                if (best < 0.0 || us < best) {
                    best = us;
                    *best_tile_nodes = cand[c];
                }
            }
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
        }
        svlg_model_destroy(h);
    }
    SVLG_CHECK(best > 0.0, "no candidate tile size could be built and timed");
    return 0;
}

int svlg_cd_steps(svlg_model *h, int32_t k0, int32_t nsteps, int32_t nrec, const int32_t *rec_dofs, double *hist) {
    SVLG_CHECK(h, "null model");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    SVLG_CHECK(nsteps >= 0 && nrec >= 0, "negative count");
    RecRef rec{nullptr, nullptr, nullptr, 0};
    std::vector<int32_t> pos, dup;
    // The step kernels record, except where support motion moves DOFs after them or the
    // element-colored kernels run: there a kernel per step does.
    const bool inside = m.sm_ndofs == 0 && (m.variant == 1 || m.variant == 3);
    if (nrec > 0) {
        SVLG_CHECK(rec_dofs && hist, "recorder arrays missing");
        if (int rc = record_positions(m, nrec, rec_dofs, pos)) return rc;
        const size_t want = size_t(nrec) * std::max(nsteps, 1);
        if (m.hist.n < want) SVLG_HIP(m.hist.alloc(want));
        if (m.rec.n < pos.size()) SVLG_HIP(m.rec.alloc(pos.size()));
        if (inside) {
            // A DOF asked for more than once is recorded in its first column and copied. Columns in
            // ascending free order (a whole field, a line of nodes) hold none; otherwise one pass finds
            // them (a sort took 68 of 70 ms of a one-step call that recorded 1.56M DOFs).
            bool distinct = rec_dofs[0] >= 0;
            for (int r = 1; r < nrec && distinct; ++r) distinct = rec_dofs[r] > rec_dofs[r - 1];
            if (!distinct) {
                std::vector<int32_t> first(m.ndofn, -1);
                for (int r = 0; r < nrec; ++r) {
                    int32_t &f = first[pos[r]];
                    if (f < 0) {
                        f = r;
                    } else {
                        dup.push_back(r);
                        dup.push_back(f);
                        pos[r] = -1;
                    }
                }
            }
            if (!m.rectile.p) {
                SVLG_HIP(m.recmap.alloc(m.ndofn));
                SVLG_HIP(hipMemsetAsync(m.recmap.p, 0xff, sizeof(int32_t) * m.ndofn, m.stream));
                SVLG_HIP(m.rectile.alloc(m.tiles.ntiles));
                SVLG_HIP(hipMemsetAsync(m.rectile.p, 0, sizeof(int32_t) * m.tiles.ntiles, m.stream));
            }
        }
        SVLG_HIP(hipMemcpyAsync(m.rec.p, pos.data(), sizeof(int32_t) * pos.size(), hipMemcpyHostToDevice, m.stream));
        if (inside) {
            rec = RecRef{m.recmap.p, m.rectile.p, m.hist.p, nrec};
            rec_columns(m, nrec, 1);
        }
    }
    int rc = 0;
    if (inside || nrec == 0) {
        rc = cd_advance(m, k0, nsteps, rec);
    } else {
        for (int s = 0; s < nsteps && rc == 0; ++s) {
            rc = cd_one_step(m, k0 + s);
            if (rc == 0)
                hipLaunchKernelGGL(k_record, dim3((nrec + 63) / 64), dim3(64), 0, m.stream, nrec, m.rec.p,
                                   m.U[m.ring].p, m.hist.p + size_t(s) * nrec);
        }
    }
    if (rec.map) rec_columns(m, nrec, 0);
    if (rc) {
        (void)hipStreamSynchronize(m.stream);  // pos is on its way to the device
        return rc;
    }
    SVLG_HIP(hipGetLastError());
    if (nrec > 0 && nsteps > 0)
        SVLG_HIP(hipMemcpyAsync(hist, m.hist.p, sizeof(double) * size_t(nrec) * nsteps, hipMemcpyDeviceToHost,
                                m.stream));
    SVLG_HIP(hipStreamSynchronize(m.stream));
    // (On the host: columns times steps may pass 2^31.)
    for (int s = 0; s < nsteps && !dup.empty(); ++s) {
        double *row = hist + size_t(s) * nrec;
        for (size_t i = 0; i < dup.size(); i += 2) row[dup[i]] = row[dup[i + 1]];
    }
    return 0;
}

int svlg_cd_effective_force(svlg_model *h, int32_t k, double factor, double *Feff) {
    (void)factor;  // unused by CentralDifference::ComputeEffectiveForce as well
    SVLG_CHECK(h && Feff, "null argument");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    double *Ucur = m.U[m.ring].p;
    const double *Up = m.U[(m.ring + 2) % 3].p;
    if (int rc = sm_lag_in(m, Ucur, Up, nullptr)) return rc;
    if (m.nload > 0)
        hipLaunchKernelGGL(k_loads, dim3(1), dim3(64), 0, m.stream, k, m.nload, m.load_nt, m.ndim,
                           (int)m.h_load_dofs.size(), m.load_dofs.p, m.load_node.p, m.load_dir.p, m.load_factor.p,
                           m.load_series.p, m.Fext.p);
    if (int rc = drm_add_fext(m, k, m.Fext.p)) return rc;
    if (int rc = launch_fint_colored(m, Ucur, m.ftol, m.F.p)) return rc;
    DevBuf<double> fn, ff;
    SVLG_HIP(fn.alloc(m.ndofn));
    SVLG_HIP(ff.alloc(std::max(m.nfree, 1)));
    const int nb = (m.ndofn + 255) / 256;
    hipLaunchKernelGGL(k_cd_feff, dim3(nb), dim3(256), 0, m.stream, m.ndofn, Ucur, Up, m.F.p, m.Fext.p, m.keff.p,
                       m.kforce.p, fn.p);
    if (int rc = sm_finish(m, 0, k, Ucur, nullptr)) return rc;
    if (int rc = gather_free(m, fn.p, ff.p)) return rc;
    SVLG_HIP(hipMemcpyAsync(Feff, ff.p, sizeof(double) * m.nfree, hipMemcpyDeviceToHost, m.stream));
    SVLG_HIP(hipStreamSynchronize(m.stream));
    return 0;
}

int svlg_external_force(svlg_model *h, int32_t k, double *F) {
    SVLG_CHECK(h && F, "null argument");
    Model &m = h->m;
    DevBuf<double> fe;
    SVLG_HIP(fe.alloc(m.ndofn));
    SVLG_HIP(hipMemsetAsync(fe.p, 0, sizeof(double) * m.ndofn, m.stream));
    if (m.nload > 0)
        hipLaunchKernelGGL(k_loads, dim3(1), dim3(64), 0, m.stream, k, m.nload, m.load_nt, m.ndim,
                           (int)m.h_load_dofs.size(), m.load_dofs.p, m.load_node.p, m.load_dir.p, m.load_factor.p,
                           m.load_series.p, fe.p);
    if (int rc = drm_add_fext(m, k, fe.p)) return rc;
    SVLG_HIP(hipGetLastError());
    std::vector<double> h_fe(m.ndofn);
    SVLG_HIP(hipMemcpyAsync(h_fe.data(), fe.p, sizeof(double) * m.ndofn, hipMemcpyDeviceToHost, m.stream));
    SVLG_HIP(hipStreamSynchronize(m.stream));
    // Device node order -> description order.
    for (int n = 0; n < m.nnodes; ++n)
        for (int c = 0; c < m.ndim; ++c) F[size_t(n) * m.ndim + c] = h_fe[size_t(m.inv[n]) * m.ndim + c];
    return 0;
}

int svlg_cd_effective_stiffness(svlg_model *h, double *Kdiag) {
    SVLG_CHECK(h && Kdiag, "null argument");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    DevBuf<double> ff;
    SVLG_HIP(ff.alloc(std::max(m.nfree, 1)));
    if (int rc = gather_free(m, m.keff.p, ff.p)) return rc;
    SVLG_HIP(hipMemcpyAsync(Kdiag, ff.p, sizeof(double) * m.nfree, hipMemcpyDeviceToHost, m.stream));
    SVLG_HIP(hipStreamSynchronize(m.stream));
    return 0;
}

int svlg_cd_apply_increment(svlg_model *h, int32_t k, const double *dU) {
    SVLG_CHECK(h && dU, "null argument");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    DevBuf<double> ff, dn;
    SVLG_HIP(ff.upload(dU, std::max(m.nfree, 1), m.stream));
    SVLG_HIP(dn.alloc(m.ndofn));
    if (int rc = scatter_free(m, ff.p, dn.p)) return rc;
    const int nb = (m.ndofn + 255) / 256;
    hipLaunchKernelGGL(k_cd_increment, dim3(nb), dim3(256), 0, m.stream, m.ndofn, m.U[m.ring].p, dn.p, m.keff.p,
                       m.U[(m.ring + 1) % 3].p);
    SVLG_HIP(hipGetLastError());
    if (int rc = sm_add_increment(m, k, m.U[m.ring].p, m.U[(m.ring + 1) % 3].p)) return rc;
    m.ring = (m.ring + 1) % 3;
    m.steps_done++;
    SVLG_HIP(hipStreamSynchronize(m.stream));
    return 0;
}

int svlg_cd_get_state(svlg_model *h, double *U, double *V, double *A) {
    SVLG_CHECK(h, "null model");
    Model &m = h->m;
    SVLG_CHECK(m.cd_ready, "svlg_cd_init has not been called");
    double *outs[3] = {U, V, A};
    if (!U && !V && !A) return 0;
    const size_t nf = std::max(m.nfree, 1);
    if (m.snap.n < 3 * nf) {
        SVLG_HIP(m.snap.alloc(3 * nf));
        SVLG_HIP(hipMemsetAsync(m.snap.p, 0, sizeof(double) * m.snap.n, m.stream));
    }
    double *dev[3] = {U ? m.snap.p : nullptr, V ? m.snap.p + nf : nullptr, A ? m.snap.p + 2 * nf : nullptr};
    hipLaunchKernelGGL(k_cd_state, dim3((m.ndofn + 255) / 256), dim3(256), 0, m.stream, m.ndofn, m.dt,
                       m.h_dt_dof.empty() ? nullptr : m.dt_dof.p, m.steps_done > 0 ? 1 : 0, m.fdof.p, m.U[m.ring].p,
                       m.U[(m.ring + 2) % 3].p, m.U[(m.ring + 1) % 3].p, dev[0], dev[1], dev[2]);
    SVLG_HIP(hipGetLastError());
    for (int i = 0; i < 3; ++i)
        if (outs[i])
            SVLG_HIP(hipMemcpyAsync(outs[i], dev[i], sizeof(double) * m.nfree, hipMemcpyDeviceToHost, m.stream));
    SVLG_HIP(hipStreamSynchronize(m.stream));
    return 0;
}

}  // extern "C"
