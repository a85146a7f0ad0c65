// Learned HLLD surrogate (no counterpart in the reference; it stands in for
// riemannSolver_HLLD, computeFlux.cpp:178-425, inside computeFlux,
// computeFlux.cpp:6-148).
//
//   featurisation   the HLLD inputs of a face in the face frame (rotation and
//                   Dedner B_n/psi exactly as computeFlux, FP64), divided by two
//                   exact symmetries of the HLLD flux: the Galilean boost
//                   V = w_n n + u_t and the MHD scaling (rho_s, c_s); the
//                   network answers the residual over the HLL flux of the two
//                   sides per unit normalised jump (fvm_mlp.h)
//   training        Adam over bf16-operand MFMAs (v_mfma_f32_16x16x32_bf16,
//                   FP32 accumulation), two launches a step (fvm_sg_train.h)
//   inference       one fused kernel: each wavefront featurises 64 faces, runs
//                   the four layers as chained MFMAs with every activation kept
//                   in registers (the K order of each weight fragment is the
//                   order in which the previous layer's accumulator tiles land
//                   in the lanes, so no transpose is needed between layers),
//                   then gates and assembles the FP64 flux; weights stay in LDS
//   fallback        every face the gate rejects is appended to a list (gathered
//                   in LDS, one atomic addition per 128 of a wavefront's and
//                   one per block) and a second launch runs the FP64
//                   computeFlux on it
//
// Compiled with -ffp-contract=off so the FP64 Dedner terms and the fallback
// are operation-for-operation the reference's.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/fvm_gpu.h"
#include "../../include/fvm_surrogate.h"
#include "fvm_internal.h"
#include "fvm_physics.h"
#include "fvm_mlp.h"
#include "fvm_sg_train.h"

namespace fvm {
namespace sg {

using Frame = FrameT<double>;

__device__ __forceinline__ int gid() { return (int)(blockIdx.x * blockDim.x + threadIdx.x); }

// ---------------------------------------------------------------------------
// face frame (computeFlux.cpp:17-107), interior faces
// ---------------------------------------------------------------------------
__device__ __forceinline__ void frame_rows(const double *nrm, double A[3][3]) {
  const double ex = nrm[0], ey = nrm[1], ez = nrm[2];
  const double ds = dsqrt(ex * ex + ey * ey);
  const double ids = (ds != 0.0) ? 1.0 / ds : 0.0;
  const double cosph = (ids == 0.0) ? 1.0 : ex * ids;
  const double sinph = (ids == 0.0) ? 0.0 : ey * ids;
  const double costh = ez, sinth = ds;
  A[0][0] = cosph * sinth;
  A[0][1] = sinth * sinph;
  A[0][2] = costh;
  A[1][0] = -sinph;
  A[1][1] = cosph;
  A[1][2] = 0.0;
  A[2][0] = -costh * cosph;
  A[2][1] = -costh * sinph;
  A[2][2] = sinth;
}

__device__ __forceinline__ void to_frame(double gamma, const double *wij, const double *Wi, const double *Wj,
                                         const double *nrm, Frame &s) {
  frame_rows(nrm, s.A);
  for (int d = 0; d < 3; d++) {
    s.vL[d] = s.A[d][0] * Wi[VELX] + s.A[d][1] * Wi[VELY] + s.A[d][2] * Wi[VELZ];
    s.BL[d] = s.A[d][0] * Wi[BX] + s.A[d][1] * Wi[BY] + s.A[d][2] * Wi[BZ];
    s.vR[d] = s.A[d][0] * Wj[VELX] + s.A[d][1] * Wj[VELY] + s.A[d][2] * Wj[VELZ];
    s.BR[d] = s.A[d][0] * Wj[BX] + s.A[d][1] * Wj[BY] + s.A[d][2] * Wj[BZ];
  }
  s.rL = Wi[DENS];
  s.eL = Wi[ETHM];
  s.rR = Wj[DENS];
  s.eR = Wj[ETHM];
  s.psiL = Wi[PSI];
  s.psiR = Wj[PSI];
  s.entrL = Wi[ENTR];
  s.entrR = Wj[ENTR];
  s.pL = pressure(gamma, Wi[ETHM]);
  s.pR = pressure(gamma, Wj[ETHM]);
  s.wn = s.A[0][0] * wij[0] + s.A[0][1] * wij[1] + s.A[0][2] * wij[2];
  const double cfl2 = (gamma * s.pL + sqr(s.BL[0]) + sqr(s.BL[1]) + sqr(s.BL[2])) / s.rL;
  const double cfr2 = (gamma * s.pR + sqr(s.BR[0]) + sqr(s.BR[1]) + sqr(s.BR[2])) / s.rR;
  const double chL = dsqrt(cfl2 + 0.0 * sqr(s.vL[0] - s.wn));
  const double chR = dsqrt(cfr2 + 0.0 * sqr(s.vR[0] - s.wn));
  s.Bn = (s.BL[0] * chL + s.BR[0] * chR + (s.psiL - s.psiR)) / (chL + chR);
  s.psi = (s.psiL * chR + s.psiR * chL + chR * chL * (s.BL[0] - s.BR[0])) / (chL + chR);
}

__device__ __forceinline__ void load_face(int f, const double *wij, const double *Wi, const double *Wj,
                                          const double *nrm, double *w3, double *L, double *R, double *n3) {
  for (int d = 0; d < 3; d++) {
    w3[d] = wij[3 * (size_t)f + d];
    n3[d] = nrm[3 * (size_t)f + d];
  }
  for (int k = 0; k < NF; k++) {
    L[k] = Wi[(size_t)NF * f + k];
    R[k] = Wj[(size_t)NF * f + k];
  }
}

// ---------------------------------------------------------------------------
// training samples: features + normalised moving-frame HLLD fluxes (FP64 HLLD)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_samples(int n, double gamma, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                          const double *nrm, Gate G, float *Xs, float *Ts, int *flag) {
  const int f = gid();
  bool keep = false;
  float x[NIN], t[NOUT];
  if (f < n) {
    double w3[3], L[NF], R[NF], n3[3];
    load_face(f, wij, Wi, Wj, nrm, w3, L, R, n3);
    Frame s;
    to_frame(gamma, w3, L, R, n3, s);
    double Fc[7], J, sc[4];
    keep = features<double>(gamma, s, jbnd[f], G, x, Fc, J, sc);
    if (keep) {
      const double rs = sc[0], cs = sc[1], Ps = rs * cs * cs, Bs = dsqrt(Ps);
      double F[NF];
      riemann_hlld<double>(gamma, F, s.Bn, s.wn, s.rL, s.pL, s.eL, s.vL[0], s.vL[1], s.vL[2], s.BL[1], s.BL[2], s.rR,
                           s.pR, s.eR, s.vR[0], s.vR[1], s.vR[2], s.BR[1], s.BR[2]);
      // moving-frame flux: G' = G - boost(V), V = (w_n, u_t1, u_t2)
      const double V[3] = {s.wn, sc[2], sc[3]};
      const double Gm = F[MASS];
      const double Gp[3] = {F[MOMX] - V[0] * Gm, F[MOMY] - V[1] * Gm, F[MOMZ] - V[2] * Gm};
      const double GE = F[ENER] - (V[0] * Gp[0] + V[1] * Gp[1] + V[2] * Gp[2]) -
                        0.5 * (V[0] * V[0] + V[1] * V[1] + V[2] * V[2]) * Gm;
      const double Gb1 = F[WBY] + s.Bn * V[1], Gb2 = F[WBZ] + s.Bn * V[2];
      // residual over the HLL base flux, per unit jump
      const double g[7] = {Gm / (rs * cs), Gp[0] / Ps, Gp[1] / Ps, Gp[2] / Ps, GE / (Ps * cs), Gb1 / (Bs * cs),
                           Gb2 / (Bs * cs)};
      for (int k = 0; k < 7; k++) t[k] = (float)((g[k] - Fc[k]) / J);
      t[7] = 0.0f;
      for (int k = 0; k < 7; k++) keep = keep && __builtin_isfinite(t[k]);
    }
  }
  // staged at the face's own index; k_pack_samples keeps the face order, so
  // the training set (and the minibatches drawn from it) is the same every run
  if (f < n) {
    flag[f] = keep ? 1 : 0;
    if (keep) {
      for (int k = 0; k < NIN; k++) Xs[(size_t)f * NIN + k] = x[k];
      for (int k = 0; k < NOUT; k++) Ts[(size_t)f * NOUT + k] = t[k];
    }
  }
}

// kept samples, in face order, appended at base (pos: exclusive scan of flag)
__global__ void k_pack_samples(int n, const int *flag, const int *pos, const float *Xs, const float *Ts, float *X,
                               float *T, long long base) {
  const int f = gid();
  if (f >= n || !flag[f]) return;
  const size_t i = (size_t)(base + pos[f]);
  for (int k = 0; k < NIN; k++) X[i * NIN + k] = Xs[(size_t)f * NIN + k];
  for (int k = 0; k < NOUT; k++) T[i * NOUT + k] = Ts[(size_t)f * NOUT + k];
}

// ---------------------------------------------------------------------------
// inference: weight fragments in the lane order of the MFMA A operand
//   L0 (16x16x16): frag[mt][lane] 4 x bf16 = W0[4g+e][16mt+r16]
//   L1, L2 (16x16x32): frag[mt][c][lane] 8 x bf16 = W[f(c,g,e)][16mt+r16]
//   L3: frag[c][lane] 8 x bf16 = W3[f(c,g,e)][r16] (r16 < 8, else 0)
// with f(c,g,e) = 32c + 4g + e (e < 4), 32c + 16 + 4g + e - 4 (e >= 4): the
// input feature that lane group g holds in K slot e after the previous layer's
// accumulator tiles 2c and 2c+1 are concatenated.
// ---------------------------------------------------------------------------
constexpr int IB = 512;                        // threads per inference block
constexpr int FEAT_B = 64 * NIN * 2;           // per wave: features (bf16), reused for outputs (f32)
constexpr int OUT_B = 64 * NOUT * 4;
struct FaceCtx {
  float nrm[3];
  float wn, ut1, ut2, rs, cs, psiL, psiR, entrL, entrR;
  float Fc[7], J;
  float pad[2];
  double Bn, psi;
};
constexpr int CTX_B = 64 * (int)sizeof(FaceCtx);
constexpr int WAVE_B = (FEAT_B > OUT_B ? FEAT_B : OUT_B) + CTX_B;
constexpr int REJ_N = 128;                     // rejected faces a wavefront gathers
constexpr int LDS_B = P_BYTES + (IB / 64) * (WAVE_B + REJ_N * 4 + 8);
static_assert(sizeof(FaceCtx) == 104, "FaceCtx layout");
static_assert(LDS_B <= 160 * 1024, "LDS budget");

__global__ void k_pack(const float *P, __bf16 *frag, float *bias) {
  const int i = gid();
  if (i < P_BF) {
    float v = 0.0f;
    if (i < P_L0) {
      const int e = i & 3, lane = (i >> 2) & 63, mt = i >> 8;
      v = P[OW0 + (4 * (lane >> 4) + e) * NH + 16 * mt + (lane & 15)];
    } else if (i < P_L0 + 2 * P_L1) {
      const int j = (i - P_L0) % P_L1, layer = (i - P_L0) / P_L1;
      const int e = j & 7, lane = (j >> 3) & 63, c = (j >> 9) & 3, mt = j >> 11;
      v = P[(layer ? OW2 : OW1) + kfeat(c, lane >> 4, e) * NH + 16 * mt + (lane & 15)];
    } else {
      const int j = i - P_L0 - 2 * P_L1;
      const int e = j & 7, lane = (j >> 3) & 63, c = j >> 9;
      v = (lane & 15) < NOUT ? P[OW3 + kfeat(c, lane >> 4, e) * NOUT + (lane & 15)] : 0.0f;
    }
    frag[i] = (__bf16)v;
  }
  if (i < P_BIAS) {
    float v = 0.0f;
    if (i < NH) v = P[OB0 + i];
    else if (i < 2 * NH) v = P[OB1 + i - NH];
    else if (i < 3 * NH) v = P[OB2 + i - 2 * NH];
    else if (i < 3 * NH + NOUT) v = P[OB3 + i - 3 * NH];
    bias[i] = v;
  }
}

// MODE 0: computeFlux batch (features from the faces, gate, FP64 assembly,
// fallback list); MODE 1: raw features x[n][16] -> y[n][8]
// The rejected faces: each wavefront gathers its own in LDS and takes their place
// in the list with one atomic addition per 128, what is left with one per block.
// An addition per batch of 64 faces was the bound of the launch: at about 10 ns
// each on one address, 156 of 181 us for 10^6 faces.  Now (10^6 faces, with the
// fallback launch: 214 -> 130 us a call) it waits on its inputs, two wavefronts a
// SIMD: no faster with a third (the network in two passes of 32 faces), nor with
// inputs loaded in whole lines, with or without a batch's lead.
template <int MODE>
__global__ void __launch_bounds__(IB) k_infer(int n, double gamma, const double *__restrict__ wij,
                                              const double *__restrict__ Wi, const double *__restrict__ Wj,
                                              const int *__restrict__ jbnd, const double *__restrict__ nrm,
                                              const __bf16 *__restrict__ pfrag, const float *__restrict__ pbias,
                                              Gate G, double *__restrict__ psi_out, double *__restrict__ Bn_out,
                                              double *__restrict__ flux, int *__restrict__ fb_list,
                                              unsigned long long *__restrict__ fb_count, const float *__restrict__ xin,
                                              float *__restrict__ yout) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __bf16 *wl = reinterpret_cast<__bf16 *>(smem);
  float *bias = reinterpret_cast<float *>(smem + P_BF * 2);
  {
    const int4 *src = reinterpret_cast<const int4 *>(pfrag);
    int4 *dst = reinterpret_cast<int4 *>(smem);
    for (int i = threadIdx.x; i < P_BF * 2 / 16; i += IB) dst[i] = src[i];
    for (int i = threadIdx.x; i < P_BIAS; i += IB) bias[i] = pbias[i];
  }
  __syncthreads();
  const int lane = __lane_id(), wv = threadIdx.x >> 6;
  char *wb = smem + P_BYTES + wv * WAVE_B;
  __bf16 *feat = reinterpret_cast<__bf16 *>(wb);
  float *out = reinterpret_cast<float *>(wb);
  FaceCtx *ctx = reinterpret_cast<FaceCtx *>(wb + (FEAT_B > OUT_B ? FEAT_B : OUT_B));
  int *rejs = reinterpret_cast<int *>(smem + P_BYTES + (IB / 64) * WAVE_B) + wv * REJ_N;
  unsigned long long *wrej = reinterpret_cast<unsigned long long *>(smem + P_BYTES + (IB / 64) * (WAVE_B + REJ_N * 4));
  int nrej = 0;
  const int nbatch = (n + 63) / 64;
  const int wstride = gridDim.x * (IB / 64);
  for (int bw = blockIdx.x * (IB / 64) + wv; bw < nbatch; bw += wstride) {
    const int f = bw * 64 + lane;
    const bool live = f < n;
    bool ok = false;
    float x[NIN];
    if constexpr (MODE == 1) {
      for (int k = 0; k < NIN; k++) x[k] = live ? xin[(size_t)f * NIN + k] : 0.0f;
      ok = live;
    } else {
      for (int k = 0; k < NIN; k++) x[k] = 0.0f;
      if (live) {
        double w3[3], L[NF], R[NF], n3[3];
        load_face(f, wij, Wi, Wj, nrm, w3, L, R, n3);
        Frame s;
        to_frame(gamma, w3, L, R, n3, s);
        float Fc[7], J, sc[4];
        ok = features<float>(gamma, s, jbnd[f], G, x, Fc, J, sc);
        FaceCtx &cx = ctx[lane];
        for (int k = 0; k < 7; k++) cx.Fc[k] = Fc[k];
        cx.J = J;
        for (int d = 0; d < 3; d++) cx.nrm[d] = (float)n3[d];
        cx.wn = (float)s.wn;
        cx.ut1 = sc[2];
        cx.ut2 = sc[3];
        cx.rs = sc[0];
        cx.cs = sc[1];
        cx.psiL = (float)s.psiL;
        cx.psiR = (float)s.psiR;
        cx.entrL = (float)s.entrL;
        cx.entrR = (float)s.entrR;
        cx.Bn = s.Bn;
        cx.psi = s.psi;
        if (!ok)
          for (int k = 0; k < NIN; k++) x[k] = 0.0f;
      }
    }
    {
      bf16x8 lo, hi;
      for (int k = 0; k < 8; k++) {
        lo[k] = (__bf16)x[k];
        hi[k] = (__bf16)x[8 + k];
      }
      *reinterpret_cast<bf16x8 *>(feat + lane * NIN) = lo;
      *reinterpret_cast<bf16x8 *>(feat + lane * NIN + 8) = hi;
    }
    wave_sync();
    mlp64(wl, bias, feat, out, lane);
    wave_sync();
    float y[NOUT];
    for (int k = 0; k < NOUT; k++) y[k] = out[lane * NOUT + k];
    wave_sync();  // outputs read before the next batch's features land
    if constexpr (MODE == 1) {
      if (live)
        for (int k = 0; k < NOUT; k++) yout[(size_t)f * NOUT + k] = y[k];
    } else {
      ok = ok && y[7] <= G.max_log10_err;
      if (live && ok) {
        const FaceCtx &cx = ctx[lane];
        const float rs = cx.rs, cs = cx.cs, Ps = rs * cs * cs, Bs = __builtin_sqrtf(Ps);
        const float V[3] = {cx.wn, cx.ut1, cx.ut2};
        float g[7];
        for (int k = 0; k < 7; k++) g[k] = cx.Fc[k] + cx.J * y[k];
        const float Gm = g[0] * rs * cs;
        const float Gp[3] = {g[1] * Ps, g[2] * Ps, g[3] * Ps};
        const float GE = g[4] * Ps * cs + (V[0] * Gp[0] + V[1] * Gp[1] + V[2] * Gp[2]) +
                         0.5f * (V[0] * V[0] + V[1] * V[1] + V[2] * V[2]) * Gm;
        const float Bn = (float)cx.Bn;
        const float Gmom[3] = {Gp[0] + V[0] * Gm, Gp[1] + V[1] * Gm, Gp[2] + V[2] * Gm};
        const float GB[3] = {-cx.wn * Bn, g[5] * Bs * cs - Bn * V[1], g[6] * Bs * cs - Bn * V[2]};
        double A[3][3];
        const double n3[3] = {(double)cx.nrm[0], (double)cx.nrm[1], (double)cx.nrm[2]};
        frame_rows(n3, A);
        double *o = flux + (size_t)NF * f;
        o[MASS] = (double)Gm;
        o[ENER] = (double)GE;
        for (int d = 0; d < 3; d++) {
          o[MOMX + d] = A[0][d] * Gmom[0] + A[1][d] * Gmom[1] + A[2][d] * Gmom[2];
          o[WBX + d] = A[0][d] * GB[0] + A[1][d] * GB[1] + A[2][d] * GB[2];
        }
        o[MPSI] = (double)Gm * (double)(Gm > 0.0f ? cx.psiL : cx.psiR);
        o[MENTR] = (double)Gm * (double)(Gm > 0.0f ? cx.entrL : cx.entrR);
        psi_out[f] = cx.psi;
        Bn_out[f] = cx.Bn;
      }
      // rejected faces gather in the wavefront's list
      const bool rej = live && !ok;
      const unsigned long long m = __ballot(rej);
      const int nr = __popcll(m);
      if (nrej + nr > REJ_N) {
        unsigned long long b0 = 0;
        if (lane == 0) b0 = atomicAdd(fb_count, (unsigned long long)nrej);
        b0 = __shfl(b0, 0);
        for (int i = lane; i < nrej; i += 64) fb_list[b0 + i] = rejs[i];
        nrej = 0;
        wave_sync();
      }
      if (rej) rejs[nrej + __popcll(m & ((1ULL << lane) - 1ULL))] = f;
      nrej += nr;
      wave_sync();
    }
  }
  if constexpr (MODE == 0) {
    // what is left, with one addition to the count for the block
    if (lane == 0) wrej[wv] = (unsigned long long)nrej;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long t = 0;
      for (int w = 0; w < IB / 64; w++) t += wrej[w];
      unsigned long long b0 = t ? atomicAdd(fb_count, t) : 0;
      for (int w = 0; w < IB / 64; w++) {
        const unsigned long long k = wrej[w];
        wrej[w] = b0;
        b0 += k;
      }
    }
    __syncthreads();
    for (int i = lane; i < nrej; i += 64) fb_list[wrej[wv] + i] = rejs[i];
  }
}

// FP64 computeFlux on the rejected faces; passes their number on to the host and
// clears the counter of the next call, so that a call makes two launches and no
// copy (1000 faces: 44 -> 32 us a call)
__global__ void __launch_bounds__(256) k_fallback(const int *list, const unsigned long long *count,
                                                  unsigned long long *next, unsigned long long *host, double gamma,
                                                  const double *wij, const double *Wi, const double *Wj,
                                                  const int *jbnd, const double *nrm, double *psi, double *Bn,
                                                  double *flux) {
  const unsigned long long nf = *count;
  if (gid() == 0) {
    *next = 0;
    *host = nf;
  }
  for (unsigned long long i = (unsigned long long)gid(); i < nf; i += (unsigned long long)gridDim.x * blockDim.x) {
    const int f = list[i];
    double w3[3], L[NF], R[NF], n3[3], F[NF], p, b;
    load_face(f, wij, Wi, Wj, nrm, w3, L, R, n3);
    compute_flux<double>(gamma, w3, L, R, jbnd[f], n3, p, b, F);
    psi[f] = p;
    Bn[f] = b;
    for (int k = 0; k < NF; k++) flux[(size_t)NF * f + k] = F[k];
  }
}

// computeFlux on every face in precision T (the comparison kernels)
template <typename T>
__global__ void __launch_bounds__(256) k_hlld(int n, double gamma, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                       const double *nrm, double *psi, double *Bn, double *flux) {
  const int f = gid();
  if (f >= n) return;
  double w3[3], L[NF], R[NF], n3[3];
  load_face(f, wij, Wi, Wj, nrm, w3, L, R, n3);
  T wt[3], Lt[NF], Rt[NF], nt[3], F[NF], p, b;
  for (int d = 0; d < 3; d++) {
    wt[d] = (T)w3[d];
    nt[d] = (T)n3[d];
  }
  for (int k = 0; k < NF; k++) {
    Lt[k] = (T)L[k];
    Rt[k] = (T)R[k];
  }
  compute_flux<T>((T)gamma, wt, Lt, Rt, jbnd[f], nt, p, b, F);
  psi[f] = (double)p;
  Bn[f] = (double)b;
  for (int k = 0; k < NF; k++) flux[(size_t)NF * f + k] = (double)F[k];
}

}  // namespace sg
}  // namespace fvm

// ===========================================================================
// host side
// ===========================================================================
namespace {
struct Buf {
  void *p = nullptr;
  size_t bytes = 0;
};
}  // namespace

struct fvm_sg {
  int device = 0;
  hipStream_t stream = nullptr;
  double gamma = 5.0 / 3.0;
  std::string err;
  fvm::sg::Gate gate{0.5f, 1.0f, 3.0f, -3.0f};
  fvm::sg::LossW lossw{{1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f}};
  Buf params, grads, am, av, pfrag, pbias;
  Buf X, T;
  long long nsamp = 0, cap = 0;
  Buf xb, tb, y, loss;     // fvm_sg_gradients' batch and outputs; the steps' losses
  Buf tfrag, tops, tcols, tloss;  // training: packed weights; the tiles' operands, FP32 gradients and losses
  Buf stage, fbl, fbc;
  unsigned long long *nfb = nullptr;  // pinned: rejected faces of the last batch
  int fslot = -1;                     // the counter in turn (of the two of fbc); -1: neither is clear
  Buf sx, st, sflag, spos;  // sample staging of one add_faces call
  fvm::ScanScratch scan;
  int adam_t = 0;
  bool packed = false;
};

using namespace fvm::sg;

static int sg_fail(fvm_sg *s, int code, const std::string &m) {
  if (s) s->err = m;
  return code;
}
#define SGCHK(s, call)                                                             \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess) return sg_fail(s, FVM_EHIP, std::string(#call ": ") + hipGetErrorString(e_)); \
  } while (0)

static void sg_release(Buf &b) {
  if (b.p) (void)hipFree(b.p);
  b.p = nullptr;
  b.bytes = 0;
}
static int sg_ensure(fvm_sg *s, Buf &b, size_t bytes, bool keep = false) {
  if (b.bytes >= bytes && b.p) return FVM_OK;
  void *p = nullptr;
  if (hipMalloc(&p, std::max<size_t>(bytes, 256)) != hipSuccess) return sg_fail(s, FVM_EHIP, "hipMalloc failed");
  if (keep && b.p && b.bytes) (void)hipMemcpy(p, b.p, b.bytes, hipMemcpyDeviceToDevice);
  sg_release(b);
  b.p = p;
  b.bytes = std::max<size_t>(bytes, 256);
  return FVM_OK;
}
static unsigned nblk(long long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// fragments of the current parameters for the training kernels; their padding
// is cleared when they are first allocated
static int train_pack(fvm_sg *s) {
  if (!s->tfrag.p) {
    int rc = sg_ensure(s, s->tfrag, sizeof(__bf16) * (size_t)T_FRAG);
    if (rc) return rc;
    SGCHK(s, hipMemsetAsync(s->tfrag.p, 0, s->tfrag.bytes, s->stream));
  }
  hipLaunchKernelGGL(k_train_pack, dim3(nblk(NPARAM)), dim3(256), 0, s->stream, (const float *)s->params.p,
                     (__bf16 *)s->tfrag.p);
  SGCHK(s, hipGetLastError());
  return FVM_OK;
}
// buffers of a batch of B samples, and what both launches of a step share
static int train_args(fvm_sg *s, int B, float lam, TrainArgs &A, GradArgs &D) {
  const size_t nt = ((size_t)B + TS - 1) / TS;
  int rc;
  if ((rc = train_pack(s)) || (rc = sg_ensure(s, s->tops, sizeof(__bf16) * N_OP * OP_E * nt)) ||
      (rc = sg_ensure(s, s->tcols, sizeof(float) * N_COL * COL_E * nt)) || (rc = sg_ensure(s, s->tloss, sizeof(float) * nt)))
    return rc;
  A = TrainArgs{};
  A.B = B;
  A.frag = (const __bf16 *)s->tfrag.p;
  A.P = (const float *)s->params.p;
  A.lam = lam;
  A.lw = s->lossw;
  A.ops = (__bf16 *)s->tops.p;
  A.cols = (float *)s->tcols.p;
  A.tloss = (float *)s->tloss.p;
  D = GradArgs{};
  D.ntile = (int)nt;
  D.ops = A.ops;
  D.cols = A.cols;
  D.tloss = A.tloss;
  D.G = (float *)s->grads.p;
  D.P = (float *)s->params.p;
  D.M = (float *)s->am.p;
  D.V = (float *)s->av.p;
  D.frag = (__bf16 *)s->tfrag.p;
  return FVM_OK;
}

static int pack(fvm_sg *s) {
  if (s->packed) return FVM_OK;
  int rc;
  if ((rc = sg_ensure(s, s->pfrag, (size_t)P_BF * 2)) || (rc = sg_ensure(s, s->pbias, (size_t)P_BIAS * 4))) return rc;
  hipLaunchKernelGGL(k_pack, dim3(nblk(P_BF)), dim3(256), 0, s->stream, (const float *)s->params.p,
                     (__bf16 *)s->pfrag.p, (float *)s->pbias.p);
  SGCHK(s, hipGetLastError());
  s->packed = true;
  return FVM_OK;
}

// one block a CU, all resident: the weights are loaded once (over 1024 blocks:
// 10^6 faces 15 us more)
static unsigned infer_grid(int n) {
  const unsigned nb = (unsigned)(((long long)n + IB - 1) / IB);
  return std::max(1u, std::min(nb, 256u));
}

template <int MODE>
static int launch_infer(fvm_sg *s, int n, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                        const double *nrm, double *psi, double *Bn, double *flux, int *fbl,
                        unsigned long long *fbc, const float *xin, float *yout) {
  static bool attr = false;
  if (!attr) {
    SGCHK(s, hipFuncSetAttribute((const void *)k_infer<MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_B));
    attr = true;
  }
  hipLaunchKernelGGL(k_infer<MODE>, dim3(infer_grid(n)), dim3(IB), LDS_B, s->stream, n, s->gamma, wij, Wi, Wj, jbnd,
                     nrm, (const __bf16 *)s->pfrag.p, (const float *)s->pbias.p, s->gate, psi, Bn, flux, fbl, fbc,
                     xin, yout);
  SGCHK(s, hipGetLastError());
  return FVM_OK;
}

// surrogate fluxes of a batch and the FP64 fluxes of the faces it rejects
static int launch_flux(fvm_sg *s, int n, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                       const double *nrm, double *psi, double *Bn, double *flux) {
  int rc;
  if ((rc = sg_ensure(s, s->fbl, sizeof(int) * (size_t)n)) ||
      (rc = sg_ensure(s, s->fbc, 2 * sizeof(unsigned long long))))
    return rc;
  unsigned long long *cnt = (unsigned long long *)s->fbc.p;
  if (s->fslot < 0) SGCHK(s, hipMemsetAsync(cnt, 0, 2 * sizeof(unsigned long long), s->stream));
  const int slot = s->fslot < 0 ? 0 : s->fslot;
  s->fslot = -1;  // until both launches are made
  if ((rc = launch_infer<0>(s, n, wij, Wi, Wj, jbnd, nrm, psi, Bn, flux, (int *)s->fbl.p, cnt + slot, nullptr, nullptr)))
    return rc;
  hipLaunchKernelGGL(k_fallback, dim3(std::min(nblk(n), 1024u)), dim3(256), 0, s->stream, (const int *)s->fbl.p,
                     cnt + slot, cnt + (slot ^ 1), s->nfb, s->gamma, wij, Wi, Wj, jbnd, nrm, psi, Bn, flux);
  SGCHK(s, hipGetLastError());
  s->fslot = slot ^ 1;
  return FVM_OK;
}

int fvm_sg_device_weights(fvm_sg *s, const void **frag, const float **bias, float gate[4]) {
  if (!s || !frag || !bias || !gate) return FVM_EARG;
  (void)hipSetDevice(s->device);
  int rc = pack(s);
  if (rc) return rc;
  SGCHK(s, hipStreamSynchronize(s->stream));
  *frag = s->pfrag.p;
  *bias = (const float *)s->pbias.p;
  gate[0] = s->gate.max_log_rho;
  gate[1] = s->gate.max_log_p;
  gate[2] = s->gate.max_vn;
  gate[3] = s->gate.max_log10_err;
  return FVM_OK;
}

int fvm_sg_device_of(const fvm_sg *s) { return s ? s->device : -1; }

extern "C" {

int fvm_sg_create(fvm_sg **out, int device, double gamma_gas) {
  if (!out) return FVM_EARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return FVM_EHIP;
  fvm_sg *s = new (std::nothrow) fvm_sg();
  if (!s) return FVM_EARG;
  s->device = device;
  s->gamma = gamma_gas;
  (void)hipSetDevice(device);
  if (hipStreamCreate(&s->stream) != hipSuccess) {
    delete s;
    return FVM_EHIP;
  }
  if (sg_ensure(s, s->params, 4 * NPARAM) || sg_ensure(s, s->grads, 4 * NPARAM) || sg_ensure(s, s->am, 4 * NPARAM) ||
      sg_ensure(s, s->av, 4 * NPARAM) ||
      hipHostMalloc((void **)&s->nfb, sizeof(unsigned long long), hipHostMallocDefault) != hipSuccess) {
    fvm_sg_destroy(s);
    return FVM_EHIP;
  }
  (void)hipMemset(s->params.p, 0, 4 * NPARAM);
  (void)hipMemset(s->am.p, 0, 4 * NPARAM);
  (void)hipMemset(s->av.p, 0, 4 * NPARAM);
  *out = s;
  return FVM_OK;
}

void fvm_sg_destroy(fvm_sg *s) {
  if (!s) return;
  (void)hipSetDevice(s->device);
  for (Buf *b : {&s->params, &s->grads, &s->am, &s->av, &s->pfrag, &s->pbias, &s->X, &s->T, &s->xb, &s->tb, &s->y,
                 &s->loss, &s->tfrag, &s->tops, &s->tcols, &s->tloss, &s->stage, &s->fbl, &s->fbc,
                 &s->sx, &s->st, &s->sflag, &s->spos})
    sg_release(*b);
  if (s->nfb) (void)hipHostFree(s->nfb);
  fvm::scan_release(s->scan);
  if (s->stream) (void)hipStreamDestroy(s->stream);
  delete s;
}

const char *fvm_sg_last_error(const fvm_sg *s) { return s ? s->err.c_str() : "null handle"; }

int fvm_sg_set_params(fvm_sg *s, const float *params, int n) {
  if (!s || !params || n != NPARAM) return sg_fail(s, FVM_EARG, "set_params: need FVM_SG_NPARAM floats");
  (void)hipSetDevice(s->device);
  SGCHK(s, hipMemcpyAsync(s->params.p, params, 4 * (size_t)NPARAM, hipMemcpyHostToDevice, s->stream));
  SGCHK(s, hipMemsetAsync(s->am.p, 0, 4 * NPARAM, s->stream));
  SGCHK(s, hipMemsetAsync(s->av.p, 0, 4 * NPARAM, s->stream));
  SGCHK(s, hipStreamSynchronize(s->stream));
  s->adam_t = 0;
  s->packed = false;
  return FVM_OK;
}

int fvm_sg_get_params(fvm_sg *s, float *params, int n) {
  if (!s || !params || n != NPARAM) return sg_fail(s, FVM_EARG, "get_params: need FVM_SG_NPARAM floats");
  (void)hipSetDevice(s->device);
  SGCHK(s, hipMemcpyAsync(params, s->params.p, 4 * (size_t)NPARAM, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipStreamSynchronize(s->stream));
  return FVM_OK;
}

int fvm_sg_set_loss_weights(fvm_sg *s, const double *w, int n) {
  if (!s || !w || n != 7) return sg_fail(s, FVM_EARG, "set_loss_weights: need 7 weights");
  for (int k = 0; k < 7; k++) {
    if (!(w[k] > 0.0)) return sg_fail(s, FVM_EARG, "set_loss_weights: weights must be positive");
    s->lossw.w[k] = (float)w[k];
  }
  return FVM_OK;
}

int fvm_sg_set_gate(fvm_sg *s, const fvm_sg_gate *g) {
  if (!s || !g) return sg_fail(s, FVM_EARG, "set_gate: NULL");
  s->gate = Gate{(float)g->max_log_rho_jump, (float)g->max_log_p_jump, (float)g->max_vn, (float)g->max_log10_err};
  return FVM_OK;
}

static int stage_faces(fvm_sg *s, int n, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                       const double *normal, bool outputs, double **d) {
  const size_t N = (size_t)n;
  const size_t nd = (3 + 10 + 10 + 3 + (outputs ? 12 : 0)) * N;
  int rc = sg_ensure(s, s->stage, sizeof(double) * nd + sizeof(int) * N + 64);
  if (rc) return rc;
  double *b = (double *)s->stage.p;
  d[0] = b;
  d[1] = d[0] + 3 * N;
  d[2] = d[1] + 10 * N;
  d[3] = d[2] + 10 * N;
  d[4] = d[3] + 3 * N;  // outputs: psi, Bn, flux
  d[5] = d[4] + N;
  d[6] = d[5] + N;
  d[7] = (double *)((char *)s->stage.p + sizeof(double) * nd);  // jbnd
  SGCHK(s, hipMemcpyAsync(d[0], wij, sizeof(double) * 3 * N, hipMemcpyHostToDevice, s->stream));
  SGCHK(s, hipMemcpyAsync(d[1], Wi, sizeof(double) * 10 * N, hipMemcpyHostToDevice, s->stream));
  SGCHK(s, hipMemcpyAsync(d[2], Wj, sizeof(double) * 10 * N, hipMemcpyHostToDevice, s->stream));
  SGCHK(s, hipMemcpyAsync(d[3], normal, sizeof(double) * 3 * N, hipMemcpyHostToDevice, s->stream));
  SGCHK(s, hipMemcpyAsync(d[7], jbnd, sizeof(int) * N, hipMemcpyHostToDevice, s->stream));
  return FVM_OK;
}

int fvm_sg_add_faces(fvm_sg *s, int n, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                     const double *normal, int *n_kept) {
  if (!s || n < 0) return sg_fail(s, FVM_EARG, "add_faces: bad arguments");
  if (n == 0) {
    if (n_kept) *n_kept = 0;
    return FVM_OK;
  }
  if (!wij || !Wi || !Wj || !jbnd || !normal) return sg_fail(s, FVM_EARG, "add_faces: NULL array");
  (void)hipSetDevice(s->device);
  int rc;
  const long long need = s->nsamp + n;
  if (need > s->cap) {
    const long long cap = std::max(need, 2 * s->cap);
    if ((rc = sg_ensure(s, s->X, 4 * (size_t)cap * NIN, true)) || (rc = sg_ensure(s, s->T, 4 * (size_t)cap * NOUT, true)))
      return rc;
    s->cap = cap;
  }
  double *d[8];
  if ((rc = stage_faces(s, n, wij, Wi, Wj, jbnd, normal, false, d))) return rc;
  if ((rc = sg_ensure(s, s->sx, sizeof(float) * NIN * (size_t)n)) ||
      (rc = sg_ensure(s, s->st, sizeof(float) * NOUT * (size_t)n)) || (rc = sg_ensure(s, s->sflag, sizeof(int) * (size_t)n)) ||
      (rc = sg_ensure(s, s->spos, sizeof(int) * (size_t)n)))
    return rc;
  hipLaunchKernelGGL(k_samples, dim3(nblk(n)), dim3(256), 0, s->stream, n, s->gamma, d[0], d[1], d[2],
                     (const int *)d[7], d[3], s->gate, (float *)s->sx.p, (float *)s->st.p, (int *)s->sflag.p);
  SGCHK(s, hipGetLastError());
  int kept = 0;
  if (fvm::exclusive_scan_flags(s->scan, (const int *)s->sflag.p, (int *)s->spos.p, n, &kept, s->stream))
    return sg_fail(s, FVM_EHIP, "add_faces: sample scan failed");
  hipLaunchKernelGGL(k_pack_samples, dim3(nblk(n)), dim3(256), 0, s->stream, n, (const int *)s->sflag.p,
                     (const int *)s->spos.p, (const float *)s->sx.p, (const float *)s->st.p, (float *)s->X.p,
                     (float *)s->T.p, s->nsamp);
  SGCHK(s, hipGetLastError());
  SGCHK(s, hipStreamSynchronize(s->stream));
  s->nsamp += (long long)kept;
  if (n_kept) *n_kept = (int)kept;
  return FVM_OK;
}

int fvm_sg_clear_samples(fvm_sg *s) {
  if (!s) return FVM_EARG;
  s->nsamp = 0;
  return FVM_OK;
}

int fvm_sg_num_samples(fvm_sg *s, long long *n) {
  if (!s || !n) return FVM_EARG;
  *n = s->nsamp;
  return FVM_OK;
}

int fvm_sg_get_samples(fvm_sg *s, long long first, int n, float *x, float *t) {
  if (!s || n < 0 || first < 0 || first + n > s->nsamp || !x || !t) return sg_fail(s, FVM_EARG, "get_samples: range");
  (void)hipSetDevice(s->device);
  SGCHK(s, hipMemcpyAsync(x, (float *)s->X.p + first * NIN, 4 * (size_t)n * NIN, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipMemcpyAsync(t, (float *)s->T.p + first * NOUT, 4 * (size_t)n * NOUT, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipStreamSynchronize(s->stream));
  return FVM_OK;
}

int fvm_sg_train(fvm_sg *s, int steps, int batch, double lr, double lam, unsigned long long seed, float *loss_hist) {
  if (!s || steps < 0 || batch < 64 || !(lr > 0.0)) return sg_fail(s, FVM_EARG, "train: bad arguments");
  if (s->nsamp < 1) return sg_fail(s, FVM_ESTATE, "train: no samples");
  (void)hipSetDevice(s->device);
  int rc;
  TrainArgs A;
  GradArgs D;
  if ((rc = train_args(s, batch, (float)lam, A, D)) || (rc = sg_ensure(s, s->loss, 4 * (size_t)std::max(steps, 1)))) return rc;
  A.X = (const float *)s->X.p;
  A.T = (const float *)s->T.p;
  A.nsamp = s->nsamp;
  A.seed = seed;
  D.lr = (float)lr;
  D.b1 = 0.9f;
  D.b2 = 0.999f;
  D.eps = 1e-8f;
  for (int k = 0; k < steps; k++) {
    A.step = (unsigned long long)s->adam_t;
    hipLaunchKernelGGL(k_train_tile<true>, dim3(D.ntile), dim3(TB), 0, s->stream, A);
    s->adam_t++;
    D.c1 = 1.0f - powf(D.b1, (float)s->adam_t);
    D.c2 = 1.0f - powf(D.b2, (float)s->adam_t);
    D.loss = (float *)s->loss.p + k;
    hipLaunchKernelGGL(k_train_grad<true>, dim3(GRAD_BLOCKS), dim3(64), 0, s->stream, D);
    SGCHK(s, hipGetLastError());
  }
  s->packed = false;
  if (loss_hist && steps > 0)
    SGCHK(s, hipMemcpyAsync(loss_hist, s->loss.p, 4 * (size_t)steps, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipStreamSynchronize(s->stream));
  return FVM_OK;
}

int fvm_sg_gradients(fvm_sg *s, int n, const float *x, const float *t, double lam, float *y, float *grads,
                     double *loss) {
  if (!s || n < 1 || !x || !t) return sg_fail(s, FVM_EARG, "gradients: bad arguments");
  (void)hipSetDevice(s->device);
  int rc;
  TrainArgs A;
  GradArgs D;
  if ((rc = train_args(s, n, (float)lam, A, D)) || (rc = sg_ensure(s, s->xb, 4 * (size_t)n * NIN)) ||
      (rc = sg_ensure(s, s->tb, 4 * (size_t)n * NOUT)) || (rc = sg_ensure(s, s->y, 4 * (size_t)n * NOUT)) ||
      (rc = sg_ensure(s, s->loss, 4)))
    return rc;
  SGCHK(s, hipMemcpyAsync(s->xb.p, x, 4 * (size_t)n * NIN, hipMemcpyHostToDevice, s->stream));
  SGCHK(s, hipMemcpyAsync(s->tb.p, t, 4 * (size_t)n * NOUT, hipMemcpyHostToDevice, s->stream));
  A.X = (const float *)s->xb.p;
  A.T = (const float *)s->tb.p;
  A.Y = (float *)s->y.p;
  D.loss = (float *)s->loss.p;
  hipLaunchKernelGGL(k_train_tile<false>, dim3(D.ntile), dim3(TB), 0, s->stream, A);
  hipLaunchKernelGGL(k_train_grad<false>, dim3(GRAD_BLOCKS), dim3(64), 0, s->stream, D);
  SGCHK(s, hipGetLastError());
  float l = 0.0f;
  if (y) SGCHK(s, hipMemcpyAsync(y, s->y.p, 4 * (size_t)n * NOUT, hipMemcpyDeviceToHost, s->stream));
  if (grads) SGCHK(s, hipMemcpyAsync(grads, s->grads.p, 4 * (size_t)NPARAM, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipMemcpyAsync(&l, s->loss.p, 4, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipStreamSynchronize(s->stream));
  if (loss) *loss = (double)l;
  return FVM_OK;
}

int fvm_sg_forward(fvm_sg *s, int n, const float *x, float *y) {
  if (!s || n < 0 || (n > 0 && (!x || !y))) return sg_fail(s, FVM_EARG, "forward: bad arguments");
  if (n == 0) return FVM_OK;
  (void)hipSetDevice(s->device);
  int rc;
  if ((rc = pack(s)) || (rc = sg_ensure(s, s->stage, 4 * (size_t)n * (NIN + NOUT)))) return rc;
  float *dx = (float *)s->stage.p, *dy = dx + (size_t)n * NIN;
  SGCHK(s, hipMemcpyAsync(dx, x, 4 * (size_t)n * NIN, hipMemcpyHostToDevice, s->stream));
  if ((rc = launch_infer<1>(s, n, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                            nullptr, dx, dy)))
    return rc;
  SGCHK(s, hipMemcpyAsync(y, dy, 4 * (size_t)n * NOUT, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipStreamSynchronize(s->stream));
  return FVM_OK;
}

int fvm_sg_compute_flux_device(fvm_sg *s, int n, const double *wij, const double *Wi, const double *Wj,
                               const int *jbnd, const double *normal, double *psi, double *Bn, double *flux,
                               int *n_fallback) {
  if (!s || n < 0) return sg_fail(s, FVM_EARG, "compute_flux: bad arguments");
  if (n == 0) {
    if (n_fallback) *n_fallback = 0;
    return FVM_OK;
  }
  if (!wij || !Wi || !Wj || !jbnd || !normal || !psi || !Bn || !flux)
    return sg_fail(s, FVM_EARG, "compute_flux: NULL array");
  (void)hipSetDevice(s->device);
  int rc;
  if ((rc = pack(s)) || (rc = launch_flux(s, n, wij, Wi, Wj, jbnd, normal, psi, Bn, flux))) return rc;
  SGCHK(s, hipStreamSynchronize(s->stream));
  if (n_fallback) *n_fallback = (int)*s->nfb;
  return FVM_OK;
}

int fvm_sg_compute_flux(fvm_sg *s, int n, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                        const double *normal, double *psi, double *Bn, double *flux, int *n_fallback) {
  if (!s || n < 0) return sg_fail(s, FVM_EARG, "compute_flux: bad arguments");
  if (n == 0) {
    if (n_fallback) *n_fallback = 0;
    return FVM_OK;
  }
  if (!wij || !Wi || !Wj || !jbnd || !normal || !psi || !Bn || !flux)
    return sg_fail(s, FVM_EARG, "compute_flux: NULL array");
  (void)hipSetDevice(s->device);
  double *d[8];
  int rc = stage_faces(s, n, wij, Wi, Wj, jbnd, normal, true, d);
  if (rc) return rc;
  if ((rc = fvm_sg_compute_flux_device(s, n, d[0], d[1], d[2], (const int *)d[7], d[3], d[4], d[5], d[6], n_fallback)))
    return rc;
  const size_t N = (size_t)n;
  SGCHK(s, hipMemcpyAsync(psi, d[4], sizeof(double) * N, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipMemcpyAsync(Bn, d[5], sizeof(double) * N, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipMemcpyAsync(flux, d[6], sizeof(double) * 10 * N, hipMemcpyDeviceToHost, s->stream));
  SGCHK(s, hipStreamSynchronize(s->stream));
  return FVM_OK;
}

int fvm_sg_time_flux(fvm_sg *s, int n, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                     const double *normal, int iters, double *ms, int *n_fallback) {
  if (!s || n < 1 || iters < 1 || !ms) return sg_fail(s, FVM_EARG, "time_flux: bad arguments");
  (void)hipSetDevice(s->device);
  double *d[8];
  int rc = stage_faces(s, n, wij, Wi, Wj, jbnd, normal, true, d);
  if (rc) return rc;
  const int *jb = (const int *)d[7];
  if ((rc = fvm_sg_compute_flux_device(s, n, d[0], d[1], d[2], jb, d[3], d[4], d[5], d[6], n_fallback))) return rc;
  hipEvent_t e[4];
  for (auto &x : e) SGCHK(s, hipEventCreate(&x));
  SGCHK(s, hipEventRecord(e[0], s->stream));
  for (int k = 0; k < iters; k++)
    if ((rc = launch_flux(s, n, d[0], d[1], d[2], jb, d[3], d[4], d[5], d[6]))) return rc;
  SGCHK(s, hipEventRecord(e[1], s->stream));
  for (int k = 0; k < iters; k++)
    hipLaunchKernelGGL(k_hlld<double>, dim3(nblk(n)), dim3(256), 0, s->stream, n, s->gamma, d[0], d[1], d[2], jb, d[3],
                       d[4], d[5], d[6]);
  SGCHK(s, hipEventRecord(e[2], s->stream));
  for (int k = 0; k < iters; k++)
    hipLaunchKernelGGL(k_hlld<float>, dim3(nblk(n)), dim3(256), 0, s->stream, n, s->gamma, d[0], d[1], d[2], jb, d[3],
                       d[4], d[5], d[6]);
  SGCHK(s, hipEventRecord(e[3], s->stream));
  SGCHK(s, hipGetLastError());
  SGCHK(s, hipEventSynchronize(e[3]));
  for (int k = 0; k < 3; k++) {
    float t = 0.0f;
    SGCHK(s, hipEventElapsedTime(&t, e[k], e[k + 1]));
    ms[k] = (double)t / iters;
  }
  for (auto &x : e) (void)hipEventDestroy(x);
  return FVM_OK;
}

}  // extern "C"
