// The ONLY_DIAG Classic model on the device (getFM_diag_tnlm_vect_cls_,
// src/bsa/functions/functionsImpl.F90:1747-1970; getRM_diag_vect_cls_,
// :1975-2101): loaded nodes without coherence between them and only the
// diagonal modal entries.  Per mode m, with W_m(k) = Psi_q Psi_l^2 of the K
// index k = (component, node) and S_k the nodal PSD,
//   B_m(f1, f2) = 2 sum_k W_m(k) [S_k(f1) S_k(f2) + S_k(f1+f2) S_k(f2) + S_k(f1+f2) S_k(f1)]
//               = 2 [T_m(|f1|, |f2|) + T_m(|f1+f2|, |f2|) + T_m(|f1+f2|, |f1|)],
//   T_m(u, v)   = sum_k S_k(u) W_m(k) S_k(v),
// with S(f1+f2) = 0 beyond +-fmax (the reference's zero padding), and
// psd_m(f) = sum_k Psi_l^2 S_k(f).  The moments integrate B_m and psd_m with
// the response factors Re[H_m(f1) H_m(f2) conj H_m(f1+f2)] and |H_m(f)|^2.
// T_m is G[m](m,u; m,v) of the full model for a structure of that one mode with the
// table S and Psi_b = W_m: the third moments are its contraction with the plane
// epilogue (k_gsym_diag), each T value formed once and never stored, and the second
// moments its modal PSD kernel (k_m2 with diag).  Bound by launches and latency at
// these sizes: T stored by a GEMM per mode, read back over the whole plane and a
// serial loop over k per PSD value took 530 us for 500 nodes with 2 components, 20
// modes, 257 frequencies; now 64 us, with the 15 us of k_m2 beside.  Selected bispectra
// still store their T_m (one GEMM per mode).

// X[k*ldX + u] = S_k(u df), zero for u >= nh and in the padding rows k >= kv; from the
// nodal parameters prm, formula as k_psd_sqrt.  grid (ceil(ldX/64), K), block 64
__global__ void k_diag_psd(const double *__restrict__ fl, int nh, int nnl, int kv,
                           const double *__restrict__ prm, const int *__restrict__ formula,
                           int pulsation, long ldX, double *__restrict__ X)
{
   const int u = blockIdx.x * 64 + threadIdx.x;
   const int k = blockIdx.y;
   if (u >= ldX) return;
   double s = 0.0;
   if (k < kv && u < nh) s = psd_sqrt(prm + (size_t)k * 4, formula[k / nnl], fl[u], pulsation);
   X[(size_t)k * ldX + u] = s * s;
}

// W[m*K + k] = Psi_q Psi_l^2, A2[m*K + k] = Psi_l^2
__global__ void k_diag_weights(const double *__restrict__ pa, const double *__restrict__ pb, long n,
                               double *__restrict__ W, double *__restrict__ A2)
{
   const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (t >= n) return;
   const double a = pa[t];
   W[t] = pb[t] * a * a;
   A2[t] = a * a;
}

// Y[(m*K + k)*ldX + u] = W_m(k) X[k*ldX + u]; grid (ceil(ldX/64), K, nm), block 64
__global__ void k_diag_scaled(const double *__restrict__ X, long ldX, const double *__restrict__ W,
                              int K, double *__restrict__ Y)
{
   const int u = blockIdx.x * 64 + threadIdx.x;
   const int k = blockIdx.y, m = blockIdx.z;
   if (u < ldX) Y[((size_t)m * K + k) * ldX + u] = W[(size_t)m * K + k] * X[(size_t)k * ldX + u];
}

// Diagonal bispectra of selected modes on the Classic grid from T, by the
// formula of B_m above: out[q1 + nf*q2 + nf*nf*s] for mode sel[s] (the reference's
// bisp(i, j, m) of getFM_diag_tnlm_vect_cls_ / getRM_diag_vect_cls_).
// grid (ceil(nf*nf/256), nsel), block 256
__global__ __launch_bounds__(256) void k_diag_bisp_sel(const double *__restrict__ T, int nh,
                                                       const double2 *__restrict__ H, int nft,
                                                       const int *__restrict__ sel,
                                                       double *__restrict__ bfm,
                                                       double *__restrict__ brm)
{
   const int n = nh - 1, nf = 2 * nh - 1;
   const long npts = (long)nf * nf;
   const long pt = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (pt >= npts) return;
   const int m = sel[blockIdx.y];
   const double *Tm = T + (size_t)m * nh * nh;
   const int F1 = (int)(pt % nf) - n, F2 = (int)(pt / nf) - n, s = F1 + F2;
   const int a1 = abs(F1), a2 = abs(F2), as = abs(s);
   double b = Tm[a1 + (size_t)a2 * nh];
   if (as <= n) b += Tm[as + (size_t)a2 * nh] + Tm[as + (size_t)a1 * nh];
   b *= 2.0;
   const size_t o = (size_t)blockIdx.y * npts + pt;
   if (bfm) bfm[o] = b;
   if (brm) brm[o] = b * re3(hget(H, nft, m, F1), hget(H, nft, m, F2), hget(H, nft, m, s));
}

// Diagonal-model force bispectrum at points, the Mesher's ONLY_DIAG BFM
// (getFM_diag_tnm_scalar_msh_, functionsImpl.F90:1123-1216, with S(f1+f2) in
// its second and third products as the Classic model has them):
//   out[slot[q]*nm + m] = 2 sum_k W_m(k) [S_k(f1) S_k(f2) + S_k(f1+f2) (S_k(f2) + S_k(f1))],
// W_m(k) = Psi_q Psi_l^2, S_k = sq^2 from the table sq[(c*nu + u)*nnl + n] at rows
// i1, i2, i3 (|f1|, |f2|, |f1+f2|).  grid (ceil(npts*nm/256)), block 256
__global__ __launch_bounds__(256) void k_diag_points(
   const double *__restrict__ sq, int nu, int nnl, int kv, const double *__restrict__ pa,
   const double *__restrict__ pb, int K, int nm, int npts, const int *__restrict__ i1,
   const int *__restrict__ i2, const int *__restrict__ i3, const long *__restrict__ slot,
   double *__restrict__ out)
{
   const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (gid >= (long)npts * nm) return;
   const int q = (int)(gid / nm), m = (int)(gid % nm);
   const int a1 = i1[q], a2 = i2[q], a3 = i3[q];
   double s = 0.0;
   for (int k = 0; k < kv; ++k) {                      // rows k >= kv are padding
      const int c = k / nnl, n = k % nnl;
      const double *col = sq + (size_t)c * nu * nnl + n;
      const double r1 = col[(size_t)a1 * nnl], r2 = col[(size_t)a2 * nnl];
      const double r3 = a3 >= 0 ? col[(size_t)a3 * nnl] : 0.0;
      const double S1 = r1 * r1, S2 = r2 * r2, S3 = r3 * r3;
      const double a = pa[(size_t)m * K + k], b = pb[(size_t)m * K + k];
      s += b * a * a * (S1 * S2 + S3 * S2 + S3 * S1);
   }
   out[(size_t)slot[q] * nm + m] = 2.0 * s;
}
