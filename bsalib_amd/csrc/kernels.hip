// Device kernels of the BFM hot path for gfx950 (CDNA4).
//
// Notation (the reference's, src/bsa/functions/functionsImpl.F90:1312-1587):
//   nodes i,j,k (NNL loaded), modes m,n,p (NM kept), components tc (NTC),
//   Psi_a / Psi_b = phi_times_A_ndegw_(:,:,tc) / (:,:,tc+3),
//   S_ij(f) = rho_ij^|f| sqrt(S_i(f) S_j(f)),   A(n,i;f) = sum_j Psi_a(n,j) S_ji(f).
// The reference's modal force bispectrum is
//   B(m,n,p)(f1,f2) = 2 sum_tc [ G[m](n,f1; p,f2) + G[n](m,f3; p,f2) + G[p](m,f3; n,f1) ],
//   G[x](y,f; z,g)  = sum_i Psi_b(x,i) A(y,i;f) A(z,i;g),          f3 = f1 + f2,
// i.e. its three node sums (functionsImpl.F90:1523-1528) are one tensor G read
// at three argument permutations.  G is symmetric in (y,f)<->(z,g) and depends
// on |f|, |g| only (PSD and coherence are even in f).  k_gsym_f64 computes each
// distinct G value once on FP64 MFMA and its epilogue adds it, weighted by the
// quadrature weight and the modal FRF product, to the up to 12 (m,n,p,f1,f2)
// places it occupies in the plane.
//
// K index of every contraction: k = tc*NNLp + i (NNLp = NNL padded, zeros).
// U table (A values): U[k*ldU + y*nhp + u], u = |f|/df on the half grid.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

typedef double d4 __attribute__((ext_vector_type(4)));

#define KC 32          // table K rows are padded to a multiple of this

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__global__ void k_fill(double *__restrict__ p, size_t n, double v)
{
   size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
   const size_t st = (size_t)gridDim.x * blockDim.x;
   for (; i < n; i += st) p[i] = v;
}

// U[k*ld + c] = 0 for c >= c0, the first n / (ld - c0) rows
__global__ void k_zero_tail(double *__restrict__ U, long ld, long c0, long n)
{
   const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (t >= n) return;
   const long w = ld - c0;
   U[t / w * ld + c0 + t % w] = 0.0;
}

// Nodal one-sided PSD, then its square root, on a list of |f| values.
// formula: 1 von Karman u (WindPSDImpl.F90:166-188), 2 von Karman v/w (:190-222),
// 3 Davenport-Greisch (:249-277), 5 Davenport-Uliege (:283-316), 0 zero (Kaimal,
// :231-243).  Pulsation convention divides by 4 pi (:143).
// prm[(tc*nnl + i)*4 + {0,1,2,3}] = {L, sigma, U_node, U_mean_ref(zone)}.
__device__ __forceinline__ double psd_sqrt(const double *__restrict__ pp, int formula, double f,
                                           int pulsation)
{
   const double L = pp[0], sg = pp[1], U = pp[2], Um = pp[3];
   double S = 0.0;
   switch (formula) {
   case 1: {
      const double LU = L / U;
      const double x = f * LU;
      S = 4.0 * (LU * sg * sg) / pow(1.0 + 70.7 * x * x, 5.0 / 6.0);
   } break;
   case 2: {
      double d = 2.0 * f * (L / U);
      d = d * d;
      const double r2 = pow(1.0 + 70.7 * d, 11.0 / 6.0) * U;
      S = 4.0 * (L * (1.0 + 188.4 * d) / r2 * (sg * sg));
   } break;
   case 3: {
      const double c = 0.65 * 1200.0;
      const double x = c * f / Um;
      S = (c * sg * sg / Um) / pow(1.0 + x * x, 5.0 / 6.0);
   } break;
   case 5: {
      const double cLU = L / U;
      const double cF = f * cLU;
      S = ((2.0 / 3.0) * cF * cLU * (sg * sg)) / pow(1.0 + cF * cF, 4.0 / 3.0);
   } break;
   default: S = 0.0;
   }
   if (pulsation) S = S / (4.0 * M_PI);
   return sqrt(S);
}

__global__ void k_psd_sqrt(const double *__restrict__ fabs_list, int nfl,
                           const double *__restrict__ prm, const int *__restrict__ formula,
                           int nnl, int ntc, int pulsation, double *__restrict__ sq)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   const int q = blockIdx.y;
   const int tc = blockIdx.z;
   if (i >= nnl || q >= nfl) return;
   sq[((size_t)tc * nfl + q) * nnl + i] =
      psd_sqrt(prm + ((size_t)tc * nnl + i) * 4, formula[tc], fabs_list[q], pulsation);
}

// ln rho_ji for the loaded nodes from the packed coherence vector
// (util_getCorrVectIndex, src/utils/utility.F90:60-79): lnr[c][j][i].
// col[c] is the 0-based nod_corr column of component c; clamp > 0 replaces
// rho < clamp by clamp (BsaCL convention, bsacl.cl:243-245).
__global__ void k_lnrho(const double *__restrict__ corr, long ncorr_rows, const int *__restrict__ col,
                        const int *__restrict__ n_load, int nnl, long nn, double clamp,
                        double *__restrict__ lnr)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   const int j = blockIdx.y;
   const int c = blockIdx.z;
   if (i >= nnl || j >= nnl) return;
   long a = n_load[j], b = n_load[i];
   if (a > b) {
      const long t = a;
      a = b;
      b = t;
   }
   const long id = (a - 1) * nn + b - (a * a - a) / 2;
   double r = corr[(size_t)col[c] * ncorr_rows + (id - 1)];
   if (clamp > 0.0 && r < clamp) r = clamp;
   lnr[((size_t)c * nnl + j) * nnl + i] = log(r);
}

// Modal FRF table H[m*nft + q] = 1/(K - w^2 M + i w C), w = 2 pi q df, q >= 0
// (functionsImpl.F90:1641-1651).  Negative frequencies use conj.
__device__ __forceinline__ double2 frf_grid(const double *__restrict__ Mm,
                                            const double *__restrict__ Km,
                                            const double *__restrict__ Cm, int m, int q, double df)
{
   const double w = 2.0 * M_PI * ((double)q * df);
   const double r = -(w * w * Mm[m]) + Km[m];
   const double im = w * Cm[m];
   const double d = r * r + im * im;
   return make_double2(r / d, -im / d);
}

__global__ void k_frf_table(const double *__restrict__ Mm, const double *__restrict__ Km,
                            const double *__restrict__ Cm, int nm, int nft, double df,
                            double2 *__restrict__ H)
{
   const int q = blockIdx.x * blockDim.x + threadIdx.x;
   const int m = blockIdx.y;
   if (q >= nft || m >= nm) return;
   H[(size_t)m * nft + q] = frf_grid(Mm, Km, Cm, m, q, df);
}

// ---------------------------------------------------------------------------
// projection A(y,i;f) = s_i(f) sum_j Psi_a(y,j) s_j(f) exp(|f| ln rho_ji) on
// FP64 MFMA: per frequency an (MT*16 x nnl) x (nnl x 16) product per wave.  The right
// operand s_j rho_ji^|f| is formed in the lane that feeds it to the MFMA, once for all
// modes, so the waves need no LDS and no barrier.  A wave takes F frequencies that are
// neighbours in the table: they share its loads of ln rho and Psi_a, and its stores
// become runs of F values (a table row is contiguous in the frequency).  Bound by the
// FP64 exp (about 25 multiply-adds each); the form this replaces staged 8 nodes of a
// 64-node coherence tile in LDS between two barriers and stored single doubles a table
// row apart: 1000 nodes, 30 modes, 2 components, 513 frequencies 3.0 -> 1.8 ms; 200
// nodes, 10 modes, some 4600 frequencies of the Mesher's point layout 1.7 (with the
// transpose it no longer needs) -> 0.85 ms.  The f64 MFMAs and the FP64 vector
// instructions add up here: 128 + 80 of the 255 cycles per 64 coherences and 32 modes.
// Waves: column tile of 16 nodes x group of F frequencies x component x chunk of 64
// modes; F from project_group() so that small tables still fill the chip.
// v_mfma_f64_16x16x4f64: A lane l holds (row l%16, k l/16), B (k l/16, col l%16),
// D register t of lane l holds (row l/16 + 4t, col l%16).
// VLAY: the point layout U[(q*K + k)*ldU + y] of the Mesher (ldU modes, zero from nm
// on, K rows) instead of U[k*ldU + y*row_stride + q]; its padding rows k are cleared.
// ---------------------------------------------------------------------------
// exp(x) of the projection's inner loop by Cody-Waite reduction: x = n ln 2 + r,
// |r| <= ln 2 / 2 (the high part of ln 2 cut to 33 bits so that n times it is exact), a
// degree-11 polynomial on r whose coefficients interpolate (e^r - 1 - r) / r^2 at the
// Chebyshev nodes (relative error 2e-17), and a power of two.  0.85 ulp at most (5000
// arguments from -690 to 0 against 60 digits), within the 1 ulp of the library's exp;
// here the coefficients stay in scalar registers, where the library call reloads eighteen
// vector registers with them for every value.  Results below the subnormals are 0, those
// above the largest double infinite.
struct ExpC {
   double magic, inv, hi, lo, c3, c4, c5, c6, c7, c8, c9, c10, c11;
};

__device__ __forceinline__ ExpC exp_consts()
{
   ExpC e = {0x1.8p52, 0x1.71547652b82fep+0, 0x1.62e42fef00000p-1, 0x1.473de6af278edp-34,
             0x1.5555555555555p-3, 0x1.5555555553d63p-5, 0x1.11111111109b3p-7,
             0x1.6c16c1788bd90p-10, 0x1.a01a01a7c41d5p-13, 0x1.a019b90d2ae7ap-16,
             0x1.71de0dae63bb3p-19, 0x1.289185613a3d6p-22, 0x1.af38a9b0ec855p-26};
   // opaque to the compiler, so that they are not rematerialised in the loop
   asm volatile("" : "+v"(e.magic), "+s"(e.inv), "+s"(e.hi), "+s"(e.lo), "+s"(e.c3), "+s"(e.c4),
                     "+s"(e.c5), "+s"(e.c6), "+s"(e.c7), "+s"(e.c8), "+s"(e.c9), "+s"(e.c10));
   asm volatile("" : "+v"(e.c11));
   return e;
}

// NaN is left to the caller: the clamps drop it
__device__ __forceinline__ double exp_fast(double x, const ExpC &e)
{
   x = __builtin_fmin(__builtin_fmax(x, -800.0), 720.0);
   const double t = __builtin_fma(x, e.inv, e.magic);
   const int n = (int)(uint32_t)__double_as_longlong(t);   // rounded to nearest
   const double nf = t - e.magic;
   double r = __builtin_fma(-nf, e.hi, x);
   r = __builtin_fma(-nf, e.lo, r);
   double p = __builtin_fma(e.c11, r, e.c10);
   p = __builtin_fma(p, r, e.c9);
   p = __builtin_fma(p, r, e.c8);
   p = __builtin_fma(p, r, e.c7);
   p = __builtin_fma(p, r, e.c6);
   p = __builtin_fma(p, r, e.c5);
   p = __builtin_fma(p, r, e.c4);
   p = __builtin_fma(p, r, e.c3);
   p = __builtin_fma(p, r, 0.5);
   p = __builtin_fma(p, r, 1.0);
   p = __builtin_fma(p, r, 1.0);
   return __builtin_amdgcn_ldexp(p, n);
}

// Two waves per SIMD at least: 256 registers, so that the accumulators stay in ordinary
// ones (with 512 the compiler moves them to and from the accumulation registers).
struct ProjArgs {
   const double *pak;        // [nm][K]  Psi_a per K index
   const double *lnr;        // [tc][nnl][nnl]  ln rho_ji (row j, col i)
   const double *sq;         // [tc][nfl][nnl]  sqrt(S)
   const double *fabs_list;
   int nfl, nnl, nm, nnlp, K;
   int row_stride;           // rows per mode in U (nhp)
   int ntc, ncoltile;        // components, column tiles
   double *U;
   long ldU;
   long nqg;                 // frequency groups
};

// One wave: column tile and frequency group `wid` of component tc, modes from y0 on.
// Consecutive waves take consecutive frequency groups of one column tile: they share
// its ln rho lines.
template <int MT, int F, bool VLAY>
__device__ __forceinline__ void project_wave(const ProjArgs &P, long wid, int tc, int y0)
{
   const int lane = threadIdx.x & 63;
   const int nfl = P.nfl, nnl = P.nnl, nm = P.nm, nnlp = P.nnlp, K = P.K, ntc = P.ntc;
   const double *__restrict__ pak = P.pak;
   const double *__restrict__ lnr = P.lnr;
   const double *__restrict__ sq = P.sq;
   const double *__restrict__ fabs_list = P.fabs_list;
   double *__restrict__ U = P.U;
   const long ldU = P.ldU;
   const int row_stride = P.row_stride;
   const int i0 = (int)(wid / P.nqg) * 16;
   const int q0 = (int)(wid % P.nqg) * F;
   const int lr = lane & 15, lk = lane >> 4;
   const int i = i0 + lr;
   const int ic = min(i, nnl - 1);
   const double *lnt = lnr + (size_t)tc * nnl * nnl + ic;
   const double *pat[MT];              // rows y >= nm repeat the last mode: not stored
#pragma unroll
   for (int r = 0; r < MT; ++r)
      pat[r] = pak + (size_t)min(y0 + 16 * r + lr, nm - 1) * K + tc * nnlp;
   const double *sqt = sq + (size_t)tc * nfl * nnl;
   double af[F];
   const double *sqq[F];
#pragma unroll
   for (int f = 0; f < F; ++f) {
      const int q = min(q0 + f, nfl - 1);
      af[f] = fabs_list[q];
      sqq[f] = sqt + (size_t)q * nnl;
   }
   d4 acc[F][MT];
#pragma unroll
   for (int f = 0; f < F; ++f)
#pragma unroll
      for (int r = 0; r < MT; ++r) acc[f][r] = (d4){0.0, 0.0, 0.0, 0.0};
   const ExpC ec = exp_consts();
   unsigned long long nan = 0;                // lanes that met a NaN of ln rho
   // one MFMA step: ln rho l of the lane's (j, i), Psi_a a of its (y, j), s_j
   auto step = [&](double l, const double (&a)[MT], const double (&sj)[F]) {
      // |f| = 0 gives 1 for any rho: the infinity of rho == 0 becomes a finite number, the
      // NaN of rho < 0 is noted and joins its column at the end where |f| is another
      nan |= __ballot(l != l);
      const double lc = __builtin_fmin(__builtin_fmax(l, -0x1.fffffffffffffp1023), 0x1.fffffffffffffp1023);
#pragma unroll
      for (int f = 0; f < F; ++f) {
         const double e = exp_fast(af[f] * lc, ec) * sj[f];
#pragma unroll
         for (int r = 0; r < MT; ++r)
            acc[f][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], e, acc[f][r], 0, 0, 0);
      }
   };
   // pairs of steps: lane group lk takes the nodes j0 + 2 lk and j0 + 2 lk + 1, so that
   // Psi_a and s_j come as 16-byte loads; the next pair's operands are loaded while
   // this one's are used
   struct pair { double v[2]; };
   auto ld2 = [](const double *p) {
      pair v;
      __builtin_memcpy(&v, p, sizeof(v));
      return v;
   };
   double l0, l1;
   pair a2[MT], s2[F];
   auto load = [&](int j0) {
      const int j = j0 + 2 * lk;
      l0 = lnt[(size_t)j * nnl];
      l1 = lnt[(size_t)(j + 1) * nnl];
#pragma unroll
      for (int r = 0; r < MT; ++r) a2[r] = ld2(pat[r] + j);
#pragma unroll
      for (int f = 0; f < F; ++f) s2[f] = ld2(sqq[f] + j);
   };
   const int n8 = nnl & ~7;
   if (n8 > 0) load(0);
   for (int j0 = 0; j0 < n8; j0 += 8) {
      const double c0 = l0, c1 = l1;
      double a0[MT], a1[MT], x0[F], x1[F];
#pragma unroll
      for (int r = 0; r < MT; ++r) {
         a0[r] = a2[r].v[0];
         a1[r] = a2[r].v[1];
      }
#pragma unroll
      for (int f = 0; f < F; ++f) {
         x0[f] = s2[f].v[0];
         x1[f] = s2[f].v[1];
      }
      if (j0 + 8 < n8) load(j0 + 8);
      step(c0, a0, x0);
      step(c1, a1, x1);
   }
   for (int j0 = n8; j0 < nnl; j0 += 4) {
      const int j = j0 + lk, jc = min(j, nnl - 1);
      double a[MT], x[F];
#pragma unroll
      for (int r = 0; r < MT; ++r) a[r] = j < nnl ? pat[r][jc] : 0.0;
#pragma unroll
      for (int f = 0; f < F; ++f) x[f] = j < nnl ? sqq[f][jc] : 0.0;
      step(lnt[(size_t)jc * nnl], a, x);
   }
   nan |= nan >> 32;
   nan |= nan >> 16;
   const double bad = (nan >> lr) & 1 ? __builtin_nan("") : 0.0;      // the lane's column
   // s_i; a frequency that is not a number, or infinite (rho_ii = 1), gives NaN as well
   auto row = [&](int f) { return sqq[f][i] + (af[f] - af[f]) + (af[f] == 0.0 ? 0.0 : bad); };
   const int k = tc * nnlp + i;
   const bool ok = i < nnl;
   if constexpr (VLAY) {
      if (!ok && !(tc == ntc - 1 && k < K)) return;
#pragma unroll
      for (int f = 0; f < F; ++f) {
         if (q0 + f >= nfl) break;
         const double si = ok ? row(f) : 0.0;
         double *d = U + ((size_t)(q0 + f) * K + k) * ldU + y0 + lk;
#pragma unroll
         for (int r = 0; r < MT; ++r)
#pragma unroll
            for (int t = 0; t < 4; ++t)
               d[16 * r + 4 * t] = ok && y0 + lk + 16 * r + 4 * t < nm ? acc[f][r][t] * si : 0.0;
      }
   } else {
      if (!ok) return;
      double si[F];
#pragma unroll
      for (int f = 0; f < F; ++f) si[f] = row(f);
#pragma unroll
      for (int r = 0; r < MT; ++r)
#pragma unroll
         for (int t = 0; t < 4; ++t) {
            const int y = y0 + 16 * r + lk + 4 * t;
            if (y >= nm) continue;
            double *d = U + (size_t)k * ldU + (size_t)y * row_stride + q0;
#pragma unroll
            for (int f = 0; f < F; ++f)
               if (q0 + f < nfl) d[f] = acc[f][r][t] * si[f];
         }
   }
}

template <int MT, int F, bool VLAY>
__global__ __launch_bounds__(256, 2) void k_project(ProjArgs P)
{
   const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const long wid = (long)blockIdx.x * 4 + w;
   if (wid >= P.nqg * P.ncoltile) return;
   project_wave<MT, F, VLAY>(P, wid, blockIdx.y, blockIdx.z * (MT * 16));
}

// ---------------------------------------------------------------------------
// FRF helpers and quadrature weights (FP64)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double2 hget(const double2 *__restrict__ H, int nft, int m, int F)
{
   double2 h = H[(size_t)m * nft + abs(F)];
   if (F < 0) h.y = -h.y;
   return h;
}

// Re[a b conj(c)]  (functionsImpl.F90:1706-1710 / bsacl.cl:892-897)
__device__ __forceinline__ double re3(double2 a, double2 b, double2 c)
{
   const double pr = a.x * b.x - a.y * b.y;
   const double pi = a.x * b.y + a.y * b.x;
   return pr * c.x + pi * c.y;
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
   for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
   return v;
}

// ---------------------------------------------------------------------------
// G contraction on FP64 MFMA + plane epilogue
// grid: (n_tile_pairs * nm) workgroups, 256 threads (4 waves, 2x2 of 32x32)
// ---------------------------------------------------------------------------
struct GsymArgs {
   const double *U;       // [K][ldU]
   long ldU;
   const double *pb;      // [nm][K]  Psi_b per K index
   int K;                 // multiple of KC
   int nm, nhp, nh;       // modes, rows per mode, half-grid points of the plane
   int nu;                // table rows holding A (nh, or 2nh-1 when S(f1+f2)
                          // is evaluated beyond the plane)
   const double2 *H;      // [nm][nft]
   int nft;               // >= 2*nu - 1
   double d2;             // (2 pi df)^2 or df^2
   int rule;
   int epi_plain;         // 1: every 16x16 block through the generic epilogue
   double *m3f, *m3r;     // [nm^3] accumulated (atomic)
   double *slots;         // NULL, or fixed-order mode: the flushes of a wave write
                          // their m3 contributions one after the other to slots +
                          // slot0[item*4 + wave] instead of the atomics
   const long *slot0;
   int copies;            // of m3f and m3r, 2 nm^3 doubles apart (gsym_f64_wave)
};

// Quadrature weight / d^2 from edge flags of |F1| (p) and |F2| (q) on the
// half grid [0, n]: outside the plane 0; corner c_corner; edge c_edge; else 1.
struct QRule {
   double c_edge, c_corner;
};

__device__ __forceinline__ QRule qrule(int rule)
{
   if (rule == 0) return QRule{0.5, 1.0 - 1.5};   // intgSpectraVect_ (BsaClassicImpl.F90:604-631)
   if (rule == 1) return QRule{1.0, 1.0};         // Riemann (BsaClassicImpl.F90:331,341)
   return QRule{0.5, 0.25};                       // tensor trapezoid (_shared_poly2d.fi:827-832)
}

__device__ __forceinline__ double qw(bool ep, bool op, bool eq, bool oq, const QRule &r)
{
   return (op || oq) ? 0.0 : ((ep && eq) ? r.c_corner : ((ep || eq) ? r.c_edge : 1.0));
}

// Plane epilogue.  A G value G[x](y,u; z,v) enters the moments at up to twelve
// (m,n,p,f1,f2) places; per lane they make nine sums:
//   s0 force (x,y,z)=(x,z,y)  s1 resp (x,y,z)  s2 force (y,x,z)=(y,z,x)
//   s3 resp (y,x,z)  s4 resp (y,z,x)  s5 resp (x,z,y)
//   s6 force (z,x,y)=(z,y,x)  s7 resp (z,x,y)  s8 resp (z,y,x)
// (s5..s8 and the second entry of s0 only off the tile diagonal).  Re[a b conj c] does
// not change when all three factors are conjugated, so of the eight FRF products that
// weight them four differ:
//   F1s = Re[H_x(u) H_y(v) conj H_z(u+v)]         F1o = Re[H_x(u) conj H_y(v) conj H_z(u-v)]
//   F2s = Re[H_y(u-v) H_x(v) conj H_z(u)]         F2o = Re[H_y(u+v) conj H_x(v) conj H_z(u)]
// and with the sign multiplicities ms, mo of (+-u, +-v) and the weights W of the places
//   s0 += g Wa (ms + mo)            s1 += g Wa (ms F1s + mo F1o)
//   s2 += g (ms Wb + mo Wd)         s3 += g (ms Wb F2s + mo Wd F2o)
//   s4 += g (ms Wb F1o + mo Wd F1s) s5 += g Wa (ms F2o + mo F2s)
//   s6 += g (ms We + mo Wf)         s7 += g (ms We F1o + mo Wf F1s)
//   s8 += g (ms We F2s + mo Wf F2o)
// Wa = w(u,v), Wb = w(|u-v|,v), Wd = w(u+v,v), We = w(|u-v|,u), Wf = w(u+v,u).  H(0) is
// real, so at u = 0 or v = 0 the s and the o terms are equal and the multiplicities (2, 0)
// and (1, 0) act as (1, 1) and (1/2, 1/2): a factor 1/2 on g per zero.  All sums are
// kept in units of 4 g (interior multiplicity 2, B = 2 G).
//
// Each 16x16 block is handled by its class, uniform per wave (epi_class):
//   1  u, v < n and u + v < n: every weight 1
//   2  u, v < n and u + v > n: Wd = Wf = 0
//   3  u + v on both sides of n, or with the edge u = n or v = n
//   4  holds (n,n), (n,0) or (0,n), where two edges meet, or lies beyond the plane
//      (SUM_EXACT): every weight by the rule, qw()
// In classes 1 to 3 one factor each of u and of v goes onto g: 1/2 at 0, the edge weight
// c at n, 0 for rows (columns) of another mode.  That is Wa; Wb and Wd have no factor of
// u and We and Wf none of v, so the row u = n gets the missing (1 - c) of s2..s4 by itself
// (w(u+v) is 0 there) and the column v = n its s6..s8 divided by c.  The sums over a lane's
// rows are taken before the factors of its column: sum h H_x(u) conj H_z(u+v) first,
// H_y(v) once per column block (21 FP64 instructions per value of class 1 instead of 33).
// The FRF values at u+v and u-v are read from a window in LDS, those of the rows
// broadcast from registers (a lane of each 16-lane row holds one row's).  With one
// window load per value and two passes (interior, then edges point by point) the BF16x3
// kernel took 842 us at 333 nodes, 17 modes, 193 frequencies and 208 us at 40, 20, 65,
// now 741 and 150, of which 388 and 21 are the contraction.

// FRF values of a wave's (y, z) pair in LDS, indexed by the offset from its origin
// (ub, vb) within the modes (either may be negative; entries of points outside the modes
// are never used):
//   [0, 128)   H_z(u+v)      at u+v - (ub+vb)
//   [128, 256) H_y(u+v)      at u+v - (ub+vb)
//   [256, 384) H_y(u-v)      at u-v - (ub-vb-16BC+1), conjugated for u < v
//   [384, 512) H_z(u-v)      likewise
//   [512, 576) H_x(u), [576, 640) H_z(u)   at u - ub
//   [640, 704) H_x(v), [704, 768) H_y(v)   at v - vb
template <int BR, int BC>
__device__ __forceinline__ void epi_window(const GsymArgs &a, int x, int y, int z, int ub, int vb,
                                           int lane, double2 *win)
{
   constexpr int NS = 16 * (BR + BC);
   static_assert(NS <= 128 && 16 * BR <= 64 && 16 * BC <= 64, "FRF windows of 128 and 64 entries");
   const double2 *Hx = a.H + (size_t)x * a.nft;
   const double2 *Hy = a.H + (size_t)y * a.nft;
   const double2 *Hz = a.H + (size_t)z * a.nft;
   const int wsb = ub + vb, wdb = ub - vb - (16 * BC - 1);
   // the previous pair's reads before these writes
   __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
   __builtin_amdgcn_wave_barrier();
   for (int e = lane; e < NS; e += 64) {
      const int sp = min(abs(wsb + e), a.nft - 1);
      const int dm = wdb + e;
      const int ad = min(abs(dm), a.nft - 1);
      double2 hym = Hy[ad], hzm = Hz[ad];
      if (dm < 0) {
         hym.y = -hym.y;
         hzm.y = -hzm.y;
      }
      win[e] = Hz[sp];
      win[128 + e] = Hy[sp];
      win[256 + e] = hym;
      win[384 + e] = hzm;
   }
   if (lane < 16 * BR) {
      const int u = min(max(ub + lane, 0), a.nft - 1);
      win[512 + lane] = Hx[u];
      win[576 + lane] = Hz[u];
   }
   if (lane < 16 * BC) {
      const int v = min(max(vb + lane, 0), a.nft - 1);
      win[640 + lane] = Hx[v];
      win[704 + lane] = Hy[v];
   }
   // the wave's own LDS writes before its reads (other waves never touch it)
   __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
   __builtin_amdgcn_wave_barrier();
   __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Class of the 16x16 block at (u0, v0) within the modes, see above.
__device__ __forceinline__ int epi_class(const GsymArgs &a, int u0, int v0)
{
   const int n = a.nh - 1;
   const bool ue = u0 + 15 >= n, ve = v0 + 15 >= n;
   if (a.epi_plain || (a.nu != a.nh && (ue || ve))) return 4;
   if ((ue && (ve || v0 <= 0)) || (ve && u0 <= 0)) return 4;
   if (ue || ve) return 3;
   if (u0 + v0 + 30 <= n - 1) return 1;
   return u0 + v0 >= n + 1 ? 2 : 3;
}

// broadcast within each 16-lane row from its lane C
template <int C>
__device__ __forceinline__ double row_bcast(double v)
{
   const long b = __double_as_longlong(v);
   const int lo = __builtin_amdgcn_mov_dpp((int)b, 0x150 + C, 0xf, 0xf, true);
   const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x150 + C, 0xf, 0xf, true);
   return __longlong_as_double(((long)hi << 32) | (unsigned)lo);
}

// Sums of a column block (classes 1 to 3) before the column's factors; w: the part of h
// that w(u+v) leaves to the u + v terms (class 1: all), r: the rest (class 2: all).
struct EpiZ {
   double z1wr, z1wi, z1rr, z1ri;      // sum h H_x(u) conj H_z(u+v)
   double z2r, z2i;                    // sum h H_x(u) conj H_z(u-v)
   double z3r, z3i;                    // sum h H_y(u-v) conj H_z(u)
   double z4wr, z4wi, z4rr, z4ri;      // sum h H_y(u+v) conj H_z(u)
   double hw, hr;                      // sum h
};

// Value T of row block I, column block at window offsets ps (u+v) and pd (u-v), class 1,
// 2 or 3 (w: w(u+v)).  rx, rz: the lane's row of H_x(u), H_z(u) (lane c = 4 i + t of each
// 16-lane row holds row register t of block i).  ST: u step of the row registers.
template <int CLS, int I, int T, int ST>
__device__ __forceinline__ void epi_value(const double2 *ps, const double2 *pd, double h, double w,
                                          const double2 &rx, const double2 &rz, EpiZ &Z)
{
   const double2 hzs = ps[ST * T], hys = ps[128 + ST * T];
   const double2 hyd = pd[ST * T], hzd = pd[128 + ST * T];
   const double xr = h * row_bcast<4 * I + T>(rx.x), xi = h * row_bcast<4 * I + T>(rx.y);
   const double zr = h * row_bcast<4 * I + T>(rz.x), zi = h * row_bcast<4 * I + T>(rz.y);
   if constexpr (CLS == 1) {
      Z.z1wr = fma(xi, hzs.y, fma(xr, hzs.x, Z.z1wr));
      Z.z1wi = fma(-xr, hzs.y, fma(xi, hzs.x, Z.z1wi));
      Z.z4wr = fma(zi, hys.y, fma(zr, hys.x, Z.z4wr));
      Z.z4wi = fma(-zi, hys.x, fma(zr, hys.y, Z.z4wi));
      Z.hw += h;
   } else if constexpr (CLS == 2) {
      Z.z1rr = fma(xi, hzs.y, fma(xr, hzs.x, Z.z1rr));
      Z.z1ri = fma(-xr, hzs.y, fma(xi, hzs.x, Z.z1ri));
      Z.z4rr = fma(zi, hys.y, fma(zr, hys.x, Z.z4rr));
      Z.z4ri = fma(-zi, hys.x, fma(zr, hys.y, Z.z4ri));
      Z.hr += h;
   } else {
      const double r = 1.0 - w;
      const double p1r = fma(xi, hzs.y, xr * hzs.x), p1i = fma(-xr, hzs.y, xi * hzs.x);
      const double p4r = fma(zi, hys.y, zr * hys.x), p4i = fma(-zi, hys.x, zr * hys.y);
      Z.z1wr = fma(w, p1r, Z.z1wr);
      Z.z1wi = fma(w, p1i, Z.z1wi);
      Z.z4wr = fma(w, p4r, Z.z4wr);
      Z.z4wi = fma(w, p4i, Z.z4wi);
      Z.z1rr = fma(r, p1r, Z.z1rr);
      Z.z1ri = fma(r, p1i, Z.z1ri);
      Z.z4rr = fma(r, p4r, Z.z4rr);
      Z.z4ri = fma(r, p4i, Z.z4ri);
      Z.hw = fma(w, h, Z.hw);
      Z.hr = fma(r, h, Z.hr);
   }
   Z.z2r = fma(xi, hzd.y, fma(xr, hzd.x, Z.z2r));
   Z.z2i = fma(-xr, hzd.y, fma(xi, hzd.x, Z.z2i));
   Z.z3r = fma(zi, hyd.y, fma(zr, hyd.x, Z.z3r));
   Z.z3i = fma(-zi, hyd.x, fma(zr, hyd.y, Z.z3i));
}

// Row block I of a column block, class cls 1 to 3; win, ub, wdb: the wave's window.
template <int I, int ST>
__device__ __forceinline__ void epi_rows(const GsymArgs &a, int cls, int ur0, int vq0, int lane,
                                         const double (&g)[4], const double2 *ps, const double2 *pd,
                                         const double2 &rx, const double2 &rz, EpiZ &Z, double (&s)[9],
                                         const double2 *win, int ub, int vb)
{
   const int n = a.nh - 1;
   const double ce = qrule(a.rule).c_edge;
   double h[4] = {g[0], g[1], g[2], g[3]};
   const int v = vq0 + (lane & 15), ul = ur0 + (ST == 4 ? lane >> 4 : 4 * (lane >> 4));
   if (ur0 <= 0 || vq0 <= 0 || ur0 + 15 >= n || vq0 + 15 >= n) {       // uniform
      const bool vok = v >= 0 && v <= n;
      const double fv = v == 0 ? 0.5 : (v == n ? ce : 1.0);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
         const int u = ul + ST * t;
         const double fu = u == 0 ? 0.5 : (u == n ? ce : 1.0);
         h[t] = vok && u >= 0 && u <= n ? h[t] * (fu * fv) : 0.0;
      }
      if (ur0 + 15 >= n && ce != 1.0) {
         // the row u = n: one register of one lane group
         const int rn = n - ur0, tn = ST == 4 ? rn >> 2 : rn & 3, kn = ST == 4 ? rn & 3 : rn >> 2;
         const double gn = tn == 0 ? g[0] : (tn == 1 ? g[1] : (tn == 2 ? g[2] : g[3]));
         const double c = vok && lane >> 4 == kn ? gn * (fv * (1.0 - ce)) : 0.0;
         const double2 hxn = win[512 + n - ub], hzn = win[576 + n - ub];
         const double2 hxv = win[640 + v - vb], hyv = win[704 + v - vb];
         const double2 hyd = pd[n - ul], hzd = pd[128 + n - ul];
         s[2] += c;
         s[3] += c * re3(hyd, hxv, hzn);
         s[4] += c * re3(hxn, make_double2(hyv.x, -hyv.y), hzd);
      }
   }
   if (cls == 1) {
      epi_value<1, I, 0, ST>(ps, pd, h[0], 1.0, rx, rz, Z);
      epi_value<1, I, 1, ST>(ps, pd, h[1], 1.0, rx, rz, Z);
      epi_value<1, I, 2, ST>(ps, pd, h[2], 1.0, rx, rz, Z);
      epi_value<1, I, 3, ST>(ps, pd, h[3], 1.0, rx, rz, Z);
   } else if (cls == 2) {
      epi_value<2, I, 0, ST>(ps, pd, h[0], 0.0, rx, rz, Z);
      epi_value<2, I, 1, ST>(ps, pd, h[1], 0.0, rx, rz, Z);
      epi_value<2, I, 2, ST>(ps, pd, h[2], 0.0, rx, rz, Z);
      epi_value<2, I, 3, ST>(ps, pd, h[3], 0.0, rx, rz, Z);
   } else {
      const int s0 = ul + v;
      double w[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) w[t] = s0 + ST * t < n ? 1.0 : (s0 + ST * t == n ? ce : 0.0);
      epi_value<3, I, 0, ST>(ps, pd, h[0], w[0], rx, rz, Z);
      epi_value<3, I, 1, ST>(ps, pd, h[1], w[1], rx, rz, Z);
      epi_value<3, I, 2, ST>(ps, pd, h[2], w[2], rx, rz, Z);
      epi_value<3, I, 3, ST>(ps, pd, h[3], w[3], rx, rz, Z);
   }
}

// Block of class 4: every weight of every point by the rule, FRF values from the window.
template <int ST>
__device__ __forceinline__ void epi_rule(const GsymArgs &a, int ur0, int vq0, int lane,
                                         const double (&gval)[4], double (&s)[9], const double2 *win,
                                         int ub, int vb, int wdb)
{
   const int n = a.nh - 1;
   const QRule qr = qrule(a.rule);
   const int vr = vq0 + (lane & 15);
   const bool vok = vr >= 0 && vr < a.nu;
   const int v = vok ? vr : max(vb, 0);                      // a column of the window
   const double2 hxv = win[640 + v - vb], hyv = win[704 + v - vb];
   const double2 cyv = make_double2(hyv.x, -hyv.y);
   const double2 cxv = make_double2(hxv.x, -hxv.y);
   const bool ev = (v == n), ov = (v > n);
#pragma unroll
   for (int t = 0; t < 4; ++t) {
      // rows past the mode's last row (the next mode's rows, or padding) add
      // nothing: stop once the lowest row of this register is one of them (uniform)
      if (ur0 + ST * t >= a.nu) break;
      const int ur = ur0 + (ST == 4 ? lane >> 4 : 4 * (lane >> 4)) + ST * t;
      const bool ok = vok && ur >= 0 && ur < a.nu;
      const int u = ok ? ur : max(ub, 0);
      const int sp = u + v, dm = u - v, ad = abs(dm);
      const double2 hxu = win[512 + u - ub], hzu = win[576 + u - ub];
      const double2 hzp = win[sp - ub - vb], hyp = win[128 + sp - ub - vb];
      const double2 hym = win[256 + dm - wdb], hzm = win[384 + dm - wdb];
      const double F1s = re3(hxu, hyv, hzp);
      const double F1o = re3(hxu, cyv, hzm);
      const double F2s = re3(hym, hxv, hzu);
      const double F2o = re3(hyp, cxv, hzu);
      const double g = ok ? 0.5 * gval[t] : 0.0;             // sums in units of 4 g
      const double ms = (u == 0 && v == 0) ? 1.0 : 2.0;
      const double mo = (u > 0 && v > 0) ? 2.0 : 0.0;
      const bool eu = (u == n), ou = (u > n), es = (sp == n), os = (sp > n);
      const bool ed = (ad == n), od = (ad > n);
      const double ga = g * qw(eu, ou, ev, ov, qr);
      const double gas = ms * ga, gao = mo * ga;
      const double gbs = ms * g * qw(ed, od, ev, ov, qr), gdo = mo * g * qw(es, os, ev, ov, qr);
      const double ges = ms * g * qw(ed, od, eu, ou, qr), gfo = mo * g * qw(es, os, eu, ou, qr);
      s[0] += gas + gao;
      s[1] += gas * F1s + gao * F1o;
      s[2] += gbs + gdo;
      s[3] += gbs * F2s + gdo * F2o;
      s[4] += gbs * F1o + gdo * F1s;
      s[5] += gas * F2o + gao * F2s;
      s[6] += ges + gfo;
      s[7] += ges * F1o + gfo * F1s;
      s[8] += ges * F2s + gfo * F2o;
   }
}

// One exchange of epi_flush: of the N values a lane holds it keeps the lower half (or,
// with its bit `m` set, the upper one), summed with the partner's.
template <int N, int M>
__device__ __forceinline__ void epi_halve(double (&v)[9], int lane)
{
   constexpr int H = (N + 1) / 2;
   const bool up = (lane & M) != 0;
#pragma unroll
   for (int k = 0; k < H; ++k) {
      const double hi = H + k < N ? v[H + k] : 0.0;
      const double send = up ? v[k] : hi, keep = up ? hi : v[k];
      v[k] = keep + __shfl_xor(send, M, 64);
   }
}

// Reduce the nine sums over the wave and add them (times 4 d^2) to the m3 entries, or
// in the fixed-order mode store them from the wave's slot on (det_slot_lists of
// bsahip_api.hip builds the matching lists).  The exchanges halve the values a lane
// holds as they halve the lanes that share one, 13 instead of 54, and leave sum k on
// the lanes of one 4-lane group, so that the contributions (slot t: permutation t / 2 of
// xyz, yxz, yzx, xzy, zxy, zyx; even force, odd response) leave as one atomic.
// F64 (the FP64 kernels; the others' tiles of 64 x 64 make a quarter of the flushes, and the
// longer code costs them 0.8 %): contributions that meet in one entry leave as one.  With
// y == z, off the tile diagonal, the second six are those of the first again, with x == y ==
// z two of them are left.  An atomic to one address takes some 40 ns however many waves
// wait, and the entries of one mode are the ones that most waves share: 300 nodes, 1 mode,
// 193 frequencies 42 -> 27 us (with one copy of the moments).
// ONE: a structure of one mode.
__host__ __device__ inline int epi_count(bool f64, int x, int y, int z, bool diag)
{
   if (f64 && y == z) return x == y ? 2 : 6;
   return diag ? 6 : 12;
}

__device__ __forceinline__ void epi_put(const GsymArgs &a, int t, size_t e, double q, unsigned wave, int f)
{
   if (a.slots) {
      a.slots[a.slot0[wave] + f + t] = q;
      return;
   }
   atomicAdd((t & 1 ? a.m3r : a.m3f) + e, q);
}

template <bool ONE, bool F64>
__device__ __forceinline__ void epi_flush(const GsymArgs &a, int x, int y, int z, bool diag,
                                          int lane, double (&s)[9], unsigned wave, int f)
{
   const double d2 = 4.0 * a.d2;
   if (F64 && y == z && !diag) {
      s[0] *= 2.0;
      s[1] += s[5];
      s[2] += s[6];
      s[3] += s[7];
      s[4] += s[8];
   }
   const int n = ONE ? 2 : epi_count(F64, x, y, z, diag);
   if (n == 2) {
      s[0] += 2.0 * s[2];
      s[1] = (s[1] + s[3]) + s[4];
      epi_halve<2, 32>(s, lane);
      double q = s[0];
#pragma unroll
      for (int o = 16; o >= 1; o >>= 1) q += __shfl_xor(q, o, 64);
      if ((lane & 31) == 0) epi_put(a, lane >> 5, (size_t)x * (1 + a.nm + (size_t)a.nm * a.nm), q * d2, wave, f);
   } else {
      epi_halve<9, 32>(s, lane);
      epi_halve<5, 16>(s, lane);
      epi_halve<3, 8>(s, lane);
      epi_halve<2, 4>(s, lane);
      double q = s[0];
      q += __shfl_xor(q, 2, 64);
      q += __shfl_xor(q, 1, 64);
      q *= d2;
      // value index of the lane's group; groups of padding (a lower half is the larger)
      const int b5 = lane >> 5, b4 = (lane >> 4) & 1, b3 = (lane >> 3) & 1, b2 = (lane >> 2) & 1;
      const int k = 5 * b5 + 3 * b4 + 2 * b3 + b2;
      const bool pad = (b3 && (b4 || b2)) || (b5 && b4 && b2);
      // slots of value k: {0,6} 1 {2,4} 3 5 7 {8,10} 9 11
      const int second = lane & 3;
      int t = -1;
      if (!pad && second == 0) t = k == 0 ? 0 : (k <= 3 ? k : (k == 4 ? 5 : (k == 5 ? 7 : (k == 6 ? 8 : (k == 7 ? 9 : 11)))));
      if (!pad && second == 1) t = k == 0 ? 6 : (k == 2 ? 4 : (k == 6 ? 10 : -1));
      if (t >= 0 && t < n) {
         const int p = t >> 1;
         const int i0 = p == 0 || p == 3 ? x : (p == 1 || p == 2 ? y : z);
         const int i1 = p == 0 || p == 5 ? y : (p == 1 || p == 4 ? x : z);
         const int i2 = p == 0 || p == 1 ? z : (p == 2 || p == 5 ? x : y);
         epi_put(a, t, i0 + (size_t)a.nm * (i1 + (size_t)a.nm * i2), q, wave, f);
      }
   }
#pragma unroll
   for (int t = 0; t < 9; ++t) s[t] = 0.0;
}

// Epilogue of a wave's BR x BC blocks of 16x16 (rows rw0.., cols cw0..), one accumulation
// and reduction per (y, z) mode pair they meet: the rows of consecutive modes are packed,
// so a block can hold the end of one mode and the start of the next and is then visited
// for each, the other mode's rows (columns) masked.  win: 768 double2 of LDS owned by this
// wave.  getv<i>(j, g): values of block (i, j).
template <int BR, int BC, bool IL, bool ONE, class GetVal>
__device__ __forceinline__ void epi_wave(const GsymArgs &a, int x, bool diag, int rw0, int cw0,
                                         int lane, unsigned wave, GetVal getv, double2 *win)
{
   constexpr int ST = IL ? 4 : 1;
   const int nm = a.nm;
   int f = 0;                                         // slots of this wave so far
   const int y0 = rw0 / a.nhp, y1 = min((rw0 + 16 * BR - 1) / a.nhp, nm - 1);
   const int z0 = cw0 / a.nhp, z1 = min((cw0 + 16 * BC - 1) / a.nhp, nm - 1);
   const int lr = lane & 15, lk = lane >> 4;
#pragma unroll 1
   for (int y = y0; y <= y1; ++y)
#pragma unroll 1
      for (int z = z0; z <= z1; ++z) {
         const int ub = rw0 - y * a.nhp, vb = cw0 - z * a.nhp;
         const int wdb = ub - vb - (16 * BC - 1);
         epi_window<BR, BC>(a, x, y, z, ub, vb, lane, win);
         double s[9];
#pragma unroll
         for (int t = 0; t < 9; ++t) s[t] = 0.0;
         // row values of this lane: row register lr % 4 of block lr / 4 (of its lk group)
         const int rr = min(16 * (lr >> 2) + (IL ? lk + 4 * (lr & 3) : 4 * lk + (lr & 3)), 16 * BR - 1);
         const double2 rx = win[512 + rr], rz = win[576 + rr];
         const int us = IL ? lk : 4 * lk;                  // u of row register 0 in its block
         unsigned rule = 0;                                // blocks of class 4
#pragma unroll 1
         for (int j = 0; j < BC; ++j) {
            const int v0 = vb + 16 * j;
            if (v0 + 15 < 0 || v0 >= a.nu) continue;       // no column of this mode
            EpiZ Z = {};
            const double2 *ps = win + us + lr + 16 * j;
            const double2 *pd = win + 256 + us - lr - 16 * j + 16 * BC - 1;
            double g[4];
            auto rows = [&](auto ic) {
               constexpr int I = decltype(ic)::value;
               if constexpr (I < BR) {
                  const int u0 = ub + 16 * I;
                  if (u0 + 15 < 0 || u0 >= a.nu) return;   // no row of this mode
                  const int cls = epi_class(a, u0, v0);    // uniform per block
                  if (cls == 4) {
                     rule |= 1u << (I * BC + j);
                     return;
                  }
                  getv(ic, j, g);
                  epi_rows<I, ST>(a, cls, u0, v0, lane, g, ps + 16 * I, pd + 16 * I, rx, rz, Z, s, win, ub, vb);
               }
            };
            rows(std::integral_constant<int, 0>());
            rows(std::integral_constant<int, 1>());
            rows(std::integral_constant<int, 2>());
            rows(std::integral_constant<int, 3>());
            const double2 hx = win[640 + 16 * j + lr], hy = win[704 + 16 * j + lr];
            const double a1w = hy.x * Z.z1wr - hy.y * Z.z1wi, a1r = hy.x * Z.z1rr - hy.y * Z.z1ri;
            const double a2 = hy.x * Z.z2r + hy.y * Z.z2i;
            const double a3 = hx.x * Z.z3r - hx.y * Z.z3i;
            const double a4w = hx.x * Z.z4wr + hx.y * Z.z4wi, a4r = hx.x * Z.z4rr + hx.y * Z.z4ri;
            const double h2 = 2.0 * Z.hw + Z.hr, b1 = a2 + a1w, b3 = a3 + a4w;
            const double iv = v0 + lr == a.nh - 1 ? 1.0 / qrule(a.rule).c_edge : 1.0;
            s[0] += 2.0 * (Z.hw + Z.hr);
            s[1] += b1 + a1r;
            s[2] += h2;
            s[3] += b3;
            s[4] += b1;
            s[5] += b3 + a4r;
            s[6] += iv * h2;
            s[7] += iv * b1;
            s[8] += iv * b3;
         }
         while (rule) {                                    // uniform per wave
            const int b = __builtin_ctz(rule);
            rule &= rule - 1;
            const int i = b / BC, j = b % BC;
            double g[4];
            switch (i) {
            case 0: getv(std::integral_constant<int, 0>(), j, g); break;
            case 1: if constexpr (BR > 1) getv(std::integral_constant<int, 1>(), j, g); break;
            case 2: if constexpr (BR > 2) getv(std::integral_constant<int, 2>(), j, g); break;
            default: if constexpr (BR > 3) getv(std::integral_constant<int, 3>(), j, g); break;
            }
            const int u0 = ub + 16 * i, v0 = vb + 16 * j;
            epi_rule<ST>(a, u0, v0, lane, g, s, win, ub, vb, wdb);
         }
         epi_flush<ONE, IL>(a, x, y, z, diag, lane, s, wave, f);
         f += epi_count(IL, x, y, z, diag);
      }
}

__device__ __forceinline__ void pair_from_index(long t, int &R, int &Q)
{
   long q = (long)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
   while ((q + 1) * (q + 2) / 2 <= t) ++q;
   while (q * (q + 1) / 2 > t) --q;
   Q = (int)q;
   R = (int)(t - q * (q + 1) / 2);
}

// XCD-aware order: workgroups dispatched to one XCD take consecutive logical
// ids, so the nm modes x that share one (R,Q) tile pair run on the same L2.
__device__ __forceinline__ long xcd_lid()
{
   const long nwg = (long)gridDim.x;
   const long wid = blockIdx.x;
   long lid = wid;
   const long per = nwg / 8;
   if (wid < per * 8) lid = (wid % 8) * per + wid / 8;
   return lid;
}

// Tiles of the FP64 G kernel: a wave takes 16 BR table rows x 16 BC table columns
// (r = BR / BC, 1 or 2).  G is symmetric: row tile R goes with the column tiles c from r R
// on, the first r of them diagonal.  The waves of a mode are numbered by groups of r
// columns, rows R <= g of group g one after the other; a workgroup takes four that follow
// one another and none of them idles (with four column tiles and a row tile per workgroup,
// those below the diagonal and beyond the last column did, on the same SIMDs throughout:
// 270 rows, 30 modes, 700 nodes 394 us where 64 x 64 tiles take 297).  Numbered by rows
// instead, 14 nodes, 28 modes, 81 frequencies take 589 us where this takes 561, and 166,
// 13, 374 1514 / 1493, but 22, 13, 176 255 / 261.
// Counts fit 32 bits: a plan's grid has at most 2^24 tile pairs of 64.
__host__ __device__ inline unsigned f64_group(unsigned g, unsigned r) { return r * (g * (g + 1) / 2); }

__host__ __device__ inline void f64_tile(unsigned i, unsigned nc, unsigned r, int &R, int &c)
{
   unsigned g = (unsigned)((sqrtf(8.0f * (float)i / r + 1.0f) - 1.0f) * 0.5f);   // the loops make it exact
   while (g > 0 && f64_group(g, r) > i) --g;
   while (f64_group(g + 1, r) <= i) ++g;
   const unsigned o = i - f64_group(g, r), n = nc - r * g < r ? nc - r * g : r;
   R = (int)(o / n);
   c = (int)(r * g + o % n);
}

// waves of a mode, workgroups of a mode
__host__ __device__ inline unsigned f64_waves(long rows, int BR, int BC)
{
   const unsigned nc = (unsigned)((rows + 16 * BC - 1) / (16 * BC)), r = BR / BC, g = nc / r;
   return f64_group(g, r) + nc % r * (g + 1);
}

__host__ __device__ inline long f64_tiles(long rows, int BR, int BC)
{
   return (f64_waves(rows, BR, BC) + 3L) / 4;
}

// One wave item of the FP64 G contraction: mode x, tile t.  The operands go from L1 / L2
// straight into the MFMA fragments (a fragment row is 16 contiguous table rows, 128
// bytes), D steps of 4 K rows ahead: no LDS, no barrier, so the two waves of a SIMD
// run out of phase and each hides the other's loads and epilogue.  FP64 MFMA and FP64
// vector instructions share one pipe (4 fma beside each MFMA cost their 16 cycles on
// top of its 64), so what is left to win is the vector work: the scaling by Psi_b
// (BR multiplies per 4 BR BC MFMAs) and the epilogue.  Staged through LDS with two
// barriers per chunk of 32 K rows it took 254 ms at 1000 nodes, 30 modes, 513
// frequencies (61 TFLOP/s where bare MFMA reaches 76.9) and 2690 / 262 us at 333, 17,
// 193 / 40, 20, 65; now 231.7 ms, of which the epilogue 24, and 2395 / 192 us, of which
// 497 / 130.
// The blocks near the origin and the resonances hold most of a moment, and with hundreds
// of small additions after them the order alone costs ten roundings and more; waves that
// add to one address wait for each other, too (some 40 ns each).  The workgroups of a mode
// therefore take the copies of the moments in turn, summed up at the end (k_sum_copies).
// Largest difference from the compensated sums of the same contributions over the largest
// moment, one copy -> gsym_copies of them: 30 nodes, 2 modes, 1025 frequencies 5.7e-15 ->
// 2.1e-16, 60, 16, 257 1.3e-15 -> 2.0e-16, 200, 24, 513 3.0e-15 -> 1.6e-16, 40, 9, 101
// 8.4e-16 -> 2.2e-16; times 18 nodes, 3 modes, 405 frequencies 92 -> 34 us, 132, 3, 504
// 136 -> 69, 27, 2, 254 30 -> 22.
template <int BR, int BC, bool ONE>
__device__ __forceinline__ void gsym_f64_wave(const GsymArgs &args, int x, long t)
{
   GsymArgs a = args;
   if (!ONE) {
      const long own = t % a.copies * (2L * a.nm * a.nm * a.nm);
      a.m3f += own;
      a.m3r += own;
   }
   constexpr int D = 4;                                      // K is a multiple of 32 = 8 D
   __shared__ double2 wins[4 * 768];
   const int lane = threadIdx.x & 63;
   const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int rows = a.nm * a.nhp, nc = (rows + 16 * BC - 1) / (16 * BC);
   const unsigned i = 4 * (unsigned)t + w;
   if (i >= f64_waves(rows, BR, BC)) return;                 // uniform per wave
   int R, c;
   f64_tile(i, nc, BR / BC, R, c);
   R = __builtin_amdgcn_readfirstlane(R);
   c = __builtin_amdgcn_readfirstlane(c);
   const int lr = lane & 15, lk = lane >> 4;
   const double *pA = a.U + (size_t)lk * a.ldU + R * 16 * BR + lr;
   const double *pB = a.U + (size_t)lk * a.ldU + c * 16 * BC + lr;
   const double *pbx = a.pb + (size_t)x * a.K + lk;
   d4 acc[BR][BC];
#pragma unroll
   for (int i = 0; i < BR; ++i)
#pragma unroll
      for (int j = 0; j < BC; ++j) acc[i][j] = (d4){0.0, 0.0, 0.0, 0.0};
   double ra[D][BR], rb[D][BC], rp[D];
   auto load = [&](int d, int k) {
      const size_t o = (size_t)k * a.ldU;
#pragma unroll
      for (int i = 0; i < BR; ++i) ra[d][i] = pA[o + 16 * i];
#pragma unroll
      for (int j = 0; j < BC; ++j) rb[d][j] = pB[o + 16 * j];
      rp[d] = pbx[k];
   };
#pragma unroll
   for (int d = 0; d < D; ++d) load(d, 4 * d);
   for (int k0 = 0; k0 < a.K; k0 += 4 * D) {
      const int kn = min(k0 + 4 * D, a.K - 4 * D);           // the last group again at the end: unused
#pragma unroll
      for (int d = 0; d < D; ++d) {
         double fa[BR], fb[BC];
#pragma unroll
         for (int i = 0; i < BR; ++i) fa[i] = ra[d][i] * rp[d];
#pragma unroll
         for (int j = 0; j < BC; ++j) fb[j] = rb[d][j];
         load(d, kn + 4 * d);
#pragma unroll
         for (int i = 0; i < BR; ++i)
#pragma unroll
            for (int j = 0; j < BC; ++j)
               acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
   }

   // ---- epilogue: for v_mfma_f64_16x16x4f64, register t of lane l holds
   // D[(l/16) + 4t][l%16] of its 16x16 block (rows interleaved by 4).
   const unsigned wave = (unsigned)((t * a.nm + x) * 4 + w);
   epi_wave<BR, BC, true, ONE>(a, x, c < (R + 1) * (BR / BC), R * 16 * BR, c * 16 * BC, lane, wave,
                  [&](auto ic, int j, double (&g)[4]) {
                     constexpr int I = decltype(ic)::value;
#pragma unroll
                     for (int q = 0; q < 4; ++q) {
                        double v = acc[I][0][q], u = acc[I][BC - 1][q];
                        // opaque: a select of the two addresses would put acc into memory
                        asm("" : "+v"(v), "+v"(u));
                        g[q] = j == 0 ? v : u;
                     }
                  },
                  wins + w * 768);
}

// Two waves per SIMD (registers; LDS allows three).  The bound of 4 for the tiles up to
// 2x2 makes the compiler keep the accumulators in AGPRs, without copies: with 2 it takes
// 96 us where 4 takes 93 at 151 nodes, 9 modes, 101 frequencies, 67 / 64 at 60, 8, 129,
// 32 / 27 at 300, 1, 193, and a call of the diagonal model 248 / 242 at 500, 20, 257.
// A bound of 3 spills: 153, 105, 32 and 245.
constexpr int f64_bound(int blocks) { return blocks > 4 ? 2 : 4; }

template <int BR, int BC>
__global__ __launch_bounds__(256, f64_bound(BR * BC)) void k_gsym_f64(GsymArgs a)
{
   const long lid = xcd_lid();
   gsym_f64_wave<BR, BC, false>(a, (int)(lid % a.nm), lid / a.nm);
}

// The ONLY_DIAG model's plane sums: mode x alone, i.e. the contraction and epilogue
// above for a one-mode structure whose table is the nodal PSDs X, with Psi_b W_x, FRF
// row x and the moments of mode x.  grid (tiles * nm).  Cutting K into slices that
// run side by side (the plane sums are linear in G) would fill the chip better at a few
// hundred nodes, but the slices' sums cancel: 5e-15 of the moments against 1e-15.
template <int BR, int BC>
__global__ __launch_bounds__(256, f64_bound(BR * BC)) void k_gsym_diag(GsymArgs a, int nmodes)
{
   const long lid = blockIdx.x;
   const int x = (int)(lid % nmodes);
   GsymArgs b = a;
   b.pb = a.pb + (size_t)x * a.K;
   b.H = a.H + (size_t)x * a.nft;
   b.m3f = a.m3f + x;
   b.m3r = a.m3r + x;
   gsym_f64_wave<BR, BC, true>(b, 0, lid / nmodes);
}

// ---------------------------------------------------------------------------
// G contraction in split-bf16 x3 on v_mfma_f32_16x16x32_bf16 (FP32 accumulate)
//   a*b ~= a_hi*b_hi + a_hi*b_lo + a_lo*b_hi,  a_hi = bf16(a), a_lo = bf16(a - a_hi)
// Operands come from the FP32 copy of the A table; the row operand is scaled
// by Psi_b(x,k) in FP32 before the split.  Same plane epilogue (FP64) as
// k_gsym_f64.  Workgroup tile 128x128, 4 waves of 64x64 (4x4 blocks of
// 16x16), K chunk 32 double-buffered in LDS.  LDS rows (64 bytes) hold four
// 16-byte k-groups stored at slot g ^ ((row >> 1) & 3): the 8 rows 0-7 (8-15)
// of a fragment read fill the 8 distinct 16-byte slots of a 128-byte line
// (SQ_LDS_BANK_CONFLICT reads zero for this kernel).
// ---------------------------------------------------------------------------
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));

#define T2 128
#define KC2 32

__device__ __forceinline__ uint32_t bf16_rne_bits(float f)
{
   const uint32_t b = __float_as_uint(f);
   return (b + 0x7FFFu + ((b >> 16) & 1u)) >> 16;
}

__device__ __forceinline__ int swz(int row, int g) { return row * 4 + (g ^ ((row >> 1) & 3)); }

struct GsymArgs16 {
   const float *UR;       // [rows][ldk]  A table, FP32, K contiguous (row operand source)
   const uint4 *UCh;      // [rows][ldk/8] bf16 hi of the A table (column operand)
   const uint4 *UCl;      // [rows][ldk/8] bf16 lo
   const float *pb32;     // [nm][ldk]  Psi_b per K index, FP32
   long ldk;              // K stride (multiple of 32)
};

// One work item of the split-bf16x3 G contraction: mode x, tile pair tp.
__device__ __forceinline__ void gsym_bf16x3_item(const GsymArgs &a, const GsymArgs16 &b, int x,
                                                 long tp)
{
   __shared__ uint4 Ah[2][T2 * 4], Al[2][T2 * 4], Bh[2][T2 * 4], Bl[2][T2 * 4];
   int R, Q;
   pair_from_index(tp, R, Q);
   const bool diag = (R == Q);

   const int tid = threadIdx.x;
   const int lane = tid & 63;
   const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform
   const int wr = w >> 1, wc = w & 1;

   // staging: items tid and tid+256 -> (row = item/4, k-group = item%4 of 8)
   const int srow0 = tid >> 2, srow1 = srow0 + 64;
   const int sgrp = tid & 3;
   const long ldk = b.ldk;
   const float *gA0 = b.UR + ((size_t)R * T2 + srow0) * ldk + sgrp * 8;
   const float *gA1 = b.UR + ((size_t)R * T2 + srow1) * ldk + sgrp * 8;
   const uint4 *gBh0 = b.UCh + (((size_t)Q * T2 + srow0) * ldk + sgrp * 8) / 8;
   const uint4 *gBh1 = b.UCh + (((size_t)Q * T2 + srow1) * ldk + sgrp * 8) / 8;
   const uint4 *gBl0 = b.UCl + (((size_t)Q * T2 + srow0) * ldk + sgrp * 8) / 8;
   const uint4 *gBl1 = b.UCl + (((size_t)Q * T2 + srow1) * ldk + sgrp * 8) / 8;
   const float *pbx = b.pb32 + (size_t)x * ldk + sgrp * 8;

   f4v acc[4][4];
#pragma unroll
   for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = (f4v){0.f, 0.f, 0.f, 0.f};

   float4 ra0, ra1, ra2, ra3, sc0, sc1;
   uint4 rbh0, rbh1, rbl0, rbl1;
   auto gload = [&](int k0) {
      ra0 = *(const float4 *)(gA0 + k0);
      ra1 = *(const float4 *)(gA0 + k0 + 4);
      ra2 = *(const float4 *)(gA1 + k0);
      ra3 = *(const float4 *)(gA1 + k0 + 4);
      sc0 = *(const float4 *)(pbx + k0);
      sc1 = *(const float4 *)(pbx + k0 + 4);
      rbh0 = gBh0[k0 / 8];
      rbh1 = gBh1[k0 / 8];
      rbl0 = gBl0[k0 / 8];
      rbl1 = gBl1[k0 / 8];
   };
   auto split2 = [](float v0, float v1, uint32_t &h, uint32_t &l) {
      const f2v vv = (f2v){v0, v1};
      const bf2v hv = __builtin_convertvector(vv, bf2v);              // v_cvt_pk_bf16_f32 (RNE)
      const f2v r = vv - __builtin_convertvector(hv, f2v);             // exact in FP32
      h = __builtin_bit_cast(uint32_t, hv);
      l = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf2v));
   };
   auto split8 = [&](float4 p0, float4 p1, uint4 &hi, uint4 &lo) {
      split2(p0.x * sc0.x, p0.y * sc0.y, hi.x, lo.x);
      split2(p0.z * sc0.z, p0.w * sc0.w, hi.y, lo.y);
      split2(p1.x * sc1.x, p1.y * sc1.y, hi.z, lo.z);
      split2(p1.z * sc1.z, p1.w * sc1.w, hi.w, lo.w);
   };
   auto lstore = [&](int buf) {
      uint4 hi, lo;
      split8(ra0, ra1, hi, lo);
      Ah[buf][swz(srow0, sgrp)] = hi;
      Al[buf][swz(srow0, sgrp)] = lo;
      split8(ra2, ra3, hi, lo);
      Ah[buf][swz(srow1, sgrp)] = hi;
      Al[buf][swz(srow1, sgrp)] = lo;
      Bh[buf][swz(srow0, sgrp)] = rbh0;
      Bh[buf][swz(srow1, sgrp)] = rbh1;
      Bl[buf][swz(srow0, sgrp)] = rbl0;
      Bl[buf][swz(srow1, sgrp)] = rbl1;
   };

   const int nchunk = a.K / KC2;
   // the K loop at raised wave priority, the epilogue at the default: where the
   // two workgroups of a CU are in different phases, the MFMA-issuing waves are
   // served first and the epilogue's FP64 VALU work fills the gaps (measured:
   // 1-1.4 % shorter kernel; the reverse order gains nothing)
   __builtin_amdgcn_s_setprio(1);
   gload(0);
   __syncthreads();      // a previous item's epilogue (persistent batch) may still read LDS
   lstore(0);
   __syncthreads();
   for (int c = 0; c < nchunk; ++c) {
      const int buf = c & 1;
      if (c + 1 < nchunk) gload((c + 1) * KC2);
      const int g = lane >> 4;
      bf8 ah[4], al[4], bh[4], bl[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
         const int row = wr * 64 + i * 16 + (lane & 15);
         const int col = wc * 64 + i * 16 + (lane & 15);
         ah[i] = __builtin_bit_cast(bf8, Ah[buf][swz(row, g)]);
         al[i] = __builtin_bit_cast(bf8, Al[buf][swz(row, g)]);
         bh[i] = __builtin_bit_cast(bf8, Bh[buf][swz(col, g)]);
         bl[i] = __builtin_bit_cast(bf8, Bl[buf][swz(col, g)]);
      }
      // small products first; product-major order keeps consecutive MFMAs independent
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
         for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
         for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
         for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
      if (c + 1 < nchunk) lstore(buf ^ 1);
      __syncthreads();
   }

   __builtin_amdgcn_s_setprio(0);
   // epilogue: f32-output 16x16 MFMAs hold D[4(l/16)+t][l%16]
   const unsigned wave = (unsigned)((tp * a.nm + x) * 4 + w);
   // each wave's FRF window: 12 KB of one operand plane (16 KB), free after the
   // last chunk's barrier
   uint4 *plane = w == 0 ? &Ah[0][0] : (w == 1 ? &Al[0][0] : (w == 2 ? &Bh[0][0] : &Bl[0][0]));
   double2 *win = reinterpret_cast<double2 *>(plane);
   epi_wave<4, 4, false, false>(a, x, diag, R * T2 + wr * 64, Q * T2 + wc * 64, lane, wave,
                  [&](auto ic, int j, double (&g)[4]) {
                     constexpr int I = decltype(ic)::value;
                     f4v v = acc[I][3];
                     switch (j) {       // uniform branch: constant register indices
                     case 0: v = acc[I][0]; break;
                     case 1: v = acc[I][1]; break;
                     case 2: v = acc[I][2]; break;
                     default: break;
                     }
#pragma unroll
                     for (int t = 0; t < 4; ++t) g[t] = (double)v[t];
                  },
                  win);
}

__global__ __launch_bounds__(256, 2) void k_gsym_bf16x3(GsymArgs a, GsymArgs16 b)
{
   const long lid = xcd_lid();
   gsym_bf16x3_item(a, b, (int)(lid % a.nm), lid / a.nm);
}

// ---------------------------------------------------------------------------
// G contraction in FP32 on v_mfma_f32_16x16x4f32 (FP32 operands, FP32
// accumulate); same plane epilogue (FP64) as k_gsym_f64.  Workgroup tile
// 128x128, 4 waves of 64x64 (4x4 blocks of 16x16), K chunk 32 double-buffered
// in LDS (two FP32 planes, 64 KB).  Within a chunk, MFMA step s (0..7) takes
// k = 8 (l/16) + s for lane l in both operands (any assignment of the chunk's
// 32 k to (step, lane group) gives the same sum), so a lane reads its 8 k of
// one row as two 16-byte LDS loads.  LDS rows (128 bytes) hold eight 16-byte
// k-groups stored at slot q ^ (row & 7).  Measured at NN=1000, NM=30: half the
// bank-conflict cycles of slot q ^ ((row >> 1) & 7) and 2.4 % faster; slot
// q ^ ((row ^ (row >> 3)) & 7) has none but ran 1.7 % slower than this one.
// ---------------------------------------------------------------------------
#define KC4 32

__device__ __forceinline__ int swz8(int row, int q) { return row * 8 + (q ^ (row & 7)); }

__device__ __forceinline__ void gsym_f32_item(const GsymArgs &a, const GsymArgs16 &b, int x, long tp)
{
   __shared__ float4 As[2][T2 * 8], Bs[2][T2 * 8];
   int R, Q;
   pair_from_index(tp, R, Q);
   const bool diag = (R == Q);

   const int tid = threadIdx.x;
   const int lane = tid & 63;
   const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform
   const int wr = w >> 1, wc = w & 1;

   // staging: thread -> (row = tid/2, k-groups 4h..4h+3 of 4 floats), h = tid%2
   const int srow = tid >> 1, sh = tid & 1;
   const long ldk = b.ldk;
   const float *gA = b.UR + ((size_t)R * T2 + srow) * ldk + sh * 16;
   const float *gB = b.UR + ((size_t)Q * T2 + srow) * ldk + sh * 16;
   const float *pbx = b.pb32 + (size_t)x * ldk + sh * 16;

   f4v acc[4][4];
#pragma unroll
   for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = (f4v){0.f, 0.f, 0.f, 0.f};

   float4 ra[4], rb[4], sc[4];
   auto gload = [&](int k0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
         ra[j] = *(const float4 *)(gA + k0 + 4 * j);
         rb[j] = *(const float4 *)(gB + k0 + 4 * j);
         sc[j] = *(const float4 *)(pbx + k0 + 4 * j);
      }
   };
   auto lstore = [&](int buf) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
         const float4 v = ra[j], s = sc[j];
         As[buf][swz8(srow, 4 * sh + j)] = make_float4(v.x * s.x, v.y * s.y, v.z * s.z, v.w * s.w);
         Bs[buf][swz8(srow, 4 * sh + j)] = rb[j];
      }
   };

   const int nchunk = a.K / KC4;
   __builtin_amdgcn_s_setprio(1);   // K loop at raised wave priority, as k_gsym_bf16x3
   gload(0);
   __syncthreads();      // a previous item's epilogue (persistent batch) may still read LDS
   lstore(0);
   __syncthreads();
   const int g = lane >> 4;            // lane group: k = 8g .. 8g+7 of the chunk
   for (int c = 0; c < nchunk; ++c) {
      const int buf = c & 1;
      if (c + 1 < nchunk) gload((c + 1) * KC4);
#pragma unroll
      for (int hsel = 0; hsel < 2; ++hsel) {       // steps 4 hsel .. 4 hsel + 3
         float4 fa[4], fb[4];
#pragma unroll
         for (int i = 0; i < 4; ++i) {
            const int row = wr * 64 + i * 16 + (lane & 15);
            const int col = wc * 64 + i * 16 + (lane & 15);
            fa[i] = As[buf][swz8(row, 2 * g + hsel)];
            fb[i] = Bs[buf][swz8(col, 2 * g + hsel)];
         }
#pragma unroll
         for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
               for (int j = 0; j < 4; ++j)
                  acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                     ((const float *)&fa[i])[s], ((const float *)&fb[j])[s], acc[i][j], 0, 0, 0);
      }
      if (c + 1 < nchunk) lstore(buf ^ 1);
      __syncthreads();
   }

   // epilogue: f32-output 16x16 MFMAs hold D[4(l/16)+t][l%16]
   const unsigned wave = (unsigned)((tp * a.nm + x) * 4 + w);
   __builtin_amdgcn_s_setprio(0);
   // each wave's FRF window: 12 KB of the operand planes (2 x 32 KB), free after
   // the last chunk's barrier
   double2 *win = reinterpret_cast<double2 *>(w < 2 ? &As[0][0] : &Bs[0][0]) + (w & 1) * 768;
   epi_wave<4, 4, false, false>(a, x, diag, R * T2 + wr * 64, Q * T2 + wc * 64, lane, wave,
                  [&](auto ic, int j, double (&gv)[4]) {
                     constexpr int I = decltype(ic)::value;
                     f4v v = acc[I][3];
                     switch (j) {       // uniform branch: constant register indices
                     case 0: v = acc[I][0]; break;
                     case 1: v = acc[I][1]; break;
                     case 2: v = acc[I][2]; break;
                     default: break;
                     }
#pragma unroll
                     for (int t = 0; t < 4; ++t) gv[t] = (double)v[t];
                  },
                  win);
}

__global__ __launch_bounds__(256, 2) void k_gsym_f32(GsymArgs a, GsymArgs16 b)
{
   const long lid = xcd_lid();
   gsym_f32_item(a, b, (int)(lid % a.nm), lid / a.nm);
}

// Lane-layout self test of v_mfma_f32_16x16x4f32 (one wave, 512 floats):
// out[t*64 + l] = D[4(l/16)+t][l%16] of A[i][k] = i + 16 k, B = identity
// columns k == j % 4 (so D[i][j] = i + 16 (j % 4)); out[256 + t*64 + l] of
// A[i][k] = 1, B[k][j] = k + 4 j (D[i][j] = 6 + 16 j).
__global__ void k_mfma_f32_layout(float *__restrict__ out)
{
   const int l = threadIdx.x;
   const int i = l & 15, k = l >> 4;
   const f4v z = (f4v){0.f, 0.f, 0.f, 0.f};
   const f4v d1 = __builtin_amdgcn_mfma_f32_16x16x4f32((float)(i + 16 * k),
                                                       (k == (i & 3)) ? 1.f : 0.f, z, 0, 0, 0);
   const f4v d2 = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, (float)(k + 4 * i), z, 0, 0, 0);
#pragma unroll
   for (int t = 0; t < 4; ++t) {
      out[t * 64 + l] = d1[t];
      out[256 + t * 64 + l] = d2[t];
   }
}

// A table [K][ldU] (FP64) -> row operand [rows][ldk] FP32 and column operand
// [rows][ldk] split into bf16 hi/lo (Ch, Cl NULL: the FP32 copy only).  32x32
// tiles transposed through LDS.
__device__ __forceinline__ void split_tile(int r0, int k0, const double *__restrict__ U, long ldU,
                                           int K, int rows, long ldk, float *__restrict__ UR,
                                           uint16_t *__restrict__ Ch, uint16_t *__restrict__ Cl)
{
   __shared__ float tile[32][33];
   const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;     // 256 threads: 32 x 8
   for (int j = ty; j < 32; j += 8) {
      const int k = k0 + j, r = r0 + tx;
      tile[j][tx] = (k < K && r < rows) ? (float)U[(size_t)k * ldU + r] : 0.f;
   }
   __syncthreads();
   for (int j = ty; j < 32; j += 8) {
      const int r = r0 + j, k = k0 + tx;
      if (r < rows && k < ldk) {
         const float v = tile[tx][j];
         const size_t o = (size_t)r * ldk + k;
         UR[o] = v;
         if (Ch) {                 // bf16 planes (split-bf16x3 only)
            const __bf16 h = (__bf16)v;
            const __bf16 l = (__bf16)(v - (float)h);
            Ch[o] = __builtin_bit_cast(uint16_t, h);
            Cl[o] = __builtin_bit_cast(uint16_t, l);
         }
      }
   }
}

__global__ void k_split_table(const double *__restrict__ U, long ldU, int K, int rows, long ldk,
                              float *__restrict__ UR, uint16_t *__restrict__ Ch,
                              uint16_t *__restrict__ Cl)
{
   split_tile(blockIdx.x * 32, blockIdx.y * 32, U, ldU, K, rows, ldk, UR, Ch, Cl);
}

// Lane-layout self test of v_mfma_f32_16x16x32_bf16 (one wave, 768 floats):
// three products with known answers, see bsahip_selftest_mfma_layout.
__global__ void k_mfma_bf16_layout(float *__restrict__ out)
{
   const int l = threadIdx.x;
   const int row = l & 15, g = l >> 4;
   uint32_t a1[8], b1[8], a2[8], b2[8], b3[8];
#pragma unroll
   for (int j = 0; j < 8; ++j) {
      const int k = 8 * g + j;                    // k index this element holds (assumed)
      a1[j] = bf16_rne_bits(k == 0 ? (float)row : 0.f);
      b1[j] = bf16_rne_bits(k == 0 ? 1.f : 0.f);
      a2[j] = bf16_rne_bits((float)k);
      b2[j] = bf16_rne_bits(k == row ? 1.f : 0.f);          // B[k][col=row-of-lane]
      b3[j] = bf16_rne_bits(k == row + 16 ? 1.f : 0.f);
   }
   auto pack = [](const uint32_t (&v)[8]) {
      uint4 q = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
      return __builtin_bit_cast(bf8, q);
   };
   const f4v z = (f4v){0.f, 0.f, 0.f, 0.f};
   const f4v d1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pack(a1), pack(b1), z, 0, 0, 0);
   const f4v d2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pack(a2), pack(b2), z, 0, 0, 0);
   const f4v d3 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pack(a2), pack(b3), z, 0, 0, 0);
#pragma unroll
   for (int t = 0; t < 4; ++t) {
      out[t * 64 + l] = d1[t];
      out[256 + t * 64 + l] = d2[t];
      out[512 + t * 64 + l] = d3[t];
   }
}

// ---------------------------------------------------------------------------
// modal PSD and second moments (functionsImpl.F90:1546-1558, 1686-1689;
// BsaClassicImpl.F90:197-210, 567-589).
// psd(n,p;u) = sum_k U[k][n*nhp+u] Psi_a(p,k); the grid holds +-u.
// ---------------------------------------------------------------------------
// Modal PSD moments: PSD(n,p;u) = sum_k A(n,k;u) Psi_a(p,k) on the half grid,
// weighted with the vect rule (+u and -u), times Re[H_p conj(H_n)] and w^2.
// A block takes 64 frequencies of mode n and 16 MT modes p as FP64 MFMA tiles (rows u,
// columns p), its four waves a quarter of K each; the weights are linear, so each wave
// reduces its own partial PSDs over u and only 3 x 16 MT sums meet in LDS.  Reads the
// table once per 32 modes p (once per pair (n, p) before, on the vector unit): bound by
// those reads.  1000 nodes, 30 modes, 513 frequencies: 1.55 -> 0.35 ms beside the G kernel.
// Partial sums of the blocks are added atomically (the outputs start at zero), or with
// m2part stored per frequency block for a fixed-order sum (k_sum_fixed).
struct M2Args {
   const double *U;
   long ldU;
   const double *pa;          // [nm][K]
   int K, nm, nhp, nh;        // K a multiple of 16
   const double2 *H;
   int nft;
   double d, om_step;
   double *m2f, *m2r, *m2o;
   double *m2part;            // NULL, or [frequency block][3][nm^2]
   int diag;                  // ONLY_DIAG: n = 0, pa = Psi_l^2, entry p weighed by |H_p|^2
   int kper;                  // K rows per slice (a multiple of 16; K: no slices)
};

template <int MT>
__device__ __forceinline__ void m2_block(const M2Args &A, int n, int by, int p0, int sl)
{
   __shared__ double red[4][3][16 * MT];
   const int lane = threadIdx.x & 63;
   const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int lr = lane & 15, lk = lane >> 4;
   const int u0 = by * 64;
   const double *ua[4], *pb[MT];
#pragma unroll
   for (int i = 0; i < 4; ++i)                         // frequencies beyond the grid: weight 0
      ua[i] = A.U + (size_t)n * A.nhp + min(u0 + 16 * i + lr, A.nh - 1) + (size_t)(4 * w + lk) * A.ldU;
#pragma unroll
   for (int j = 0; j < MT; ++j) pb[j] = A.pa + (size_t)min(p0 + 16 * j + lr, A.nm - 1) * A.K + 4 * w + lk;
   d4 acc[4][MT];
#pragma unroll
   for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = (d4){0.0, 0.0, 0.0, 0.0};
   double av[4], bv[MT];
   auto load = [&](int k) {
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = ua[i][(size_t)k * A.ldU];
#pragma unroll
      for (int j = 0; j < MT; ++j) bv[j] = pb[j][k];
   };
   const int k0 = sl * A.kper, k1 = min(A.K, k0 + A.kper);
   load(k0);
#pragma unroll 2
   for (int k = k0; k < k1; k += 16) {
      double a[4], b[MT];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = av[i];
#pragma unroll
      for (int j = 0; j < MT; ++j) b[j] = bv[j];
      if (k + 16 < k1) load(k + 16);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
         for (int j = 0; j < MT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
   }
#pragma unroll
   for (int j = 0; j < MT; ++j) {
      const int p = min(p0 + 16 * j + lr, A.nm - 1);
      double sf = 0.0, sr = 0.0, so = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
         for (int t = 0; t < 4; ++t) {
            const int u = u0 + 16 * i + lk + 4 * t;
            if (u < A.nh) {
               double wt = (u == A.nh - 1) ? 0.5 * A.d : A.d;
               if (u > 0) wt *= 2.0;                                // +u and -u
               const double2 hp = A.H[(size_t)p * A.nft + u], hn = A.H[(size_t)(A.diag ? p : n) * A.nft + u];
               const double fr = hp.x * hn.x + hp.y * hn.y;         // Re[H_p conj(H_n)]
               const double om = A.om_step * u;
               const double v = wt * acc[i][j][t];
               sf += v;
               sr += v * fr;
               so += v * fr * om * om;
            }
         }
      sf += __shfl_xor(sf, 16, 64);
      sr += __shfl_xor(sr, 16, 64);
      so += __shfl_xor(so, 16, 64);
      sf += __shfl_xor(sf, 32, 64);
      sr += __shfl_xor(sr, 32, 64);
      so += __shfl_xor(so, 32, 64);
      if (lk == 0) {
         red[w][0][16 * j + lr] = sf;
         red[w][1][16 * j + lr] = sr;
         red[w][2][16 * j + lr] = so;
      }
   }
   __syncthreads();
   const int pl = threadIdx.x, p = p0 + pl;
   if (pl < 16 * MT && p < A.nm) {
      const size_t nm2 = (size_t)A.nm * A.nm, id = A.diag ? (size_t)p : n + (size_t)A.nm * p;
      double s[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) s[c] = (red[0][c][pl] + red[1][c][pl]) + (red[2][c][pl] + red[3][c][pl]);
      if (A.m2part) {
         double *o = A.m2part + (size_t)by * 3 * nm2 + id;
         o[0] = s[0];
         o[nm2] = s[1];
         o[2 * nm2] = s[2];
      } else {
         atomicAdd(A.m2f + id, s[0]);
         atomicAdd(A.m2r + id, s[1]);
         atomicAdd(A.m2o + id, s[2]);
      }
   }
}

// grid (nm (diag: 1), ceil(nh/64), ceil(nm / (16 MT)) * K slices)
template <int MT>
__global__ __launch_bounds__(256, 2) void k_m2(M2Args A)
{
   const int np = (A.nm + 16 * MT - 1) / (16 * MT);
   m2_block<MT>(A, blockIdx.x, blockIdx.y, (int)blockIdx.z % np * 16 * MT, (int)blockIdx.z / np);
}

// Fixed-order compensated sums.  k_sum_lists: out[e] = sum over the slot list
// idx[off[e] .. off[e+1]) of vals (ascending slot order), Kahan-compensated;
// k_sum_fixed: out[i] = sum_b part[b * stride + i] for b = 0 .. nb-1, likewise.
__device__ __forceinline__ void kahan_add(double &s, double &c, double v)
{
   const double y = v - c;
   const double t = s + y;
   c = (t - s) - y;
   s = t;
}

// Sum of nc doubles v(0 .. nc-1), compensated; the plain sum where it is no longer finite
// (the correction of an infinity would be NaN).  W loads go out together: on the device
// 192 of them one after the other took 35 us.
template <class Get>
__device__ __forceinline__ double sum_all(int nc, Get v)
{
   constexpr int W = 16;
   double s = v(0), c = 0.0, plain = s, q[W];
   for (int k = 1; k < nc; k += W) {
#pragma unroll
      for (int j = 0; j < W; ++j) q[j] = k + j < nc ? v(k + j) : 0.0;
#pragma unroll
      for (int j = 0; j < W; ++j) {
         kahan_add(s, c, q[j]);
         plain += q[j];
      }
   }
   return plain - plain == 0.0 ? s : plain;
}

// p[i] = sum of the nc copies p[c * n + i], n doubles each
__global__ void k_sum_copies(double *p, long n, int nc)
{
   const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (i < n) p[i] = sum_all(nc, [&](int c) { return p[c * n + i]; });
}

__global__ void k_sum_lists(const double *__restrict__ vals, const long *__restrict__ off,
                            const long *__restrict__ idx, long n, double *__restrict__ out)
{
   const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (e >= n) return;
   double s = 0.0, c = 0.0;
   for (long q = off[e]; q < off[e + 1]; ++q) kahan_add(s, c, vals[idx[q]]);
   out[e] = s;
}

__global__ void k_sum_fixed(const double *__restrict__ part, int nb, long stride, long n,
                            double *__restrict__ out)
{
   const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= n) return;
   double s = 0.0, c = 0.0;
   for (int b = 0; b < nb; ++b) kahan_add(s, c, part[(size_t)b * stride + i]);
   out[i] = s;
}

// Modal PSD on grid indices (for the spectra output): psd(q, n+p*nm).
__global__ void k_psd_grid(const double *__restrict__ U, long ldU, const double *__restrict__ pa,
                           int K, int nm, int nhp, int nf, int c, const double2 *__restrict__ H,
                           int nft, double *__restrict__ psd_f, double *__restrict__ psd_r)
{
   const int q = blockIdx.x * blockDim.x + threadIdx.x;
   const int np = blockIdx.y;
   if (q >= nf) return;
   const int n = np % nm, p = np / nm;
   const int u = abs(q - c);
   double s = 0.0;
   for (int k = 0; k < K; ++k) s = fma(U[(size_t)k * ldU + (size_t)n * nhp + u], pa[(size_t)p * K + k], s);
   const double2 hp = H[(size_t)p * nft + u], hn = H[(size_t)n * nft + u];
   if (psd_f) psd_f[(size_t)np * nf + q] = s;
   if (psd_r) psd_r[(size_t)np * nf + q] = s * (hp.x * hn.x + hp.y * hn.y);
}

// ---------------------------------------------------------------------------
// Modal force bispectrum of triple (m, n, p) at one point from the projection
// table U: rows a1 -> |f1|, a2 -> |f2|, a3 -> |f1+f2| (a3 < 0: S(f1+f2) = 0).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double bfm_point(const double *__restrict__ U, long ldU, int rows,
                                            const double *__restrict__ pb, int K, int m, int n,
                                            int p, int a1, int a2, int a3)
{
   double s = 0.0;
   for (int k = 0; k < K; ++k) {
      const double *row = U + (size_t)k * ldU;
      const double An1 = row[(size_t)n * rows + a1], Ap2 = row[(size_t)p * rows + a2];
      double v = pb[(size_t)m * K + k] * An1 * Ap2;
      if (a3 >= 0) {
         const double Am3 = row[(size_t)m * rows + a3];
         v += pb[(size_t)n * K + k] * Am3 * Ap2 + pb[(size_t)p * K + k] * Am3 * An1;
      }
      s += v;
   }
   return 2.0 * s;
}

// One G value G[x](y,u; z,v) = sum_k Psi_b(x,k) A(y,k;u) A(z,k;v) with the
// operand rounding of the mixed-precision G kernels: the operand of the lower
// table row (the kernels' row operand) is fl32(A) fl32(Psi_b) in FP32, the
// other fl32(A); PREC 1 (FP32) accumulates their FP32 product, PREC 2
// (split-bf16x3) the three bf16 products lo*hi + hi*lo + hi*hi, all in FP32
// and in K order (the MFMA path sums in another order; its error per term is
// the same).
template <int PREC>
__device__ __forceinline__ float g_value_mixed(const double *__restrict__ U, long ldU, int rows,
                                               const double *__restrict__ pb, int K, int x, int y,
                                               int u, int z, int v)
{
   if ((long)z * rows + v < (long)y * rows + u) {
      const int ty = y, tu = u;
      y = z;
      u = v;
      z = ty;
      v = tu;
   }
   float acc = 0.f;
   for (int k = 0; k < K; ++k) {
      const double *row = U + (size_t)k * ldU;
      const float a = (float)row[(size_t)y * rows + u] * (float)pb[(size_t)x * K + k];
      const float b = (float)row[(size_t)z * rows + v];
      if constexpr (PREC == 1) {
         acc = fmaf(a, b, acc);
      } else {
         const float ah = (float)(__bf16)a, bh = (float)(__bf16)b;
         const float al = (float)(__bf16)(a - ah), bl = (float)(__bf16)(b - bh);
         acc = fmaf(al, bh, acc);
         acc = fmaf(ah, bl, acc);
         acc = fmaf(ah, bh, acc);
      }
   }
   return acc;
}

// bfm_point with the G values of the mixed-precision kernels (g_value_mixed).
template <int PREC>
__device__ __forceinline__ double bfm_point_mixed(const double *__restrict__ U, long ldU, int rows,
                                                  const double *__restrict__ pb, int K, int m,
                                                  int n, int p, int a1, int a2, int a3)
{
   double s = (double)g_value_mixed<PREC>(U, ldU, rows, pb, K, m, n, a1, p, a2);
   if (a3 >= 0) {
      s += (double)g_value_mixed<PREC>(U, ldU, rows, pb, K, n, m, a3, p, a2);
      s += (double)g_value_mixed<PREC>(U, ldU, rows, pb, K, p, m, a3, n, a1);
   }
   return 2.0 * s;
}

// Response factor Re[H_m(f1) H_n(f2) conj H_p(f1+f2)] from the modal mass,
// stiffness and damping; H at f1+f2 uses w1 + w2 as the reference does
// (functionsImpl.F90:1659-1663).
__device__ __forceinline__ double brm_factor(double f1, double f2, int m, int n, int p,
                                             const double *__restrict__ Mm,
                                             const double *__restrict__ Km,
                                             const double *__restrict__ Cm)
{
   auto H = [&](int mo, double w) {
      const double r = -(w * w * Mm[mo]) + Km[mo];
      const double im = w * Cm[mo];
      const double d = r * r + im * im;
      return make_double2(r / d, -im / d);
   };
   const double w1 = 2.0 * M_PI * f1, w2 = 2.0 * M_PI * f2;
   return re3(H(m, w1), H(n, w2), H(p, w1 + w2));
}

// ---------------------------------------------------------------------------
// Per-point bispectrum: B(m,n,p) at points given by row indices into U
// (i1 -> f1, i2 -> f2, i3 -> f1+f2, i3 < 0 means S(f1+f2) = 0) and the
// signed frequencies for the FRF.  out index = pt*nm^3 + mnp.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_bfm_points(
   const double *__restrict__ U, long ldU, int rows, const double *__restrict__ pb, int K,
   int nm, int npts, const int *__restrict__ i1, const int *__restrict__ i2,
   const int *__restrict__ i3, const double *__restrict__ f1s, const double *__restrict__ f2s,
   const double *__restrict__ Mm, const double *__restrict__ Km, const double *__restrict__ Cm,
   double *__restrict__ bfm, double *__restrict__ brm)
{
   const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
   const long nm3 = (long)nm * nm * nm;
   if (gid >= nm3 * npts) return;
   const long pt = gid / nm3;
   const int mnp = (int)(gid % nm3);
   const int m = mnp % nm, n = (mnp / nm) % nm, p = mnp / (nm * nm);
   const double s = bfm_point(U, ldU, rows, pb, K, m, n, p, i1[pt], i2[pt], i3[pt]);
   bfm[gid] = s;
   if (brm) brm[gid] = s * brm_factor(f1s[pt], f2s[pt], m, n, p, Mm, Km, Cm);
}

// brm[e] = bfm[e] Re[H_m(f1) H_n(f2) conj H_p(f1+f2)] at points, e = pt nm^3 + mnp
__global__ __launch_bounds__(256) void k_brm_points(const double *__restrict__ bfm, int nm, long total,
                                                    const double *__restrict__ f1s,
                                                    const double *__restrict__ f2s,
                                                    const double *__restrict__ Mm,
                                                    const double *__restrict__ Km,
                                                    const double *__restrict__ Cm,
                                                    double *__restrict__ brm)
{
   const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
   const long nm3 = (long)nm * nm * nm;
   if (e >= total) return;
   const long pt = e / nm3;
   const int mnp = (int)(e % nm3);
   brm[e] = bfm[e] * brm_factor(f1s[pt], f2s[pt], mnp % nm, (mnp / nm) % nm, mnp / (nm * nm), Mm, Km, Cm);
}

// ---------------------------------------------------------------------------
// Bispectra of mode triples on the Classic grid f = (q - c) df, q = 0 .. nf-1:
// out[q1 + nf*q2 + nf*nf*s] for triple sel[s] (linear index m + n*nm + p*nm^2,
// m fastest; sel null: triple s), the reference's bisp(i, j, k) layout.
// Rows of U: |F| for F within the grid; with exact, |f1+f2| up to 2c as well,
// otherwise S(f1+f2) = 0 beyond the grid.
//
// FP64: one workgroup per 16x16 tile (|F1|, |F2|) and triple,
//   B = 2 (G_m[(n,F1),(p,F2)] + G_n[(m,F3),(p,F2)] + G_p[(m,F3),(n,F1)]),
// F3 = |F1 + F2| and |F1 - F2| in windows of 32 from |16 (a+b)| and 16 (a-b) - 16 on:
// nine 16x16 blocks by MFMA.  A tile gives the four sign combinations of its points,
// which are two values.  Its waves share the contraction (k = 16 i + 4 wave + 0..3) and
// their parts are added in wave order, so a value does not depend on which launch formed
// it.  One value per lane with a serial loop over k, five loads per term, took 286 us
// for 3 triples, 300 nodes and 2 components, 257^2 points; now 33 us.
// grid (tiles^2, min(nsel, 65535), ceil(nsel / 65535)), block 256
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256, 2) void k_bisp_grid_f64(
   const double *__restrict__ U, long ldU, int rows, const double *__restrict__ pb, int K,
   int nm, int nf, double df, long nsel, const int *__restrict__ sel,
   const double *__restrict__ Mm, const double *__restrict__ Km, const double *__restrict__ Cm,
   double *__restrict__ bfm, double *__restrict__ brm)
{
   __shared__ double part[4][9][256];
   const long s = blockIdx.y + (long)gridDim.y * blockIdx.z;
   if (s >= nsel) return;
   const int c = (nf - 1) / 2, nt = (c + 16) / 16;
   const int ta = (int)(blockIdx.x % nt), tb = (int)(blockIdx.x / nt);
   const int mnp = sel ? sel[s] : (int)s;
   const int m = mnp % nm, n = (mnp / nm) % nm, p = mnp / (nm * nm);
   const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 15, kk = 4 * wv + (lane >> 4);
   // table rows of the lane's operands; those beyond the table are clamped and their
   // products never used
   const int last = rows - 1, d0 = 16 * (ta - tb) - 16 + l;
   const double *An = U + (size_t)kk * ldU + (size_t)n * rows + min(16 * ta + l, last);
   const double *Ap = U + (size_t)kk * ldU + (size_t)p * rows + min(16 * tb + l, last);
   const double *Am = U + (size_t)kk * ldU + (size_t)m * rows;
   const int r0 = min(16 * (ta + tb) + l, last), r1 = min(16 * (ta + tb) + 16 + l, last);
   const int r2 = min(abs(d0), last), r3 = min(abs(d0 + 16), last);
   const double *bm = pb + (size_t)m * K + kk, *bn = pb + (size_t)n * K + kk, *bp = pb + (size_t)p * K + kk;
   d4 acc[9];
#pragma unroll
   for (int t = 0; t < 9; ++t) acc[t] = (d4){0.0, 0.0, 0.0, 0.0};
   // K is a multiple of 32: every wave has K / 16 steps
#pragma unroll 2
   for (int k = 0; k < K; k += 16) {
      const size_t o = (size_t)k * ldU;
      const double an = An[o], ap = Ap[o], a0 = Am[o + r0], a1 = Am[o + r1], a2 = Am[o + r2], a3 = Am[o + r3];
      const double x = bm[k] * an, y = bn[k] * ap, z = bp[k] * an;
      acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, ap, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, y, acc[1], 0, 0, 0);
      acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, y, acc[2], 0, 0, 0);
      acc[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, z, acc[3], 0, 0, 0);
      acc[4] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, z, acc[4], 0, 0, 0);
      acc[5] = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, y, acc[5], 0, 0, 0);
      acc[6] = __builtin_amdgcn_mfma_f64_16x16x4f64(a3, y, acc[6], 0, 0, 0);
      acc[7] = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, z, acc[7], 0, 0, 0);
      acc[8] = __builtin_amdgcn_mfma_f64_16x16x4f64(a3, z, acc[8], 0, 0, 0);
   }
#pragma unroll
   for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) part[wv][t][16 * ((lane >> 4) + 4 * j) + l] = acc[t][j];
   __syncthreads();
   // F1 along the threads: it is the fastest index of the output
   const int i = threadIdx.x & 15, j = threadIdx.x >> 4, u = 16 * ta + i, v = 16 * tb + j;
   if (u > c || v > c) return;
   const auto val = [&](int t, int row, int col) {
      const int e = 16 * row + col;
      return ((part[0][t][e] + part[1][t][e]) + part[2][t][e]) + part[3][t][e];
   };
   const double g = val(0, i, j);
   const size_t o = (size_t)s * nf * nf;
   const auto put = [&](int F1, int F2, double b, double fac) {
      const size_t q = o + (size_t)(F1 + c) + (size_t)nf * (F2 + c);
      if (bfm) bfm[q] = b;
      if (brm) brm[q] = b * fac;
   };
#pragma unroll
   for (int h = 0; h < 2; ++h) {                             // F1 + F2, then F1 - F2
      const int w = h ? i - j + 16 : i + j, F2 = h ? -v : v;
      double b = g;
      if (abs(u + F2) <= last) {
         b += val(1 + 4 * h + (w >> 4), w & 15, j);
         b += val(3 + 4 * h + (w >> 4), w & 15, i);
      }
      b *= 2.0;
      // both signs: H(-f) is the conjugate, the factor's real part the same
      const double fac = brm ? brm_factor(u * df, F2 * df, m, n, p, Mm, Km, Cm) : 0.0;
      put(u, F2, b, fac);
      put(-u, -F2, b, fac);
   }
}

// The same by the G values of the FP32 (PREC 1) and split-bf16x3 (2) kernels
// (bfm_point_mixed).  grid (ceil(nf*nf/256), nsel)
template <int PREC>
__global__ __launch_bounds__(256) void k_bisp_grid_sel(
   const double *__restrict__ U, long ldU, int rows, const double *__restrict__ pb, int K,
   int nm, int nf, int exact, double df, const int *__restrict__ sel,
   const double *__restrict__ Mm, const double *__restrict__ Km, const double *__restrict__ Cm,
   double *__restrict__ bfm, double *__restrict__ brm)
{
   const long npts = (long)nf * nf;
   const long pt = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (pt >= npts) return;
   const int c = (nf - 1) / 2;
   const int mnp = sel[blockIdx.y];
   const int m = mnp % nm, n = (mnp / nm) % nm, p = mnp / (nm * nm);
   const int F1 = (int)(pt % nf) - c, F2 = (int)(pt / nf) - c, F3 = F1 + F2;
   const int a3 = (exact || abs(F3) <= c) ? abs(F3) : -1;
   const double s = bfm_point_mixed<PREC>(U, ldU, rows, pb, K, m, n, p, abs(F1), abs(F2), a3);
   const size_t o = (size_t)blockIdx.y * npts + pt;
   if (bfm) bfm[o] = s;
   if (brm) brm[o] = s * brm_factor(F1 * df, F2 * df, m, n, p, Mm, Km, Cm);
}

// Lane-layout self test of v_mfma_f64_16x16x4f64 (one wave, 512 doubles out):
// out[t*64 + l] = row index seen by register t of lane l, out[256 + t*64 + l]
// = its column index (A = row index in column 0, B = column index in row 0).
__global__ void k_mfma_f64_layout(double *__restrict__ out)
{
   const int l = threadIdx.x;
   const bool k0 = (l >> 4) == 0;
   d4 z = (d4){0.0, 0.0, 0.0, 0.0};
   d4 rows = __builtin_amdgcn_mfma_f64_16x16x4f64(k0 ? (double)(l & 15) : 0.0, k0 ? 1.0 : 0.0, z, 0, 0, 0);
   d4 cols = __builtin_amdgcn_mfma_f64_16x16x4f64(k0 ? 1.0 : 0.0, k0 ? (double)(l & 15) : 0.0, z, 0, 0, 0);
#pragma unroll
   for (int t = 0; t < 4; ++t) {
      out[t * 64 + l] = rows[t];
      out[256 + t * 64 + l] = cols[t];
   }
}

// ---------------------------------------------------------------------------
// Sum over a point list of w_pt * B(m,n,p)(pt) [* FRF]: one thread per mode
// triple and chunk of points, one atomic per thread.  Used for point sets that
// are not a symmetric uniform grid (BsaCL computation frequencies).
// grid (ceil(nm3/256), nchunk).
// ---------------------------------------------------------------------------
// FRF weighting of given modal spectra (getRM_full_vect_cls_,
// functionsImpl.F90:1598-1738, and getRM_full_scalar_msh_, :1031-1115), in
// place, H_m(f) = 1 / (K_m - w^2 M_m + i w C_mm), w = 2 pi f:
//   kind 0: psd(n1, NM^2), column n + p NM: times Re[H_p(f1_i) conj H_n(f1_i)]
//   kind 1: bisp(n1, n2, NM^3), entry m + n NM + p NM^2 at (f1_i, f2_j):
//           times Re[H_m(f1_i) H_n(f2_j) conj H_p(f1_i + f2_j)]
//   kind 2: bisp(NM^3, n1) at the points (f1_q, f2_q): the same factor.
// grid (ceil(total/256)), block 256
// ---------------------------------------------------------------------------
// U[k*ldU + y*nu + u] = 0 for u >= u0 (n = K * nm * (nu - u0) values)
__global__ void k_zero_cols(double *__restrict__ U, long ldU, int nu, long u0, int nm, long n)
{
   const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (t >= n) return;
   const long w = nu - u0;
   const long u = u0 + t % w, y = (t / w) % nm, k = t / (w * nm);
   U[k * ldU + y * nu + u] = 0.0;
}

__device__ __forceinline__ double2 frf_at(double f, const double *Mm, const double *Km,
                                          const double *Cm, int m)
{
   const double w = 2.0 * M_PI * f;
   const double r = Km[m] - w * w * Mm[m], im = w * Cm[m], d = r * r + im * im;
   return make_double2(r / d, -im / d);
}

// FRF weighting in place (bsahip_frf_apply).  kind 0: (n1, E2) spectra at f1,
// column c = n + p NM times Re[H_p conj H_n] (diag: column m times |H_m|^2);
// kind 1: (n1, n2, E3) at (f1_i, f2_j); kind 2: (E3, n1) at (f1_q, f2_q); entry
// e = m + n NM + p NM^2 times Re[H_m(a) H_n(b) conj H_p(a+b)] (diag: e = m, all
// three modes m).  E2 = NM^2, E3 = NM^3, or NM both for the diagonal model.
__global__ void k_frf_apply(int kind, int diag, long n1, const double *__restrict__ f1, long n2,
                            const double *__restrict__ f2, int nm, const double *__restrict__ Mm,
                            const double *__restrict__ Km, const double *__restrict__ Cm,
                            long total, double *__restrict__ data)
{
   const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (t >= total) return;
   if (kind == 0) {
      const long i = t % n1, c = t / n1;
      const int n = diag ? (int)c : (int)(c % nm), p = diag ? (int)c : (int)(c / nm);
      const double2 hn = frf_at(f1[i], Mm, Km, Cm, n), hp = frf_at(f1[i], Mm, Km, Cm, p);
      data[t] *= hp.x * hn.x + hp.y * hn.y;
      return;
   }
   const long ne = diag ? (long)nm : (long)nm * nm * nm;
   double a, b;
   long e;
   if (kind == 1) {
      const long i = t % n1, j = (t / n1) % n2;
      e = t / (n1 * n2);
      a = f1[i];
      b = f2[j];
   } else {
      const long q = t / ne;
      e = t % ne;
      a = f1[q];
      b = f2[q];
   }
   int m, n, p;
   if (diag) {
      m = n = p = (int)e;
   } else {
      m = (int)(e % nm);
      n = (int)((e / nm) % nm);
      p = (int)(e / ((long)nm * nm));
   }
   data[t] *= re3(frf_at(a, Mm, Km, Cm, m), frf_at(b, Mm, Km, Cm, n), frf_at(a + b, Mm, Km, Cm, p));
}

// Diagonal-model modal PSD at points: psd[q nm + m] = sum_k pa(m,k)^2 S_k(f_q),
// S from the sqrt-PSD table sq (ntc, nu, nnl) at row iu[q] (getFM_diag_tnlm_*'s
// psd, functionsImpl.F90:1747-1970).
__global__ void k_diag_psd_points(const double *__restrict__ sq, int nu, int nnl, int kv,
                                  const double *__restrict__ pa, int K, int nm, int npts,
                                  const int *__restrict__ iu, double *__restrict__ psd)
{
   const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
   if (gid >= (long)npts * nm) return;
   const int q = (int)(gid / nm), m = (int)(gid % nm);
   const int u = iu[q];
   double s = 0.0;
   for (int k = 0; k < kv; ++k) {                      // rows k >= kv are padding
      const int c = k / nnl, n = k % nnl;
      const double r = sq[((size_t)c * nu + u) * nnl + n];
      const double a = pa[(size_t)m * K + k];
      s += a * a * r * r;
   }
   psd[gid] = s;
}

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_bfm_points_sum(
   const double *__restrict__ U, long ldU, int rows, const double *__restrict__ pb, int K,
   int nm, int npts, const int *__restrict__ i1, const int *__restrict__ i2,
   const int *__restrict__ i3, const double *__restrict__ f1s, const double *__restrict__ f2s,
   const double *__restrict__ wpt, const double *__restrict__ Mm, const double *__restrict__ Km,
   const double *__restrict__ Cm, int with_frf, double *__restrict__ out)
{
   const int nm3 = nm * nm * nm;
   const int mnp = blockIdx.x * blockDim.x + threadIdx.x;
   if (mnp >= nm3) return;
   const int m = mnp % nm, n = (mnp / nm) % nm, p = mnp / (nm * nm);
   const int per = (npts + gridDim.y - 1) / gridDim.y;
   const int p0 = blockIdx.y * per, p1 = min(npts, p0 + per);
   double acc = 0.0;
   for (int pt = p0; pt < p1; ++pt) {
      const int a1 = i1[pt], a2 = i2[pt], a3 = i3[pt];
      double s = 0.0;
      for (int k = 0; k < K; ++k) {
         const double *row = U + (size_t)k * ldU;
         const double An1 = row[(size_t)n * rows + a1], Ap2 = row[(size_t)p * rows + a2];
         double v = pb[(size_t)m * K + k] * An1 * Ap2;
         if (a3 >= 0) {
            const double Am3 = row[(size_t)m * rows + a3];
            v += pb[(size_t)n * K + k] * Am3 * Ap2 + pb[(size_t)p * K + k] * Am3 * An1;
         }
         s += v;
      }
      s *= 2.0 * wpt[pt];
      if (with_frf) {
         const double w1 = 2.0 * M_PI * f1s[pt], w2 = 2.0 * M_PI * f2s[pt], w3 = w1 + w2;
         double r, im, d;
         r = -(w1 * w1 * Mm[m]) + Km[m]; im = w1 * Cm[m]; d = r * r + im * im;
         const double2 h1 = make_double2(r / d, -im / d);
         r = -(w2 * w2 * Mm[n]) + Km[n]; im = w2 * Cm[n]; d = r * r + im * im;
         const double2 h2 = make_double2(r / d, -im / d);
         r = -(w3 * w3 * Mm[p]) + Km[p]; im = w3 * Cm[p]; d = r * r + im * im;
         const double2 h3 = make_double2(r / d, -im / d);
         s *= re3(h1, h2, h3);
      }
      acc += s;
   }
   atomicAdd(out + mnp, acc);
}
