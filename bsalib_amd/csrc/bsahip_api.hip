// C ABI of libbsahip.so (declarations and layouts: include/bsahip.h).
//
// Host side of the MI355X BFM path.  A plan holds one structure resident on
// the device (Psi per K index, ln rho, PSD parameters, modal data) and every
// buffer its Classic run needs; bsahip_plan_run is the per-step hot path
// (nodal PSD -> projection A(f) -> [bf16 split] -> G contraction with the
// plane epilogue -> modal PSD moments -> copy of the moments).  There is no
// CPU fallback: without a usable GPU every entry point returns BSAHIP_EDEVICE.
#include "kernels.hip"
#include "gemm.hip"
#include "pod.hip"
#include "diag.hip"
#include "../../include/bsahip.h"
#include "bsahip_internal.h"

#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <initializer_list>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg)
{
   g_err = msg;
   return code;
}

#define HIPC(x)                                                                              \
   do {                                                                                      \
      hipError_t e_ = (x);                                                                   \
      if (e_ != hipSuccess)                                                                  \
         return fail(BSAHIP_EDEVICE, std::string(#x) + ": " + hipGetErrorString(e_));       \
   } while (0)

#define CHK(x)                                                                               \
   do {                                                                                      \
      int r_ = (x);                                                                          \
      if (r_ != 0) return r_;                                                                \
   } while (0)

struct Bufs;
bool give_back(const Bufs *asking);

// Named, grow-only device buffers.  With an arena (set_arena), get() carves
// the buffers out of that fixed device region instead and never allocates.
struct Bufs {
   struct Buf {
      void *p = nullptr;
      size_t n = 0;
   };
   std::map<std::string, Buf> m;
   char *arena = nullptr;
   size_t arena_cap = 0, arena_used = 0;
   Bufs() = default;
   Bufs(const Bufs &) = delete;                              // owns its buffers
   ~Bufs() { release(); }
   void release()
   {
      if (!arena)
         for (auto &kv : m)
            if (kv.second.p) (void)hipFree(kv.second.p);
      m.clear();
      arena_used = 0;
   }
   void set_arena(void *base, size_t cap)
   {
      release();
      arena = static_cast<char *>(base);
      arena_cap = cap;
   }
   // gives single buffers back; nothing may be using them
   void drop(std::initializer_list<const char *> names)
   {
      if (arena) return;
      (void)hipDeviceSynchronize();
      for (const char *name : names) {
         const auto it = m.find(name);
         if (it == m.end()) continue;
         if (it->second.p) (void)hipFree(it->second.p);
         m.erase(it);
      }
   }
   size_t total() const
   {
      size_t n = 0;
      for (const auto &kv : m) n += kv.second.n;
      return n;
   }
   template <class T>
   int get(const char *name, size_t count, T **out)
   {
      Buf &b = m[name];
      const size_t bytes = std::max<size_t>(count * sizeof(T), 256);
      if (arena) {
         if (b.n < bytes) {
            const size_t need = (bytes + 255) / 256 * 256;
            if (arena_used + need > arena_cap)
               return fail(BSAHIP_EINVAL,
                           std::string("the problem needs more than the ") +
                              std::to_string(arena_cap >> 20) +
                              " MiB of static device scratch of this entry point (at buffer " + name +
                              "); use the allocating entry point");
            b.p = arena + arena_used;
            b.n = need;
            arena_used += need;
         }
         *out = static_cast<T *>(b.p);
         return 0;
      }
      if (b.n < bytes) {
         // work queued earlier may still read the old buffer
         if (b.p) {
            (void)hipDeviceSynchronize();
            (void)hipFree(b.p);
         }
         b.p = nullptr;
         b.n = 0;
         hipError_t e = hipMalloc(&b.p, bytes);
         if (e == hipErrorOutOfMemory && give_back(this)) {
            (void)hipGetLastError();
            e = hipMalloc(&b.p, bytes);
         }
         if (e != hipSuccess) {
            (void)hipGetLastError();             // or the next launch's check reports it
            b.p = nullptr;
            return fail(BSAHIP_ENOMEM, std::string("hipMalloc(") + name + ", " +
                                           std::to_string(bytes) + " B): " + hipGetErrorString(e));
         }
         b.n = bytes;
      }
      *out = static_cast<T *>(b.p);
      return 0;
   }
};

// Static device scratch of bsahip_classic_run_noalloc: every buffer of its
// run (problem tables, A table, split planes, FRF table, moment accumulators)
// is carved out of this array, so that entry point never allocates.  Each
// device holds its own copy, at the address hipGetSymbolAddress returns with
// that device current (kept in Ctx::scratch_dev); the name itself is a host
// stand-in and is never passed to a kernel or a copy.
#define BSAHIP_NOALLOC_SCRATCH_BYTES ((size_t)64 << 20)
#define BSAHIP_MAX_DEVICES 64
static __device__ __align__(256) unsigned char scratch[BSAHIP_NOALLOC_SCRATCH_BYTES];

struct Ctx {
   bool ready = false;
   int dev = 0;
   void *scratch_dev[BSAHIP_MAX_DEVICES] = {};   // device address of `scratch` per device
   hipStream_t s = nullptr;
   hipStream_t s2 = nullptr;             // side stream: modal PSD moments beside the G kernel
   hipEvent_t e0 = nullptr, e1 = nullptr, e2 = nullptr, e3 = nullptr;
   Bufs *bufs = nullptr;                 // scratch of the one-shot entry points
   Bufs *plan_bufs = nullptr;            // buffers kept for the plans of one call (PlanLoan)
   char *stage = nullptr;                // pinned host memory of Pack, then of Pull
   hipEvent_t es = nullptr;              // Pack's last copy out of it
   // load_problem's host tables, kept up to HOST_KEPT values each: fresh ones cost a page
   // fault every 4 KB
   std::vector<double> pa_t, pa_k, pb_k;
   std::vector<float> pb32;
   double last_ms = 0.0;
   int last_launches = 0;
   rocblas_handle blas = nullptr;        // created on first use (truncated POD)
   std::recursive_mutex mu;
};

Ctx g;

// Kept scratch freed for an owner of buffers that found no memory.  No call uses the
// one-shot scratch beside other buffers, and a plan on loan has taken its own out.
bool give_back(const Bufs *asking)
{
   bool any = false;
   for (Bufs *b : {g.bufs, g.plan_bufs}) {
      if (!b || b == asking || b->m.empty()) continue;
      if (!any) (void)hipDeviceSynchronize();
      b->release();
      any = true;
   }
   return any;
}

// Host arrays and device results of one call travel in few copies: a copy from or to
// pageable memory costs about 5 us up and 20 us down however small it is (13 uploads of a
// small problem 62 us, one of the same bytes out of pinned memory 12 us; 4 KB down 23 us,
// by pinned memory 12 us).  From about a megabyte on there is nothing to win (1.6 MB down
// 317 us either way: the page faults of the caller's array).
constexpr size_t STAGE_UP = (size_t)4 << 20, STAGE_DOWN = (size_t)512 << 10, PART_UP = STAGE_UP / 4;

// Uploads gathered into one device buffer (src null: room only).  The host arrays have to
// live until send(), which has read them when it returns.
struct Pack {
   struct Part {
      const void *src;
      size_t bytes, off;
      void **out;
   };
   std::vector<Part> parts;
   size_t n = 0;
   // every array starts where a buffer of its own would in an arena: at a multiple of 256
   void add(const void *src, size_t bytes, void **out)
   {
      parts.push_back({src, bytes, n, out});
      n += std::max<size_t>((bytes + 255) / 256 * 256, 256);
   }
   template <class T>
   void add(const std::vector<T> &h, T **out)
   {
      add(h.data(), h.size() * sizeof(T), reinterpret_cast<void **>(out));
   }
   int send(Bufs &B, const char *name)
   {
      char *dev;
      CHK(B.get(name, n, &dev));
      size_t lo = 0, hi = 0;                                 // staged, not yet sent
      bool direct = false;                                   // the caller's memory is read
      const auto flush = [&]() -> int {
         if (hi > lo) {
            HIPC(hipMemcpyAsync(dev + lo, g.stage, hi - lo, hipMemcpyHostToDevice, g.s));
            HIPC(hipEventRecord(g.es, g.s));
         }
         lo = hi;
         return 0;
      };
      for (const Part &p : parts) {
         if (p.out) *p.out = dev + p.off;
         if (!p.bytes || !p.src) continue;
         if (!g.stage || p.bytes > PART_UP) {
            CHK(flush());
            HIPC(hipMemcpyAsync(dev + p.off, p.src, p.bytes, hipMemcpyHostToDevice, g.s));
            lo = hi = p.off + p.bytes;
            direct = true;
            continue;
         }
         if (p.off + p.bytes - lo > STAGE_UP) CHK(flush());
         if (hi == lo) {
            HIPC(hipEventSynchronize(g.es));                 // an earlier copy may still read it
            lo = hi = p.off;
         }
         std::memcpy(g.stage + (p.off - lo), p.src, p.bytes);
         hi = p.off + p.bytes;
      }
      CHK(flush());
      // a copy out of pageable memory is over when it returns, one out of the caller's
      // pinned memory is not
      if (direct) HIPC(hipStreamSynchronize(g.s));
      parts.clear();
      n = 0;
      return 0;
   }
};

// Results brought to the host: finish() waits for the stream.
struct Pull {
   struct Seg {
      void *dst;
      const char *src;
      size_t bytes;
   };
   std::vector<Seg> segs;
   size_t n = 0;
   int add(void *dst, const void *src, size_t bytes)
   {
      if (!dst || !bytes) return 0;
      if (!g.stage || n + bytes > STAGE_DOWN) {
         HIPC(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g.s));
         return 0;
      }
      segs.push_back({dst, static_cast<const char *>(src), bytes});
      n += bytes;
      return 0;
   }
   int finish()
   {
      char *stage = g.stage + STAGE_UP;
      size_t at = 0;
      for (size_t i = 0, j; i < segs.size(); i = j) {        // neighbours on the device in one copy
         size_t len = segs[i].bytes;
         for (j = i + 1; j < segs.size() && segs[j].src == segs[i].src + len; ++j) len += segs[j].bytes;
         HIPC(hipMemcpyAsync(stage + at, segs[i].src, len, hipMemcpyDeviceToHost, g.s));
         at += len;
      }
      HIPC(hipStreamSynchronize(g.s));
      at = 0;
      for (const Seg &q : segs) {
         std::memcpy(q.dst, stage + at, q.bytes);
         at += q.bytes;
      }
      segs.clear();
      n = 0;
      return 0;
   }
};

template <class T>
int upload(Bufs &B, const char *name, const std::vector<T> &h, T **out)
{
   CHK(B.get(name, h.size(), out));
   if (!h.empty())
      HIPC(hipMemcpyAsync(*out, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, g.s));
   return 0;
}

int fill(double *p, size_t n, double v)
{
   if (n == 0) return 0;
   const int blocks = (int)std::min<size_t>((n + 255) / 256, 65536);
   k_fill<<<blocks, 256, 0, g.s>>>(p, n, v);
   HIPC(hipGetLastError());
   return 0;
}

int ensure_init()
{
   if (g.ready) return 0;
   return bsahip_init(0) == 0 ? 0 : BSAHIP_EDEVICE;
}

inline int round_up(int a, int b) { return (a + b - 1) / b * b; }

int validate(const bsahip_problem *p)
{
   if (!p) return fail(BSAHIP_EINVAL, "problem pointer is NULL");
   if (p->nn <= 0 || p->nnl <= 0 || p->nm <= 0 || p->ntc <= 0 || p->ntc > 3 || p->nwz <= 0)
      return fail(BSAHIP_EINVAL, "invalid sizes (nn, nnl, nm, ntc in 1..3, nwz must be > 0)");
   if (p->nnl > p->nn) return fail(BSAHIP_EINVAL, "nnl > nn");
   if (p->nm > 256) return fail(BSAHIP_EUNSUPPORTED, "more than 256 modes");
   if (p->ndegw < 6) return fail(BSAHIP_EINVAL, "ndegw must be >= 6 (3 linear + 3 quadratic)");
   if ((long)p->ncorr_rows != ((long)p->nn * p->nn + p->nn) / 2)
      return fail(BSAHIP_EINVAL, "ncorr_rows must equal (nn*nn+nn)/2");
   if (!p->n_load || !p->tc || !p->psi || !p->nod_corr || !p->u_node || !p->wz_node ||
       !p->turb_scales || !p->turb_std || !p->Mm || !p->Km || !p->Cm)
      return fail(BSAHIP_EINVAL, "a required problem array is NULL");
   if (p->psd_id == 3 && !p->u_mean_ref) return fail(BSAHIP_EINVAL, "psd_id 3 needs u_mean_ref");
   if (!(p->psd_id == 1 || p->psd_id == 2 || p->psd_id == 3 || p->psd_id == 5))
      return fail(BSAHIP_EINVAL, "psd_id must be 1, 2, 3 or 5");
   for (int a = 0; a < p->nnl; ++a)
      if (p->n_load[a] < 1 || p->n_load[a] > p->nn) return fail(BSAHIP_EINVAL, "n_load out of range");
   for (int c = 0; c < p->ntc; ++c)
      if (p->tc[c] < 1 || p->tc[c] > 3) return fail(BSAHIP_EINVAL, "tc must be in 1..3");
   for (int a = 0; a < p->nn; ++a)
      if (p->wz_node[a] < 1 || p->wz_node[a] > p->nwz) return fail(BSAHIP_EINVAL, "wz_node out of range");
   return 0;
}

// Device-resident description of one structure.
struct Prob {
   // K rows: component c, loaded node i at k = c*nnlp + i (nnlp = nnl), the
   // kv = ntc*nnl valid rows padded with zero rows to a multiple of the K chunk
   int nn = 0, nnl = 0, nnlp = 0, nm = 0, ntc = 0, K = 0, kv = 0, pulsation = 1;
   double *pa_t = nullptr;   // [tc][m][nnl]
   double *pa_k = nullptr;   // [m][K]
   double *pb_k = nullptr;   // [m][K]
   float *pb32 = nullptr;    // [m][K]
   double *lnr = nullptr;    // [tc][nnl(j)][nnl(i)]
   double *prm = nullptr;    // [tc][nnl][4]
   int *formula = nullptr;   // [tc]
   double *Mm = nullptr, *Km = nullptr, *Cm = nullptr;
   // truncated POD of S(f) in the point tables (0/0: none, direct projection)
   int pod_nmodes = 0;
   double pod_lim = 0.0;
};

// psd_mode 0: reference Classic/Mesher semantics (evalPSD per component);
// psd_mode 1: BsaCL semantics (u formula for every component, zone 1, rho clamped).
constexpr size_t HOST_KEPT = (size_t)1 << 18;

// more: arrays of the caller that go up with the problem's; coh false: no coherence table
// (D.lnr null), for callers that do not project.
int load_problem(const bsahip_problem *p, int psd_mode, Bufs &B, Prob &D, Pack *more = nullptr,
                 bool coh = true)
{
   CHK(validate(p));
   D.nn = p->nn;
   D.nnl = p->nnl;
   D.nm = p->nm;
   D.ntc = p->ntc;
   D.nnlp = p->nnl;
   D.kv = D.ntc * D.nnl;
   D.K = round_up(D.kv, KC);
   D.pulsation = p->pulsation;
   const int nm = D.nm, nnl = D.nnl, K = D.K;
   // only the truncated POD reads Psi_a by components
   const bool pod = p->pod_nmodes != 0 || p->pod_trunc_lim != 0.0;
   const size_t npt = (size_t)D.ntc * nm * nnl, npk = (size_t)nm * K;
   std::vector<double> &pa_t = g.pa_t, &pa_k = g.pa_k, &pb_k = g.pb_k;
   std::vector<float> &pb32 = g.pb32;
   pa_t.resize(pod ? npt : 0);
   pa_k.assign(npk, 0.0);
   pb_k.assign(npk, 0.0);
   for (int c = 0; c < D.ntc; ++c) {
      const int t = p->tc[c];
      for (int i = 0; i < nnl; ++i)
         for (int m = 0; m < nm; ++m) {
            const double a = p->psi[m + (size_t)nm * (i + (size_t)nnl * (t - 1))];
            const double b = p->psi[m + (size_t)nm * (i + (size_t)nnl * (t + 2))];
            if (pod) pa_t[((size_t)c * nm + m) * nnl + i] = a;
            pa_k[(size_t)m * K + (size_t)c * D.nnlp + i] = a;
            pb_k[(size_t)m * K + (size_t)c * D.nnlp + i] = b;
         }
   }
   pb32.assign(pb_k.begin(), pb_k.end());
   // coherence columns actually read (nod_corr_(:, tc), or column 1 for all)
   std::vector<int> col(D.ntc);
   for (int c = 0; c < D.ntc; ++c)
      col[c] = (p->corr_col_mode == 1 || psd_mode == 1) ? 0 : p->tc[c] - 1;
   std::vector<int> ucol = col;
   std::sort(ucol.begin(), ucol.end());
   ucol.erase(std::unique(ucol.begin(), ucol.end()), ucol.end());
   std::vector<int> colmap(D.ntc);
   for (int c = 0; c < D.ntc; ++c)
      colmap[c] = (int)(std::lower_bound(ucol.begin(), ucol.end(), col[c]) - ucol.begin());
   // the table itself when they are its first ones, in order
   std::vector<double> corr;
   const double *corr_h = p->nod_corr;
   const size_t ncorr = coh ? ucol.size() * (size_t)p->ncorr_rows : 0;
   if (coh && ucol.back() != (int)ucol.size() - 1) {
      corr.resize(ncorr);
      for (size_t k = 0; k < ucol.size(); ++k)
         std::memcpy(corr.data() + k * p->ncorr_rows, p->nod_corr + (size_t)ucol[k] * p->ncorr_rows,
                     sizeof(double) * p->ncorr_rows);
      corr_h = corr.data();
   }
   std::vector<int> nl(p->n_load, p->n_load + nnl);
   std::vector<double> prm((size_t)D.ntc * nnl * 4, 0.0);
   std::vector<int> formula(D.ntc, 0);
   for (int c = 0; c < D.ntc; ++c) {
      const int t = p->tc[c];
      int f = 0;
      if (psd_mode == 1) f = (p->psd_id == 5) ? 5 : (p->psd_id == 1 ? 1 : 0);
      else if (p->psd_id == 1) f = (t == 1) ? 1 : 2;
      else f = (p->psd_id == 2) ? 0 : p->psd_id;
      formula[c] = f;
      for (int i = 0; i < nnl; ++i) {
         const int node = p->n_load[i] - 1;
         const int wz = (psd_mode == 1) ? 0 : p->wz_node[node] - 1;
         // L(component, direction 1, zone): von Karman u reads component 1
         // (WindPSDImpl.F90:167), the other formulas component tc.
         const int lc = (psd_mode == 0 && f == 1) ? 1 : t;
         double *q = prm.data() + ((size_t)c * nnl + i) * 4;
         q[0] = p->turb_scales[(lc - 1) + 9 * (size_t)wz];
         q[1] = p->turb_std[(t - 1) + 3 * (size_t)wz];
         q[2] = p->u_node[node];
         q[3] = p->u_mean_ref ? p->u_mean_ref[wz] : 1.0;
      }
   }
   std::vector<double> Mm(p->Mm, p->Mm + nm), Km(p->Km, p->Km + nm), Cm(p->Cm, p->Cm + nm);
   double *dcorr;
   int *dcol, *dnl;
   Pack own, &pk = more ? *more : own;
   // room for Psi_a by components in any case: a problem needs the same scratch with a POD
   pk.add(pod ? pa_t.data() : nullptr, npt * sizeof(double), reinterpret_cast<void **>(&D.pa_t));
   pk.add(pa_k, &D.pa_k);
   pk.add(pb_k, &D.pb_k);
   pk.add(pb32, &D.pb32);
   pk.add(colmap, &dcol);
   pk.add(nl, &dnl);
   pk.add(prm, &D.prm);
   pk.add(formula, &D.formula);
   pk.add(Mm, &D.Mm);
   pk.add(Km, &D.Km);
   pk.add(Cm, &D.Cm);
   if (coh) pk.add(corr_h, ncorr * sizeof(double), reinterpret_cast<void **>(&dcorr));
   CHK(pk.send(B, "problem"));
   if (npk > HOST_KEPT) {
      for (auto *v : {&pa_t, &pa_k, &pb_k}) std::vector<double>().swap(*v);
      std::vector<float>().swap(pb32);
   }
   if (!coh) return 0;
   CHK(B.get("lnr", (size_t)D.ntc * nnl * nnl, &D.lnr));
   dim3 gl((nnl + 255) / 256, nnl, D.ntc);
   k_lnrho<<<gl, 256, 0, g.s>>>(dcorr, p->ncorr_rows, dcol, dnl, nnl, p->nn,
                                psd_mode == 1 ? 2.2250738585072014e-308 : 0.0, D.lnr);
   HIPC(hipGetLastError());
   return 0;
}

// Truncated POD for the point paths (pod_nmodes / pod_trunc_lim of the problem).
int set_pod(const bsahip_problem *p, Prob &D)
{
   D.pod_nmodes = 0;
   D.pod_lim = 0.0;
   if (p->pod_nmodes < 0 || !std::isfinite(p->pod_trunc_lim) || p->pod_trunc_lim < 0.0)
      return fail(BSAHIP_EINVAL, "pod_nmodes must be >= 0 and pod_trunc_lim finite and >= 0");
   if (p->pod_nmodes == 0 && p->pod_trunc_lim == 0.0) return 0;
   if (p->corr_col_mode != 1)
      return fail(BSAHIP_EINVAL, "a truncated POD reads coherence column 1 (corr_col_mode must be 1)");
   D.pod_nmodes = p->pod_nmodes;
   D.pod_lim = p->pod_trunc_lim;
   return 0;
}

#define BLASC(x)                                                                             \
   do {                                                                                      \
      rocblas_status st_ = (x);                                                              \
      if (st_ != rocblas_status_success)                                                     \
         return fail(BSAHIP_EDEVICE, std::string(#x) + ": " + rocblas_status_to_string(st_)); \
   } while (0)

// rocBLAS / rocSOLVER handle on the library stream, created on first use.
int blas_handle()
{
   if (!g.blas) {
      BLASC(rocblas_create_handle(&g.blas));
      BLASC(rocblas_set_stream(g.blas, g.s));
   }
   return 0;
}

// C_b = alpha op(A_b) op(B_b) + beta C_b on the library stream (k_dgemm_sb).
int dgemm_sb(int transa, int transb, int M, int N, int K, double alpha, const double *A, long lda,
             long sA, const double *B, long ldb, long sB, double beta, double *C, long ldc,
             long sC, int batch)
{
   if (M <= 0 || N <= 0 || batch <= 0) return 0;
   if (batch > 65535) return fail(BSAHIP_EUNSUPPORTED, "GEMM batch above 65535");
   dim3 gr((unsigned)((M + 63) / 64), (unsigned)((N + 63) / 64), (unsigned)batch);
   k_dgemm_sb<<<gr, 256, 0, g.s>>>(transa, transb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C,
                                    ldc, sC);
   HIPC(hipGetLastError());
   return 0;
}

// A_K(y, i; f) = (Psi_a V) diag(w) V^T for the truncated POD of S(f) (see
// pod.hip), written into the table layout of k_project.  sq: sqrt(S_i) at fl.
int pod_project(Bufs &B, const Prob &D, const double *sq, const double *fl, int nfl,
                int rows_per_mode, double *U, long ldU)
{
   CHK(blas_handle());
   const int n = D.nnl, nm = D.nm;
   const size_t nn2 = (size_t)n * n, mn = (size_t)nm * n;
   const long total = (long)D.ntc * nfl;
   // at most 2^28 doubles (2 GiB) of matrices and 65535 matrices per chunk
   const long cap = std::max<long>(1, std::min<long>({total, 65535L, (1L << 28) / (long)nn2}));
   double *S, *lam, *E, *w, *T, *A;
   int *info, *kept;
   CHK(B.get("pod_S", (size_t)cap * nn2, &S));
   CHK(B.get("pod_lam", (size_t)cap * n, &lam));
   CHK(B.get("pod_E", (size_t)cap * n, &E));
   CHK(B.get("pod_w", (size_t)cap * n, &w));
   CHK(B.get("pod_T", (size_t)cap * mn, &T));
   CHK(B.get("pod_A", (size_t)cap * mn, &A));
   CHK(B.get("pod_info", (size_t)cap, &info));
   CHK(B.get("pod_kept", (size_t)cap, &kept));
   std::vector<int> hk((size_t)cap);
   for (long b0 = 0; b0 < total; b0 += cap) {
      const int nb = (int)std::min<long>(cap, total - b0);
      k_pod_smat<<<dim3((unsigned)((nn2 + 255) / 256), nb), 256, 0, g.s>>>(D.lnr, sq, fl, nfl, n, b0, S);
      HIPC(hipGetLastError());
      BLASC(rocsolver_dsyevd_strided_batched(g.blas, rocblas_evect_original, rocblas_fill_lower, n, S,
                                             n, (rocblas_stride)nn2, lam, n, E, n, info, nb));
      k_pod_weights<<<nb, 64, 0, g.s>>>(lam, info, n, D.pod_nmodes, D.pod_lim, w, kept);
      HIPC(hipGetLastError());
      // T = Psi_a(c) V: Psi_a(c) is pa_t[c] read as the column-major n x nm
      // matrix P, so T = P^T V; one strided batch per component in the chunk
      for (long bb = b0; bb < b0 + nb;) {
         const int c = (int)(bb / nfl);
         const long be = std::min<long>(b0 + nb, (long)(c + 1) * nfl);
         CHK(dgemm_sb(1, 0, nm, n, n, 1.0, D.pa_t + (size_t)c * mn, n, 0, S + (size_t)(bb - b0) * nn2,
                      n, (long)nn2, 0.0, T + (size_t)(bb - b0) * mn, nm, (long)mn, (int)(be - bb)));
         bb = be;
      }
      k_pod_scale<<<dim3((unsigned)((mn + 255) / 256), nb), 256, 0, g.s>>>(T, w, nm, n);
      HIPC(hipGetLastError());
      CHK(dgemm_sb(0, 1, nm, n, n, 1.0, T, nm, (long)mn, S, n, (long)nn2, 0.0, A, nm, (long)mn, nb));
      k_pod_scatter<<<dim3((unsigned)((mn + 255) / 256), nb), 256, 0, g.s>>>(A, nm, n, nfl, b0, D.nnlp,
                                                                         rows_per_mode, U, ldU);
      HIPC(hipGetLastError());
      HIPC(hipMemcpyAsync(hk.data(), kept, (size_t)nb * sizeof(int), hipMemcpyDeviceToHost, g.s));
      HIPC(hipStreamSynchronize(g.s));
      for (int b = 0; b < nb; ++b)
         if (hk[b] < 0) return fail(BSAHIP_EDEVICE, "POD eigendecomposition of S(f) did not converge");
   }
   return 0;
}

// Neighbouring frequencies per wave of k_project: 8 (64-byte stores, loads of ln rho
// and Psi_a shared by eight) while that still leaves 2 waves per SIMD of the chip, fewer
// for small tables, where latency counts; at most 4 beyond 16 modes (accumulators).
int project_group(long ncoltile, int nfl, int planes, int mt)
{
   int F = mt == 1 ? 8 : (mt == 2 ? 4 : 2);
   while (F > 1 && ncoltile * ((nfl + F - 1) / F) * planes < 2048) F /= 2;
   return F;
}

// Projection tables at the |f| list fl (nodal sqrt-PSDs sq): k_project in the layout
// U[k*ldU + y*rows + q], or (vlay) the Mesher's U[(q*K + k)*ldU + y] with every padding
// entry written.  proj_args leaves nqg to the caller, who knows F.
ProjArgs proj_args(const Prob &D, const double *sq, const double *fl, int nfl, int rows, double *U,
                   long ldU, bool vlay)
{
   ProjArgs P;
   P.pak = D.pa_k;
   P.lnr = D.lnr;
   P.sq = sq;
   P.fabs_list = fl;
   P.nfl = nfl;
   P.nnl = D.nnl;
   P.nm = D.nm;
   P.nnlp = D.nnlp;
   P.K = D.K;
   P.row_stride = rows;
   P.ntc = D.ntc;
   // the point layout's tiles cover its padding rows
   P.ncoltile = ((vlay ? D.nnl + D.K - D.kv : D.nnl) + 15) / 16;
   P.U = U;
   P.ldU = ldU;
   P.nqg = 0;
   return P;
}

// 16-mode tiles of a projection wave, chunks of modes (grid z)
int proj_mt(int nm) { return nm <= 64 ? (nm + 15) / 16 : 4; }
int proj_chunks(int nm) { return (nm + 63) / 64; }

// f(integral constants MT, F) for the tiles mt and the group F of project_group
template <class Fn>
void proj_dispatch(int mt, int F, Fn f)
{
   auto g = [&](auto MT, auto FM) {
      constexpr int M = decltype(MT)::value, X = decltype(FM)::value;
      if (F >= X) f(MT, FM);
      else if (F >= 4 && X > 4) f(MT, std::integral_constant<int, X < 4 ? X : 4>());
      else if (F >= 2 && X > 2) f(MT, std::integral_constant<int, X < 2 ? X : 2>());
      else f(MT, std::integral_constant<int, 1>());
      (void)M;
   };
   if (mt <= 1) g(std::integral_constant<int, 1>(), std::integral_constant<int, 8>());
   else if (mt <= 2) g(std::integral_constant<int, 2>(), std::integral_constant<int, 4>());
   else if (mt <= 3) g(std::integral_constant<int, 3>(), std::integral_constant<int, 2>());
   else g(std::integral_constant<int, 4>(), std::integral_constant<int, 2>());
}

int project(const Prob &D, const double *sq, const double *fl, int nfl, int rows, double *U, long ldU,
            bool vlay)
{
   ProjArgs P = proj_args(D, sq, fl, nfl, rows, U, ldU, vlay);
   const int mt = proj_mt(D.nm), nch = proj_chunks(D.nm);
   const int F = project_group(P.ncoltile, nfl, D.ntc * nch, mt);
   P.nqg = (nfl + F - 1) / F;
   const dim3 gr((unsigned)((P.nqg * P.ncoltile + 3) / 4), (unsigned)D.ntc, (unsigned)nch);
   proj_dispatch(mt, F, [&](auto MT, auto FF) {
      constexpr int M = decltype(MT)::value, X = decltype(FF)::value;
      if (vlay) k_project<M, X, true><<<gr, 256, 0, g.s>>>(P);
      else k_project<M, X, false><<<gr, 256, 0, g.s>>>(P);
   });
   HIPC(hipGetLastError());
   return 0;
}

// Nodal sqrt-PSD table [tc][nfl][nnl] at the |f| list fl
int psd_table(Bufs &B, const Prob &D, const double *fl, int nfl, double **sq)
{
   if (nfl > 65535) return fail(BSAHIP_EUNSUPPORTED, "more than 65535 distinct frequencies in one table");
   CHK(B.get("sq", (size_t)D.ntc * nfl * D.nnl, sq));
   dim3 gp((D.nnl + 63) / 64, nfl, D.ntc);
   k_psd_sqrt<<<gp, 64, 0, g.s>>>(fl, nfl, D.prm, D.formula, D.nnl, D.ntc, D.pulsation, *sq);
   HIPC(hipGetLastError());
   return 0;
}

// The entries of a table U[K][ldU] that no projection writes: the K rows from kv on and
// the columns from nm*rows on.
int zero_padding(const Prob &D, int rows, double *U, long ldU)
{
   CHK(fill(U + (size_t)D.kv * ldU, (size_t)(D.K - D.kv) * ldU, 0.0));
   const long c0 = (long)D.nm * rows, n = (ldU - c0) * D.kv;
   if (n > 0) {
      k_zero_tail<<<(unsigned)((n + 255) / 256), 256, 0, g.s>>>(U, ldU, c0, n);
      HIPC(hipGetLastError());
   }
   return 0;
}

// A table on a list of nfl = rows_per_mode |f| values (device array fl): U[K][ldU], rows
// y*rows_per_mode + q, everything outside the valid rows and columns zero (padded: the
// caller's U already holds those zeros).
int build_table(Bufs &B, const Prob &D, const double *fl, int nfl, int rows_per_mode, double *U,
                long ldU, bool padded = false)
{
   double *sq;
   CHK(psd_table(B, D, fl, nfl, &sq));
   if (!padded) CHK(zero_padding(D, rows_per_mode, U, ldU));
   if (D.pod_nmodes > 0 || D.pod_lim > 0.0)
      return pod_project(B, D, sq, fl, nfl, rows_per_mode, U, ldU);
   return project(D, sq, fl, nfl, rows_per_mode, U, ldU, false);
}

int launch_frf(const Prob &D, int nft, double df, double2 *H)
{
   dim3 gh((nft + 255) / 256, D.nm);
   k_frf_table<<<gh, 256, 0, g.s>>>(D.Mm, D.Km, D.Cm, D.nm, nft, df, H);
   HIPC(hipGetLastError());
   return 0;
}

// FP64 bispectra of nsel triples (device list sel; null: triple s of all) on the grid of
// nf points per axis from the table U of nu rows per mode
void bisp_grid_f64(const Prob &D, const double *U, long ldU, int nu, int nf, double df, long nsel,
                   const int *sel, double *bfm, double *brm)
{
   const unsigned nt = (unsigned)((nf - 1) / 2 + 16) / 16;
   const long ny = std::min(nsel, 65535L);
   k_bisp_grid_f64<<<dim3(nt * nt, (unsigned)ny, (unsigned)((nsel + ny - 1) / ny)), 256, 0, g.s>>>(
      U, ldU, nu, D.pb_k, D.K, D.nm, nf, df, nsel, sel, D.Mm, D.Km, D.Cm, bfm, brm);
}

int check_flags(int32_t flags, bool grid, bool allow_mixed)
{
   const int prec = flags & BSAHIP_PREC_MASK;
   const int quad = (flags & BSAHIP_QUAD_MASK) >> 4;
   if (prec != BSAHIP_PREC_FP64 &&
       !(allow_mixed && (prec == BSAHIP_PREC_BF16X3 || prec == BSAHIP_PREC_FP32)))
      return fail(BSAHIP_EUNSUPPORTED, "precision not available in this entry point");
   if (grid && quad > 2) return fail(BSAHIP_EINVAL, "unknown quadrature rule");
   return 0;
}

// Distinct |f| over f1, f2, f1+f2 of a point list and the index maps into it.
void point_tables(int npts, const double *fi, const double *fj, std::vector<double> &uq,
                  std::vector<int> &i1, std::vector<int> &i2, std::vector<int> &i3)
{
   // distinct values by open addressing on their bits, then sorted: a sort of all 3 npts
   // and a search for each took 3/5 of a Mesher's refinement (40 nodes, 3 modes: 10.4 ms of
   // zones built, refined and integrated, now 4.3)
   size_t cap = 16;
   int shift = 60;
   while (cap < 6 * (size_t)npts) {
      cap *= 2;
      --shift;
   }
   std::vector<int> table(cap, -1), id(3 * (size_t)npts);
   std::vector<double> keys;
   const auto look = [&](double v) {
      v = std::fabs(v);
      uint64_t bits;
      std::memcpy(&bits, &v, sizeof bits);
      for (size_t h = (size_t)((bits * 0x9E3779B97F4A7C15ull) >> shift);; h = (h + 1) & (cap - 1)) {
         const int k = table[h];
         if (k < 0) {
            table[h] = (int)keys.size();
            keys.push_back(v);
            return table[h];
         }
         if (std::memcmp(&keys[k], &bits, sizeof bits) == 0) return k;
      }
   };
   for (int q = 0; q < npts; ++q) {
      id[3 * (size_t)q] = look(fi[q]);
      id[3 * (size_t)q + 1] = look(fj[q]);
      id[3 * (size_t)q + 2] = look(fi[q] + fj[q]);
   }
   std::vector<int> order(keys.size()), rank(keys.size());
   for (size_t k = 0; k < order.size(); ++k) order[k] = (int)k;
   std::sort(order.begin(), order.end(), [&](int a, int b) { return keys[a] < keys[b]; });
   uq.resize(keys.size());
   for (size_t k = 0; k < order.size(); ++k) {
      uq[k] = keys[order[k]];
      rank[order[k]] = (int)k;
   }
   i1.resize(npts);
   i2.resize(npts);
   i3.resize(npts);
   for (int q = 0; q < npts; ++q) {
      i1[q] = rank[id[3 * (size_t)q]];
      i2[q] = rank[id[3 * (size_t)q + 1]];
      i3[q] = rank[id[3 * (size_t)q + 2]];
   }
}

}  // namespace

// A Classic run of one structure on one grid, resident on the device.
struct bsahip_plan {
   Bufs B;
   Prob D;
   int32_t flags = 0, prec = 0;
   int nh = 0, nf = 0, nu = 0, nhp = 0, rows = 0, ntile = 0, nft = 0;
   int f64_br = 0, f64_bc = 0;           // FP64 wave tile in blocks of 16 (0: f64_shape's)
   long ldU = 0;
   double df = 0.0, d = 0.0;
   double *fl = nullptr, *U = nullptr, *m3 = nullptr, *m2 = nullptr;
   int copies = 1;                       // of m3 (gsym_copies)
   double2 *H = nullptr;
   float *UR = nullptr;
   uint16_t *Ch = nullptr, *Cl = nullptr;
   double last_ms = 0.0;
   // fixed-order summation (BSAHIP_DETERMINISTIC): per-flush slots of the G
   // epilogue, the slot list of every m3 entry, per-block m2 partials
   double *slots = nullptr, *m2part = nullptr;
   long *det_off = nullptr, *det_idx = nullptr, *det_slot0 = nullptr;
};

namespace {

// Host pair index of a tile pair as the kernels' pair_from_index: t ->
// (R, Q), R <= Q, t = Q (Q + 1) / 2 + R.
void host_pair(long t, int &R, int &Q)
{
   long q = (long)((std::sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
   while ((q + 1) * (q + 2) / 2 <= t) ++q;
   while (q * (q + 1) / 2 > t) --q;
   Q = (int)q;
   R = (int)(t - q * (q + 1) / 2);
}

// FP64 wave tile (blocks of 16 rows x columns) for nm modes x and nm (diagonal model: one)
// runs of `per` table rows: the larger tiles load and scale less per MFMA, the smaller ones
// give more waves.  Measured in us at (rows, nm, K), tiles 1x1 / 2x2 / 4x2: full model
// (193, 1, 608) 27 / 39 / 61, (195, 3, 32) 16 / 21 / 31, (390, 5, 608) 44 / 51 / -,
// (516, 4, 2016) 165 / 115 / -, (771, 3, 608) 72 / 50 / 76, (780, 12, 608) 239 / 135 / 161,
// (3084, 12, 608) 3146 / 1481 / 1391, (2910, 30, 608) 7131 / 3394 / 3189; diagonal model
// (257, 4, 608) 33 / 39 / -, (65, 60, 128) 11 / 14 / -, (257, 20, 3008) 297 / 243 / -.
// `least` is the count of waves from which 2x2 is taken.  In both models 1x1 is the faster
// while all its waves run at once, up to some 400 to 512 of 2x2; the full model takes 2x2
// from 32 on all the same, since it is the batches' tile: a structure's moments are then
// sums of the same contributions in a batch as alone.  A wave sums for each pair of modes
// it meets, one after the other: tiles that would meet more than some four keep to 2x2,
// (270, 30, 608) 148 / 153 / 235, (990, 30, 608) 924 / 476 / 503, (900, 100, 32)
// 2431 / 2090 / 2548.
constexpr long F64_LARGE = 48;

void f64_shape(long rows, long per, int nm, double least, int &br, int &bc)
{
   const auto waves = [&](int r, int c) { return (double)rows * (double)rows / (512.0 * r * c) * nm; };
   if (per >= F64_LARGE && waves(4, 2) >= 4096.0) {
      br = 4;
      bc = 2;
   } else if (waves(2, 2) >= least) {
      br = bc = 2;
   } else {
      br = bc = 1;
   }
}

// Copies of the third moments that the FP64 contraction adds into (gsym_f64_wave): about one
// for every COPY_ADDS additions to an entry, three for each tile of a mode pair, while all of
// them stay within COPY_MAX doubles and the last sum, serial per entry, within COPY_MOST.
// One where a fixed arena keeps the scratch it had or the sums have an order of their own,
// and for the other precisions, whose own error is 1e-7.
constexpr long COPY_ADDS = 4, COPY_MAX = 1L << 20, COPY_MOST = 256;

int gsym_copies(const bsahip_plan *P)
{
   if (P->prec != BSAHIP_PREC_FP64 || (P->flags & (BSAHIP_NO_BISP | BSAHIP_DETERMINISTIC)) || P->B.arena) return 1;
   const long n = 2L * P->D.nm * P->D.nm * P->D.nm;
   const long adds = 3L * (P->nhp / (16 * P->f64_br) + 1) * (P->nhp / (16 * P->f64_bc) + 1);
   return (int)std::max(1L, std::min({adds / COPY_ADDS, COPY_MAX / n, COPY_MOST}));
}

constexpr double F64_LEAST = 32.0, F64_LEAST_DIAG = 384.0;

// workgroups of one G launch
long plan_items(const bsahip_plan *P)
{
   const long t = P->prec == BSAHIP_PREC_FP64 ? f64_tiles(P->rows, P->f64_br, P->f64_bc)
                                              : (long)P->ntile * (P->ntile + 1) / 2;
   return t * P->D.nm;
}

// Slot lists of the fixed-order mode: the flushes of every wave of every G
// item in the order epi_wave makes them (kernels.hip), each with its m3 entries
// in the order of epi_flush (m3f entries 0 .. NM^3-1, m3r entries NM^3 ..
// 2 NM^3-1).  off (2 NM^3 + 1) and idx list, per entry, its slots in ascending
// order, slot0 the first slot of each wave.
void det_slot_lists(const bsahip_plan *P, std::vector<long> &off, std::vector<long> &idx,
                    std::vector<long> &slot0)
{
   const int nm = P->D.nm, nhp = P->nhp;
   const bool f64 = (P->prec == BSAHIP_PREC_FP64);
   const int BR = f64 ? P->f64_br : 4, BC = f64 ? P->f64_bc : 4;
   const long nm3 = (long)nm * nm * nm, nent = 2 * nm3, nitems = plan_items(P);
   auto walk = [&](auto wave, auto flush) {
      for (long lid = 0; lid < nitems; ++lid) {
         const int x = (int)(lid % nm);
         int R = 0, Q = 0;
         if (!f64) host_pair(lid / nm, R, Q);
         for (int w = 0; w < 4; ++w) {
            int rw0 = R * T2 + (w >> 1) * 64, cw0 = Q * T2 + (w & 1) * 64;
            bool diag = (R == Q);
            if (f64) {                     // gsym_f64_wave
               const long i = 4 * (lid / nm) + w;
               if (i >= f64_waves(P->rows, BR, BC)) continue;
               int c;
               f64_tile(i, (P->rows + 16 * BC - 1) / (16 * BC), BR / BC, R, c);
               rw0 = R * 16 * BR;
               cw0 = c * 16 * BC;
               diag = c < (R + 1) * (BR / BC);
            }
            const int y0 = rw0 / nhp, y1 = std::min((rw0 + 16 * BR - 1) / nhp, nm - 1);
            const int z0 = cw0 / nhp, z1 = std::min((cw0 + 16 * BC - 1) / nhp, nm - 1);
            wave(lid * 4 + w);
            for (int y = y0; y <= y1; ++y)
               for (int z = z0; z <= z1; ++z) flush(x, y, z, diag);
         }
      }
   };
   auto entries = [&](int x, int y, int z, bool diag, auto entry) {
      const long xyz = x + (long)nm * y + (long)nm * nm * z, yxz = y + (long)nm * x + (long)nm * nm * z,
                 yzx = y + (long)nm * z + (long)nm * nm * x, xzy = x + (long)nm * z + (long)nm * nm * y,
                 zxy = z + (long)nm * x + (long)nm * nm * y, zyx = z + (long)nm * y + (long)nm * nm * x;
      const long v[12] = {xyz, nm3 + xyz, yxz, nm3 + yxz, yzx, nm3 + yzx,
                          xzy, nm3 + xzy, zxy, nm3 + zxy, zyx, nm3 + zyx};
      const int n = epi_count(f64, x, y, z, diag);
      for (int t = 0; t < n; ++t) entry(v[t]);
   };
   off.assign(nent + 1, 0);
   slot0.assign(nitems * 4, 0);
   long slot = 0;
   walk([&](long w) { slot0[w] = slot; },
        [&](int x, int y, int z, bool diag) {
           entries(x, y, z, diag, [&](long e) {
              ++off[e + 1];
              ++slot;
           });
        });
   for (long e = 0; e < nent; ++e) off[e + 1] += off[e];
   idx.assign(slot, 0);
   std::vector<long> pos(off.begin(), off.end() - 1);
   slot = 0;
   walk([](long) {},
        [&](int x, int y, int z, bool diag) {
           entries(x, y, z, diag, [&](long e) { idx[pos[e]++] = slot++; });
        });
}

int plan_setup(bsahip_plan *P, const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
               int psd_mode)
{
   CHK(check_flags(flags, true, true));
   if (nfh < 2 || !(df > 0.0)) return fail(BSAHIP_EINVAL, "need nfh >= 2 and df > 0");
   if (flags & BSAHIP_ONLY_DIAG)
      return fail(BSAHIP_EUNSUPPORTED, "the ONLY_DIAG model runs through bsahip_classic_run");
   CHK(validate(p));
   const long nul = (flags & BSAHIP_SUM_EXACT) ? 2L * nfh - 1 : nfh;
   const int tile = (flags & BSAHIP_PREC_MASK) == BSAHIP_PREC_FP64 ? 64 : T2;
   const long nt = (p->nm * nul + tile - 1) / tile;
   // one workgroup of 256 threads per (tile pair, mode): the launch's global
   // size must fit 32 bits.  Before any table of that size is made.
   if ((double)nt * (nt + 1) / 2 * p->nm * 256.0 > 4294967295.0)
      return fail(BSAHIP_EUNSUPPORTED, "grid too large for one launch: (tile pairs x modes) x 256 "
                                       "threads exceeds 2^32; use a coarser grid or fewer modes");
   const int nu = (int)nul;
   std::vector<double> fl(nu);
   for (int u = 0; u < nu; ++u) fl[u] = (double)u * df;
   Pack pk;
   pk.add(fl, &P->fl);
   CHK(load_problem(p, psd_mode, P->B, P->D, &pk));
   P->flags = flags;
   P->prec = flags & BSAHIP_PREC_MASK;
   P->df = df;
   P->nh = nfh;
   P->nf = 2 * nfh - 1;
   P->nu = nu;                                                  // rows of A per mode
   // rows of consecutive modes packed (no padding to 16 per mode): a 16-row
   // block may span two modes, and the epilogue masks the other mode's rows
   P->nhp = P->nu;
   P->rows = P->D.nm * P->nhp;
   P->ntile = (int)nt;
   if (P->f64_br == 0) f64_shape(P->rows, P->nhp, P->D.nm, F64_LEAST, P->f64_br, P->f64_bc);
   P->ldU = (long)round_up(P->rows, T2);
   P->nft = 2 * P->nu - 1;
   P->d = p->pulsation ? df * 2.0 * M_PI : df;
   CHK(P->B.get("U", (size_t)P->D.K * P->ldU, &P->U));
   CHK(zero_padding(P->D, P->nhp, P->U, P->ldU));      // the runs write the valid entries only
   CHK(P->B.get("H", (size_t)P->D.nm * P->nft, &P->H));
   const size_t nm3 = (size_t)P->D.nm * P->D.nm * P->D.nm, nm2 = (size_t)P->D.nm * P->D.nm;
   P->copies = gsym_copies(P);
   // one buffer: the results come back in one copy
   CHK(P->B.get("moments", 3 * nm2 + 2 * nm3 * P->copies, &P->m2));
   P->m3 = P->m2 + 3 * nm2;
   if ((flags & BSAHIP_DETERMINISTIC) && !(flags & BSAHIP_NO_BISP)) {
      std::vector<long> off, idx, slot0;
      det_slot_lists(P, off, idx, slot0);
      CHK(upload(P->B, "det_off", off, &P->det_off));
      CHK(upload(P->B, "det_idx", idx, &P->det_idx));
      CHK(upload(P->B, "det_slot0", slot0, &P->det_slot0));
      CHK(P->B.get("det_slots", idx.size(), &P->slots));
   }
   if ((flags & BSAHIP_DETERMINISTIC) && !(flags & BSAHIP_NO_PSD))
      CHK(P->B.get("m2part", (size_t)((P->nh + 63) / 64) * 3 * nm2, &P->m2part));
   if (P->prec != BSAHIP_PREC_FP64) {
      const size_t n = (size_t)P->ldU * P->D.K;
      CHK(P->B.get("UR32", n, &P->UR));
      if (P->prec == BSAHIP_PREC_BF16X3) {
         CHK(P->B.get("UCh", n, &P->Ch));
         CHK(P->B.get("UCl", n, &P->Cl));
      }
   }
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

// Phases of a plan run (all stream-ordered on g.s, no host synchronisation):
// tables (PSD, projection, FRF, split planes), G contraction, modal PSD moments.
int plan_prepare(bsahip_plan *P)
{
   Prob &D = P->D;
   const size_t nm3 = (size_t)D.nm * D.nm * D.nm;
   CHK(build_table(P->B, D, P->fl, P->nu, P->nhp, P->U, P->ldU, true));
   CHK(launch_frf(D, P->nft, P->df, P->H));
   if (!(P->flags & BSAHIP_NO_BISP)) {
      CHK(fill(P->m3, 2 * nm3 * P->copies, 0.0));
      if (P->prec != BSAHIP_PREC_FP64) {
         dim3 gs((unsigned)(P->ldU / 32), (unsigned)((D.K + 31) / 32));
         k_split_table<<<gs, 256, 0, g.s>>>(P->U, P->ldU, D.K, (int)P->ldU, D.K, P->UR, P->Ch, P->Cl);
         HIPC(hipGetLastError());
      }
   }
   return 0;
}

void plan_args(const bsahip_plan *P, GsymArgs &a, GsymArgs16 &b16)
{
   const Prob &D = P->D;
   const size_t nm3 = (size_t)D.nm * D.nm * D.nm;
   a.U = P->U;
   a.ldU = P->ldU;
   a.pb = D.pb_k;
   a.K = D.K;
   a.nm = D.nm;
   a.nhp = P->nhp;
   a.nh = P->nh;
   a.nu = P->nu;
   a.H = P->H;
   a.nft = P->nft;
   a.d2 = P->d * P->d;
   a.rule = (P->flags & BSAHIP_QUAD_MASK) >> 4;
   a.epi_plain = (P->flags & BSAHIP_EPI_GENERIC) ? 1 : 0;
   a.m3f = P->m3;
   a.m3r = P->m3 + nm3;
   a.slots = P->slots;
   a.slot0 = P->det_slot0;
   a.copies = P->copies;
   b16.UR = P->UR;
   b16.UCh = reinterpret_cast<const uint4 *>(P->Ch);
   b16.UCl = reinterpret_cast<const uint4 *>(P->Cl);
   b16.pb32 = D.pb32;
   b16.ldk = D.K;
}

int plan_gsym(bsahip_plan *P)
{
   GsymArgs a;
   GsymArgs16 b16;
   plan_args(P, a, b16);
   const long nwg = plan_items(P);
   if (P->prec == BSAHIP_PREC_BF16X3)
      k_gsym_bf16x3<<<dim3((unsigned)nwg), 256, 0, g.s>>>(a, b16);
   else if (P->prec == BSAHIP_PREC_FP32)
      k_gsym_f32<<<dim3((unsigned)nwg), 256, 0, g.s>>>(a, b16);
   else if (P->f64_br == 4)
      k_gsym_f64<4, 2><<<dim3((unsigned)nwg), 256, 0, g.s>>>(a);
   else if (P->f64_br == 2)
      k_gsym_f64<2, 2><<<dim3((unsigned)nwg), 256, 0, g.s>>>(a);
   else
      k_gsym_f64<1, 1><<<dim3((unsigned)nwg), 256, 0, g.s>>>(a);
   HIPC(hipGetLastError());
   if (P->slots) {
      // fixed order: every m3 entry sums its slots in ascending order
      const long n = 2 * (long)P->D.nm * P->D.nm * P->D.nm;
      k_sum_lists<<<(unsigned)((n + 255) / 256), 256, 0, g.s>>>(P->slots, P->det_off, P->det_idx, n,
                                                                P->m3);
      HIPC(hipGetLastError());
   }
   return 0;
}

// K rows per slice of k_m2 so that some `want` blocks run (each at least 64 rows, 4 MFMA
// steps per wave: shorter slices are all reduction); want 1: no slices
int m2_slice(int want, long blocks, int K)
{
   const int n = (int)std::max<long>(1, std::min<long>(want / std::max<long>(1, blocks), K / 64));
   return round_up((K + n - 1) / n, 16);
}

M2Args plan_m2_args(const bsahip_plan *P)
{
   const Prob &D = P->D;
   const size_t nm2 = (size_t)D.nm * D.nm;
   M2Args a;
   a.U = P->U;
   a.ldU = P->ldU;
   a.pa = D.pa_k;
   a.K = D.K;
   a.nm = D.nm;
   a.nhp = P->nhp;
   a.nh = P->nh;
   a.H = P->H;
   a.nft = P->nft;
   a.d = P->d;
   a.om_step = 2.0 * M_PI * P->df;
   a.m2f = P->m2;
   a.m2r = P->m2 + nm2;
   a.m2o = P->m2 + 2 * nm2;
   a.m2part = P->m2part;
   a.diag = 0;
   a.kper = m2_slice(P->m2part ? 1 : 1024, (long)D.nm * ((P->nh + 63) / 64), D.K);
   return a;
}

int plan_m2(bsahip_plan *P)
{
   Prob &D = P->D;
   const size_t nm2 = (size_t)D.nm * D.nm;
   const int nby = (P->nh + 63) / 64, mt = D.nm <= 16 ? 1 : 2;
   if (!P->m2part) CHK(fill(P->m2, 3 * nm2, 0.0));
   const M2Args a = plan_m2_args(P);
   const dim3 gm((unsigned)D.nm, (unsigned)nby,
                 (unsigned)(((D.nm + 16 * mt - 1) / (16 * mt)) * ((D.K + a.kper - 1) / a.kper)));
   if (mt == 1) k_m2<1><<<gm, 256, 0, g.s>>>(a);
   else k_m2<2><<<gm, 256, 0, g.s>>>(a);
   HIPC(hipGetLastError());
   if (P->m2part) {
      const long n = 3 * (long)nm2;
      k_sum_fixed<<<(unsigned)((n + 255) / 256), 256, 0, g.s>>>(P->m2part, nby, n, n, P->m2);
      HIPC(hipGetLastError());
   }
   return 0;
}

int plan_copyout(bsahip_plan *P, double *m2mf, double *m2mr, double *m2o2mr, double *m3mf,
                 double *m3mr)
{
   const Prob &D = P->D;
   const size_t nm3 = (size_t)D.nm * D.nm * D.nm, nm2 = (size_t)D.nm * D.nm;
   Pull pl;
   if (!(P->flags & BSAHIP_NO_PSD)) {
      CHK(pl.add(m2mf, P->m2, nm2 * sizeof(double)));
      CHK(pl.add(m2mr, P->m2 + nm2, nm2 * sizeof(double)));
      CHK(pl.add(m2o2mr, P->m2 + 2 * nm2, nm2 * sizeof(double)));
   }
   if (P->copies > 1 && (m3mf || m3mr)) {
      k_sum_copies<<<(unsigned)((2 * nm3 + 63) / 64), 64, 0, g.s>>>(P->m3, (long)(2 * nm3), P->copies);
      HIPC(hipGetLastError());
   }
   if (!(P->flags & BSAHIP_NO_BISP)) {
      CHK(pl.add(m3mf, P->m3, nm3 * sizeof(double)));
      CHK(pl.add(m3mr, P->m3 + nm3, nm3 * sizeof(double)));
   }
   return pl.finish();
}

int plan_exec(bsahip_plan *P, double *m2mf, double *m2mr, double *m2o2mr, double *m3mf, double *m3mr)
{
   const bool want_psd = !(P->flags & BSAHIP_NO_PSD);
   const bool want_bisp = !(P->flags & BSAHIP_NO_BISP);
   CHK(plan_prepare(P));
   P->last_ms = 0.0;
   // the modal PSD moments only read the tables: they run on the side stream
   // while the G kernel runs, and the copy-out waits for both
   const bool side = want_psd && want_bisp;
   if (side) {
      HIPC(hipEventRecord(g.e2, g.s));
      HIPC(hipStreamWaitEvent(g.s2, g.e2, 0));
      hipStream_t main_s = g.s;
      g.s = g.s2;
      const int rc = plan_m2(P);
      g.s = main_s;
      CHK(rc);
      HIPC(hipEventRecord(g.e3, g.s2));
   }
   if (want_bisp) {
      HIPC(hipEventRecord(g.e0, g.s));
      CHK(plan_gsym(P));
      HIPC(hipEventRecord(g.e1, g.s));
   }
   if (want_psd && !side) CHK(plan_m2(P));
   if (side) HIPC(hipStreamWaitEvent(g.s, g.e3, 0));
   CHK(plan_copyout(P, m2mf, m2mr, m2o2mr, m3mf, m3mr));
   g.last_ms = 0.0;
   g.last_launches = 0;
   if (want_bisp) {
      float ms = 0.f;
      HIPC(hipEventElapsedTime(&ms, g.e0, g.e1));
      P->last_ms = ms;
      g.last_ms = ms;
      g.last_launches = 1;
   }
   return 0;
}

Bufs &oneshot_bufs()
{
   if (!g.bufs) g.bufs = new Bufs();
   return *g.bufs;
}

// A plan of one call works in buffers kept for the next one: allocated and freed by each
// call, 151 nodes, 9 modes, 101 frequencies took 296 us, so 248.  Beyond KEPT bytes they are
// freed with the plan; the other entry points' scratch is not touched.
struct PlanLoan {
   static constexpr size_t KEPT = (size_t)256 << 20;
   Bufs &B;
   explicit PlanLoan(Bufs &b) : B(b)
   {
      if (!g.plan_bufs) g.plan_bufs = new Bufs();
      B.m.swap(g.plan_bufs->m);
   }
   ~PlanLoan()
   {
      if (B.total() > KEPT) B.release();
      B.m.swap(g.plan_bufs->m);
   }
};

}  // namespace

extern "C" {

int bsahip_version(void) { return 110; }

const char *bsahip_last_error(void) { return g_err.c_str(); }

int bsahip_init(int device)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (g.ready) return 0;
   int n = 0;
   hipError_t e = hipGetDeviceCount(&n);
   if (e != hipSuccess || n <= 0)
      return fail(BSAHIP_EDEVICE, std::string("no HIP device available: ") + hipGetErrorString(e));
   if (device < 0 || device >= n) return fail(BSAHIP_EINVAL, "device index out of range");
   if (device >= BSAHIP_MAX_DEVICES) return fail(BSAHIP_EUNSUPPORTED, "device index above 63");
   HIPC(hipSetDevice(device));
   if (!g.scratch_dev[device]) {
      void *sp = nullptr;
      HIPC(hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch)));
      if (!sp) return fail(BSAHIP_EDEVICE, "hipGetSymbolAddress(scratch) returned NULL");
      g.scratch_dev[device] = sp;
   }
   HIPC(hipStreamCreateWithFlags(&g.s, hipStreamNonBlocking));
   HIPC(hipStreamCreateWithFlags(&g.s2, hipStreamNonBlocking));
   HIPC(hipEventCreate(&g.e0));
   HIPC(hipEventCreate(&g.e1));
   HIPC(hipEventCreateWithFlags(&g.e2, hipEventDisableTiming));
   HIPC(hipEventCreateWithFlags(&g.e3, hipEventDisableTiming));
   HIPC(hipEventCreateWithFlags(&g.es, hipEventDisableTiming));
   if (hipHostMalloc(reinterpret_cast<void **>(&g.stage), STAGE_UP + STAGE_DOWN, hipHostMallocDefault) !=
       hipSuccess) {
      g.stage = nullptr;                                     // copies from pageable memory instead
      (void)hipGetLastError();
   }
   g.dev = device;
   g.ready = true;
   return 0;
}

int bsahip_finalise(void)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (!g.ready) return 0;
   (void)hipStreamSynchronize(g.s);
   delete g.bufs;
   delete g.plan_bufs;
   g.bufs = g.plan_bufs = nullptr;
   if (g.blas) (void)rocblas_destroy_handle(g.blas);
   g.blas = nullptr;
   (void)hipStreamSynchronize(g.s2);
   (void)hipEventDestroy(g.e0);
   (void)hipEventDestroy(g.e1);
   (void)hipEventDestroy(g.e2);
   (void)hipEventDestroy(g.e3);
   (void)hipEventDestroy(g.es);
   if (g.stage) (void)hipHostFree(g.stage);
   g.stage = nullptr;
   (void)hipStreamDestroy(g.s2);
   (void)hipStreamDestroy(g.s);
   g.ready = false;
   return 0;
}

int bsahip_last_kernel_time(double *ms, int32_t *launches)
{
   if (ms) *ms = g.last_ms;
   if (launches) *launches = g.last_launches;
   return 0;
}

int bsahip_plan_create(const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
                       bsahip_plan **out)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (!out) return fail(BSAHIP_EINVAL, "NULL plan output");
   *out = nullptr;
   CHK(ensure_init());
   std::unique_ptr<bsahip_plan> P(new bsahip_plan());
   CHK(plan_setup(P.get(), p, nfh, df, flags, 0));
   *out = P.release();
   return 0;
}

int bsahip_plan_run(bsahip_plan *plan, double *m2mf, double *m2mr, double *m2o2mr,
                    double *m3mf, double *m3mr)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (!plan) return fail(BSAHIP_EINVAL, "NULL plan");
   CHK(ensure_init());
   return plan_exec(plan, m2mf, m2mr, m2o2mr, m3mf, m3mr);
}

int bsahip_plan_destroy(bsahip_plan *plan)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (plan) {
      if (g.ready) (void)hipStreamSynchronize(g.s);
      delete plan;
   }
   return 0;
}

int bsahip_classic_run(const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
                       double *m2mf, double *m2mr, double *m2o2mr, double *m3mf, double *m3mr)
{
   return bsahip__classic_moments(p, nfh, df, flags, 0, m2mf, m2mr, m2o2mr, m3mf, m3mr);
}

int bsahip_classic_run_noalloc(const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
                               double *m2mf, double *m2mr, double *m2o2mr, double *m3mf,
                               double *m3mr)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (!g.ready) return fail(BSAHIP_ESTATE, "call bsahip_init first (it sets up the static scratch)");
   if (flags & BSAHIP_ONLY_DIAG)
      return fail(BSAHIP_EUNSUPPORTED, "the ONLY_DIAG model runs through bsahip_classic_run");
   void *base = g.scratch_dev[g.dev];
   if (!base) return fail(BSAHIP_ESTATE, "no static scratch on the current device");
   // the plan's buffers come from the static array; the plan is never
   // destroyed with buffers of its own (Bufs in arena mode frees nothing)
   bsahip_plan P;
   P.B.set_arena(base, BSAHIP_NOALLOC_SCRATCH_BYTES);
   CHK(plan_setup(&P, p, nfh, df, flags, 0));
   return plan_exec(&P, m2mf, m2mr, m2o2mr, m3mf, m3mr);
}

}  // extern "C"

namespace {

// Tables of the ONLY_DIAG model on the half grid u df, u < nh: X (K, ldX) the nodal
// PSDs, W and A2 (nm, K) the weights Psi_q Psi_l^2 and Psi_l^2, H (nm, 2 nh - 1) the FRFs.
struct DiagTab {
   double *X, *W, *A2;
   double2 *H;
   long ldX;
};

int diag_tables(Bufs &B, const Prob &D, const double *dfl, int nh, double df, long ldX, DiagTab &T)
{
   const int nft = 2 * nh - 1, nm = D.nm, K = D.K;
   T.ldX = ldX;
   CHK(B.get("dg_X", (size_t)K * T.ldX, &T.X));
   CHK(B.get("dg_W", (size_t)nm * K, &T.W));
   CHK(B.get("dg_A2", (size_t)nm * K, &T.A2));
   CHK(B.get("dg_H", (size_t)nm * nft, &T.H));
   k_diag_psd<<<dim3((unsigned)((T.ldX + 63) / 64), (unsigned)K), 64, 0, g.s>>>(
      dfl, nh, D.nnl, D.kv, D.prm, D.formula, D.pulsation, T.ldX, T.X);
   HIPC(hipGetLastError());
   const long n = (long)nm * K;
   k_diag_weights<<<(unsigned)((n + 255) / 256), 256, 0, g.s>>>(D.pa_k, D.pb_k, n, T.W, T.A2);
   HIPC(hipGetLastError());
   return launch_frf(D, nft, df, T.H);
}

// T (nm, nh, nh) = X W_m X^T per mode, for the bispectra
int diag_products(Bufs &B, const Prob &D, int nh, const DiagTab &T, double **out)
{
   double *Y;
   const int nm = D.nm, K = D.K;
   CHK(B.get("dg_Y", (size_t)nm * K * T.ldX, &Y));
   CHK(B.get("dg_T", (size_t)nm * nh * nh, out));
   k_diag_scaled<<<dim3((unsigned)((T.ldX + 63) / 64), (unsigned)K, (unsigned)nm), 64, 0, g.s>>>(
      T.X, T.ldX, T.W, K, Y);
   HIPC(hipGetLastError());
   return dgemm_sb(0, 1, nh, nh, K, 1.0, T.X, T.ldX, 0, Y, T.ldX, (long)K * T.ldX, 0.0, *out, nh,
                   (long)nh * nh, nm);
}

// The ONLY_DIAG Classic model (diag.hip): outputs have NM entries each.
int classic_diag(const bsahip_problem *p, int32_t nfh, double df, int32_t flags, double *m2mf,
                 double *m2mr, double *m2o2mr, double *m3mf, double *m3mr)
{
   if ((flags & BSAHIP_PREC_MASK) != BSAHIP_PREC_FP64)
      return fail(BSAHIP_EUNSUPPORTED, "the ONLY_DIAG model runs in FP64");
   if (nfh < 2 || !(df > 0.0)) return fail(BSAHIP_EINVAL, "need nfh >= 2 and df > 0");
   CHK(validate(p));
   const bool psd = !(flags & BSAHIP_NO_PSD), bisp = !(flags & BSAHIP_NO_BISP);
   int br, bc;
   f64_shape(nfh, nfh, p->nm, F64_LEAST_DIAG, br, bc);
   // (2^20 frequencies: past any accepted plane, within the 32 bits of f64_waves)
   const long items = nfh > 1 << 20 ? LONG_MAX : f64_tiles(nfh, br, bc) * p->nm;
   if (bisp && items > 0xffffffL)
      return fail(BSAHIP_EUNSUPPORTED, "grid too large for one launch: use a coarser grid or fewer modes");
   Bufs &B = oneshot_bufs();
   Prob D;
   Pack pk;
   std::vector<double> fl(nfh);
   for (int u = 0; u < nfh; ++u) fl[u] = (double)u * df;
   double *dfl;
   pk.add(fl, &dfl);
   CHK(load_problem(p, 0, B, D, &pk, false));
   const int nh = nfh, nft = 2 * nh - 1, nm = D.nm, K = D.K;
   const double d = p->pulsation ? df * 2.0 * M_PI : df;
   DiagTab T;
   double *mom;
   CHK(diag_tables(B, D, dfl, nh, df, (nh + 127L) / 128 * 128, T));      // whole tiles
   CHK(B.get("dg_mom", 5 * (size_t)nm, &mom));
   CHK(fill(mom, 5 * (size_t)nm, 0.0));
   double *m2f = mom, *m2r = mom + nm, *m2o = mom + 2 * nm, *m3f = mom + 3 * nm, *m3r = mom + 4 * nm;
   if (psd) {
      // beside the third moments, on the side stream
      HIPC(hipEventRecord(g.e2, g.s));
      HIPC(hipStreamWaitEvent(g.s2, g.e2, 0));
      const int nby = (nh + 63) / 64, mt = nm <= 16 ? 1 : 2, np = (nm + 16 * mt - 1) / (16 * mt);
      M2Args a{T.X, T.ldX, T.A2, K, nm, 0, nh, T.H, nft, d, 2.0 * M_PI * df, m2f, m2r, m2o, nullptr, 1,
               m2_slice(256, (long)nby * np, K)};
      const dim3 gm(1, (unsigned)nby, (unsigned)(np * ((K + a.kper - 1) / a.kper)));
      if (mt == 1) k_m2<1><<<gm, 256, 0, g.s2>>>(a);
      else k_m2<2><<<gm, 256, 0, g.s2>>>(a);
      HIPC(hipGetLastError());
      HIPC(hipEventRecord(g.e3, g.s2));
   }
   if (bisp) {
      GsymArgs a{};
      a.U = T.X;
      a.ldU = T.ldX;
      a.pb = T.W;
      a.K = K;
      a.nm = 1;
      a.nhp = a.nh = a.nu = nh;
      a.H = T.H;
      a.nft = nft;
      a.d2 = d * d;
      a.rule = (flags & BSAHIP_QUAD_MASK) >> 4;
      a.epi_plain = (flags & BSAHIP_EPI_GENERIC) ? 1 : 0;
      a.m3f = m3f;
      a.m3r = m3r;
      if (br == 4) k_gsym_diag<4, 2><<<(unsigned)items, 256, 0, g.s>>>(a, nm);
      else if (br == 2) k_gsym_diag<2, 2><<<(unsigned)items, 256, 0, g.s>>>(a, nm);
      else k_gsym_diag<1, 1><<<(unsigned)items, 256, 0, g.s>>>(a, nm);
      HIPC(hipGetLastError());
   }
   if (psd) HIPC(hipStreamWaitEvent(g.s, g.e3, 0));
   Pull pl;
   const size_t nb = nm * sizeof(double);
   if (psd) {
      CHK(pl.add(m2mf, m2f, nb));
      CHK(pl.add(m2mr, m2r, nb));
      CHK(pl.add(m2o2mr, m2o, nb));
   }
   if (bisp) {
      CHK(pl.add(m3mf, m3f, nb));
      CHK(pl.add(m3mr, m3r, nb));
   }
   return pl.finish();
}

}  // namespace

extern "C" {

int bsahip__classic_moments(const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
                            int32_t psd_mode, double *m2mf, double *m2mr, double *m2o2mr,
                            double *m3mf, double *m3mr)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (flags & BSAHIP_ONLY_DIAG) {
      if (psd_mode != 0) return fail(BSAHIP_EUNSUPPORTED, "the ONLY_DIAG model has no BsaCL form");
      if (flags & BSAHIP_DETERMINISTIC)
         return fail(BSAHIP_EUNSUPPORTED, "the ONLY_DIAG model has no fixed-order mode");
      const int rc = classic_diag(p, nfh, df, flags, m2mf, m2mr, m2o2mr, m3mf, m3mr);
      if (rc != 0) (void)hipDeviceSynchronize();             // nothing in flight on the one-shot scratch
      return rc;
   }
   bsahip_plan P;
   PlanLoan loan(P.B);
   int rc = plan_setup(&P, p, nfh, df, flags, psd_mode);
   if (rc == 0) rc = plan_exec(&P, m2mf, m2mr, m2o2mr, m3mf, m3mr);
   if (rc != 0) (void)hipDeviceSynchronize();                // nothing in flight on kept buffers
   return rc;
}

int bsahip__points_sum(const bsahip_problem *p, int32_t npts, const double *fi, const double *fj,
                       const double *w, int32_t psd_mode, int32_t with_frf, double *m3)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (npts < 0 || (npts > 0 && (!fi || !fj || !w || !m3)))
      return fail(BSAHIP_EINVAL, "npts < 0 or NULL point/weight/output arrays");
   Bufs &B = oneshot_bufs();
   Prob D;
   CHK(load_problem(p, psd_mode, B, D));
   const size_t nm3 = (size_t)D.nm * D.nm * D.nm;
   if (npts == 0) {
      std::fill(m3, m3 + nm3, 0.0);
      return 0;
   }
   std::vector<double> uq;
   std::vector<int> i1, i2, i3;
   point_tables(npts, fi, fj, uq, i1, i2, i3);
   const int nu = (int)uq.size();
   const long ldU = (long)D.nm * nu;
   double *fl, *U;
   CHK(upload(B, "fl", uq, &fl));
   CHK(B.get("U", (size_t)D.K * ldU, &U));
   CHK(build_table(B, D, fl, nu, nu, U, ldU));
   std::vector<double> f1(fi, fi + npts), f2(fj, fj + npts), ww(w, w + npts);
   int *di1, *di2, *di3;
   double *df1, *df2, *dw, *out;
   CHK(upload(B, "i1", i1, &di1));
   CHK(upload(B, "i2", i2, &di2));
   CHK(upload(B, "i3", i3, &di3));
   CHK(upload(B, "f1", f1, &df1));
   CHK(upload(B, "f2", f2, &df2));
   CHK(upload(B, "wpt", ww, &dw));
   CHK(B.get("m3sum", nm3, &out));
   CHK(fill(out, nm3, 0.0));
   const int nchunk = (int)std::min<long>(1024, std::max<long>(1, npts / 16));
   dim3 gs((unsigned)((nm3 + 255) / 256), nchunk);
   k_bfm_points_sum<<<gs, 256, 0, g.s>>>(U, ldU, nu, D.pb_k, D.K, D.nm, npts, di1, di2, di3,
                                         df1, df2, dw, D.Mm, D.Km, D.Cm, with_frf, out);
   HIPC(hipGetLastError());
   HIPC(hipMemcpyAsync(m3, out, nm3 * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

int bsahip_classic_spectra(const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
                           double *psd_f, double *psd_r, double *bfm, double *brm)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   CHK(check_flags(flags, true, false));
   if (flags & BSAHIP_ONLY_DIAG)
      return fail(BSAHIP_EUNSUPPORTED, "bsahip_classic_spectra is the full model; the diagonal model's "
                                       "spectra: bsahip_diag_psd_points, bsahip_classic_bispectra_sel");
   if (nfh < 2 || !(df > 0.0)) return fail(BSAHIP_EINVAL, "need nfh >= 2 and df > 0");
   Bufs &B = oneshot_bufs();
   Prob D;
   CHK(load_problem(p, 0, B, D));
   const int nh = nfh, nf = 2 * nh - 1, c = nh - 1;
   const bool exact = (flags & BSAHIP_SUM_EXACT) != 0;
   const int nu = exact ? nf : nh;
   const long ldU = (long)D.nm * nu;
   std::vector<double> fl(nu);
   for (int u = 0; u < nu; ++u) fl[u] = (double)u * df;
   double *dfl, *U;
   double2 *H;
   CHK(upload(B, "fl", fl, &dfl));
   CHK(B.get("U", (size_t)D.K * ldU, &U));
   CHK(build_table(B, D, dfl, nu, nu, U, ldU));
   CHK(B.get("H", (size_t)D.nm * nf, &H));
   CHK(launch_frf(D, nf, df, H));
   const size_t nm2 = (size_t)D.nm * D.nm, nm3 = nm2 * D.nm;
   if (psd_f || psd_r) {
      double *pf, *pr;
      CHK(B.get("psd_f", nm2 * nf, &pf));
      CHK(B.get("psd_r", nm2 * nf, &pr));
      dim3 gq((nf + 255) / 256, (unsigned)nm2);
      k_psd_grid<<<gq, 256, 0, g.s>>>(U, ldU, D.pa_k, D.K, D.nm, nu, nf, c, H, nf, pf, pr);
      HIPC(hipGetLastError());
      if (psd_f) HIPC(hipMemcpyAsync(psd_f, pf, nm2 * nf * sizeof(double), hipMemcpyDeviceToHost, g.s));
      if (psd_r) HIPC(hipMemcpyAsync(psd_r, pr, nm2 * nf * sizeof(double), hipMemcpyDeviceToHost, g.s));
   }
   if (bfm || brm) {
      const long npts = (long)nf * nf;
      double *ob, *orr;
      CHK(B.get("bfm_out", nm3 * npts, &ob));
      CHK(B.get("brm_out", nm3 * npts, &orr));
      if ((long)nm3 * npts > 0xffffff00L)
         return fail(BSAHIP_EUNSUPPORTED, "NF^2 * NM^3 exceeds 2^32 bispectrum values in one call");
      bisp_grid_f64(D, U, ldU, nu, nf, df, (long)nm3, nullptr, ob, orr);
      HIPC(hipGetLastError());
      if (bfm) HIPC(hipMemcpyAsync(bfm, ob, nm3 * npts * sizeof(double), hipMemcpyDeviceToHost, g.s));
      if (brm) HIPC(hipMemcpyAsync(brm, orr, nm3 * npts * sizeof(double), hipMemcpyDeviceToHost, g.s));
   }
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

int bsahip_classic_bispectra_sel(const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
                                 int32_t nsel, const int32_t *sel, double *bfm, double *brm)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   CHK(check_flags(flags, true, true));
   const int prec = flags & BSAHIP_PREC_MASK;
   if (nfh < 2 || !(df > 0.0)) return fail(BSAHIP_EINVAL, "need nfh >= 2 and df > 0");
   if (prec != BSAHIP_PREC_FP64 && (flags & BSAHIP_ONLY_DIAG))
      return fail(BSAHIP_EUNSUPPORTED, "the ONLY_DIAG model runs in FP64");
   if (nsel < 0 || nsel > 65535 || (nsel > 0 && !sel))
      return fail(BSAHIP_EINVAL, "nsel outside 0..65535 or NULL selection");
   const bool diag = (flags & BSAHIP_ONLY_DIAG) != 0, exact = (flags & BSAHIP_SUM_EXACT) != 0;
   if (diag && exact)
      return fail(BSAHIP_EUNSUPPORTED, "the ONLY_DIAG model pads S(f1+f2) with zeros (no SUM_EXACT)");
   if (nsel == 0 || (!bfm && !brm)) return 0;
   if (nfh > 46341) return fail(BSAHIP_EINVAL, "nfh too large for one selected bispectrum");
   Bufs &B = oneshot_bufs();
   Prob D;
   CHK(validate(p));
   const long ncol = diag ? p->nm : (long)p->nm * p->nm * p->nm;
   const int nh = nfh, nf = 2 * nh - 1, nu = exact ? nf : nh;
   std::vector<int> s0(nsel);
   std::vector<double> fl(nu);
   for (int u = 0; u < nu; ++u) fl[u] = (double)u * df;
   for (int s = 0; s < nsel; ++s) {
      if (sel[s] < 1 || sel[s] > ncol)
         return fail(BSAHIP_EINVAL, "selection index out of 1..NM^3 (1..NM with ONLY_DIAG)");
      s0[s] = sel[s] - 1;
   }
   const size_t npts = (size_t)nf * nf, nout = npts * (size_t)nsel;
   int *dsel;
   double *dfl, *ob = nullptr, *orr = nullptr;
   Pack pk;
   pk.add(s0, &dsel);
   pk.add(fl, &dfl);
   CHK(load_problem(p, 0, B, D, &pk, !diag));
   if (bfm) CHK(B.get("bisp_sel_f", nout, &ob));
   if (brm) CHK(B.get("bisp_sel_r", nout, &orr));
   const dim3 gs((unsigned)((npts + 255) / 256), (unsigned)nsel);
   if (diag) {
      DiagTab X;
      double *T;
      CHK(diag_tables(B, D, dfl, nh, df, nh, X));
      CHK(diag_products(B, D, nh, X, &T));
      k_diag_bisp_sel<<<gs, 256, 0, g.s>>>(T, nh, X.H, 2 * nh - 1, dsel, ob, orr);
   } else {
      const long ldU = (long)D.nm * nu;
      double *U;
      CHK(B.get("U", (size_t)D.K * ldU, &U));
      CHK(build_table(B, D, dfl, nu, nu, U, ldU));
#define LAUNCH_SEL(PR)                                                                        \
   k_bisp_grid_sel<PR><<<gs, 256, 0, g.s>>>(U, ldU, nu, D.pb_k, D.K, D.nm, nf, exact ? 1 : 0, df, \
                                            dsel, D.Mm, D.Km, D.Cm, ob, orr)
      if (prec == BSAHIP_PREC_FP32) LAUNCH_SEL(1);
      else if (prec == BSAHIP_PREC_BF16X3) LAUNCH_SEL(2);
      else bisp_grid_f64(D, U, ldU, nu, nf, df, nsel, dsel, ob, orr);
#undef LAUNCH_SEL
   }
   HIPC(hipGetLastError());
   if (bfm) HIPC(hipMemcpyAsync(bfm, ob, nout * sizeof(double), hipMemcpyDeviceToHost, g.s));
   if (brm) HIPC(hipMemcpyAsync(brm, orr, nout * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

}  // extern "C"

namespace {
int bfm_points_impl(const bsahip_problem *p, int32_t npts, const double *fi, const double *fj,
                    double *bfm, double *brm, double fmax, bool diag);
int diag_sq_table(Bufs &B, const Prob &D, const std::vector<double> &uq, double fmax, double **sq);
}  // namespace

extern "C" {

int bsahip_bfm_points(const bsahip_problem *p, int32_t npts, const double *fi, const double *fj,
                      int32_t flags, double *bfm, double *brm)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   CHK(check_flags(flags, false, false));
   if (flags & ~(BSAHIP_PREC_MASK | BSAHIP_ONLY_DIAG))
      return fail(BSAHIP_EINVAL, "bsahip_bfm_points takes BSAHIP_ONLY_DIAG and FP64 only");
   return bfm_points_impl(p, npts, fi, fj, bfm, brm, -1.0, (flags & BSAHIP_ONLY_DIAG) != 0);
}

int bsahip_bfm_points_cls(const bsahip_problem *p, int32_t nfh, double df, int32_t flags,
                          int32_t npts, const double *fi, const double *fj, double *bfm,
                          double *brm)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (nfh < 2 || !(df > 0.0)) return fail(BSAHIP_EINVAL, "need nfh >= 2 and df > 0");
   if (flags & ~BSAHIP_ONLY_DIAG)
      return fail(BSAHIP_EINVAL, "bsahip_bfm_points_cls takes BSAHIP_ONLY_DIAG only");
   return bfm_points_impl(p, npts, fi, fj, bfm, brm, (nfh - 1) * df,
                          (flags & BSAHIP_ONLY_DIAG) != 0);
}

int bsahip_diag_psd_points(const bsahip_problem *p, int32_t npts, const double *f, double *psd)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (npts < 0 || (npts > 0 && (!f || !psd))) return fail(BSAHIP_EINVAL, "npts < 0 or NULL arrays");
   if (npts == 0) return 0;
   Bufs &B = oneshot_bufs();
   Prob D;
   CHK(load_problem(p, 0, B, D, nullptr, false));
   std::vector<double> af(npts);
   for (int q = 0; q < npts; ++q) af[q] = std::fabs(f[q]);
   std::vector<double> uq(af);
   std::sort(uq.begin(), uq.end());
   uq.erase(std::unique(uq.begin(), uq.end()), uq.end());
   std::vector<int> iu(npts);
   for (int q = 0; q < npts; ++q)
      iu[q] = (int)(std::lower_bound(uq.begin(), uq.end(), af[q]) - uq.begin());
   double *sq, *out;
   int *diu;
   CHK(diag_sq_table(B, D, uq, -1.0, &sq));
   CHK(upload(B, "dp_iu", iu, &diu));
   const long tot = (long)npts * D.nm;
   CHK(B.get("dp_out", (size_t)tot, &out));
   k_diag_psd_points<<<(unsigned)((tot + 255) / 256), 256, 0, g.s>>>(
      sq, (int)uq.size(), D.nnl, D.kv, D.pa_k, D.K, D.nm, npts, diu, out);
   HIPC(hipGetLastError());
   HIPC(hipMemcpyAsync(psd, out, (size_t)tot * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

}  // extern "C"

namespace {

// the Mesher's point evaluation (mesher.hip)
int point_table(Bufs &B, const Prob &D, const double *fl, int nu, int nmp, double **V);
int point_psib(Bufs &B, const Prob &D, int nmp, double **PB);
int bfm_batch(const Prob &D, const double *V, const double *PB, int nmp, int npts, const int *i1,
              const int *i2, const int *i3, const long *slot, double *out);

// sqrt-PSD table (ntc, nu, nnl) of the nodes at the distinct |f| uq; fmax > 0:
// rows with |f| beyond fmax zero (the Classic grid's truncation)
int diag_sq_table(Bufs &B, const Prob &D, const std::vector<double> &uq, double fmax, double **sq)
{
   const int nu = (int)uq.size();
   if (nu > 65535) return fail(BSAHIP_EUNSUPPORTED, "more than 65535 distinct frequencies in one table");
   double *fl;
   CHK(upload(B, "dg_fl", uq, &fl));
   CHK(B.get("dg_sq", (size_t)D.ntc * nu * D.nnl, sq));
   dim3 gp((D.nnl + 63) / 64, nu, D.ntc);
   k_psd_sqrt<<<gp, 64, 0, g.s>>>(fl, nu, D.prm, D.formula, D.nnl, D.ntc, D.pulsation, *sq);
   HIPC(hipGetLastError());
   if (fmax > 0.0) {
      const long u0 = std::upper_bound(uq.begin(), uq.end(), fmax * (1.0 + 1e-12)) - uq.begin();
      for (int c = 0; c < D.ntc && u0 < nu; ++c)
         CHK(fill(*sq + ((size_t)c * nu + u0) * D.nnl, (size_t)(nu - u0) * D.nnl, 0.0));
   }
   return 0;
}

// Point BFM/BRM; fmax > 0: the Classic grid's truncation, S(|f|) = 0 beyond
// fmax (it reaches only f1 + f2 of grid points); diag: the ONLY_DIAG model,
// NM entries per point (k_diag_points, the Mesher's diagonal evaluation)
int bfm_points_impl(const bsahip_problem *p, int32_t npts, const double *fi, const double *fj,
                    double *bfm, double *brm, double fmax, bool diag)
{
   if (npts < 0 || (npts > 0 && (!fi || !fj || !bfm)))
      return fail(BSAHIP_EINVAL, "npts < 0 or NULL point/output arrays");
   if (npts == 0) return 0;
   Bufs &B = oneshot_bufs();
   Prob D;
   CHK(validate(p));
   std::vector<double> uq;
   std::vector<int> i1, i2, i3;
   point_tables(npts, fi, fj, uq, i1, i2, i3);
   int *di1, *di2, *di3;
   double *dfl, *df1, *df2;
   Pack pk;
   pk.add(uq, &dfl);
   pk.add(i1, &di1);
   pk.add(i2, &di2);
   pk.add(i3, &di3);
   pk.add(fi, npts * sizeof(double), reinterpret_cast<void **>(&df1));
   pk.add(fj, npts * sizeof(double), reinterpret_cast<void **>(&df2));
   CHK(load_problem(p, 0, B, D, &pk, !diag));
   if (diag) {
      const long tot = (long)npts * D.nm;
      if (tot > 0xffffff00L) return fail(BSAHIP_EUNSUPPORTED, "npts * NM exceeds 2^32 values");
      double *sq, *ob;
      long *ds;
      std::vector<long> slot(npts);
      for (int q = 0; q < npts; ++q) slot[q] = q;
      CHK(diag_sq_table(B, D, uq, fmax, &sq));
      CHK(upload(B, "dg_slot", slot, &ds));
      CHK(B.get("bfm_out", (size_t)tot, &ob));
      k_diag_points<<<(unsigned)((tot + 255) / 256), 256, 0, g.s>>>(
         sq, (int)uq.size(), D.nnl, D.kv, D.pa_k, D.pb_k, D.K, D.nm, npts, di1, di2, di3, ds, ob);
      HIPC(hipGetLastError());
      HIPC(hipMemcpyAsync(bfm, ob, (size_t)tot * sizeof(double), hipMemcpyDeviceToHost, g.s));
      if (brm) {
         double *orr;
         CHK(B.get("brm_out", (size_t)tot, &orr));
         HIPC(hipMemcpyAsync(orr, ob, (size_t)tot * sizeof(double), hipMemcpyDeviceToDevice, g.s));
         k_frf_apply<<<(unsigned)((tot + 255) / 256), 256, 0, g.s>>>(
            BSAHIP_FRF_POINTS, 1, npts, df1, npts, df2, D.nm, D.Mm, D.Km, D.Cm, tot, orr);
         HIPC(hipGetLastError());
         HIPC(hipMemcpyAsync(brm, orr, (size_t)tot * sizeof(double), hipMemcpyDeviceToHost, g.s));
      }
      HIPC(hipStreamSynchronize(g.s));
      return 0;
   }
   CHK(set_pod(p, D));
   const int nu = (int)uq.size();
   const size_t nm3 = (size_t)D.nm * D.nm * D.nm;
   const long tot = (long)nm3 * npts;
   if (tot > 0xffffff00L)
      return fail(BSAHIP_EUNSUPPORTED, "npts * NM^3 exceeds 2^32 bispectrum values in one call");
   // uq is ascending: rows u0.. lie beyond the grid
   const long u0 = fmax > 0.0 ? std::upper_bound(uq.begin(), uq.end(), fmax * (1.0 + 1e-12)) - uq.begin() : nu;
   double *ob, *orr = nullptr;
   CHK(B.get("bfm_out", nm3 * npts, &ob));
   if (brm) CHK(B.get("brm_out", nm3 * npts, &orr));
   const unsigned nblk = (unsigned)((tot + 255) / 256);
   // the Mesher's point kernel up to 32 modes; where its table, 16 or 32 columns for any
   // count of modes, finds no memory, the general one with its own of nm columns
   const int nmp = (D.nm + 15) / 16 * 16;
   double *V = nullptr, *PB = nullptr;
   int rc = D.nm <= 32 ? point_table(B, D, dfl, nu, nmp, &V) : BSAHIP_ENOMEM;
   if (rc == 0) rc = point_psib(B, D, nmp, &PB);
   if (rc != 0 && rc != BSAHIP_ENOMEM) return rc;
   if (rc == 0) {
      const size_t slab = (size_t)D.K * nmp;
      if (u0 < nu) CHK(fill(V + u0 * slab, (size_t)(nu - u0) * slab, 0.0));
      CHK(bfm_batch(D, V, PB, nmp, npts, di1, di2, di3, nullptr, ob));
      if (brm) {
         k_brm_points<<<nblk, 256, 0, g.s>>>(ob, D.nm, tot, df1, df2, D.Mm, D.Km, D.Cm, orr);
         HIPC(hipGetLastError());
      }
   } else {
      if (D.nm <= 32) B.drop({"m_V", "m_PB", "m_U"});
      const long ldU = (long)D.nm * nu;
      double *U;
      CHK(B.get("U", (size_t)D.K * ldU, &U));
      CHK(build_table(B, D, dfl, nu, nu, U, ldU));
      if (u0 < nu) {
         const long n = (long)D.K * D.nm * (nu - u0);
         k_zero_cols<<<(unsigned)((n + 255) / 256), 256, 0, g.s>>>(U, ldU, nu, u0, D.nm, n);
         HIPC(hipGetLastError());
      }
      k_bfm_points<<<nblk, 256, 0, g.s>>>(U, ldU, nu, D.pb_k, D.K, D.nm, npts, di1, di2, di3, df1, df2,
                                          D.Mm, D.Km, D.Cm, ob, orr);
      HIPC(hipGetLastError());
   }
   HIPC(hipMemcpyAsync(bfm, ob, nm3 * npts * sizeof(double), hipMemcpyDeviceToHost, g.s));
   if (brm) HIPC(hipMemcpyAsync(brm, orr, nm3 * npts * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

}  // namespace

extern "C" {

int bsahip_frf_apply(const bsahip_problem *p, int32_t flags, int32_t kind, int64_t n1,
                     const double *f1, int64_t n2, const double *f2, double *data)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (flags & ~BSAHIP_ONLY_DIAG) return fail(BSAHIP_EINVAL, "bsahip_frf_apply takes BSAHIP_ONLY_DIAG only");
   const bool diag = (flags & BSAHIP_ONLY_DIAG) != 0;
   if (kind < BSAHIP_FRF_PSD || kind > BSAHIP_FRF_POINTS)
      return fail(BSAHIP_EINVAL, "kind must be BSAHIP_FRF_PSD, _GRID or _POINTS");
   if (n1 < 0 || n2 < 0 || (kind == BSAHIP_FRF_GRID && n2 == 0 && n1 > 0))
      return fail(BSAHIP_EINVAL, "negative sizes, or a grid without f2");
   if (n1 == 0) return 0;
   if (!f1 || !data || (kind != BSAHIP_FRF_PSD && !f2))
      return fail(BSAHIP_EINVAL, "NULL frequencies or data");
   Bufs &B = oneshot_bufs();
   Prob D;
   CHK(load_problem(p, 0, B, D, nullptr, false));
   const long nm = D.nm, nm2 = diag ? nm : nm * nm, nm3 = diag ? nm : nm * nm * nm;
   const long nf2 = kind == BSAHIP_FRF_GRID ? n2 : (kind == BSAHIP_FRF_POINTS ? n1 : 0);
   const double tot_d = kind == BSAHIP_FRF_PSD ? (double)n1 * nm2
                       : (kind == BSAHIP_FRF_GRID ? (double)n1 * n2 * nm3 : (double)n1 * nm3);
   if (tot_d > (double)0xffffff00L)  // one thread per value, grid within 2^32 threads
      return fail(BSAHIP_EUNSUPPORTED, "more than 2^32 spectral values in one call");
   const long total = (long)tot_d;
   std::vector<double> h1(f1, f1 + n1), h2;
   if (nf2) h2.assign(f2, f2 + nf2);
   double *d1, *d2 = nullptr, *dd;
   CHK(upload(B, "frf_f1", h1, &d1));
   if (nf2) CHK(upload(B, "frf_f2", h2, &d2));
   CHK(B.get("frf_data", (size_t)total, &dd));
   HIPC(hipMemcpyAsync(dd, data, (size_t)total * sizeof(double), hipMemcpyHostToDevice, g.s));
   k_frf_apply<<<(unsigned)((total + 255) / 256), 256, 0, g.s>>>(kind, diag ? 1 : 0, n1, d1, n2, d2,
                                                                  D.nm, D.Mm, D.Km, D.Cm, total, dd);
   HIPC(hipGetLastError());
   HIPC(hipMemcpyAsync(data, dd, (size_t)total * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

int bsahip_selftest_mfma_layout(double *out512)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (!out512) return fail(BSAHIP_EINVAL, "NULL output");
   double *d;
   CHK(oneshot_bufs().get("selftest", 512, &d));
   k_mfma_f64_layout<<<1, 64, 0, g.s>>>(d);
   HIPC(hipGetLastError());
   HIPC(hipMemcpyAsync(out512, d, 512 * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

int bsahip_dgemm_strided_batched(int32_t transa, int32_t transb, int32_t M, int32_t N, int32_t K,
                                 double alpha, const double *A, int64_t lda, int64_t sA,
                                 const double *B, int64_t ldb, int64_t sB, double beta, double *C,
                                 int64_t ldc, int64_t sC, int32_t batch)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (M < 0 || N < 0 || K < 0 || batch < 1 || !A || !B || !C || (transa != 0 && transa != 1) ||
       (transb != 0 && transb != 1) || lda < (transa ? K : M) || ldb < (transb ? N : K) || ldc < M ||
       sA < 0 || sB < 0 || sC < 0)
      return fail(BSAHIP_EINVAL, "bad GEMM arguments");
   // extents of the host arrays (column-major, last batch included)
   const size_t na = (size_t)sA * (batch - 1) + (size_t)lda * (transa ? M : K);
   const size_t nb = (size_t)sB * (batch - 1) + (size_t)ldb * (transb ? K : N);
   const size_t nc = (size_t)sC * (batch - 1) + (size_t)ldc * N;
   Bufs &Bf = oneshot_bufs();
   double *dA, *dB, *dC;
   CHK(Bf.get("gemm_A", std::max<size_t>(na, 1), &dA));
   CHK(Bf.get("gemm_B", std::max<size_t>(nb, 1), &dB));
   CHK(Bf.get("gemm_C", std::max<size_t>(nc, 1), &dC));
   HIPC(hipMemcpyAsync(dA, A, na * sizeof(double), hipMemcpyHostToDevice, g.s));
   HIPC(hipMemcpyAsync(dB, B, nb * sizeof(double), hipMemcpyHostToDevice, g.s));
   HIPC(hipMemcpyAsync(dC, C, nc * sizeof(double), hipMemcpyHostToDevice, g.s));
   CHK(dgemm_sb(transa, transb, M, N, K, alpha, dA, lda, sA, dB, ldb, sB, beta, dC, ldc, sC, batch));
   HIPC(hipMemcpyAsync(C, dC, nc * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

int bsahip_selftest_mfma_f32_layout(float *out512)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (!out512) return fail(BSAHIP_EINVAL, "NULL output");
   float *d;
   CHK(oneshot_bufs().get("selftest32", 512, &d));
   k_mfma_f32_layout<<<1, 64, 0, g.s>>>(d);
   HIPC(hipGetLastError());
   HIPC(hipMemcpyAsync(out512, d, 512 * sizeof(float), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

int bsahip_selftest_mfma_bf16_layout(float *out768)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   CHK(ensure_init());
   if (!out768) return fail(BSAHIP_EINVAL, "NULL output");
   float *d;
   CHK(oneshot_bufs().get("selftest16", 768, &d));
   k_mfma_bf16_layout<<<1, 64, 0, g.s>>>(d);
   HIPC(hipGetLastError());
   HIPC(hipMemcpyAsync(out768, d, 768 * sizeof(float), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   return 0;
}

}  // extern "C"

#include "mesher.hip"
#include "recomb.hip"
#include "mlp.hip"
#include "batch.hip"
