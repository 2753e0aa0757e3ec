// Batches of structures of uneven size (node, mode, component and frequency
// counts): every structure is a resident plan; one step builds all their tables
// in one launch per kind (PSD, FRF and cleared sums; projection; operand split),
// then ONE persistent G-contraction launch whose workgroups take work items
// (structure, tile pair, mode) from a device queue, while one launch on a side
// stream computes every structure's modal PSD moments.  The step is captured once
// in a HIP graph (the side stream becomes a parallel branch) and replayed.  The
// item list is ordered by decreasing cost per item (longest-processing-time
// first) and split into one queue per XCD; a small autotuner picks the persistent
// grid size and the items per ticket.

__device__ __forceinline__ long uniform_long(long v)
{
   const int lo = __builtin_amdgcn_readfirstlane((int)(v & 0xffffffffL));
   const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
   return ((long)hi << 32) | (long)(unsigned)lo;
}

// structure of item `it`: offs[s] <= it < offs[s+1] (offs has ns+1 entries)
__device__ __forceinline__ int batch_struct(const long *__restrict__ offs, int ns, long it)
{
   int lo = 0, hi = ns;
   while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (offs[mid] <= it) lo = mid;
      else hi = mid;
   }
   return lo;
}

__global__ void k_zero_u64(unsigned long long *c, int n)
{
   if ((int)threadIdx.x < n) c[threadIdx.x] = 0ull;
}

// Work queues: the ordered item list is cut into 8 contiguous slices, one per
// XCD (a persistent workgroup stays on XCD blockIdx.x % 8), so the nm items of
// one tile pair -- which read the same U tiles -- share that XCD's L2.  A
// workgroup drains its own slice, then takes items from the other slices.
#define BATCH_QUEUES 8

template <class Item>
__device__ __forceinline__ void batch_drain(const long *__restrict__ offs, int ns,
                                            const long *__restrict__ qbeg,
                                            unsigned long long *counters, int chunk, Item item)
{
   __shared__ long s_i0;
   const int own = blockIdx.x % BATCH_QUEUES;
   for (int k = 0; k < BATCH_QUEUES; ++k) {
      const int q = (own + k) % BATCH_QUEUES;
      const long b0 = qbeg[q], len = qbeg[q + 1] - qbeg[q];
      for (;;) {
         __syncthreads();
         if (threadIdx.x == 0) s_i0 = (long)atomicAdd(counters + q, (unsigned long long)chunk);
         __syncthreads();
         const long i0 = uniform_long(s_i0);
         if (i0 >= len) break;
         const long i1 = i0 + chunk < len ? i0 + chunk : len;
         for (long it = b0 + i0; it < b0 + i1; ++it) {
            const int s = batch_struct(offs, ns, it);
            item(s, it - offs[s]);
         }
      }
   }
}

// 2x2 blocks for every structure: the launch has one tile shape, and small structures, which
// batches are for, need the smaller one.  The launch bound of the single form's 2x2 (4)
// changes nothing here (-1 to +2 % over batches of 4 to 64 structures).
__global__ __launch_bounds__(256, 2) void k_gsym_f64_batch(const GsymArgs *__restrict__ args,
                                                        const long *__restrict__ offs, int ns,
                                                        const long *__restrict__ qbeg,
                                                        unsigned long long *counters, int chunk)
{
   batch_drain(offs, ns, qbeg, counters, chunk, [&](int s, long li) {
      const GsymArgs a = args[s];
      gsym_f64_wave<2, 2, false>(a, (int)(li % a.nm), li / a.nm);
   });
}

__global__ __launch_bounds__(256, 2) void k_gsym_bf16x3_batch(
   const GsymArgs *__restrict__ args, const GsymArgs16 *__restrict__ args16,
   const long *__restrict__ offs, int ns, const long *__restrict__ qbeg,
   unsigned long long *counters, int chunk)
{
   batch_drain(offs, ns, qbeg, counters, chunk, [&](int s, long li) {
      const GsymArgs a = args[s];
      const GsymArgs16 b = args16[s];
      gsym_bf16x3_item(a, b, (int)(li % a.nm), li / a.nm);
   });
}

__global__ __launch_bounds__(256, 2) void k_gsym_f32_batch(
   const GsymArgs *__restrict__ args, const GsymArgs16 *__restrict__ args16,
   const long *__restrict__ offs, int ns, const long *__restrict__ qbeg,
   unsigned long long *counters, int chunk)
{
   batch_drain(offs, ns, qbeg, counters, chunk, [&](int s, long li) {
      const GsymArgs a = args[s];
      const GsymArgs16 b = args16[s];
      gsym_f32_item(a, b, (int)(li % a.nm), li / a.nm);
   });
}

// The table launches over every structure: block (or wave) -> structure by binary
// search over the offsets, then the single-structure kernel's work.  A launch per
// structure and table kind left the chip to one small structure at a time and cost
// eight launches each: 64 towers (NN 20-60, NM 3-6, 65-129 points a side) 1.67 ms
// a step, 0.52 ms with these.
struct BatchTab {
   const double *fl, *prm, *Mm, *Km, *Cm;
   const int *formula;
   double *sq, *m3, *m2;
   double2 *H;
   double df;
   int nu, nnl, nm, nft, pulsation;
   long npsd, nfrf, nm3, nm2;          // values of each kind (sums to clear: nm3, nm2)
};

__global__ __launch_bounds__(256) void k_batch_tables(const BatchTab *__restrict__ tab,
                                                      const long *__restrict__ offs, int ns)
{
   const int s = batch_struct(offs, ns, blockIdx.x);
   const BatchTab T = tab[s];
   long t = ((long)blockIdx.x - offs[s]) * 256 + threadIdx.x;
   if (t < T.npsd) {
      const int i = (int)(t % T.nnl);
      const long r = t / T.nnl;                       // tc * nu + q
      const int q = (int)(r % T.nu), tc = (int)(r / T.nu);
      T.sq[t] = psd_sqrt(T.prm + ((size_t)tc * T.nnl + i) * 4, T.formula[tc], T.fl[q], T.pulsation);
      return;
   }
   t -= T.npsd;
   if (t < T.nfrf) {
      T.H[t] = frf_grid(T.Mm, T.Km, T.Cm, (int)(t / T.nft), (int)(t % T.nft), T.df);
      return;
   }
   t -= T.nfrf;
   if (t < T.nm3) T.m3[t] = 0.0;
   else if (t - T.nm3 < T.nm2) T.m2[t - T.nm3] = 0.0;
}

template <int MT, int F>
__global__ __launch_bounds__(256, 2) void k_project_batch(const ProjArgs *__restrict__ args,
                                                          const long *__restrict__ offs, int ns)
{
   const long wid = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   if (wid >= offs[ns]) return;
   const int s = batch_struct(offs, ns, wid);
   const ProjArgs P = args[s];
   const long l = wid - offs[s], per = P.nqg * P.ncoltile;
   const int r = (int)(l / per);
   project_wave<MT, F, false>(P, l % per, r % P.ntc, (r / P.ntc) * (MT * 16));
}

struct SplitArgs {
   const double *U;
   float *UR;
   uint16_t *Ch, *Cl;
   long ldU;
   int K;
};

__global__ __launch_bounds__(256) void k_split_batch(const SplitArgs *__restrict__ args,
                                                     const long *__restrict__ offs, int ns)
{
   const int s = batch_struct(offs, ns, blockIdx.x);
   const SplitArgs a = args[s];
   const long l = (long)blockIdx.x - offs[s], nr = a.ldU / 32;
   split_tile((int)(l % nr) * 32, (int)(l / nr) * 32, a.U, a.ldU, a.K, (int)a.ldU, a.K, a.UR, a.Ch, a.Cl);
}

template <int MT>
__global__ __launch_bounds__(256, 2) void k_m2_batch(const M2Args *__restrict__ args,
                                                     const long *__restrict__ offs, int ns)
{
   const int s = batch_struct(offs, ns, blockIdx.x);
   const M2Args a = args[s];
   const int l = (int)((long)blockIdx.x - offs[s]), nby = (a.nh + 63) / 64;
   m2_block<MT>(a, l % a.nm, (l / a.nm) % nby, l / (a.nm * nby) * 16 * MT, 0);
}

// results of every structure into one contiguous buffer: array j = srcs[j]
// (lens[j] doubles) to dst + offs[j], its copies[j] copies summed; grid (arrays, any)
__global__ void k_pack(const double *const *__restrict__ srcs, const long *__restrict__ lens,
                       const int *__restrict__ copies, const long *__restrict__ offs,
                       double *__restrict__ dst)
{
   const int j = blockIdx.x;
   const double *src = srcs[j];
   double *d = dst + offs[j];
   for (long t = blockIdx.y * blockDim.x + threadIdx.x; t < lens[j]; t += gridDim.y * blockDim.x)
      d[t] = sum_all(copies[j], [&](int c) { return src[c * lens[j] + t]; });
}

struct bsahip_batch {
   std::vector<std::unique_ptr<bsahip_plan>> plans;
   std::vector<int> order;            // queue order of the structures
   int prec = 0;
   int32_t flags = 0;
   Bufs B;
   GsymArgs *args = nullptr;
   GsymArgs16 *args16 = nullptr;
   long *offs = nullptr;
   unsigned long long *counter = nullptr;   // one per queue
   long *qbeg = nullptr;                    // queue slices of the item list
   std::vector<long> qb;                    // host copy
   long total = 0;
   int ncu = 0, occ = 1;
   int grid_mult = 2, chunk = 1;
   hipGraph_t graph = nullptr;
   hipGraphExec_t gexec = nullptr;
   double ms_total = 0.0, ms_gsym = 0.0;
   // side stream (default priority) of the PSD moments, forked from and joined to
   // the library stream
   hipStream_t side = nullptr;
   hipEvent_t ev_fork = nullptr, ev_m2 = nullptr;
   // launches over every structure: descriptors and their block (wave) offsets, the
   // structures of one template instance together
   BatchTab *tab = nullptr;
   SplitArgs *split = nullptr;
   long *tab_offs = nullptr, *split_offs = nullptr;
   long tab_blocks = 0, split_blocks = 0;
   struct Group {
      int mt, F, n;              // template arguments, structures
      long total;                // blocks or waves
      long *offs;
      ProjArgs *proj;
      M2Args *m2;
   };
   std::vector<Group> proj, m2;
   bool joint = true;            // one table launch per kind (batch_descriptors)
   // packed results: per structure m3 (m3f, m3r) then m2 (f, r, o)
   const double **psrc = nullptr;
   long *plen = nullptr, *poff = nullptr;
   int *pcopies = nullptr;
   long longest = 0;                        // doubles of the longest result
   double *pack = nullptr, *hpack = nullptr;   // device buffer, pinned host copy
   std::vector<long> m3off, m2off;
   long npack = 0;
   ~bsahip_batch()
   {
      if (hpack) (void)hipHostFree(hpack);
      if (gexec) (void)hipGraphExecDestroy(gexec);
      if (graph) (void)hipGraphDestroy(graph);
      if (ev_m2) (void)hipEventDestroy(ev_m2);
      if (ev_fork) (void)hipEventDestroy(ev_fork);
      if (side) (void)hipStreamDestroy(side);
   }
};

namespace {

// queue slices for the first `total` items: 8 equal contiguous ranges
int batch_slices(bsahip_batch *b, long total)
{
   b->qb.assign(BATCH_QUEUES + 1, 0);
   for (int q = 0; q <= BATCH_QUEUES; ++q) b->qb[q] = total * q / BATCH_QUEUES;
   HIPC(hipMemcpyAsync(b->qbeg, b->qb.data(), (BATCH_QUEUES + 1) * sizeof(long),
                       hipMemcpyHostToDevice, g.s));
   return 0;
}

int batch_launch(bsahip_batch *b)
{
   const unsigned grid = (unsigned)std::max(BATCH_QUEUES, b->grid_mult * b->ncu * b->occ);
   const int ns = (int)b->order.size();
   k_zero_u64<<<1, 64, 0, g.s>>>(b->counter, BATCH_QUEUES);
   HIPC(hipGetLastError());
   if (b->prec == BSAHIP_PREC_BF16X3)
      k_gsym_bf16x3_batch<<<grid, 256, 0, g.s>>>(b->args, b->args16, b->offs, ns, b->qbeg,
                                                 b->counter, b->chunk);
   else if (b->prec == BSAHIP_PREC_FP32)
      k_gsym_f32_batch<<<grid, 256, 0, g.s>>>(b->args, b->args16, b->offs, ns, b->qbeg,
                                              b->counter, b->chunk);
   else
      k_gsym_f64_batch<<<grid, 256, 0, g.s>>>(b->args, b->offs, ns, b->qbeg, b->counter, b->chunk);
   HIPC(hipGetLastError());
   return 0;
}

// results of every structure into `pack`
int batch_pack(bsahip_batch *b)
{
   const dim3 grid((unsigned)(2 * b->plans.size()), (unsigned)std::min<long>((b->longest + 255) / 256, 64));
   k_pack<<<grid, 256, 0, g.s>>>(b->psrc, b->plen, b->pcopies, b->poff, b->pack);
   HIPC(hipGetLastError());
   return 0;
}

// descriptors of the launches over every structure, on the device
int batch_descriptors(bsahip_batch *b)
{
   const bool bisp = !(b->flags & BSAHIP_NO_BISP), psd = !(b->flags & BSAHIP_NO_PSD);
   const int n = (int)b->plans.size();
   auto up = [&](const char *name, const auto &h, auto **d) -> int { return upload(b->B, name, h, d); };
   std::vector<BatchTab> tab;
   std::vector<SplitArgs> sp;
   std::vector<long> toff(1, 0), soff(1, 0);
   for (auto &P : b->plans) {
      const Prob &D = P->D;
      BatchTab T;
      CHK(P->B.get("sq", (size_t)D.ntc * P->nu * D.nnl, &T.sq));
      T.fl = P->fl;
      T.prm = D.prm;
      T.Mm = D.Mm;
      T.Km = D.Km;
      T.Cm = D.Cm;
      T.formula = D.formula;
      T.m3 = P->m3;
      T.m2 = P->m2;
      T.H = P->H;
      T.df = P->df;
      T.nu = P->nu;
      T.nnl = D.nnl;
      T.nm = D.nm;
      T.nft = P->nft;
      T.pulsation = D.pulsation;
      T.npsd = (long)D.ntc * P->nu * D.nnl;
      T.nfrf = (long)D.nm * P->nft;
      T.nm3 = bisp ? 2L * D.nm * D.nm * D.nm * P->copies : 0;
      T.nm2 = psd ? 3L * D.nm * D.nm : 0;
      tab.push_back(T);
      toff.push_back(toff.back() + (T.npsd + T.nfrf + T.nm3 + T.nm2 + 255) / 256);
      sp.push_back(SplitArgs{P->U, P->UR, P->Ch, P->Cl, P->ldU, D.K});
      soff.push_back(soff.back() + P->ldU / 32 * ((D.K + 31) / 32));
   }
   b->tab_blocks = toff.back();
   b->split_blocks = bisp && b->prec != BSAHIP_PREC_FP64 ? soff.back() : 0;
   CHK(up("bt_tab", tab, &b->tab));
   CHK(up("bt_toff", toff, &b->tab_offs));
   CHK(up("bt_split", sp, &b->split));
   CHK(up("bt_soff", soff, &b->split_offs));
   for (int mt = 1; mt <= 4; ++mt) {
      // one frequency group size per template, as if the structures were one table
      std::vector<int> in;
      long tiles = 0;
      int nfl = 1;
      for (int i = 0; i < n; ++i) {
         const bsahip_plan *P = b->plans[i].get();
         if (proj_mt(P->D.nm) != mt) continue;
         in.push_back(i);
         nfl = std::max(nfl, P->nu);
      }
      if (in.empty()) continue;
      std::vector<ProjArgs> pa;
      for (int i : in) {
         const bsahip_plan *P = b->plans[i].get();
         pa.push_back(proj_args(P->D, tab[i].sq, P->fl, P->nu, P->nhp, P->U, P->ldU, false));
         tiles += (long)pa.back().ncoltile * P->D.ntc * proj_chunks(P->D.nm) * P->nu / nfl + 1;
      }
      bsahip_batch::Group G;
      G.mt = mt;
      G.F = project_group(tiles, nfl, 1, mt);
      G.n = (int)in.size();
      std::vector<long> off(1, 0);
      for (size_t k = 0; k < in.size(); ++k) {
         ProjArgs &A = pa[k];
         A.nqg = (A.nfl + G.F - 1) / G.F;
         off.push_back(off.back() + A.nqg * A.ncoltile * A.ntc * proj_chunks(A.nm));
      }
      G.total = off.back();
      G.m2 = nullptr;
      const std::string id = std::to_string(mt);
      CHK(up(("bt_proj" + id).c_str(), pa, &G.proj));
      CHK(up(("bt_poff" + id).c_str(), off, &G.offs));
      b->proj.push_back(G);
   }
   for (int mt = 1; psd && mt <= 2; ++mt) {
      std::vector<M2Args> a;
      std::vector<long> off(1, 0);
      for (auto &P : b->plans) {
         const int nm = P->D.nm;
         if ((nm <= 16 ? 1 : 2) != mt) continue;
         a.push_back(plan_m2_args(P.get()));
         a.back().kper = a.back().K;               // one slice
         off.push_back(off.back() + (long)nm * ((P->nh + 63) / 64) * ((nm + 16 * mt - 1) / (16 * mt)));
      }
      if (a.empty()) continue;
      bsahip_batch::Group G;
      G.mt = mt;
      G.F = 0;
      G.n = (int)a.size();
      G.total = off.back();
      G.proj = nullptr;
      const std::string id = std::to_string(mt);
      CHK(up(("bt_m2" + id).c_str(), a, &G.m2));
      CHK(up(("bt_m2off" + id).c_str(), off, &G.offs));
      b->m2.push_back(G);
   }
   // a launch holds at most 2^32 threads: batches beyond that (thousands of large
   // structures) build their tables structure by structure
   b->joint = b->tab_blocks <= 0xffffffL && b->split_blocks <= 0xffffffL;
   for (const auto *v : {&b->proj, &b->m2})
      for (const auto &G : *v) b->joint = b->joint && G.total <= 0xffffffL;
   return 0;
}

// tables of every structure on the library stream
int batch_tables(bsahip_batch *b)
{
   const int n = (int)b->plans.size();
   if (!b->joint) {
      for (auto &P : b->plans) CHK(plan_prepare(P.get()));
      return 0;
   }
   k_batch_tables<<<(unsigned)b->tab_blocks, 256, 0, g.s>>>(b->tab, b->tab_offs, n);
   HIPC(hipGetLastError());
   for (const auto &G : b->proj) {
      proj_dispatch(G.mt, G.F, [&](auto MT, auto F) {
         k_project_batch<decltype(MT)::value, decltype(F)::value>
            <<<(unsigned)((G.total + 3) / 4), 256, 0, g.s>>>(G.proj, G.offs, G.n);
      });
      HIPC(hipGetLastError());
   }
   if (b->split_blocks) {
      k_split_batch<<<(unsigned)b->split_blocks, 256, 0, g.s>>>(b->split, b->split_offs, n);
      HIPC(hipGetLastError());
   }
   return 0;
}

// one step, stream-ordered, no host synchronisation (capturable).
// mode 1: everything on the library stream, one launch per structure and kind.
// mode 0: the tables of every structure, then the persistent G launch on the
// library stream while the side stream computes the PSD moments.
int batch_step(bsahip_batch *b, int mode)
{
   const bool bisp = !(b->flags & BSAHIP_NO_BISP), psd = !(b->flags & BSAHIP_NO_PSD);
   if (mode == 1) {
      for (auto &P : b->plans) CHK(plan_prepare(P.get()));
      if (bisp)
         for (int s : b->order) CHK(plan_gsym(b->plans[s].get()));
      if (psd)
         for (auto &P : b->plans) CHK(plan_m2(P.get()));
      return batch_pack(b);
   }
   CHK(batch_tables(b));
   if (psd) {
      HIPC(hipEventRecord(b->ev_fork, g.s));
      HIPC(hipStreamWaitEvent(b->side, b->ev_fork, 0));
      if (!b->joint) {
         const hipStream_t keep = g.s;
         int rc = 0;
         g.s = b->side;
         for (size_t i = 0; i < b->plans.size() && rc == 0; ++i) rc = plan_m2(b->plans[i].get());
         g.s = keep;
         CHK(rc);
      }
      for (const auto &G : b->m2) {
         if (!b->joint) break;
         if (G.mt == 1) k_m2_batch<1><<<(unsigned)G.total, 256, 0, b->side>>>(G.m2, G.offs, G.n);
         else k_m2_batch<2><<<(unsigned)G.total, 256, 0, b->side>>>(G.m2, G.offs, G.n);
         HIPC(hipGetLastError());
      }
      HIPC(hipEventRecord(b->ev_m2, b->side));
   }
   if (bisp) CHK(batch_launch(b));
   if (psd) HIPC(hipStreamWaitEvent(g.s, b->ev_m2, 0));
   return batch_pack(b);
}

void batch_drop_graph(bsahip_batch *b)
{
   if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
   if (b->graph) (void)hipGraphDestroy(b->graph);
   b->gexec = nullptr;
   b->graph = nullptr;
}

int batch_capture(bsahip_batch *b)
{
   batch_drop_graph(b);
   HIPC(hipStreamBeginCapture(g.s, hipStreamCaptureModeRelaxed));
   const int rc = batch_step(b, 0);
   hipGraph_t gr = nullptr;
   const hipError_t e = hipStreamEndCapture(g.s, &gr);
   if (rc) {
      if (gr) (void)hipGraphDestroy(gr);
      return rc;
   }
   if (e != hipSuccess) return fail(BSAHIP_EDEVICE, std::string("graph capture: ") + hipGetErrorString(e));
   b->graph = gr;
   HIPC(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
   return 0;
}

}  // namespace

extern "C" {

int bsahip_batch_create(const bsahip_problem *const *probs, const int32_t *nfh, const double *df,
                        int32_t n, int32_t flags, bsahip_batch **out)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (!probs || !nfh || !df || !out || n < 1) return fail(BSAHIP_EINVAL, "bad batch arguments");
   *out = nullptr;
   CHK(ensure_init());
   CHK(check_flags(flags, true, true));
   if (flags & BSAHIP_SUM_EXACT) return fail(BSAHIP_EUNSUPPORTED, "batches use the Classic truncated sum");
   if (flags & BSAHIP_DETERMINISTIC)
      return fail(BSAHIP_EUNSUPPORTED, "batches sum with atomics (no fixed-order mode)");
   std::unique_ptr<bsahip_batch> B(new bsahip_batch());
   B->prec = flags & BSAHIP_PREC_MASK;
   B->flags = flags;
   for (int i = 0; i < n; ++i) {
      std::unique_ptr<bsahip_plan> P(new bsahip_plan());
      P->f64_br = P->f64_bc = 2;               // the persistent kernel's tile
      const int rc = plan_setup(P.get(), probs[i], nfh[i], df[i], flags, 0);
      if (rc) {
         g_err = "structure " + std::to_string(i) + ": " + g_err;
         return rc;
      }
      B->plans.push_back(std::move(P));
   }
   // queue order: decreasing contraction length K (cost of one item), then modes
   B->order.resize(n);
   for (int i = 0; i < n; ++i) B->order[i] = i;
   std::stable_sort(B->order.begin(), B->order.end(), [&](int x, int y) {
      const Prob &a = B->plans[x]->D, &c = B->plans[y]->D;
      return a.K != c.K ? a.K > c.K : a.nm > c.nm;
   });
   std::vector<GsymArgs> a(n);
   std::vector<GsymArgs16> a16(n);
   std::vector<long> offs(n + 1, 0);
   for (int q = 0; q < n; ++q) {
      const bsahip_plan *P = B->plans[B->order[q]].get();
      plan_args(P, a[q], a16[q]);
      offs[q + 1] = offs[q] + plan_items(P);
   }
   B->total = offs[n];
   CHK(B->B.get("args", (size_t)n, &B->args));
   CHK(B->B.get("args16", (size_t)n, &B->args16));
   CHK(B->B.get("offs", (size_t)n + 1, &B->offs));
   CHK(B->B.get("counter", BATCH_QUEUES, &B->counter));
   CHK(B->B.get("qbeg", BATCH_QUEUES + 1, &B->qbeg));
   HIPC(hipMemcpyAsync(B->args, a.data(), n * sizeof(GsymArgs), hipMemcpyHostToDevice, g.s));
   HIPC(hipMemcpyAsync(B->args16, a16.data(), n * sizeof(GsymArgs16), hipMemcpyHostToDevice, g.s));
   HIPC(hipMemcpyAsync(B->offs, offs.data(), (n + 1) * sizeof(long), hipMemcpyHostToDevice, g.s));
   CHK(batch_slices(B.get(), B->total));
   int dev = 0;
   HIPC(hipGetDevice(&dev));
   HIPC(hipDeviceGetAttribute(&B->ncu, hipDeviceAttributeMultiprocessorCount, dev));
   int occ = 1;
   if (B->prec == BSAHIP_PREC_BF16X3)
      HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_gsym_bf16x3_batch, 256, 0));
   else if (B->prec == BSAHIP_PREC_FP32)
      HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_gsym_f32_batch, 256, 0));
   else
      HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_gsym_f64_batch, 256, 0));
   B->occ = std::max(1, occ);
   HIPC(hipStreamCreateWithFlags(&B->side, hipStreamNonBlocking));
   HIPC(hipEventCreateWithFlags(&B->ev_m2, hipEventDisableTiming));
   HIPC(hipEventCreateWithFlags(&B->ev_fork, hipEventDisableTiming));
   {
      std::vector<const double *> src;
      std::vector<long> len, off;
      std::vector<int> copies;
      long o = 0;
      for (auto &P : B->plans) {
         const long nm = P->D.nm;
         B->m3off.push_back(o);
         src.push_back(P->m3);
         len.push_back(2 * nm * nm * nm);
         copies.push_back(P->copies);
         off.push_back(o);
         o += 2 * nm * nm * nm;
         B->longest = std::max({B->longest, len.back(), 3 * nm * nm});
         B->m2off.push_back(o);
         src.push_back(P->m2);
         len.push_back(3 * nm * nm);
         copies.push_back(1);
         off.push_back(o);
         o += 3 * nm * nm;
      }
      B->npack = o;
      CHK(B->B.get("psrc", src.size(), &B->psrc));
      CHK(B->B.get("plen", len.size(), &B->plen));
      CHK(B->B.get("poff", off.size(), &B->poff));
      CHK(B->B.get("pack", (size_t)o, &B->pack));
      CHK(upload(B->B, "pcopies", copies, &B->pcopies));
      HIPC(hipMemcpyAsync(B->psrc, src.data(), src.size() * sizeof(double *), hipMemcpyHostToDevice, g.s));
      HIPC(hipMemcpyAsync(B->plen, len.data(), len.size() * sizeof(long), hipMemcpyHostToDevice, g.s));
      HIPC(hipMemcpyAsync(B->poff, off.data(), off.size() * sizeof(long), hipMemcpyHostToDevice, g.s));
      HIPC(hipHostMalloc((void **)&B->hpack, (size_t)o * sizeof(double), hipHostMallocDefault));
   }
   CHK(batch_descriptors(B.get()));
   // warm-up run: every buffer reaches its size before a graph is captured
   CHK(batch_step(B.get(), 1));
   HIPC(hipStreamSynchronize(g.s));
   *out = B.release();
   return 0;
}

int bsahip_batch_autotune(bsahip_batch *b, int32_t *grid_mult, int32_t *chunk)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (!b) return fail(BSAHIP_EINVAL, "NULL batch");
   if (b->flags & BSAHIP_NO_BISP) return 0;
   // the tables of every structure are current after any step; time the
   // persistent contraction alone on the first quarter of the queue (the
   // structures with the longest items)
   const long part = std::max(1L, b->total / 4);
   static const int mults[] = {1, 2, 4};
   static const int chunks[] = {1, 4, 16};
   double best = 1e300;
   int bm = b->grid_mult, bc = b->chunk;
   for (int m : mults)
      for (int c : chunks) {
         b->grid_mult = m;
         b->chunk = c;
         CHK(batch_slices(b, part));
         HIPC(hipEventRecord(g.e0, g.s));
         CHK(batch_launch(b));
         HIPC(hipEventRecord(g.e1, g.s));
         HIPC(hipStreamSynchronize(g.s));
         float ms = 0.f;
         HIPC(hipEventElapsedTime(&ms, g.e0, g.e1));
         if (ms < best) {
            best = ms;
            bm = m;
            bc = c;
         }
      }
   b->grid_mult = bm;
   b->chunk = bc;
   CHK(batch_slices(b, b->total));
   HIPC(hipStreamSynchronize(g.s));
   batch_drop_graph(b);
   if (grid_mult) *grid_mult = bm;
   if (chunk) *chunk = bc;
   return 0;
}

int bsahip_batch_run(bsahip_batch *b, int32_t mode, double *const *m3mf, double *const *m3mr,
                     double *const *m2mr)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   if (!b) return fail(BSAHIP_EINVAL, "NULL batch");
   if (mode < 0 || mode > 2)
      return fail(BSAHIP_EINVAL, "mode must be 0 (graph), 1 (per structure) or 2 (streams)");
   if (mode == 0 && !b->gexec) CHK(batch_capture(b));
   HIPC(hipEventRecord(g.e0, g.s));
   if (mode == 0) HIPC(hipGraphLaunch(b->gexec, g.s));
   else CHK(batch_step(b, mode == 1 ? 1 : 0));
   HIPC(hipEventRecord(g.e1, g.s));
   HIPC(hipMemcpyAsync(b->hpack, b->pack, (size_t)b->npack * sizeof(double), hipMemcpyDeviceToHost, g.s));
   HIPC(hipStreamSynchronize(g.s));
   for (size_t i = 0; i < b->plans.size(); ++i) {
      const size_t nm = b->plans[i]->D.nm, nm3 = nm * nm * nm, nm2 = nm * nm;
      const double *m3 = b->hpack + b->m3off[i], *m2 = b->hpack + b->m2off[i];
      if (m3mf && m3mf[i]) std::memcpy(m3mf[i], m3, nm3 * sizeof(double));
      if (m3mr && m3mr[i]) std::memcpy(m3mr[i], m3 + nm3, nm3 * sizeof(double));
      if (m2mr && m2mr[i]) std::memcpy(m2mr[i], m2 + nm2, nm2 * sizeof(double));
   }
   float ms = 0.f;
   HIPC(hipEventElapsedTime(&ms, g.e0, g.e1));
   b->ms_total = ms;
   return 0;
}

int bsahip_batch_info(const bsahip_batch *b, double *ms_step, int64_t *items, int32_t *grid_mult,
                      int32_t *chunk)
{
   if (!b) return fail(BSAHIP_EINVAL, "NULL batch");
   if (ms_step) *ms_step = b->ms_total;
   if (items) *items = b->total;
   if (grid_mult) *grid_mult = b->grid_mult;
   if (chunk) *chunk = b->chunk;
   return 0;
}

int bsahip_batch_destroy(bsahip_batch *b)
{
   std::lock_guard<std::recursive_mutex> lk(g.mu);
   delete b;
   return 0;
}

}  // extern "C"
