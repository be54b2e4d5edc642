/*
 * cpsd_api.hip -- host orchestration of the MI355X SD step and the C-ABI
 * entry points declared in include/cpsd_abi.h.
 *
 * One SD step (ccpsdv3/cpsd.c:169-491) on the device, FP64, one HIP stream:
 *   1  C1 <- C2 (buffer role swap, no copy)                    :173
 *   2  z pass G->r of every orbital into T                      :177-181
 *   3  y+x passes per z plane, psi^2 summed per orbital block   :185-194
 *   4  dn = scal2 sum psi^2, LDA xcp/xce at every point         :185, :370-371
 *   5  dng = mask(FFT(2 dn / N^3))                              :198-205
 *   6  V(r) = FFT^-1(vall/Omega + dng vc) + xcp                 :373-382, :388
 *   7  per plane: psi -> V psi -> forward x,y (in place in T)   :384-392
 *   8  z pass r->G, CP = -scal1 mask(V psi) - tg C1             :212-221, :394-395
 *   9  P = beta^T W C1 (split-K MFMA), KB coefficients          :287-289
 *  10  CP += beta X ; C2 = C1 + dte CP (tall MFMA, fused)       :290, :399-400
 *  11  Gram of [C1|C2] (split-K MFMA, symmetric tiles)          :415-437
 *  12  Lagrange fixed point (persistent kernel)                 :439-478
 *  13  C2 += dte C1 lmd (tall MFMA)                             :482-488
 * then the energy tail (:494-672).  Structure factors and projectors are
 * rebuilt from the positions at the start of every call (ions fixed).
 */
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <math.h>
#include <cmath>
#include <vector>
#include <string>
#include <map>
#include <mutex>
#include <condition_variable>
#include <thread>
#include <algorithm>

#include "cpsd_internal.h"
#include "sd_kernels.h"
#include "../../include/cpsd_abi.h"

/* ---------------------------------------------------------- errors */

static char g_err[1024];
static int g_abort_on_error = 1;

void cpsd_set_error(const char *fmt, ...)
{
   va_list ap;
   va_start(ap, fmt);
   vsnprintf(g_err, sizeof g_err, fmt, ap);
   va_end(ap);
}

extern "C" const char *cpsd_last_error(void) { return g_err; }
extern "C" void cpsd_set_abort_on_error(int on) { g_abort_on_error = on; }

static void fail_loudly(const char *where)
{
   fprintf(stderr, "libcpsd_hip: %s: %s\n", where, g_err);
   fflush(stderr);
   if (g_abort_on_error) abort();
}

#define TRY(x) do { if ((x) != 0) return -1; } while (0)

/* ---------------------------------------------------------- context */

/* one phase per hot kernel where the bench reports a roofline for it;
 * the split-K reductions are phases of their own */
enum { PH_ZG2R, PH_DENSITY, PH_DNRED, PH_DNG, PH_VTOT, PH_VPSI, PH_ZR2G, PH_KBPROJ, PH_KBRED,
       PH_KBAPPLY, PH_GRAM, PH_GRAMRED, PH_LAGRANGE, PH_CONSTRAINT, PH_ENERGY, PH_FORCE, PH_PRECOND,
       PH_COUNT };
static const char *ph_names[PH_COUNT] = {
   "zpass_g2r", "plane_density", "dn_reduce_xc", "dng_r2c", "vtot_c2r", "plane_vpsi",
   "zpass_r2g_hpsi", "kb_projection", "kb_reduce", "kb_apply_sd", "gram", "gram_reduce",
   "lagrange", "constraint", "energy_tail", "ion_forces", "precondition"};

template<typename T>
static int dalloc(T **p, size_t n)
{
   *p = nullptr;
   if (n == 0) n = 1;
   CPSD_CHECK(hipMalloc((void **)p, n * sizeof(T)));
   return 0;
}

template<typename T>
static int h2d(T *d, const T *h, size_t n, hipStream_t s)
{
   CPSD_CHECK(hipMemcpyAsync(d, h, n * sizeof(T), hipMemcpyHostToDevice, s));
   return 0;
}

struct cpsd_dev {
   int n, nh, ne, nion, nkind, nproj, ng, ngp, nfft3d, n2ft3d, nyq, ncol, nsh;   /* ncol: columns of a plane of T */
   size_t n3;
   hipStream_t stream;
   /* packed-G tables */
   int *crows, *gmap, *gidx, *pidx, *kx, *ky, *kz;   /* crows, gmap: the columns of T (ColTable) */
   double2 *tw;
   double *w, *tg, *vc, *vg, *vl, *vnl, *pnrm, *zv, *unitg, *r1, *rcell;
   int *katm, *lmmax;
   double2 *ex1, *ex2, *ex3;
   /* state */
   double2 *Cbase, *CP;   /* Cbase: 2 orbital blocks */
   int cur;               /* C2 lives in block cur */
   double2 *T, *Tv;
   double *dnpart, *dn, *xcp, *xce, *V;
   int ndnblk[2], nob[2], fb;   /* density blocks of the FP64 [0] and FP32 [1] pass */
   int wgt;                     /* split-K workgroup target (launch plan) */
   size_t dnpart_cap;
   /* precision of the orbital transforms and KB products of every step but
    * the last of a call: 0 FP64; 1 FP32; 2 FP32 with a BF16-input KB
    * projection; 3 FP32 transforms with every product of the step (KB
    * projection and apply, preconditioned update, overlaps, constraint) in
    * split BF16 (the last step, which feeds the energy, is FP64) */
   int mixed;
   /* FP64 refresh period of the mixed modes: step k of the run (counted from
    * the last cpsd_dev_set_orbitals) is FP64 when (k + 1) % refresh == 0,
    * besides the last step of every call; 0: the last step of each call only */
   int refresh;
   long nstep;
   /* fallback: a call whose energy rises above the previous call's by more
    * than 1e-8 |E| while a mixed mode or a preconditioner is on turns both
    * off for the following calls (the reference's FP64 step) */
   int fallback_on, fallbacks, have_prevE;
   int poisoned;          /* a call produced non-finite values: clear the state first */
   int lag_itmax;         /* Lagrange iteration cap of the last step */
   double prevE, fallback_rise;
   float *Bf;             /* FP32 copy of the projectors B, [nproj][2 ngp] */
   int bf_valid;          /* Bf matches B */
   __bf16 *Bb;            /* BF16 copy of the projectors (mode 2) */
   int bb_valid;
   /* mode 3: the split-BF16 projectors, [nproj][2 ngp] (projection) and
    * transposed [2 ngp][npad] (apply), npad = nproj rounded up to 32; the
    * split X^T scratch of the apply, ne (npad + ne) each */
   __bf16 *BsH, *BsL, *BtH, *BtL, *XTh, *XTl;
   int bs_valid, npad;
   /* <c1|c1> of the next step, carried from this step's overlaps and lmd
    * (ne a multiple of 128): g11c[g11_idx] is valid when g11_valid */
   double *g11c[2], *g11w;
   double *DP;          /* preconditioned step: D = <c1|c2> - I, A11 D and D^T <c1|c2> */
   int g11_idx, g11_valid;
   /* mode 3: the FP32 steps form the overlaps from split-BF16 products of
    * their step d = c2 - c1 and the carried <c1|c1> (Gx: the reduced
    * products, ne x 2ne).  g11_drift: the carried <c1|c1> came from
    * such overlaps; an FP64 step after them forms the full Gram, which
    * returns the carried value to the FP64 one */
   int g11_drift;
   double *Gx;
   /* preconditioned step (cpsd_dev_set_preconditioner): one factor per
    * packed coefficient; the steps of a call use it when hml holds the
    * Lagrange matrix of the current orbitals' last energy evaluation */
   double *Kp;
   int precond, hml_valid;
   /* learned preconditioner: features of the packed G [ngp][4]; training
    * statistics against converged orbitals Cinf (Rh = C1 hml scratch) */
   float *Xf, *Pmlp;
   double2 *Cinf, *Rh;
   double *SA, *SB;
   int stats_on;          /* the energy evaluations accumulate SA, SB */
   long gram_wgs;         /* workgroups of the full Gram launch */
   /* HIP graphs of whole calls (inner steps + energy tail), keyed on what
    * the captured launches bake in; see ctx_run */
   int graphs;
   int ran_mode[4];       /* an eager call has run in this precision mode */
   /* a started call's results (E[0..11], Lagrange info, error flag) land in
    * pinned host memory; pending until cpsd_dev_run_finish */
   double *hout;
   int *herr;
   int pending;
   struct GraphEntry {
      int inner, mixed, cur0, g11i0, g11v0, pre, rk, rph;
      double dt, dte;
      int cur1, g11i1, g11v1;
      hipGraphExec_t exec;
   } gcache[8];
   int ngc;
   double2 *dng, *s, *vall, *B;
   double *partial; size_t partial_cap;
   double *Gm, *P, *Xkb, *s11, *s12, *s21, *s22, *LX, *st1, *lmd, *wgmax, *info, *hml, *Mh;
   unsigned *bar; int *err; int *flag;
   double *gsum_part, *xc_part, *orb_part, *ewald_part, *E;
   int ngsum_parts, nxc_parts, norb_parts;
   double2 *fullbuf;      /* ne * nfft3d staging of the reference layout */
   double *realbuf;       /* n2ft3d staging */
   int stager;            /* counted among the users of StageRings */
   double omega, cewald, rcut;
   int have_run;
   /* moving ions (move = 1): positions r2 after the step, forces, packed
    * Cartesian G, first projector of each ion, force partials; host copies
    * of katm and the per-kind masses for dt/sqrt(M) */
   int move;
   int struct_valid;      /* structure factors and projectors match r1 */
   double *r2d, *fion, *dti, *Gp, *fgpart, *fnlpart, *fnlsum;
   int *poff, fchunk;
   int *katm_h; double *amass_h;
   int *gidx_h;           /* grid index of each packed coefficient */
   double *Gp_h;
   /* profiling: event pairs recorded on the stream without synchronising;
    * they are resolved when the pool fills or the profile is read */
   int prof;
   hipEvent_t *pool;
   int *pool_ph;
   int pool_cap, pool_used;
   double prof_ms[PH_COUNT];
   int prof_calls[PH_COUNT];
   int last_lag_iters; double last_lag_adiff;
};

static int ph_flush(cpsd_dev *c)
{
   if (!c->pool_used) return 0;
   CPSD_CHECK(hipEventSynchronize(c->pool[2 * c->pool_used - 1]));
   for (int i = 0; i < c->pool_used; ++i) {
      float ms = 0.f;
      CPSD_CHECK(hipEventElapsedTime(&ms, c->pool[2 * i], c->pool[2 * i + 1]));
      c->prof_ms[c->pool_ph[i]] += ms;
      c->prof_calls[c->pool_ph[i]] += 1;
   }
   c->pool_used = 0;
   return 0;
}

static int ph_begin(cpsd_dev *c, int ph)
{
   (void)ph;
   if (c->prof) {
      if (c->pool_used == c->pool_cap) TRY(ph_flush(c));
      CPSD_CHECK(hipEventRecord(c->pool[2 * c->pool_used], c->stream));
   }
   return 0;
}

static int ph_end(cpsd_dev *c, int ph)
{
   if (c->prof) {
      CPSD_CHECK(hipEventRecord(c->pool[2 * c->pool_used + 1], c->stream));
      c->pool_ph[c->pool_used++] = ph;
   }
   return 0;
}

/* Pinned rings that the read-backs of all contexts share, one to a call at a
 * time: at most RINGS of 8 MB, and when the last context that has used one goes
 * they are given back but one.  That one stays because a ring takes up to 1.1 ms
 * to pin: made by each context's first call, a call of 11 MB took 1.5 ms where
 * the plain copy takes 0.7 and the ring 0.45. */
class StageRings {
public:
   enum { SLOTS = 4, RINGS = 4 };
   static constexpr size_t CHUNK = (size_t)2 << 20;
   struct Ring { char *mem; hipEvent_t ev[SLOTS]; int dev, busy; };

   static void join()
   {
      std::lock_guard<std::mutex> lk(mu);
      ++users;
   }
   static void leave()
   {
      std::lock_guard<std::mutex> lk(mu);
      if (--users > 0) return;
      bool kept = false;
      for (Ring &r : rings) {
         if (!r.mem) continue;
         r.busy = 0;   /* the streams of its calls are gone */
         if (!kept) { kept = true; continue; }
         for (hipEvent_t e : r.ev) (void)hipEventDestroy(e);
         (void)hipHostFree(r.mem);
         r.mem = nullptr;
      }
   }
   /* a ring for the device, or null */
   static Ring *take(int dev)
   {
      std::lock_guard<std::mutex> lk(mu);
      Ring *none = nullptr;
      for (Ring &r : rings) {
         if (r.mem && r.dev == dev && !r.busy) { r.busy = 1; return &r; }
         if (!r.mem && !none) none = &r;
      }
      if (!none || !make(none, dev)) return nullptr;
      none->busy = 1;
      return none;
   }
   static void give(Ring *r)
   {
      std::lock_guard<std::mutex> lk(mu);
      r->busy = 0;
   }

private:
   static bool make(Ring *r, int dev)
   {
      int n = 0;
      for (; n < SLOTS; ++n)
         if (hipEventCreateWithFlags(&r->ev[n], hipEventDisableTiming) != hipSuccess) break;
      void *p = nullptr;
      if (n == SLOTS && hipHostMalloc(&p, SLOTS * CHUNK, hipHostMallocPortable) == hipSuccess) {
         r->mem = static_cast<char *>(p);
         r->dev = dev;
         return true;
      }
      while (n > 0) (void)hipEventDestroy(r->ev[--n]);
      (void)hipGetLastError();
      return false;
   }
   static std::mutex mu;
   static Ring rings[RINGS];
   static int users;
};
std::mutex StageRings::mu;
StageRings::Ring StageRings::rings[StageRings::RINGS];
int StageRings::users = 0;

static void ctx_free(cpsd_dev *c)
{
   void *ptrs[] = {c->crows, c->gmap, c->gidx, c->pidx,
                   c->kx, c->ky, c->kz, c->tw, c->w, c->tg, c->vc, c->vg, c->vl, c->vnl, c->pnrm,
                   c->zv, c->unitg, c->r1, c->rcell, c->katm, c->lmmax, c->ex1, c->ex2, c->ex3,
                   c->Cbase, c->CP, c->T, c->Tv, c->dnpart, c->dn, c->xcp, c->xce, c->V, c->dng,
                   c->s, c->vall, c->B, c->partial, c->Gm, c->P, c->Xkb, c->s11, c->s12, c->s21,
                   c->s22, c->LX, c->st1, c->lmd, c->wgmax, c->info, c->hml, c->Mh, c->bar, c->err,
                   c->flag, c->gsum_part, c->xc_part, c->orb_part, c->ewald_part, c->E,
                   c->fullbuf, c->realbuf, c->r2d, c->fion, c->dti, c->Gp, c->fgpart,
                   c->fnlpart, c->fnlsum, c->poff, c->Bf, c->g11c[0], c->g11c[1], c->g11w, c->DP, c->Bb, c->Kp,
                   c->Gx, c->BsH, c->BsL, c->BtH, c->BtL, c->XTh, c->XTl, c->Xf, c->Pmlp, c->Cinf, c->Rh, c->SA, c->SB};
   for (void *p : ptrs)
      if (p) (void)hipFree(p);
   free(c->katm_h);
   free(c->amass_h);
   free(c->gidx_h);
   free(c->Gp_h);
   for (int i = 0; i < c->ngc; ++i) (void)hipGraphExecDestroy(c->gcache[i].exec);
   if (c->hout) (void)hipHostFree(c->hout);
   if (c->herr) (void)hipHostFree(c->herr);
   if (c->pool) {
      for (int i = 0; i < 2 * c->pool_cap; ++i) (void)hipEventDestroy(c->pool[i]);
      free(c->pool);
      free(c->pool_ph);
   }
   if (c->stream) (void)hipStreamDestroy(c->stream);
   if (c->stager) StageRings::leave();
   memset(c, 0, sizeof(*c));
}

int gemm_tn_tiles(int M, int N, int symm);

/* split-K count of a product: about wgt workgroups (the context's launch
 * plan, 2048 unless tuned) over its tiles */
static int splits_for_wgt(int wgt, int M, int N, size_t K, int symm)
{
   const int tiles = gemm_tn_tiles(M, N, symm);
   int sp = wgt / (tiles > 0 ? tiles : 1);
   const int maxsp = (int)(K / (16 * 8));
   if (sp > maxsp) sp = maxsp;
   if (sp > 256) sp = 256;
   if (sp < 1) sp = 1;
   return sp;
}

static int splits_for(const cpsd_dev *c, int M, int N, size_t K, int symm)
{
   return splits_for_wgt(c->wgt, M, N, K, symm);
}

/* The launch plan of a context: orbitals per FFT launch pair (fb), orbitals
 * per density partial plane of the FP64 and FP32 passes (nob; 0: as the
 * workgroup slots of plane_density_occupancy, a table that stands for the
 * rounding of the density sum and no longer counts what a CU holds, are best
 * filled) and the
 * split-K workgroup target of the small-output products (wgt).  The
 * buffers whose sizes depend on it (density partials, split-K partials)
 * grow as needed; graphs captured before are dropped. */
static int ctx_plan(cpsd_dev *c, int fb, const int *nob_req, int wgt)
{
   const int n = c->n, ne = c->ne, nproj = c->nproj;
   c->fb = fb < 1 ? 1 : (fb > ne ? ne : fb);
   c->wgt = wgt;
   int dev = 0, cus = 0;
   CPSD_CHECK(hipGetDevice(&dev));
   CPSD_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
   for (int f = 0; f < 2; ++f) {
      if (nob_req && nob_req[f] > 0) {
         c->nob[f] = nob_req[f] < c->fb ? nob_req[f] : c->fb;
      } else {
         const long slots = (long)(cus > 0 ? cus : 1) * plane_density_occupancy(n, f);
         int best = 1;
         double beff = -1.0;
         for (int d = 1; d <= (c->fb < 32 ? c->fb : 32); ++d) {
            const int nob = (c->fb + d - 1) / d, dd = (c->fb + nob - 1) / nob;
            const long wgs = (long)n * dd;
            const double eff = (double)wgs / ((double)slots * (double)((wgs + slots - 1) / slots));
            if (eff >= 0.9) { best = dd; break; }
            if (eff > beff + 1e-12) { beff = eff; best = dd; }
         }
         const char *env = getenv("CPSD_DN_BLOCKS");   /* tuning override */
         if (env && atoi(env) > 0) best = atoi(env) < c->fb ? atoi(env) : c->fb;
         c->nob[f] = (c->fb + best - 1) / best;
      }
      c->ndnblk[f] = (c->fb + c->nob[f] - 1) / c->nob[f];
   }
   const size_t dnp = (size_t)(c->ndnblk[0] > c->ndnblk[1] ? c->ndnblk[0] : c->ndnblk[1]) * c->n3;
   if (dnp > c->dnpart_cap) {
      if (c->dnpart) (void)hipFree(c->dnpart);
      c->dnpart = nullptr;
      TRY(dalloc(&c->dnpart, dnp));
      c->dnpart_cap = dnp;
   }
   const size_t K = 2 * (size_t)c->ngp;
   size_t cap = 0;
   int sp = splits_for(c, 2 * ne, 2 * ne, K, 1), so, sd;
   gemm_tn_symm_splits(2 * ne, K, sp, &so, &sd);
   cap = (size_t)(so > sd ? so : sd) * 4 * ne * ne;
   sp = splits_for(c, ne, ne, K, 1);   /* the epilogue's Gram of c1 */
   gemm_tn_symm_splits(ne, K, sp, &so, &sd);
   if ((size_t)(so > sd ? so : sd) * ne * ne > cap) cap = (size_t)(so > sd ? so : sd) * ne * ne;
   sp = splits_for(c, nproj, ne, K, 0);
   if ((size_t)sp * nproj * ne > cap) cap = (size_t)sp * nproj * ne;
   /* the Gram without its C1 x C1 block (ne a multiple of 128): the same
    * number of workgroups over the tiles that touch C2 */
   c->gram_wgs = (long)gemm_tn_tiles(2 * ne, 2 * ne, 1) * splits_for(c, 2 * ne, 2 * ne, K, 1);
   if (ne % 128 == 0 && ne <= 512) {
      const int q = ne / 128, nt = 2 * q;
      int so2, sd2;
      gemm_tn_list_splits(nt * (nt - 1) / 2 - q * (q - 1) / 2, q, K, c->gram_wgs, &so2, &sd2);
      const size_t z = (size_t)(so2 > 2 * sd2 ? so2 : 2 * sd2);
      if (z * 4 * ne * ne > cap) cap = z * 4 * ne * ne;
   }
   sp = splits_for(c, ne, ne, K, 0);
   if ((size_t)sp * ne * ne > cap) cap = (size_t)sp * ne * ne;
   if (cap > c->partial_cap) {
      if (c->partial) (void)hipFree(c->partial);
      c->partial = nullptr;
      TRY(dalloc(&c->partial, cap));
      c->partial_cap = cap;
   }
   for (int i = 0; i < c->ngc; ++i) (void)hipGraphExecDestroy(c->gcache[i].exec);
   c->ngc = 0;
   return 0;
}

static int ctx_build(cpsd_dev *c, int nfft, int ne, int nion, const int *katm, const double *zv,
                     const int *lmmax, const double *vnlnrm, const double *vl, const double *vnl,
                     const int *masker, const double *tg, const double *vc, const double *vg,
                     const double *unitg, double omega, int nsh, const double *rcell,
                     double cewald, double rcut, const double *r)
{
   if (!fft_supported(nfft)) { cpsd_set_error("FFT grid %d is not supported", nfft); return -1; }
   if (ne < 1 || nion < 1) { cpsd_set_error("need ne >= 1 and nion >= 1 (ne=%d nion=%d)", ne, nion); return -1; }
   if (ne > 512) { cpsd_set_error("ne=%d above 512 is not supported", ne); return -1; }
   const int n = nfft, nh = n / 2 + 1;
   c->n = n; c->nh = nh; c->ne = ne; c->nion = nion; c->nsh = nsh;
   c->nfft3d = nh * n * n; c->n2ft3d = (n + 2) * n * n; c->n3 = (size_t)n * n * n;
   c->omega = omega; c->cewald = cewald; c->rcut = rcut;
   int nkind = 0;
   for (int i = 0; i < nion; ++i) {
      if (katm[i] < 0) { cpsd_set_error("katm[%d]=%d is negative", i, katm[i]); return -1; }
      if (katm[i] + 1 > nkind) nkind = katm[i] + 1;
   }
   c->nkind = nkind;
   int nproj = 0;
   for (int i = 0; i < nion; ++i) {
      const int lm = lmmax[katm[i]];
      if (lm < 0 || lm > 9) { cpsd_set_error("lmmax=%d out of range", lm); return -1; }
      nproj += lm;
   }
   c->nproj = nproj;
   std::vector<int> poff(nion);
   for (int i = 0, m = 0; i < nion; ++i) { poff[i] = m; m += lmmax[katm[i]]; }

   /* masked rows: each (ky,kz) row must hold one contiguous kx interval */
   std::vector<int> clen(n, 0), pidx(c->nfft3d, -1);
   std::vector<int> gidx, kxv, kyv, kzv;
   int ng = 0;
   for (int kz = 0; kz < n; ++kz)
      for (int ky = 0; ky < n; ++ky) {
         const int r = ky + n * kz;
         int first = -1, last = -1;
         for (int kx = 0; kx < nh; ++kx) {
            const int g = kx + nh * r;
            const int m0 = masker[2 * g], m1 = masker[2 * g + 1];
            if (m0 != m1 || (m0 != 0 && m0 != 1)) {
               cpsd_set_error("masker must be 0/1 and equal on re/im (entry %d)", g);
               return -1;
            }
            if (m0) {
               if (first < 0) first = kx;
               else if (last != kx - 1) { cpsd_set_error("mask row %d is not an interval", r); return -1; }
               last = kx;
            }
         }
         if (first < 0) continue;
         for (int kx = first; kx <= last; ++kx) {
            pidx[kx + nh * r] = ng++;
            gidx.push_back(kx + nh * r);
            kxv.push_back(kx); kyv.push_back(ky); kzv.push_back(kz);
         }
         if (last + 1 > clen[ky]) clen[ky] = last + 1;
      }
   if (ng == 0) { cpsd_set_error("empty mask"); return -1; }
   c->ng = ng;
   c->ngp = (ng + 63) / 64 * 64;
   /* columns of T: row ky holds kx < clen[ky], rows padded to 8 columns */
   std::vector<int> crows(n);
   c->ncol = 0;
   c->nyq = 0;
   for (int ky = 0; ky < n; ++ky) {
      crows[ky] = clen[ky] << 16 | c->ncol;
      c->ncol += (clen[ky] + 7) / 8 * 8;
      if (clen[ky] == nh) c->nyq = 1;
   }
   const int ngp = c->ngp;
   for (int p = ng; p < ngp; ++p) { gidx.push_back(0); kxv.push_back(0); kyv.push_back(0); kzv.push_back(0); }

   std::vector<double2> tw(n);
   for (int m = 0; m < n; ++m) {
      const double a = 2.0 * M_PI * (double)m / (double)n;
      tw[m] = make_double2(cos(a), sin(a));
   }
   std::vector<double> w(2 * (size_t)ngp, 0.0), tgp(ngp, 0.0), vcp(ngp, 0.0), vgp(ngp, 0.0);
   std::vector<double> vlp((size_t)nkind * ngp, 0.0), vnlp((size_t)nkind * 9 * ngp, 0.0);
   for (int p = 0; p < ng; ++p) {
      const int g = gidx[p];
      const double wp = (kxv[p] == 0) ? 1.0 : 2.0;
      w[2 * p] = w[2 * p + 1] = wp;
      tgp[p] = tg[g]; vcp[p] = vc[g]; vgp[p] = vg[g];
      for (int k = 0; k < nkind; ++k) {
         vlp[(size_t)k * ngp + p] = vl[(size_t)k * c->nfft3d + g];
         for (int l = 0; l < lmmax[k]; ++l)
            vnlp[((size_t)k * 9 + l) * ngp + p] = vnl[((size_t)k * 9 + l) * c->nfft3d + g];
      }
   }
   std::vector<double> pnrm(nproj > 0 ? nproj : 1);
   {
      int m = 0;
      for (int i = 0; i < nion; ++i)
         for (int l = 0; l < lmmax[katm[i]]; ++l) pnrm[m++] = vnlnrm[katm[i] * 9 + l];
   }

   CPSD_CHECK(hipStreamCreate(&c->stream));
   CPSD_CHECK(hipHostMalloc((void **)&c->hout, 16 * sizeof(double), hipHostMallocDefault));
   CPSD_CHECK(hipHostMalloc((void **)&c->herr, sizeof(int), hipHostMallocDefault));
   hipStream_t st = c->stream;
   TRY(dalloc(&c->crows, n)); TRY(dalloc(&c->gmap, (size_t)n * c->ncol));
   TRY(dalloc(&c->gidx, ngp)); TRY(dalloc(&c->pidx, c->nfft3d));
   TRY(dalloc(&c->kx, ngp)); TRY(dalloc(&c->ky, ngp)); TRY(dalloc(&c->kz, ngp));
   TRY(dalloc(&c->tw, n)); TRY(dalloc(&c->w, 2 * (size_t)ngp));
   TRY(dalloc(&c->tg, ngp)); TRY(dalloc(&c->vc, ngp)); TRY(dalloc(&c->vg, ngp));
   TRY(dalloc(&c->vl, (size_t)nkind * ngp)); TRY(dalloc(&c->vnl, (size_t)nkind * 9 * ngp));
   TRY(dalloc(&c->pnrm, pnrm.size())); TRY(dalloc(&c->zv, nkind)); TRY(dalloc(&c->unitg, 9));
   TRY(dalloc(&c->r1, 3 * (size_t)nion)); TRY(dalloc(&c->rcell, 3 * (size_t)nsh));
   TRY(dalloc(&c->katm, nion)); TRY(dalloc(&c->lmmax, nkind));
   TRY(dalloc(&c->ex1, (size_t)nion * nh)); TRY(dalloc(&c->ex2, (size_t)nion * n));
   TRY(dalloc(&c->ex3, (size_t)nion * n));
   TRY(h2d(c->crows, crows.data(), n, st));
   TRY(h2d(c->gidx, gidx.data(), ngp, st)); TRY(h2d(c->pidx, pidx.data(), c->nfft3d, st));
   TRY(sd_gmap(n, c->crows, c->pidx, c->ncol, c->gmap, st));
   TRY(h2d(c->kx, kxv.data(), ngp, st)); TRY(h2d(c->ky, kyv.data(), ngp, st));
   TRY(h2d(c->kz, kzv.data(), ngp, st));
   TRY(h2d(c->tw, tw.data(), n, st)); TRY(h2d(c->w, w.data(), w.size(), st));
   TRY(h2d(c->tg, tgp.data(), ngp, st)); TRY(h2d(c->vc, vcp.data(), ngp, st));
   TRY(h2d(c->vg, vgp.data(), ngp, st));
   TRY(h2d(c->vl, vlp.data(), vlp.size(), st)); TRY(h2d(c->vnl, vnlp.data(), vnlp.size(), st));
   TRY(h2d(c->pnrm, pnrm.data(), pnrm.size(), st)); TRY(h2d(c->zv, zv, nkind, st));
   TRY(h2d(c->unitg, unitg, 9, st)); TRY(h2d(c->r1, r, 3 * (size_t)nion, st));
   TRY(h2d(c->rcell, rcell, 3 * (size_t)nsh, st));
   TRY(h2d(c->katm, katm, nion, st)); TRY(h2d(c->lmmax, lmmax, nkind, st));
   TRY(dalloc(&c->poff, nion)); TRY(h2d(c->poff, poff.data(), nion, st));
   c->gidx_h = (int *)malloc((size_t)ngp * sizeof(int));
   if (!c->gidx_h) { cpsd_set_error("host allocation failed"); return -1; }
   memcpy(c->gidx_h, gidx.data(), (size_t)ngp * sizeof(int));
   c->katm_h = (int *)malloc((size_t)nion * sizeof(int));
   c->Gp_h = (double *)calloc(3 * (size_t)ngp, sizeof(double));
   if (!c->katm_h || !c->Gp_h) { cpsd_set_error("host allocation failed"); return -1; }
   memcpy(c->katm_h, katm, (size_t)nion * sizeof(int));
   /* Cartesian G of the packed entries, the expression of ccpsdv3/get_g.c:
    * k1 b1 + k2 b2 + k3 b3 with ky, kz taken back to (-N/2, N/2] */
   for (int p = 0; p < c->ng; ++p) {
      const int k1 = kxv[p];
      const int k2 = kyv[p] <= n / 2 ? kyv[p] : kyv[p] - n;
      const int k3 = kzv[p] <= n / 2 ? kzv[p] : kzv[p] - n;
      for (int d = 0; d < 3; ++d)
         c->Gp_h[(size_t)d * ngp + p] = k1 * unitg[d] + k2 * unitg[3 + d] + k3 * unitg[6 + d];
   }

   /* state and scratch */
   const size_t orb = (size_t)ne * ngp;
   TRY(dalloc(&c->Cbase, 2 * orb)); TRY(dalloc(&c->CP, orb));
   CPSD_CHECK(hipMemsetAsync(c->Cbase, 0, 2 * orb * sizeof(double2), st));
   CPSD_CHECK(hipMemsetAsync(c->CP, 0, orb * sizeof(double2), st));
   const size_t plane = (size_t)n * c->ncol;
   TRY(dalloc(&c->T, (size_t)ne * plane)); TRY(dalloc(&c->Tv, plane));
   /* launch plan: all orbitals per FFT launch pair by default
    * (CPSD_FFT_BATCH sets fewer, whose z-transformed planes then stay in the
    * Infinity Cache between the two launches), density blocks that fill the
    * GPU, 2048 split-K workgroups; cpsd_dev_autotune measures others */
   {
      long fb = ne;
      const char *env = getenv("CPSD_FFT_BATCH");
      if (env && atol(env) > 0) fb = atol(env);
      c->wgt = 2048;
      c->dnpart_cap = 0;
      c->partial_cap = 0;
      const size_t bsz = (size_t)(nproj > 0 ? nproj : 1) * ngp;
      TRY(dalloc(&c->B, bsz));
      TRY(ctx_plan(c, (int)(fb > ne ? ne : fb), nullptr, 2048));
   }
   TRY(dalloc(&c->dn, c->n3)); TRY(dalloc(&c->xcp, c->n3)); TRY(dalloc(&c->xce, c->n3));
   TRY(dalloc(&c->V, c->n3));
   TRY(dalloc(&c->dng, ngp)); TRY(dalloc(&c->s, ngp)); TRY(dalloc(&c->vall, ngp));
   /* the packed tail p >= ng is never written by the kernels: keep it zero */
   CPSD_CHECK(hipMemsetAsync(c->dng, 0, ngp * sizeof(double2), st));
   const size_t ee = (size_t)ne * ne;
   TRY(dalloc(&c->Gm, 4 * ee));
   if (ne % 128 == 0 && ne <= 512) {
      TRY(dalloc(&c->g11c[0], ee)); TRY(dalloc(&c->g11c[1], ee)); TRY(dalloc(&c->g11w, 2 * ee));
   }
   TRY(dalloc(&c->DP, 3 * ee));
   TRY(dalloc(&c->P, (size_t)(nproj > 0 ? nproj : 1) * ne));
   TRY(dalloc(&c->Xkb, (size_t)(nproj > 0 ? nproj : 1) * ne));
   TRY(dalloc(&c->s11, ee)); TRY(dalloc(&c->s12, ee)); TRY(dalloc(&c->s21, ee)); TRY(dalloc(&c->s22, ee));
   TRY(dalloc(&c->LX, 2 * ee)); TRY(dalloc(&c->st1, ee)); TRY(dalloc(&c->lmd, ee));
   TRY(dalloc(&c->wgmax, 1024)); TRY(dalloc(&c->info, 4)); TRY(dalloc(&c->hml, ee)); TRY(dalloc(&c->Mh, ee));
   TRY(dalloc(&c->bar, 4)); TRY(dalloc(&c->err, 4)); TRY(dalloc(&c->flag, 4));
   c->ngsum_parts = 256; c->nxc_parts = 256; c->norb_parts = 32;
   TRY(dalloc(&c->gsum_part, 3 * (size_t)c->ngsum_parts));
   TRY(dalloc(&c->xc_part, 2 * (size_t)c->nxc_parts));
   TRY(dalloc(&c->orb_part, 2 * (size_t)c->norb_parts * ne));
   TRY(dalloc(&c->ewald_part, (size_t)nion * nion)); TRY(dalloc(&c->E, 16));
   TRY(dalloc(&c->fullbuf, (size_t)ne * c->nfft3d));
   TRY(dalloc(&c->realbuf, c->n2ft3d));
   CPSD_CHECK(hipMemsetAsync(c->err, 0, 4 * sizeof(int), st));
   CPSD_CHECK(hipStreamSynchronize(st));
   c->cur = 0;
   return 0;
}

/* ---------------------------------------------------------- one step */

static ColTable col_table(const cpsd_dev *c)
{
   ColTable t;
   t.rows = c->crows; t.gmap = c->gmap; t.P = c->ncol; t.nyq = c->nyq;
   return t;
}

static ZArgs zargs_base(const cpsd_dev *c)
{
   ZArgs z;
   memset(&z, 0, sizeof z);
   z.cols = col_table(c);
   z.tw = c->tw;
   return z;
}

static PlaneArgs pargs_base(const cpsd_dev *c)
{
   PlaneArgs pa;
   memset(&pa, 0, sizeof pa);
   pa.cols = col_table(c);
   pa.tw = c->tw;
   return pa;
}

static int run_structure(cpsd_dev *c)
{
   hipStream_t st = c->stream;
   TRY(sd_phafac(c->n, c->unitg, c->nion, c->r1, c->ex1, c->ex2, c->ex3, st));
   StructArgs a;
   a.n = c->n; a.ng = c->ng; a.ngp = c->ngp; a.nion = c->nion; a.nproj = c->nproj;
   a.kx = c->kx; a.ky = c->ky; a.kz = c->kz;
   a.ex1 = c->ex1; a.ex2 = c->ex2; a.ex3 = c->ex3;
   a.katm = c->katm; a.lmmax = c->lmmax; a.poff = c->poff; a.zv = c->zv; a.vl = c->vl; a.vnl = c->vnl;
   a.s = c->s; a.vall = c->vall; a.B = c->B;
   TRY(sd_structure(a, st));
   c->bf_valid = 0;
   c->bb_valid = 0;
   c->bs_valid = 0;
   return 0;
}

/* the BF16 projectors of mode 2's projection */
static int ensure_bb(cpsd_dev *c)
{
   const size_t n = (size_t)c->nproj * 2 * c->ngp;
   if (!c->Bb) TRY(dalloc(&c->Bb, n));
   if (!c->bb_valid) {
      TRY(launch_to_bf16(reinterpret_cast<const double *>(c->B), c->Bb, n, c->stream));
      c->bb_valid = 1;
   }
   return 0;
}

/* the split-BF16 projectors of mode 3: rows for the projection, transposed
 * for the apply */
static int ensure_bs(cpsd_dev *c)
{
   const size_t K = 2 * (size_t)c->ngp, n = (size_t)c->nproj * K;
   c->npad = (c->nproj + 31) / 32 * 32;
   if (c->nproj > 0 && !c->BsH) {
      TRY(dalloc(&c->BsH, n)); TRY(dalloc(&c->BsL, n));
      TRY(dalloc(&c->BtH, K * c->npad)); TRY(dalloc(&c->BtL, K * c->npad));
   }
   if (!c->bs_valid && c->nproj > 0) {
      TRY(launch_to_bf16x2(reinterpret_cast<const double *>(c->B), c->BsH, c->BsL, n, c->stream));
      TRY(launch_split_bt(reinterpret_cast<const double *>(c->B), c->nproj, c->npad, K, c->BtH, c->BtL,
                          c->stream));
   }
   c->bs_valid = 1;
   return 0;
}

/* the FP32 projectors of the FP32 KB products, made when first needed
 * after the projectors change */
static int ensure_bf(cpsd_dev *c)
{
   const size_t n = (size_t)c->nproj * 2 * c->ngp;
   if (!c->Bf) TRY(dalloc(&c->Bf, n));
   if (!c->bf_valid) {
      TRY(launch_to_f32(reinterpret_cast<const double *>(c->B), c->Bf, n, c->stream));
      c->bf_valid = 1;
   }
   return 0;
}

/* step `it` of the call about to run is an FP64 refresh step of the mixed
 * modes */
static int refresh_step(const cpsd_dev *c, int it)
{
   return c->refresh > 0 && (c->nstep + it + 1) % c->refresh == 0;
}

static int sd_step(cpsd_dev *c, double dte, int last, int fp64)
{
   hipStream_t st = c->stream;
   const int n = c->n, ne = c->ne, ngp = c->ngp;
   const size_t orb = (size_t)ne * ngp;
   const size_t K = 2 * (size_t)ngp;
   const double scal1 = 1.0 / ((double)n * n * n), scal2 = 1.0 / c->omega;
   double2 *C1 = c->Cbase + (size_t)c->cur * orb;          /* previous C2 */
   double2 *C2 = c->Cbase + (size_t)(c->cur ^ 1) * orb;

   /* moving ions: r1 <- r2 (ccpsdv3/cpsd.c:174), then phase factors,
    * structure factor, local potential and projectors at the new r1 */
   if (c->move) {
      CPSD_CHECK(hipMemcpyAsync(c->r1, c->r2d, 3 * (size_t)c->nion * sizeof(double),
                                hipMemcpyDeviceToDevice, st));
      TRY(ph_begin(c, PH_FORCE));
      TRY(run_structure(c));
      TRY(ph_end(c, PH_FORCE));
   }

   ZArgs z;
   PlaneArgs pa;
   const size_t plane = (size_t)n * c->ncol;
   const int f32 = c->mixed && !last && !fp64;
   /* 2-3: orbitals in batches of fb, so that each batch's z-transformed
    * planes are read by the density pass while they sit in the Infinity
    * Cache; T keeps every orbital for the V*psi pass */
   for (int b0 = 0; b0 < ne; b0 += c->fb) {
      const int bs = ne - b0 < c->fb ? ne - b0 : c->fb;
      TRY(ph_begin(c, PH_ZG2R));
      z = zargs_base(c);
      z.src = C1 + (size_t)b0 * ngp; z.sstride = ngp; z.T = c->T + (size_t)b0 * plane;
      z.fp32 = f32;
      TRY(launch_zpass_g2r(n, z, bs, st));
      TRY(ph_end(c, PH_ZG2R));
      TRY(ph_begin(c, PH_DENSITY));
      pa = pargs_base(c);
      pa.T = c->T + (size_t)b0 * plane;
      pa.nb = c->nob[f32]; pa.nbatch = bs; pa.dnpart = c->dnpart; pa.accumulate = b0 > 0;
      pa.fp32 = f32;
      TRY(launch_plane(n, PM_DENSITY, pa, (bs + c->nob[f32] - 1) / c->nob[f32], st));
      TRY(ph_end(c, PH_DENSITY));
   }
   /* 4 */
   TRY(ph_begin(c, PH_DNRED));
   TRY(sd_dn_reduce_xc(c->dnpart, c->ndnblk[f32], c->n3, scal2, c->dn, c->xcp, c->xce, st));
   TRY(ph_end(c, PH_DNRED));
   /* 5, and the z transform of 6 */
   TRY(ph_begin(c, PH_DNG));
   pa = pargs_base(c);
   pa.T = c->Tv; pa.dn = c->dn; pa.scal1 = scal1; pa.nbatch = 1;
   TRY(launch_plane(n, PM_R2C_DN, pa, 1, st));
   z = zargs_base(c);
   z.T = c->Tv; z.out = c->dng; z.ostride = ngp; z.vall = c->vall; z.vc = c->vc; z.scal2 = scal2;
   TRY(launch_zpass_field(n, z, st));
   TRY(ph_end(c, PH_DNG));
   if (c->move) {
      TRY(ph_begin(c, PH_FORCE));
      ForceArgs f;
      f.n = n; f.ng = c->ng; f.ngp = ngp; f.nion = c->nion; f.nchunk = c->fchunk;
      f.kx = c->kx; f.ky = c->ky; f.kz = c->kz; f.ex1 = c->ex1; f.ex2 = c->ex2; f.ex3 = c->ex3;
      f.katm = c->katm; f.zv = c->zv; f.vl = c->vl; f.vg = c->vg; f.w = c->w; f.Gp = c->Gp;
      f.dng = c->dng; f.s = c->s; f.scal2 = scal2; f.part = c->fgpart;
      TRY(sd_force_gspace(f, st));
      TRY(ph_end(c, PH_FORCE));
   }
   /* 6 */
   TRY(ph_begin(c, PH_VTOT));
   pa = pargs_base(c);
   pa.T = c->Tv; pa.Vout = c->V; pa.xcp = c->xcp; pa.nbatch = 1;
   TRY(launch_plane(n, PM_VTOT, pa, 1, st));
   TRY(ph_end(c, PH_VTOT));
   /* 7-8, batched the same way: the z pass reads what the plane pass wrote */
   for (int b0 = 0; b0 < ne; b0 += c->fb) {
      const int bs = ne - b0 < c->fb ? ne - b0 : c->fb;
      TRY(ph_begin(c, PH_VPSI));
      pa = pargs_base(c);
      pa.T = c->T + (size_t)b0 * plane; pa.V = c->V;
      pa.nbatch = bs; pa.fp32 = f32;
      pa.nb = plane_orbitals(n, (long)bs * n);
      TRY(launch_plane(n, PM_VPSI, pa, (bs + pa.nb - 1) / pa.nb, st));
      TRY(ph_end(c, PH_VPSI));
      TRY(ph_begin(c, PH_ZR2G));
      z = zargs_base(c);
      /* -H psi (local part) is kept only on the last step, for the energy
       * tail; the other steps write c1 + dte (local -H psi) straight into c2
       * and the KB apply adds dte times the nonlocal part in place */
      z.T = c->T + (size_t)b0 * plane; z.ostride = ngp;
      z.out = (last ? c->CP : C2) + (size_t)b0 * ngp;
      z.c1 = C1 + (size_t)b0 * ngp; z.tg = c->tg; z.scal1 = scal1; z.dte = dte;
      z.fp32 = f32;
      TRY(launch_zpass_r2g(n, last ? DST_HPSI : DST_SD, z, bs, st));
      TRY(ph_end(c, PH_ZR2G));
   }
   /* 9 */
   const double *A2 = reinterpret_cast<const double *>(C1);
   /* mode 3: every product of an FP32 step in split BF16 (ne 128 or 256) */
   const int sb = f32 && c->mixed == 3;
   if (c->nproj > 0) {
      TRY(ph_begin(c, PH_KBPROJ));
      const int sp = splits_for(c, c->nproj, ne, K, 0);
      const int small = gemm_tn_small_ok(c->nproj, ne);
      if (f32 && c->mixed != 3) TRY(ensure_bf(c));
      if (f32 && c->mixed == 2) TRY(ensure_bb(c));
      if (sb) TRY(ensure_bs(c));
      if (small) {
         TRY(launch_gemm_tn_small(reinterpret_cast<const double *>(c->B), K, c->nproj, A2, K, ne, c->w, K, 0,
                                  c->P, c->pnrm, scal2, c->Xkb, st));
      } else if (sb) {
         TRY(launch_kbproj_dbf16(c->BsH, c->BsL, c->nproj, A2, ne, c->w, K, sp, c->partial, c->partial_cap, st));
      } else if (f32 && c->mixed == 2) {
         TRY(launch_kbproj_bf16(c->Bb, c->nproj, A2, ne, c->w, K, sp, c->partial, c->partial_cap, st));
      } else if (f32) {
         TRY(launch_kbproj_f32(c->Bf, c->nproj, A2, ne, c->w, K, sp, c->partial, c->partial_cap, st));
      } else {
         TRY(launch_gemm_tn_splitk(reinterpret_cast<const double *>(c->B), K, c->nproj, A2, K, ne, c->w, K,
                                   sp, 0, c->partial, st));
      }
      TRY(ph_end(c, PH_KBPROJ));
      TRY(ph_begin(c, PH_KBRED));
      if (!small) TRY(launch_reduce_partials_kb(c->partial, sp, c->nproj, ne, c->P, c->pnrm, scal2, c->Xkb, st));
      TRY(ph_end(c, PH_KBRED));
   }
   if (c->move) {
      TRY(ph_begin(c, PH_FORCE));
      if (c->nproj > 0) {
         /* Z_p = sum_i sw_pi c1_i, reduced against beta_p in the epilogue */
         TallArgs t;
         t.A = A2; t.lda = K; t.X = c->Xkb; t.xsm = c->nproj; t.ldx = 1;
         t.Mr = ne; t.Nc = c->nproj; t.K = K;
         t.C2 = nullptr; t.C1 = nullptr; t.CP = nullptr; t.ldc = K; t.dte = 0.0; t.write_cp = 0;
         t.Bp = c->B; t.w = c->w; t.Gp = c->Gp; t.ngp = ngp; t.fpart = c->fnlpart;
         TRY(launch_gemm_tall(EPI_NLFORCE, t, st));
         TRY(sd_force_nlsum(c->fnlpart, (int)(K / 128), c->nproj, c->fnlsum, st));
      }
      ForceFinishArgs f;
      f.nion = c->nion; f.nchunk = c->fchunk; f.nsh = c->nsh;
      f.katm = c->katm; f.lmmax = c->lmmax; f.poff = c->poff;
      f.zv = c->zv; f.rcell = c->rcell; f.r1 = c->r1; f.dti = c->dti; f.rcut = c->rcut;
      f.gpart = c->fgpart; f.nlsum = c->fnlsum; f.fion = c->fion; f.r2 = c->r2d;
      TRY(sd_force_finish(f, st));
      TRY(ph_end(c, PH_FORCE));
   }
   /* 10 */
   const int pstep = c->precond && c->hml_valid;
   /* an FP32 preconditioned step does its KB apply inside the preconditioned
    * update (10b): one pass over C2 */
   const int fused = pstep && f32 && c->nproj > 0;
   TRY(ph_begin(c, PH_KBAPPLY));
   if (fused || (sb && pstep)) {
      /* nothing here */
   } else if (sb && c->nproj > 0) {
      TRY(launch_apply_dbf16(c->BtH, c->BtL, c->npad, c->Xkb, c->nproj, c->nproj, nullptr, 0, nullptr, 0, ne, K,
                             reinterpret_cast<double *>(C2), dte, nullptr, 0, c->XTh, c->XTl, st));
   } else if (f32 && c->nproj > 0) {
      /* C2 += dte B X with FP32 products (never the last step) */
      TRY(launch_kbapply_f32(c->Bf, c->nproj, c->Xkb, 1, c->nproj, ne, K, reinterpret_cast<double *>(C2), K,
                             dte, st));
   } else if (last || c->nproj > 0) {
      TallArgs t;
      t.A = reinterpret_cast<const double *>(c->B); t.lda = K;
      t.X = c->Xkb; t.ldx = c->nproj; t.Mr = c->nproj; t.Nc = ne; t.K = K;
      t.C2 = reinterpret_cast<double *>(C2); t.C1 = reinterpret_cast<const double *>(C1);
      t.CP = reinterpret_cast<double *>(c->CP); t.ldc = K; t.dte = dte; t.write_cp = last;
      /* last step: CP += B X, C2 = C1 + dte CP; otherwise C2 += dte B X */
      TRY(launch_gemm_tall(last ? EPI_KBAPPLY : EPI_CONSTRAINT, t, st));
   }
   TRY(ph_end(c, PH_KBAPPLY));
   /* 10b: the preconditioned step.  C2 holds c1 + dte cpsi; it becomes
    * c1 + K o dte (cpsi + c1 h), the per-G scaled residual, with h the
    * Lagrange matrix hml of the last energy evaluation (exact at the fixed
    * point, where h = <c1|H|c1>).  The overlaps below take this c2's
    * component along c1 out first (sd_smat_precond), and the constraint
    * adds it back through lmd = X - D/dte (sd_precond_lmd). */
   if (sb && pstep) {
      /* mode 3: B X + C1 h in split BF16, one pass */
      TRY(ph_begin(c, PH_PRECOND));
      TRY(launch_apply_dbf16(c->BtH, c->BtL, c->nproj > 0 ? c->npad : 0, c->Xkb, c->nproj, c->nproj, A2, ne,
                             c->hml, ne, ne, K, reinterpret_cast<double *>(C2), dte, c->Kp, 1, c->XTh, c->XTl,
                             st));
      TRY(ph_end(c, PH_PRECOND));
   } else if (fused) {
      /* the FP32 steps of the mixed modes form C1 h in FP32 as well, like
       * their FFTs and KB products, summed with B X in one pass; the update
       * itself is FP64 */
      TRY(ph_begin(c, PH_PRECOND));
      TRY(launch_kbapply_precond_f32(c->Bf, c->nproj, c->Xkb, A2, ne, c->hml, K, reinterpret_cast<double *>(C2),
                                     dte, c->Kp, st));
      TRY(ph_end(c, PH_PRECOND));
   } else if (pstep && f32) {
      TRY(ph_begin(c, PH_PRECOND));
      TRY(launch_precond_f32(A2, ne, c->hml, K, reinterpret_cast<double *>(C2), dte, c->Kp, st));
      TRY(ph_end(c, PH_PRECOND));
   } else if (pstep) {
      TRY(ph_begin(c, PH_PRECOND));
      TallArgs t;
      t.A = A2; t.lda = K; t.X = c->hml; t.xsm = 1; t.ldx = ne; t.Mr = ne; t.Nc = ne; t.K = K;
      t.C2 = reinterpret_cast<double *>(C2); t.C1 = reinterpret_cast<const double *>(C1); t.CP = nullptr;
      t.ldc = K; t.dte = dte; t.write_cp = 0; t.Kp = c->Kp;
      TRY(launch_gemm_tall(EPI_PRECOND, t, st));
      TRY(ph_end(c, PH_PRECOND));
   }
   /* 11 */
   /* with <c1|c1> carried from the previous step, the Gram skips its C1 x C1
    * block (whose reduced entries are then not read); an FP32 step of mode 3
    * forms the products of its step d = c2 - c1 only */
   const int dgram = sb && c->g11_valid;
   const int carry = c->g11_valid && (dgram || !c->g11_drift);
   const int one = !pstep && lagrange_one(ne);   /* the Lagrange kernel forms the s matrices itself */
   TRY(ph_begin(c, PH_GRAM));
   if (dgram) {
      int sp = 0;
      TRY(launch_gram_dbf16(reinterpret_cast<const double *>(C1), reinterpret_cast<const double *>(C2), ne, c->w,
                            K, c->partial, c->partial_cap, &sp, st));
      TRY(ph_end(c, PH_GRAM));
      TRY(ph_begin(c, PH_GRAMRED));
      TRY(launch_reduce_partials(c->partial, sp, ne, 2 * ne, c->Gx, 0, st));
      TRY(launch_gram_dfix(c->Gx, c->g11c[c->g11_idx], ne, c->cur, c->Gm, st));
      if (pstep)
         TRY(sd_smat_precond(c->Gm, c->g11c[c->g11_idx], ne, c->cur, dte, c->DP, c->s11, c->s12, c->s21, c->s22,
                             c->bar, st));
      else if (!one)
         TRY(sd_smat(c->Gm, c->g11c[c->g11_idx], ne, c->cur, dte, c->s11, c->s12, c->s21, c->s22, c->bar, st));
      TRY(ph_end(c, PH_GRAMRED));
   } else {
      const int sp = splits_for(c, 2 * ne, 2 * ne, K, 1);
      const double *Cb = reinterpret_cast<const double *>(c->Cbase);
      int so = 0, sdd = 0;
      const int small = !carry && gemm_tn_small_ok(2 * ne, 2 * ne);
      if (carry) {
         TRY(launch_gram_c2(Cb, K, 2 * ne, (c->cur ^ 1) * ne, c->w, K, c->gram_wgs, c->partial, c->partial_cap,
                            &so, &sdd, st));
      } else if (small) {
         TRY(launch_gemm_tn_small(Cb, K, 2 * ne, Cb, K, 2 * ne, c->w, K, 1, c->Gm, nullptr, 0.0, nullptr, st));
      } else {
         TRY(launch_gemm_tn_splitk(Cb, K, 2 * ne, Cb, K, 2 * ne, c->w, K, sp, 1, c->partial, st));
      }
      TRY(ph_end(c, PH_GRAM));
      TRY(ph_begin(c, PH_GRAMRED));
      /* diagonal tiles hold their upper 16 x 16 blocks only */
      if (carry) TRY(launch_reduce_partials_split(c->partial, so, sdd, 2 * ne, c->cur * ne, (c->cur + 1) * ne,
                                                  c->Gm, st));
      else if (!small) TRY(launch_reduce_partials_symm(c->partial, 2 * ne, K, sp, c->Gm, st));
      if (pstep)
         TRY(sd_smat_precond(c->Gm, carry ? c->g11c[c->g11_idx] : nullptr, ne, c->cur, dte, c->DP, c->s11,
                             c->s12, c->s21, c->s22, c->bar, st));
      else if (!one)
         TRY(sd_smat(c->Gm, carry ? c->g11c[c->g11_idx] : nullptr, ne, c->cur, dte, c->s11, c->s12, c->s21,
                     c->s22, c->bar, st));
      TRY(ph_end(c, PH_GRAMRED));
   }
   /* 12 */
   TRY(ph_begin(c, PH_LAGRANGE));
   {
      LagArgs l;
      l.ne = ne; l.s11 = c->s11; l.s12 = c->s12; l.s21 = c->s21; l.s22 = c->s22;
      l.X = c->LX; l.st1 = c->st1; l.lmd = c->lmd; l.wgmax = c->wgmax; l.info = c->info;
      l.bar = c->bar; l.err = c->err;
      if (one) {
         l.Gm = c->Gm; l.g11c = carry ? c->g11c[c->g11_idx] : nullptr; l.c1_second = c->cur; l.dte = dte;
      }
      l.itmax = 30;
      c->lag_itmax = l.itmax;
      TRY(sd_lagrange(l, st));
      /* the preconditioned step's Lagrange matrix of the unprojected c2 */
      if (pstep) TRY(sd_precond_lmd(c->lmd, c->DP, ne, dte, st));
   }
   TRY(ph_end(c, PH_LAGRANGE));
   /* <c2f|c2f> of the constrained orbitals, the next step's <c1|c1> */
   if (c->g11c[0]) {
      TRY(ph_begin(c, PH_GRAMRED));
      TRY(sd_gram_next(c->Gm, carry ? c->g11c[c->g11_idx] : nullptr, ne, c->cur, c->lmd, dte, c->g11w,
                       c->g11c[c->g11_idx ^ 1], st));
      c->g11_idx ^= 1;
      c->g11_valid = 1;
      c->g11_drift = dgram;
      TRY(ph_end(c, PH_GRAMRED));
   }
   /* 13 */
   TRY(ph_begin(c, PH_CONSTRAINT));
   if (sb) {
      TRY(launch_apply_dbf16(nullptr, nullptr, 0, nullptr, 0, 0, A2, ne, c->lmd, ne, ne, K,
                             reinterpret_cast<double *>(C2), dte, nullptr, 0, c->XTh, c->XTl, st));
   } else {
      TallArgs t;
      t.A = A2; t.lda = K; t.X = c->lmd; t.ldx = ne; t.Mr = ne; t.Nc = ne; t.K = K;
      t.C2 = reinterpret_cast<double *>(C2); t.C1 = nullptr; t.CP = nullptr; t.ldc = K;
      t.dte = dte; t.write_cp = 0;
      TRY(launch_gemm_tall(EPI_CONSTRAINT, t, st));
   }
   TRY(ph_end(c, PH_CONSTRAINT));
   c->cur ^= 1;
   return 0;
}

static int energy_tail(cpsd_dev *c, int inner, double dt, double dte)
{
   hipStream_t st = c->stream;
   const int ne = c->ne, ngp = c->ngp;
   const size_t orb = (size_t)ne * ngp, K = 2 * (size_t)ngp;
   const double2 *C2 = c->Cbase + (size_t)c->cur * orb;
   const double2 *C1 = c->Cbase + (size_t)(c->cur ^ 1) * orb;
   TRY(ph_begin(c, PH_ENERGY));
   {
      const int sp = splits_for(c, ne, ne, K, 0);
      if (gemm_tn_small_ok(ne, ne)) {
         TRY(launch_gemm_tn_small(reinterpret_cast<const double *>(C1), K, ne,
                                  reinterpret_cast<const double *>(c->CP), K, ne, c->w, K, 0, c->Mh,
                                  nullptr, 0.0, nullptr, st));
      } else {
         TRY(launch_gemm_tn_splitk(reinterpret_cast<const double *>(C1), K, ne,
                                   reinterpret_cast<const double *>(c->CP), K, ne, c->w, K, sp, 0,
                                   c->partial, st));
         TRY(launch_reduce_partials(c->partial, sp, ne, ne, c->Mh, 0, st));
      }
      TRY(sd_hml(c->Mh, ne, c->hml, st));
   }
   if (c->stats_on) {
      /* training statistics of this state, while CP still holds cpsi:
       * R = cpsi + c1 hml against Cinf - c1 */
      TallArgs t;
      t.A = reinterpret_cast<const double *>(C1); t.lda = K; t.X = c->hml; t.xsm = 1; t.ldx = ne;
      t.Mr = ne; t.Nc = ne; t.K = K; t.C2 = reinterpret_cast<double *>(c->Rh); t.C1 = nullptr; t.CP = nullptr;
      t.ldc = K; t.dte = 0.0; t.write_cp = 0;
      TRY(launch_gemm_tall(EPI_STORE, t, st));
      TRY(launch_precond_stats(c->CP, c->Rh, C1, c->Cinf, ne, ngp, dte, c->SA, c->SB, st));
   }
   TRY(sd_gsums(c->s, c->dng, c->vall, c->vg, c->vc, c->w, ngp, c->gsum_part, c->ngsum_parts, st));
   TRY(sd_xcsums(c->dn, c->xce, c->xcp, c->n3, c->xc_part, c->nxc_parts, st));
   TRY(sd_ewald_real(c->r1, c->katm, c->zv, c->nion, c->rcell, c->nsh, c->rcut, c->ewald_part, st));
   TRY(sd_orbsums(C1, C2, c->CP, c->tg, c->w, ngp, ne, c->orb_part, c->norb_parts, st));
   EnergyArgs e;
   e.ne = ne; e.nion = c->nion; e.nproj = c->nproj; e.inner = inner;
   e.hml = c->hml; e.P = c->P; e.pnrm = c->pnrm;
   e.gsum_part = c->gsum_part; e.ngsum_parts = c->ngsum_parts;
   e.xc_part = c->xc_part; e.nxc_parts = c->nxc_parts;
   e.orb_part = c->orb_part; e.norb_parts = c->norb_parts;
   e.ewald_part = c->ewald_part;
   e.scal2 = 1.0 / c->omega; e.omega = c->omega;
   e.dv = c->omega / ((double)c->n * c->n * c->n); e.cewald = c->cewald; e.dt = dt; e.dte = dte;
   e.E = c->E;
   TRY(sd_energy(e, st));
   TRY(ph_end(c, PH_ENERGY));
   return 0;
}

/* a call in two halves: ctx_run_start enqueues the inner steps, the energy
 * evaluation and the copy of the results to pinned host memory on the
 * context's stream and returns; ctx_run_finish waits for them.  Contexts
 * whose calls are all started before any is finished advance concurrently,
 * each on its own stream. */
static int ctx_run_start(cpsd_dev *c, int inner, double dt, double fmass, const double *E)
{
   if (inner < 1) { cpsd_set_error("inner=%d must be >= 1", inner); return -1; }
   if (c->pending) { cpsd_set_error("a started call has not been finished"); return -1; }
   const double dte = dt / sqrt(fmass);
   hipStream_t st = c->stream;
   TRY(h2d(c->E, E, 1, st));
   if (c->move) {
      /* dti = dt/sqrt(M) of each ion, ccpsdv3/cpsd.c:116-121 */
      std::vector<double> dti(c->nion);
      for (int i = 0; i < c->nion; ++i) dti[i] = dt / sqrt(c->amass_h[c->katm_h[i]]);
      TRY(h2d(c->dti, dti.data(), c->nion, st));
      CPSD_CHECK(hipStreamSynchronize(st));
   } else if (!c->struct_valid) {
      /* fixed ions: the structure factors and projectors hold until the
       * positions change */
      TRY(run_structure(c));
      c->struct_valid = 1;
   }
   /* graph replay: the steps and the energy tail are device work only (no
    * host synchronisation, no memset), and every buffer is fixed once the
    * context is built, so a captured call replays as it ran; the host state
    * the steps advance (orbital block, carried overlap) is advanced as the
    * captured run advanced it.  Moving ions, profiling and a precision
    * mode's first call (one-time kernel attributes, FP32 projectors) run
    * eagerly. */
   const bool use_graph = c->graphs && !c->move && !c->prof && !c->stats_on && c->ran_mode[c->mixed] &&
                          (c->mixed == 0 || c->mixed == 3 || c->bf_valid) && (c->mixed != 2 || c->bb_valid) &&
                          (c->mixed != 3 || c->bs_valid);
   cpsd_dev::GraphEntry *ge = nullptr;
   if (use_graph) {
      for (int i = 0; i < c->ngc; ++i) {
         cpsd_dev::GraphEntry &e = c->gcache[i];
         if (e.inner == inner && e.mixed == c->mixed && e.cur0 == c->cur && e.g11i0 == c->g11_idx &&
             e.g11v0 == c->g11_valid && e.pre == (c->precond && c->hml_valid) && e.rk == c->refresh &&
             e.rph == (c->refresh > 0 ? (int)(c->nstep % c->refresh) : 0) && e.dt == dt &&
             e.dte == dte) { ge = &e; break; }
      }
      if (!ge && c->ngc < 8) {
         cpsd_dev::GraphEntry e;
         e.inner = inner; e.mixed = c->mixed; e.cur0 = c->cur; e.g11i0 = c->g11_idx; e.g11v0 = c->g11_valid;
         e.pre = c->precond && c->hml_valid;
         e.rk = c->refresh; e.rph = c->refresh > 0 ? (int)(c->nstep % c->refresh) : 0;
         e.dt = dt; e.dte = dte;
         hipGraph_t g = nullptr;
         CPSD_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
         int rc = 0;
         for (int it = 0; it < inner && rc == 0; ++it) rc = sd_step(c, dte, it == inner - 1, refresh_step(c, it));
         if (rc == 0) rc = energy_tail(c, inner, dt, dte);
         const hipError_t ec = hipStreamEndCapture(st, &g);
         if (rc != 0) { if (g) (void)hipGraphDestroy(g); return rc; }
         CPSD_CHECK(ec);
         const hipError_t ei = hipGraphInstantiate(&e.exec, g, nullptr, nullptr, 0);
         (void)hipGraphDestroy(g);
         CPSD_CHECK(ei);
         e.cur1 = c->cur; e.g11i1 = c->g11_idx; e.g11v1 = c->g11_valid;
         /* the capture ran the host side of the steps: return to the state
          * the launch starts from */
         c->cur = e.cur0; c->g11_idx = e.g11i0; c->g11_valid = e.g11v0;
         c->gcache[c->ngc++] = e;
         ge = &c->gcache[c->ngc - 1];
      }
   }
   if (ge) {
      CPSD_CHECK(hipGraphLaunch(ge->exec, st));
      c->cur = ge->cur1; c->g11_idx = ge->g11i1; c->g11_valid = ge->g11v1;
   } else {
      for (int it = 0; it < inner; ++it) TRY(sd_step(c, dte, it == inner - 1, refresh_step(c, it)));
      TRY(energy_tail(c, inner, dt, dte));
      c->ran_mode[c->mixed] = 1;
   }
   if (c->move) c->struct_valid = 0;
   c->hml_valid = 1;   /* the energy tail formed hml of these orbitals */
   c->nstep += inner;
   CPSD_CHECK(hipMemcpyAsync(c->hout, c->E, 12 * sizeof(double), hipMemcpyDeviceToHost, st));
   CPSD_CHECK(hipMemcpyAsync(c->hout + 12, c->info, 2 * sizeof(double), hipMemcpyDeviceToHost, st));
   CPSD_CHECK(hipMemcpyAsync(c->herr, c->err, sizeof(int), hipMemcpyDeviceToHost, st));
   c->pending = 1;
   return 0;
}

/* what a finished call left in pinned memory: errors, E, deltas, the
 * fallback and the non-finite guard (the stream has been synchronised) */
static int ctx_results(cpsd_dev *c, double *E, double *deltae, double *deltac, double *deltar)
{
   const double *out = c->hout, *info = c->hout + 12;
   const int err = *c->herr;
   if (err) { cpsd_set_error("Lagrange grid barrier timed out"); return -1; }
   c->last_lag_iters = (int)info[0];
   c->last_lag_adiff = info[1];
   if (c->last_lag_iters >= c->lag_itmax && !(info[1] < 1e-15)) printf("ierr=10 adiff=%f\n", info[1]);
   for (int i = 0; i < 12; ++i)
      if (!std::isfinite(out[i])) {
         cpsd_set_error("the SD step produced a non-finite %s (%g): the orbitals are lost; restart from "
                        "cpsd_dev_set_orbitals", i < 10 ? "energy" : (i == 10 ? "deltae" : "deltac"), out[i]);
         c->have_prevE = 0;
         c->poisoned = 1;
         return -1;
      }
   for (int i = 0; i < 10; ++i) E[i] = out[i];
   *deltae = out[10];
   *deltac = out[11];
   if (c->fallback_on && c->have_prevE && (c->mixed || c->precond) &&
       E[0] > c->prevE + c->fallback_rise * (fabs(c->prevE) > 1.0 ? fabs(c->prevE) : 1.0)) {
      c->mixed = 0;
      c->precond = 0;
      c->fallbacks += 1;
   }
   c->prevE = E[0];
   c->have_prevE = 1;
   *deltar = 0.0;
   if (c->move) {
      /* largest |F_I|, ccpsdv3/cpsd.c:675-683 */
      std::vector<double> f(3 * (size_t)c->nion);
      CPSD_CHECK(hipMemcpy(f.data(), c->fion, f.size() * sizeof(double), hipMemcpyDeviceToHost));
      for (int i = 0; i < c->nion; ++i) {
         const double a = sqrt(f[3 * i] * f[3 * i] + f[3 * i + 1] * f[3 * i + 1] + f[3 * i + 2] * f[3 * i + 2]);
         if (a > *deltar) *deltar = a;
      }
   }
   c->have_run = 1;
   return 0;
}

static int ctx_run_finish(cpsd_dev *c, double *E, double *deltae, double *deltac, double *deltar)
{
   if (!c->pending) { cpsd_set_error("no started call to finish"); return -1; }
   c->pending = 0;
   CPSD_CHECK(hipStreamSynchronize(c->stream));
   return ctx_results(c, E, deltae, deltac, deltar);
}

static int ctx_run(cpsd_dev *c, int inner, double dt, double fmass, double *E, double *deltae,
                   double *deltac, double *deltar)
{
   TRY(ctx_run_start(c, inner, dt, fmass, E));
   return ctx_run_finish(c, E, deltae, deltac, deltar);
}

/* ---------------------------------------------------- many cells, one graph
 *
 * cpsd_batch advances independent cells (contexts) together.  A call of the
 * batch is captured once into ONE HIP graph: a fork on the batch's stream,
 * then per cell on its own stream the upload of E[0] from pinned memory,
 * its inner steps and energy evaluation and the copy of its results to
 * pinned memory, then a join back; later calls replay it with a single
 * hipGraphLaunch while every cell is in the state the capture started from
 * (orbital block, carried overlap, mode, preconditioner and refresh phase).
 * Calls that cannot be captured (a cell's first call in its precision mode,
 * moving ions, profiling, training statistics) run as concurrent eager
 * calls, one stream per cell. */
struct BatchCellState {
   int cur, g11i, g11v, mixed, pre, rph;
   long nstep;
};

struct BatchGraph {
   hipGraphExec_t exec;
   int inner;
   double dt, dte;
   std::vector<BatchCellState> start, end;
};

struct cpsd_batch {
   std::vector<cpsd_dev *> cells;
   hipStream_t stream;
   hipEvent_t fork;
   std::vector<hipEvent_t> join;
   double *hin;                      /* pinned E[0] of each cell */
   std::vector<BatchGraph> graphs;   /* up to 4, oldest first (an odd inner
                                      * alternates between two start states) */
   long launches, captures, eager;
};

static BatchCellState cell_state(const cpsd_dev *c)
{
   BatchCellState s;
   s.cur = c->cur; s.g11i = c->g11_idx; s.g11v = c->g11_valid; s.mixed = c->mixed;
   s.pre = c->precond && c->hml_valid;
   s.rph = c->refresh > 0 ? (int)(c->nstep % c->refresh) : 0;
   s.nstep = c->nstep;
   return s;
}

static bool same_start(const BatchCellState &a, const BatchCellState &b)
{
   return a.cur == b.cur && a.g11i == b.g11i && a.g11v == b.g11v && a.mixed == b.mixed && a.pre == b.pre &&
          a.rph == b.rph;
}

static bool cell_capturable(const cpsd_dev *c)
{
   return !c->move && !c->prof && !c->stats_on && !c->pending && !c->poisoned && c->struct_valid &&
          c->ran_mode[c->mixed] && (c->mixed == 0 || c->mixed == 3 || c->bf_valid) &&
          (c->mixed != 2 || c->bb_valid) && (c->mixed != 3 || c->bs_valid);
}

static void batch_drop_graphs(cpsd_batch *b)
{
   for (auto &g : b->graphs) (void)hipGraphExecDestroy(g.exec);
   b->graphs.clear();
}

static BatchGraph *batch_capture(cpsd_batch *b, int inner, double dt, double dte)
{
   const size_t n = b->cells.size();
   hipStream_t s0 = b->stream;
   std::vector<BatchCellState> st0(n);
   for (size_t i = 0; i < n; ++i) st0[i] = cell_state(b->cells[i]);
   hipGraph_t g = nullptr;
   if (hipStreamBeginCapture(s0, hipStreamCaptureModeThreadLocal) != hipSuccess) {
      cpsd_set_error("batch capture could not begin");
      return nullptr;
   }
   int rc = hipEventRecord(b->fork, s0) == hipSuccess ? 0 : -1;
   for (size_t i = 0; i < n && rc == 0; ++i) {
      cpsd_dev *c = b->cells[i];
      hipStream_t st = c->stream;
      if (hipStreamWaitEvent(st, b->fork, 0) != hipSuccess ||
          hipMemcpyAsync(c->E, b->hin + i, sizeof(double), hipMemcpyHostToDevice, st) != hipSuccess) {
         rc = -1;
         break;
      }
      for (int it = 0; it < inner && rc == 0; ++it) rc = sd_step(c, dte, it == inner - 1, refresh_step(c, it));
      if (rc == 0) rc = energy_tail(c, inner, dt, dte);
      if (rc == 0 &&
          (hipMemcpyAsync(c->hout, c->E, 12 * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
           hipMemcpyAsync(c->hout + 12, c->info, 2 * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
           hipMemcpyAsync(c->herr, c->err, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
           hipEventRecord(b->join[i], st) != hipSuccess || hipStreamWaitEvent(s0, b->join[i], 0) != hipSuccess))
         rc = -1;
   }
   const hipError_t ec = hipStreamEndCapture(s0, &g);
   /* the capture ran the host side of the steps; what it advanced is what a
    * launch advances: record it and return to the start */
   BatchGraph e;
   e.end.resize(n);
   for (size_t i = 0; i < n; ++i) {
      cpsd_dev *c = b->cells[i];
      e.end[i] = cell_state(c);
      c->cur = st0[i].cur; c->g11_idx = st0[i].g11i; c->g11_valid = st0[i].g11v;
   }
   if (rc != 0 || ec != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      if (rc == 0) cpsd_set_error("batch capture failed: %s", hipGetErrorString(ec));
      return nullptr;
   }
   const hipError_t ei = hipGraphInstantiate(&e.exec, g, nullptr, nullptr, 0);
   (void)hipGraphDestroy(g);
   if (ei != hipSuccess) {
      cpsd_set_error("batch graph instantiation failed: %s", hipGetErrorString(ei));
      return nullptr;
   }
   if (b->graphs.size() >= 4) {
      (void)hipGraphExecDestroy(b->graphs.front().exec);
      b->graphs.erase(b->graphs.begin());
   }
   e.start = st0;
   e.inner = inner; e.dt = dt; e.dte = dte;
   b->graphs.push_back(e);
   b->captures += 1;
   return &b->graphs.back();
}

extern "C" int cpsd_batch_create(cpsd_batch **out, cpsd_dev *const *cells, int n)
{
   if (!out || !cells || n < 1) { cpsd_set_error("cpsd_batch_create: needs n >= 1 cells"); return -1; }
   for (int i = 0; i < n; ++i)
      for (int j = 0; j < i; ++j)
         if (!cells[i] || cells[i] == cells[j]) {
            cpsd_set_error("cpsd_batch_create: cell %d is null or repeated", i);
            return -1;
         }
   cpsd_batch *b = new cpsd_batch();
   b->cells.assign(cells, cells + n);
   b->join.assign(n, nullptr);
   b->launches = b->captures = b->eager = 0;
   if (hipStreamCreate(&b->stream) != hipSuccess ||
       hipEventCreateWithFlags(&b->fork, hipEventDisableTiming) != hipSuccess ||
       hipHostMalloc((void **)&b->hin, (size_t)n * sizeof(double), hipHostMallocDefault) != hipSuccess) {
      cpsd_set_error("cpsd_batch_create: stream, event or pinned memory allocation failed");
      delete b;
      return -1;
   }
   for (int i = 0; i < n; ++i)
      if (hipEventCreateWithFlags(&b->join[i], hipEventDisableTiming) != hipSuccess) {
         cpsd_set_error("cpsd_batch_create: event creation failed");
         return -1;
      }
   *out = b;
   return 0;
}

extern "C" int cpsd_batch_run(cpsd_batch *b, int inner, double dt, double fmass, double *E, double *deltae,
                              double *deltac, double *deltar)
{
   if (!b || !E || !deltae || !deltac || !deltar) { cpsd_set_error("cpsd_batch_run: null argument"); return -1; }
   if (inner < 1) { cpsd_set_error("inner=%d must be >= 1", inner); return -1; }
   const size_t n = b->cells.size();
   const double dte = dt / sqrt(fmass);
   bool graph = true;
   for (size_t i = 0; i < n; ++i) graph = graph && cell_capturable(b->cells[i]);
   if (!graph) {
      /* eager: every call started before any is finished */
      for (size_t i = 0; i < n; ++i)
         if (ctx_run_start(b->cells[i], inner, dt, fmass, E + 10 * i) != 0) return -1;
      int rc = 0;
      for (size_t i = 0; i < n; ++i)
         if (ctx_run_finish(b->cells[i], E + 10 * i, deltae + i, deltac + i, deltar + i) != 0) rc = -1;
      b->eager += 1;
      return rc;
   }
   BatchGraph *ge = nullptr;
   for (auto &gr : b->graphs) {
      bool match = gr.inner == inner && gr.dt == dt && gr.dte == dte;
      for (size_t i = 0; i < n && match; ++i) match = same_start(cell_state(b->cells[i]), gr.start[i]);
      if (match) { ge = &gr; break; }
   }
   if (!ge && !(ge = batch_capture(b, inner, dt, dte))) return -1;
   for (size_t i = 0; i < n; ++i) b->hin[i] = E[10 * i];
   CPSD_CHECK(hipGraphLaunch(ge->exec, b->stream));
   CPSD_CHECK(hipStreamSynchronize(b->stream));
   b->launches += 1;
   int rc = 0;
   for (size_t i = 0; i < n; ++i) {
      cpsd_dev *c = b->cells[i];
      c->cur = ge->end[i].cur; c->g11_idx = ge->end[i].g11i; c->g11_valid = ge->end[i].g11v;
      c->hml_valid = 1;
      c->nstep += inner;
      if (ctx_results(c, E + 10 * i, deltae + i, deltac + i, deltar + i) != 0) rc = -1;
   }
   return rc;
}

extern "C" int cpsd_batch_info(cpsd_batch *b, long *graph_launches, long *captures, long *eager_calls)
{
   if (!b) { cpsd_set_error("null batch"); return -1; }
   if (graph_launches) *graph_launches = b->launches;
   if (captures) *captures = b->captures;
   if (eager_calls) *eager_calls = b->eager;
   return 0;
}

extern "C" void cpsd_batch_destroy(cpsd_batch *b)
{
   if (!b) return;
   (void)hipStreamSynchronize(b->stream);
   batch_drop_graphs(b);
   for (hipEvent_t e : b->join)
      if (e) (void)hipEventDestroy(e);
   if (b->fork) (void)hipEventDestroy(b->fork);
   if (b->hin) (void)hipHostFree(b->hin);
   if (b->stream) (void)hipStreamDestroy(b->stream);
   delete b;
}

static int ctx_set_ions(cpsd_dev *c, int move, const double *amass, const double *r2)
{
   hipStream_t st = c->stream;
   if (move != 0 && move != 1) { cpsd_set_error("move=%d must be 0 or 1", move); return -1; }
   if (!r2 || (move && !amass)) { cpsd_set_error("set_ions needs positions and, for move=1, masses"); return -1; }
   if (move && c->mixed >= 2) {
      cpsd_set_error("set_ions: moving ions need precision mode 0 or 1 (mode 2 moves forces by ~3e-4 Ha/bohr; "
                     "mode 3 is for electronic convergence)");
      return -1;
   }
   const size_t n3i = 3 * (size_t)c->nion;
   if (move && !c->r2d) {
      c->fchunk = 64;
      TRY(dalloc(&c->r2d, n3i)); TRY(dalloc(&c->fion, n3i)); TRY(dalloc(&c->dti, c->nion));
      TRY(dalloc(&c->Gp, 3 * (size_t)c->ngp));
      TRY(h2d(c->Gp, c->Gp_h, 3 * (size_t)c->ngp, st));
      TRY(dalloc(&c->fgpart, (size_t)c->nion * c->fchunk * 3));
      TRY(dalloc(&c->fnlpart, (size_t)(2 * (size_t)c->ngp / 128) * (c->nproj > 0 ? c->nproj : 1) * 3));
      TRY(dalloc(&c->fnlsum, 3 * (size_t)(c->nproj > 0 ? c->nproj : 1)));
      CPSD_CHECK(hipMemsetAsync(c->fion, 0, n3i * sizeof(double), st));
   }
   if (move) {
      double *m = (double *)realloc(c->amass_h, (size_t)c->nkind * sizeof(double));
      if (!m) { cpsd_set_error("host allocation failed"); return -1; }
      c->amass_h = m;
      for (int k = 0; k < c->nkind; ++k) {
         if (!(amass[k] > 0.0)) { cpsd_set_error("amass[%d]=%g must be positive", k, amass[k]); return -1; }
         c->amass_h[k] = amass[k];
      }
      TRY(h2d(c->r2d, r2, n3i, st));
   }
   c->move = move;
   TRY(h2d(c->r1, r2, n3i, st));
   c->struct_valid = 0;
   CPSD_CHECK(hipStreamSynchronize(st));
   return 0;
}

static int ctx_get_ions(cpsd_dev *c, double *r1, double *r2, double *fion)
{
   const size_t n3i = 3 * (size_t)c->nion;
   if (r1) CPSD_CHECK(hipMemcpy(r1, c->r1, n3i * sizeof(double), hipMemcpyDeviceToHost));
   if (r2) CPSD_CHECK(hipMemcpy(r2, c->move ? c->r2d : c->r1, n3i * sizeof(double), hipMemcpyDeviceToHost));
   if (fion && c->fion) CPSD_CHECK(hipMemcpy(fion, c->fion, n3i * sizeof(double), hipMemcpyDeviceToHost));
   return 0;
}

/* after a call with non-finite results every buffer the steps carry from
 * one step to the next is cleared, so that new orbitals start clean */
static int ctx_clear_state(cpsd_dev *c)
{
   hipStream_t st = c->stream;
   const size_t orb = (size_t)c->ne * c->ngp, ee = (size_t)c->ne * c->ne;
   const size_t plane = (size_t)c->n * c->ncol;
   struct { void *p; size_t bytes; } z[] = {
      {c->Cbase, 2 * orb * sizeof(double2)}, {c->CP, orb * sizeof(double2)},
      {c->T, (size_t)c->ne * plane * sizeof(double2)}, {c->Tv, plane * sizeof(double2)},
      {c->dnpart, (size_t)(c->ndnblk[0] > c->ndnblk[1] ? c->ndnblk[0] : c->ndnblk[1]) * c->n3 * sizeof(double)},
      {c->dn, c->n3 * sizeof(double)}, {c->xcp, c->n3 * sizeof(double)}, {c->xce, c->n3 * sizeof(double)},
      {c->V, c->n3 * sizeof(double)}, {c->dng, (size_t)c->ngp * sizeof(double2)},
      {c->partial, c->partial_cap * sizeof(double)}, {c->Gm, 4 * ee * sizeof(double)},
      {c->s11, ee * sizeof(double)}, {c->s12, ee * sizeof(double)}, {c->s21, ee * sizeof(double)},
      {c->s22, ee * sizeof(double)}, {c->LX, 2 * ee * sizeof(double)}, {c->st1, ee * sizeof(double)},
      {c->lmd, ee * sizeof(double)}, {c->hml, ee * sizeof(double)}, {c->Mh, ee * sizeof(double)},
      {c->g11c[0], ee * sizeof(double)}, {c->g11c[1], ee * sizeof(double)}, {c->g11w, 2 * ee * sizeof(double)},
      {c->DP, 3 * ee * sizeof(double)}, {c->err, 4 * sizeof(int)}};
   for (auto &e : z)
      if (e.p) CPSD_CHECK(hipMemsetAsync(e.p, 0, e.bytes, st));
   CPSD_CHECK(hipStreamSynchronize(st));
   c->poisoned = 0;
   return 0;
}

/* Copies from the device to the caller's (pageable) arrays.  The runtime's own
 * path empties its staging with one thread, about 9 GB/s; here a ring of
 * pinned chunks is emptied by a few threads while the DMA engine fills the
 * others (59 MB: 3.4 -> 1.6 ms, into fresh pages 6.2 -> 2.1; uploads run at
 * 27 GB/s either way).  The threads live for one call of ctx_get.  Calls below
 * 8 MB, arrays below 4, arrays in pinned memory (59 MB: 1.07 ms, 1.60 through
 * the ring), and every copy if no ring or threads can be had, take the plain
 * path. */
class HostCopier {
   enum { SLOTS = StageRings::SLOTS, THREADS = 4 };
   static constexpr size_t CHUNK = StageRings::CHUNK, LEAST = (size_t)4 << 20;
   struct Job { int slot; char *host; size_t n; };
   cpsd_dev *c;
   StageRings::Ring *ring = nullptr;
   int dev = 0;
   bool on = false, tried, stop = false;   /* the ring and its threads: there; there or not to be had */
   bool finished = false;
   long issued = 0;                      /* chunks given a slot so far */
   int failed = 0;
   std::mutex mu;
   std::condition_variable cv;
   Job jobs[SLOTS];                      /* queued jobs [head, tail): at most one per slot */
   long head = 0, tail = 0;
   long done[SLOTS] = {0};               /* jobs finished on a slot */
   std::thread th[THREADS];
   uintptr_t lo = UINTPTR_MAX, hi = 0;   /* the host addresses of the arrays so far */

   void work()
   {
      int bad = hipSetDevice(dev) != hipSuccess;
      std::unique_lock<std::mutex> lk(mu);
      for (;;) {
         cv.wait(lk, [&] { return stop || head < tail; });
         if (head == tail) return;
         const Job j = jobs[head++ % SLOTS];
         lk.unlock();
         if (hipEventSynchronize(ring->ev[j.slot]) != hipSuccess) bad = 1;   /* the chunk has arrived */
         memcpy(j.host, ring->mem + (size_t)j.slot * CHUNK, j.n);
         lk.lock();
         done[j.slot]++;
         if (bad) failed = 1;
         cv.notify_all();
      }
   }
   void push(const Job &j)
   {
      std::lock_guard<std::mutex> lk(mu);
      jobs[tail++ % SLOTS] = j;
      cv.notify_all();
   }
   void await(int slot, long count)
   {
      std::unique_lock<std::mutex> lk(mu);
      cv.wait(lk, [&] { return done[slot] >= count; });
   }
   /* every chunk issued so far is in its array */
   void drain()
   {
      for (long j = std::max(0L, issued - SLOTS); j < issued; ++j) await((int)(j % SLOTS), j / SLOTS + 1);
   }
   /* memory the runtime knows (pinned, registered, managed): the DMA engine
    * writes it itself, 55 GB/s */
   static bool known(const void *host)
   {
      hipPointerAttribute_t at;
      if (hipPointerGetAttributes(&at, host) == hipSuccess) return at.type != hipMemoryTypeUnregistered;
      (void)hipGetLastError();   /* the question's own error */
      return false;
   }
   /* the ring and its threads, when the first array needs them */
   bool start()
   {
      if (tried) return on;
      tried = true;
      if (hipGetDevice(&dev) != hipSuccess) return false;
      if (!c->stager) { StageRings::join(); c->stager = 1; }
      ring = StageRings::take(dev);
      if (!ring) return false;
      int n = 0;
      try {
         for (; n < THREADS; ++n) th[n] = std::thread([this] { work(); });
      } catch (...) {
      }
      return on = n > 0;
   }

public:
   /* total: bytes of the call that may go through the ring */
   HostCopier(cpsd_dev *ctx, size_t total) : c(ctx), tried(total < 2 * LEAST) {}
   ~HostCopier()
   {
      {
         std::lock_guard<std::mutex> lk(mu);
         stop = true;
         cv.notify_all();
      }
      for (std::thread &t : th)
         if (t.joinable()) t.join();
      /* a call that failed may have chunks on their way: the ring is nobody's
       * until they have arrived */
      if (ring && (finished || hipStreamSynchronize(c->stream) == hipSuccess)) StageRings::give(ring);
   }
   /* after what is on the stream; the data is there after finish().  Where a
    * caller passes the same memory for several arrays, the last one stays in
    * it: such an array waits for the chunks of those before it.  staged: the
    * array may go through the ring */
   int get(void *host, const void *d, size_t n, bool staged)
   {
      const uintptr_t h = reinterpret_cast<uintptr_t>(host);
      if (h < hi && h + n > lo) drain();
      lo = std::min(lo, h);
      hi = std::max(hi, h + n);
      if (!staged || n < LEAST || known(host) || !start()) {
         CPSD_CHECK(hipMemcpyAsync(host, d, n, hipMemcpyDeviceToHost, c->stream));
         return 0;
      }
      for (size_t o = 0; o < n; o += CHUNK, ++issued) {
         const int slot = (int)(issued % SLOTS);
         const size_t m = std::min(CHUNK, n - o);
         await(slot, issued / SLOTS);
         CPSD_CHECK(hipMemcpyAsync(ring->mem + (size_t)slot * CHUNK, static_cast<const char *>(d) + o, m,
                                   hipMemcpyDeviceToHost, c->stream));
         CPSD_CHECK(hipEventRecord(ring->ev[slot], c->stream));
         push(Job{slot, static_cast<char *>(host) + o, m});
      }
      return 0;
   }
   /* everything is where it belongs */
   int finish()
   {
      CPSD_CHECK(hipStreamSynchronize(c->stream));
      drain();
      finished = true;
      if (failed) { cpsd_set_error("copy to the host failed"); return -1; }
      return 0;
   }
};

static int ctx_set_orbitals(cpsd_dev *c, const double *cin)
{
   hipStream_t st = c->stream;
   if (c->poisoned) TRY(ctx_clear_state(c));
   const size_t fstride = c->nfft3d;
   CPSD_CHECK(hipMemcpyAsync(c->fullbuf, cin, (size_t)c->ne * c->n2ft3d * sizeof(double),
                             hipMemcpyHostToDevice, st));
   CPSD_CHECK(hipMemsetAsync(c->flag, 0, sizeof(int), st));
   /* a timed-out Lagrange barrier of an earlier run does not outlive it */
   CPSD_CHECK(hipMemsetAsync(c->err, 0, sizeof(int), st));
   TRY(sd_check_unmasked(c->fullbuf, fstride, c->pidx, c->nfft3d, c->ne, c->flag, st));
   c->cur = 0;
   c->g11_valid = 0;
   c->hml_valid = 0;
   c->nstep = 0;
   c->have_prevE = 0;
   TRY(sd_pack(c->fullbuf, fstride, c->gidx, c->ng, c->ngp, c->Cbase, c->ngp, c->ne, st));
   int flag = 0;
   CPSD_CHECK(hipMemcpyAsync(&flag, c->flag, sizeof(int), hipMemcpyDeviceToHost, st));
   CPSD_CHECK(hipStreamSynchronize(st));
   if (flag) {
      cpsd_set_error("orbital coefficients outside the cutoff mask are nonzero; the GPU path "
                     "stores masked coefficients only");
      return -1;
   }
   return 0;
}

static int ctx_get(cpsd_dev *c, double *c1, double *c2, double *cpsi, double *dn, double *hml,
                   double *lmd)
{
   const size_t orb = (size_t)c->ne * c->ngp, bytes = (size_t)c->ne * c->n2ft3d * sizeof(double);
   hipStream_t st = c->stream;
   HostCopier hc(c, ((c1 != nullptr) + (c2 != nullptr) + (cpsi != nullptr)) * bytes);
   auto get_orb = [&](const double2 *packed, double *host) {
      TRY(sd_unpack(packed, c->ngp, c->pidx, c->nfft3d, c->fullbuf, c->nfft3d, c->ne, st));
      return hc.get(host, c->fullbuf, bytes, true);
   };
   if (c1) TRY(get_orb(c->Cbase + (size_t)(c->cur ^ 1) * orb, c1));
   if (c2) TRY(get_orb(c->Cbase + (size_t)c->cur * orb, c2));
   if (cpsi) TRY(get_orb(c->CP, cpsi));
   if (dn) {
      TRY(sd_pad_real(c->dn, fft_slots(c->n), 2, c->realbuf, st));
      TRY(hc.get(dn, c->realbuf, (size_t)c->n2ft3d * sizeof(double), false));
   }
   const size_t ee = (size_t)c->ne * c->ne;
   if (hml) TRY(hc.get(hml, c->hml, ee * sizeof(double), false));
   if (lmd) TRY(hc.get(lmd, c->lmd, ee * sizeof(double), false));
   return hc.finish();
}

/* The run epilogue of ccpsdv3/main.c:451-484 on the resident state:
 * ortho = gcdotc(c1_i, c1_j) of the last step's starting orbitals (:456-464),
 * the eigenpairs of hml in eigsrt order (:466-476), and c1 <- c2 V on the
 * device (:478-483).  c2 is left as it is. */
static int ctx_epilogue(cpsd_dev *c, double *ortho, double *eig, double *V)
{
   if (!c->have_run) { cpsd_set_error("epilogue: no SD step has run on this context"); return -1; }
   c->g11_valid = 0;
   c->hml_valid = 0;   /* c1 is rotated below */
   const int ne = c->ne;
   const size_t K = 2 * (size_t)c->ngp, orb = (size_t)ne * c->ngp, ee = (size_t)ne * ne;
   hipStream_t st = c->stream;
   double2 *C1 = c->Cbase + (size_t)(c->cur ^ 1) * orb;
   const double2 *C2 = c->Cbase + (size_t)c->cur * orb;
   if (ortho) {
      const int sp = splits_for(c, ne, ne, K, 1);
      int so, sd;
      gemm_tn_symm_splits(ne, K, sp, &so, &sd);
      if ((size_t)(so > sd ? so : sd) * ee > c->partial_cap) {
         cpsd_set_error("epilogue: split-K buffer too small");
         return -1;
      }
      const double *c1r = reinterpret_cast<const double *>(C1);
      if (gemm_tn_small_ok(ne, ne)) {
         TRY(launch_gemm_tn_small(c1r, K, ne, c1r, K, ne, c->w, K, 1, c->Gm, nullptr, 0.0, nullptr, st));
      } else {
         TRY(launch_gemm_tn_splitk(c1r, K, ne, c1r, K, ne, c->w, K, sp, 1, c->partial, st));
         TRY(launch_reduce_partials_symm(c->partial, ne, K, sp, c->Gm, st));
      }
      CPSD_CHECK(hipMemcpyAsync(ortho, c->Gm, ee * sizeof(double), hipMemcpyDeviceToHost, st));
   }
   std::vector<double> a(ee), w(ne);
   CPSD_CHECK(hipMemcpyAsync(a.data(), c->hml, ee * sizeof(double), hipMemcpyDeviceToHost, st));
   CPSD_CHECK(hipStreamSynchronize(st));
   TRY(cpsd_syev_sorted(ne, a.data(), w.data()));
   /* Mh (the energy tail's scratch) takes V: X[m][n] = V[m + n ne] */
   CPSD_CHECK(hipMemcpyAsync(c->Mh, a.data(), ee * sizeof(double), hipMemcpyHostToDevice, st));
   TallArgs t;
   t.A = reinterpret_cast<const double *>(C2); t.lda = K;
   t.X = c->Mh; t.ldx = ne; t.xsm = 1; t.Mr = ne; t.Nc = ne; t.K = K;
   t.C2 = reinterpret_cast<double *>(C1); t.ldc = K;
   TRY(launch_gemm_tall(EPI_STORE, t, st));
   CPSD_CHECK(hipStreamSynchronize(st));
   if (eig) memcpy(eig, w.data(), (size_t)ne * sizeof(double));
   if (V) memcpy(V, a.data(), ee * sizeof(double));
   return 0;
}

/* ---------------------------------------------------- public C-ABI */

extern "C" int cpsd_dev_create(cpsd_dev **h, int nfft, int ne, int nion, const int *katm,
                               const double *zv, const int *lmmax, const double *vnlnrm,
                               const double *vl, const double *vnl, const int *masker,
                               const double *tg, const double *vc, const double *vg,
                               const double *unitg, double omega, int nsh, const double *rcell,
                               double cewald, double rcut, const double *r)
{
   cpsd_dev *c = (cpsd_dev *)calloc(1, sizeof(cpsd_dev));
   if (!c) { cpsd_set_error("out of host memory"); return -1; }
   if (ctx_build(c, nfft, ne, nion, katm, zv, lmmax, vnlnrm, vl, vnl, masker, tg, vc, vg, unitg,
                 omega, nsh, rcell, cewald, rcut, r) != 0) {
      ctx_free(c);
      free(c);
      *h = nullptr;
      return -1;
   }
   c->fallback_on = 1;
   c->fallback_rise = 1e-8;
   *h = c;
   return 0;
}

extern "C" int cpsd_dev_set_orbitals(cpsd_dev *h, const double *c)
{
   if (!h || !c) { cpsd_set_error("cpsd_dev_set_orbitals: null handle or orbitals"); return -1; }
   return ctx_set_orbitals(h, c);
}

extern "C" int cpsd_dev_run(cpsd_dev *h, int inner, double dt, double fmass, double *E,
                            double *deltae, double *deltac, double *deltar)
{
   if (!h || !E || !deltae || !deltac || !deltar) {
      cpsd_set_error("cpsd_dev_run: null handle or output");
      return -1;
   }
   return ctx_run(h, inner, dt, fmass, E, deltae, deltac, deltar);
}

extern "C" int cpsd_dev_run_start(cpsd_dev *h, int inner, double dt, double fmass, const double *E)
{
   if (!h || !E) { cpsd_set_error("cpsd_dev_run_start: null handle or E"); return -1; }
   return ctx_run_start(h, inner, dt, fmass, E);
}

extern "C" int cpsd_dev_run_finish(cpsd_dev *h, double *E, double *deltae, double *deltac, double *deltar)
{
   if (!h || !E || !deltae || !deltac || !deltar) {
      cpsd_set_error("cpsd_dev_run_finish: null handle or output");
      return -1;
   }
   return ctx_run_finish(h, E, deltae, deltac, deltar);
}

extern "C" int cpsd_dev_set_ions(cpsd_dev *h, int move, const double *amass, const double *r2)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   return ctx_set_ions(h, move, amass, r2);
}

extern "C" int cpsd_dev_get_ions(cpsd_dev *h, double *r1, double *r2, double *fion)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   return ctx_get_ions(h, r1, r2, fion);
}

extern "C" int cpsd_dev_get(cpsd_dev *h, double *c1, double *c2, double *cpsi, double *dn,
                            double *hml, double *lmd)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   return ctx_get(h, c1, c2, cpsi, dn, hml, lmd);
}

extern "C" int cpsd_dev_epilogue(cpsd_dev *h, double *ortho, double *eig, double *V)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   return ctx_epilogue(h, ortho, eig, V);
}

extern "C" int cpsd_dev_set_precision(cpsd_dev *h, int mode)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   if (mode < 0 || mode > 3) {
      cpsd_set_error("cpsd_dev_set_precision: mode %d is not 0 (FP64), 1 (FP32), 2 (FP32, BF16 projection) or 3 "
                     "(FP32 transforms, split-BF16 products)", mode);
      return -1;
   }
   if (mode >= 2 && h->move) {
      cpsd_set_error("cpsd_dev_set_precision: mode %d is for electronic convergence (mode 2's BF16 projection "
                     "moves forces by ~3e-4 Ha/bohr); with moving ions use mode 0 or 1", mode);
      return -1;
   }
   if (mode == 3) {
      const size_t K = 2 * (size_t)h->ngp;
      if (!gram_dbf16_ok(h->ne) || !apply_dbf16_ok(h->ne)) {
         cpsd_set_error("cpsd_dev_set_precision: mode 3 needs ne = 128 or 256 (ne=%d)", h->ne);
         return -1;
      }
      if (!gram_dbf16_fits(h->ne, K)) {
         cpsd_set_error("cpsd_dev_set_precision: mode 3: %d orbitals of %zu reals exceed 4 GiB", h->ne, K);
         return -1;
      }
      const int npad = (h->nproj + 31) / 32 * 32;
      if (!h->Gx) TRY(dalloc(&h->Gx, 2 * (size_t)h->ne * h->ne));
      if (!h->XTh) {
         TRY(dalloc(&h->XTh, (size_t)h->ne * (npad + h->ne)));
         TRY(dalloc(&h->XTl, (size_t)h->ne * (npad + h->ne)));
      }
   }
   h->mixed = mode;
   return 0;
}

extern "C" int cpsd_dev_set_refresh(cpsd_dev *h, int period)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   if (period < 0) { cpsd_set_error("cpsd_dev_set_refresh: period %d must be >= 0", period); return -1; }
   h->refresh = period;
   return 0;
}

extern "C" int cpsd_dev_set_fallback(cpsd_dev *h, int enable, double rise)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   if (!std::isfinite(rise)) { cpsd_set_error("cpsd_dev_set_fallback: rise must be finite"); return -1; }
   h->fallback_on = enable ? 1 : 0;
   h->fallback_rise = rise;
   return 0;
}

extern "C" int cpsd_dev_fallback_info(cpsd_dev *h, int *fallbacks, int *mode, int *precond)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   if (fallbacks) *fallbacks = h->fallbacks;
   if (mode) *mode = h->mixed;
   if (precond) *precond = h->precond;
   return 0;
}

/* ------------------------------------------------------------ autotuner
 *
 * The launch plan (ctx_plan) of each size class -- grid, orbitals,
 * projectors, precision mode, preconditioner on or off -- is chosen by
 * measurement: knob by knob (split-K workgroup target, orbitals per FFT
 * launch pair, orbitals per density plane), each candidate runs a few SD
 * steps of the context's own orbitals, timed with HIP events, and the
 * fastest is kept; the result is remembered for the process, so other
 * cells of the class take it without measuring.  Tuning leaves the
 * orbitals as they were and resets the run state as
 * cpsd_dev_set_orbitals() does.  The knobs change launch shapes and
 * reduction blockings only, so results change at rounding level. */
struct PlanKey {
   int n, ne, nproj, mixed, pre;
   bool operator<(const PlanKey &o) const
   {
      if (n != o.n) return n < o.n;
      if (ne != o.ne) return ne < o.ne;
      if (nproj != o.nproj) return nproj < o.nproj;
      if (mixed != o.mixed) return mixed < o.mixed;
      return pre < o.pre;
   }
};
struct Plan {
   int fb, nob[2], wgt;
   double ms;
};
static std::mutex g_plan_mu;
static std::map<PlanKey, Plan> g_plans;

static void reset_run_state(cpsd_dev *c)
{
   c->cur = 0; c->g11_valid = 0; c->hml_valid = 0; c->nstep = 0; c->have_prevE = 0;
}

static int time_plan(cpsd_dev *c, const double2 *backup, const Plan &p, int steps, double *ms)
{
   TRY(ctx_plan(c, p.fb, p.nob, p.wgt));
   hipStream_t st = c->stream;
   const size_t orb = (size_t)c->ne * c->ngp;
   CPSD_CHECK(hipMemcpyAsync(c->Cbase, backup, orb * sizeof(double2), hipMemcpyDeviceToDevice, st));
   reset_run_state(c);
   c->hml_valid = c->precond ? 1 : 0;   /* time the preconditioned step when it is on */
   const double dte = 5.8 / sqrt(400000.0);
   TRY(sd_step(c, dte, 0, 0));           /* warm-up (first launches, carried overlap) */
   hipEvent_t e0, e1;
   CPSD_CHECK(hipEventCreate(&e0));
   CPSD_CHECK(hipEventCreate(&e1));
   CPSD_CHECK(hipEventRecord(e0, st));
   int rc = 0;
   for (int i = 0; i < steps && rc == 0; ++i) rc = sd_step(c, dte, 0, 0);
   CPSD_CHECK(hipEventRecord(e1, st));
   CPSD_CHECK(hipEventSynchronize(e1));
   float t = 0.f;
   CPSD_CHECK(hipEventElapsedTime(&t, e0, e1));
   (void)hipEventDestroy(e0);
   (void)hipEventDestroy(e1);
   *ms = rc == 0 ? (double)t / steps : 1e30;
   return rc;
}

extern "C" int cpsd_dev_autotune(cpsd_dev *h, int steps, int *plan)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   if (h->pending || h->move || h->stats_on) {
      cpsd_set_error("cpsd_dev_autotune: needs fixed ions and no started call or statistics");
      return -1;
   }
   if (steps < 1) steps = 3;
   const PlanKey key{h->n, h->ne, h->nproj, h->mixed, h->precond};
   Plan best;
   int cached = 0;
   {
      std::lock_guard<std::mutex> lk(g_plan_mu);
      auto it = g_plans.find(key);
      if (it != g_plans.end()) { best = it->second; cached = 1; }
   }
   if (!cached) {
      const size_t orb = (size_t)h->ne * h->ngp;
      double2 *backup = nullptr;
      TRY(dalloc(&backup, orb));
      const double2 *C2 = h->Cbase + (size_t)h->cur * orb;
      int rc = hipMemcpyAsync(backup, C2, orb * sizeof(double2), hipMemcpyDeviceToDevice, h->stream) == hipSuccess
                  ? 0 : -1;
      if (rc == 0 && !h->struct_valid) { rc = run_structure(h); h->struct_valid = rc == 0; }
      if (h->mixed && h->mixed != 3 && rc == 0) rc = ensure_bf(h);
      if (h->mixed == 2 && rc == 0) rc = ensure_bb(h);
      if (h->mixed == 3 && rc == 0) rc = ensure_bs(h);
      Plan cur{h->ne, {0, 0}, 2048, 0.0};
      if (rc == 0) rc = time_plan(h, backup, cur, steps, &cur.ms);
      best = cur;
      /* split-K target */
      for (int w : {1024, 4096}) {
         Plan p = best; p.wgt = w;
         if (rc == 0) rc = time_plan(h, backup, p, steps, &p.ms);
         if (rc == 0 && p.ms < best.ms) best = p;
      }
      /* orbitals per FFT launch pair */
      for (int fb : {h->ne / 2, 32}) {
         if (fb < 8 || fb >= h->ne) continue;
         Plan p = best; p.fb = fb; p.nob[0] = p.nob[1] = 0;
         if (rc == 0) rc = time_plan(h, backup, p, steps, &p.ms);
         if (rc == 0 && p.ms < best.ms) best = p;
      }
      /* orbitals per density partial plane, around the filling default */
      if (rc == 0) {
         TRY(ctx_plan(h, best.fb, best.nob, best.wgt));
         const int f = h->mixed ? 1 : 0, d = h->nob[f];
         for (int nb : {2 * d, d / 2}) {
            if (nb < 1 || nb > best.fb || nb == d) continue;
            Plan p = best; p.nob[f] = nb;
            if (rc == 0) rc = time_plan(h, backup, p, steps, &p.ms);
            if (rc == 0 && p.ms < best.ms) best = p;
         }
      }
      /* the orbitals as they were */
      if (rc == 0) rc = ctx_plan(h, best.fb, best.nob, best.wgt);
      if (rc == 0 && hipMemcpyAsync(h->Cbase, backup, orb * sizeof(double2), hipMemcpyDeviceToDevice,
                                    h->stream) != hipSuccess)
         rc = -1;
      (void)hipStreamSynchronize(h->stream);
      (void)hipFree(backup);
      reset_run_state(h);
      if (rc != 0) return -1;
      std::lock_guard<std::mutex> lk(g_plan_mu);
      g_plans[key] = best;
   } else {
      TRY(ctx_plan(h, best.fb, best.nob, best.wgt));
      const size_t orb = (size_t)h->ne * h->ngp;
      if (h->cur != 0)
         CPSD_CHECK(hipMemcpyAsync(h->Cbase, h->Cbase + orb, orb * sizeof(double2), hipMemcpyDeviceToDevice,
                                   h->stream));
      CPSD_CHECK(hipStreamSynchronize(h->stream));
      reset_run_state(h);
   }
   if (plan) {
      plan[0] = h->fb; plan[1] = h->nob[0]; plan[2] = h->nob[1]; plan[3] = h->wgt; plan[4] = cached;
   }
   return 0;
}

/* K[nfft3d]: one factor per half-complex G of the reference's layout (the
 * factors outside the cutoff mask are not used); NULL turns it off */
static int ctx_set_preconditioner(cpsd_dev *c, const double *K)
{
   if (!K) { c->precond = 0; return 0; }
   std::vector<double> kp(c->ngp, 0.0);
   for (int p = 0; p < c->ng; ++p) {
      const double f = K[c->gidx_h[p]];
      if (!(f >= 0.0) || !(f < 1e6)) {
         cpsd_set_error("cpsd_dev_set_preconditioner: K at G index %d is %g, not a finite factor >= 0",
                        c->gidx_h[p], f);
         return -1;
      }
      kp[p] = f;
   }
   /* the buffer is allocated once, so captured calls keep reading it */
   if (!c->Kp) TRY(dalloc(&c->Kp, c->ngp));
   CPSD_CHECK(hipMemcpyAsync(c->Kp, kp.data(), (size_t)c->ngp * sizeof(double), hipMemcpyHostToDevice,
                             c->stream));
   CPSD_CHECK(hipStreamSynchronize(c->stream));
   c->precond = 1;
   return 0;
}

/* structure factors, local potential and projectors of the current ions
 * (what the features read), formed now if no step has formed them */
static int ensure_structure(cpsd_dev *c)
{
   if (!c->struct_valid) {
      TRY(run_structure(c));
      if (!c->move) c->struct_valid = 1;
   }
   return 0;
}

static int ctx_precond_features(cpsd_dev *c)
{
   TRY(ensure_structure(c));
   if (!c->Xf) TRY(dalloc(&c->Xf, 4 * (size_t)c->ngp));
   return launch_precond_features(c->tg, c->B, c->pnrm, c->nproj, c->vall, c->omega, c->ng, c->ngp, c->Xf,
                                  c->stream);
}

extern "C" int cpsd_dev_precond_features(cpsd_dev *h, float *X)
{
   if (!h || !X) { cpsd_set_error("cpsd_dev_precond_features: null handle or output"); return -1; }
   TRY(ctx_precond_features(h));
   CPSD_CHECK(hipMemcpyAsync(X, h->Xf, 4 * (size_t)h->ng * sizeof(float), hipMemcpyDeviceToHost, h->stream));
   CPSD_CHECK(hipStreamSynchronize(h->stream));
   return 0;
}

extern "C" int cpsd_dev_set_learned_preconditioner(cpsd_dev *h, const float *params, double alpha, double kmin,
                                                   double kmax)
{
   if (!h || !params) { cpsd_set_error("cpsd_dev_set_learned_preconditioner: null handle or parameters"); return -1; }
   if (!(alpha > 0.0) || !(kmin >= 0.0) || !(kmax >= kmin) || !(kmax < 1e6)) {
      cpsd_set_error("cpsd_dev_set_learned_preconditioner: needs alpha > 0 and 0 <= kmin <= kmax < 1e6");
      return -1;
   }
   if (h->pending) { cpsd_set_error("cpsd_dev_set_learned_preconditioner: a started call has not been finished"); return -1; }
   for (int q = 0; q < CPSD_MLP_NPARAM; ++q)
      if (!std::isfinite(params[q])) { cpsd_set_error("cpsd_dev_set_learned_preconditioner: parameter %d is not finite", q); return -1; }
   hipStream_t st = h->stream;
   TRY(ctx_precond_features(h));
   if (!h->Pmlp) TRY(dalloc(&h->Pmlp, CPSD_MLP_NPARAM));
   if (!h->Kp) TRY(dalloc(&h->Kp, h->ngp));
   CPSD_CHECK(hipMemcpyAsync(h->Pmlp, params, CPSD_MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice, st));
   if (h->ngp > h->ng) CPSD_CHECK(hipMemsetAsync(h->Kp + h->ng, 0, (size_t)(h->ngp - h->ng) * sizeof(double), st));
   TRY(launch_mlp_predict(h->Xf, h->ng, h->Pmlp, nullptr, h->Kp, alpha, kmin, kmax, st));
   CPSD_CHECK(hipStreamSynchronize(st));
   h->precond = 1;
   return 0;
}

/* training statistics: _begin takes the converged orbitals cinf (ELCIN
 * layout), clears the sums and makes every following energy evaluation add
 * its state (energy_tail), _end stops that, _read returns the per-G sums of
 * the masked G in packed order (the order of cpsd_dev_precond_features) */
extern "C" int cpsd_dev_stats_begin(cpsd_dev *h, const double *cinf)
{
   if (!h || !cinf) { cpsd_set_error("cpsd_dev_stats_begin: null handle or orbitals"); return -1; }
   const size_t orb = (size_t)h->ne * h->ngp;
   if (!h->Cinf) {
      TRY(dalloc(&h->Cinf, orb)); TRY(dalloc(&h->Rh, orb));
      TRY(dalloc(&h->SA, h->ngp)); TRY(dalloc(&h->SB, h->ngp));
   }
   hipStream_t st = h->stream;
   CPSD_CHECK(hipMemcpyAsync(h->fullbuf, cinf, (size_t)h->ne * h->n2ft3d * sizeof(double), hipMemcpyHostToDevice, st));
   TRY(sd_pack(h->fullbuf, h->nfft3d, h->gidx, h->ng, h->ngp, h->Cinf, h->ngp, h->ne, st));
   CPSD_CHECK(hipMemsetAsync(h->SA, 0, h->ngp * sizeof(double), st));
   CPSD_CHECK(hipMemsetAsync(h->SB, 0, h->ngp * sizeof(double), st));
   CPSD_CHECK(hipStreamSynchronize(st));
   h->stats_on = 1;
   return 0;
}

extern "C" int cpsd_dev_stats_end(cpsd_dev *h)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   h->stats_on = 0;
   return 0;
}

extern "C" int cpsd_dev_stats_read(cpsd_dev *h, double *A, double *B)
{
   if (!h || !h->Cinf || !A || !B) { cpsd_set_error("cpsd_dev_stats_read: no statistics or null output"); return -1; }
   CPSD_CHECK(hipMemcpy(A, h->SA, (size_t)h->ng * sizeof(double), hipMemcpyDeviceToHost));
   CPSD_CHECK(hipMemcpy(B, h->SB, (size_t)h->ng * sizeof(double), hipMemcpyDeviceToHost));
   return 0;
}

extern "C" int cpsd_dev_set_preconditioner(cpsd_dev *h, const double *K)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   if (h->pending) { cpsd_set_error("cpsd_dev_set_preconditioner: a started call has not been finished"); return -1; }
   return ctx_set_preconditioner(h, K);
}

extern "C" int cpsd_dev_set_graphs(cpsd_dev *h, int enable)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   h->graphs = enable ? 1 : 0;
   return 0;
}

extern "C" int cpsd_dev_lagrange_info(cpsd_dev *h, int *iterations, double *adiff)
{
   if (!h || !iterations || !adiff) { cpsd_set_error("cpsd_dev_lagrange_info: null handle or output"); return -1; }
   *iterations = h->last_lag_iters;
   *adiff = h->last_lag_adiff;
   return 0;
}

extern "C" int cpsd_dev_sizes(cpsd_dev *h, int *sizes)
{
   if (!h || !sizes) { cpsd_set_error("cpsd_dev_sizes: null handle or output"); return -1; }
   sizes[0] = h->ng; sizes[1] = h->ngp; sizes[2] = h->nproj;
   return 0;
}

extern "C" int cpsd_dev_profile(cpsd_dev *h, int enable)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   TRY(ph_flush(h));
   if (enable && !h->pool) {
      h->pool_cap = 2048;
      h->pool = (hipEvent_t *)calloc(2 * h->pool_cap, sizeof(hipEvent_t));
      h->pool_ph = (int *)calloc(h->pool_cap, sizeof(int));
      if (!h->pool || !h->pool_ph) { cpsd_set_error("out of host memory"); return -1; }
      for (int i = 0; i < 2 * h->pool_cap; ++i) CPSD_CHECK(hipEventCreate(&h->pool[i]));
   }
   h->prof = enable;
   for (int i = 0; i < PH_COUNT; ++i) { h->prof_ms[i] = 0.0; h->prof_calls[i] = 0; }
   return 0;
}

extern "C" int cpsd_dev_profile_read(cpsd_dev *h, char *names, int names_len, double *ms, int *calls,
                                     int max_phases)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   std::string s;
   int k = 0;
   TRY(ph_flush(h));
   for (int i = 0; i < PH_COUNT && i < max_phases; ++i, ++k) {
      if (i) s += ";";
      s += ph_names[i];
      ms[i] = h->prof_ms[i];
      calls[i] = h->prof_calls[i];
   }
   if (names && names_len > 0) {
      strncpy(names, s.c_str(), names_len - 1);
      names[names_len - 1] = 0;
   }
   return k;
}

/* copy an internal device buffer to the host (test hook): returns the number
 * of doubles written, or -1 */
extern "C" long cpsd_dev_debug_fetch(cpsd_dev *h, int what, double *out, long cap)
{
   if (!h) { cpsd_set_error("null handle"); return -1; }
   const size_t orb = (size_t)h->ne * h->ngp;
   const void *src = nullptr;
   size_t nd = 0;
   switch (what) {
   case 0: src = h->dn; nd = h->n3; break;
   case 1: src = h->V; nd = h->n3; break;
   case 2: src = h->dng; nd = 2 * (size_t)h->ngp; break;
   case 3: src = h->CP; nd = 2 * orb; break;
   case 4: src = h->P; nd = (size_t)h->nproj * h->ne; break;
   case 5: src = h->Gm; nd = 4 * (size_t)h->ne * h->ne; break;
   case 6: src = h->s11; nd = (size_t)h->ne * h->ne; break;
   case 7: src = h->s12; nd = (size_t)h->ne * h->ne; break;
   case 8: src = h->s21; nd = (size_t)h->ne * h->ne; break;
   case 9: src = h->s22; nd = (size_t)h->ne * h->ne; break;
   case 10: src = h->lmd; nd = (size_t)h->ne * h->ne; break;
   case 11: src = h->Cbase; nd = 4 * orb; break;
   case 12: src = h->xcp; nd = h->n3; break;
   case 13: src = h->vall; nd = 2 * (size_t)h->ngp; break;
   case 14: src = h->Xkb; nd = (size_t)h->nproj * h->ne; break;
   case 15: src = h->B; nd = 2 * (size_t)h->nproj * h->ngp; break;
   case 16: src = h->info; nd = 2; break;
   default: cpsd_set_error("debug_fetch: unknown buffer %d", what); return -1;
   }
   if ((long)nd > cap) { cpsd_set_error("debug_fetch: capacity %ld < %zu", cap, nd); return -1; }
   if (what == 0 || what == 1 || what == 12) {   /* real-space fields, in natural order */
      TRY(sd_pad_real(static_cast<const double *>(src), fft_slots(h->n), 0, h->realbuf, h->stream));
      CPSD_CHECK(hipStreamSynchronize(h->stream));
      src = h->realbuf;
   }
   if (hipMemcpy(out, src, nd * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess) {
      cpsd_set_error("debug_fetch: copy failed");
      return -1;
   }
   return (long)nd;
}

extern "C" void cpsd_dev_destroy(cpsd_dev *h)
{
   if (!h) return;
   ctx_free(h);
   free(h);
}

/* ------------------------------------------- drop-in cpsd() of cpsd.c */

static cpsd_dev *g_ctx = nullptr;
/* what the drop-in context was built from, and the positions it holds */
struct DropinKey {
   int nfft, ne, nion, nsh, nkind, pad;
   double omega, cewald, rcut;
   uint64_t h;
};
static DropinKey g_key;
static std::vector<double> g_r2;
static int g_ctx_reusable = 0;

/* 64-bit hash of a byte range: 8-byte words mixed with the splitmix64
 * finaliser (tail bytes zero-padded), chained through h.  Whole 64-byte blocks
 * run through eight chains, folded into one at their end: one chain waits for
 * its own two multiplications at every word (3 ms for the tables of two kinds
 * at 48^3, 0.5 with eight). */
static uint64_t hash_bytes(uint64_t h, const void *p, size_t n)
{
   const unsigned char *b = static_cast<const unsigned char *>(p);
   auto mix = [](uint64_t z) {
      z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
      z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
      return z ^ (z >> 31);
   };
   const uint64_t step = 0x9e3779b97f4a7c15ull;
   size_t i = 0;
   if (n >= 64) {
      uint64_t l[8];
      for (int q = 0; q < 8; ++q) l[q] = mix(h + (uint64_t)(q + 1) * step);
      for (; i + 64 <= n; i += 64) {
         uint64_t w[8];
         memcpy(w, b + i, 64);
         for (int q = 0; q < 8; ++q) l[q] = mix(l[q] ^ (w[q] + step));
      }
      for (int q = 0; q < 8; ++q) h = mix(h ^ (l[q] + step));
   }
   for (; i + 8 <= n; i += 8) {
      uint64_t w;
      memcpy(&w, b + i, 8);
      h = mix(h ^ (w + step));
   }
   if (i < n) {
      uint64_t w = 0;
      memcpy(&w, b + i, n - i);
      h = mix(h ^ (w + step));
   }
   return mix(h ^ n);
}

extern "C" void cpsd(const int inner, const int move, const int nion, const int ispin, const int *ne,
                     const int nfft, const int nfft3d, const int n2ft3d, const double *unitg,
                     const double omega, const double dt, const double fmass, const int *katm,
                     const double *amass, const double *zv, const int nsh, const double *rcell,
                     const double cewald, const double rcut, const int *masker, const double *G,
                     const double *tg, const double *vc, const double *vg, int *lmmax,
                     double *vnlnrm, double *vl, double *vnl, double *r1, double *r2, double *fion,
                     double *c1, double *c2, double *cpsi, double *dn, double *hml, double *lmd,
                     double *cpsdwork, double *E, double *deltae, double *deltac, double *deltar)
{
   (void)G; (void)cpsdwork;
   if (ispin != 1 || ne[1] != 0 || (move != 0 && move != 1)) {
      cpsd_set_error("only ispin=1 (ne[1]=0), move=0 or 1 is supported (got ispin=%d move=%d ne[1]=%d)",
                     ispin, move, ne[1]);
      fail_loudly("cpsd");
      return;
   }
   if (nfft3d != (nfft / 2 + 1) * nfft * nfft || n2ft3d != (nfft + 2) * nfft * nfft) {
      cpsd_set_error("inconsistent grid sizes nfft=%d nfft3d=%d n2ft3d=%d", nfft, nfft3d, n2ft3d);
      fail_loudly("cpsd");
      return;
   }
   /* r1 <- r2 before anything reads the positions (ccpsdv3/cpsd.c:174) */
   memcpy(r1, r2, 3 * (size_t)nion * sizeof(double));
   /* The device context of the previous call is kept when this call's
    * static inputs are those it was built from (sizes, scalars and a hash
    * of every table), as they are across the outer loop of
    * ccpsdv3/main.c:417-445; only the orbitals (c2) and, when they moved,
    * the ions go up again.  Anything else rebuilds the context. */
   int nkind = 0;
   for (int i = 0; i < nion; ++i)
      if (katm[i] + 1 > nkind) nkind = katm[i] + 1;
   DropinKey key;
   memset(&key, 0, sizeof key);
   key.nfft = nfft; key.ne = ne[0]; key.nion = nion; key.nsh = nsh; key.nkind = nkind;
   key.omega = omega; key.cewald = cewald; key.rcut = rcut;
   {
      uint64_t h = 0x6a09e667f3bcc908ull;
      h = hash_bytes(h, katm, (size_t)nion * sizeof(int));
      if (nkind > 0) {
         h = hash_bytes(h, zv, (size_t)nkind * sizeof(double));
         h = hash_bytes(h, lmmax, (size_t)nkind * sizeof(int));
         h = hash_bytes(h, vnlnrm, (size_t)nkind * 9 * sizeof(double));
         h = hash_bytes(h, vl, (size_t)nkind * nfft3d * sizeof(double));
         for (int k = 0; k < nkind; ++k)
            h = hash_bytes(h, vnl + (size_t)k * 9 * nfft3d, (size_t)(lmmax[k] > 0 ? lmmax[k] : 0) * nfft3d * sizeof(double));
      }
      h = hash_bytes(h, masker, (size_t)n2ft3d * sizeof(int));
      h = hash_bytes(h, tg, (size_t)nfft3d * sizeof(double));
      h = hash_bytes(h, vc, (size_t)nfft3d * sizeof(double));
      h = hash_bytes(h, vg, (size_t)nfft3d * sizeof(double));
      h = hash_bytes(h, unitg, 9 * sizeof(double));
      h = hash_bytes(h, rcell, 3 * (size_t)nsh * sizeof(double));
      key.h = h;
   }
   const bool reuse = g_ctx && g_ctx_reusable && memcmp(&key, &g_key, sizeof key) == 0;
   if (!reuse) {
      if (g_ctx) { cpsd_dev_destroy(g_ctx); g_ctx = nullptr; }
      g_ctx_reusable = 0;
      if (cpsd_dev_create(&g_ctx, nfft, ne[0], nion, katm, zv, lmmax, vnlnrm, vl, vnl, masker, tg, vc,
                          vg, unitg, omega, nsh, rcell, cewald, rcut, r1) != 0) {
         fail_loudly("cpsd");
         return;
      }
      g_key = key;
      g_r2.assign(r1, r1 + 3 * (size_t)nion);
   } else if (!move && (g_ctx->move || memcmp(g_r2.data(), r1, 3 * (size_t)nion * sizeof(double)) != 0)) {
      /* fixed ions that are not where the kept context has them */
      if (ctx_set_ions(g_ctx, 0, nullptr, r1) != 0) { fail_loudly("cpsd"); return; }
      g_r2.assign(r1, r1 + 3 * (size_t)nion);
   }
   g_ctx_reusable = 0;   /* set again only when this call completes */
   if ((move && ctx_set_ions(g_ctx, 1, amass, r2) != 0) ||
       ctx_set_orbitals(g_ctx, c2) != 0 ||
       ctx_run(g_ctx, inner, dt, fmass, E, deltae, deltac, deltar) != 0 ||
       ctx_get(g_ctx, c1, c2, cpsi, dn, hml, lmd) != 0 ||
       (move && ctx_get_ions(g_ctx, r1, r2, fion) != 0)) {
      fail_loudly("cpsd");
      return;
   }
   if (move) g_r2.assign(r2, r2 + 3 * (size_t)nion);
   g_ctx_reusable = 1;
}

/* ccpsdv3/main.c:466-484 for ispin = 1 with host arrays: esyev('V','U') and
 * eigsrt of hml (hml <- eigenvectors in columns, eig <- eigenvalues,
 * descending), then c1 = c2 hml over the n2ft3d reals of each orbital.  It
 * reuses the device tables of the preceding cpsd() call (same nfft and ne),
 * as the reference's epilogue follows its SD loop; c2 is uploaded again, so
 * the host arrays are the ones rotated. */
extern "C" void cpsd_rotate(const int ispin, const int *ne, const int n2ft3d, double *hml, double *eig,
                            const double *c2, double *c1)
{
   if (ispin != 1 || ne[1] != 0) {
      cpsd_set_error("cpsd_rotate: only ispin=1 (ne[1]=0) is supported (got ispin=%d ne[1]=%d)", ispin, ne[1]);
      fail_loudly("cpsd_rotate");
      return;
   }
   if (!g_ctx || g_ctx->ne != ne[0] || g_ctx->n2ft3d != n2ft3d) {
      cpsd_set_error("cpsd_rotate: needs a preceding cpsd() call with ne=%d and n2ft3d=%d", ne[0], n2ft3d);
      fail_loudly("cpsd_rotate");
      return;
   }
   cpsd_dev *c = g_ctx;
   const size_t ee = (size_t)c->ne * c->ne;
   if (ctx_set_orbitals(c, c2) != 0) { fail_loudly("cpsd_rotate"); return; }
   std::vector<double> a(hml, hml + ee), w(c->ne);
   if (cpsd_syev_sorted(c->ne, a.data(), w.data()) != 0) { fail_loudly("cpsd_rotate"); return; }
   const size_t K = 2 * (size_t)c->ngp, orb = (size_t)c->ne * c->ngp;
   hipStream_t st = c->stream;
   TallArgs t;
   t.A = reinterpret_cast<const double *>(c->Cbase + (size_t)c->cur * orb); t.lda = K;
   t.X = c->Mh; t.ldx = c->ne; t.xsm = 1; t.Mr = c->ne; t.Nc = c->ne; t.K = K;
   t.C2 = reinterpret_cast<double *>(c->Cbase + (size_t)(c->cur ^ 1) * orb); t.ldc = K;
   if (hipMemcpyAsync(c->Mh, a.data(), ee * sizeof(double), hipMemcpyHostToDevice, st) != hipSuccess ||
       launch_gemm_tall(EPI_STORE, t, st) != 0 || ctx_get(c, c1, nullptr, nullptr, nullptr, nullptr, nullptr) != 0) {
      fail_loudly("cpsd_rotate");
      return;
   }
   memcpy(hml, a.data(), ee * sizeof(double));
   memcpy(eig, w.data(), (size_t)c->ne * sizeof(double));
}

/* ---------------------------------------- FFT entry points (Fortran) */

struct FftCtx {
   int n, nbatch;
   hipStream_t stream;
   double2 *tw, *T, *A;
};
static FftCtx g_fft = {0, 0, nullptr, nullptr, nullptr, nullptr};

static int fft_ctx(int n, int nbatch)
{
   if (!fft_supported(n)) { cpsd_set_error("FFT grid %d is not supported", n); return -1; }
   if (g_fft.n == n && g_fft.nbatch >= nbatch) return 0;
   if (g_fft.stream) {
      (void)hipFree(g_fft.tw); (void)hipFree(g_fft.T); (void)hipFree(g_fft.A);
   } else {
      CPSD_CHECK(hipStreamCreate(&g_fft.stream));
   }
   const int nh = n / 2 + 1;
   std::vector<double2> tw(n);
   for (int m = 0; m < n; ++m) {
      const double a = 2.0 * M_PI * (double)m / (double)n;
      tw[m] = make_double2(cos(a), sin(a));
   }
   g_fft.n = n; g_fft.nbatch = nbatch;
   TRY(dalloc(&g_fft.tw, n));
   TRY(dalloc(&g_fft.T, (size_t)nbatch * n * n * nh));
   TRY(dalloc(&g_fft.A, (size_t)nbatch * n * n * nh));
   hipStream_t st = g_fft.stream;
   TRY(h2d(g_fft.tw, tw.data(), n, st));
   CPSD_CHECK(hipStreamSynchronize(st));
   return 0;
}

static int fft_run(int dir, int n, int nbatch, double *Ah)
{
   TRY(fft_ctx(n, nbatch));
   hipStream_t st = g_fft.stream;
   const size_t per = (size_t)n * n * (n / 2 + 1);  /* complex = (n+2) n n / 2 */
   CPSD_CHECK(hipMemcpyAsync(g_fft.A, Ah, (size_t)nbatch * per * sizeof(double2), hipMemcpyHostToDevice, st));
   TRY(launch_fft3d(dir, n, nbatch, g_fft.A, g_fft.T, g_fft.tw, st));
   CPSD_CHECK(hipMemcpyAsync(Ah, g_fft.A, (size_t)nbatch * per * sizeof(double2), hipMemcpyDeviceToHost, st));
   CPSD_CHECK(hipStreamSynchronize(st));
   return 0;
}

static int fft_args_ok(int *inc2c, int *inc3c, int *inc2r, int *inc3r, int *nx, int *ny, int *nz)
{
   const int n = *nx;
   if (*ny != n || *nz != n || *inc2c != n / 2 + 1 || *inc3c != (n / 2 + 1) * n || *inc2r != n + 2 ||
       *inc3r != (n + 2) * n) {
      cpsd_set_error("only nx=ny=nz with the reference increments is supported");
      return -1;
   }
   return 0;
}

extern "C" void cr_fft3b_(double *A, int *inc2c, int *inc3c, int *inc2r, int *inc3r, int *nx, int *ny,
                          int *nz, double *tmp, int *ntmp)
{
   (void)tmp; (void)ntmp;
   if (fft_args_ok(inc2c, inc3c, inc2r, inc3r, nx, ny, nz) != 0 || fft_run(+1, *nx, 1, A) != 0)
      fail_loudly("cr_fft3b_");
}

extern "C" void rc_fft3f_(double *A, int *inc2c, int *inc3c, int *inc2r, int *inc3r, int *nx, int *ny,
                          int *nz, double *tmp, int *ntmp)
{
   (void)tmp; (void)ntmp;
   if (fft_args_ok(inc2c, inc3c, inc2r, inc3r, nx, ny, nz) != 0 || fft_run(-1, *nx, 1, A) != 0)
      fail_loudly("rc_fft3f_");
}

extern "C" int cpsd_fft3d_batch(int dir, int nfft, int nbatch, double *A)
{
   return fft_run(dir, nfft, nbatch, A);
}

extern "C" int cpsd_lda_device(int n, const double *dn, double *xcp, double *xce)
{
   double *d = nullptr, *p = nullptr, *e = nullptr;
   TRY(dalloc(&d, n)); TRY(dalloc(&p, n)); TRY(dalloc(&e, n));
   CPSD_CHECK(hipMemcpy(d, dn, n * sizeof(double), hipMemcpyHostToDevice));
   TRY(sd_lda(d, n, p, e, 0));
   CPSD_CHECK(hipMemcpy(xcp, p, n * sizeof(double), hipMemcpyDeviceToHost));
   CPSD_CHECK(hipMemcpy(xce, e, n * sizeof(double), hipMemcpyDeviceToHost));
   (void)hipFree(d); (void)hipFree(p); (void)hipFree(e);
   return 0;
}

extern "C" int cpsd_erfc_device(int n, const double *w, double *out)
{
   double *d = nullptr, *o = nullptr;
   TRY(dalloc(&d, n)); TRY(dalloc(&o, n));
   CPSD_CHECK(hipMemcpy(d, w, n * sizeof(double), hipMemcpyHostToDevice));
   TRY(sd_erfc_as(d, n, o, 0));
   CPSD_CHECK(hipMemcpy(out, o, n * sizeof(double), hipMemcpyDeviceToHost));
   (void)hipFree(d); (void)hipFree(o);
   return 0;
}
