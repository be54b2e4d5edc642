/*
 * gemm_kernels.hip -- FP64 MFMA contractions over the packed G vectors.
 *
 * The reference forms these as level-1 BLAS loops:
 *   - KB projections  sw = gcdotc(beta, c1_i)      ccpsdv3/cpsd.c:287-290
 *   - overlaps        gcdotc(c_i, c_j) x 4          ccpsdv3/cpsd.c:415-437
 *   - hml             -gcdotc(c1_i, cpsi_j)         ccpsdv3/cpsd.c:497-513
 *   - KB apply        c2_i += sw * beta (daxpy)     ccpsdv3/cpsd.c:290
 *   - constraint      c2 += dte c1 lmd (dgemm)      ccpsdv3/cpsd.c:482-488
 * Here they are two kernels built on v_mfma_f64_16x16x4_f64 (mfma64.h):
 *   k_gemm_tn_splitk : small M x N output, reduction over the huge K = 2*ngp
 *                      real coefficients, split over blockIdx.z; 128 x 128
 *                      output tiles; the G-space weight
 *                      (1 on the kx = 0 plane, 2 elsewhere: the
 *                      2*sum - sum_{kx=0} of ccpsdv3/gcdotc.c:25-27) is
 *                      applied to the A operand.
 *   k_gemm_tall      : tall output [ncol][K] = X^T A with a short reduction
 *                      (projectors or orbitals), 128-, 64- or 32-column x 128-row
 *                      output tiles over 4 waves, SD epilogues fused; the
 *                      nonlocal force (ccpsdv3/cpsd.c:291-304) reduces its
 *                      output against the projectors instead of storing it.
 */
#include "cpsd_internal.h"
#include "mfma64.h"
#include <type_traits>
#include <cstring>

/* 16 bytes at base + off: a scalar base and a 32-bit lane offset */
__device__ __forceinline__ double2 load2(const char *base, unsigned off)
{
   typedef double d2 __attribute__((ext_vector_type(2)));
   const d2 v = *reinterpret_cast<const d2 *>(base + off);
   return make_double2(v[0], v[1]);
}

/* sum over the 64 lanes of a wave, same tree in every wave */
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
   for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
   return v;
}

/* ------------------------------------------------------- split-K TN */

/* scheduling hint: N times, one instruction of the kind MASK (0x100 LDS read,
 * 0x200 LDS write, 0x20 global read) after M MFMAs */
template<int MASK, int N, int M>
__device__ __forceinline__ void sched_mix()
{
#pragma unroll
   for (int i = 0; i < N; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, M, 0);
      __builtin_amdgcn_sched_group_barrier(MASK, 1, 0);
   }
}

template<int V> using template_int = std::integral_constant<int, V>;

#define TT 128  /* output tile edge */
#define KC 32   /* K ranges are multiples of this */

/* The blocks of a diagonal tile.  Its 36 upper 16 x 16 blocks are split
 * evenly between the four waves: waves 0-2 take 3 x 3 squares on or above the
 * diagonal (rows dg_row.., columns dg_col..), wave 3 the three remaining
 * corners (p, p), (p, p+1), (p+1, p+1) at p = 0, 3, 6. */
__device__ __forceinline__ int dg_row(int wave) { return wave == 1 ? 3 : 0; }
__device__ __forceinline__ int dg_col(int wave) { return wave == 2 ? 2 : 5; }
/* operand fragment f of a corner wave is block row dg_tri(f); block b of it
 * multiplies fragments dg_ta(b) and dg_tb(b) */
__device__ constexpr int dg_tri(int f) { return 3 * (f >> 1) + (f & 1); }
__device__ constexpr int dg_ta(int b) { return 2 * (b / 3) + (b % 3 == 2); }
__device__ constexpr int dg_tb(int b) { return 2 * (b / 3) + (b % 3 != 0); }

/* partial[z][m][n] = sum_{k in split z} w[k] A[m][k] B[n][k].  TM x TN output
 * tiles, four waves of (TM/2) x (TN/2), K steps of KT double-buffered in LDS.
 * 128 x 128 (or 96 x 128 when that pads the row count less, e.g. 192
 * projectors) in 72 KB: two workgroups share a CU, so one's barriers and loads
 * overlap the other's MFMAs.  32 x 32 (35 KB, K steps of 32) where 128 would
 * leave CUs without work (tn_tile).  The operands of the next 8 k are read from LDS between
 * the MFMAs of the current ones; the weight is applied to the A rows on their
 * way into LDS.  Each sum runs over k in order, one fused multiply-add per
 * term (what the FP64 MFMA does with its four k), so a split's result does
 * not depend on the tiling.
 *
 * One workgroup per (tile, K split); the grid is 1D over the pairs.
 * Workgroups go to the 8 XCDs round-robin by block id, so block b is given
 * pair (b % 8) * per + b / 8 with per = pairs / 8 rounded up (ids past the
 * last pair exit): the workgroups one XCD runs together hold consecutive
 * pairs, i.e. all tiles of the same K range, which then share that XCD's L2.
 *
 * A symmetric product (SYM: A = B, M = N) forms the listed tiles only: tiles
 * above the diagonal in full, 128 x 128 diagonal tiles by their upper 36
 * blocks, nine to a wave against 16 in a full tile.  Split z of a diagonal tile is the
 * whole range z of kchunk_dd (tl.halves 1) or half h of range z' (z = 2 z' +
 * h, tl.halves 2).
 *
 * Bound by the MFMA issue: at 64 waters (128^3, 256 orbitals, 384
 * projectors) the KB projection takes 3.39 ms (64 TFLOP/s) and the Gram with
 * <c1|c1> carried 3.68 ms (60); the form with four v_mfma_f64_4x4x4_4b
 * per 16 x 16 block, 8 waves of 64 x 32 and one workgroup per CU took 4.24 and
 * 4.46 ms (51 and 49 TFLOP/s). */
template<int TM, int TN, int KT, bool SYM>
__global__ void __launch_bounds__(256, TN == 128 ? 2 : 4)
k_gemm_tn_splitk(const double *__restrict__ A, size_t lda, int M,
                 const double *__restrict__ B, size_t ldb, int N,
                 const double *__restrict__ w, size_t K, size_t kchunk, size_t kchunk_dd,
                 int ntm, int ntile, long poff, long pairs, GramTiles tl, double *__restrict__ partial)
{
   /* a symmetric product's off-diagonal pairs and its shorter diagonal pairs
    * are spread over the XCDs each by themselves, the longer ones first */
   const long x = blockIdx.x & 7, t8 = blockIdx.x >> 3, po = SYM ? (poff + 7) >> 3 : gridDim.x >> 3;
   const bool dd = SYM && t8 >= po;
   const long g = dd ? x * ((gridDim.x >> 3) - po) + t8 - po : x * po + t8;
   if (g >= (SYM && !dd ? poff : dd ? pairs - poff : pairs)) return;
   int tm, tn, kz;
   size_t kc = kchunk;
   if (dd) {
      tm = tn = tl.dt[g % tl.nd];
      kz = (int)(g / tl.nd);
      kc = kchunk_dd;
   } else if (SYM) {
      const int t = (int)(g % tl.noff);
      kz = (int)(g / tl.noff);
      tm = tl.otm[t];
      tn = tl.otn[t];
   } else {
      const int t = (int)(g % ntile);
      kz = (int)(g / ntile);
      tm = t % ntm;
      tn = t / ntm;
   }
   size_t kb = (size_t)(SYM && dd && tl.halves == 2 ? kz >> 1 : kz) * kc;
   size_t ke = min(K, kb + kc);
   if (SYM && dd && tl.halves == 2) {
      const size_t khalf = ke > kb ? ((ke - kb) / KC + 1) / 2 * KC : 0;
      if (kz & 1) kb += khalf;
      else ke = min(ke, kb + khalf);
   }
   /* S[buf][0]: the weighted A rows, S[buf][1]: the B rows (of a diagonal
    * tile the same rows without the weight).  Of each 8 k the pairs (q, q + 4)
    * are adjacent: one 16-byte read hands a lane its slot of two successive
    * instructions.  The pitch lets a 16-byte read of 8 rows cover the banks
    * once. */
   constexpr int KP = KT + 2;
   __shared__ __align__(16) double S[2][2][TM > TN ? TM : TN][KP];
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int wm = wave & 1, wn = wave >> 1;
   const int l16 = lane & 15, lq4 = lane >> 4;
   constexpr int BI = TM / 32, BJ = TN / 32;   /* 16-row and 16-column blocks per wave */

   /* Row addresses without branches: rows past M or N repeat the last one
    * (their outputs are not written), so a load is a 32-bit lane offset on a
    * scalar base that moves along K.  PR lanes to the K step of a row. */
   constexpr int PR = KT / 2, RP = 256 / PR;
   constexpr int HA = TM / RP, HB = TN / RP;
   const int lr = tid / PR, lc = tid % PR;
   const int ar0 = tm * TM, br0 = tn * TN;
   const char *const abase = reinterpret_cast<const char *>(A + (size_t)ar0 * lda);
   const char *const bbase = reinterpret_cast<const char *>(B + (size_t)br0 * ldb);
   unsigned aoff[HA], boff[HB];
#pragma unroll
   for (int h = 0; h < HA; ++h) aoff[h] = (unsigned)min(lr + RP * h, M - 1 - ar0) * (unsigned)(lda * 8) + lc * 16;
#pragma unroll
   for (int h = 0; h < HB; ++h) boff[h] = (unsigned)min(lr + RP * h, N - 1 - br0) * (unsigned)(ldb * 8) + lc * 16;
   /* K tile t + 1 waits in registers while tile t is multiplied */
   double2 ra[HA], rb[HB], rw;
   auto gload = [&](size_t k0) {
      const char *const ak = abase + k0 * 8;
      const char *const bk = bbase + k0 * 8;
#pragma unroll
      for (int h = 0; h < HA; ++h) ra[h] = load2(ak, aoff[h]);
      if (!SYM || !dd) {
#pragma unroll
         for (int h = 0; h < HB; ++h) rb[h] = load2(bk, boff[h]);
      }
      rw = load2(reinterpret_cast<const char *>(w + k0), lc * 16);
   };
   /* k = 2 lc, 2 lc + 1 of rows lr + RP h */
   const int sq = 8 * (lc >> 2) + 4 * (lc & 1) + ((lc >> 1) & 1);
   auto lput = [&](double *row, double2 v) {
      row[sq] = v.x;
      row[sq + 2] = v.y;
   };
   auto lstore = [&](int bf) {
#pragma unroll
      for (int h = 0; h < HA; ++h) lput(S[bf][0][lr + RP * h], make_double2(ra[h].x * rw.x, ra[h].y * rw.y));
      if (SYM && dd) {
#pragma unroll
         for (int h = 0; h < HA; ++h) lput(S[bf][1][lr + RP * h], ra[h]);
      } else {
#pragma unroll
         for (int h = 0; h < HB; ++h) lput(S[bf][1][lr + RP * h], rb[h]);
      }
   };
   /* k = 8 ks + lq4 and 8 ks + 4 + lq4 of a row */
   auto pair_at = [&](int bf, int half, int row, int ks) {
      return *reinterpret_cast<const double2 *>(&S[bf][half][row][8 * ks + 2 * lq4]);
   };

   /* the K loop, specialised per wave role: NA x NB fragments, blocks
    * (ia(b), jb(b)), b < NBLK */
   auto kloop = [&](auto na_, auto nb_, auto nblk_, auto arow, auto brow, auto ia, auto jb, mfma_d4 *acc) {
      constexpr int NA = decltype(na_)::value, NB = decltype(nb_)::value, NBLK = decltype(nblk_)::value;
      constexpr int NK = KT / 8;
      struct Frag { double2 a[NA], b[NB]; };
      auto fread = [&](Frag &f, int bf, int ks) {
#pragma unroll
         for (int i = 0; i < NA; ++i) f.a[i] = pair_at(bf, 0, 16 * arow(i) + l16, ks);
#pragma unroll
         for (int j = 0; j < NB; ++j) f.b[j] = pair_at(bf, 1, 16 * brow(j) + l16, ks);
      };
      auto mma = [&](const Frag &f) {
#pragma unroll
         for (int b = 0; b < NBLK; ++b) acc[b] = mfma16(f.a[ia(b)].x, f.b[jb(b)].x, acc[b]);
#pragma unroll
         for (int b = 0; b < NBLK; ++b) acc[b] = mfma16(f.a[ia(b)].y, f.b[jb(b)].y, acc[b]);
      };
#pragma unroll
      for (int b = 0; b < NBLK; ++b) acc[b] = mfma_d4{0.0, 0.0, 0.0, 0.0};
      if (kb >= ke) return;
      const int nt = (int)((ke - kb + KT - 1) / KT);
      gload(kb);
      lstore(0);
      gload(kb + (nt > 1 ? KT : 0));
      __syncthreads();
      Frag f[2];
      fread(f[0], 0, 0);
      int buf = 0;
      /* branch-free body: one workgroup's MFMA stream has to stay fed from one
       * wave per SIMD, so the LDS reads and writes and the loads of the next
       * tile are spread between the MFMAs (64 cycles each) */
      for (int t = 0; t + 1 < nt; ++t) {
#pragma unroll
         for (int ks = 0; ks + 1 < NK; ++ks) {
            fread(f[(ks + 1) & 1], buf, ks + 1);
            mma(f[ks & 1]);
            if (ks + 2 == NK) lstore(buf ^ 1);
            sched_mix<0x100, NA + NB, 1>();
            if (ks + 2 == NK) sched_mix<0x200, HA + HB, 1>();
         }
         __syncthreads();   /* every read of this tile has been issued and has returned */
         buf ^= 1;
         fread(f[0], buf, 0);
         gload(kb + (size_t)min(t + 2, nt - 1) * KT);
         mma(f[1]);
         sched_mix<0x100, NA + NB, 1>();
         sched_mix<0x20, HA + HB + 1, 1>();
      }
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) {
         if (ks + 1 < NK) fread(f[(ks + 1) & 1], buf, ks + 1);
         mma(f[ks & 1]);
      }
   };
   auto store_block = [&](int m0, int n0, const mfma_d4 &v) {
      const int n = n0 + l16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
         const int m = m0 + mfma16_row(r, lane);
         if (m < M && n < N) partial[((size_t)kz * M + m) * N + n] = v[r];
      }
   };
   if (TN != 128 || !SYM || !dd) {
      /* a diagonal tile of 32 is formed in full */
      mfma_d4 acc[BI * BJ];
      kloop(template_int<BI>{}, template_int<BJ>{}, template_int<BI * BJ>{}, [&](int i) { return BI * wm + i; },
            [&](int j) { return BJ * wn + j; }, [](int b) { return b % BI; }, [](int b) { return b / BI; }, acc);
#pragma unroll
      for (int b = 0; b < BI * BJ; ++b)
         store_block(ar0 + 16 * (BI * wm + b % BI), br0 + 16 * (BJ * wn + b / BI), acc[b]);
   } else if constexpr (TN == 128 && TM == 128 && SYM) {
      mfma_d4 acc[9];
      if (wave < 3) {
         const int r0 = dg_row(wave), c0 = dg_col(wave);
         kloop(template_int<3>{}, template_int<3>{}, template_int<9>{}, [&](int i) { return r0 + i; },
               [&](int j) { return c0 + j; }, [](int b) { return b % 3; }, [](int b) { return b / 3; }, acc);
#pragma unroll
         for (int b = 0; b < 9; ++b) store_block(ar0 + 16 * (r0 + b % 3), br0 + 16 * (c0 + b / 3), acc[b]);
      } else {
         kloop(template_int<6>{}, template_int<6>{}, template_int<9>{}, [](int i) { return dg_tri(i); },
               [](int j) { return dg_tri(j); }, [](int b) { return dg_ta(b); }, [](int b) { return dg_tb(b); }, acc);
#pragma unroll
         for (int b = 0; b < 9; ++b)
            store_block(ar0 + 16 * dg_tri(dg_ta(b)), br0 + 16 * dg_tri(dg_tb(b)), acc[b]);
      }
   }
}

/* K splits of a symmetric product: the tiles above the diagonal take sp_off
 * and the diagonal tiles sp_dd, in the ratio 16 : 18 of a full tile's blocks to
 * those of two diagonal tiles, `splits` workgroups per full tile and pair of
 * diagonal tiles.  The launch forms every diagonal tile by itself, which gives
 * it more workgroups than that; the counts stay because they decide the rounding
 * of the sums */
void gemm_tn_symm_splits(int M, size_t K, int splits, int *sp_off, int *sp_dd)
{
   const int ntm = (M + TT - 1) / TT;
   const int noff = ntm * (ntm - 1) / 2, ndd = (ntm + 1) / 2;
   const int kmax = (int)(K / KC) > 0 ? (int)(K / KC) : 1;
   if (noff == 0) {
      *sp_off = 0;
      *sp_dd = splits < kmax ? splits : kmax;
      return;
   }
   const long W = (long)(noff + ndd) * splits;
   int so = (int)(W * 16 / (16L * noff + 18L * ndd));
   if (so < 1) so = 1;
   int sd = (int)((W - (long)noff * so + ndd - 1) / ndd);
   if (sd < 1) sd = 1;
   *sp_off = so < kmax ? so : kmax;
   *sp_dd = sd < kmax ? sd : kmax;
}

/* the same for a product restricted to noff off-diagonal and nd diagonal
 * tiles over about wgs workgroups, each diagonal range formed as two halves
 * (2 sp_dd partials) */
void gemm_tn_list_splits(int noff, int nd, size_t K, long wgs, int *sp_off, int *sp_dd)
{
   const int kmax = (int)(K / KC) > 0 ? (int)(K / KC) : 1;
   const int kmax2 = kmax / 2 > 0 ? kmax / 2 : 1;
   int so = noff > 0 ? (int)(16 * wgs / (16L * noff + 9L * nd)) : 0;
   if (noff > 0 && so < 1) so = 1;
   if (so > kmax) so = kmax;
   int sd = nd > 0 ? (int)((wgs - (long)noff * so + nd - 1) / nd) : 0;
   if (nd > 0 && sd < 1) sd = 1;
   if (sd > kmax2) sd = kmax2;
   *sp_off = so;
   *sp_dd = sd;
}

/* tiles of one K split; pairs of diagonal tiles count as one, for the reason
 * given at gemm_tn_symm_splits */
int gemm_tn_tiles(int M, int N, int symm)
{
   if (symm) {
      const int ntm = (M + TT - 1) / TT;
      return ntm * (ntm - 1) / 2 + (ntm + 1) / 2;
   }
   const int pad128 = (M + 127) / 128 * 128 - M, pad96 = (M + 95) / 96 * 96 - M;
   const int tmr = pad96 < pad128 ? 96 : TT;
   return ((M + tmr - 1) / tmr) * ((N + TT - 1) / TT);
}

/* whole rounds of the 8 XCDs */
static dim3 xcd_grid(long blocks) { return dim3((unsigned)((blocks + 7) / 8 * 8)); }

static size_t k_chunk(size_t K, int sp)
{
   const size_t kc = (K + sp - 1) / sp;
   return (kc + KC - 1) / KC * KC;
}

/* The tile edge of a product formed in `splits` K ranges: 32 when 128 x 128
 * tiles would give a CU less than two workgroups and eight 32 x 32 tiles cover
 * the output, which then spread each range over several workgroups (more of
 * them read the rows too often).  The K ranges, hence the results, do not
 * depend on it.  32 against 128, 256 ranges: Gram of 64 rows at 64^3 26 and
 * 53 us, of 128 rows (ten tiles) at 80^3 136 and 118; projection 48 x 32 at
 * 64^3 24 and 60, 96 x 64 at 80^3 103 and 130. */
static int tn_tile(int M, int N, int splits, int symm)
{
   auto tiles = [&](int e) {
      const long nm = (M + e - 1) / e, nn = (N + e - 1) / e;
      return symm ? nm * (nm + 1) / 2 : nm * nn;
   };
   return tiles(TT) * splits < 512 && tiles(32) <= 8 ? 32 : TT;
}

/* the listed tiles of the symmetric product A W A^T, so and sd K ranges */
template<int TE, int KT>
static int launch_tn_list(const GramTiles &tl, const double *A, size_t lda, int M, const double *w, size_t K, int so,
                          int sd, double *partial, hipStream_t s)
{
   const long poff = (long)tl.noff * so;
   const long pairs = poff + (long)tl.nd * sd * tl.halves;
   hipLaunchKernelGGL((k_gemm_tn_splitk<TE, TE, KT, true>), dim3(xcd_grid(poff).x + xcd_grid(pairs - poff).x), dim3(256),
                      0, s, A, lda, M, A, lda, M, w, K, so > 0 ? k_chunk(K, so) : 0, sd > 0 ? k_chunk(K, sd) : 0, 0, 0,
                      poff, pairs, tl, partial);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

template<int TM, int TN, int KT>
static int launch_tn_tiles(const double *A, size_t lda, int M, const double *B, size_t ldb, int N, const double *w,
                           size_t K, int splits, double *partial, hipStream_t s)
{
   GramTiles tl;
   memset(&tl, 0, sizeof tl);
   const int ntm = (M + TM - 1) / TM, ntile = ntm * ((N + TN - 1) / TN);
   const long pairs = (long)ntile * splits;
   hipLaunchKernelGGL((k_gemm_tn_splitk<TM, TN, KT, false>), xcd_grid(pairs), dim3(256), 0, s, A, lda, M, B, ldb, N, w,
                      K, k_chunk(K, splits), 0, ntm, ntile, 0, pairs, tl, partial);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

int launch_gemm_tn_splitk(const double *A, size_t lda, int M, const double *B, size_t ldb,
                          int N, const double *w, size_t K, int splits, int symm,
                          double *partial, hipStream_t s)
{
   if (K % KC) { cpsd_set_error("gemm_tn: K=%zu not a multiple of %d", K, KC); return -1; }
   if (symm && (M != N || M > 8 * TT)) { cpsd_set_error("gemm_tn: symmetric product of %d x %d", M, N); return -1; }
   /* 32-bit lane offsets of the rows of a tile */
   if (lda * 8 * TT >= (1ull << 32) || ldb * 8 * TT >= (1ull << 32)) {
      cpsd_set_error("gemm_tn: rows of %zu doubles", lda > ldb ? lda : ldb);
      return -1;
   }
   if (symm) {
      int so, sd;
      gemm_tn_symm_splits(M, K, splits, &so, &sd);
      /* one 128 x 128 tile or less takes sd ranges throughout; more tiles
       * than that fill the GPU */
      const int te = M <= TT ? tn_tile(M, M, sd, 1) : TT;
      if (M <= TT) so = sd;
      GramTiles tl;
      memset(&tl, 0, sizeof tl);
      const int ntm = (M + te - 1) / te;
      for (int i = 0; i < ntm; ++i) {
         for (int j = i + 1; j < ntm; ++j) { tl.otm[tl.noff] = (unsigned char)i; tl.otn[tl.noff] = (unsigned char)j; ++tl.noff; }
         tl.dt[tl.nd++] = (unsigned char)i;
      }
      tl.halves = 1;
      if (te == 32) return launch_tn_list<32, 32>(tl, A, lda, M, w, K, so, sd, partial, s);
      return launch_tn_list<TT, 16>(tl, A, lda, M, w, K, so, sd, partial, s);
   }
   const int te = tn_tile(M, N, splits, 0);
   if (te == 32) return launch_tn_tiles<32, 32, 32>(A, lda, M, B, ldb, N, w, K, splits, partial, s);
   /* row tile: 128, or 96 when that leaves fewer padding rows */
   const int pad128 = (M + 127) / 128 * 128 - M, pad96 = (M + 95) / 96 * 96 - M;
   if (pad96 < pad128) return launch_tn_tiles<96, 128, 16>(A, lda, M, B, ldb, N, w, K, splits, partial, s);
   return launch_tn_tiles<128, 128, 16>(A, lda, M, B, ldb, N, w, K, splits, partial, s);
}

/* the Gram of [C1 C2] (M = 2 ne rows of stride lda, ne a multiple of 128)
 * without the C1 x C1 block: every 128 x 128 tile with a row or column in the
 * C2 block (rows [c2row, c2row + ne)) */
int launch_gram_c2(const double *A, size_t lda, int M, int c2row, const double *w, size_t K, long wgs,
                   double *partial, size_t partial_cap, int *sp_off, int *sp_dd, hipStream_t s)
{
   if (K % KC || lda * 8 * TT >= (1ull << 32)) { cpsd_set_error("gram: K=%zu not a multiple of %d, or too long", K, KC); return -1; }
   if (M % TT || c2row % TT || M > 8 * TT) {
      cpsd_set_error("gram: %d rows (C2 from row %d) are not whole 128-row tiles (at most 8)", M, c2row);
      return -1;
   }
   const int ntm = M / TT, c0 = c2row / TT, c1 = c0 + M / 2 / TT;
   auto in_c2 = [&](int t) { return t >= c0 && t < c1; };
   GramTiles tl;
   memset(&tl, 0, sizeof tl);
   for (int i = 0; i < ntm; ++i)
      for (int j = i + 1; j < ntm; ++j)
         if (in_c2(i) || in_c2(j)) { tl.otm[tl.noff] = (unsigned char)i; tl.otn[tl.noff] = (unsigned char)j; ++tl.noff; }
   for (int i = 0; i < ntm; ++i)
      if (in_c2(i)) tl.dt[tl.nd++] = (unsigned char)i;
   int so, sd;
   gemm_tn_list_splits(tl.noff, tl.nd, K, wgs, &so, &sd);
   tl.halves = 2;
   const int zmax = so > 2 * sd ? so : 2 * sd;
   if ((size_t)zmax * M * M > partial_cap) {
      cpsd_set_error("gram: %d splits of %d x %d do not fit the partial buffer", zmax, M, M);
      return -1;
   }
   *sp_off = so;
   *sp_dd = 2 * sd;
   return launch_tn_list<TT, 16>(tl, A, lda, M, w, K, so, sd, partial, s);
}

/* out[m][n] = sum_z partial[z][m][n] over the splits that formed (m, n):
 * `splits`, or for a symmetric product (symm = block edge of the formed
 * blocks) sp_dd inside the 128 x 128 diagonal tiles and `splits` elsewhere;
 * only blocks with block(m) <= block(n) exist and the rest is mirrored.  A
 * workgroup covers 64 consecutive outputs with RW waves: wave g sums the splits
 * z = g mod RW in eight interleaved chains, and the waves' sums are added in g
 * order, so the result does not depend on scheduling. */
#define RW 16   /* waves per reduction workgroup, each over every RW-th split */

/* with X non-null (KB projections: out = P, nproj x ne), also the apply
 * coefficients X[m + n M] = -P[m][n] scal2 / pnrm[m] (ccpsdv3/cpsd.c:289) */
__global__ void __launch_bounds__(64 * RW) k_reduce_partials(const double *__restrict__ partial, int splits,
                                                         int sp_dd, int M, int N, int symm, int skip0,
                                                         int skip1, double *__restrict__ out,
                                                         const double *__restrict__ pnrm, double scal2,
                                                         double *__restrict__ X)
{
   __shared__ double red[RW][64];
   const int g = threadIdx.x >> 6, l = threadIdx.x & 63;
   const size_t idx = (size_t)blockIdx.x * 64 + l;
   const int m = (int)(idx / N), n = (int)(idx % N);
   /* symmetric: the blocks below the diagonal are written from their mirror;
    * rows and columns both in [skip0, skip1) were not formed */
   const bool valid = idx < (size_t)M * N && !(symm && (m / symm) > (n / symm)) &&
                      !(m >= skip0 && m < skip1 && n >= skip0 && n < skip1);
   const int nz = (symm && m / TT == n / TT) ? sp_dd : splits;
   /* wave g sums splits g, g + RW, ... into eight accumulators, so that eight
    * loads are in flight per lane, then adds them in a fixed tree */
   double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
   if (valid) {
      const size_t stride = (size_t)M * N;
      const double *p = partial + (size_t)m * N + n;
      int z = g;
      for (; z + 7 * RW < nz; z += 8 * RW) {
#pragma unroll
         for (int u = 0; u < 8; ++u) acc[u] += p[(size_t)(z + RW * u) * stride];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
         if (z + RW * u < nz) acc[u] += p[(size_t)(z + RW * u) * stride];
   }
   red[g][l] = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
   __syncthreads();
   if (g == 0 && valid) {
      double v = red[0][l];
#pragma unroll
      for (int w = 1; w < RW; ++w) v += red[w][l];
      out[idx] = v;
      if (symm && (m / symm) < (n / symm)) out[(size_t)n * N + m] = v;
      if (X) X[m + (size_t)n * M] = -v * scal2 / pnrm[m];
   }
}

int launch_reduce_partials(const double *partial, int splits, int M, int N, double *out,
                           int symm, hipStream_t s)
{
   const size_t tot = (size_t)M * N;
   hipLaunchKernelGGL(k_reduce_partials, dim3((tot + 63) / 64), dim3(64 * RW), 0, s, partial,
                      splits, splits, M, N, symm, 0, 0, out, nullptr, 0.0, nullptr);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

int launch_reduce_partials_kb(const double *partial, int splits, int nproj, int ne, double *P, const double *pnrm,
                              double scal2, double *X, hipStream_t s)
{
   const size_t tot = (size_t)nproj * ne;
   hipLaunchKernelGGL(k_reduce_partials, dim3((tot + 63) / 64), dim3(64 * RW), 0, s, partial,
                      splits, splits, nproj, ne, 0, 0, 0, P, pnrm, scal2, X);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

int launch_reduce_partials_split(const double *partial, int sp_off, int sp_dd, int M, int skip0, int skip1,
                                 double *out, hipStream_t s)
{
   const size_t tot = (size_t)M * M;
   hipLaunchKernelGGL(k_reduce_partials, dim3((tot + 63) / 64), dim3(64 * RW), 0, s, partial,
                      sp_off, sp_dd, M, M, 16, skip0, skip1, out, nullptr, 0.0, nullptr);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

int launch_reduce_partials_symm(const double *partial, int M, size_t K, int splits, double *out,
                                hipStream_t s)
{
   int so, sd;
   gemm_tn_symm_splits(M, K, splits, &so, &sd);
   const size_t tot = (size_t)M * M;
   hipLaunchKernelGGL(k_reduce_partials, dim3((tot + 63) / 64), dim3(64 * RW), 0, s, partial,
                      so, sd, M, M, 16, 0, 0, out, nullptr, 0.0, nullptr);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

/* ------------------------------------------------- small M x N (TN) */

/* out[m][n] = sum_k w[k] A[m][k] B[n][k] for small M, N: one 1024-thread
 * workgroup per output (per upper-triangle pair m <= n when symm, mirrored),
 * its 16 waves taking interleaved 16-byte pieces of K so that many loads are
 * in flight, eight per thread; wave sums by a fixed shuffle tree, then the 16
 * wave sums in order: no split-K partials, no reduction launch, and the KB
 * apply's coefficients X in the same one.  Latency-bound: 7 us at 32^3, a
 * launch of 2 us less with X formed here. */
__global__ void __launch_bounds__(1024) k_gemm_tn_small(const double *__restrict__ A, size_t lda, int M,
                                                        const double *__restrict__ B, size_t ldb, int N,
                                                        const double *__restrict__ w, size_t K, int symm,
                                                        double *__restrict__ out, const double *__restrict__ pnrm,
                                                        double scal2, double *__restrict__ X)
{
   __shared__ double ws[16];
   const int o = blockIdx.x, t = threadIdx.x, lane = t & 63, wv = t >> 6;
   int m, n;
   if (symm) {
      int r = o;
      m = 0;
      while (r >= M - m) { r -= M - m; ++m; }
      n = m + r;
   } else {
      m = o / N;
      n = o % N;
   }
   const double *a = A + (size_t)m * lda, *b = B + (size_t)n * ldb;
   double s0 = 0.0, s1 = 0.0;
#pragma unroll 8
   for (size_t k = 2 * (size_t)t; k < K; k += 2048) {
      const double2 av = *reinterpret_cast<const double2 *>(a + k);
      const double2 bv = *reinterpret_cast<const double2 *>(b + k);
      const double2 wk = *reinterpret_cast<const double2 *>(w + k);
      s0 += (wk.x * av.x) * bv.x;
      s1 += (wk.y * av.y) * bv.y;
   }
   const double v = wave_sum(s0 + s1);
   if (lane == 0) ws[wv] = v;
   __syncthreads();
   if (t == 0) {
      double tot = 0.0;
      for (int i = 0; i < 16; ++i) tot += ws[i];
      out[(size_t)m * N + n] = tot;
      if (symm) out[(size_t)n * N + m] = tot;
      if (X) X[m + (size_t)n * M] = -tot * scal2 / pnrm[m];
   }
}

int gemm_tn_small_ok(int M, int N) { return M <= 16 && N <= 16; }

int launch_gemm_tn_small(const double *A, size_t lda, int M, const double *B, size_t ldb, int N,
                         const double *w, size_t K, int symm, double *out, const double *pnrm, double scal2, double *X,
                         hipStream_t s)
{
   if (K % 2) { cpsd_set_error("gemm_tn_small: K=%zu is odd", K); return -1; }
   if (symm && M != N) { cpsd_set_error("gemm_tn_small: symmetric product needs M == N"); return -1; }
   const long outs = symm ? (long)M * (M + 1) / 2 : (long)M * N;
   hipLaunchKernelGGL(k_gemm_tn_small, dim3((unsigned)outs), dim3(1024), 0, s, A, lda, M, B, ldb, N, w, K, symm,
                      out, pnrm, scal2, X);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

/* ---------------------------------------------------------- tall NN */

#define TK 128  /* output rows (K) per workgroup */
#define MC 16   /* reduction step */


/* Output tile: TK = 128 rows of K x NT columns over 4 waves: 64 K rows x 64
 * columns each (NT = 128), or 32 K rows x 64 columns (NT = 64).  32 K rows are
 * two 16-column MFMA blocks, the even and the odd ones, so that one 16-byte
 * LDS read feeds both and a lane ends up with whole complex coefficients: 16
 * lanes hold 256 contiguous bytes of an output row and the SD epilogues run
 * straight from the accumulators.  At most 256 VGPRs and 70 KB of LDS: two
 * workgroups share a CU and one's epilogue traffic overlaps the other's MFMA
 * stream.  Bound by the MFMA issue and, for short reductions, by the C2
 * update: at 64 waters the KB apply takes 3.6 ms (60
 * TFLOP/s) and the constraint 2.5 (4.28 and 2.93 ms with v_mfma_f64_4x4x4_4b
 * and DPP-rotated operands). */
template<int EPI, int NT>
__global__ void __launch_bounds__(256, 2) k_gemm_tall(TallArgs a)
{
   constexpr int BJ = NT < 64 ? NT / 16 : 4;                  /* 16-column blocks per wave */
   constexpr int WN = NT == 128 ? 2 : 1, WK = 4 / WN;         /* waves along the columns and along K */
   constexpr int BP = TK / WK / 32;          /* block pairs along K per wave */
   constexpr int XP = MC + 2;                /* X pitch: 16-byte reads of 8 rows cover the banks once */
   __shared__ __align__(16) double panels[2 * MC * TK + 2 * NT * XP];
   double (*const As)[MC][TK] = reinterpret_cast<double (*)[MC][TK]>(panels);
   double (*const Xs)[NT][XP] = reinterpret_cast<double (*)[NT][XP]>(panels + 2 * MC * TK);
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int l16 = lane & 15, lq4 = lane >> 4;
   const int wk = wave % WK, wn = wave / WK;
   /* block -> (K block, column tile) with the column tile fastest, remapped
    * so that the workgroups one XCD runs together (block id mod 8) hold
    * consecutive pairs: the column tiles of one K block then read its A
    * rows through the same L2 */
   const int g = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
   if (g >= a.blocks) return;
   const size_t k0 = (size_t)(g / a.ntn) * TK;
   const int n0 = (g % a.ntn) * NT;
   mfma_d4 acc[BJ][BP][2];   /* [column block][K pair][even, odd K rows] */
#pragma unroll
   for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int p = 0; p < BP; ++p) acc[j][p][0] = acc[j][p][1] = mfma_d4{0.0, 0.0, 0.0, 0.0};

   /* loaders: A chunk MC x TK, rows ar + 4 h with 64 lanes per 1 KB row; X
    * chunk NT x MC.  No branches: rows past Mr repeat the last one with X = 0,
    * columns past Nc repeat the last one and are not written. */
   constexpr int XQ = NT * MC / 256;
   static_assert(TK == 128 && MC == 16, "A loader covers 16 rows of 128");
   const int ar = tid >> 6, ac = (tid & 63) * 2;
   double2 ra[4];
   double rx[XQ];
   const char *const xbase = reinterpret_cast<const char *>(a.X);
   unsigned xo[XQ];
#pragma unroll
   for (int u = 0; u < XQ; ++u) xo[u] = (unsigned)min(n0 + (tid + 256 * u) / MC, a.Nc - 1) * (unsigned)(a.ldx * 8);
   const int xm = tid % MC, xp = (xm & 8) + 2 * (xm & 3) + ((xm >> 2) & 1);   /* m and m + 4 adjacent */
   auto gload = [&](int m0) {
      const char *const ab = reinterpret_cast<const char *>(a.A + (size_t)m0 * a.lda + k0);
      const int last = a.Mr - 1 - m0;
#pragma unroll
      for (int h = 0; h < 4; ++h)
         ra[h] = load2(ab, (unsigned)min(ar + 4 * h, last) * (unsigned)(a.lda * 8) + ac * 8);
      const unsigned xr = (unsigned)(m0 + min(xm, last)) * (unsigned)(a.xsm * 8);
#pragma unroll
      for (int u = 0; u < XQ; ++u) rx[u] = *reinterpret_cast<const double *>(xbase + (xo[u] + xr));
   };
   auto lstore = [&](int bf, int m0) {
#pragma unroll
      for (int h = 0; h < 4; ++h) *reinterpret_cast<double2 *>(&As[bf][ar + 4 * h][ac]) = ra[h];
#pragma unroll
      for (int u = 0; u < XQ; ++u) Xs[bf][(tid + 256 * u) / MC][xp] = m0 + xm < a.Mr ? rx[u] : 0.0;
   };
   /* 8 of the chunk's rows m, in order: lane group lq4 supplies rows 8 ks +
    * lq4 and 8 ks + 4 + lq4 to two successive instructions */
   struct Frag { double2 x[BJ], b[BP][2]; };
   auto fread = [&](Frag &f, int bf, int ks) {
#pragma unroll
      for (int j = 0; j < BJ; ++j)
         f.x[j] = *reinterpret_cast<const double2 *>(&Xs[bf][64 * wn + 16 * j + l16][8 * ks + 2 * lq4]);
#pragma unroll
      for (int p = 0; p < BP; ++p)
#pragma unroll
         for (int u = 0; u < 2; ++u)
            f.b[p][u] = *reinterpret_cast<const double2 *>(&As[bf][8 * ks + 4 * u + lq4][(TK / WK) * wk + 32 * p + 2 * l16]);
   };
   auto mma = [&](const Frag &f) {
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
         for (int p = 0; p < BP; ++p) {
            acc[j][p][0] = mfma16(f.x[j].x, f.b[p][0].x, acc[j][p][0]);
            acc[j][p][1] = mfma16(f.x[j].x, f.b[p][0].y, acc[j][p][1]);
         }
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
         for (int p = 0; p < BP; ++p) {
            acc[j][p][0] = mfma16(f.x[j].y, f.b[p][1].x, acc[j][p][0]);
            acc[j][p][1] = mfma16(f.x[j].y, f.b[p][1].y, acc[j][p][1]);
         }
   };

   /* chunk c+1 waits in registers while chunk c is multiplied; the operands of
    * the next 8 rows are read from LDS between the current ones' MFMAs; one
    * barrier per chunk, after which every read of the chunk has returned */
   if (a.Mr > 0) {   /* an empty reduction (no projectors) leaves the product zero */
      const int nc = (a.Mr + MC - 1) / MC;
      gload(0);
      lstore(0, 0);
      gload(nc > 1 ? MC : 0);
      __syncthreads();
      Frag f0, f1;
      fread(f0, 0, 0);
      int buf = 0;
      for (int c = 0; c + 1 < nc; ++c) {
         fread(f1, buf, 1);
         mma(f0);
         lstore(buf ^ 1, (c + 1) * MC);
         sched_mix<0x100, BJ + 2 * BP, 1>();
         sched_mix<0x200, 4 + XQ, 1>();
         __syncthreads();
         buf ^= 1;
         fread(f0, buf, 0);
         gload(min(c + 2, nc - 1) * MC);
         mma(f1);
         sched_mix<0x100, BJ + 2 * BP, 1>();
         sched_mix<0x20, 4 + XQ, 1>();
      }
      fread(f1, buf, 1);
      mma(f0);
      mma(f1);
   }

   /* epilogue: register r of block (j, p) is row n of the output at complex
    * coefficient (k0 + 32 p') / 2 + l16; the loads of a block pair are issued
    * before its stores */
   const size_t kw = k0 + (TK / WK) * wk + 2 * l16;
   if constexpr (EPI == EPI_NLFORCE) {
      /* Z_n(G) against the projectors (ccpsdv3/cpsd.c:296-302 with the orbital
       * sum moved inside): 32 columns at a time staged in LDS, then a wave
       * per row with a lane per G and the wave's fixed shuffle tree */
      double (*T)[TK + 2] = reinterpret_cast<double (*)[TK + 2]>(panels);
      static_assert(32 * (TK + 2) <= 2 * MC * TK + 2 * NT * XP, "staging fits the panels");
#pragma unroll
      for (int half = 0; half < NT / 32; ++half) {
         __syncthreads();
         if (wn == half >> 1) {
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
               for (int p = 0; p < BP; ++p)
#pragma unroll
                  for (int r = 0; r < 4; ++r) {
                     const int j = 2 * (half & 1) + jj;
                     *reinterpret_cast<double2 *>(&T[16 * jj + mfma16_row(r, lane)][(TK / WK) * wk + 32 * p + 2 * l16]) =
                        make_double2(acc[j][p][0][r], acc[j][p][1][r]);
                  }
         }
         __syncthreads();
         for (int nl = wave; nl < 32; nl += 4) {
            const int n = n0 + 32 * half + nl;
            if (n >= a.Nc) break;
            const double2 v = make_double2(T[nl][2 * lane], T[nl][2 * lane + 1]);
            const size_t gq = (k0 >> 1) + lane;
            const double2 b = a.Bp[(size_t)n * a.ngp + gq];
            const double t = a.w[k0 + 2 * lane] * (v.y * b.x - v.x * b.y);
            const double f0 = wave_sum(a.Gp[gq] * t);
            const double f1 = wave_sum(a.Gp[(size_t)a.ngp + gq] * t);
            const double f2 = wave_sum(a.Gp[2 * (size_t)a.ngp + gq] * t);
            if (lane == 0) {
               double *o = a.fpart + ((size_t)(k0 / TK) * a.Nc + n) * 3;
               o[0] = f0; o[1] = f1; o[2] = f2;
            }
         }
      }
   } else {
      /* column blocks whose rows are fetched together: the operands' registers
       * are free now, and the compiler may not move a load over a store (one
       * block at a time: constraint of 64 orbitals at 80^3 93 -> 85 us, KB apply
       * and constraint of 256 at 128^3 2.98 -> 2.92 ms on average; four at 128
       * columns spill, 3.00) */
      constexpr int EJ = BJ < 2 || (EPI == EPI_CONSTRAINT && NT < 128) ? BJ : 2;
#pragma unroll
      for (int p = 0; p < BP; ++p) {
         const size_t kc = kw + 32 * p;
         double f = 0.0;
         if (EPI == EPI_PRECOND) f = a.Kp[kc >> 1];
#pragma unroll
         for (int j0 = 0; j0 < BJ; j0 += EJ) {
            double2 c2[EJ][4], c1[EJ][4], cp[EJ][4];
            auto at = [&](int j, int r) {   /* columns past Nc load the last one */
               return (size_t)min(n0 + 64 * wn + 16 * j + mfma16_row(r, lane), a.Nc - 1) * a.ldc + kc;
            };
#pragma unroll
            for (int j = j0; j < j0 + EJ; ++j)
#pragma unroll
               for (int r = 0; r < 4; ++r) {
                  const size_t o = at(j, r);
                  if (EPI == EPI_CONSTRAINT || EPI == EPI_PRECOND) c2[j - j0][r] = *reinterpret_cast<const double2 *>(a.C2 + o);
                  if (EPI == EPI_KBAPPLY || EPI == EPI_PRECOND) c1[j - j0][r] = *reinterpret_cast<const double2 *>(a.C1 + o);
                  if (EPI == EPI_KBAPPLY) cp[j - j0][r] = *reinterpret_cast<const double2 *>(a.CP + o);
               }
#pragma unroll
            for (int j = j0; j < j0 + EJ; ++j)
#pragma unroll
               for (int r = 0; r < 4; ++r) {
                  if (n0 + 64 * wn + 16 * j + mfma16_row(r, lane) >= a.Nc) continue;
                  const double2 v = make_double2(acc[j][p][0][r], acc[j][p][1][r]);
                  const double2 d2 = c2[j - j0][r], d1 = c1[j - j0][r];
                  const size_t e = at(j, r);
                  double2 o = v;
                  if (EPI == EPI_KBAPPLY) {
                     double2 h = cp[j - j0][r];
                     h.x += v.x; h.y += v.y;
                     o = make_double2(d1.x + a.dte * h.x, d1.y + a.dte * h.y);
                     if (a.write_cp) *reinterpret_cast<double2 *>(a.CP + e) = h;
                  } else if (EPI == EPI_CONSTRAINT) {
                     o = make_double2(d2.x + a.dte * v.x, d2.y + a.dte * v.y);
                  } else if (EPI == EPI_PRECOND) {
                     o.x = d1.x + f * (d2.x - d1.x + a.dte * v.x);
                     o.y = d1.y + f * (d2.y - d1.y + a.dte * v.y);
                  }
                  *reinterpret_cast<double2 *>(a.C2 + e) = o;
               }
         }
      }
   }
}

template<int NT>
static void gemm_tall_go(int epi, TallArgs &a, hipStream_t s)
{
   a.ntn = (a.Nc + NT - 1) / NT;
   a.blocks = (int)(a.K / TK) * a.ntn;
   const dim3 g = xcd_grid(a.blocks), t(256);
   if (epi == EPI_KBAPPLY) hipLaunchKernelGGL((k_gemm_tall<EPI_KBAPPLY, NT>), g, t, 0, s, a);
   else if (epi == EPI_CONSTRAINT) hipLaunchKernelGGL((k_gemm_tall<EPI_CONSTRAINT, NT>), g, t, 0, s, a);
   else if (epi == EPI_STORE) hipLaunchKernelGGL((k_gemm_tall<EPI_STORE, NT>), g, t, 0, s, a);
   else if (epi == EPI_PRECOND) hipLaunchKernelGGL((k_gemm_tall<EPI_PRECOND, NT>), g, t, 0, s, a);
   else hipLaunchKernelGGL((k_gemm_tall<EPI_NLFORCE, NT>), g, t, 0, s, a);
}

int launch_gemm_tall(int epi, const TallArgs &args, hipStream_t s)
{
   if (args.K % TK) { cpsd_set_error("gemm_tall: K=%zu not a multiple of %d", args.K, TK); return -1; }
   /* 32-bit lane offsets of the MC rows of a chunk */
   if (args.lda * 8 * MC >= (1ull << 32)) { cpsd_set_error("gemm_tall: rows of %zu doubles", args.lda); return -1; }
   TallArgs a = args;
   /* 128 columns per workgroup read A and X half as often as 64; 64 where
    * they pad less; 32 for small outputs, whose workgroups then hold less and
    * overlap more of each other's loads (constraint of 32 orbitals at 64^3 30
    * -> 21 us, nonlocal force of 48 projectors 49 -> 45) */
   if (a.Nc <= 32 || (epi == EPI_NLFORCE && a.Nc <= 64)) gemm_tall_go<32>(epi, a, s);
   else if ((a.Nc + 127) / 128 * 2 == (a.Nc + 63) / 64) gemm_tall_go<128>(epi, a, s);
   else gemm_tall_go<64>(epi, a, s);
   CPSD_CHECK(hipGetLastError());
   return 0;
}
