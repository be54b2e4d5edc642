/*
 * fft_kernels.hip -- batched 3D real<->half-complex FFTs of the SD step on
 * gfx950, FP64, with FP32 variants of the orbital passes (the transforms
 * run on float2 in LDS and T; inputs, the density sum and the outputs stay
 * FP64).
 *
 * The 3D transform of cr_fft3b / rc_fft3f (fftpack3d/fftpack3d.f:22-96,
 * 107-196) is split into
 *   z pass   : one workgroup per (32 columns, orbitals).  G->r reads the packed
 *              masked coefficients directly (zero fill outside the sphere);
 *              r->G writes only masked coefficients, with the SD epilogue
 *              fused.  One trip through LDS: a workgroup's global reads are the
 *              items of pass 1, its writes those of pass 2.
 *   y+x pass : one workgroup per (z plane, orbital [block]); the (ky, kx) plane
 *              of N x (N/2+1) complex lives in LDS (133 KB at N = 128), the y
 *              transforms and the real x transform run back to back, and the
 *              real-space work (density, V*psi) is fused between the inverse
 *              and forward x transforms.
 * The y and z passes run over kx = 0..N/2 before the x pass, as the
 * reference does, so the imaginary parts of kx = 0 and kx = N/2 are dropped
 * at the same point (the complex-to-real x transform); rc_fft3f's zeroing of
 * Im(kx=0) and Im(kx=N/2) is reproduced after the forward x transform.
 *
 * The plane pass of V psi takes seven LDS trips, each one barrier:
 *   y pass 1 from the registers the plane was fetched into; y pass 2; the
 *   half-length x transform's pre-twiddle with x pass 1 (the mirror pairs k,
 *   N/2 - k lie in items n2 and NX2 - n2, which one thread takes together); x
 *   pass 2, times V, forward x pass 1 (the same slots); forward x pass 2 with
 *   the post-twiddle; forward y pass 1; forward y pass 2 straight to T.
 * Stages are kept from contracting into each other (opaque), so results are
 * those of one trip per pass.  At 128^3 and 256 orbitals V psi takes 2.37 ms
 * (3.27 with eleven trips and 0.27 more of T), the density 1.16 (1.41), FP32
 * 1.26 (1.47) and 0.73 (0.97).  An FP64 V psi plane takes a CU about 44,000
 * cycles: 25,000 of HBM traffic at the rate of a large copy, 18,000 of vector ALU
 * (busy 0.44) and 13,000 of LDS (twelve passes over the plane at 128 bytes a
 * cycle), in part one after the other, as one workgroup of eight waves fits a CU.
 * The FP32 passes are bound by the vector ALU (busy 0.87 and 0.72).
 */
#include "cpsd_internal.h"
#include "fft_core.h"
#include <string.h>
#include <algorithm>

/* ------------------------------------------------------------ z passes */

/* block -> (column block, orbital group), column blocks fastest.  Workgroups
 * go to the 8 XCDs round-robin, and neighbouring column blocks share lines of
 * the packed orbitals at their edges, so every XCD runs a contiguous range. */
__device__ __forceinline__ bool zpass_block(int ncb, int ngrp, int &cb, int &grp)
{
   const int l = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
   cb = l % ncb;
   grp = l / ncb;
   return grp < ngrp;
}

/* packed coefficient of (kz, column c), -1 outside the mask */
template<int N, bool FULL>
__device__ __forceinline__ int zpass_index(const ColTable &t, int kz, int c)
{
   if (FULL) return c < t.P ? kz * N * (N / 2 + 1) + c : -1;
   return c < t.P ? at(t.gmap, kz * t.P + c) : -1;
}

/* waves per SIMD: what the LDS column block admits, at most 3 */
template<int N, typename V>
constexpr int zpass_waves()
{
   constexpr int wg = (int)(160L * 1024 / ((long)(N * ZKB + N) * (long)sizeof(V)));
   return wg < 1 ? 1 : wg > 3 ? 3 : wg;
}

/* G -> r along kz for bper orbitals: the gather of orbital b+1 goes into the
 * registers pass 1 leaves free while orbital b is in LDS.  HBM-bound: at 128^3
 * and 256 orbitals 1.16 ms, 4.9 TB/s (1.83 with whole rows of T and four LDS
 * passes), FP32 0.80 (1.37). */
template<int N, bool FULL, typename V>
__global__ void __launch_bounds__(ZT, (zpass_waves<N, V>())) k_zpass_g2r(ZArgs a)
{
   using C = GridCfg<N>;
   constexpr int N1 = C::NY1, N2 = C::NY2;
   constexpr int I1 = (ZKB * N2 + ZT - 1) / ZT, I2 = (ZKB * N1 + ZT - 1) / ZT;
   __shared__ __align__(16) V sm[N * ZKB];
   __shared__ V tws[N];
   int cb, grp;
   const int ncb = (a.cols.P + ZKB - 1) / ZKB;
   if (!zpass_block(ncb, (a.nbatch + a.bper - 1) / a.bper, cb, grp)) return;
   const int c0 = cb * ZKB, P = a.cols.P, tid0 = threadIdx.x;
   int tid;
   const int b0 = grp * a.bper, b1 = min(a.nbatch, b0 + a.bper);
   for (int m = tid0; m < N; m += ZT) tws[m] = cvt<V>(a.tw[m]);
   int pe[I1][N1];
   tid = fresh(tid0);
#pragma unroll
   for (int q = 0; q < I1; ++q)
#pragma unroll
      for (int n1 = 0; n1 < N1; ++n1) {
         const int it = tid + ZT * q;
         pe[q][n1] = it < ZKB * N2 ? zpass_index<N, FULL>(a.cols, N2 * n1 + it / ZKB, c0 + it % ZKB) : -1;
      }
   V v[I1][N1];
   auto gather = [&](int b) {
      const double2 *src = a.src + (size_t)b * a.sstride;
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < I1; ++q)
#pragma unroll
         for (int n1 = 0; n1 < N1; ++n1) {
            const int p = fresh(pe[q][n1]);
            v[q][n1] = cvt<V>(p >= 0 ? at(src, p) : make_double2(0.0, 0.0));
         }
   };
   gather(b0);
   __syncthreads();
   for (int b = b0; b < b1; ++b) {
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < I1; ++q) {
         const int it = tid + ZT * q, col = it % ZKB, n2 = it / ZKB;
         if (it < ZKB * N2) {
            pass_dft_tw<N, N1, +1>(v[q], n2, tws, 1);
#pragma unroll
            for (int k1 = 0; k1 < N1; ++k1) sm[(N2 * k1 + n2) * ZKB + col] = v[q][k1];
         }
         item_end();
      }
      __syncthreads();
      if (b + 1 < b1) gather(b + 1);
      V *T = reinterpret_cast<V *>(a.T) + (size_t)b * N * P;
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < I2; ++q) {
         const int it = tid + ZT * q, col = it % ZKB, k1 = it / ZKB;
         if (it < ZKB * N1) {
            V u[N2];
#pragma unroll
            for (int n2 = 0; n2 < N2; ++n2) u[n2] = sm[(N2 * k1 + n2) * ZKB + col];
            pass_dft<N2, +1>(u);
            if (c0 + col < P) {
#pragma unroll
               for (int k2 = 0; k2 < N2; ++k2) at(T, (k1 + N1 * k2) * P + c0 + col) = u[k2];
            }
         }
      }
      __syncthreads();
   }
}

/* r -> G along kz for bper orbitals, each with its kinetic inputs fetched
 * before the LDS trip (the workgroups of a CU overlap one another).  At 128^3
 * and 256 orbitals (DST_SD) 1.91 ms, 4.2 TB/s (2.03 before), FP32 1.59 (1.83). */
template<int N, int DST, typename V>
__global__ void __launch_bounds__(ZT, (zpass_waves<N, V>())) k_zpass_r2g(ZArgs a)
{
   using C = GridCfg<N>;
   constexpr int N1 = C::NY1, N2 = C::NY2;
   constexpr int I1 = (ZKB * N1 + ZT - 1) / ZT, I2 = (ZKB * N2 + ZT - 1) / ZT;
   constexpr bool FULL = DST == DST_FULL;
   __shared__ __align__(16) V sm[N * ZKB];
   __shared__ V tws[N];
   int cb, grp;
   const int ncb = (a.cols.P + ZKB - 1) / ZKB;
   if (!zpass_block(ncb, (a.nbatch + a.bper - 1) / a.bper, cb, grp)) return;
   const int c0 = cb * ZKB, P = a.cols.P, tid0 = threadIdx.x;
   int tid;
   const int b0 = grp * a.bper, b1 = min(a.nbatch, b0 + a.bper);
   for (int m = tid0; m < N; m += ZT) tws[m] = cvt<V>(a.tw[m]);
   V v[I1][N2];
   auto fetch = [&](int b) {
      const V *T = reinterpret_cast<const V *>(a.T) + (size_t)b * N * P;
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < I1; ++q) {
         const int it = tid + ZT * q, c = min(c0 + it % ZKB, P - 1), n1 = it / ZKB;
         if (it < ZKB * N1) {
#pragma unroll
            for (int n2 = 0; n2 < N2; ++n2) v[q][n2] = at(T, (n1 + N1 * n2) * P + c);
         }
      }
   };
   int pe[I2][N1];
   tid = fresh(tid0);
#pragma unroll
   for (int q = 0; q < I2; ++q)
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) {
         const int it = tid + ZT * q;
         pe[q][k1] = it < ZKB * N2 ? zpass_index<N, FULL>(a.cols, N2 * k1 + it / ZKB, c0 + it % ZKB) : -1;
      }
   for (int b = b0; b < b1; ++b) {
      fetch(b);
      __syncthreads();   /* twiddles; the previous orbital's pass 2 has read the columns */
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < I1; ++q) {
         const int it = tid + ZT * q, col = it % ZKB, n1 = it / ZKB;
         if (it < ZKB * N1) {
            pass_dft_tw<N, N2, -1>(v[q], n1, tws, 1);
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) sm[(N2 * n1 + k2) * ZKB + col] = v[q][k2];
         }
         item_end();
      }
      double2 c[N1];
      double t[N1];
      auto kinetic = [&](int q) {
         const double2 *c1 = a.c1 + (size_t)b * a.ostride;
#pragma unroll
         for (int k1 = 0; k1 < N1; ++k1) {
            const int p = fresh(max(pe[q][k1], 0));   /* outside the mask: not used */
            c[k1] = at(c1, p);
            t[k1] = at(a.tg, p);
         }
         item_end();
      };
      if (!FULL) kinetic(0);
      __syncthreads();
      double2 *out = a.out + (size_t)b * a.ostride;
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < I2; ++q) {
         const int it = tid + ZT * q, col = it % ZKB, k2 = it / ZKB;
         if (!FULL && q > 0) kinetic(q);
         if (it < ZKB * N2) {
            V u[N1];
#pragma unroll
            for (int n1 = 0; n1 < N1; ++n1) u[n1] = sm[(N2 * n1 + k2) * ZKB + col];
            pass_dft<N1, -1>(u);
#pragma unroll
            for (int k1 = 0; k1 < N1; ++k1) {
               const double2 f = to_d2(u[k1]);
               double2 r = f;
               if (!FULL) {
                  r = make_double2(-a.scal1 * f.x - t[k1] * c[k1].x, -a.scal1 * f.y - t[k1] * c[k1].y);
                  if (DST == DST_SD) r = make_double2(c[k1].x + a.dte * r.x, c[k1].y + a.dte * r.y);
               }
               const int p = fresh(pe[q][k1]);
               if (p >= 0) at(out, p) = r;
            }
         }
         item_end();
      }
   }
}

/* One field in place along z: T (the density's planes) -> out = dng, its
 * masked G coefficients -> T of the local potential vall scal2 + dng vc.  The
 * columns hold the whole kz range, so both transforms of a column run in one
 * workgroup. */
template<int N>
__global__ void __launch_bounds__(ZT) k_zpass_field(ZArgs a)
{
   using C = GridCfg<N>;
   using V = double2;
   constexpr int N1 = C::NY1, N2 = C::NY2;
   constexpr int I1 = (ZKB * N1 + ZT - 1) / ZT, I2 = (ZKB * N2 + ZT - 1) / ZT;
   __shared__ __align__(16) V sm[N * ZKB];
   __shared__ V tws[N];
   const int c0 = blockIdx.x * ZKB, P = a.cols.P, tid0 = threadIdx.x;
   int tid;
   for (int m = tid0; m < N; m += ZT) tws[m] = a.tw[m];
   V v[I1][N2];
   tid = fresh(tid0);
#pragma unroll
   for (int q = 0; q < I1; ++q) {
      const int it = tid + ZT * q, c = min(c0 + it % ZKB, P - 1), n1 = it / ZKB;
      if (it < ZKB * N1) {
#pragma unroll
         for (int n2 = 0; n2 < N2; ++n2) v[q][n2] = at(a.T, (n1 + N1 * n2) * P + c);
      }
   }
   V vl[I2][N1];
   double vc[I2][N1];
   int pe[I2][N1];
   tid = fresh(tid0);
#pragma unroll
   for (int q = 0; q < I2; ++q)
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) {
         const int it = tid + ZT * q;
         pe[q][k1] = it < ZKB * N2 ? zpass_index<N, false>(a.cols, N2 * k1 + it / ZKB, c0 + it % ZKB) : -1;
         vl[q][k1] = pe[q][k1] >= 0 ? a.vall[pe[q][k1]] : make_double2(0.0, 0.0);
         vc[q][k1] = pe[q][k1] >= 0 ? a.vc[pe[q][k1]] : 0.0;
      }
   __syncthreads();
   tid = fresh(tid0);
#pragma unroll
   for (int q = 0; q < I1; ++q) {
      const int it = tid + ZT * q, col = it % ZKB, n1 = it / ZKB;
      if (it < ZKB * N1) {
         pass_dft_tw<N, N2, -1>(v[q], n1, tws, 1);
#pragma unroll
         for (int k2 = 0; k2 < N2; ++k2) sm[(N2 * n1 + k2) * ZKB + col] = v[q][k2];
      }
   }
   __syncthreads();
   /* pass 2 of the forward transform holds the kz of pass 1 of the inverse */
   tid = fresh(tid0);
#pragma unroll
   for (int q = 0; q < I2; ++q) {
      const int it = tid + ZT * q, col = it % ZKB, k2 = it / ZKB;
      if (it < ZKB * N2) {
         V u[N1];
#pragma unroll
         for (int n1 = 0; n1 < N1; ++n1) u[n1] = sm[(N2 * n1 + k2) * ZKB + col];
         pass_dft<N1, -1>(u);
#pragma unroll
         for (int k1 = 0; k1 < N1; ++k1) {
            const int p = pe[q][k1];
            const double2 dg = u[k1];
            if (p >= 0) a.out[p] = dg;
            u[k1] = p >= 0 ? make_double2(fma(vl[q][k1].x, a.scal2, dg.x * vc[q][k1]),
                                          fma(vl[q][k1].y, a.scal2, dg.y * vc[q][k1]))
                           : make_double2(0.0, 0.0);
         }
         pass_dft_tw<N, N1, +1>(u, k2, tws, 1);
#pragma unroll
         for (int n1 = 0; n1 < N1; ++n1) sm[(N2 * n1 + k2) * ZKB + col] = u[n1];
      }
   }
   __syncthreads();
   tid = fresh(tid0);
#pragma unroll
   for (int q = 0; q < I1; ++q) {
      const int it = tid + ZT * q, col = it % ZKB, k1 = it / ZKB;
      if (it < ZKB * N1) {
         V u[N2];
#pragma unroll
         for (int n2 = 0; n2 < N2; ++n2) u[n2] = sm[(N2 * k1 + n2) * ZKB + col];
         pass_dft<N2, +1>(u);
         if (c0 + col < P) {
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) at(a.T, (k1 + N1 * k2) * P + c0 + col) = u[k2];
         }
      }
   }
}

/* ------------------------------------------------------ plane stages */

/* The half-length complex transform of the real x transform, M = N/2.
 * Inverse (pre): Z_k = (X_k + conj X_{M-k}) + i W^k (X_k - conj X_{M-k}), W =
 * e^{2 pi i/N}; only Re X_0 and Re X_M are used (drfftb ignores their
 * imaginary parts).  Here for the pair k < M - k. */
template<typename V>
__device__ __forceinline__ void pre_pair(V &xk, V &xm, V w)
{
   opaque(xk);
   opaque(xm);
   const V a = xk, b = xm;
   const V wm = Cx<V>::mk(-w.x, w.y);  /* W^{M-k} = -conj(W^k) */
   xk = cadd(cadd(a, cconj(b)), cmuli(cmul(w, csub(a, cconj(b)))));
   xm = cadd(cadd(b, cconj(a)), cmuli(cmul(wm, csub(b, cconj(a)))));
   opaque(xk);
   opaque(xm);
}
template<typename V>
__device__ __forceinline__ void pre_self(V &x, V w)   /* k = M/2 */
{
   opaque(x);
   const V a = x;
   x = cadd(cadd(a, cconj(a)), cmuli(cmul(w, csub(a, cconj(a)))));
   opaque(x);
}
/* forward (post): X_k = (Z_k + conj Z_{M-k})/2 - (i/2) W^{-k} (Z_k - conj
 * Z_{M-k}) */
template<typename V>
__device__ __forceinline__ void post_pair(V &xk, V &xm, V tw)
{
   using R = typename Cx<V>::R;
   opaque(xk);
   opaque(xm);
   const V za = xk, zb = xm;
   const V w = cconj(tw);                        /* W^{-k} */
   const V wm = Cx<V>::mk(-tw.x, -tw.y);         /* W^{-(M-k)} = -W^k */
   const V sa = cadd(za, cconj(zb)), da = csub(za, cconj(zb));
   const V sb = cadd(zb, cconj(za)), db = csub(zb, cconj(za));
   const V ta = cmuli(cmul(w, da)), tb = cmuli(cmul(wm, db));
   xk = Cx<V>::mk(R(0.5) * (sa.x - ta.x), R(0.5) * (sa.y - ta.y));
   xm = Cx<V>::mk(R(0.5) * (sb.x - tb.x), R(0.5) * (sb.y - tb.y));
   opaque(xk);
   opaque(xm);
}
template<typename V>
__device__ __forceinline__ void post_self(V &x, V tw)
{
   using R = typename Cx<V>::R;
   opaque(x);
   const V z = x;
   const V w = cconj(tw);
   const V sa = cadd(z, cconj(z)), ta = cmuli(cmul(w, csub(z, cconj(z))));
   x = Cx<V>::mk(R(0.5) * (sa.x - ta.x), R(0.5) * (sa.y - ta.y));
   opaque(x);
}

/* Units of the x passes that carry the mirror pairs: unit 0 takes item 0 and,
 * for even NX2, item NX2/2, which mirror into themselves; unit u > 0 takes
 * items u and NX2 - u, which mirror into each other.  Element n1 of item i is
 * k = NX2 n1 + i; NP the inverse pre-twiddle (then DFT and twiddles), the
 * forward post-twiddle otherwise (after the DFT). */
template<int NX2> constexpr int x_units() { return NX2 / 2 + (NX2 & 1); }

template<int N, bool NYQ, bool INV, typename V>
__device__ __forceinline__ void x_unit(V *row, int u, const V *__restrict__ tw)
{
   using C = GridCfg<N>;
   using R = typename Cx<V>::R;
   constexpr int X1 = C::NX1, X2 = C::NX2, M = N / 2;
   constexpr bool EVEN = X2 % 2 == 0;
   const int i0 = u, i1 = u == 0 ? (EVEN ? X2 / 2 : 0) : X2 - u;
   const bool two = u > 0 || EVEN;
   V a[X1], b[X1];
   auto load = [&](V (&v)[X1], int i) {
#pragma unroll
      for (int n = 0; n < X1; ++n) v[n] = row[X2 * n + i];
      if (!INV) {
         pass_dft<X1, -1>(v);
         item_end();
      }
   };
   auto store = [&](V (&v)[X1], int i) {
      if (INV) {
         item_end();
         pass_dft_tw<M, X1, +1>(v, i, tw, 2);
      }
#pragma unroll
      for (int n = 0; n < X1; ++n) row[X2 * n + i] = v[n];
   };
   load(a, i0);
   if (two) load(b, i1);
   auto pair = [&](V &xk, V &xm, int k) {
      if (INV) pre_pair(xk, xm, tw[k]);
      else post_pair(xk, xm, tw[k]);
   };
   auto self = [&](V &x) {
      if (INV) pre_self(x, tw[M / 2]);
      else post_self(x, tw[M / 2]);
   };
   if (u == 0) {
      if (INV) {
         const R x0 = a[0].x, xm = NYQ ? row[M].x : R(0);
         a[0] = Cx<V>::mk(x0 + xm, x0 - xm);
      } else {
         const V z0 = a[0];
         a[0] = Cx<V>::mk(z0.x + z0.y, R(0));
         if (NYQ) row[M] = Cx<V>::mk(z0.x - z0.y, R(0));
      }
#pragma unroll
      for (int n = 1; n < (X1 + 1) / 2; ++n) pair(a[n], a[X1 - n], X2 * n);
      if (X1 % 2 == 0) self(a[X1 / 2]);
      if (EVEN) {
#pragma unroll
         for (int n = 0; n < X1 / 2; ++n) pair(b[n], b[X1 - 1 - n], X2 * n + X2 / 2);
         if (X1 % 2 == 1) self(b[X1 / 2]);
      }
   } else {
#pragma unroll
      for (int n = 0; n < X1; ++n) {
         /* k = X2 n + u; below M/2 for n <= (X1 - 1) / 2 as u < X2/2 */
         if (2 * n + 1 <= X1) pair(a[n], b[X1 - 1 - n], X2 * n + u);
         else pair(b[X1 - 1 - n], a[n], X2 * (X1 - 1 - n) + X2 - u);
      }
   }
   store(a, i0);
   if (two) store(b, i1);
}

/* ------------------------------------------------------- plane kernel */

/* threads of a plane workgroup: two FP64 planes at N = 96 fit a CU; the density
 * sums of 512 threads would leave 128 registers and spill (0.50 ms on 32
 * waters at 512, 0.33 at 256; V psi 0.54 and 0.56) */
template<int N, int MODE, typename V>
constexpr int plane_threads()
{
   return N == 96 && sizeof(V) == 16 && MODE == PM_DENSITY ? 256 : GridCfg<N>::PLANE_THREADS;
}

/* The V psi and density passes fetch the next orbital's plane into registers
 * while the current one is in LDS where a plane fills at least a third of
 * the LDS (N = 128): such planes leave one or two workgroups per CU. */
template<int N, int MODE, typename V>
constexpr bool plane_prefetch()
{
   return N >= 112 && (sizeof(V) == 16 || MODE == PM_DENSITY);
}

/* waves per SIMD the registers are sized for: what the LDS admits, at most
 * four; two for the FP32 density pass that prefetches and three for the
 * FP64 one, whose sums need the registers (in workgroups of at most four
 * waves, which spread evenly over the SIMDs) */
template<int N, int MODE, typename V>
constexpr int plane_min_waves()
{
   constexpr long bytes = ((long)N * (N / 2 + 1) + N) * (long)sizeof(V) + N * 4;
   constexpr int nw = (plane_threads<N, MODE, V>() + 63) / 64;
   constexpr int lw = (int)(160L * 1024 / bytes) * nw / 4;
   constexpr int cap = MODE == PM_DENSITY && sizeof(V) == 8 && plane_prefetch<N, MODE, V>() ? 2
                     : MODE == PM_DENSITY && sizeof(V) == 16 && nw <= 4                    ? 3
                                                                                          : 4;
   return lw < 1 ? 1 : lw < cap ? lw : cap;
}

extern __shared__ __align__(16) unsigned char plane_lds[];

template<int N, int MODE, typename V, bool NYQ>
__global__ void __launch_bounds__((plane_threads<N, MODE, V>()), (plane_min_waves<N, MODE, V>())) k_plane(PlaneArgs a)
{
   using C = GridCfg<N>;
   constexpr int NH = N / 2 + 1, M = N / 2, NT = plane_threads<N, MODE, V>();
   constexpr int Y1 = C::NY1, Y2 = C::NY2, X1 = C::NX1, X2 = C::NX2;
   constexpr int NC = NYQ ? NH : M;                     /* columns that can be nonzero */
   constexpr int IY1 = (NC * Y2 + NT - 1) / NT, IY2 = (NC * Y1 + NT - 1) / NT;
   constexpr int IX1 = (N * x_units<X2>() + NT - 1) / NT, IX2 = (N * X1 + NT - 1) / NT;
   constexpr bool FULL = MODE == PM_C2R_OUT || MODE == PM_R2C_IN;
   constexpr bool PF = plane_prefetch<N, MODE, V>();
   V *sm = reinterpret_cast<V *>(plane_lds);
   V *tws = sm + (size_t)N * NH;
   const int tid0 = threadIdx.x;
   int tid;
   /* the V psi pass runs the orbital groups of one z plane in consecutive
    * workgroups (blockIdx.x the group), which the 8 XCDs take round-robin,
    * so the plane's potential is fetched by few L2s at about the same time;
    * the other modes keep blockIdx.x = z */
   const int z = MODE == PM_VPSI ? blockIdx.y : blockIdx.x, grp = MODE == PM_VPSI ? blockIdx.x : blockIdx.y;
   const int P = a.cols.P;
   for (int m = tid0; m < N; m += NT) tws[m] = cvt<V>(a.tw[m]);
   const int nb = MODE == PM_DENSITY || MODE == PM_VPSI ? a.nb : 1;
   const int b0 = grp * nb, b1 = min(b0 + nb, a.nbatch);
   auto plane_of = [&](int b) { return reinterpret_cast<V *>(a.T) + ((size_t)b * N + z) * P; };

   /* (ky, kx) of T: element n1 of y pass 1's item it, and element k1 of the
    * forward y pass 2's, is ky = Y2 n1 + it / NC, kx = it % NC */
   int *rows = reinterpret_cast<int *>(tws + N);
   if (!FULL) {
      for (int ky = tid0; ky < N; ky += NT) rows[ky] = a.cols.rows[ky];
      __syncthreads();
   }
   auto column = [&](int ky, int kx) {
      if (FULL) return ky * NH + kx;
      const int r = rows[ky];
      return kx < (r >> 16) ? (r & 0xffff) + kx : -1;
   };
   V y[IY1][Y1];
   auto fetch = [&](int b) {
      const V *Tp = plane_of(b);
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < IY1; ++q) {
         const int it = tid + NT * q;
#pragma unroll
         for (int n1 = 0; n1 < Y1; ++n1) {
            const int c = it < NC * Y2 ? column(Y2 * n1 + it / NC, it % NC) : -1;
            y[q][n1] = c >= 0 ? at(Tp, c) : Cx<V>::mk(0, 0);
         }
      }
   };
   /* y passes 1 and 2, the x pre-twiddle and x pass 1; x pass 2 is the caller's */
   auto inverse_to_x2 = [&]() {
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < IY1; ++q) {
         const int it = tid + NT * q, kx = it % NC, n2 = it / NC;
         if (it < NC * Y2) {
            pass_dft_tw<N, Y1, +1>(y[q], n2, tws, 1);
#pragma unroll
            for (int k1 = 0; k1 < Y1; ++k1) sm[(Y2 * k1 + n2) * NH + kx] = y[q][k1];
         }
         item_end();
      }
      __syncthreads();
   };
   auto inverse_rest = [&]() {
      tid = fresh(tid0);
#pragma unroll 1
      for (int q = 0; q < IY2; ++q) {
         const int it = tid + NT * q, kx = it % NC, k1 = it / NC;
         if (it < NC * Y1) {
            V u[Y2];
#pragma unroll
            for (int n2 = 0; n2 < Y2; ++n2) u[n2] = sm[(Y2 * k1 + n2) * NH + kx];
            pass_dft<Y2, +1>(u);
#pragma unroll
            for (int k2 = 0; k2 < Y2; ++k2) sm[(Y2 * k1 + k2) * NH + kx] = u[k2];
         }
      }
      __syncthreads();
      tid = fresh(tid0);
#pragma unroll 1
      for (int q = 0; q < IX1; ++q) {
         const int it = tid + NT * q;
         if (it < N * x_units<X2>()) x_unit<N, NYQ, true>(sm + (it % N) * NH, it / N, tws);
      }
   };
   /* forward x pass 1 of a row's item n1 held in u, back to its slots */
   auto forward_x1 = [&](V (&u)[X2], V *row, int n1) {
      pass_dft_tw<M, X2, -1>(u, n1, tws, 2);
#pragma unroll
      for (int k2 = 0; k2 < X2; ++k2) row[X2 * n1 + k2] = u[k2];
   };
   /* from forward x pass 2 to T */
   auto forward_rest = [&](int b) {
      __syncthreads();
      tid = fresh(tid0);
#pragma unroll 1
      for (int q = 0; q < IX1; ++q) {
         const int it = tid + NT * q;
         if (it < N * x_units<X2>()) x_unit<N, NYQ, false>(sm + (it % N) * NH, it / N, tws);
      }
      __syncthreads();
      tid = fresh(tid0);
#pragma unroll 1
      for (int q = 0; q < IY2; ++q) {
         const int it = tid + NT * q, kx = it % NC, n1 = it / NC;
         if (it < NC * Y1) {
            V u[Y2];
#pragma unroll
            for (int n2 = 0; n2 < Y2; ++n2) u[n2] = sm[(Y2 * n1 + n2) * NH + kx];
            pass_dft_tw<N, Y2, -1>(u, n1, tws, 1);
#pragma unroll
            for (int k2 = 0; k2 < Y2; ++k2) sm[(Y2 * n1 + k2) * NH + kx] = u[k2];
         }
      }
      __syncthreads();
      V *Tp = plane_of(b);
      tid = fresh(tid0);
#pragma unroll 1
      for (int q = 0; q < IY1; ++q) {
         const int it = tid + NT * q, kx = it % NC, k2 = it / NC;
         if (it < NC * Y2) {
            V u[Y1];
#pragma unroll
            for (int n1 = 0; n1 < Y1; ++n1) u[n1] = sm[(Y2 * n1 + k2) * NH + kx];
            pass_dft<Y1, -1>(u);
#pragma unroll
            for (int k1 = 0; k1 < Y1; ++k1) {
               const int c = column(Y2 * k1 + k2, kx);
               if (c >= 0) at(Tp, c) = u[k1];
            }
         }
      }
   };
   /* pair index of (row slot s, k1, k2) in a slot-ordered field */
   auto field = [&](int s, int k1, int k2) { return (unsigned)(((z * X1 + k1) * X2 + k2) * N + s); };

   if constexpr (MODE == PM_DENSITY) {
      double2 acc[IX2][X2];
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < IX2; ++q)
#pragma unroll
         for (int k2 = 0; k2 < X2; ++k2) acc[q][k2] = make_double2(0.0, 0.0);
      if (PF && b0 < b1) fetch(b0);
      for (int b = b0; b < b1; ++b) {
         if (!PF) fetch(b);
         __syncthreads();   /* the previous orbital's sums have read the plane */
         inverse_to_x2();
         if (PF && b + 1 < b1) fetch(b + 1);
         inverse_rest();
         __syncthreads();
         tid = fresh(tid0);
#pragma unroll
         for (int q = 0; q < IX2; ++q) {
            const int it = tid + NT * q;
            if (it < N * X1) {
               const V *row = sm + (it % N) * NH;
               const int k1 = it / N;
               V u[X2];
#pragma unroll
               for (int n2 = 0; n2 < X2; ++n2) u[n2] = row[X2 * k1 + n2];
               pass_dft<X2, +1>(u);
#pragma unroll
               for (int k2 = 0; k2 < X2; ++k2) {
                  const double vx = u[k2].x, vy = u[k2].y;
                  acc[q][k2].x += vx * vx;
                  acc[q][k2].y += vy * vy;
               }
            }
            item_end();
         }
      }
      double2 *dst = reinterpret_cast<double2 *>(a.dnpart + (size_t)grp * N * N * N);
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < IX2; ++q) {
         const int it = tid + NT * q;
         if (it < N * X1) {
#pragma unroll
            for (int k2 = 0; k2 < X2; ++k2) {
               double2 *d = &at(dst, field(it % N, it / N, k2));
               *d = a.accumulate ? make_double2(d->x + acc[q][k2].x, d->y + acc[q][k2].y) : acc[q][k2];
            }
         }
      }
   } else if constexpr (MODE == PM_VPSI) {
      /* orbitals [b0, b1) of plane z; with prefetch the potential stays in
       * registers for all of them */
      V vv[IX2][X2];
      auto load_v = [&]() {
         const double2 *Vz = reinterpret_cast<const double2 *>(a.V);
         tid = fresh(tid0);
#pragma unroll
         for (int q = 0; q < IX2; ++q) {
            const int it = tid + NT * q;
#pragma unroll
            for (int k2 = 0; k2 < X2; ++k2)
               vv[q][k2] = it < N * X1 ? cvt<V>(at(Vz, field(it % N, it / N, k2))) : Cx<V>::mk(0, 0);
         }
      };
      if (PF && b0 < b1) {
         fetch(b0);
         load_v();
      }
      for (int b = b0; b < b1; ++b) {
         if (!PF) fetch(b);
         __syncthreads();   /* twiddles; the previous orbital's write-out has read the plane */
         inverse_to_x2();
         if (PF && b + 1 < b1) fetch(b + 1);
         inverse_rest();
         if (!PF) load_v();
         __syncthreads();
         tid = fresh(tid0);
#pragma unroll
         for (int q = 0; q < IX2; ++q) {
            const int it = tid + NT * q;
            if (it < N * X1) {
               V *row = sm + (it % N) * NH;
               const int k1 = it / N;
               V u[X2];
#pragma unroll
               for (int n2 = 0; n2 < X2; ++n2) u[n2] = row[X2 * k1 + n2];
               pass_dft<X2, +1>(u);
#pragma unroll
               for (int k2 = 0; k2 < X2; ++k2) {
                  u[k2].x *= vv[q][k2].x;
                  u[k2].y *= vv[q][k2].y;
               }
               forward_x1(u, row, k1);
            }
            item_end();
         }
         forward_rest(b);
      }
   } else if constexpr (MODE == PM_VTOT) {
      fetch(b0);
      __syncthreads();
      inverse_to_x2();
      inverse_rest();
      __syncthreads();
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < IX2; ++q) {
         const int it = tid + NT * q;
         if (it < N * X1) {
            const V *row = sm + (it % N) * NH;
            const int k1 = it / N;
            V u[X2];
#pragma unroll
            for (int n2 = 0; n2 < X2; ++n2) u[n2] = row[X2 * k1 + n2];
            pass_dft<X2, +1>(u);
#pragma unroll
            for (int k2 = 0; k2 < X2; ++k2) {
               const unsigned g = field(it % N, k1, k2);
               const double2 xc = at(reinterpret_cast<const double2 *>(a.xcp), g);
               at(reinterpret_cast<double2 *>(a.Vout), g) = make_double2(u[k2].x + xc.x, u[k2].y + xc.y);
            }
         }
      }
   } else if constexpr (MODE == PM_C2R_OUT) {
      fetch(b0);
      __syncthreads();
      inverse_to_x2();
      inverse_rest();
      __syncthreads();
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < IX2; ++q) {
         const int it = tid + NT * q;
         if (it < N * X1) {
            V *row = sm + (it % N) * NH;
            const int k1 = it / N;
            V u[X2];
#pragma unroll
            for (int n2 = 0; n2 < X2; ++n2) u[n2] = row[X2 * k1 + n2];
            pass_dft<X2, +1>(u);
#pragma unroll
            for (int k2 = 0; k2 < X2; ++k2) row[X2 * k1 + k2] = u[k2];
         }
      }
      __syncthreads();
      /* whole rows of the padded output, its two pad reals zero */
      double2 *dst = reinterpret_cast<double2 *>(a.rout + ((size_t)b0 * N + z) * N * (N + 2));
      for (int it = tid0; it < N * NH; it += NT) {
         const int yy = it / NH, j = it % NH;
         dst[it] = j < M ? to_d2(sm[tr_slot<Y1, Y2>(yy) * NH + tr_slot<X1, X2>(j)]) : make_double2(0.0, 0.0);
      }
   } else {  /* PM_R2C_DN, PM_R2C_IN */
      if (MODE == PM_R2C_IN) {
         const double2 *src = reinterpret_cast<const double2 *>(a.rin + ((size_t)b0 * N + z) * N * (N + 2));
         for (int it = tid0; it < N * NH; it += NT) {
            const int yy = it / NH, j = it % NH;
            if (j < M) sm[tr_slot<Y1, Y2>(yy) * NH + tr_slot<X1, X2>(j)] = cvt<V>(src[it]);
         }
      }
      __syncthreads();
      tid = fresh(tid0);
#pragma unroll
      for (int q = 0; q < IX2; ++q) {
         const int it = tid + NT * q;
         if (it < N * X1) {
            V *row = sm + (it % N) * NH;
            const int n1 = it / N;
            V u[X2];
#pragma unroll
            for (int n2 = 0; n2 < X2; ++n2) {
               if (MODE == PM_R2C_DN) {
                  const double2 d = at(reinterpret_cast<const double2 *>(a.dn), field(it % N, n1, n2));
                  u[n2] = cvt<V>(make_double2((d.x + d.x) * a.scal1, (d.y + d.y) * a.scal1));
               } else {
                  u[n2] = row[X2 * n1 + n2];
               }
            }
            forward_x1(u, row, n1);
         }
      }
      forward_rest(b0);
   }
}

/* ------------------------------------------------------------ launchers */

int fft_supported(int n)
{
   switch (n) {
#define CASE(nn) case nn: return 1;
      CPSD_FOR_EACH_GRID(CASE)
#undef CASE
   default: return 0;
   }
}

FftSlots fft_slots(int n)
{
   switch (n) {
#define CASE(nn) case nn: return {nn, GridCfg<nn>::NY1, GridCfg<nn>::NY2, GridCfg<nn>::NX1, GridCfg<nn>::NX2};
      CPSD_FOR_EACH_GRID(CASE)
#undef CASE
   }
   return {0, 1, 1, 1, 1};
}

/* orbitals per workgroup: up to four while the grid still has eight
 * workgroups per CU to spread (they share the index table and prefetch) */
static dim3 zpass_grid(ZArgs &a, int nbatch)
{
   const long ncb = (a.cols.P + ZKB - 1) / ZKB;
   a.nbatch = nbatch;
   a.bper = 1;
   while (a.bper < 4 && ncb * ((nbatch + 2 * a.bper - 1) / (2 * a.bper)) >= 2048) a.bper *= 2;
   const long blocks = ncb * ((nbatch + a.bper - 1) / a.bper);
   return dim3((unsigned)((blocks + 7) / 8 * 8));
}

template<int N>
static int zg2r(const ZArgs &args, int nbatch, hipStream_t s)
{
   ZArgs a = args;
   const dim3 grid = zpass_grid(a, nbatch);
   const bool full = !a.cols.rows;
   if (a.fp32 && full) { cpsd_set_error("zpass g2r: FP32 only for packed orbitals"); return -1; }
   if (a.fp32) hipLaunchKernelGGL((k_zpass_g2r<N, false, float2>), grid, dim3(ZT), 0, s, a);
   else if (full) hipLaunchKernelGGL((k_zpass_g2r<N, true, double2>), grid, dim3(ZT), 0, s, a);
   else hipLaunchKernelGGL((k_zpass_g2r<N, false, double2>), grid, dim3(ZT), 0, s, a);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

template<int N>
static int zr2g(int dst, const ZArgs &args, int nbatch, hipStream_t s)
{
   ZArgs a = args;
   const dim3 grid = zpass_grid(a, nbatch);
   if (a.fp32) {
      if (dst == DST_HPSI) hipLaunchKernelGGL((k_zpass_r2g<N, DST_HPSI, float2>), grid, dim3(ZT), 0, s, a);
      else if (dst == DST_SD) hipLaunchKernelGGL((k_zpass_r2g<N, DST_SD, float2>), grid, dim3(ZT), 0, s, a);
      else {
         cpsd_set_error("zpass r2g: FP32 only for the orbital outputs");
         return -1;
      }
   } else if (dst == DST_HPSI) hipLaunchKernelGGL((k_zpass_r2g<N, DST_HPSI, double2>), grid, dim3(ZT), 0, s, a);
   else if (dst == DST_SD) hipLaunchKernelGGL((k_zpass_r2g<N, DST_SD, double2>), grid, dim3(ZT), 0, s, a);
   else hipLaunchKernelGGL((k_zpass_r2g<N, DST_FULL, double2>), grid, dim3(ZT), 0, s, a);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

template<int N>
static int zfield(const ZArgs &a, hipStream_t s)
{
   hipLaunchKernelGGL((k_zpass_field<N>), dim3((a.cols.P + ZKB - 1) / ZKB), dim3(ZT), 0, s, a);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

template<int N, typename V>
static constexpr size_t plane_lds_bytes()
{
   return ((size_t)N * (N / 2 + 1) + N) * sizeof(V) + N * sizeof(int);   /* plane, twiddles, rows */
}

template<int N, int MODE, typename V, bool NYQ>
static int plane_launch(const PlaneArgs &a, int nblocks, hipStream_t s)
{
   const size_t lds = plane_lds_bytes<N, V>();
   static std::atomic<unsigned long long> attr_set{0};
   if (dyn_lds_once((const void *)k_plane<N, MODE, V, NYQ>, (int)lds, attr_set) != 0) return -1;
   const dim3 grid = MODE == PM_VPSI ? dim3(nblocks, N) : dim3(N, nblocks);
   hipLaunchKernelGGL((k_plane<N, MODE, V, NYQ>), grid, dim3(plane_threads<N, MODE, V>()), lds, s, a);
   CPSD_CHECK(hipGetLastError());
   return 0;
}

template<int N, int MODE, typename V>
static int plane_nyq(const PlaneArgs &a, int nblocks, hipStream_t s)
{
   return a.cols.nyq ? plane_launch<N, MODE, V, true>(a, nblocks, s) : plane_launch<N, MODE, V, false>(a, nblocks, s);
}

template<int N>
static int plane_dispatch(int mode, const PlaneArgs &a, int nblocks, hipStream_t s)
{
   if (a.fp32) {
      switch (mode) {
      case PM_DENSITY: return plane_nyq<N, PM_DENSITY, float2>(a, nblocks, s);
      case PM_VPSI:    return plane_nyq<N, PM_VPSI, float2>(a, nblocks, s);
      }
      cpsd_set_error("plane: mode %d has no FP32 form", mode);
      return -1;
   }
   switch (mode) {
   case PM_DENSITY: return plane_nyq<N, PM_DENSITY, double2>(a, nblocks, s);
   case PM_VTOT:    return plane_nyq<N, PM_VTOT, double2>(a, nblocks, s);
   case PM_VPSI:    return plane_nyq<N, PM_VPSI, double2>(a, nblocks, s);
   case PM_R2C_DN:  return plane_nyq<N, PM_R2C_DN, double2>(a, nblocks, s);
   case PM_C2R_OUT: return plane_launch<N, PM_C2R_OUT, double2, true>(a, nblocks, s);
   case PM_R2C_IN:  return plane_launch<N, PM_R2C_IN, double2, true>(a, nblocks, s);
   }
   cpsd_set_error("plane: bad mode %d", mode);
   return -1;
}

int launch_zpass_g2r(int n, const ZArgs &a, int nbatch, hipStream_t s)
{
   switch (n) {
#define CASE(nn) case nn: return zg2r<nn>(a, nbatch, s);
      CPSD_FOR_EACH_GRID(CASE)
#undef CASE
   }
   cpsd_set_error("FFT grid %d not supported", n);
   return -1;
}

int launch_zpass_r2g(int n, int dst, const ZArgs &a, int nbatch, hipStream_t s)
{
   switch (n) {
#define CASE(nn) case nn: return zr2g<nn>(dst, a, nbatch, s);
      CPSD_FOR_EACH_GRID(CASE)
#undef CASE
   }
   cpsd_set_error("FFT grid %d not supported", n);
   return -1;
}

int launch_zpass_field(int n, const ZArgs &a, hipStream_t s)
{
   switch (n) {
#define CASE(nn) case nn: return zfield<nn>(a, s);
      CPSD_FOR_EACH_GRID(CASE)
#undef CASE
   }
   cpsd_set_error("FFT grid %d not supported", n);
   return -1;
}

/* N = 128 (one or two workgroups per CU): up to 4 while the grid keeps about 4
 * workgroups per CU.  FP32 at 256 orbitals: 1 orbital 1.38 ms, 4 1.26.  Below,
 * one each: at 96^3 and 128 orbitals 1 and 4 measured the same, at 80^3 and
 * 64 one was faster (0.087 and 0.095 ms). */
int plane_orbitals(int n, long planes) { return n < 112 ? 1 : (int)std::max(1L, std::min(4L, planes / 1024)); }

/* The density sum is grouped by how many workgroups of its pass a CU held when
 * the grouping was chosen; it stays so, because the grouping decides the
 * rounding of the density. */
int plane_density_occupancy(int n, int fp32)
{
   switch (n) {
   case 8: case 12: case 16: return 8;
   case 20: case 24: return fp32 ? 8 : 7;
   case 32: return fp32 ? 8 : 5;
   case 40: return fp32 ? 7 : 4;
   case 48: return fp32 ? 6 : 4;
   case 64: return fp32 ? 5 : 3;
   case 80: case 96: return 2;
   }
   return 1;
}

int launch_plane(int n, int mode, const PlaneArgs &a, int nblocks, hipStream_t s)
{
   switch (n) {
#define CASE(nn) case nn: return plane_dispatch<nn>(mode, a, nblocks, s);
      CPSD_FOR_EACH_GRID(CASE)
#undef CASE
   }
   cpsd_set_error("FFT grid %d not supported", n);
   return -1;
}

int launch_fft3d(int dir, int n, int nbatch, double2 *A, double2 *T, const double2 *tw, hipStream_t s)
{
   const size_t per = (size_t)n * n * (n / 2 + 1);
   ColTable cols;
   cols.rows = cols.gmap = nullptr; cols.P = n * (n / 2 + 1); cols.nyq = 1;
   ZArgs z;
   memset(&z, 0, sizeof z);
   z.cols = cols; z.tw = tw; z.T = T;
   z.src = A; z.sstride = per; z.out = A; z.ostride = per;
   PlaneArgs pa;
   memset(&pa, 0, sizeof pa);
   pa.cols = cols; pa.T = T; pa.tw = tw; pa.nbatch = nbatch;
   pa.rout = reinterpret_cast<double *>(A); pa.rin = reinterpret_cast<const double *>(A);
   if (dir > 0) {
      if (launch_zpass_g2r(n, z, nbatch, s) != 0) return -1;
      return launch_plane(n, PM_C2R_OUT, pa, nbatch, s);
   }
   if (launch_plane(n, PM_R2C_IN, pa, nbatch, s) != 0) return -1;
   return launch_zpass_r2g(n, DST_FULL, z, nbatch, s);
}
