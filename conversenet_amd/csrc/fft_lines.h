// In-place prime-factor FFTs of any length up to 1024 on a batch of lines held in LDS, for gfx950.
//
// Layout: element n of line b sits at buf[n kLineLd + b], b < kLines = 16: the lines run along the
// lanes, so a butterfly's LDS accesses are 16 consecutive float2 and need no transposition between
// passes, and the odd kLineLd spreads accesses that run along n (global loads and stores) over all banks.
// (32 lines per block measured the same to 15 % slower at most lengths: fewer blocks per CU.)
//
// A length is split into pairwise coprime parts Q (Good-Thomas: I. J. Good, J. Roy. Statist. Soc. B 20,
// 1958; L. H. Thomas, 1963).  With M = L / Q and the index map n = sum_Q M a_Q mod L, position n holds
// the coordinates a_Q and the transform is a Q-point DFT along each coordinate, in place and without
// twiddles; afterwards the position with coordinates b_Q holds the bin k = b_Q mod Q of every part.  A
// part is
//   * one register butterfly of radix 2 .. 32, where prime powers of different primes may share one
//     (a radix of 24 = 8 x 3 inside the registers saves a pass over LDS);
//   * a prime power above 32: Cooley-Tukey stages inside the part, the twiddles W_Q on the outputs of a
//     stage (digit-reversed result; the inverse runs the stages backwards, twiddles on the inputs);
//   * a prime above 31: a dense DFT on the fp32 matrix cores (dense_pass).
// Two passes serve most lengths; every length up to 1024 has a plan.  Twiddle-free passes of large radix
// keep both the number of LDS round trips and the rounding errors low.
//
// All transforms run forward; an inverse transform is the forward one with real and imaginary parts
// exchanged before and after, which the callers fold into their stores and loads.
#pragma once
#include <atomic>
#include <new>

#include "fft_device.h"

namespace cvn {

// Kernel arguments are read in place, in the constant address space: a plan indexed by a loop variable
// stays scalar loads (as an ordinary reference the whole argument struct was copied to scratch).
#define CVN_KARG __attribute__((address_space(4)))

// ------------------------------------------------------------------------------------------------
// Register DFTs of the composite radices: coprime factors (Good-Thomas) and prime powers (Cooley-Tukey).
// ------------------------------------------------------------------------------------------------
// out[map(k1, k2)] = DFT_{A B}: n = (B n1 + A n2) mod N, k = k1 mod A and k = k2 mod B.
template <int A, int B> struct DftCoprime {
  static constexpr int N = A * B;
  static constexpr int bin(int k1, int k2) {
    for (int k = 0; k < N; ++k)
      if (k % A == k1 && k % B == k2) return k;
    return 0;
  }
  template <int K1, int K2>
  static __device__ __forceinline__ void put(float2* u, const float2* v) {
    u[bin(K1, K2)] = v[K2];
    if constexpr (K2 + 1 < B) put<K1, K2 + 1>(u, v);
  }
  template <int K1>
  static __device__ __forceinline__ void second(float2* u, const float2 (&t)[B][A]) {
    float2 v[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) v[n2] = t[n2][K1];
    Dft<B, false>::run(v);
    put<K1, 0>(u, v);
    if constexpr (K1 + 1 < A) second<K1 + 1>(u, t);
  }
  static __device__ __forceinline__ void run(float2* u) {
    float2 t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = u[(B * n1 + A * n2) % N];
      Dft<A, false>::run(t[n2]);
    }
    second<0>(u, t);
  }
};
// n = B n1 + n2, k = k1 + A k2, twiddles W_{A B}^(n2 k1) as literals.
template <int A, int B> struct DftPower {
  static constexpr int N = A * B;
  template <int N2, int K1>
  static __device__ __forceinline__ void twiddle(float2* t) {
    if constexpr (N2 * K1 != 0) {
      constexpr CosSin w = cos_sin_turn(N2 * K1, N);
      t[K1] = cmul(t[K1], make_float2((float)w.c, (float)-w.s));
    }
    if constexpr (K1 + 1 < A) twiddle<N2, K1 + 1>(t);
  }
  template <int N2>
  static __device__ __forceinline__ void first(const float2* u, float2 (&t)[B][A]) {
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) t[N2][n1] = u[B * n1 + N2];
    Dft<A, false>::run(t[N2]);
    twiddle<N2, 0>(t[N2]);
    if constexpr (N2 + 1 < B) first<N2 + 1>(u, t);
  }
  static __device__ __forceinline__ void run(float2* u) {
    float2 t[B][A];
    first<0>(u, t);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      float2 v[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) v[n2] = t[n2][k1];
      Dft<B, false>::run(v);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) u[k1 + A * k2] = v[k2];
    }
  }
};
template <> struct Dft<6, false> : DftCoprime<3, 2> {};
template <> struct Dft<9, false> : DftPower<3, 3> {};
template <> struct Dft<10, false> : DftCoprime<5, 2> {};
template <> struct Dft<12, false> : DftCoprime<4, 3> {};
template <> struct Dft<14, false> : DftCoprime<7, 2> {};
template <> struct Dft<15, false> : DftCoprime<5, 3> {};
template <> struct Dft<18, false> : DftCoprime<9, 2> {};
template <> struct Dft<20, false> : DftCoprime<5, 4> {};
template <> struct Dft<21, false> : DftCoprime<7, 3> {};
template <> struct Dft<22, false> : DftCoprime<11, 2> {};
template <> struct Dft<24, false> : DftCoprime<8, 3> {};
template <> struct Dft<25, false> : DftPower<5, 5> {};
template <> struct Dft<26, false> : DftCoprime<13, 2> {};
template <> struct Dft<27, false> : DftPower<9, 3> {};
template <> struct Dft<28, false> : DftCoprime<7, 4> {};
template <> struct Dft<30, false> : DftCoprime<15, 2> {};
template <> struct Dft<32, false> : DftPower<8, 4> {};

// ------------------------------------------------------------------------------------------------
// Plans
// ------------------------------------------------------------------------------------------------
constexpr int kLineMax = 1024;     // longest length
constexpr int kLines = 16;         // lines per block
constexpr int kLineLd = kLines + 1;
constexpr int kLinePasses = 6;
constexpr int kLineRadix = 32;     // largest register butterfly
// One pass: nl = L / R butterflies.  Butterfly l = (i bt + beta) mt + e has its legs at
// (base + j d) mod L, base = (Q i + M (beta nt + e)) mod L; single-stage parts have bt = mt = 1.
struct LinePass {
  int R;                 // radix; dense: the prime
  int dense;
  int nl, d, Q;
  int mt, bt, eM, bM;    // e step M, beta step M nt
  uint32_t mg_m, mg_b;   // ceil(2^32 / mt), ceil(2^32 / bt)
  int tw;                // twiddle step: output leg j times W_T^(e j tw); 0: none
};
struct LineStages {      // the part that runs in several stages, if any: digit reversal of its coordinate
  int Q, M, nst;
  uint32_t mgQ;
  int R[3], m[3];        // radices and their slot strides
  uint32_t mgR[3];
};
struct LinePlan {
  int L, np;
  int T, tws;            // LDS table of W_T^m, m < T (T = 1: none), read from W_L^(m tws)
  int kappa;             // position of bin k: (kappa k + M reversed(k mod Q)) mod L
  uint32_t mgL;
  LineStages ms;         // nst = 0: none
  LinePass ps[kLinePasses];
};

__device__ __forceinline__ int mg_div(int a, uint32_t mg, int d) { return d > 1 ? (int)__umulhi((uint32_t)a, mg) : a; }

// Position of bin k.  A single-stage part puts M (k mod Q) there, which is M k mod L, so those parts
// together are one multiplication; at most one part of a length up to 1024 has several stages.
__device__ __forceinline__ int line_pos(const CVN_KARG LinePlan& p, int k) {
  int a = p.kappa * k;  // < 2^20
  if (p.ms.nst) {
    int b = k - mg_div(k, p.ms.mgQ, p.ms.Q) * p.ms.Q, slot = 0;
#pragma unroll
    for (int s = 0; s < 3; ++s)
      if (s < p.ms.nst) {
        const int hi = mg_div(b, p.ms.mgR[s], p.ms.R[s]);
        slot += (b - hi * p.ms.R[s]) * p.ms.m[s];
        b = hi;
      }
    a += slot * p.ms.M;  // < L
  }
  return a - mg_div(a, p.mgL, p.L) * p.L;
}

// Fills the block's LDS tables: ipos[k] (position of bin k) and tw[m] = W_T^m.  The caller synchronises.
__device__ __forceinline__ void line_tables(const CVN_KARG LinePlan& p, const float2* __restrict__ gtw, unsigned short* ipos,
                                            float2* tw, int tid, int nth) {
  if (p.T > 1)
    for (int m = tid; m < p.T; m += nth) tw[m] = gtw[m * p.tws];
  for (int k = tid; k < p.L; k += nth) ipos[k] = (unsigned short)line_pos(p, k);
}

// Butterfly l of a pass: its first position (before the legs' steps) and its twiddle row e.
__device__ __forceinline__ uint32_t line_base(const CVN_KARG LinePass& ps, int L, int l, int* e) {
  *e = 0;
  if (ps.mt == 1 && ps.bt == 1) return ps.Q * l;
  const int r = mg_div(l, ps.mg_m, ps.mt);
  *e = l - r * ps.mt;
  const int i = mg_div(r, ps.mg_b, ps.bt);
  const uint32_t base = ps.Q * i + ps.bM * (r - i * ps.bt) + ps.eM * *e;
  return min(base, base - (uint32_t)L);
}

// Odd prime radix R > 13 by conjugate pairs (DftOdd): each pair of outputs is stored as it is formed,
// so the registers hold the (R - 1) / 2 sums and differences only.  Every index is a template argument:
// nested loops of this size stop being unrolled, and the arrays would live in scratch.
template <int R> struct PrimePass {
  static constexpr int H = (R - 1) / 2;
  template <int Q, int J>
  static __device__ __forceinline__ void terms(const float2* a, const float2* b, float2& A, float2& Bv) {
    constexpr CosSin w = cos_sin_turn(J * Q % R, R);
    A.x = fmaf((float)w.c, a[J - 1].x, A.x);
    A.y = fmaf((float)w.c, a[J - 1].y, A.y);
    Bv.x = fmaf((float)w.s, b[J - 1].x, Bv.x);
    Bv.y = fmaf((float)w.s, b[J - 1].y, Bv.y);
    if constexpr (J < H) terms<Q, J + 1>(a, b, A, Bv);
  }
  template <int Q>
  static __device__ __forceinline__ void bins(char* buf, uint32_t lo, uint32_t hi, uint32_t dS, uint32_t LS, float2 x0,
                                              const float2* a, const float2* b, const float2* tw, int st) {
    float2 A = x0, Bv = make_float2(0.f, 0.f);
    terms<Q, 1>(a, b, A, Bv);
    float2 xl = make_float2(A.x + Bv.y, A.y - Bv.x), xh = make_float2(A.x - Bv.y, A.y + Bv.x);
    if (st >= 0) {
      xl = cmul(xl, tw[Q * st]);
      xh = cmul(xh, tw[(R - Q) * st]);
    }
    *(float2*)(buf + lo) = xl;
    *(float2*)(buf + hi) = xh;
    lo += dS;
    lo = min(lo, lo - LS);
    hi -= dS;
    hi = min(hi, hi + LS);
    if constexpr (Q < H) bins<Q + 1>(buf, lo, hi, dS, LS, x0, a, b, tw, st);
  }
};
template <int R>
__device__ __forceinline__ void prime_pass(char* buf, const CVN_KARG LinePass& ps, int L, int b, int grp, int ngrp,
                                           const float2* tw, bool dit) {
  constexpr uint32_t S = kLineLd * sizeof(float2);
  constexpr int H = (R - 1) / 2;
  const uint32_t dS = ps.d * S, LS = L * S;
  const int twm = ps.tw, nl = ps.nl;
  for (int l = grp; l < nl; l += ngrp) {
    int e;
    const uint32_t a0 = line_base(ps, L, l, &e) * S + b * (uint32_t)sizeof(float2);
    const int st = e * twm;
    float2 p[H], m[H];
    const float2 x0 = *(const float2*)(buf + a0);
    float2 sum = x0;
    uint32_t lo0 = a0 + dS;
    lo0 = min(lo0, lo0 - LS);
    uint32_t hi0 = a0 + (R - 1) * dS;  // (R d = L only where the part has one stage)
    hi0 = min(hi0, hi0 - LS);
    uint32_t lo = lo0, hi = hi0;
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      float2 ul = *(const float2*)(buf + lo), uh = *(const float2*)(buf + hi);
      if (twm && dit) {
        ul = cmul(ul, tw[j * st]);
        uh = cmul(uh, tw[(R - j) * st]);
      }
      p[j - 1] = cadd(ul, uh);
      m[j - 1] = csub(ul, uh);
      sum = cadd(sum, p[j - 1]);
      lo += dS;
      lo = min(lo, lo - LS);
      hi -= dS;
      hi = min(hi, hi + LS);
    }
    *(float2*)(buf + a0) = sum;
    PrimePass<R>::template bins<1>(buf, lo0, hi0, dS, LS, x0, p, m, tw, twm && !dit ? st : -1);
  }
}

// One radix-R pass.  grp / ngrp: this thread's butterfly index and the number of butterflies in flight.
// dit: the twiddles multiply the inputs (inverse order) instead of the outputs.
template <int R>
__device__ __forceinline__ void line_pass(char* buf, const CVN_KARG LinePass& ps, int L, int b, int grp, int ngrp,
                                          const float2* tw, bool dit) {
  constexpr uint32_t S = kLineLd * sizeof(float2);
  const uint32_t dS = ps.d * S, LS = L * S;
  const int twm = ps.tw, nl = ps.nl;
  for (int l = grp; l < nl; l += ngrp) {
    int e;
    const uint32_t a0 = line_base(ps, L, l, &e) * S + b * (uint32_t)sizeof(float2);
    float2 u[R];
    uint32_t ad = a0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      u[j] = *(const float2*)(buf + ad);
      ad += dS;
      ad = min(ad, ad - LS);
    }
    if (twm && dit) {
      const int st = e * twm;
#pragma unroll
      for (int j = 1; j < R; ++j) u[j] = cmul(u[j], tw[j * st]);
    }
    Dft<R, false>::run(u);
    if (twm && !dit) {
      const int st = e * twm;
#pragma unroll
      for (int j = 1; j < R; ++j) u[j] = cmul(u[j], tw[j * st]);
    }
    uint32_t aw = a0;
    asm volatile("" : "+v"(aw));  // the store addresses are formed again instead of held in R registers
#pragma unroll
    for (int j = 0; j < R; ++j) {
      *(float2*)(buf + aw) = u[j];
      aw += dS;
      aw = min(aw, aw - LS);
    }
  }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Dense DFT of prime length p = ps.R on the fp32 matrix cores, in place on ps.nl lines.  With
// a_j = u_j + u_{p-j}, b_j = u_j - u_{p-j}, j = 1 .. h = (p - 1) / 2:
//   A_q = u_0 + sum_j cos(2 pi j q / p) a_j,  B_q = sum_j sin(2 pi j q / p) b_j,  q = 0 .. h,
//   X_q = A_q - i B_q,  X_{p-q} = A_q + i B_q,
// four real products of an (h + 1) x h coefficient matrix (entries read from the p-entry table) with
// the real and imaginary parts of a and b: a quarter of the multiplications of the plain complex form.
// A unit is one line's 16 bins q for all 16 batch lanes: v_mfma_f32_16x16x4f32 with lane 16 g + c
// holding coefficient (q = 16 tile + c, j = 4 step + g + 1) and sample j of batch lane c.  The block
// takes as many whole lines per round as its waves hold units (kDenseUnits), synchronises when
// every unit of the round has read its line, and writes in place.  ceil((h + 1) / 16) must not
// exceed kDenseUnits nwaves (line_min_threads).
// Sums run in chunks of kDenseChunk steps (32 samples), added up afterwards: the rounding error of a
// 257-point transform is half of one running sum's.
constexpr int kDenseChunk = 8;
constexpr int kDenseUnits = 2;
__device__ __forceinline__ void dense_pass(char* buf, const CVN_KARG LinePass& ps, int L, const float2* tw, int tid, int nth) {
  constexpr uint32_t S = kLineLd * sizeof(float2);
  const int p = ps.R, h = (p - 1) / 2, M = ps.d;
  const int per = (h + 16) / 16;  // tiles of 16 bins
  const int lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nth >> 6;
  const int lines = min(ps.nl, nw * kDenseUnits / per);  // whole lines per round (at least 1)
  const int steps = (h + 3) / 4;
  for (int l0 = 0; l0 < ps.nl; l0 += lines) {
    const int units = min(lines, ps.nl - l0) * per;
    f32x4 are[kDenseUnits], aim[kDenseUnits], bre[kDenseUnits], bim[kDenseUnits];
#pragma unroll
    for (int k = 0; k < kDenseUnits; ++k) {
      const int un = wave + k * nw;
      if (un < units) {
        const int line = un / per, tile = un - line * per;
        const int base = ps.Q * (l0 + line);
        const uint32_t col = c * sizeof(float2);
        const int q = tile * 16 + c;
        int ci = (int)(((unsigned)q * (unsigned)(g + 1)) % (unsigned)p);
        const int cs = (int)((4u * (unsigned)q) % (unsigned)p);
        // positions of samples j and p - j: base + j M and base + (p - j) M, mod L
        uint32_t lo = base + (g + 1) * M, hi = base + (p - 1 - g) * M;
        lo = min(lo, lo - (uint32_t)L);
        hi = min(hi, hi - (uint32_t)L);
        const uint32_t MS = (4 * M) * S, LS = L * S;  // 4 M < L: p > 31
        lo = lo * S + col;
        hi = hi * S + col;
        const float2 u0 = *(const float2*)(buf + base * S + col);
        f32x4 xr = {u0.x, u0.x, u0.x, u0.x}, xi = {u0.y, u0.y, u0.y, u0.y};
        f32x4 yr = {0.f, 0.f, 0.f, 0.f}, yi = {0.f, 0.f, 0.f, 0.f};
        f32x4 txr = yr, txi = yr, tyr = yr, tyi = yr;
        for (int t = 0; t < steps; ++t) {
          if (t > 0 && t % kDenseChunk == 0) {
            txr += xr;
            txi += xi;
            tyr += yr;
            tyi += yi;
            xr = xi = yr = yi = f32x4{0.f, 0.f, 0.f, 0.f};
          }
          const float2 w = tw[ci];
          float2 ul = *(const float2*)(buf + lo), uh = *(const float2*)(buf + hi);
          if (4 * t + g >= h) ul = uh = make_float2(0.f, 0.f);
          xr = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, ul.x + uh.x, xr, 0, 0, 0);
          xi = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, ul.y + uh.y, xi, 0, 0, 0);
          yr = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, ul.x - uh.x, yr, 0, 0, 0);
          yi = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, ul.y - uh.y, yi, 0, 0, 0);
          ci += cs;
          ci = ci >= p ? ci - p : ci;
          lo += MS;
          lo = min(lo, lo - LS);
          hi -= MS;                 // below zero: wraps past hi + LS, which min picks
          hi = min(hi, hi + LS);
        }
        are[k] = xr + txr;
        aim[k] = xi + txi;
        bre[k] = yr + tyr;
        bim[k] = yi + tyi;
      }
    }
    __syncthreads();  // every unit of these lines has read its samples
#pragma unroll
    for (int k = 0; k < kDenseUnits; ++k) {
      const int un = wave + k * nw;
      if (un < units) {
        const int line = un / per, tile = un - line * per;
        const int base = ps.Q * (l0 + line);
        const uint32_t col = c * sizeof(float2);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int q = tile * 16 + 4 * g + e;
          if (q <= h) {
            // the table holds -sin: y = -B
            uint32_t lo = base + q * M, hi = base + (p - q) * M;
            lo = min(lo, lo - (uint32_t)L);
            hi = min(hi, hi - (uint32_t)L);
            *(float2*)(buf + lo * S + col) = make_float2(are[k][e] - bim[k][e], aim[k][e] + bre[k][e]);
            if (q > 0)
              *(float2*)(buf + hi * S + col) = make_float2(are[k][e] + bim[k][e], aim[k][e] - bre[k][e]);
          }
        }
      }
    }
  }
}

// The whole transform of the block's lines; synchronises after every pass.  FWD: natural order to positions
// (line_pos); otherwise positions to natural order (passes backwards).  Every thread of the block calls.
template <bool FWD>
__device__ __forceinline__ void line_fft(const CVN_KARG LinePlan& p, char* buf, const float2* tw, int tid, int nth) {
  const int b = tid % kLines, grp = tid / kLines, ngrp = nth / kLines;
  for (int t = 0; t < p.np; ++t) {
    const CVN_KARG LinePass& ps = p.ps[FWD ? t : p.np - 1 - t];
    if (ps.dense) {
      dense_pass(buf, ps, p.L, tw, tid, nth);
    } else {
      switch (ps.R) {
#define CVN_LINE_PRIME(r) \
  case r: prime_pass<r>(buf, ps, p.L, b, grp, ngrp, tw, !FWD); break;
#define CVN_LINE_RADIX(r) \
  case r: line_pass<r>(buf, ps, p.L, b, grp, ngrp, tw, !FWD); break;
        CVN_LINE_RADIX(2) CVN_LINE_RADIX(3) CVN_LINE_RADIX(4) CVN_LINE_RADIX(5) CVN_LINE_RADIX(6)
        CVN_LINE_RADIX(7) CVN_LINE_RADIX(8) CVN_LINE_RADIX(9) CVN_LINE_RADIX(10) CVN_LINE_RADIX(11)
        CVN_LINE_RADIX(12) CVN_LINE_RADIX(13) CVN_LINE_RADIX(14) CVN_LINE_RADIX(15) CVN_LINE_RADIX(16)
        CVN_LINE_PRIME(17) CVN_LINE_RADIX(18) CVN_LINE_PRIME(19) CVN_LINE_RADIX(20) CVN_LINE_RADIX(21)
        CVN_LINE_RADIX(22) CVN_LINE_PRIME(23) CVN_LINE_RADIX(24) CVN_LINE_RADIX(25) CVN_LINE_RADIX(26)
        CVN_LINE_RADIX(27) CVN_LINE_RADIX(28) CVN_LINE_PRIME(29) CVN_LINE_RADIX(30) CVN_LINE_PRIME(31)
        default: line_pass<32>(buf, ps, p.L, b, grp, ngrp, tw, !FWD); break;
#undef CVN_LINE_RADIX
#undef CVN_LINE_PRIME
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------------------
// Planner (host)
// ------------------------------------------------------------------------------------------------
inline uint32_t line_magic(int d) { return d > 1 ? 0xFFFFFFFFu / (uint32_t)d + 1u : 0u; }

// Plan of length L (1 .. kLineMax), false outside.
inline bool make_line_plan(int L, LinePlan* p) {
  if (L < 1 || L > kLineMax) return false;
  *p = LinePlan{};
  p->L = L;
  p->T = 1;
  int q[8], pr[8], nq = 0;  // prime powers and their primes
  for (int n = L, f = 2; n > 1; ++f)
    if (n % f == 0) {
      pr[nq] = f;
      q[nq] = 1;
      while (n % f == 0) { q[nq] *= f; n /= f; }
      ++nq;
    }
  // parts that fit a register butterfly share one where the product does too: the grouping with the
  // fewest groups, then the smallest sum of radices (the register butterflies' work per sample)
  int small[8], ns = 0;
  for (int t = 0; t < nq; ++t)
    if (q[t] <= kLineRadix && (pr[t] <= 31)) small[ns++] = q[t];
  int best[8], bestn = 99, bestsum = 1 << 20;
  int grp[8] = {0};
  // all assignments of the (at most 4) small parts to groups
  int total = 1;
  for (int t = 0; t < ns; ++t) total *= ns;
  for (int code = 0; code < (ns ? total : 0); ++code) {
    int prod[8];
    for (int t = 0; t < ns; ++t) prod[t] = 1;
    for (int t = 0, c = code; t < ns; ++t, c /= ns) {
      grp[t] = c % ns;
      prod[grp[t]] *= small[t];
    }
    int n = 0, sum = 0;
    bool ok = true;
    for (int t = 0; t < ns; ++t)
      if (prod[t] > 1) {
        ++n;
        sum += prod[t];
        ok = ok && prod[t] <= kLineRadix;
      }
    if (ok && (n < bestn || (n == bestn && sum < bestsum))) {
      bestn = n;
      bestsum = sum;
      int k = 0;
      for (int t = 0; t < ns; ++t)
        if (prod[t] > 1) best[k++] = prod[t];
    }
  }
  p->mgL = line_magic(L);
  auto part = [&](int Q, int nst, const int* R, bool dense) {
    const int M = L / Q;
    if (nst == 1) p->kappa = (p->kappa + M) % L;
    else p->ms = LineStages{Q, M, nst, line_magic(Q), {}, {}, {}};
    int bt = 1, nt = Q;
    for (int s = 0; s < nst; ++s) {
      const int m = nt / R[s];
      if (nst > 1) {
        p->ms.R[s] = R[s];
        p->ms.m[s] = m;
        p->ms.mgR[s] = line_magic(R[s]);
      }
      LinePass& ps = p->ps[p->np++];
      ps.R = R[s];
      ps.dense = dense ? 1 : 0;
      ps.nl = L / R[s];
      ps.Q = Q;
      ps.mt = m;
      ps.bt = bt;
      ps.mg_m = line_magic(m);
      ps.mg_b = line_magic(bt);
      ps.eM = M;
      ps.bM = M * nt;
      ps.d = M * m;
      ps.tw = m > 1 ? Q / nt : 0;
      if (m > 1 || dense) {
        p->T = Q;
        p->tws = L / Q;
      }
      bt *= R[s];
      nt = m;
    }
  };
  for (int t = 0; t < nq; ++t) {
    if (pr[t] > 31) {
      part(q[t], 1, &q[t], true);  // a prime above 31 divides a length up to 1024 once
    } else if (q[t] > kLineRadix) {  // Cooley-Tukey inside the part: balanced stages
      int R[3] = {1, 1, 1}, n = 0;
      for (int rest = q[t]; rest > 1; ++n) {
        // fewest stages, then nearly equal: the smallest power r of the prime with r^k >= rest
        int k = 1;
        auto fits = [&](int stages) {
          int r = pr[t];
          while (r * pr[t] <= kLineRadix) r *= pr[t];
          long long v = 1;
          for (int i = 0; i < stages; ++i) v *= r;
          return v >= rest;
        };
        while (!fits(k)) ++k;
        int r = pr[t];
        auto powk = [&](int b) { long long v = 1; for (int i = 0; i < k; ++i) v *= b; return v; };
        while (powk(r) < rest) r *= pr[t];
        if (r > rest) r = rest;
        R[n] = r;
        rest /= r;
      }
      part(q[t], n, R, false);
    }
  }
  for (int k = 0; k < (ns ? bestn : 0); ++k) part(best[k], 1, &best[k], false);
  return true;
}

// The plan of length L, made once per process (at most kLineMax of them; the planner takes microseconds,
// as much as a small launch); null outside 1 .. kLineMax (and without memory).
inline const LinePlan* line_plan(int L) {
  static std::atomic<const LinePlan*> memo[kLineMax + 1] = {};
  if (L < 1 || L > kLineMax) return nullptr;
  const LinePlan* p = memo[L].load(std::memory_order_acquire);
  if (p) return p;
  LinePlan* made = new (std::nothrow) LinePlan;
  if (!made) return nullptr;
  make_line_plan(L, made);
  if (memo[L].compare_exchange_strong(p, made, std::memory_order_acq_rel)) return made;
  delete made;  // another thread was first
  return p;
}

// LDS of a block's lines of length L, and of their tables (twiddles, positions); 16-byte multiples.
inline size_t line_buf_bytes(int L) { return ((size_t)L * kLineLd * sizeof(float2) + 15) / 16 * 16; }
inline size_t line_tab_bytes(const LinePlan& p) {
  return ((size_t)p.T * sizeof(float2) + (size_t)p.L * sizeof(unsigned short) + 15) / 16 * 16;
}
// Threads per block that the dense pass needs at least (the units of one line).
inline int line_min_threads(const LinePlan& p) {
  int n = 64;
  for (int t = 0; t < p.np; ++t)
    if (p.ps[t].dense) n = 64 * ((((p.ps[t].R - 1) / 2 + 16) / 16 + kDenseUnits - 1) / kDenseUnits);
  return n;
}

}  // namespace cvn
