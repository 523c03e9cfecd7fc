// Row and column passes of the multi-pass routes for any transform length up to 1024, on the in-place
// prime-factor engine of fft_lines.h.  Same spectra scratch and transfer table as the runtime-plan passes
// of converse2d_generic.hip (half spectra S[plane][col][row], tables (psf plane, col, row), twiddles
// exp(-2 pi i m / L)), which keep the longer lengths.
//
// Every block transforms 16 lines (row pairs or columns) of any planes: lines are numbered through all
// planes, so small planes fill their blocks.
//
// What bounds them: each pass is one trip of the plane through HBM or the MALL (4.6 to 6 bytes moved per
// byte of plane and pass), overlapped by the 2 to 16 blocks of a CU with two or three LDS passes.  Measured
// (one layer, us, runtime-plan passes -> these): 128 planes 333 x 493: 679 -> 210 (rows 214 -> 58, columns
// 282 -> 90, inverse rows 214 -> 58); 512 planes 136 x 136: 282 -> 90; 256 planes 499 x 509 (primes):
// 1283 ms -> 1.7 ms; the backward's 1024 x 260 rows of 260, compile-time plan before: 172 -> 127; the
// backward's column pass at 1024 planes 108 x 108: 240 -> 127; the operator's 192 planes 63 x 88 at scale 3:
// 336 -> 176 (whole call).
#include <algorithm>

#include "cvn_common.h"
#include "fft_lines.h"

namespace cvn {
namespace {

constexpr int kLineThreads = 1024;
constexpr size_t kLineLds = 160 * 1024;

__device__ __forceinline__ int line_pad_src(int i, int n, int p, int mode) {
  int j = i - p;
  if (j >= 0 && j < n) return j;
  switch (mode) {
    case CVN_PAD_CIRCULAR: j %= n; return j < 0 ? j + n : j;
    case CVN_PAD_REPLICATE: return j < 0 ? 0 : n - 1;
    case CVN_PAD_REFLECT: return j < 0 ? -j : 2 * (n - 1) - j;
    default: return -1;
  }
}

// The dispatcher places block i on XCD i mod 8; items run contiguously per XCD, so that neighbouring
// batches (which share 128-byte lines of the spectra) and the planes of one psf meet in one L2.
__device__ __forceinline__ int line_item(int blk, int nblk) {
  const int x = blk & 7, k = blk >> 3, per = nblk >> 3, rem = nblk & 7;
  return x * per + min(x, rem) + k;
}

// ------------------------------------------------------------------------------------------------
// Forward row pass: real row pairs (2 t, 2 t + 1) as one complex line, half spectra to S[plane][v][row].
// ------------------------------------------------------------------------------------------------
struct RowsFwdArgs {
  const float* x;   // (P, Hin, Win)
  float2* S;        // (P, NC, h)
  const float2* tw;
  int Hin, Win, h, pad, mode, NC, npair, total, nblk;  // total = P npair lines
  int vec;          // S allows 16-byte stores of a row pair (h even, S 16-byte aligned)
  LinePlan plan;
};

__global__ void __launch_bounds__(kLineThreads) k_lines_rows_fwd(RowsFwdArgs) {
  const CVN_KARG RowsFwdArgs& a = *(const CVN_KARG RowsFwdArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NB = kLines, LD = kLineLd;
  const int tid = threadIdx.x, nth = blockDim.x, L = a.plan.L;
  float2* buf = (float2*)smem;
  char* tab = smem + ((size_t)L * LD * sizeof(float2) + 15) / 16 * 16;
  int64_t* src = (int64_t*)tab;  // 2 NB: element offset of each line's source rows, -1: zeros
  float2* tw = (float2*)(src + 2 * NB);
  unsigned short* ipos = (unsigned short*)(tw + a.plan.T);
  const int g0 = line_item(blockIdx.x, a.nblk) * NB;
  if (tid < 2 * NB) {
    const int gp = g0 + (tid >> 1);
    const int plane = gp / a.npair, r = 2 * (gp - plane * a.npair) + (tid & 1);
    const int sr = (gp < a.total && r < a.h) ? line_pad_src(r, a.Hin, a.pad, a.mode) : -1;
    src[tid] = sr >= 0 ? ((int64_t)plane * a.Hin + sr) * a.Win : -1;
  }
  __syncthreads();
  // items (8 lines, sample n), n fastest; the tables are filled while the first loads are on their way
  const int nitem = L * (NB / 8);
  for (int i0 = tid; i0 < nitem || i0 == tid; i0 += nth) {
    const int idx = min(i0, nitem - 1);
    const int q = mg_div(idx, a.plan.mgL, L), n = idx - q * L, b0 = 8 * q;
    const int sc = line_pad_src(n, a.Win, a.pad, a.mode);
    const float* xc = a.x + max(sc, 0);
    float va[8], vb[8];
    int64_t oa[8], ob[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      oa[k] = src[2 * (b0 + k)];
      ob[k] = src[2 * (b0 + k) + 1];
      va[k] = xc[oa[k] < 0 ? 0 : oa[k]];
      vb[k] = xc[ob[k] < 0 ? 0 : ob[k]];
    }
    if (i0 == tid) line_tables(a.plan, a.tw, ipos, tw, tid, nth);
    if (i0 < nitem) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        buf[n * LD + b0 + k] =
            make_float2(sc < 0 || src[2 * (b0 + k)] < 0 ? 0.f : va[k], sc < 0 || src[2 * (b0 + k) + 1] < 0 ? 0.f : vb[k]);
    }
  }
  __syncthreads();
  line_fft<true>(a.plan, smem, tw, tid, nth);
  // Ya = (Z[v] + conj Z[-v]) / 2, Yb = (Z[v] - conj Z[-v]) / (2 i)
  const int b = tid % NB, gp = g0 + b;
  if (gp >= a.total) return;
  const int plane = gp / a.npair, r = 2 * (gp - plane * a.npair);
  float2* out = a.S + (int64_t)plane * a.NC * a.h + r;
  const bool two = r + 1 < a.h;
  const int step = nth / NB;
  for (int v0 = tid / NB; v0 < a.NC; v0 += 4 * step) {
    float2 z[4], zm[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int v = min(v0 + k * step, a.NC - 1);
      z[k] = buf[ipos[v] * LD + b];
      zm[k] = buf[ipos[v ? L - v : 0] * LD + b];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int v = v0 + k * step;
      if (v >= a.NC) break;
      const float2 ya = make_float2(0.5f * (z[k].x + zm[k].x), 0.5f * (z[k].y - zm[k].y));
      const float2 yb = make_float2(0.5f * (z[k].y + zm[k].y), 0.5f * (zm[k].x - z[k].x));
      float2* o = out + (int64_t)v * a.h;
      if (a.vec) {
        *(float4*)o = make_float4(ya.x, ya.y, yb.x, yb.y);
      } else {
        o[0] = ya;
        if (two) o[1] = yb;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Module column pass: forward LR column transform, times Phi, inverse HR column transform.  Above scale 1
// the LR bins pass through registers, so that one line buffer serves both transforms: 4 instead of 3 blocks per
// CU at 132 -> 264 points (layer call, us, two buffers -> one: 256 planes 132 -> 264: 114 -> 97; 64 planes
// 330 -> 990: 566 -> 372; 128 planes 16 -> 32, where the waves limit the blocks: 53 -> 54).
// ------------------------------------------------------------------------------------------------
constexpr int kUpRounds = 6;  // items of 2 lines per thread: 6 nth >= 8 h (launch_lines_cols)
struct ColsArgs {
  const float2* S;    // (P, NC, h)
  const float2* phi;  // (Cp, NCs, Hs)
  float2* SH;         // (P, NCs, Hs); S itself at scale 1
  const float2 *tw_h, *tw_H;
  int B, C, psf_batch;
  int w, Hs, NC, NCs, total, nblk;
  LinePlan ph, pH;    // column lengths h and Hs (pH unused at scale 1)
};

template <bool ONE>  // ONE: scale 1, in place
__global__ void __launch_bounds__(kLineThreads) k_lines_cols(ColsArgs) {
  const CVN_KARG ColsArgs& a = *(const CVN_KARG ColsArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NB = kLines, LD = kLineLd;
  const int tid = threadIdx.x, nth = blockDim.x, h = a.ph.L, Hs = ONE ? h : a.Hs;
  float2* X = (float2*)smem;  // the LR lines, then the HR lines
  char* p = smem + ((size_t)Hs * LD * sizeof(float2) + 15) / 16 * 16;
  int64_t* in = (int64_t*)p;  // per line: offset in S (complemented: the conjugate), in Phi, in SH
  int64_t *fi = in + NB, *oo = fi + NB;
  float2* twh = (float2*)(oo + NB);
  float2* twH = ONE ? twh : twh + a.ph.T;
  unsigned short* ih = (unsigned short*)(twH + (ONE ? a.ph.T : a.pH.T));
  unsigned short* iH = ONE ? ih : ih + h;
  const int g0 = line_item(blockIdx.x, a.nblk) * NB;
  const int nb = min(NB, a.total - g0);
  if (tid < NB) {
    // lines channel by channel: the planes that share a psf follow each other
    const int gc = min(g0 + tid, a.total - 1);
    const int q = gc / a.NCs, v = gc - q * a.NCs;
    const int c = q / a.B;
    const int64_t plane = (int64_t)(q - c * a.B) * a.C + c;
    const int64_t cp = a.psf_batch == 1 ? c : plane;
    oo[tid] = (plane * a.NCs + v) * Hs;
    fi[tid] = (cp * a.NCs + v) * Hs;
    const int vv = ONE ? v : v % a.w;  // a real row's spectrum is Hermitian in the column
    in[tid] = vv < a.NC ? (plane * a.NC + vv) * h : ~((plane * a.NC + (a.w - vv)) * h);
  }
  __syncthreads();
  const int nin = h * (NB / 8), nout = Hs * (NB / 8);
  for (int i0 = tid; i0 < nin || i0 == tid; i0 += nth) {
    const int idx = min(i0, nin - 1);
    const int q = mg_div(idx, a.ph.mgL, h), u = idx - q * h, b0 = 8 * q;
    float2 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t o = in[b0 + k];
      v[k] = a.S[(o < 0 ? ~o : o) + u];
      if (!ONE && o < 0) v[k].y = -v[k].y;
    }
    if (i0 == tid) {
      line_tables(a.ph, a.tw_h, ih, twh, tid, nth);
      if (!ONE) line_tables(a.pH, a.tw_H, iH, twH, tid, nth);
    }
    if (i0 < nin) {
#pragma unroll
      for (int k = 0; k < 8; ++k) X[u * LD + b0 + k] = v[k];
    }
  }
  __syncthreads();
  line_fft<true>(a.ph, smem, twh, tid, nth);
  if constexpr (ONE) {
    for (int idx = tid; idx < nout; idx += nth) {
      const int q = mg_div(idx, a.ph.mgL, h), u = idx - q * h, b0 = 8 * q;
      float2 f[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) f[k] = a.phi[fi[b0 + k] + u];
      float2* x = X + ih[u] * LD + b0;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float2 t = cmul(x[k], f[k]);
        x[k] = make_float2(t.y, t.x);
      }
    }
  } else {
    // each LR bin times Phi at its s aliases u + e h; items of 2 lines at one LR row, rows fastest
    const int n = h * (NB / 2);
    float2 y[kUpRounds][2];
    int ul[kUpRounds], bl[kUpRounds];
#pragma unroll
    for (int r = 0; r < kUpRounds; ++r) {
      if (r * nth >= n) break;
      const int idx = min(tid + r * nth, n - 1), q = mg_div(idx, a.ph.mgL, h);
      ul[r] = idx - q * h;
      bl[r] = 2 * q;
#pragma unroll
      for (int j = 0; j < 2; ++j) y[r][j] = X[ih[ul[r]] * LD + bl[r] + j];
    }
    __syncthreads();
    for (int u0 = 0; u0 < Hs; u0 += h) {
      float2 f[kUpRounds][2];
#pragma unroll
      for (int r = 0; r < kUpRounds; ++r) {
        if (r * nth >= n) break;  // (a wave's last rounds may hold nothing)
#pragma unroll
        for (int j = 0; j < 2; ++j) f[r][j] = a.phi[fi[bl[r] + j] + u0 + ul[r]];
      }
#pragma unroll
      for (int r = 0; r < kUpRounds; ++r)
        if (tid + r * nth < n) {
          float2* x = X + iH[u0 + ul[r]] * LD + bl[r];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float2 t = cmul(y[r][j], f[r][j]);
            x[j] = make_float2(t.y, t.x);
          }
        }
    }
  }
  __syncthreads();
  line_fft<false>(ONE ? a.ph : a.pH, smem, twH, tid, nth);
  for (int idx = tid; idx < nout; idx += nth) {
    const int q = mg_div(idx, ONE ? a.ph.mgL : a.pH.mgL, Hs), u = idx - q * Hs, b0 = 8 * q;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (b0 + k < nb) {
        const float2 t = X[u * LD + b0 + k];
        a.SH[oo[b0 + k] + u] = make_float2(t.y, t.x);
      }
  }
}

// ------------------------------------------------------------------------------------------------
// Inverse row pass: half spectra SH[plane][v][row] -> real rows; crop and activation on store, or the
// padding adjoint (pad >= 0, see k_rows_inv).
// ------------------------------------------------------------------------------------------------
struct RowsInvArgs {
  const float2* SH;
  float* out;
  float* side;
  const float2* tw;
  int Hs, NCs, row0, nrows, col0, ncols, act, npair, total, nblk;
  int vec;          // 16-byte loads of a row pair (Hs and row0 even, SH 16-byte aligned)
  int pad, pmode, dst_off;
  uint32_t mg_cols;
  LinePlan plan;
};

__global__ void __launch_bounds__(kLineThreads) k_lines_rows_inv(RowsInvArgs) {
  const CVN_KARG RowsInvArgs& a = *(const CVN_KARG RowsInvArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NB = kLines, LD = kLineLd;
  const int tid = threadIdx.x, nth = blockDim.x, L = a.plan.L;
  float2* buf = (float2*)smem;
  float2* tw = (float2*)(smem + ((size_t)L * LD * sizeof(float2) + 15) / 16 * 16);
  unsigned short* ipos = (unsigned short*)(tw + a.plan.T);
  float** dst = (float**)(smem + a.dst_off);  // 2 NB: each row's destination, null: none
  int* csrc = (int*)(dst + 2 * NB);
  const int g0 = line_item(blockIdx.x, a.nblk) * NB;
  const int Hd = a.nrows - 2 * a.pad, Wd = a.ncols - 2 * a.pad;  // the unpadded grid (pad >= 0)
  const int cols = a.pad >= 0 ? Wd : a.ncols, c0 = a.pad >= 0 ? a.pad : a.col0;
  const int nbd = (a.pad < 0 || a.pmode == CVN_PAD_ZEROS) ? 0 : 2 * a.pad;
  if (tid < 2 * NB) {
    const int gp = g0 + (tid >> 1);
    const int plane = gp / a.npair, r = 2 * (gp - plane * a.npair) + (tid & 1);
    float* d = nullptr;
    if (gp < a.total && r < a.nrows) {
      if (a.pad < 0) d = a.out + ((int64_t)plane * a.nrows + r) * cols;
      else if (r >= a.pad && r < a.pad + Hd) d = a.out + ((int64_t)plane * Hd + (r - a.pad)) * cols;
      else if (nbd > 0) d = a.side + ((int64_t)plane * nbd + (r < a.pad ? r : r - Hd)) * cols;
    }
    dst[tid] = d;
  }
  line_tables(a.plan, a.tw, ipos, tw, tid, nth);
  for (int q = tid; q < nbd; q += nth)
    csrc[q] = line_pad_src(q < a.pad ? q : Wd + q, Wd, a.pad, a.pmode);
  __syncthreads();
  {
    const int b = tid % NB, gp = min(g0 + b, a.total - 1);
    const int plane = gp / a.npair, r = 2 * (gp - plane * a.npair);
    const float2* in = a.SH + (int64_t)plane * a.NCs * a.Hs + a.row0 + r;
    const bool two = r + 1 < a.nrows;
    for (int v0 = tid / NB; v0 < a.NCs; v0 += 4 * (nth / NB)) {
      float2 fa[4], fb[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int v = min(v0 + k * (nth / NB), a.NCs - 1);
        const float2* s = in + (int64_t)v * a.Hs;
        if (a.vec) {
          const float4 t = *(const float4*)s;
          fa[k] = make_float2(t.x, t.y);
          fb[k] = make_float2(t.z, t.w);
        } else {
          fa[k] = s[0];
          fb[k] = two ? s[1] : make_float2(0.f, 0.f);
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int v = v0 + k * (nth / NB);
        if (v >= a.NCs) break;
        if (v == 0 || 2 * v == L) fa[k].y = fb[k].y = 0.f;
        // Z = Fa + i Fb and its mirror conj Fa + i conj Fb, real and imaginary parts exchanged
        buf[ipos[v] * LD + b] = make_float2(fa[k].y + fb[k].x, fa[k].x - fb[k].y);
        if (v > 0 && 2 * v < L) buf[ipos[L - v] * LD + b] = make_float2(fb[k].x - fa[k].y, fa[k].x + fb[k].y);
      }
    }
  }
  __syncthreads();
  line_fft<false>(a.plan, smem, tw, tid, nth);
  // buf[n LD + b] = (row 2 t + 1, row 2 t) of line b
  if (nbd > 0) {
    // border columns onto their padding sources: columns j <= pad or j >= Wd - 1 - pad
    const bool all = Wd <= 2 * a.pad + 2;
    const int ne = all ? Wd : 2 * a.pad + 2, b = tid % NB;
    for (int e = tid / NB; e < ne; e += nth / NB) {
      const int j = (all || e <= a.pad) ? e : Wd - 1 - a.pad + (e - a.pad - 1);
      float2 v = buf[(j + a.pad) * LD + b];
      for (int q = 0; q < nbd; ++q)
        if (csrc[q] == j) {
          const float2 z = buf[(q < a.pad ? q : Wd + q) * LD + b];
          v.x += z.x;
          v.y += z.y;
        }
      buf[(j + a.pad) * LD + b] = v;
    }
    __syncthreads();
  }
  for (int idx = tid; idx < cols * (NB / 4); idx += nth) {
    const int q = mg_div(idx, a.mg_cols, cols), j = idx - q * cols, b0 = 4 * q;
    float2 z[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      z[k] = buf[(c0 + j) * LD + b0 + k];
      if (a.act == CVN_ACT_GELU) z[k] = make_float2(gelu_fast(z[k].x), gelu_fast(z[k].y));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float *da = dst[2 * (b0 + k)], *db = dst[2 * (b0 + k) + 1];
      if (da) da[j] = z[k].y;
      if (db) db[j] = z[k].x;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Backward column pass (see k_cols_bwd): 16 LR column classes v0 per block, numbered through the psf
// groups; the block loops over the planes that share a psf.  Per plane: Y (LR columns of pad x) and, member
// by member, dZ (HR columns v0 + b w of the output gradient's rows) are transformed; dY = alias sum of
// conj(Phi') dZ goes back through the inverse LR transform to dS, in place over Sx; dPhi += conj(Y) dZ.
// dPhi is summed in global memory: every entry belongs to one thread, which adds its planes in order (no
// atomics, the same bits each time), and the block's 16 columns stay in L2; in registers the sums would
// have to live across the transforms, in LDS they would halve the blocks per CU.
// ------------------------------------------------------------------------------------------------
struct ColsBwdArgs {
  const float2* Sg;   // (P, NCs, Hs)
  float2* Sx;         // (P, NC, h): in (dphi != null) and out
  const float2* phi;  // (Cp, NCs, Hs)
  float2* dphi;       // (Cp, Ws, Hs) or null
  const float2 *tw_h, *tw_H;
  int nplanes, C;     // planes per psf: B (shared psf) or 1
  int w, s, Hs, Ws, NC, NCs, total, nblk;
  LinePlan ph, pH;
};

template <bool ONE>  // ONE: scale 1 (dY in place of dZ)
__global__ void __launch_bounds__(kLineThreads) k_lines_cols_bwd(ColsBwdArgs) {
  const CVN_KARG ColsBwdArgs& a = *(const CVN_KARG ColsBwdArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NB = kLines, LD = kLineLd;
  const int tid = threadIdx.x, nth = blockDim.x, h = a.ph.L, Hs = ONE ? h : a.Hs;
  const bool wg = a.dphi != nullptr;
  const size_t nh = ((size_t)h * LD * sizeof(float2) + 15) / 16 * 16;
  float2* Y = (float2*)smem;             // LR lines of pad x
  float2* X = (float2*)(smem + nh);      // HR lines of one member
  char* p = smem + nh + ((size_t)Hs * LD * sizeof(float2) + 15) / 16 * 16;
  float2* D = ONE ? X : (float2*)p;      // dY
  if (!ONE) p += nh;
  // per line, for the current plane and member: offsets in Sx, Sg and Phi' (complemented: the mirrored
  // column, conjugated) and dPhi
  int64_t* xo = (int64_t*)p;
  int64_t *go = xo + NB, *fo = go + NB, *po = fo + NB;
  float2* twh = (float2*)(po + NB);
  float2* twH = ONE ? twh : twh + a.ph.T;
  unsigned short* ih = (unsigned short*)(twH + (ONE ? a.ph.T : a.pH.T));
  unsigned short* iH = ONE ? ih : ih + h;
  const int g0 = line_item(blockIdx.x, a.nblk) * NB;
  const int nb = min(NB, a.total - g0);
  line_tables(a.ph, a.tw_h, ih, twh, tid, nth);
  if (!ONE) line_tables(a.pH, a.tw_H, iH, twH, tid, nth);
  const int members = ONE ? 1 : a.s;
  for (int ib = 0; ib < a.nplanes; ++ib) {
    for (int b = 0; b < members; ++b) {
      // the index arithmetic of each phase is formed again per plane: hoisted out of the loop, it would be
      // held (spilled) across the transforms
      int tl = tid;
      asm volatile("" : "+v"(tl));
      const int nih = h * (NB / 4), niH = Hs * (NB / 4);  // items of 4 lines at one row, rows fastest
      const uint32_t mgh = a.ph.mgL, mgH = ONE ? mgh : a.pH.mgL;
      __syncthreads();  // the previous member's product and the previous plane's stores have read theirs
      if (tl < NB) {
        const int gc = min(g0 + tl, a.total - 1), grp = gc / a.NC, col = gc - grp * a.NC, vb = col + b * a.w;
        const int64_t plane = (int64_t)ib * a.C + grp;
        const bool mir = !ONE && vb > a.Ws / 2;  // a real row's spectrum is Hermitian in the column
        const int vm = mir ? a.Ws - vb : vb;
        const int64_t g = (plane * a.NCs + vm) * Hs, f = ((int64_t)grp * a.NCs + vm) * Hs;
        xo[tl] = (plane * a.NC + col) * h;
        go[tl] = mir ? ~g : g;
        fo[tl] = mir ? ~f : f;
        po[tl] = ((int64_t)grp * a.Ws + vb) * Hs;
      }
      __syncthreads();
      if (wg && b == 0)
        for (int idx = tl; idx < nih; idx += nth) {
          const int q = mg_div(idx, mgh, h), u = idx - q * h;
          float2 v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = a.Sx[xo[4 * q + j] + u];
#pragma unroll
          for (int j = 0; j < 4; ++j) Y[u * LD + 4 * q + j] = v[j];
        }
      for (int idx = tl; idx < niH; idx += nth) {
        const int q = mg_div(idx, mgH, Hs), u = idx - q * Hs;
        float2 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t o = go[4 * q + j];
          v[j] = a.Sg[(!ONE && o < 0 ? ~o : o) + u];
          if (!ONE && o < 0) v[j].y = -v[j].y;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) X[u * LD + 4 * q + j] = v[j];
      }
      __syncthreads();
      for (int t = wg && b == 0 ? 0 : 1; t < 2; ++t) {
        const CVN_KARG LinePlan* pl = (ONE || t == 0) ? &a.ph : &a.pH;
        line_fft<true>(*pl, (char*)(t ? X : Y), t ? twH : twh, tl, nth);
      }
      // dY (+)= sum over the member's rows of a class of conj(Phi') dZ, real and imaginary parts exchanged
      // for the inverse transform; dPhi (+)= conj(Y) dZ / (Hs Ws).  Items of 2 lines at one LR row.
      const float norm = 1.0f / ((float)Hs * (float)a.Ws);
      int tp = tid;
      asm volatile("" : "+v"(tp));
      for (int idx = tp; idx < 2 * nih; idx += nth) {
        const int q = mg_div(idx, mgh, h), u0 = idx - q * h;
        const int py = ih[u0] * LD + 2 * q;
        float2 m[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) m[j] = make_float2(0.f, 0.f);
        for (int e = 0; e < members; ++e) {
          const int u = ONE ? u0 : u0 + e * h;
          const float2* xz = X + iH[u] * LD + 2 * q;
          float2 f[2], d[2];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int64_t o = fo[2 * q + j];
            f[j] = !ONE && o < 0 ? a.phi[~o + (u ? Hs - u : 0)] : a.phi[o + u];
            if (!ONE && o < 0) f[j].y = -f[j].y;
            d[j] = make_float2(0.f, 0.f);
            if (wg && ib > 0) d[j] = a.dphi[po[2 * q + j] + u];
          }
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float2 z = xz[j];
            const float2 t = cmul(cconj(f[j]), z);
            m[j].x += t.x;
            m[j].y += t.y;
            if (wg && 2 * q + j < nb) {
              const float2 g = cmul(cconj(Y[py + j]), z);
              a.dphi[po[2 * q + j] + u] = make_float2(fmaf(g.x, norm, d[j].x), fmaf(g.y, norm, d[j].y));
            }
          }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float2 t = make_float2(m[j].y, m[j].x);
          if (!ONE && b > 0) {
            const float2 o = D[py + j];
            t.x += o.x;
            t.y += o.y;
          }
          D[py + j] = t;
        }
      }
    }
    __syncthreads();
    int ts = tid;
    asm volatile("" : "+v"(ts));
    line_fft<false>(a.ph, (char*)D, twh, ts, nth);
    for (int idx = ts; idx < h * (NB / 4); idx += nth) {
      const int q = mg_div(idx, a.ph.mgL, h), u = idx - q * h;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * q + j < nb) {
          const float2 t = D[u * LD + 4 * q + j];
          a.Sx[xo[4 * q + j] + u] = make_float2(t.y, t.x);
        }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Operator column pass (arbitrary x0, see k_cols_op): 16 alias classes v0 in [0, w / 2] per block with all
// their members v0 + b w in LDS.  Rows are real, so column Ws - v of a row spectrum is the conjugate of
// column v: the members past Ws / 2 are read from, and written to, the mirrored stored columns, which
// covers the classes above w / 2 too (half the column transforms of one block per class).
// ------------------------------------------------------------------------------------------------
struct ColsOpArgs {
  const float2* S;   // (P, NC, h)    row spectra of y
  const float2* S0;  // (P, NCs, Hs)  row spectra of x0
  const float2* kf;  // (C, Ws, Hs)
  const float2* A;   // (C, Ws, Hs)   conj(K) / D / (Hs Ws)
  float2* SH;        // (P, NCs, Hs)
  const float2 *tw_h, *tw_H;
  int B, C, w, s, Hs, Ws, NC, NCs, total, nblk;
  LinePlan ph, pH;
};
constexpr int64_t kNoCol = INT64_MIN;

__global__ void __launch_bounds__(kLineThreads) k_lines_cols_op(ColsOpArgs) {
  const CVN_KARG ColsOpArgs& a = *(const CVN_KARG ColsOpArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NB = kLines, LD = kLineLd;
  const int tid = threadIdx.x, nth = blockDim.x, h = a.ph.L, Hs = a.Hs;
  const size_t nh = ((size_t)h * LD * sizeof(float2) + 15) / 16 * 16;
  const size_t nH = ((size_t)Hs * LD * sizeof(float2) + 15) / 16 * 16;
  float2* Y = (float2*)smem;
  char* X = smem + nh;  // member b at X + b nH
  // per line: offset in S; per member and line: offsets in S0 (complemented: mirrored and conjugated), the
  // tables, and SH (complemented: conjugated; kNoCol: a member whose mirror is another member, which stores it)
  int64_t* yo = (int64_t*)(X + a.s * nH);
  int64_t *xo = yo + NB, *ko = xo + a.s * NB, *oo = ko + a.s * NB;
  float2* twh = (float2*)(oo + a.s * NB);
  float2* twH = twh + a.ph.T;
  unsigned short* ih = (unsigned short*)(twH + a.pH.T);
  unsigned short* iH = ih + h;
  const int g0 = line_item(blockIdx.x, a.nblk) * NB;
  const int nb = min(NB, a.total - g0);
  for (int i = tid; i < a.s * NB; i += nth) {
    const int b = i / NB, gc = min(g0 + i - b * NB, a.total - 1);
    const int q = gc / a.NC, v0 = gc - q * a.NC, c = q / a.B;  // planes of a channel follow each other
    const int64_t plane = (int64_t)(q - c * a.B) * a.C + c;
    const int vb = v0 + b * a.w;
    const bool mir = vb > a.Ws / 2;
    const int64_t o = (plane * a.NCs + (mir ? a.Ws - vb : vb)) * Hs;
    if (b == 0) yo[i] = (plane * a.NC + v0) * h;
    xo[i] = mir ? ~o : o;
    ko[i] = ((int64_t)c * a.Ws + vb) * Hs;
    oo[i] = !mir ? o : (v0 == 0 || 2 * v0 == a.w) ? kNoCol : ~o;
  }
  line_tables(a.ph, a.tw_h, ih, twh, tid, nth);
  line_tables(a.pH, a.tw_H, iH, twH, tid, nth);
  __syncthreads();
  const int nih = h * (NB / 4), niH = Hs * (NB / 4);  // items of 4 lines at one row, rows fastest
  for (int idx = tid; idx < nih; idx += nth) {
    const int q = mg_div(idx, a.ph.mgL, h), u = idx - q * h;
    float2 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = a.S[yo[4 * q + j] + u];
#pragma unroll
    for (int j = 0; j < 4; ++j) Y[u * LD + 4 * q + j] = v[j];
  }
  for (int b = 0; b < a.s; ++b)
    for (int idx = tid; idx < niH; idx += nth) {
      const int q = mg_div(idx, a.pH.mgL, Hs), u = idx - q * Hs;
      float2 v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t o = xo[b * NB + 4 * q + j];
        v[j] = a.S0[(o < 0 ? ~o : o) + u];
        if (o < 0) v[j].y = -v[j].y;
      }
      float2* d = (float2*)(X + b * nH) + u * LD + 4 * q;
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = v[j];
    }
  __syncthreads();
  for (int t = 0; t <= a.s; ++t) {
    const CVN_KARG LinePlan* pl = t == 0 ? &a.ph : &a.pH;
    line_fft<true>(*pl, t == 0 ? (char*)Y : X + (t - 1) * nH, t == 0 ? twh : twH, tid, nth);
  }
  // X = X0 + A (Y - mean(K X0)) of every class, real and imaginary parts exchanged for the inverse
  {
    int ts = tid;
    asm volatile("" : "+v"(ts));  // (its index arithmetic is not to be held across the transforms)
    const float inv_s2 = 1.0f / (float)(a.s * a.s), norm = 1.0f / ((float)Hs * (float)a.Ws);
    for (int idx = ts; idx < 2 * nih; idx += nth) {
      const int q = mg_div(idx, a.ph.mgL, h), u0 = idx - q * h;
      float2 m[2] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
      for (int b = 0; b < a.s; ++b)
        for (int e = 0; e < a.s; ++e) {
          const int u = u0 + e * h;
          const float2* x = (const float2*)(X + b * nH) + iH[u] * LD + 2 * q;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float2 t = cmul(a.kf[ko[b * NB + 2 * q + j] + u], x[j]);
            m[j].x += t.x;
            m[j].y += t.y;
          }
        }
      const float2* y = Y + ih[u0] * LD + 2 * q;
#pragma unroll
      for (int j = 0; j < 2; ++j) m[j] = make_float2(y[j].x - m[j].x * inv_s2, y[j].y - m[j].y * inv_s2);
      for (int b = 0; b < a.s; ++b)
        for (int e = 0; e < a.s; ++e) {
          const int u = u0 + e * h;
          float2* x = (float2*)(X + b * nH) + iH[u] * LD + 2 * q;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float2 t = cmul(a.A[ko[b * NB + 2 * q + j] + u], m[j]), x0 = x[j];
            x[j] = make_float2(fmaf(x0.y, norm, t.y), fmaf(x0.x, norm, t.x));
          }
        }
    }
  }
  __syncthreads();
  for (int b = 0; b < a.s; ++b) line_fft<false>(a.pH, X + b * nH, twH, tid, nth);
  int ts = tid;
  asm volatile("" : "+v"(ts));
  for (int b = 0; b < a.s; ++b)
    for (int idx = ts; idx < niH; idx += nth) {
      const int q = mg_div(idx, a.pH.mgL, Hs), u = idx - q * Hs;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t o = oo[b * NB + 4 * q + j];
        if (4 * q + j < nb && o != kNoCol) {
          const float2 t = ((const float2*)(X + b * nH))[u * LD + 4 * q + j];
          a.SH[(o < 0 ? ~o : o) + u] = make_float2(t.y, o < 0 ? -t.x : t.x);
        }
      }
    }
}

std::atomic<uint64_t> g_line_attr{0};
void line_attrs() {
  once_per_device(g_line_attr, [] {
    for (const void* k : {(const void*)k_lines_rows_fwd, (const void*)k_lines_rows_inv, (const void*)k_lines_cols<true>,
                          (const void*)k_lines_cols<false>, (const void*)k_lines_cols_bwd<true>,
                          (const void*)k_lines_cols_bwd<false>, (const void*)k_lines_cols_op})
      (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kLineLds);
    (void)hipGetLastError();
  });
}

constexpr int kCus = 256;  // compute units of the device

// Threads per block.  The kernels take up to 128 VGPRs, so a CU holds 16 waves.  Measured over 27 lengths
// from 24 to 560 (1 to 16 waves per block): a power of two near one wave per 64 elements of length (16
// elements per thread) is the fastest or within 6 % of it, and an uneven share of the 16 waves (3, 5) up to
// 30 % slower.  Where the blocks are too few to fill the chip, waves are doubled while all blocks stay
// resident and the widest pass still gives every wave a butterfly per lane (64 planes of 136 x 136: 37 -> 28 us), or,
// for the loads and stores, a thread has 4 elements or more and the chip is half empty (a call on 2 to 64 planes of 16 to
// 264 rows or columns of 64: 1 to 3 us of 20 to 27 us less; 2 elements: 0.5 us more than 4; beyond half full 1 to 4 %
// slower).
// lds: the block's LDS, where it holds more than one line buffer (fewer blocks per CU, more waves each).
int line_threads(const LinePlan& p, int nblk, size_t lds = 0) {
  int w = 1, most = 1;
  while (w < 16 && w * 64 * 1.41421 < p.L) w *= 2;
  for (int t = 0; t < p.np; ++t) most = std::max(most, p.ps[t].nl * kLines);
  if (lds) most = std::max(most, p.L * 8);  // the product's items
  while (lds && 2 * w * (int)(kLineLds / lds) <= 16 && 64 * w < most) w *= 2;
  while (2 * w <= 16 && (int64_t)nblk * 2 * w <= kCus * 16 && 64 * w < most) w *= 2;
  while (2 * w <= 16 && (int64_t)nblk * 2 * w <= kCus * 8 && 4 * 64 * w < p.L * kLines) w *= 2;
  return std::max(64 * w, line_min_threads(p));
}

// Whether the runtime-plan passes' transform of length L has no prime above 13: with one, they are never the faster
// (136 = 8 17: 1.8 times this engine's time at any number of blocks).
bool plain_plan(int L) {
  const FftPlan* p = fft_plan(L);
  if (!p) return false;
  for (int i = 0; i < p->nst; ++i)
    if (p->radix[i] > 13) return false;
  return true;
}

// Butterflies of the widest radix.
int narrowest(const LinePlan& p) {
  int n = p.L;
  for (int t = 0; t < p.np; ++t) n = std::min(n, p.ps[t].nl);
  return n;
}

}  // namespace

// Rows of lengths up to 1024, except where the blocks leave much of the chip idle and the runtime-plan pass, with 2 to 8
// rows to a block instead of 32, is the faster one (two row passes and a column pass of 64 rows, us, that / this):
//   one or two butterflies per line, so that most of a block idles: rows of 24: 18.7 / 19.3, 32: 19.2 / 21.2, 50:
//     21.2 / 22.3 (of 16: 18.4 / 18.4; three of 48: 20.7 / 19.9); at 128 blocks 19.5 / 19.9, 20.0 / 21.2, 22.3 / 22.3, at 256
//     20.8 / 19.6, 21.5 / 20.9, 24.6 / 22.6;
//   the lengths with a compile-time form of that pass: 132: 19.5 / 22.4, 256: 22.8 / 24.6, 260: 22.4 / 24.9; at 128
//     blocks 21.9 / 23.4, 27.5 / 26.7, 30.0 / 27.1; at 192 23.8 / 23.9, 32.7 / 27.8, 34.7 / 28.3;
//   long rows in few blocks, one per CU: 640: 31.2 / 33.2, 768: 29.0 / 35.2, 1024: 31.6 / 37.5 (600: 31.7 / 32.0); at 48
//     blocks 40.3 / 35.2, 42.2 / 37.8, 49.3 / 40.8.
bool lines_rows_ok(int64_t P, int h, int w) {
  const LinePlan* p = line_plan(w);
  const int64_t lines = P * ((h + 1) / 2), nblk = (lines + kLines - 1) / kLines;
  if (!p || lines >= (1 << 30)) return false;
  const bool few = narrowest(*p) <= 2 ? 4 * nblk < 3 * kCus
                   : fixed_len(w)        ? nblk * w < 100 * kCus
                                         : w >= 640 && 8 * nblk < kCus;
  return !few || !plain_plan(w);
}

int launch_lines_rows_fwd(const float* x, int64_t P, int Hin, int Win, int pad, int mode, int h, int w,
                          const float2* tw, float2* S, hipStream_t st) {
  RowsFwdArgs a;
  const LinePlan* lp = line_plan(w);
  if (!lp) return fail(CVN_ERR_UNSUPPORTED, "no plan for length %d", w);
  a.plan = *lp;
  line_attrs();
  a.x = x; a.S = S; a.tw = tw; a.Hin = Hin; a.Win = Win; a.h = h; a.pad = pad; a.mode = mode;
  a.NC = w / 2 + 1;
  a.npair = (h + 1) / 2;
  a.total = (int)(P * a.npair);
  a.vec = h % 2 == 0 && ((uintptr_t)S & 15) == 0;
  const size_t lds = line_buf_bytes(w) + line_tab_bytes(a.plan) + 2 * kLines * sizeof(int64_t);
  a.nblk = (a.total + kLines - 1) / kLines;
  hipLaunchKernelGGL(k_lines_rows_fwd, dim3((unsigned)a.nblk), dim3(line_threads(a.plan, a.nblk)), lds, st, a);
  return check_launch("row forward pass");
}

// Columns that fit the LDS, except long ones in few blocks, where k_cols_module has more and smaller ones (a call of
// 64 columns of the length at scale 1, us, that / this): 512: 27.8 / 33.5, 768: 28.9 / 40.4, 1024: 30.6 / 45.3, at 50 blocks
// 31.3 / 34.9, 35.5 / 43.1, 39.8 / 48.8, at 132 blocks 43.7 / 40.2, 57.4 / 52.3, 64.4 / 60.0; with other factors only from 900
// on: 800 30.9 / 30.6, 1000 32.1 / 38.2, at 50 blocks 37.5 / 32.3, 40.4 / 40.8.
bool lines_cols_ok(int64_t P, int h, int Hs, int NCs) {
  if (!line_plan(h) || !line_plan(Hs) || P * NCs >= (1 << 30)) return false;
  const int64_t nblk = (P * NCs + kLines - 1) / kLines;
  if ((Hs % 128 == 0 ? Hs >= 512 && 8 * nblk < 3 * kCus : Hs >= 900 && 8 * nblk < kCus) && plain_plan(h) && plain_plan(Hs))
    return false;
  return line_buf_bytes(Hs) + line_tab_bytes(*line_plan(h)) + line_tab_bytes(*line_plan(Hs)) +
                 3 * kLines * sizeof(int64_t) <= kLineLds;
}

int launch_lines_cols(const float2* S, const float2* phi, float2* SH, int64_t B, int64_t C, int64_t psf_batch, int h,
                      int w, int Hs, int Ws, const float2* tw_h, const float2* tw_H, hipStream_t st) {
  ColsArgs a;
  const LinePlan *lh = line_plan(h), *lH = line_plan(Hs);
  if (!lh || !lH) return fail(CVN_ERR_UNSUPPORTED, "no plan for column length");
  a.ph = *lh;
  a.pH = *lH;
  line_attrs();
  const bool one = Hs == h;
  a.S = S; a.phi = phi; a.SH = SH; a.tw_h = tw_h; a.tw_H = tw_H;
  a.B = (int)B; a.C = (int)C; a.psf_batch = (int)psf_batch;
  a.w = w; a.Hs = Hs; a.NC = w / 2 + 1; a.NCs = Ws / 2 + 1;
  a.total = (int)(B * C * a.NCs);
  size_t lds = line_buf_bytes(Hs) + line_tab_bytes(a.ph) + 3 * kLines * sizeof(int64_t);
  if (!one) lds += line_tab_bytes(a.pH);
  a.nblk = (a.total + kLines - 1) / kLines;
  int nth = std::max(line_threads(a.ph, a.nblk), line_threads(a.pH, a.nblk));
  if (!one) nth = std::max(nth, ((kLines / 2 * h + kUpRounds - 1) / kUpRounds + 63) / 64 * 64);  // at most 704
  const dim3 grid((unsigned)a.nblk), block(nth);
  if (one) hipLaunchKernelGGL(k_lines_cols<true>, grid, block, lds, st, a);
  else hipLaunchKernelGGL(k_lines_cols<false>, grid, block, lds, st, a);
  return check_launch("column pass");
}

namespace {
size_t cols_bwd_lines_lds(int h, int Hs, int s) {
  size_t n = 2 * line_buf_bytes(h) + line_tab_bytes(*line_plan(h)) + 4 * kLines * sizeof(int64_t);
  if (s > 1) n += line_buf_bytes(Hs) + line_tab_bytes(*line_plan(Hs));
  return n;
}
}  // namespace

namespace {
// Whether k_cols_bwd (1 to 8 columns per block) is the faster one: with less than about a block per CU, the lines
// pass is a serial chain over the planes of a psf beside idle CUs.  Time of the whole backward with that one over the
// time with this one, columns of h, B planes per psf, 4 to 84 blocks (it hardly depends on their number there):
//   scale > 1: B 2 0.97 to 0.87, B 4 0.96 to 0.78, B 16 0.89 to 0.64 at h s = 32 to 400; B 1 1.04 to 0.97 at scale 2, 0.99 to
//     0.93 at scale 3.  Columns up to 192: still at 132 blocks (192 rows, B 16 523 / 643 us); longer ones: 98 blocks
//     313 / 363, 102 blocks of 400 rows 184 / 177, 392 blocks of 256 265 / 213.
//   scale 1, where a block holds one column buffer less: h 24 1.00 at B 2, 0.96 at B 4, 0.85 at B 16, and 32 0.95, 0.88, 0.74, one
//     butterfly per line; 64 (k_cols_bwd in two stages) 1.00 at B 4, 0.96 at B 8, 0.93 at B 16; 320 and 400 0.93 at B 4, 0.85 at B 16,
//     but 1.02 at 84 blocks; otherwise 36 1.12, 48 1.08, 120 1.10 at any B, 100 and 128 1.00 at B 4, 0.95 at B 16, 200 1.00.
bool few_bwd_blocks(int64_t nblk, int64_t nplanes, int h, int s) {
  if (!plain_plan(h) || !plain_plan(h * s)) return false;
  const int64_t part = h * s <= 192 ? 4 * nblk : 8 * nblk;  // of 3 blocks per CU
  if (s > 1) return part < 3 * kCus && (nplanes > 1 || s > 2);
  if (narrowest(*line_plan(h)) <= 2) return 8 * nblk < 3 * kCus && nplanes > 1;
  return h >= 256 ? 5 * nblk < kCus && nplanes >= 4 : 8 * nblk < 3 * kCus && nplanes >= 8 && fft_plan(h)->nst <= 2;
}
}  // namespace

bool lines_cols_bwd_ok(int64_t P, int64_t nplanes, int h, int Hs, int s, int NC) {
  if (line_plan(h) && few_bwd_blocks((P / nplanes * NC + kLines - 1) / kLines, nplanes, h, s)) return false;
  return line_plan(h) && line_plan(Hs) && P * NC < (1 << 30) && cols_bwd_lines_lds(h, Hs, s) <= kLineLds;
}

int launch_lines_cols_bwd(const float2* Sg, float2* Sx, const float2* phi, float2* dphi, int64_t B, int64_t C,
                          int64_t psf_batch, int h, int w, int s, const float2* tw_h, const float2* tw_H, hipStream_t st) {
  ColsBwdArgs a;
  const LinePlan *lh = line_plan(h), *lH = line_plan(h * s);
  if (!lh || !lH) return fail(CVN_ERR_UNSUPPORTED, "no plan for column length");
  a.ph = *lh;
  a.pH = *lH;
  line_attrs();
  a.Sg = Sg; a.Sx = Sx; a.phi = phi; a.dphi = dphi; a.tw_h = tw_h; a.tw_H = tw_H;
  a.nplanes = psf_batch == 1 ? (int)B : 1;
  a.C = (int)C;
  a.w = w; a.s = s; a.Hs = h * s; a.Ws = w * s; a.NC = w / 2 + 1; a.NCs = w * s / 2 + 1;
  a.total = (int)(psf_batch == 1 ? C : B * C) * a.NC;
  a.nblk = (a.total + kLines - 1) / kLines;
  const size_t lds = cols_bwd_lines_lds(h, h * s, s);
  const dim3 grid((unsigned)a.nblk), block(std::max(line_threads(a.ph, a.nblk, lds), line_threads(a.pH, a.nblk, lds)));
  if (s == 1) hipLaunchKernelGGL(k_lines_cols_bwd<true>, grid, block, lds, st, a);
  else hipLaunchKernelGGL(k_lines_cols_bwd<false>, grid, block, lds, st, a);
  return check_launch("backward column pass");
}

namespace {
size_t cols_op_lines_lds(int h, int Hs, int s) {
  return line_buf_bytes(h) + s * line_buf_bytes(Hs) + line_tab_bytes(*line_plan(h)) + line_tab_bytes(*line_plan(Hs)) +
         (1 + 3 * (size_t)s) * kLines * sizeof(int64_t);
}
}  // namespace

// A block runs s + 1 transforms and s^2 bins per class one after another, k_cols_op one block per class: with
// few blocks that one is faster (us, this / that: 36 blocks at s = 4 50 / 40, 24 at s = 3 52 / 47, 36 and 42 at
// s = 2 40 / 38 and 36 / 42, 33 at s = 1 37 / 44; 104 at s = 3 45 / 65, 216 at s = 4 57 / 104).
bool lines_cols_op_ok(int64_t P, int h, int Hs, int s, int w) {
  if (P * (w / 2 + 1) < (int64_t)kLines * 20 * s) return false;
  return line_plan(h) && line_plan(Hs) && P * (w / 2 + 1) < (1 << 30) && cols_op_lines_lds(h, Hs, s) <= kLineLds;
}

int launch_lines_cols_op(const float2* S, const float2* S0, const float2* kf, const float2* A, float2* SH, int64_t B,
                         int64_t C, int h, int w, int s, const float2* tw_h, const float2* tw_H, hipStream_t st) {
  ColsOpArgs a;
  const LinePlan *lh = line_plan(h), *lH = line_plan(h * s);
  if (!lh || !lH) return fail(CVN_ERR_UNSUPPORTED, "no plan for column length");
  a.ph = *lh;
  a.pH = *lH;
  line_attrs();
  a.S = S; a.S0 = S0; a.kf = kf; a.A = A; a.SH = SH; a.tw_h = tw_h; a.tw_H = tw_H;
  a.B = (int)B; a.C = (int)C;
  a.w = w; a.s = s; a.Hs = h * s; a.Ws = w * s; a.NC = w / 2 + 1; a.NCs = w * s / 2 + 1;
  a.total = (int)(B * C * a.NC);
  a.nblk = (a.total + kLines - 1) / kLines;
  const size_t lds = cols_op_lines_lds(h, h * s, s);
  const dim3 block(std::max(line_threads(a.ph, a.nblk, lds), line_threads(a.pH, a.nblk, lds)));
  hipLaunchKernelGGL(k_lines_cols_op, dim3((unsigned)a.nblk), block, lds, st, a);
  return check_launch("op column pass");
}

int launch_lines_rows_inv(const float2* SH, int64_t P, int Hs, int Ws, int row0, int nrows, int col0, int ncols, int act,
                          const float2* tw, float* out, hipStream_t st, int pad, int pmode, float* side) {
  RowsInvArgs a;
  const LinePlan* lp = line_plan(Ws);
  if (!lp) return fail(CVN_ERR_UNSUPPORTED, "no plan for length %d", Ws);
  a.plan = *lp;
  line_attrs();
  a.SH = SH; a.out = out; a.side = side; a.tw = tw; a.Hs = Hs; a.NCs = Ws / 2 + 1;
  a.row0 = row0; a.nrows = nrows; a.col0 = col0; a.ncols = ncols; a.act = act;
  a.pad = pad; a.pmode = pmode;
  a.npair = (nrows + 1) / 2;
  a.total = (int)(P * a.npair);
  a.vec = Hs % 2 == 0 && row0 % 2 == 0 && nrows % 2 == 0 && ((uintptr_t)SH & 15) == 0;
  a.mg_cols = line_magic(pad >= 0 ? ncols - 2 * pad : ncols);
  a.dst_off = (int)(line_buf_bytes(Ws) + line_tab_bytes(a.plan));
  const size_t lds = a.dst_off + 2 * kLines * sizeof(float*) + sizeof(int) * 2 * std::max(pad, 0);
  a.nblk = (a.total + kLines - 1) / kLines;
  hipLaunchKernelGGL(k_lines_rows_inv, dim3((unsigned)a.nblk), dim3(line_threads(a.plan, a.nblk)), lds, st, a);
  return check_launch("row inverse pass");
}

}  // namespace cvn
