// dps_spread_fx.hip -- spreading of FP64 arrays onto FP32 grids by int32 fixed
// point, whose sums do not depend on their order.  FP64 results of a
// mixed-precision solver stay the same to the last bits as before the matrix
// products, whose sums differ by 1e-7 -- within the accuracy of either, but not
// within an FP64 comparison with stored results; so this pair of types keeps
// these kernels
// (SpreadInterp.cpp:302-448 + BoundaryConditions.h:22-361 +
// SpreadInterpWrapper.cpp:66-107).
//
//  k_fx_cells    the (tile, z chunk) cells that a pass's entries reach: counts,
//                then (after k_fx_scan) the entry lists; with the positions, once
//                a solver has had a product of this pass
//  k_fx_absmax   partial maxima of |F|, |T| for the fixed-point scale, and
//                partial sums for the choice of a finer one
//  k_spread_fx   one workgroup per cell, LDS accumulation, one coalesced write
//                per grid element
#include <hip/hip_runtime.h>
#include <algorithm>
#include "dps_core.h"
#include "dps_internal.h"

namespace dps {

namespace {

// exclusive scan of counts[0..n) into start[0..n], counts turned into cursors
__global__ void __launch_bounds__(1024) k_fx_scan(int* counts, int* start, int n)
{
  __shared__ int part[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int per = (n + 1023) / 1024;
  const int b = min(n, t * per), e = min(n, b + per);
  int s = 0;
  for (int i = b; i < e; ++i) s += counts[i];
  int inc = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  if (lane == 63) part[wave] = inc;
  __syncthreads();
  int run = inc - s;
  for (int w = 0; w < wave; ++w) run += part[w];
  for (int i = b; i < e; ++i) {
    const int c = counts[i];
    start[i] = run;
    counts[i] = run;
    run += c;
  }
  if (t == 1023) start[n] = run;
}

__global__ void __launch_bounds__(256) k_fx_zero(int* a, int n)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) a[i] = 0;
}

// each (particle, kind) entry once per cell its support reaches: kind 0 over
// the rows of kernel 0, or (pair) of both kernels, kind 1 those of kernel 1
template <bool SCATTER>
__global__ void __launch_bounds__(256) k_fx_cells(FxArgs A)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= A.N * A.nkind) return;
  const int p = i / A.nkind, kind = i - p * A.nkind;
  const int4 s = (kind ? A.sup1 : A.sup0)[p];
  int klo = s.z, n = s.w;
  if (A.pair) {
    const int4 d = A.sup1[p];
    if (d.w > 0) {
      const int hi = n > 0 ? max(klo + n, d.z + d.w) : d.z + d.w;
      klo = n > 0 ? min(klo, d.z) : d.z;
      n = hi - klo;
    }
  }
  const int wx = kind ? A.wx1 : A.wx0, wy = kind ? A.wy1 : A.wy0;
  for_run_tiles(s.y, wy, A.Ny, FX_TY, [&](int ty) {
    for_run_tiles(s.x, wx, A.Nx, FX_TX, [&](int tx) {
      // rows wrap when z is periodic, else they are interior rows
      for_run_tiles(klo, n, A.periodic_z ? A.Nz : (1 << 30), A.ZC, [&](int ch) {
        const int cell = (ty * A.ntx + tx) * A.nch + ch;
        if (!SCATTER) {
          atomicAdd(&A.counts[cell], 1);
        } else {
          const int at = atomicAdd(&A.counts[cell], 1);
          if (at < A.cap) A.entries[at] = 2 * p + kind;
        }
      });
    });
  });
}

// per block: the largest |F| and |T| (NaN propagates), and the sums of squares
// and numbers of nonzero values of F and T
__global__ void __launch_bounds__(256) k_fx_absmax(const double* __restrict__ F, const double* __restrict__ Tq, int n3,
                                                FxStats* __restrict__ out)
{
  __shared__ FxStats red[4];
  FxStats v{};
  auto max2 = [](float m, float a) { return (a > m || a != a) ? a : m; };
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n3; i += gridDim.x * 256) {
    const double f = F[i], t = Tq ? Tq[i] : 0.0;
    v.fm = max2(v.fm, fabsf((float)f));
    v.tm = max2(v.tm, fabsf((float)t));
    v.f2 += f * f;
    v.t2 += t * t;
    v.nf += f != 0;
    v.nt += t != 0;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    v.fm = max2(v.fm, __shfl_xor(v.fm, o, 64));
    v.tm = max2(v.tm, __shfl_xor(v.tm, o, 64));
    v.f2 += __shfl_xor(v.f2, o, 64);
    v.t2 += __shfl_xor(v.t2, o, 64);
    v.nf += __shfl_xor(v.nf, o, 64);
    v.nt += __shfl_xor(v.nt, o, 64);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      v.fm = max2(v.fm, red[w].fm);
      v.tm = max2(v.tm, red[w].tm);
      v.f2 += red[w].f2;
      v.t2 += red[w].t2;
      v.nf += red[w].nf;
      v.nt += red[w].nt;
    }
    out[blockIdx.x] = v;
  }
}

// one contiguous piece of a periodic support range intersected with a tile:
// support columns b..b+w-1 (unwrapped) against [t0, t0+n), images shifted by
// multiples of the period.  Returns count, first support index in *i0 and the
// tile-local column of that index in *l0.
__device__ __forceinline__ int clip_piece(int b, int w, int t0, int n, int period, int shift,
                                          int* i0, int* l0)
{
  const int lo = max(b + shift, t0), hi = min(b + shift + w, t0 + n);
  if (hi <= lo) return 0;
  *i0 = lo - (b + shift);
  *l0 = lo - t0;
  return hi - lo;
}

// word `off` of an unpadded record's spreading parts ([x][y][z], derivative
// kernels [x][y][dx][dy][z][dz]) in the padded layout
__device__ __forceinline__ int padded(int off, int wx, int wy, int W, int deriv)
{
  int n = 1 + (off >= wx) + (off >= wx + wy);
  if (deriv) n += (off >= 2 * wx + wy) + (off >= 2 * (wx + wy)) + (off >= 2 * (wx + wy) + W);
  return off + n;
}

// A cell's scale from bounds on its columns: the first row of its tile sums, entry
// by entry (one per thread), the largest |contribution| of the entry at any level
// of a column, in units four times the present scale's (an entry's bound here is
// at most 1.5 times the one that scale allows for).
__device__ __forceinline__ void tight_scale(const FxArgs& A, const double* __restrict__ F, const double* __restrict__ Tq,
                                         int e0, int ncand, int X0, int Y0, int nX, int nY, int* acc, int RS, int* red,
                                         float* scl)
{
  const float u = 0.25f * scl[0];
  auto largest = [](const double* v) { return fmaxf(fmaxf(fabsf((float)v[0]), fabsf((float)v[1])), fabsf((float)v[2])); };
  for (int k = threadIdx.x; k < ncand; k += 256) {
    const int ent = A.entries[e0 + k], p = ent >> 1, kind = ent & 1;
    const int4 s = (kind ? A.sup1 : A.sup0)[p];
    const float* rm = (const float*)A.rec + (size_t)p * A.rs;
    const float* rd = rm + A.off1;
    const bool plain = !kind, deriv = kind || A.pair;
    const RecLayout R = rec_layout(A.wx0, A.wy0, A.W0, 0, 1), D = rec_layout(A.wx1, A.wy1, A.W1, 1, 1);
    float m = 0, a = 0, b = 0;   // largest z weight; z factors of the x and y derivatives, of the z derivative
    if (plain) {
      for (int q = 0; q < A.W0; ++q) m = fmaxf(m, fabsf(rm[R.z + q]));
      m *= u * largest(F + 3 * (size_t)p);
    }
    if (deriv) {
      for (int q = 0; q < A.W1; ++q) {
        a = fmaxf(a, fabsf(rd[D.z + q]));
        b = fmaxf(b, fabsf(rd[D.dz + q]));
      }
      const float t = 0.5f * u * largest(Tq + 3 * (size_t)p);
      a *= t;
      b *= t;
    }
    const int wx = kind ? A.wx1 : A.wx0, wy = kind ? A.wy1 : A.wy0;
    for (int j = 0; j < wy; ++j) {
      int y = s.y + j;
      y += y < 0 ? A.Ny : (y >= A.Ny ? -A.Ny : 0);
      if ((unsigned)(y - Y0) >= (unsigned)nY) continue;
      for (int i = 0; i < wx; ++i) {
        int x = s.x + i;
        x += x < 0 ? A.Nx : (x >= A.Nx ? -A.Nx : 0);
        if ((unsigned)(x - X0) >= (unsigned)nX) continue;
        float v = 0;
        if (plain) v = fabsf(rm[R.x + i] * rm[R.y + j]) * m;
        if (deriv)
          v += (fabsf(rd[D.dx + i] * rd[D.y + j]) + fabsf(rd[D.x + i] * rd[D.dy + j])) * a +
               fabsf(rd[D.x + i] * rd[D.y + j]) * b;
        atomicAdd(&acc[(y - Y0) * RS + x - X0], __float2int_ru(v));
      }
    }
  }
  __syncthreads();
  int m = 0;
  for (int i = threadIdx.x; i < FX_TY * RS; i += 256) {
    m = max(m, acc[i]);
    acc[i] = 0;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = max(max(max(red[0], red[1]), max(red[2], red[3])), 1);
    int S = 0;
    (void)frexpf(scl[0], &S);              // the scale is 2^(S - 1)
    S = min(S - 1 - 2 + __clz(m) - 2, 120);   // 4 m < 2^(34 - clz): partial sums below 2^30 again
    scl[0] = ldexpf(1.0f, S);
    scl[1] = ldexpf(1.0f, -S);
  }
  __syncthreads();
}

// One workgroup owns a cell: FX_TX x FX_TY columns and ZC z rows.  Its entries
// are staged in batches, 16 threads per entry loading record, support and
// force one batch ahead; a wavefront spreads one entry at a time, a lane per
// column of the entry's clipped support (with at most 32 columns the wave
// splits the rows into phases).  Every grid element of the cell is written to
// HBM once, coalesced.
template <int NPF, bool PAIR>
__global__ void __launch_bounds__(256) k_spread_fx(FxArgs A, const double* __restrict__ F,
                                                   const double* __restrict__ Tq)
{
  typedef float T;
  typedef double Tin;
  constexpr int B = FX_BATCH;     // queued entries staged per batch, 16 threads each
  constexpr int SLOT = 16 * NPF;          // words per staged entry: record, then header at rs_max
  constexpr int TX = FX_TX, TY = FX_TY;
  // padded tile [c][z][y][x]: row stride TX+1, odd plane stride, so that the
  // lanes of one atomic instruction spread over the LDS banks
  constexpr int RS = TX + 1, PL = TY * RS + 1;
  // int32 fixed point: ds_add_u32 is the fastest LDS atomic (~6 cycles per
  // 64-lane instruction per CU, ds_add_f32 ~193, measured on gfx950), and
  // integer sums do not depend on the order of the additions.  The scale 2^S
  // keeps every partial sum below 2^30: a point receives at most one term
  // per entry of the cell, each at most K0 max|F| + K1 max|T|.  Where that bound
  // is far above the sums -- many entries, which do not all meet at one point, or a
  // few large values among many -- its unit would be too coarse (1500 particles
  // under one tile: grid 2.8e-5 off; 8000 with one force 100 times the others
  // 3.3e-3), and the cell's columns are bounded one by one (tight_scale): 1.5e-6 and
  // 4.1e-6, at 493 and 2837 us a product of either with torques (532 and 2989 with
  // the coarse unit and the kernel before).
  typedef int TA;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  TA* acc = reinterpret_cast<TA*>(smem_raw);
  const int vol = A.ZC * PL;
  T* bst = reinterpret_cast<T*>(acc + 3 * vol);           // [B][SLOT] staged entries
  int* queue = reinterpret_cast<int*>(bst + B * SLOT);     // p * 2 + kind
  // fixed-point scale and its inverse; the bound on the cell's sums, and the
  // root mean square of an entry's
  float* scl = reinterpret_cast<float*>(queue + 2 * 256);
  T* __restrict__ grid = reinterpret_cast<T*>(A.grid);
  // cells in list order, consecutive cells (the chunks of a tile, then the
  // next tile) on one XCD, whose L2 then holds their shared records
  const int cell = xcd_group(blockIdx.x, gridDim.x);
  const int zc = cell % A.nch, tile = cell / A.nch;
  const int tx = tile % A.ntx, ty = tile / A.ntx;
  const int X0 = tx * TX, Y0 = ty * TY, Z0 = zc * A.ZC;
  const int nX = min(TX, A.Nx - X0), nY = min(TY, A.Ny - Y0), nZ = min(A.ZC, A.Nz - Z0);
  for (int i = threadIdx.x; i < 3 * vol; i += blockDim.x) acc[i] = (TA)0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwaves = blockDim.x >> 6;
  // this cell's entries (launch_fx_lists)
  const int e0 = A.start[cell];
  const int ncand = max(0, min(A.start[cell + 1], A.cap) - e0);   // within the list's capacity
  if (wave == 0) {
    // the scale: a NaN in the inputs propagates to the whole tile
    float fm = 0.0f, tm = 0.0f;
    for (int i = lane; i < FX_AMAX_BLOCKS; i += 64) {
      const float a = A.stats[i].fm, b = A.stats[i].tm;
      fm = (a > fm || a != a) ? a : fm;
      tm = (b > tm || b != b) ? b : tm;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const float a = __shfl_xor(fm, o, 64), b = __shfl_xor(tm, o, 64);
      fm = (a > fm || a != a) ? a : fm;
      tm = (b > tm || b != b) ? b : tm;
    }
    if (lane == 0) {
      const double bound = (double)ncand * (A.K0 * fm + A.K1 * tm);
      int e = 0;
      (void)frexp(bound, &e);   // bound < 2^e
      const int S = min(30 - e, 120);
      scl[0] = ldexpf(1.0f, S);
      scl[1] = isfinite(bound) ? ldexpf(1.0f, -S) : __builtin_nanf("");
      scl[2] = (float)bound;
    }
  } else if (wave == 1) {
    double f2 = 0, t2 = 0;
    int nf = 0, nt = 0;
    for (int i = lane; i < FX_AMAX_BLOCKS; i += 64) {
      f2 += A.stats[i].f2;
      t2 += A.stats[i].t2;
      nf += A.stats[i].nf;
      nt += A.stats[i].nt;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      f2 += __shfl_xor(f2, o, 64);
      t2 += __shfl_xor(t2, o, 64);
      nf += __shfl_xor(nf, o, 64);
      nt += __shfl_xor(nt, o, 64);
    }
    if (lane == 0)
      scl[3] = (float)sqrt((A.K0 * A.K0 * f2 + A.K1 * A.K1 * t2) / max(1, A.pair ? max(nf, nt) : nf + nt));
  }
  // the zeroed accumulator and the scale are complete before any thread adds
  // to the tile or, for a cell without entries, writes it out
  __syncthreads();
  // the scale is folded into each column's coefficients: add takes values
  // already in fixed-point units
  if (scl[2] > FX_COARSE * scl[3] && isfinite(scl[2])) tight_scale(A, F, Tq, e0, ncand, X0, Y0, nX, nY, acc, RS, queue, scl);
  const T sc = scl[0];
  auto add = [&](TA* d, T v) { atomicAdd(d, __float2int_rn(v)); };
  // z weight q of a row list of n entries, zero outside [0, n): the index
  // is clamped so the LDS read stays inside the slot
  auto zw = [&](const T* z, int q, int n) {
    const bool in = (unsigned)q < (unsigned)n;
    const T v = z[in ? q : 0];
    return in ? v : (T)0;
  };
  // header: sup.x, sup.y, sup.z (klo), sup.w (span), f0, f1, f2; paired
  // entries: force support, torque support, force, torque
  const int HO = A.ho;
  // Staging thread (ss, su) loads words su, su+16, ... of entry ss of a batch and
  // word su of its header.  The words' places in the padded record (0, a zero,
  // past its end) are formed once, 16 bits each, paired entries two to a
  // register, others kind 0 low and kind 1 high; so all loads of a batch are
  // issued together.  Formed per batch, with the header's words found among the
  // record's, the places took 43 registers, a quarter of the wavefronts: slit,
  // N = 16384, 256^2 x 96, forces and torques, 135 us; so, and with paired and
  // other entries in kernels of their own, 68.
  const int ss = threadIdx.x >> 4, su = threadIdx.x & 15;
  constexpr int NAT = PAIR ? (NPF + 1) / 2 : NPF;
  unsigned at[NAT];
#pragma unroll
  for (int k = 0; k < NAT; ++k) {
    auto place = [&](int off) {   // paired: force record, then torque record
      return off < A.pm ? padded(off, A.wx0, A.wy0, A.W0, 0)
                        : (off < A.pm + A.pd ? A.off1 + padded(off - A.pm, A.wx1, A.wy1, A.W1, 1) : 0);
    };
    if (PAIR)
      at[k] = place(su + 32 * k) | (unsigned)place(su + 32 * k + 16) << 16;
    else
      at[k] = (su + 16 * k < A.pm ? place(su + 16 * k) : 0) | (unsigned)place(A.pm + su + 16 * k) << 16;
    asm volatile("" : "+v"(at[k]));
  }
  constexpr int NH = PAIR ? 14 : 7;   // header words
  auto prefetch = [&](int qb, int nb, T (&v)[NPF], T& hd) {
    if (ss >= nb) return;
    const int ent = queue[qb + ss];
    const int p = ent >> 1, kind = ent & 1;
    const T* rec = (const T*)A.rec + (size_t)p * A.rs;
#pragma unroll
    for (int k = 0; k < NPF; ++k)
      v[k] = rec[PAIR ? at[PAIR ? k / 2 : 0] >> 16 * (k & 1) & 0xffff : at[PAIR ? 0 : k] >> (kind ? 16 : 0) & 0xffff];
    const bool second = PAIR ? su >= 4 : kind;   // the second kernel's support
    if (su < (PAIR ? 8 : 4)) {
      hd = (T)reinterpret_cast<const int*>((second ? A.sup1 : A.sup0) + p)[su & 3];
    } else if (su < NH) {
      const int c = su - (PAIR ? 8 : 4);
      hd = (T)((PAIR ? c >= 3 : kind) ? Tq : F)[3 * (size_t)p + (PAIR && c >= 3 ? c - 3 : c)];
    }
  };
  constexpr int QN = 2 * 256;   // queue capacity
  for (int c0 = 0; c0 < ncand; c0 += QN) {
    const int nq_entries = min(QN, ncand - c0);
    for (int i = threadIdx.x; i < nq_entries; i += blockDim.x) queue[i] = A.entries[e0 + c0 + i];
    __syncthreads();
    // ---- spread the queued entries in staged batches, one wavefront per entry ----
    T pf[NPF], ph = 0;
    prefetch(0, min(B, nq_entries), pf, ph);
    for (int qb = 0; qb < nq_entries; qb += B) {
      const int nb = min(B, nq_entries - qb);
      if (ss < nb) {
#pragma unroll
        for (int k = 0; k < NPF; ++k)
          if (su + 16 * k < HO) bst[ss * SLOT + su + 16 * k] = pf[k];
        if (su < NH) bst[ss * SLOT + HO + su] = ph;
      }
      __syncthreads();
      if (qb + B < nq_entries) prefetch(qb + B, min(B, nq_entries - qb - B), pf, ph);
      for (int si = wave; si < nb; si += nwaves) {
        const T* st = bst + si * SLOT;
        // the entry's header is the same for every lane: scalar registers
        int kind = __builtin_amdgcn_readfirstlane(queue[qb + si] & 1);
        const int bx = __builtin_amdgcn_readfirstlane((int)st[HO]);
        const int by = __builtin_amdgcn_readfirstlane((int)st[HO + 1]);
        int klo = __builtin_amdgcn_readfirstlane((int)st[HO + 2]);
        int span = __builtin_amdgcn_readfirstlane((int)st[HO + 3]);
        const int wx = kind ? A.wx1 : A.wx0, wy = kind ? A.wy1 : A.wy0;
        const int W = kind ? A.W1 : A.W0;
        const T* wxr = st;
        const T* wyr = st + wx;
        const T* dxr = wyr + wy;
        const T* dyr = dxr + wx;
        const T* zr = kind ? (dyr + wy) : (wyr + wy);   // z weights of rows klo + q
        T f0 = st[HO + 4], f1 = st[HO + 5], f2 = st[HO + 6];
        // paired entry: rows of the union of the force kernel's (klm, spm) and
        // the torque kernel's (kld, spd), torque t
        int om = 0, od = 0, spm = 0, spd = 0;
        T t0 = 0, t1 = 0, t2 = 0;
        const T* pd_w = st + A.pm;   // torque record: [wx][wy][dx][dy][z][dz]
        if (PAIR) {
          kind = 2;
          const int klm = klo;
          spm = span;
          const int kld = __builtin_amdgcn_readfirstlane((int)st[HO + 6]);
          spd = __builtin_amdgcn_readfirstlane((int)st[HO + 7]);
          if (spd > 0) {
            const int lo = (spm > 0) ? min(klm, kld) : kld;
            const int hi = (spm > 0) ? max(klm + spm, kld + spd) : kld + spd;
            klo = lo;
            span = hi - lo;
          }
          om = klo - klm;
          od = klo - kld;
          f0 = st[HO + 8]; f1 = st[HO + 9]; f2 = st[HO + 10];
          t0 = st[HO + 11]; t1 = st[HO + 12]; t2 = st[HO + 13];
        }
        // rows klo + q (+ a period when z is periodic) inside this chunk:
        // q in [qa, qb2)
        for (int szp = A.periodic_z ? -1 : 0; szp <= (A.periodic_z ? 1 : 0); ++szp) {
        const int kls = klo + szp * A.Nz;
        const int qa = max(0, Z0 - kls), qb2 = min(span, Z0 + nZ - kls);
        if (qb2 <= qa) continue;
#pragma unroll 1   // else nine copies of the point loops: 68 -> 107 us
        for (int sxp = -1; sxp <= 1; ++sxp) {
          int ix0, lx0;
          const int cx = clip_piece(bx, wx, X0, nX, A.Nx, sxp * A.Nx, &ix0, &lx0);
          if (!cx) continue;
#pragma unroll 1
          for (int syp = -1; syp <= 1; ++syp) {
            int iy0, ly0;
            const int cy = clip_piece(by, wy, Y0, nY, A.Ny, syp * A.Ny, &iy0, &ly0);
            if (!cy) continue;
            // lane -> one support column (x fastest); with at most 32 columns
            // the wave splits the rows into P phases
            const int L = cx * cy;
            const int P = (L <= 32) ? 64 / L : 1;
            for (int cb = 0; cb < L; cb += (P > 1) ? L : 64) {
              int phase = 0, col = cb + lane;
              if (P > 1) {
                phase = lane / L;
                col = lane - phase * L;
              }
              if (phase >= P || col >= L) continue;
              const int b = col / cx, a = col - b * cx;
              const int i = ix0 + a, j = iy0 + b;
              TA* dcol = acc + (kls - Z0) * PL + (ly0 + b) * RS + (lx0 + a);   // row kls + q at + q PL
              const int q1 = qb2;
              if (kind == 2) {
                // force (monopole) and torque curl at each point, one atomic
                // per component
                const T* wxd = pd_w;
                const T* wyd = wxd + wx;
                const T* dxd = wyd + wy;
                const T* dyd = dxd + wx;
                const T* zAd = dyd + wy;
                const T* zBd = zAd + A.W1;
                // with w = wm zm and g = (ax zA, ay zA, az zB) the point
                // receives w f + 1/2 g x t: per component
                //   P_c zm + Q_c zA + R_c zB  (R_2 = 0)
                // with the column's coefficients (scale included) formed once
                const T hs = (T)0.5 * sc;
                const T wm = wxr[i] * wyr[j] * sc;
                const T ax = dxd[i] * wyd[j] * hs, ay = wxd[i] * dyd[j] * hs, az = wxd[i] * wyd[j] * hs;
                const T P0 = wm * f0, P1 = wm * f1, P2 = wm * f2;
                const T Q0 = ay * t2, Q1 = -(ax * t2), Q2 = ax * t1 - ay * t0;
                const T R0 = -(az * t1), R1 = az * t0;
                for (int q = qa + phase; q < q1; q += P) {
                  const int qm = q + om, qd = q + od;
                  const T zm = zw(zr, qm, spm), zA = zw(zAd, qd, spd), zB = zw(zBd, qd, spd);
                  TA* d = dcol + q * PL;
                  add(d, zm * P0 + zA * Q0 + zB * R0);
                  add(d + vol, zm * P1 + zA * Q1 + zB * R1);
                  add(d + 2 * vol, zm * P2 + zA * Q2);
                }
              } else if (kind == 0) {
                const T wxy = wxr[i] * wyr[j] * sc;
                const T g0 = wxy * f0, g1 = wxy * f1, g2 = wxy * f2;
                int q = qa + phase;
                for (; q + 3 * P < q1; q += 4 * P) {
                  const T w0 = zr[q], w1 = zr[q + P], w2 = zr[q + 2 * P], w3 = zr[q + 3 * P];
                  TA* d0 = dcol + q * PL;
                  add(d0, (w0 * g0)); add(d0 + vol, (w0 * g1));
                  add(d0 + 2 * vol, (w0 * g2));
                  TA* d1 = d0 + P * PL;
                  add(d1, (w1 * g0)); add(d1 + vol, (w1 * g1));
                  add(d1 + 2 * vol, (w1 * g2));
                  TA* d2 = d1 + P * PL;
                  add(d2, (w2 * g0)); add(d2 + vol, (w2 * g1));
                  add(d2 + 2 * vol, (w2 * g2));
                  TA* d3 = d2 + P * PL;
                  add(d3, (w3 * g0)); add(d3 + vol, (w3 * g1));
                  add(d3 + 2 * vol, (w3 * g2));
                }
                for (; q < q1; q += P) {
                  const T w = zr[q];
                  TA* d = dcol + q * PL;
                  add(d, (w * g0)); add(d + vol, (w * g1));
                  add(d + 2 * vol, (w * g2));
                }
              } else {
                // 1/2 g x f with g = (ax zA, ay zA, az zB): per component
                // Q_c zA + R_c zB (R_2 = 0), coefficients formed once
                const T hs = (T)0.5 * sc;
                const T ax = dxr[i] * wyr[j] * hs, ay = wxr[i] * dyr[j] * hs, az = wxr[i] * wyr[j] * hs;
                const T Q0 = ay * f2, Q1 = -(ax * f2), Q2 = ax * f1 - ay * f0;
                const T R0 = -(az * f1), R1 = az * f0;
                int q = qa + phase;
                for (; q + P < q1; q += 2 * P) {
                  const T zA0 = zr[q], zB0 = zr[W + q], zA1 = zr[q + P], zB1 = zr[W + q + P];
                  {
                    TA* d = dcol + q * PL;
                    add(d, zA0 * Q0 + zB0 * R0);
                    add(d + vol, zA0 * Q1 + zB0 * R1);
                    add(d + 2 * vol, zA0 * Q2);
                  }
                  {
                    TA* d = dcol + (q + P) * PL;
                    add(d, zA1 * Q0 + zB1 * R0);
                    add(d + vol, zA1 * Q1 + zB1 * R1);
                    add(d + 2 * vol, zA1 * Q2);
                  }
                }
                for (; q < q1; q += P) {
                  const T zA = zr[q], zB = zr[W + q];
                  TA* d = dcol + q * PL;
                  add(d, zA * Q0 + zB * R0);
                  add(d + vol, zA * Q1 + zB * R1);
                  add(d + 2 * vol, zA * Q2);
                }
              }
            }
          }
        }
        }
      }
      __syncthreads();   // the batch's slots and the queue are free again
    }
  }
  // one write per grid element of the tile: thread -> fixed x, rows (z, y)
  // in steps of blockDim / TX
  {
    const int ix = threadIdx.x % TX, rstep = blockDim.x / TX;
    const int nrow = nZ * TY;
    if (ix < nX)
      for (int c = 0; c < 3; ++c) {
        T* gc = grid + ((size_t)c * A.Nz + Z0) * A.Ny * A.Nx + (size_t)Y0 * A.Nx + X0 + ix;
        const TA* ac = acc + c * vol + ix;
        const float isc = scl[1];
        for (int row = threadIdx.x / TX; row < nrow; row += rstep) {
          const int kz = row / TY, jy = row % TY;
          if (jy < nY) gc[((size_t)kz * A.Ny + jy) * A.Nx] = (float)ac[kz * PL + jy * RS] * isc;
        }
      }
  }
}


}  // namespace

size_t fx_lds_bytes(int ZC, int words)
{
  return (size_t)3 * ZC * (FX_TY * (FX_TX + 1) + 1) * 4 + (size_t)FX_BATCH * 16 * words * 4 + 2 * 256 * sizeof(int) +
         4 * sizeof(float);
}

void launch_fx_lists(const FxArgs& A, hipStream_t s)
{
  const int ncells = A.ntx * A.nty * A.nch, ne = A.N * A.nkind;
  hipLaunchKernelGGL(k_fx_zero, dim3((ncells + 255) / 256), dim3(256), 0, s, A.counts, ncells);
  if (ne > 0) hipLaunchKernelGGL(k_fx_cells<false>, dim3((ne + 255) / 256), dim3(256), 0, s, A);
  hipLaunchKernelGGL(k_fx_scan, dim3(1), dim3(1024), 0, s, A.counts, A.start, ncells);
  if (ne > 0) hipLaunchKernelGGL(k_fx_cells<true>, dim3((ne + 255) / 256), dim3(256), 0, s, A);
}

void launch_spread_fx(const FxArgs& A, int words, const double* F, const double* Tq, hipStream_t s)
{
  const int ncells = A.ntx * A.nty * A.nch;
  hipLaunchKernelGGL(k_fx_absmax, dim3(FX_AMAX_BLOCKS), dim3(256), 0, s, F, Tq, 3 * A.N, const_cast<FxStats*>(A.stats));
  const size_t lds = fx_lds_bytes(A.ZC, words);
  const dim3 grid(ncells), block(256);
  switch (words) {
#define FX_CASE(W)                                                                                 \
  case W:                                                                                          \
    if (A.pair) hipLaunchKernelGGL((k_spread_fx<W, true>), grid, block, lds, s, A, F, Tq);         \
    else hipLaunchKernelGGL((k_spread_fx<W, false>), grid, block, lds, s, A, F, Tq);               \
    break;
    FX_CASE(8) FX_CASE(10) FX_CASE(12) FX_CASE(16) FX_CASE(20) FX_CASE(24) FX_CASE(32)
#undef FX_CASE
    default: break;   // staged_words gives no other
  }
}

}  // namespace dps
