// dps_spread.hip -- spreading of forces and torques onto the grid, and the
// per-tile particle lists it reads.
//
//  k_scan_counts   exclusive scans of the list and sort counts that k_stencil
//                  took (one workgroup each), which also clear them for the
//                  next position update and hand the range flag to the host
//  k_list_scatter  particles into the lists of the tiles they reach and into
//                  the tile order that interpolation walks
//  k_list_sort     each tile's list in particle order
//  k_spread        forces + torque curl -> grid as matrix products, one write
//                  per grid element (SpreadInterp.cpp:302-448 +
//                  BoundaryConditions.h:22-361 + SpreadInterpWrapper.cpp:66-107)
#include <hip/hip_runtime.h>
#include <algorithm>
#include "dps_core.h"
#include "dps_internal.h"
#include "dps_mma.h"

namespace dps {

namespace {

constexpr int SCAN_T = 1024;

// exclusive scan of the counters, tile by tile and copy by copy of a tile, into
// cursor (same layout) and, per tile, start[0..ntiles] (either may be null);
// counters cleared; one workgroup, each thread a contiguous run
__device__ void scan_block(int* counts, int* start, int* cursor, int ntiles, int nc)
{
  __shared__ int part[SCAN_T / 64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, n = ntiles * nc, sh = __ffs(nc) - 1;
  const int per = (n + SCAN_T - 1) / SCAN_T;
  const int b = min(n, t * per), e = min(n, b + per);
  auto at = [&](int i) { return (i & (nc - 1)) * ntiles + (i >> sh); };
  int s = 0;
  for (int i = b; i < e; ++i) s += counts[at(i)];
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
    const int a = at(i), c = counts[a];
    if (start && (i & (nc - 1)) == 0) start[i >> sh] = run;
    cursor[a] = run;
    counts[a] = 0;
    run += c;
  }
  if (start && t == SCAN_T - 1) start[ntiles] = run;
}

__global__ void __launch_bounds__(SCAN_T) k_scan_counts(ListArgs A)
{
  if (blockIdx.x == 0) {
    scan_block(A.counts, A.start, A.cursor, A.ntiles, A.nc);
  } else {
    scan_block(A.kcounts, nullptr, A.kstart, A.ntiles, A.nc);
    if (threadIdx.x == 0 && A.err_host) {
      // a set of positions: its range flag to the host, both flags cleared
      *A.err_host = A.err[1];
      A.err[0] = 0;
      A.err[1] = 0;
    }
  }
}

constexpr int SCATTER_L = 4;

// Four lanes per particle, over the two to six tiles it meets.  One list by tile
// instead of one per (tile, z chunk) cell and pass, counted in k_stencil: with
// the sort below, locating 3,000 particles with torques took 155 us in 16
// launches and takes 26 in 4 (bottom wall, 160^2 x 57, one step 269 -> 121 us).
__global__ void __launch_bounds__(256) k_list_scatter(ListArgs A)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x, p = t / SCATTER_L, sl = t % SCATTER_L;
  if (p >= A.N) return;
  if (sl == 0) A.order[A.kstart[A.key[p]] + A.rank[p]] = p;
  const TileRuns r = particle_runs(A, A.sup0[p], A.sup1 ? A.sup1[p] : A.sup0[p]);
  for_tiles(A, r, sl, SCATTER_L, [&](int tile) {
    const int at = atomicAdd(&A.cursor[(p & (A.nc - 1)) * A.ntiles + tile], 1);
    if (at < A.cap) A.unsorted[at] = p;   // within the capacity (it bounds every support)
  });
}

constexpr int SORT_COUNT = 512, SORT_WORDS = 4096;

// a list of any length, through a bit per particle: 32 SORT_WORDS of them at a time
__device__ __forceinline__ void sort_bits(int* v, const int* src, int* dst, int n, int N)
{
  __shared__ int part[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int done = 0;
  for (int p0 = 0; p0 < N; p0 += 32 * SORT_WORDS) {
    const int words = min(SORT_WORDS, (N - p0 + 31) / 32), per = (words + 255) / 256;
    for (int i = t; i < words; i += 256) v[i] = 0;
    __syncthreads();
    for (int i = t; i < n; i += 256) {
      const int p = src[i] - p0;
      if (p >= 0 && p < 32 * SORT_WORDS) atomicOr(&v[p >> 5], 1 << (p & 31));
    }
    __syncthreads();
    const int b = min(words, t * per), e = min(words, b + per);
    int s = 0;
    for (int i = b; i < e; ++i) s += __popc(v[i]);
    int inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(inc, o, 64);
      if (lane >= o) inc += u;
    }
    if (lane == 63) part[wave] = inc;
    __syncthreads();
    int at = done + inc - s;
    for (int w = 0; w < 4; ++w) {
      at += w < wave ? part[w] : 0;
      done += part[w];
    }
    for (int i = b; i < e; ++i)
      for (unsigned m = v[i]; m; m &= m - 1) dst[at++] = p0 + 32 * i + __ffs(m) - 1;
    __syncthreads();   // v and part are free again
  }
}

// One workgroup per tile: the scatter above fills lists in the order its
// atomics happen to run; sums over a list in particle order are the same
// from call to call.  Particle indices are distinct: up to SORT_COUNT entries
// count the smaller ones, longer lists set a bit per particle.  An update of 600 /
// 1000 / 3000 / 9000 / 60000 particles under one tile takes 28 / 34 / 40 / 87 / 466
// us; with counting up to 1024 and a bitonic network in global memory beyond 42 /
// 71 / 184 / 644 / 5046, with that network in LDS up to 4096 39 / 43 / 99 / - / -.
__global__ void __launch_bounds__(256) k_list_sort(ListArgs A)
{
  __shared__ int v[SORT_WORDS];
  const int e0 = A.start[blockIdx.x], n = min(A.start[blockIdx.x + 1], A.cap) - e0;
  if (n <= 0) return;
  const int* src = A.unsorted + e0;
  int* dst = A.entries + e0;
  if (n > SORT_COUNT) {
    sort_bits(v, src, dst, n, A.N);
    return;
  }
  for (int i = threadIdx.x; i < n; i += 256) v[i] = src[i];
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 256) {
    const int x = v[i];
    int r = 0;
    for (int j = 0; j < n; ++j) r += v[j] < x;
    dst[r] = x;
  }
}

// 16 bytes of a grid row: rows of any length start at any element, so the
// vector is aligned to its element only
template <class T> struct Row4;
template <> struct Row4<float> { typedef float t __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct Row4<double> { typedef double t __attribute__((ext_vector_type(2), aligned(8))); };

// d modulo n for d in [-n, 2 n)
__device__ __forceinline__ int wrap1(int d, int n)
{
  d += (d < 0) ? n : 0;
  return d - ((d >= n) ? n : 0);
}

// min(max(i, -1), n) for n >= -1
__device__ __forceinline__ int clamp1(int i, int n)
{
  int r;
  asm("v_med3_i32 %0, %1, -1, %2" : "=v"(r) : "v"(i), "v"(n));
  return r;
}

// element i >= 0 of an array, by a 32-bit byte offset from its base
template <class T>
__device__ __forceinline__ T at32(const T* base, int i)
{
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (unsigned)(i * (int)sizeof(T)));
}

// Queued particles of a spreading wavefront: offsets of its columns and levels
// in the supports of both kernels, the particle and the z tiles it reaches
// (bits), and its force and half its torque: [f0 f1 f2 0 h0 h1 h2], in FP32
// followed by [-h0 -h1 -h2].  Steps of PAD particles may run past the last
// one: zeros stand there.
template <class T, bool TERMS> struct SpreadQueue {
  static constexpr int CAP = 64, PAD = 8;
  static constexpr int NF = !TERMS ? 3 : (sizeof(T) == 4 ? 10 : 7);
  int4 off[TERMS ? 2 : 1][CAP + PAD];
  int2 who[CAP + PAD];
  T f[CAP + PAD][NF];
};

// one z tile of a workgroup's columns on its way out, rows padded against
// bank conflicts
template <class T> struct SpreadOut {
  static constexpr int RS = SP_TX + 16 / (int)sizeof(T);
  T v[3][16][SP_TY][RS];
};

// Spreading as matrix products.  A wavefront owns 4 x 4 columns (16 rows M of
// the products) and NT tiles of 16 z levels (their columns N), three
// components each, accumulated in registers; the inner dimension runs over
// the terms of the particles that reach it:
//   TERMS   a particle's four terms per step: its force through the force
//           kernel, and its torque through the kernel's derivatives along x,
//           y and z (the curl, 1/2 g x t with g the kernel's gradient)
//   else    the forces of four particles per step.
// A lane forms one element of each operand: the product of an x and a y
// weight of its term, and a z weight times the term's force or torque
// coefficient per component.  Weights off the support are the zeros that pad
// the records (RecLayout), reached by clamping the index; the z weights are
// dense over the rows klo .. klo + span - 1 (folded images merged by the
// stencil).
//
// The wavefront finds its particles by testing its tile's list, 64 at a time
// (the next 64 already loading), and queues them in LDS; the loads of UN steps
// are issued together.  No atomics: sums run in list order (particle order),
// and each grid element is written once, through LDS so that the workgroup's
// eight wavefronts fill whole rows of their 32 columns.  WRAP: columns or
// levels that wrap one by one (periodic z, or a period of four columns, which
// a support may leave and enter again within one wavefront's).  Bound by vector
// instructions (addresses and operand elements; 30 per particle and z tile).
// With the particles' supports and forces re-read and masked at every step and
// direct 16-byte stores (4.7M write requests instead of 1.2M): slit N = 16384,
// 256^2 x 96, mixed 55 -> 37 us, FP64 108 -> 69; monolayer N = 262144, 1024^2 x 48
// 820 -> 397; bottom wall N = 2048, 128^2 x 64, forces 13 -> 10.  Before that, int32
// fixed point accumulated with LDS atomics took 92, 146, 1270 and 27.
template <class T, class Tin, bool TERMS, int NT, bool WRAP>
__global__ void __launch_bounds__(64 * SP_WAVES) k_spread(SpreadArgs A, const Tin* __restrict__ F,
                                                          const Tin* __restrict__ Tq)
{
  typedef SpreadQueue<T, TERMS> Queue;
  typedef SpreadOut<T> Out;
  // two steps' loads together, or four where three z tiles leave few
  // wavefronts per SIMD (monolayer 448 -> 397 us; with two z tiles 486 -> 519)
  constexpr int UN = TERMS && NT == 3 && sizeof(T) == 4 ? 4 : 2;
  constexpr int PS = TERMS ? 1 : 4;   // particles per step
  static_assert(UN * PS <= Queue::PAD, "a step's particles fit the queue's padding");
  constexpr size_t QB = sizeof(Queue) * SP_WAVES, OB = sizeof(Out);
  __shared__ __attribute__((aligned(16))) unsigned char smem[QB > OB ? QB : OB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Queue& Q = reinterpret_cast<Queue*>(smem)[wave];
  const int blk = xcd_group(blockIdx.x, gridDim.x);
  const int zg = blk % A.nzg, tile = blk / A.nzg;
  const int ty = tile / A.ntx, tx = tile - ty * A.ntx;
  const int X0 = tx * SP_TX, Y0 = ty * SP_TY;
  const int xs = X0 + 4 * (wave % (SP_TX / 4)), ys = Y0 + 4 * (wave / (SP_TX / 4));
  const int Z0 = zg * 16 * NT, Z1 = min(A.Nz, Z0 + 16 * NT);
  const int m = lane & 15, k = lane >> 4;
  // the output register index runs along x in both precisions
  const int ax = sizeof(T) == 4 ? (m & 3) : (m >> 2), ay = sizeof(T) == 4 ? (m >> 2) : (m & 3);
  typedef typename Mma<T>::acc acc_t;
  acc_t acc[NT][3];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[t][c] = acc_t{0, 0, 0, 0};
  // this lane's term: support size, record offsets of its x, y and z weights,
  // and per component the queued force or torque value
  const bool dip = TERMS && k > 0;
  const int wx = dip ? A.wx1 : A.wx0, wy = dip ? A.wy1 : A.wy0, W = dip ? A.W1 : A.W0;
  const RecLayout R = rec_layout(wx, wy, W, dip, 1);
  const int off = dip ? A.off1 : 0;
  const int ox = off + (k == 1 && dip ? R.dx : R.x);
  const int oy = off + (k == 2 && dip ? R.dy : R.y);
  const int oz = off + (k == 3 && dip ? R.dz : R.z);
  // gx: (0, -h2, h1), gy: (h2, 0, -h0), gz: (-h1, h0, 0), h = t / 2
  int fi0 = 0, fi1 = 1, fi2 = 2;
  if (dip) {
    constexpr int NEG = sizeof(T) == 4 ? 3 : 0;   // in FP64 the signs below
    if (k == 1) { fi0 = 3; fi1 = 6 + NEG; fi2 = 5; }
    else if (k == 2) { fi0 = 6; fi1 = 3; fi2 = 4 + NEG; }
    else { fi0 = 5 + NEG; fi1 = 4; fi2 = 3; }
  }
  const T sg0 = (k == 3) ? (T)-1 : (T)1, sg1 = (k == 1) ? (T)-1 : (T)1, sg2 = (k == 2) ? (T)-1 : (T)1;
  // offsets of these columns and levels in a support, and the z tiles of it
  // that it reaches here (w: bits).  Without WRAP the columns xs .. xs + 3 meet
  // a support in one run, so that one offset, -3 .. w - 1 where they meet,
  // does for all four; the same for y.
  auto reach = [&](int4 s, int w_x, int w_y) {
    int4 r = make_int4(wrap1(xs - s.x, A.Nx), wrap1(ys - s.y, A.Ny), Z0 - s.z, 0);
    const bool wrx = WRAP && A.Nx == 4, wry = WRAP && A.Ny == 4;
    r.x -= r.x > A.Nx - 4 && !wrx ? A.Nx : 0;
    r.y -= r.y > A.Ny - 4 && !wry ? A.Ny : 0;
    if ((r.x < w_x || wrx) && (r.y < w_y || wry)) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int za = Z0 + 16 * t;
        if (za >= Z1) break;
        bool in;
        if (WRAP && A.periodic_z) {
          const int d = wrap1(za - s.z, A.Nz);
          in = d < s.w || d > A.Nz - 16;
        } else {
          in = s.z < za + 16 && s.z + s.w > za;
        }
        r.w |= (in && s.w > 0) ? 1 << t : 0;
      }
    }
    return r;
  };
  const T* const rec = reinterpret_cast<const T*>(A.rec);
  const bool live = xs < A.Nx && ys < A.Ny;
  const int e0 = A.lstart[tile], e1 = live ? min(A.lstart[tile + 1], A.lcap) : e0;
  int p = 0;
  int4 s0 = make_int4(0, 0, 0, 0), s1 = s0;
  auto fetch = [&](int e) {
    if (e < e1) {
      p = A.lentries[e];
      s0 = A.sup0[p];
      if (TERMS) s1 = A.sup1[p];
    }
  };
  fetch(e0 + lane);
  for (int base = e0; base < e1; base += 64) {
    // ---- queue the particles that reach these columns and levels ----
    int zm = 0;
    int4 r0 = make_int4(0, 0, 0, 0), r1 = r0;
    if (base + lane < e1) {
      r0 = reach(s0, A.wx0, A.wy0);
      zm = r0.w;
      if (TERMS) {
        r1 = reach(s1, A.wx1, A.wy1);
        zm |= r1.w;
      }
    }
    const unsigned long long hit = __ballot(zm != 0);
    const int nq = (int)__popcll(hit);
    if (zm) {
      const int at = __popcll(hit & ((1ull << lane) - 1));
      Q.off[0][at] = r0;
      if (TERMS) Q.off[TERMS ? 1 : 0][at] = r1;
      Q.who[at] = make_int2(p, zm);
      const Tin* f = F + 3 * (size_t)p;
      T* q = Q.f[at];
      q[0] = (T)f[0];
      q[1] = (T)f[1];
      q[2] = (T)f[2];
      if constexpr (TERMS) {
        const Tin* t = Tq + 3 * (size_t)p;
        const T h0 = (T)t[0] * (T)0.5, h1 = (T)t[1] * (T)0.5, h2 = (T)t[2] * (T)0.5;
        q[3] = (T)0;
        q[4] = h0; q[5] = h1; q[6] = h2;
        if constexpr (sizeof(T) == 4) { q[7] = -h0; q[8] = -h1; q[9] = -h2; }
      }
    }
    if (lane < Queue::PAD) {
      Q.off[0][nq + lane] = make_int4(0, 0, 0, 0);
      if (TERMS) Q.off[TERMS ? 1 : 0][nq + lane] = make_int4(0, 0, 0, 0);
      Q.who[nq + lane] = make_int2(0, 0);
#pragma unroll
      for (int c = 0; c < Queue::NF; ++c) Q.f[nq + lane][c] = (T)0;
    }
    __builtin_amdgcn_wave_barrier();
    fetch(base + 64 + lane);
    // ---- the products, UN steps' loads together ----
    for (int h = 0; h < nq; h += UN * PS) {
      T av[UN], bv[UN][NT], c0[UN], c1[UN], c2[UN];
      int zms[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int at = h + u * PS + (TERMS ? 0 : k);
        const int4 s = Q.off[dip ? 1 : 0][at];
        const int2 who = Q.who[at];
        int zq = who.y;
        const T* r;
        if (TERMS) {
          r = rec + (size_t)__builtin_amdgcn_readfirstlane(who.x) * A.rs;
        } else {
          r = rec + (size_t)who.x * A.rs;
          zq |= __shfl_xor(zq, 16, 64);
          zq |= __shfl_xor(zq, 32, 64);
        }
        zms[u] = __builtin_amdgcn_readfirstlane(zq);
        int i = s.x + ax, j = s.y + ay;
        if (WRAP && A.Nx == 4) i = wrap1(i, 4);
        if (WRAP && A.Ny == 4) j = wrap1(j, 4);
        // one past either end of a part is a zero weight
        av[u] = at32(r, ox + clamp1(i, wx)) * at32(r, oy + clamp1(j, wy));
        const T* f = Q.f[at];
        c0[u] = f[fi0];
        c1[u] = f[fi1];
        c2[u] = f[fi2];
        if (dip && sizeof(T) == 8) {
          c0[u] *= sg0;
          c1[u] *= sg1;
          c2[u] *= sg2;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          bv[u][t] = (T)0;
          if (zms[u] >> t & 1) {
            int q = s.z + 16 * t + m;
            if (WRAP && A.periodic_z) q = wrap1(q, A.Nz);
            bv[u][t] = at32(r, oz + clamp1(q, W));
          }
        }
      }
#pragma unroll
      for (int u = 0; u < UN; ++u)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if (zms[u] >> t & 1) {
            acc[t][0] = Mma<T>::step(av[u], bv[u][t] * c0[u], acc[t][0]);
            acc[t][1] = Mma<T>::step(av[u], bv[u][t] * c1[u], acc[t][1]);
            acc[t][2] = Mma<T>::step(av[u], bv[u][t] * c2[u], acc[t][2]);
          }
    }
    __builtin_amdgcn_wave_barrier();
  }
  // ---- write out a z tile at a time: lane (z level m, row k) has four x
  // values; rows of 32 columns leave as 16-byte pieces, neighbours in order ----
  T* __restrict__ grid = reinterpret_cast<T*>(A.grid);
  Out& O = *reinterpret_cast<Out*>(smem);
  constexpr int VL = 16 / sizeof(T);   // values of a piece
  typedef typename Row4<T>::t piece;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int zt = Z0 + 16 * t;
    if (zt >= Z1) break;
    __syncthreads();   // the queues, or the tile before, are done with
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v) O.v[c][m][ys - Y0 + k][xs - X0 + v] = acc[t][c][v];
    __syncthreads();
    constexpr int PR = SP_TX / VL;   // pieces per row
    for (int i = threadIdx.x; i < 3 * 16 * SP_TY * PR; i += 64 * SP_WAVES) {
      const int row = i / PR, xo = (i % PR) * VL;
      const int y = row % SP_TY, cz = row / SP_TY, z = cz & 15, c = cz >> 4;
      if (zt + z >= Z1 || Y0 + y >= A.Ny || X0 + xo >= A.Nx) continue;
      const T* o = &O.v[c][z][y][xo];
      T* g = grid + (((size_t)c * A.Nz + zt + z) * A.Ny + Y0 + y) * A.Nx + X0 + xo;
      if (X0 + xo + VL <= A.Nx) {
        *reinterpret_cast<piece*>(g) = *reinterpret_cast<const piece*>(o);
      } else {
#pragma unroll
        for (int v = 0; v < VL; ++v)
          if (X0 + xo + v < A.Nx) g[v] = o[v];
      }
    }
  }
}

}  // namespace

void launch_lists(const ListArgs& A, hipStream_t s)
{
  hipLaunchKernelGGL(k_scan_counts, dim3(2), dim3(SCAN_T), 0, s, A);
  if (A.N == 0) return;
  hipLaunchKernelGGL(k_list_scatter, dim3((A.N + 256 / SCATTER_L - 1) / (256 / SCATTER_L)), dim3(256), 0, s, A);
  hipLaunchKernelGGL(k_list_sort, dim3(A.ntiles), dim3(256), 0, s, A);
}

// Three z tiles per wavefront on FP32 grids, two in FP64 (registers), as long
// as that leaves a little over three wavefronts per SIMD (1024 of them): the
// x-y operand is formed and the list tested once for all.  Fewer tiles where they make the
// same number of groups.  1 / 2 / 3 tiles: monolayer 1024^2 x 48 475 / 486 / 397 us, slit
// 256^2 x 96 42 / 37 / 37, bottom wall 160^2 x 57 15.8 / 14.4 / 17.3, bottom wall
// 128^2 x 64 10.3 / 11.0 / 12.0, periodic 96^3 19.7 / 20.6 / 25.3; FP64 slit 78 / 69 / 74.
int spread_tiles(int Nx, int Ny, int Nz, bool fp32)
{
  const long waves = (long)((Nx + 3) / 4) * ((Ny + 3) / 4);
  const int zt = (Nz + 15) / 16;
  int nt = spread_max_tiles(fp32);
  while (nt > 1 && (waves * ((zt + nt - 1) / nt) < 3200 || (zt + nt - 2) / (nt - 1) == (zt + nt - 1) / nt)) --nt;
  return nt;
}

template <class T, class Tin>
void launch_spread(const SpreadArgs& A0, const void* F, const void* Tq, hipStream_t s)
{
  SpreadArgs A = A0;
  A.nzg = (A.Nz + 16 * A.nt - 1) / (16 * A.nt);
  const dim3 grid(A.ntx * A.nty * A.nzg), block(64 * SP_WAVES);
  const Tin *f = (const Tin*)F, *t = (const Tin*)Tq;
  const bool wrap = A.periodic_z || A.Nx == 4 || A.Ny == 4;
#define SPREAD_CASE(NT)                                                                                 \
  case NT:                                                                                              \
    if (t && wrap) hipLaunchKernelGGL((k_spread<T, Tin, true, NT, true>), grid, block, 0, s, A, f, t);  \
    else if (t) hipLaunchKernelGGL((k_spread<T, Tin, true, NT, false>), grid, block, 0, s, A, f, t);    \
    else if (wrap) hipLaunchKernelGGL((k_spread<T, Tin, false, NT, true>), grid, block, 0, s, A, f, t); \
    else hipLaunchKernelGGL((k_spread<T, Tin, false, NT, false>), grid, block, 0, s, A, f, t);          \
    break;
  switch (A.nt) {
    SPREAD_CASE(1) SPREAD_CASE(2)
    default:   // three tiles: FP32 grids only
      if constexpr (sizeof(T) == 4) switch (A.nt) { SPREAD_CASE(3) default: break; }
  }
#undef SPREAD_CASE
}

template void launch_spread<float, float>(const SpreadArgs&, const void*, const void*, hipStream_t);
template void launch_spread<double, float>(const SpreadArgs&, const void*, const void*, hipStream_t);
template void launch_spread<double, double>(const SpreadArgs&, const void*, const void*, hipStream_t);

}  // namespace dps
