// dps_internal.h -- kernel argument blocks and launchers shared by the host
// orchestration (dps_api.hip) and the kernels (dps_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "dps_core.h"

#define DPS_MAX_W 32          // largest x/y support (points) a stencil may have
// spreading tile: SP_TX x SP_TY x-y cells, one wavefront per 4 x 4 of them
#define SP_TX 32
#define SP_TY 4
#define SP_WAVES (SP_TX * SP_TY / 16)

namespace dps {

template <class T> struct C2;
template <> struct C2<float> { typedef float2 t; };
template <> struct C2<double> { typedef double2 t; };

// wavenumber of FFT index i on n points over length L (Nyquist positive)
__host__ __device__ inline double kvec(int i, int n, double L)
{
  const int nn = (i <= n / 2) ? i : i - n;
  return 2 * M_PI * (double)nn / L;
}

// Block index -> work group index such that consecutive groups run on the
// same XCD (the 8 XCDs receive blocks round robin and each has its own L2).
__device__ __forceinline__ int xcd_group(int b, int nb)
{
  const int x = b & 7, q = nb >> 3, r = nb & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// Per-tile particle lists of the spreading and the tile order of the
// interpolation, rebuilt whenever positions change: k_stencil counts, then
// scans, scatter and sort (launch_lists).  A particle is listed in every tile
// that its force or torque support reaches.
struct ListArgs {
  int N, Nx, Ny, ntx, nty, ntiles;
  int wx0, wy0, wx1, wy1;      // supports of the force and torque kernels (equal without torques)
  const int4 *sup0, *sup1;     // sup1 null without torques
  int nc;                         // copies of the counters: particle p counts in copy p mod nc
  int *counts, *start, *cursor;   // [nc][ntiles], [ntiles + 1], [nc][ntiles]; counts are zero between builds
  int *unsorted, *entries;        // [cap] list entries, as scattered and in particle order
  int cap;
  int *key, *rank, *kcounts, *kstart, *order;   // tile order: [N], [N], [nc][ntiles], [nc][ntiles], [N]
  int* err;        // [2] range flags: of updates, of the set of positions under way
  int* err_host;   // where a set of positions reports its flag (null: an update)
};
void launch_lists(const ListArgs& A, hipStream_t s);
// Copies of the list counters, a power of two: additions to one counter (and to
// its cache line) from all over the chip queue up behind each other.  With one
// copy k_stencil + k_list_scatter + k_scan_counts took 32 + 12 + 5 us for 8192
// particles over 288 tiles, with 4 copies 23 + 5 + 6, with 16 the scan grows to
// 9; above 1024 tiles the counters are apart by themselves.
inline int list_copies(int ntiles) { return ntiles > 2048 ? 1 : (ntiles > 1024 ? 2 : 4); }
// upper bound of the tiles one support (points) reaches; the union of two
// kernels' supports is at most one point longer than the longer one
inline int list_tiles_bound(int wx, int wy)
{
  return ((wx + SP_TX) / SP_TX + 2) * ((wy + SP_TY) / SP_TY + 2);
}

// unwrapped columns under either of a particle's supports
struct TileRuns {
  int x, nx, y, ny;
};
__device__ __forceinline__ TileRuns particle_runs(const ListArgs& A, int4 s0, int4 s1)
{
  TileRuns r;
  r.x = min(s0.x, s1.x);
  r.nx = max(s0.x + A.wx0, s1.x + A.wx1) - r.x;
  r.y = min(s0.y, s1.y);
  r.ny = max(s0.y + A.wy0, s1.y + A.wy1) - r.y;
  return r;
}

// the tiles of size T that a periodic run of w < n of n points meets, each
// once: only the last can be the first again (a run across the end of the
// period back into the tile it starts in)
template <class Fn>
__device__ __forceinline__ void for_run_tiles(int b, int w, int n, int T, Fn&& f)
{
  int at = b % n;
  at += at < 0 ? n : 0;
  const int first = at / T;
  bool more = false;
  while (w > 0) {
    const int t = at / T;
    if (!more || t != first) f(t);
    more = true;
    const int step = min(T * (t + 1), n) - at;
    w -= step;
    at += step;
    at = at >= n ? 0 : at;
  }
}

// the same tiles by number, for the lanes of a group: k = 0 .. n - 1
struct TileSpan {
  int first, n, nt;
  __device__ __forceinline__ int tile(int k) const
  {
    const int t = first + k;
    return t >= nt ? t - nt : t;
  }
};
__device__ __forceinline__ TileSpan tile_span(int b, int w, int n, int T)
{
  int at = b % n;
  at += at < 0 ? n : 0;
  const int end = at + w - 1;   // last point, n or more past the end of the period
  TileSpan r;
  r.first = at / T;
  r.nt = (n + T - 1) / T;
  r.n = end < n ? end / T - r.first + 1 : r.nt - r.first + min((end - n) / T + 1, r.first);
  return r;
}

// f(tile) for the list tiles under a particle's supports, over L lanes (this
// one is sl)
template <class Fn>
__device__ __forceinline__ void for_tiles(const ListArgs& A, TileRuns r, int sl, int L, Fn&& f)
{
  const TileSpan sx = tile_span(r.x, r.nx, A.Nx, SP_TX), sy = tile_span(r.y, r.ny, A.Ny, SP_TY);
  for (int t = sl; t < sx.n * sy.n; t += L) {
    const int ky = t / sx.n;
    f(sy.tile(ky) * A.ntx + sx.tile(t - ky * sx.n));
  }
}

// Offsets of the parts of one kernel's weight record: x, y [, d/dx, d/dy], z
// [, d/dz] spreading weights, then the z [, d/dz] interpolation weights.  With
// pad = 1 a zero stands before, between and after the spreading parts, so that
// an index clamped to one past either end of a part reads a zero weight.
struct RecLayout {
  int x, y, dx, dy, z, dz, zi, dzi, words;
};
__host__ __device__ inline RecLayout rec_layout(int wx, int wy, int W, int deriv, int pad)
{
  RecLayout r;
  r.x = pad;
  r.y = r.x + wx + pad;
  r.dx = r.y + wy + pad;
  r.dy = r.dx + wx + pad;
  r.z = deriv ? r.dy + wy + pad : r.dx;
  r.dz = r.z + W + pad;
  r.zi = deriv ? r.dz + W + pad : r.dz;
  r.dzi = r.zi + W;
  r.words = deriv ? r.dzi + W : r.dzi;
  return r;
}

struct StencilArgs {
  int N;
  double xmin, ymin, zmin;
  double Lx, Ly, Lz, hx, hy;
  int Nx, Ny;
  int has_dip;
  KernelDesc km, kd;
  const double *zext_m, *zw_m, *zext_d, *zw_d;
  double* pos;     // 3N wrapped/shifted positions
  int* err;        // set to 1 if a particle is outside [0, Lz]
  int4 *sup_m, *sup_d;
  void *rec_m, *rec_d;   // per-particle weight records (grid precision)
  int rs_m, rs_d;        // record strides (elements)
  int pad;               // records in the padded layout
  const int* kt_m;       // z fold tables, to record the interior rows reached
  const int* kt_d;
  const double *fA_m, *fA_d, *fB_d;
  int periodic_z;        // triply periodic: uniform z nodes k hz, wrapped like x and y
  double hz;
  int dip_regular;       // the torque kernel is a plain ES kernel: records in the monopole layout
  int first_kind;        // 1: the second (kd) record set only (e.g. force-kernel derivative records)
  int move;              // the input positions take a step (by vel if given) and are rewritten in place
  const void* vel;       // 3N velocities of the positions' type, or null
  double dt;
  ListArgs L;            // counts null: no lists (records only)
};

struct SpreadArgs {
  int Nx, Ny, Nz;
  int periodic_z;   // rows of a support wrap modulo Nz
  int ntx, nty;
  int nt;           // 16-level z tiles per wavefront (1..spread_max_tiles)
  int nzg;          // z groups of nt tiles (set by the launcher)
  // particles of every tile (ty ntx + tx), in particle order:
  // lentries[lstart[tile] .. lstart[tile + 1])
  const int *lstart, *lentries;
  int lcap;         // capacity of lentries
  // padded records (stride rs): kernel 0's plain part at offset 0 and, in
  // passes with torques, kernel 1's derivative part at off1
  const int4 *sup0, *sup1;
  const void* rec;
  int rs, off1, wx0, wy0, W0, wx1, wy1, W1;
  void* grid;   // [3][Nz][Ny][Nx] grid precision
};

// Fixed-point spreading of FP64 arrays onto FP32 grids (dps_spread_fx.hip):
// cells of FX_TX x FX_TY columns and ZC rows
#define FX_TX 16
#define FX_TY 8
#define FX_BATCH 16          // entries staged together
#define FX_AMAX_BLOCKS 64
// passes, each with cell lists of its own: forces; forces and torques
// (derivative kernels); torques as a vector field (regular kernel)
enum { FX_FORCES, FX_TORQUES, FX_REGULAR };
// A cell's unit is coarse where the bound on its sums exceeds FX_COARSE times the
// root mean square of an entry's bound: the spread grid is then 7e-6 off (in
// proportion: 2.8e-5 at 6200, 1500 particles under one tile)
#define FX_COARSE 1536.0f
struct FxStats {
  float fm, tm;    // largest |F|, |T|
  double f2, t2;   // sums of squares
  int nf, nt;      // values that are not zero
};
struct FxArgs {
  int N, Nx, Ny, Nz, periodic_z;
  int ZC, ntx, nty, nch;
  // entries 2 p + kind: one per particle (pair: force and torque together,
  // the kernels share their x/y supports) or one per kernel (nkind = 2)
  int nkind, pair;
  int wx0, wy0, W0, wx1, wy1, W1;
  const int4 *sup0, *sup1;
  const void* rec;             // padded records, kernel 1's part at off1
  int rs, off1;
  int pm, pd, ho;              // spreading words of either kernel's record; header offset in a staged entry
  int *counts, *start, *entries;   // per cell; entry lists
  int cap;
  const FxStats* stats;        // [FX_AMAX_BLOCKS]
  double K0, K1;               // |contribution| <= K0 max|F| + K1 max|T|
  void* grid;
};
void launch_fx_lists(const FxArgs& A, hipStream_t s);
void launch_spread_fx(const FxArgs& A, int words, const double* F, const double* Tq, hipStream_t s);

struct InterpArgs {
  int N, Nx, Ny, Nz;
  const int* order;
  KernelDesc km, kd;
  const int4 *sup_m, *sup_d;
  const void *rec_m, *rec_d;
  int rs_m, rs_d;
  const int *kt_m, *kt_d;
  const double *fA_m, *fA_d, *fB_d;
  const void* grid;
  int periodic_z;   // rows of a support wrap modulo Nz
  int pair;         // velocities and angular velocities in one pass (shared x/y supports)
};

// Half the curl of a Fourier-Chebyshev field [c][k][Nm] (x, y derivatives i kx,
// i ky with the unpaired Nyquist entries zeroed; z derivative by the Chebyshev
// coefficient recurrence on [0, 2H]), times `scale`; added to `out` or stored.
template <class T>
void launch_curl_cheb(const void* in, void* out, int Nx, int Ny, int Nz, int Nm, const double* kxs,
                      const double* kys, double H, double scale, int add, hipStream_t s);
// Half the Fourier curl of an r2c spectrum [c][kz][ky][kx] (unpaired Nyquist
// entries of each direction zeroed); added to `out` or stored.
template <class T>
void launch_tp_curl(const void* in, void* out, int Nx, int Ny, int Nz, double Lx, double Ly, double Lz, int add,
                    hipStream_t s);

// y pass of the planar transforms: in-place c2c of length Ny along ky of the
// spectrum [nslices][Ny][Nkx], dir -1 forward / +1 inverse (unnormalised);
// tw holds exp(-2 pi i k / Ny), k < Ny, in grid precision.
// x pass of the planar transforms: real rows of NX = Nx points ([row][x]) to
// half-complex rows of Nx/2 + 1 values ([row][kx]), dir -1 forward (real ->
// complex), +1 inverse (complex -> real, unnormalised, imaginary parts of
// kx = 0 and kx = Nx/2 ignored); tw holds exp(-2 pi i k / Nx), k < Nx, in
// grid precision.  Out of place.
// fft_x_fixed / fft_y_fixed: lengths of the compile-time radices
bool fft_x_supported(int Nx);
bool fft_x_fixed(int Nx);
bool fft_y_fixed(int Ny);
template <class T>
void launch_fft_x(const void* in, void* out, int nrows, int Nx, const void* tw, int dir, hipStream_t s);
bool fft_y_supported(int Ny);
template <class T>
void launch_fft_y(void* data, int nslices, int Nkx, int Ny, const void* tw, int dir, hipStream_t s);

// Position gradient of the adjoint: per particle p (records of the force
// kernel's derivatives, dipole layout), with G_u[j][i] = D_j-interpolation of
// component i of grid gu and likewise G_v for gv,
//   grad[p][j] = -sum_i (lam[p][i] G_u[j][i] + f[p][i] G_v[j][i]).
template <class T, class Tio>
void launch_interp_grad(const InterpArgs& A, const int4* sup, const void* rec, int rs, const KernelDesc& K,
                        const void* gu, const void* gv, const void* lam, const void* f, void* grad,
                        hipStream_t s);

// Torque-kernel records of the position adjoint (4 wx + 4 wy + 4 wzmax words
// per particle, on the torque kernel's supports sup_d) and the torque terms
// of the position gradient, added to grad:
//   grad[p][k] += 1/2 sum eps_abc (mu[p][a] J_kb u_c - t[p][c] J_kb v_a).
template <class T>
void launch_stencil_d2(const StencilArgs& A, const int4* sup_d, void* rec, int rs, hipStream_t s);
template <class T, class Tio>
void launch_interp_grad_t(const InterpArgs& A, const int4* sup, const void* rec, int rs, const KernelDesc& K,
                          const void* gu, const void* gv, const void* mu, const void* t, void* grad, hipStream_t s);

// Fourier solve of the triply periodic Stokes problem on the r2c spectrum
// [c][kz][ky][kx] (kx in [0, Nx/2]), scaled by 1/(Nx Ny Nz) for the c2r
template <class T>
void launch_tp_solve(const void* in, void* out, int Nx, int Ny, int Nz, double Lx, double Ly, double Lz,
                     double eta, hipStream_t s);

struct ZArgs {
  int N, NH, NE, NO;   // nodes, node pairs, even/odd coefficient counts
  int Nm, Nkx;         // modes per z level, kx count
  const void *TfE, *TfO, *TiE, *TiO;   // grid precision
  // wall correction (inverse only)
  int nbasis;
  const double2* corr;   // [Nm][3][4]
  const double *kxs, *kys, *zpts;
  double Hs;
  double inv_nxy;   // 1/(Nx Ny): the c2r transform is unnormalised
  int accumulate;   // matrix-core inverse only: add the values to `out`
};

struct BvpArgs {
  BvpConsts B;   // pointers are device pointers
  int Nx, Ny, Nkx, Nm;
  int Ms;                  // scratch stride: Nm + nspecial lanes
  double Lx, Ly;
  const int* special;      // modes touching a Nyquist index
  int nspecial;
  double2* u2;             // [nspecial][3][Nz] mirror solutions
  double *s_ib, *s_ab;     // [Nz+1][Ms], [Nz][Ms]
  double2 *s_P, *s_CP, *s_DP, *s_U0, *s_U1, *s_U2;   // [Nz][Ms] each
  double2* corr;           // [Nm][3][4]
  double2* corr2;          // [nspecial][3][4]
};

template <class Tin, class T> void launch_stencil(const StencilArgs& A, void* pos, hipStream_t s);
void launch_reset_err(int* e, hipStream_t s);
// z tiles of 16 levels per spreading wavefront for a grid
int spread_tiles(int Nx, int Ny, int Nz, bool fp32);
constexpr int spread_max_tiles(bool fp32) { return fp32 ? 3 : 2; }
template <class T, class Tin> void launch_spread(const SpreadArgs& A, const void* F, const void* Tq, hipStream_t s);
template <class T, class Tout> void launch_interp(const InterpArgs& A, void* vel, void* ang, hipStream_t s);
size_t z_lds_bytes(const ZArgs& A, bool mixed);
// z transforms of the one-lane chain as MFMA GEMMs (false: shape not
// supported, the caller keeps the VALU kernels)
template <class T> bool zgemm_supported(const ZArgs& A);
template <class T> bool launch_zfwd_mma(const ZArgs& A, const void* in, void* out, hipStream_t s);
template <class T> bool launch_zinv_mma(const ZArgs& A, const void* in, void* out, hipStream_t s);
template <class T> void launch_zfwd(const ZArgs& A, const void* in, void* out, hipStream_t s);
template <class T> void launch_zinv(const ZArgs& A, const void* in, void* out, hipStream_t s);
template <class T> void launch_bvp(const BvpArgs& A, const void* in, void* out, hipStream_t s);
// Fused spectral solve: z transform -> per-mode BVP on lane groups ->
// Nyquist averaging -> inverse z transform with wall corrections.
struct SpecArgs {
  BvpConsts B;   // device pointers
  int Nx, Ny, Nkx, Nm;
  double Lx, Ly;
  int NH;                 // node pairs ceil(Nz/2)
  int lpm, e, G;          // lanes per mode, rows per lane, modes per block
  const void* TfP;        // [NH][LPM][E] forward rows in lane order (grid precision)
  const void* TiP;        // [ceil(Nz/2)][LPM][E] inverse rows in lane order (scaled by 1/(Nx Ny))
  // matrix-core operands of the FP32 transforms (16-lane shapes), in
  // v_mfma 16x16x4 lane order, zero-padded to LPM E / 8 steps: [2][MT][KSM][64]
  // forward (parity, coefficient tile, 4 node pairs) and inverse (parity,
  // node-pair tile, 4 coefficients of that parity; scaled by 1/(Nx Ny))
  const float* TfM;
  const float* TiM;
  // k_spectral_chains: the same operands for its rows (chain_rows), in grid
  // precision, and the row tables by parity [2][CHAIN_TABLES][rows / 2]
  const void *TfC, *TiC;
  const double* ctab;
  const double* fac_J;    // [nk][rows] k^2 over the pivots of the elimination towards row 0
  const int* fac_idx;     // [Nm] entry of each mode in the factor tables (its |k|^2)
  const double* fac_ib;   // [nk][LPM][E] reciprocal pivots of each lane's rows
  const double* fac_ab;   // [nk][LPM][E] A^{-1}B of each lane's rows
  const double* fac_G;    // [nk][4] inverse Schur complement
  const double *kxs, *kys;   // grid wavenumbers by index
  const double* zpts;
  double Hs, inv_nxy;
};
// Chains (dps_chains.hip): rows held for Nz levels, a multiple of 16 up to 128;
// 0: more levels, the lane groups below (at 128 a lane's rows and the rest fill
// 203 of the 256 registers that two workgroups per CU leave)
#define CHAIN_TABLES 8
constexpr int chain_rows(int Nz) { return Nz > 128 ? 0 : (Nz + 15) / 16 * 16; }
// modes per workgroup: two columns (re, im) of 16 modes are two matrix-core
// column blocks; 8 in FP64 fill the same LDS
constexpr int chain_modes(bool fp32) { return fp32 ? 16 : 8; }
constexpr size_t chain_lds_bytes(int nzp, bool fp32)
{
  const int G = chain_modes(fp32);
  return (size_t)((nzp > 24 ? nzp : 24) + 17) * G * 8 + (size_t)3 * nzp * (G + 1) * (fp32 ? 8 : 16);
}
// waves per SIMD that the LDS of one CU (128 blocks of 1280 bytes) and the registers allow (a
// lane holds nzp / 2 FP64 rows beside about 70 others)
constexpr int chain_waves(int nzp, bool fp32)
{
  const int w = (int)(128 / ((chain_lds_bytes(nzp, fp32) + 1279) / 1280)), v = nzp <= 64 ? 4 : (nzp <= 96 ? 3 : 2);
  return w < 1 ? 1 : (w > v ? v : w);
}
void launch_chain_factor(const BvpConsts& B, const double* ksq, int nk, int nzp, double* J, hipStream_t s);
template <class T> void launch_chains(const SpecArgs& A, int nzp, const void* in, void* out, hipStream_t s);
// lane-group shape for Nz rows: returns false when Nz is too large
bool spectral_shape(int Nz, int* lpm, int* e);
// FP32 z transforms on the matrix cores: 16-lane groups of a mixed-precision
// solve (16 modes per workgroup).  8-lane groups keep the VALU transforms:
// their 24-row parities pad to 32-row tiles and the preloaded tables push
// the solve into scratch (Nz = 48: 836 against 771 us)
constexpr bool spectral_mfma(int lpm, bool mixed) { return mixed && lpm == 16; }
// LDS of one spectral workgroup: 9 row tables of LPM E doubles, 12 wall
// corrections per mode (and |k| per mode on the matrix-core path),
// 3 components x LPM E rows x (G + 1) columns
constexpr size_t spectral_lds_bytes(int lpm, int e, int G, bool mixed)
{
  return (size_t)9 * lpm * e * 8 + (size_t)G * (12 * 16 + (spectral_mfma(lpm, mixed) ? 8 : 0)) +
         (size_t)3 * lpm * e * (G + 1) * (mixed ? 8 : 16);
}
// modes per workgroup: the most (up to 256 lanes) within 64 KiB of LDS, else 1
constexpr int spectral_modes_per_block(int lpm, int e, bool mixed)
{
  int G = 256 / lpm;
  while (G > 1 && spectral_lds_bytes(lpm, e, G, mixed) > 65536) G /= 2;
  return G;
}
// waves per SIMD that the LDS of one CU (160 KiB) allows, at most 3: the
// lane-group solve needs 136 (E = 2) to 226 (E = 8) VGPRs, and a tighter
// register cap sends it to scratch (at 4: 44, 80 and 140 bytes per lane for
// 8 x 2, 16 x 2 and 16 x 4, where 3 leaves none)
constexpr int spectral_waves_per_simd(int lpm, int e, bool mixed)
{
  const int G = spectral_modes_per_block(lpm, e, mixed);
  const int blocks = (int)(163840 / spectral_lds_bytes(lpm, e, G, mixed));
  const int w = blocks * (G * lpm / 64) / 4;
  return w < 1 ? 1 : (w > 3 ? 3 : w);
}
void launch_bvp_factor(const BvpConsts& B, const double* ksq, int nk, double* s_ib, double* s_ab, int lpm,
                       int e, double* fib, double* fab, double* fG, hipStream_t s);
template <class T> void launch_spectral(const SpecArgs& A, const void* in, void* out, hipStream_t s);
template <class T> void launch_ref_to_grid(const double* ref, void* g, int Nx, int Ny, int Nz, hipStream_t s);
template <class T> void launch_grid_to_ref(const void* g, double* ref, int Nx, int Ny, int Nz, hipStream_t s);

}  // namespace dps
