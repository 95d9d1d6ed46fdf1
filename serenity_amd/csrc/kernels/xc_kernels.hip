// HIP kernels of the XC Fock build for gfx950.
//
//   screen      block-centre shell screening (BasisFunctionOnGridController.cpp:211-255)
//   ao_eval     AO values + gradients of the significant shells into resident tiles
//               (BasisFunctionOnGridController.cpp:256-1097)
//   density     T = phi_b P_b on matrix cores, rho = rowdot(T, phi), grad rho = 2 rowdot(T, grad phi)
//               (MatrixOperatorToGridTransformer.cpp:103-165)
//   functional  per-point XC energy density and potential, block skip and E_xc partials
//               (XCFun.cpp:129-158, 751-765)
//   fock        S_b = phi_b^T G_b + G_b^T phi_b on matrix cores, the upper-triangle sub-tiles
//               of every block stored to a scratch (ScalarOperatorToMatrixAdder.cpp:179-303)
//   fock_reduce F = sum over blocks of S_b scattered by the blocks' AO lists, one AO row per
//               workgroup adding its blocks' terms in LDS, in an order that varies unless the
//               context is deterministic (the reference's thread-private F plus serial sum,
//               ScalarOperatorToMatrixAdder.cpp:101-110)
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <type_traits>

#include "mfma.h"
#include "xc_internal.h"

namespace sxc {

namespace {

__global__ __launch_bounds__(64) void screen_kernel(const double* __restrict__ pts, int64_t npts, int bs,
                                                    const DevShell* __restrict__ shells, int nshell,
                                                    const double* __restrict__ alpha,
                                                    const double* __restrict__ coef, double thr,
                                                    int* __restrict__ pos, int* __restrict__ count) {
  __shared__ double c[4], xyz[3 * kTile];
  const int b = blockIdx.x, t = threadIdx.x;
  const int64_t first = (int64_t)b * bs;
  const int B = (int)min((int64_t)bs, npts - first);
  for (int i = t; i < 3 * B; i += 64) xyz[i] = pts[3 * first + i];
  __syncthreads();
  // block centre (mean), accumulated point by point in order, one lane per coordinate; spread
  // (largest distance to the centre)
  if (t < 3) {
    double s = 0.0;
    for (int p = 0; p < B; ++p) s += xyz[3 * p + t];
    c[t] = s / B;
  }
  __syncthreads();
  double sp = 0.0;
  for (int p = t; p < B; p += 64) {
    const double dx = xyz[3 * p] - c[0], dy = xyz[3 * p + 1] - c[1], dz = xyz[3 * p + 2] - c[2];
    sp = fmax(sp, sqrt(dx * dx + dy * dy + dz * dz));
  }
  for (int m = 1; m < 64; m <<= 1) sp = fmax(sp, __shfl_xor(sp, m));
  if (t == 0) c[3] = sp;
  __syncthreads();
  // 64 shells at a time; a significant shell's compact position is the functions of those before it
  int nao = 0, nsig = 0;
  for (int s0 = 0; s0 < nshell; s0 += 64) {
    const int s = s0 + t;
    int nf = 0;
    if (s < nshell) {
      const DevShell sh = shells[s];
      const double dx = c[0] - sh.cx, dy = c[1] - sh.cy, dz = c[2] - sh.cz;
      double d = sqrt(dx * dx + dy * dy + dz * dz) - c[3];
      nf = sh.nfunc;
      if (!(d < 1.0)) {
        // radial part at the closest possible distance of any block point
        d = d * d;
        double radial = 0.0;
        for (int q = 0; q < sh.nprim; ++q) radial += coef[sh.prim_off + q] * exp(-alpha[sh.prim_off + q] * d);
        if (fabs(radial) < thr) nf = 0;
      }
    }
    int sum = nf;  // inclusive prefix over the lanes
    for (int m = 1; m < 64; m <<= 1) {
      const int v = __shfl_up(sum, m);
      if (t >= m) sum += v;
    }
    if (s < nshell) pos[(int64_t)b * nshell + s] = nf > 0 ? nao + sum - nf : -1;
    nao += __shfl(sum, 63);
    nsig += __popcll(__ballot(nf > 0));
  }
  if (t == 0) {
    count[2 * b] = nao;
    count[2 * b + 1] = nsig;
  }
}

// The lists of the blocks from their shells' compact positions: significant shells with their
// positions, and the AO index list padded with -1.
__global__ __launch_bounds__(64) void block_lists_kernel(const DevBlock* __restrict__ blocks,
                                                         const DevShell* __restrict__ shells, int nshell,
                                                         const int* __restrict__ pos, int* __restrict__ sig_shell,
                                                         int* __restrict__ sig_pos, int* __restrict__ ao_idx) {
  const int b = blockIdx.x, t = threadIdx.x;
  const DevBlock bk = blocks[b];
  int rank = bk.shell_off;
  for (int s0 = 0; s0 < nshell; s0 += 64) {
    const int s = s0 + t, p = s < nshell ? pos[(int64_t)b * nshell + s] : -1;
    const unsigned long long sig = __ballot(p >= 0);
    if (p >= 0) {
      const int at = rank + __popcll(sig & ((1ull << t) - 1));
      sig_shell[at] = s;
      sig_pos[at] = p;
      const int ao = shells[s].ao_off, nf = shells[s].nfunc;
      for (int f = 0; f < nf; ++f) ao_idx[bk.idx_off + p + f] = ao + f;
    }
    rank += __popcll(sig);
  }
  for (int i = bk.nb + t; i < bk.npad; i += 64) ao_idx[bk.idx_off + i] = -1;
}

// Row entries of the Fock reduce, for every AO the blocks holding it in block order, in three steps
// over chunks of kRowChunk blocks: the blocks of each chunk that hold a shell are counted, the counts
// become offsets (per shell over the chunks, then over the AOs), and the entries are written.
constexpr int kRowChunk = 16;
__global__ __launch_bounds__(256) void row_count_kernel(const int* __restrict__ pos, int nblocks, int nshell,
                                                        int* __restrict__ cnt) {
  const int s = blockIdx.y * 256 + threadIdx.x, b0 = blockIdx.x * kRowChunk;
  if (s >= nshell) return;
  int n = 0;
  for (int b = b0; b < min(b0 + kRowChunk, nblocks); ++b) n += pos[(int64_t)b * nshell + s] >= 0;
  cnt[(int64_t)blockIdx.x * nshell + s] = n;
}

__global__ __launch_bounds__(1024) void row_offsets_kernel(const DevShell* __restrict__ shells, int nshell, int nchunk,
                                                           int nao, int* __restrict__ cnt, int* __restrict__ row_ptr) {
  __shared__ int part[1024];
  const int t = threadIdx.x;
  int base = 0;
  for (int s0 = 0; s0 < nshell; s0 += 1024) {
    const int s = s0 + t;
    int total = 0, nf = 0, ao = 0;
    if (s < nshell) {
      nf = shells[s].nfunc;
      ao = shells[s].ao_off;
      for (int k = 0; k < nchunk; ++k) {
        const int n = cnt[(int64_t)k * nshell + s];
        cnt[(int64_t)k * nshell + s] = total;
        total += n;
      }
    }
    part[t] = total * nf;
    __syncthreads();
    for (int m = 1; m < 1024; m <<= 1) {
      const int v = t >= m ? part[t - m] : 0;
      __syncthreads();
      part[t] += v;
      __syncthreads();
    }
    for (int f = 0; f < nf; ++f) row_ptr[ao + f] = base + part[t] - total * (nf - f);
    base += part[1023];
    __syncthreads();
  }
  if (t == 0) row_ptr[nao] = base;
}

__global__ __launch_bounds__(256) void row_entries_kernel(const DevBlock* __restrict__ blocks, int nblocks,
                                                          const DevShell* __restrict__ shells, int nshell,
                                                          const int* __restrict__ pos, const int* __restrict__ cnt,
                                                          const int* __restrict__ row_ptr, RowEnt* __restrict__ ent) {
  const int s = blockIdx.y * 256 + threadIdx.x, b0 = blockIdx.x * kRowChunk;
  if (s >= nshell) return;
  const int ao = shells[s].ao_off, nf = shells[s].nfunc;
  int k = cnt[(int64_t)blockIdx.x * nshell + s];
  for (int b = b0; b < min(b0 + kRowChunk, nblocks); ++b) {
    const int p = pos[(int64_t)b * nshell + s];
    if (p < 0) continue;
    const DevBlock bk = blocks[b];
    for (int f = 0; f < nf; ++f) {
      const int l = p + f;
      RowEnt e;
      e.rowbase = bk.toff + fock_row_start(l, bk.npad) - 16 * (l / 16);
      e.c0 = l;
      e.c1 = bk.nb;
      e.idx_off = bk.idx_off;
      e.block = b;
      ent[row_ptr[ao + f] + k] = e;
    }
    ++k;
  }
}

// One workgroup per block and kAoShells of its shells, one thread per point: the exponentials of a
// shell's primitives bound it, so a block's shells are spread over workgroups (one after another
// they left most of the chip idle: (H2O)12/def2-SVP, 1175 blocks, 215 us and as much clearing;
// now 118, 360 MB of FP32 tiles at 3 TB/s).  Every element of
// the block's tiles is written, so they need no clearing.
constexpr int kAoShells = 8;
__global__ __launch_bounds__(128) void ao_kernel(const DevBlock* __restrict__ blocks, const int* __restrict__ sig_shell,
                                                 const int* __restrict__ sig_pos, const DevShell* __restrict__ shells,
                                                 const double* __restrict__ alpha, const double* __restrict__ coef,
                                                 const double* __restrict__ ang, const double* __restrict__ pts,
                                                 double thr, double exp_thr, int ncomp, double* __restrict__ t64,
                                                 float* __restrict__ t32) {
  const DevBlock bk = blocks[blockIdx.x];
  const int p = threadIdx.x;
  const int k0 = blockIdx.y * kAoShells, k1 = min(k0 + kAoShells, bk.nshell);
  if (k0 >= max(bk.nshell, 1)) return;  // uniform over the workgroup
  const int64_t cstride = (int64_t)bk.npad * kTile;
  // rows that no AO fills (padding) and points beyond the block are zero
  auto zero = [&](int64_t o) {
    for (int c = 0; c < ncomp; ++c) {
      if (t64) t64[o + c * cstride] = 0.0;
      if (t32) t32[o + c * cstride] = 0.0f;
    }
  };
  if (k0 == 0)
    for (int i = bk.nb; i < bk.npad; ++i) zero(bk.tile_off + (int64_t)i * kTile + p);
  const bool in = p < bk.npts;
  const int64_t q = bk.first + (in ? p : 0);
  const double px = pts[3 * q + 0], py = pts[3 * q + 1], pz = pts[3 * q + 2];
  for (int k = k0; k < k1; ++k) {
    const int s = sig_shell[bk.shell_off + k];
    const int pos = sig_pos[bk.shell_off + k];
    const DevShell sh = shells[s];
    const double dx = px - sh.cx, dy = py - sh.cy, dz = pz - sh.cz;
    const double r2 = dx * dx + dy * dy + dz * dz;
    double R = 0.0, dR = 0.0, ddR = 0.0;
    for (int q = 0; q < sh.nprim; ++q) {
      const double a = alpha[sh.prim_off + q];
      const double t = a * r2;
      if (t < exp_thr) {
        const double e = exp(-t);
        const double ce = coef[sh.prim_off + q] * e;
        R += ce;
        dR -= 2.0 * a * ce;
        ddR += 4.0 * a * a * ce;
      }
    }
    const int64_t base = bk.tile_off + (int64_t)pos * kTile + p;
    if (!in || fabs(R) < thr) {
      for (int f = 0; f < sh.nfunc; ++f) zero(base + (int64_t)f * kTile);
      continue;
    }
    double xp[kMaxL + 1], yp[kMaxL + 1], zp[kMaxL + 1];
    xp[0] = yp[0] = zp[0] = 1.0;
    for (int e = 1; e <= sh.l; ++e) {
      xp[e] = xp[e - 1] * dx;
      yp[e] = yp[e - 1] * dy;
      zp[e] = zp[e - 1] * dz;
    }
    const bool hess = ncomp >= 10;
    for (int f = 0; f < sh.nfunc; ++f) {
      double Y = 0.0, Yx = 0.0, Yy = 0.0, Yz = 0.0;
      double Yxx = 0.0, Yxy = 0.0, Yxz = 0.0, Yyy = 0.0, Yyz = 0.0, Yzz = 0.0;
      int ci = 0;
      for (int a = sh.l; a >= 0; --a)
        for (int b = sh.l - a; b >= 0; --b, ++ci) {
          const double m = ang[sh.ang_off + f * sh.ncart + ci];
          if (m == 0.0) continue;
          const int c = sh.l - a - b;
          Y += m * xp[a] * yp[b] * zp[c];
          if (a > 0) Yx += m * a * xp[a - 1] * yp[b] * zp[c];
          if (b > 0) Yy += m * b * xp[a] * yp[b - 1] * zp[c];
          if (c > 0) Yz += m * c * xp[a] * yp[b] * zp[c - 1];
          if (hess) {
            if (a > 1) Yxx += m * a * (a - 1) * xp[a - 2] * yp[b] * zp[c];
            if (b > 1) Yyy += m * b * (b - 1) * xp[a] * yp[b - 2] * zp[c];
            if (c > 1) Yzz += m * c * (c - 1) * xp[a] * yp[b] * zp[c - 2];
            if (a > 0 && b > 0) Yxy += m * a * b * xp[a - 1] * yp[b - 1] * zp[c];
            if (a > 0 && c > 0) Yxz += m * a * c * xp[a - 1] * yp[b] * zp[c - 1];
            if (b > 0 && c > 0) Yyz += m * b * c * xp[a] * yp[b - 1] * zp[c - 1];
          }
        }
      const int64_t o = base + (int64_t)f * kTile;
      const double val = R * Y;
      if (t64) t64[o] = val;
      if (t32) t32[o] = (float)val;
      if (ncomp > 1) {
        const double gx = R * Yx + dR * dx * Y;
        const double gy = R * Yy + dR * dy * Y;
        const double gz = R * Yz + dR * dz * Y;
        if (t64) {
          t64[o + cstride] = gx;
          t64[o + 2 * cstride] = gy;
          t64[o + 3 * cstride] = gz;
        }
        if (t32) {
          t32[o + cstride] = (float)gx;
          t32[o + 2 * cstride] = (float)gy;
          t32[o + 3 * cstride] = (float)gz;
        }
      }
      if (hess) {
        // d_i d_j (R Y) = R Y_ij + R' (x_i Y_j + x_j Y_i) + d_ij R' Y + R'' x_i x_j Y,
        // R' = sum -2 a c e^(-a r^2), R'' = sum 4 a^2 c e^(-a r^2); planes xx xy xz yy yz zz
        const double h[6] = {R * Yxx + dR * (2.0 * dx * Yx + Y) + ddR * dx * dx * Y,
                             R * Yxy + dR * (dx * Yy + dy * Yx) + ddR * dx * dy * Y,
                             R * Yxz + dR * (dx * Yz + dz * Yx) + ddR * dx * dz * Y,
                             R * Yyy + dR * (2.0 * dy * Yy + Y) + ddR * dy * dy * Y,
                             R * Yyz + dR * (dy * Yz + dz * Yy) + ddR * dy * dz * Y,
                             R * Yzz + dR * (2.0 * dz * Yz + Y) + ddR * dz * dz * Y};
        for (int c = 0; c < 6; ++c) {
          if (t64) t64[o + (4 + c) * cstride] = h[c];
          if (t32) t32[o + (4 + c) * cstride] = (float)h[c];
        }
      }
    }
  }
}

// The four FP32 tile values of a lane's MFMA accumulator rows: points 4 (lane / 16) + e,
// e = 0..3, of a 16-point row segment -- one aligned 16-byte load.
__device__ inline void quad_rows(const gmem<const float>* seg, int lane, double f[4]) {
  const f32x4 v = *reinterpret_cast<const gmem<const f32x4>*>(seg + 4 * (lane >> 4));
  f[0] = v.x;
  f[1] = v.y;
  f[2] = v.z;
  f[3] = v.w;
}

// Work item and spin of workgroup x of a launch of pairs items for two spins (0: one pass, item x):
// eight items of one spin, then the same eight of the other, so that an item's two passes run on one
// XCD shortly after each other and the second finds the tiles in its L2.
__device__ __forceinline__ int pair_item(int pairs, int x, int& spin) {
  spin = pairs ? (x >> 3) & 1 : 0;
  return pairs ? (x >> 4) * 8 + (x & 7) : x;
}

// What the density items of one launch share.
template <typename T>
struct DensityArgs {
  const int* ao_idx;
  const T* tiles;
  const T* P;
  int n, want_grad;
  double* part;
  int64_t npts;
};

// Density contraction on 16 x 16 sub-tiles.  One workgroup of 8 wavefronts
// per (block, column pass): T[p][nu] = sum_mu phi[mu][p] P[mu][nu] for the
// pass's 16 S columns, wavefront w owning points 16 w .. 16 w + 15 and all S
// column tiles (S independent accumulators).  The AO (K) dimension streams in
// chunks of KC (32 FP32 / 16 FP64) through an LDS buffer that holds phi
// point-major and the pass's P columns, both with the AO index fastest: with
// k-step t of lane group g taking AO KV g + t (KV = KC / 4) every MFMA operand
// of a chunk is one 32-byte LDS read.  The global loads of chunk k + 1 are
// issued before the MFMAs of chunk k.  The pass's partial rho and
// sum_nu T grad phi are then formed from the accumulators in registers, each
// lane dotting its T entries with the phi / grad phi values of the same
// (point, column), and summed over the columns by lane shuffles.  (FP64
// accumulates T transposed, so that its lanes read whole 128-byte point runs.)
template <typename T, int S, bool Tri>
__device__ __forceinline__ void density_item(const WorkItem& wk, const DevBlock& bk, const DensityArgs<T>& arg,
                                             unsigned char* smem, int* sIdx) {
  using M = Mfma<T>;
  constexpr int KC = 128 / (int)sizeof(T);      // AOs per chunk (128 bytes of each LDS row)
  constexpr int KV = KC / 4;
  constexpr int RS = KC + 16 / (int)sizeof(T);  // 144-byte rows
  constexpr int NC = 16 * S;
  constexpr int NB = (4 * NC + 511) / 512;      // P staging tasks per thread
  constexpr int GS = 2;
  typedef T vec_t __attribute__((ext_vector_type(KV)));
  T(*sA)[RS] = reinterpret_cast<T(*)[RS]>(smem);
  T(*sB)[RS] = reinterpret_cast<T(*)[RS]>(smem + kTile * RS * sizeof(T));
  const int* ao_idx = arg.ao_idx;
  const T* tiles = arg.tiles;
  const T* P = arg.P;
  double* part = arg.part;
  const int n = arg.n, want_grad = arg.want_grad;
  const int64_t npts = arg.npts;
  const int col0 = wk.a, ncols = wk.b;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int npad = bk.npad;
  const gmem<const T>* tb = to_global(tiles + bk.tile_off);
  const gmem<const int>* idx = to_global(ao_idx + bk.idx_off);
  const gmem<const T>* Pg = to_global(P);
  const int64_t cstride = (int64_t)npad * kTile;
  // staging: phi task = (point pa, AO quad qa); P tasks = (column cb, AO quad qb), 16
  // consecutive lanes taking 16 columns of one quad (their LDS stores then cover distinct banks)
  const int pa = tid & (kTile - 1), qa = tid >> 7;
  const int qb = (tid >> 4) & 3;
  auto col_of = [](int task) { return (task & 15) + 16 * (task >> 6); };
  int nu[NB];
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int task = tid + 512 * m, cb = col_of(task);
    nu[m] = (task < 4 * NC && cb < ncols) ? idx[col0 + cb] : -1;
  }
  typename M::acc_t acc[S];
#pragma unroll
  for (int c = 0; c < S; ++c) acc[c] = M::zero();
  vec_t rA, rB[NB];
  unsigned mu_ok = 0;  // bit e: AO KV qb + e of the chunk is not padding
  // chunk at AO k0 of the block, its AO indices at sIdx[j0 ..]
  auto load = [&](int k0, int j0) {
#pragma unroll
    for (int e = 0; e < KV; ++e) rA[e] = tb[(int64_t)(k0 + KV * qa + e) * kTile + pa];
    int mu[KV];
    mu_ok = 0;
#pragma unroll
    for (int e = 0; e < KV; ++e) {
      mu[e] = sIdx[j0 + KV * qb + e];
      mu_ok |= (unsigned)(mu[e] >= 0) << e;
    }
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      if (tid + 512 * m < 4 * NC) {  // whole wavefronts
        // P is symmetric: read P[nu][mu] so that the 16 lanes of a group (consecutive
        // columns nu, one mu) read consecutive addresses.  Padding (index -1) reads P[0][0]
        // and is zeroed at the LDS store by a multiply: a select at the load would let the
        // compiler move the load into a branch, and a multiply there would wait for it
        // before the chunk's MFMAs.
#pragma unroll
        for (int e = 0; e < KV; ++e) rB[m][e] = Pg[max(nu[m], 0) + (int64_t)n * max(mu[e], 0)];
      }
    }
  };
  auto store = [&]([[maybe_unused]] int k0) {
    *reinterpret_cast<vec_t*>(&sA[pa][KV * qa]) = rA;
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      const int task = tid + 512 * m;
      if (task < 4 * NC) {
        vec_t v = rB[m];
#pragma unroll
        for (int e = 0; e < KV; ++e) {
          const bool ok = ((mu_ok >> e) & 1u) && nu[m] >= 0;
          v[e] *= T(ok && (!Tri || k0 + KV * qb + e <= col0 + col_of(task)));
        }
        *reinterpret_cast<vec_t*>(&sB[col_of(task)][KV * qb]) = v;
      }
    }
  };
  // The block's AO index list goes to LDS (the P rows of a chunk are then gathered without a
  // dependent global load) in windows of kDensIdxLds entries: one window unless the block is
  // wider.  One LDS buffer; the global loads of chunk k + 1 of a window are in flight during the
  // MFMAs of chunk k.
  // whole chunks: at most npad, whose last AOs are zero (Tri: up to the pass's last column)
  const int kend = ((Tri ? min(bk.nb, col0 + ncols) : bk.nb) + KC - 1) / KC * KC;
  for (int wb = 0; wb < kend; wb += kDensIdxLds) {
    const int wl = min(kDensIdxLds, kend - wb);
    for (int i = tid; i < wl; i += 512) sIdx[i] = idx[wb + i];
    __syncthreads();
    const int nch = wl / KC;
    load(wb, 0);
    for (int ch = 0; ch < nch; ++ch) {
      store(wb + ch * KC);
      __syncthreads();
      if (ch + 1 < nch) load(wb + (ch + 1) * KC, (ch + 1) * KC);
      const vec_t av = *reinterpret_cast<const vec_t*>(&sA[16 * w + r][KV * g]);
#pragma unroll
      for (int s0 = 0; s0 < S; s0 += GS) {
        vec_t bv[GS];
#pragma unroll
        for (int u = 0; u < GS; ++u)
          if (s0 + u < S) bv[u] = *reinterpret_cast<const vec_t*>(&sB[16 * (s0 + u) + r][KV * g]);
#pragma unroll
        for (int t = 0; t < KV; ++t)
#pragma unroll
          for (int u = 0; u < GS; ++u)
            if (s0 + u < S) {
              // FP64 accumulates T transposed (rows: AO columns, columns: points), so that a
              // lane's entries are one point of four AO columns in the dot phase
              if constexpr (sizeof(T) == 8)
                acc[s0 + u] = M::step(bv[u][t], av[t], acc[s0 + u]);
              else
                acc[s0 + u] = M::step(av[t], bv[u][t], acc[s0 + u]);
            }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();  // (also orders the next window's index staging after this window's reads)
    }
  }

  if constexpr (sizeof(T) == 4) {
    // Dots straight from the accumulators: lane (r, g) holds T[row(lane, e)][16 s + r] of its
    // wavefront's 16 points for every column tile s, and reads the matching phi / grad phi of
    // those 4 points from the tiles (FP32: one 16-byte load per component).  All loads of the
    // phase are independent of each other and of LDS, so they are in flight together.
    double rv[4] = {0.0, 0.0, 0.0, 0.0}, xv[4] = {0.0, 0.0, 0.0, 0.0};
    double yv[4] = {0.0, 0.0, 0.0, 0.0}, zv[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < S; ++c) {
      if (16 * c < ncols) {
        const gmem<const T>* row = tb + (int64_t)(col0 + 16 * c + r) * kTile + 16 * w;
        double f[4];
        quad_rows(row, lane, f);
#pragma unroll
        for (int e = 0; e < 4; ++e) rv[e] += (double)acc[c][e] * f[e];
        if (want_grad) {
          double fx[4], fy[4], fz[4];
          quad_rows(row + cstride, lane, fx);
          quad_rows(row + 2 * cstride, lane, fy);
          quad_rows(row + 3 * cstride, lane, fz);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            xv[e] += (double)acc[c][e] * fx[e];
            yv[e] += (double)acc[c][e] * fy[e];
            zv[e] += (double)acc[c][e] * fz[e];
          }
        }
      }
    }
    // sum over the 16 lanes of a lane group (the columns), a fixed butterfly order
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        rv[e] += __shfl_xor(rv[e], m);
        if (want_grad) {
          xv[e] += __shfl_xor(xv[e], m);
          yv[e] += __shfl_xor(yv[e], m);
          zv[e] += __shfl_xor(zv[e], m);
        }
      }
    }
    if (r == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int p = 16 * w + M::row(lane, e);
        if (p < bk.npts) {
          gmem<double>* dst = to_global(part + (int64_t)wk.pass * 4 * npts + bk.first + p);
          dst[0] = rv[e];
          if (want_grad) {
            dst[npts] = xv[e];
            dst[2 * npts] = yv[e];
            dst[3 * npts] = zv[e];
          }
        }
      }
    }
  } else {
    // lane (r, g) holds T[point 16 w + r][AO column 16 c + g + 4 e]: per e the dot reads 16
    // consecutive points (128 bytes) of each of four tile rows
    double rv = 0.0, xv = 0.0, yv = 0.0, zv = 0.0;
#pragma unroll
    for (int c = 0; c < S; ++c) {
      if (16 * c < ncols) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const gmem<const T>* row = tb + (int64_t)(col0 + 16 * c + g + 4 * e) * kTile + 16 * w + r;
          const double tv = acc[c][e];
          rv += tv * row[0];
          if (want_grad) {
            xv += tv * row[cstride];
            yv += tv * row[2 * cstride];
            zv += tv * row[3 * cstride];
          }
        }
      }
    }
    // sum over the four lane groups (the AO columns g + 4 e of each tile)
    rv += __shfl_xor(rv, 16);
    rv += __shfl_xor(rv, 32);
    if (want_grad) {
      xv += __shfl_xor(xv, 16);
      xv += __shfl_xor(xv, 32);
      yv += __shfl_xor(yv, 16);
      yv += __shfl_xor(yv, 32);
      zv += __shfl_xor(zv, 16);
      zv += __shfl_xor(zv, 32);
    }
    const int p = 16 * w + r;
    if (g == 0 && p < bk.npts) {
      gmem<double>* dst = to_global(part + (int64_t)wk.pass * 4 * npts + bk.first + p);
      dst[0] = rv;
      if (want_grad) {
        dst[npts] = xv;
        dst[2 * npts] = yv;
        dst[3 * npts] = zv;
      }
    }
  }
}

// Every pass width in one kernel: a launch per width left each of them a tail of its own, and small
// systems paid the launches and the stream forks more than the work ((H2O)8/def2-SVP: 108 us of
// which the kernels ran 49).
// Tri: the density alone (no gradient) is a quadratic form, rho = sum_nu phi_nu sum_(mu <= nu) phi_mu Q_mu,nu
// with Q = P + P^T above the diagonal and P on it, so a pass contracts only the AOs up to its last
// column: half the MFMAs and elements of P on average.  The caller passes Q (fold_kernel).  FP64
// only (the other order of the sum moves FP32 densities by FP32 rounding), and for the builds: the
// densities handed out or cached are the same bits with and without their gradient.
template <typename T, bool Tri>
__global__ __launch_bounds__(512) void density_sub_kernel(const WorkItem* __restrict__ work,
                                                          const DevBlock* __restrict__ blocks, DensityArgs<T> arg,
                                                          const PackSys* __restrict__ pack,
                                                          const int* __restrict__ nwork_dev,
                                                          const unsigned char* __restrict__ skip, int pairs) {
  // a launch over a list filled on the device runs only its first *nwork_dev items
  if (nwork_dev && (int)blockIdx.x >= *nwork_dev) return;
  int spin;
  const int item = pair_item(pairs, blockIdx.x, spin);
  if (pairs && item >= pairs) return;
  __shared__ __attribute__((aligned(16))) unsigned char smem[(kTile + 16 * kDensMaxS) * 144];
  __shared__ int sIdx[kDensIdxLds];
  const WorkItem wk = work[item];
  if (skip && skip[wk.block]) return;  // a block the caller contracts in another pass
  const DevBlock bk = blocks[wk.block];
  if (pack) {
    const PackSys& ps = pack[bk.sys + spin];
    arg.tiles = static_cast<const T*>(ps.tiles);
    arg.P = static_cast<const T*>(ps.P);
    arg.ao_idx = ps.ao_idx;
    arg.part = ps.part;
    arg.npts = ps.npts;
    arg.n = ps.n;
  }
  static_assert(kDensMaxS == 6, "one case per pass width");
  switch ((wk.b + 15) / 16) {
    case 1: return density_item<T, 1, Tri>(wk, bk, arg, smem, sIdx);
    case 2: return density_item<T, 2, Tri>(wk, bk, arg, smem, sIdx);
    case 3: return density_item<T, 3, Tri>(wk, bk, arg, smem, sIdx);
    case 4: return density_item<T, 4, Tri>(wk, bk, arg, smem, sIdx);
    case 5: return density_item<T, 5, Tri>(wk, bk, arg, smem, sIdx);
    default: return density_item<T, 6, Tri>(wk, bk, arg, smem, sIdx);
  }
}

__global__ void reduce_partials_kernel(const DevBlock* __restrict__ blocks, int bs, int64_t npts,
                                       const double* __restrict__ part, int want_grad, double* __restrict__ rho,
                                       double* __restrict__ grad, int accumulate) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npts) return;
  const int np = blocks[q / bs].npass;
  double r = 0.0, x = 0.0, y = 0.0, z = 0.0;
  for (int s = 0; s < np; ++s) {
    const double* src = part + (int64_t)s * 4 * npts + q;
    r += src[0];
    if (want_grad) {
      x += src[npts];
      y += src[2 * npts];
      z += src[3 * npts];
    }
  }
  if (accumulate) {
    rho[q] += r;
    if (want_grad) {
      grad[q] += 2.0 * x;
      grad[npts + q] += 2.0 * y;
      grad[2 * npts + q] += 2.0 * z;
    }
  } else {
    rho[q] = r;
    if (want_grad) {
      grad[q] = 2.0 * x;
      grad[npts + q] = 2.0 * y;
      grad[2 * npts + q] = 2.0 * z;
    }
  }
}

__device__ inline double block_sum_128(double x, double* red) {
  // fixed-order tree reduction over 128 threads
  const int t = threadIdx.x;
  red[t] = x;
  __syncthreads();
  for (int s = 64; s > 0; s >>= 1) {
    if (t < s) red[t] += red[t + s];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(128) void functional_kernel(int func, int64_t npts, int bs,
                                                         const double* __restrict__ rho,
                                                         const double* __restrict__ grad,
                                                         const DevBlock* __restrict__ blocks,
                                                         const double* __restrict__ part,
                                                         const double* __restrict__ w, double* __restrict__ eps,
                                                         double* __restrict__ v, double* __restrict__ g,
                                                         double* __restrict__ vs, double* __restrict__ gw,
                                                         double* __restrict__ e_blk,
                                                         const PackSys* __restrict__ pack) {
  __shared__ double red[128];
  const int bm = blockIdx.x, t = threadIdx.x;  // bm: block in the (merged) block list
  int b = bm;                                  // block of this system's grid
  if (pack) {
    const PackSys& ps = pack[blocks[bm].sys];
    b = bm - ps.blk0;
    npts = ps.npts;
    part = ps.part;
    w = ps.w;
    vs = ps.vs;
    gw = ps.gw;
    e_blk = ps.eblk;
  }
  const int64_t first = (int64_t)b * bs;
  const int B = (int)min((int64_t)bs, npts - first);
  const int64_t q = first + t;
  const bool in = t < B;
  const bool gga = functional_is_gga(func);
  double r = 0.0, gx = 0.0, gy = 0.0, gz = 0.0;
  if (in) {
    if (part) {
      // sum the density passes of this block (blocks of 128 points)
      const int np = blocks[bm].npass;
      for (int s = 0; s < np; ++s) {
        const double* src = part + (int64_t)s * 4 * npts + q;
        r += src[0];
        if (gga) {
          gx += src[npts];
          gy += src[2 * npts];
          gz += src[3 * npts];
        }
      }
      gx *= 2.0;
      gy *= 2.0;
      gz *= 2.0;
    } else {
      r = rho[q];
      if (gga && grad) {
        gx = grad[q];
        gy = grad[npts + q];
        gz = grad[2 * npts + q];
      }
    }
  }
  const double sumabs = block_sum_128(fabs(r), red);
  const bool skip = sumabs < B * 1e-12;
  double e = 0.0, vv = 0.0, gg[3] = {0.0, 0.0, 0.0};
  if (in && !skip) e = xc_point(func, r, gx, gy, gz, &vv, gg);
  const double wq = in ? w[q] : 0.0;
  if (in) {
    if (eps) eps[q] = e;
    if (v) v[q] = vv;
    if (g) {
      g[q] = gg[0];
      g[npts + q] = gg[1];
      g[2 * npts + q] = gg[2];
    }
    if (vs) vs[q] = wq * vv;
    if (gw) {
      gw[q] = wq * gg[0];
      gw[npts + q] = wq * gg[1];
      gw[2 * npts + q] = wq * gg[2];
    }
  }
  const double eb = block_sum_128(wq * e, red);
  if (t == 0) e_blk[b] = eb;
}

// Sum of x[0..n) and x2[0..n2) by the first 256 threads of a workgroup, in a fixed order (every thread
// of the workgroup calls it).  Eight loads of a thread at a time: one after another they are a chain of
// memory latencies (the energy sum of a mixed (H2O)64/def2-TZVP build 39 us, 13 so).
__device__ double sum_256(const double* x, int64_t n, const double* x2, int64_t n2, double* red) {
  constexpr int U = 8;
  const int t = threadIdx.x;
  if (t < 256) {
    double s[U] = {};
    for (int64_t i = t; i < n; i += 256 * U)
#pragma unroll
      for (int u = 0; u < U; ++u) s[u] += i + 256 * u < n ? x[i + 256 * u] : 0.0;
    for (int64_t i = t; i < n2; i += 256 * U)
#pragma unroll
      for (int u = 0; u < U; ++u) s[u] += i + 256 * u < n2 ? x2[i + 256 * u] : 0.0;
    red[t] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
  }
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (t < k) red[t] += red[t + k];
    __syncthreads();
  }
  return red[0];
}

// Functional of a non-additive build.  Workgroups of y = 0: one block of v[rho_sup] - v[rho_act] (w v,
// w g) and its energy, rho_sup summed from the listed densities on the way (in list order, the active
// one first); of y > 0: a block of the energy of pend.dens.rho[y - 1] alone, into pend.eblk[y - 1]
// (y = blockIdx.y, one more without the first).  What were a pass over all densities, a launch per
// functional and one per energy sum took 36 us and as much between them (benzene and 12 waters in
// def2-SVP, 205 486 points, Thomas-Fermi); this launch and nadd_energy_kernel 19 us.
struct PendingEnergies {
  DensityList dens;
  double* eblk[kListMax];
};
__global__ __launch_bounds__(128) void nadd_functional_kernel(int func, int64_t npts, int y0,
                                                              DensityList sup, const double* __restrict__ rho_act,
                                                              const double* __restrict__ grad_act,
                                                              PendingEnergies pend, const double* __restrict__ w,
                                                              double* __restrict__ vs, double* __restrict__ gw,
                                                              double* __restrict__ e_blk) {
  __shared__ double red[128];
  const int b = blockIdx.x, t = threadIdx.x, y = y0 + blockIdx.y;
  const int64_t q = (int64_t)b * kTile + t;
  const int B = (int)min((int64_t)kTile, npts - (int64_t)b * kTile);
  const bool in = t < B, gga = functional_is_gga(func);
  double r = 0.0, g[3] = {0.0, 0.0, 0.0};
  if (in) {
    if (y == 0) {
      // four densities' loads at a time (one after another they are a chain of memory latencies:
      // 27 us for PBE over 13 densities with gradients at 205 486 points, 7 more one after another)
      constexpr int U = 4;
      for (int i0 = 0; i0 < sup.n; i0 += U) {
        double x[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = min(i0 + u, sup.n - 1);
          x[u][0] = to_global(sup.rho[i])[q];
          if (gga)
#pragma unroll
            for (int c = 0; c < 3; ++c) x[u][1 + c] = to_global(sup.grad[i])[c * npts + q];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (i0 + u < sup.n) {
            r += x[u][0];
            if (gga)
#pragma unroll
              for (int c = 0; c < 3; ++c) g[c] += x[u][1 + c];
          }
      }
    } else {
      r = pend.dens.rho[y - 1][q];
      if (gga)
        for (int c = 0; c < 3; ++c) g[c] = pend.dens.grad[y - 1][c * npts + q];
    }
  }
  const bool skip = block_sum_128(fabs(r), red) < B * 1e-12;
  double e = 0.0, vv = 0.0, gg[3] = {0.0, 0.0, 0.0};
  if (in && !skip) e = xc_point(func, r, g[0], g[1], g[2], &vv, gg);
  if (y == 0) {
    const double r2 = in ? rho_act[q] : 0.0;
    const bool skip2 = block_sum_128(fabs(r2), red) < B * 1e-12;
    if (in && !skip2) {
      double v2 = 0.0, g2[3] = {0.0, 0.0, 0.0};
      e -= xc_point(func, r2, gga ? grad_act[q] : 0.0, gga ? grad_act[npts + q] : 0.0,
                    gga ? grad_act[2 * npts + q] : 0.0, &v2, g2);
      vv -= v2;
      for (int c = 0; c < 3; ++c) gg[c] -= g2[c];
    }
  }
  const double wq = in ? w[q] : 0.0;
  if (in && y == 0) {
    vs[q] = wq * vv;
    for (int c = 0; c < 3; ++c) gw[c * npts + q] = wq * gg[c];
  }
  const double eb = block_sum_128(wq * e, red);
  if (t == 0) (y == 0 ? e_blk : pend.eblk[y - 1])[b] = eb;
}

// out = sum of e_blk (null: out itself) - env.e[0] - env.e[1] ..., where an entry with block
// energies first becomes their sum (kept where e is given); every thread of the workgroup calls it.
// red: 256 + kListMax.
__device__ void nadd_energy(const double* e_blk, int64_t n, const EnvEnergies& env, double* out, double* red) {
  double* known = red + 256;
  const int t = threadIdx.x;
  if (t < env.n && !env.eblk[t]) known[t] = env.e[t][0];
  double e = e_blk ? sum_256(e_blk, n, nullptr, 0, red) : out[0];
  __syncthreads();
  for (int i = 0; i < env.n; ++i) {
    double x = known[i];
    if (env.eblk[i]) {
      x = sum_256(env.eblk[i], n, nullptr, 0, red);
      if (t == 0 && env.e[i]) env.e[i][0] = x;
      __syncthreads();
    }
    e -= x;
  }
  if (t == 0) out[0] = e;
}
__global__ __launch_bounds__(256) void nadd_energy_kernel(const double* __restrict__ e_blk, int64_t n, EnvEnergies env,
                                                          double* __restrict__ out) {
  __shared__ double red[256 + kListMax];
  nadd_energy(e_blk, n, env, out, red);
}

// Unrestricted functional on 128-point blocks: spin densities and gradients in,
// w v_s and w g_s (the Fock kernel's inputs) per spin and the block energies out.
// The block is skipped when both spin densities are negligible (sum |rho_s| <
// B 1e-12 for each spin), as the reference's for_spin test does.
__global__ __launch_bounds__(128) void functional_pol_kernel(int func, int64_t npts, int bs,
                                                             const double* __restrict__ ra,
                                                             const double* __restrict__ ga,
                                                             const double* __restrict__ rb,
                                                             const double* __restrict__ gb,
                                                             const double* __restrict__ w, double* __restrict__ vsa,
                                                             double* __restrict__ gwa, double* __restrict__ vsb,
                                                             double* __restrict__ gwb, double* __restrict__ e_blk,
                                                             const double* __restrict__ ra2,
                                                             const double* __restrict__ ga2,
                                                             const double* __restrict__ rb2,
                                                             const double* __restrict__ gb2,
                                                             const DevBlock* __restrict__ blocks,
                                                             const double* __restrict__ part_a,
                                                             const double* __restrict__ part_b) {
  __shared__ double red[128];
  const int b = blockIdx.x, t = threadIdx.x;
  const int64_t first = (int64_t)b * bs;
  const int B = (int)min((int64_t)bs, npts - first);
  const int64_t q = first + t;
  const bool in = t < B;
  const bool gga = functional_is_gga(func);
  double a = 0.0, bb = 0.0;
  double xa[3] = {0.0, 0.0, 0.0}, xb[3] = {0.0, 0.0, 0.0};
  if (in && part_a) {
    // sum the density passes of this block (blocks of 128 points)
    const int np = blocks[b].npass;
    for (int s = 0; s < np; ++s) {
      const int64_t o = (int64_t)s * 4 * npts + q;
      a += part_a[o];
      bb += part_b[o];
      if (gga)
        for (int c = 0; c < 3; ++c) {
          xa[c] += part_a[o + (c + 1) * npts];
          xb[c] += part_b[o + (c + 1) * npts];
        }
    }
    for (int c = 0; c < 3; ++c) {
      xa[c] *= 2.0;
      xb[c] *= 2.0;
    }
  } else if (in) {
    a = ra[q];
    bb = rb[q];
    if (gga)
      for (int c = 0; c < 3; ++c) {
        xa[c] = ga[c * npts + q];
        xb[c] = gb[c * npts + q];
      }
  }
  const bool skip_a = block_sum_128(fabs(a), red) < B * 1e-12;
  const bool skip_b = block_sum_128(fabs(bb), red) < B * 1e-12;
  double e = 0.0, v[2] = {0.0, 0.0}, g[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (in && !(skip_a && skip_b)) e = xc_point_pol(func, a, bb, xa, xb, v, g);
  if (ra2) {
    // non-additive form: the same functional of a second pair of spin densities is subtracted
    // (its own block skip applies to it)
    const double a2 = in ? ra2[q] : 0.0, b2 = in ? rb2[q] : 0.0;
    double ya[3] = {0.0, 0.0, 0.0}, yb[3] = {0.0, 0.0, 0.0};
    if (in && gga)
      for (int c = 0; c < 3; ++c) {
        ya[c] = ga2[c * npts + q];
        yb[c] = gb2[c * npts + q];
      }
    const bool skip2_a = block_sum_128(fabs(a2), red) < B * 1e-12;
    const bool skip2_b = block_sum_128(fabs(b2), red) < B * 1e-12;
    if (in && !(skip2_a && skip2_b)) {
      double v2[2] = {0.0, 0.0}, g2[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      e -= xc_point_pol(func, a2, b2, ya, yb, v2, g2);
      v[0] -= v2[0];
      v[1] -= v2[1];
      for (int c = 0; c < 6; ++c) g[c] -= g2[c];
    }
  }
  const double wq = in ? w[q] : 0.0;
  if (in && vsa) {
    vsa[q] = wq * v[0];
    vsb[q] = wq * v[1];
    if (gga)
      for (int c = 0; c < 3; ++c) {
        gwa[c * npts + q] = wq * g[c];
        gwb[c * npts + q] = wq * g[3 + c];
      }
  }
  const double eb = block_sum_128(wq * e, red);
  if (t == 0) e_blk[b] = eb;
}

// Sub-tile Fock contraction.  One workgroup of W wavefronts per work item; the
// item's 16 x 16 AO sub-tiles (i, j) are dealt to the wavefronts round-robin,
// S per wavefront, each accumulating S_ij = phi_i^T G_j + G_i^T phi_j over the
// block's 128 points in registers (dummy slots of a short item compute on row
// 0 and are dropped).  The points stream in chunks of KC (32 FP32 / 16 FP64,
// one 128-byte line of each AO row): the global loads of a chunk (along the
// point axis of the AO-major tiles) are issued a chunk or two before its MFMAs,
// and a chunk is turned into phi and G = (w v / 2) phi + sum_k (w g_k) d_k phi
// rows of LDS on its way in.  Inside a chunk, k-step t of lane group g takes
// point KV g + t (KV = KC / 4), so each MFMA operand of a chunk is one 32-byte
// LDS read of KV consecutive points of one AO row.
// One kernel per workgroup shape, with one slot count each: an item's wavefronts stop at the slots
// they hold, so a shape's smaller items lose nothing but the registers of the widest (FP64 at 5
// slots spills 4; one kernel of 5 slots for every wide item was 2 to 3 % slower at (H2O)64 and 32).
// One: without gradient terms both products of an element are the same sum phi_i (w v / 2) phi_j, so
// FP64 takes one of them with w v (FP32 keeps both: its rounding would differ).
template <typename T, int W, int Rows, int S, bool One>
__global__ __launch_bounds__(64 * W) void fock_sub_kernel(const FockItem* __restrict__ work,
                                                       const DevBlock* __restrict__ blocks,
                                                       const T* __restrict__ tiles,
                                                       const double* __restrict__ vs, const double* __restrict__ gw,
                                                       int gga, double thr, T* __restrict__ Tscr, int64_t npts,
                                                       const PackSys* __restrict__ pack, int pairs) {
  using M = Mfma<T>;
  constexpr int KC = 128 / (int)sizeof(T);       // points per chunk: one 128-byte line of each AO row
  constexpr int KV = KC / 4;
  constexpr int RS = KC + 16 / (int)sizeof(T);  // 144-byte LDS rows: the 16 rows of an operand read hit distinct banks
  constexpr int NCH = kTile / KC;
  constexpr int NT = 64 * W;                     // threads
  constexpr int NTASK = Rows * 4 / NT;
  static_assert(NTASK * NT == Rows * 4, "whole staging tasks");
  typedef T vec_t __attribute__((ext_vector_type(KV)));
  // Two LDS buffers, one barrier per chunk.  FP32 stages chunk c + 1 after the MFMAs of chunk c
  // (4.25 -> 4.09 ms at (H2O)64/def2-TZVP against one buffer); FP64 stages it in the instruction
  // stream of the MFMAs of slot 0 of chunk c, from registers loaded one chunk earlier (6.22 -> 5.88
  // ms; the same order measured no faster in FP32).
  __shared__ __attribute__((aligned(16))) T sPhi2[2][Rows][RS];
  __shared__ __attribute__((aligned(16))) T sG2[2][Rows][RS];
  // w v / 2, w g_x, w g_y, w g_z of each point in the contraction type, one plane per quantity:
  // the four point runs a wavefront reads at once then start on distinct banks
  __shared__ __attribute__((aligned(16))) T spot[4][kTile];
  __shared__ double red[2];

  int spin;
  const int item = pair_item(pairs, blockIdx.x, spin);
  if (pairs && item >= pairs) return;
  const FockItem it = work[item];
  const DevBlock bk = blocks[it.block];
  if (pack) {
    const PackSys& ps = pack[bk.sys + spin];
    tiles = static_cast<const T*>(ps.tiles);
    vs = ps.vs;
    gw = ps.gw;
    Tscr = static_cast<T*>(ps.T);
    npts = ps.npts;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int npad = bk.npad;
  const bool diag = it.nb == 0;
  const int R = it.na + it.nb;
  const gmem<const T>* tb = to_global(tiles + bk.tile_off);
  const int64_t cstride = (int64_t)npad * kTile;
  vec_t raw[NTASK][4];
  if constexpr (sizeof(T) == 8) {  // LDA leaves the gradient components zero (the FP64 staging uses them)
#pragma unroll
    for (int m = 0; m < NTASK; ++m)
#pragma unroll
      for (int k = 1; k < 4; ++k) raw[m][k] = vec_t(T(0));
  }
  auto grow_of = [&](int lr) { return lr < it.na ? it.a0 + lr : it.b0 + (lr - it.na); };
  // staging task -> (row, quarter of the chunk): 16 consecutive lanes take 16 rows of one
  // quarter, so their 16-byte LDS stores (144-byte row stride) cover distinct banks
  const int q = (tid >> 4) & 3;
  auto row_of = [&](int task) { return (task & 15) + 16 * (task >> 6); };
  auto load = [&](int c) {
    const int p0 = c * KC;
#pragma unroll
    for (int m = 0; m < NTASK; ++m) {
      const int task = tid + NT * m;
      if (task < 4 * R) {
        // one 32-bit byte offset per lane from the planes' wavefront-uniform bases (a 64-bit address
        // per plane and task took the registers that made the widest FP64 items spill)
        const unsigned off = (unsigned)((grow_of(row_of(task)) * kTile + p0 + KV * q) * (int)sizeof(T));
        auto plane = [&](int k) {
          return *reinterpret_cast<const gmem<const vec_t>*>(reinterpret_cast<const gmem<const char>*>(tb + k * cstride) +
                                                             off);
        };
        raw[m][0] = plane(0);
        if (gga) {
          raw[m][1] = plane(1);
          raw[m][2] = plane(2);
          raw[m][3] = plane(3);
        }
      }
    }
  };
  load(0);  // in flight while the potentials are staged and the block skip is decided
  if (tid < kTile) {
    const bool in = tid < bk.npts;
    const int64_t q = bk.first + tid;
    const gmem<const double>* vsg = to_global(vs);
    const gmem<const double>* gwg = to_global(gw);
    const double v0 = in ? vsg[q] : 0.0;
    const double v1 = (in && gga) ? gwg[q] : 0.0;
    const double v2 = (in && gga) ? gwg[npts + q] : 0.0;
    const double v3 = (in && gga) ? gwg[2 * npts + q] : 0.0;
    spot[0][tid] = (T)(One ? v0 : 0.5 * v0);
    spot[1][tid] = (T)v1;
    spot[2][tid] = (T)v2;
    spot[3][tid] = (T)v3;
    double a = fabs(v0) + fabs(v1) + fabs(v2) + fabs(v3);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a += __shfl_down(a, off, 64);
    if (lane == 0) red[w] = a;
  }
  __syncthreads();


  // sub-tile t of the item -> (i, j) in 16-row units (i <= j on a diagonal item)
  auto decode = [&](int t, int& i, int& j) {
    i = 0;
    if (diag) {
      const int nt = it.na / 16;
      int start = 0;
      while (start + (nt - i) <= t) {
        start += nt - i;
        ++i;
      }
      j = i + (t - start);
    } else {
      const int ntb = it.nb / 16;
      i = t / ntb;
      j = t - i * ntb;
    }
  };
  // a skipped block (every item of it takes the same decision from the same values) leaves zeros
  // in its sub-tiles, so the reduce needs no per-block test
  if ((red[0] + red[1]) / bk.npts < thr) {
    gmem<T>* out0 = to_global(Tscr + bk.toff);
    for (int t = w; t < it.nsub; t += W) {
      int i, j;
      decode(t, i, j);
      const int I = it.a0 / 16 + i, J = (diag ? it.a0 : it.b0) / 16 + j;
      gmem<T>* sub = out0 + fock_row_start(16 * I, npad) + 16 * (J - I);
      for (int e = lane; e < 256; e += 64) sub[(int64_t)(e >> 4) * (npad - 16 * I) + (e & 15)] = T(0);
    }
    return;
  }
  // this wavefront's sub-tiles as LDS row offsets (wavefront-uniform)
  int li[S], lj[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int t = w + W * s;
    int i = 0, j = 0;
    if (t < it.nsub) decode(t, i, j);
    li[s] = __builtin_amdgcn_readfirstlane(t < it.nsub ? 16 * i : 0);
    lj[s] = __builtin_amdgcn_readfirstlane(t < it.nsub ? (diag ? 16 * j : it.na + 16 * j) : 0);
  }

  auto store = [&](int c) {
    T(*sPhi)[RS] = sPhi2[c & 1];
    T(*sG)[RS] = sG2[c & 1];
    // the KV points of this thread's tasks are the same for every task; their potentials are
    // read as whole vectors, the GGA test taken once (a test per value branches around each
    // LDS read and waits for it)
    const int p0 = c * KC + KV * q;
    vec_t gv[NTASK];
    auto pot = [&](int k) { return *reinterpret_cast<const vec_t*>(&spot[k][p0]); };
    const vec_t w0 = pot(0);
    if (gga) {
      const vec_t w1 = pot(1), w2 = pot(2), w3 = pot(3);
#pragma unroll
      for (int m = 0; m < NTASK; ++m)
#pragma unroll
        for (int e = 0; e < KV; ++e)
          gv[m][e] = w0[e] * raw[m][0][e] + w1[e] * raw[m][1][e] + w2[e] * raw[m][2][e] + w3[e] * raw[m][3][e];
    } else {
#pragma unroll
      for (int m = 0; m < NTASK; ++m)
#pragma unroll
        for (int e = 0; e < KV; ++e) gv[m][e] = w0[e] * raw[m][0][e];
    }
#pragma unroll
    for (int m = 0; m < NTASK; ++m) {
      const int task = tid + NT * m;
      if (task < 4 * R) {
        const int lr = row_of(task);
        *reinterpret_cast<vec_t*>(&sPhi[lr][KV * q]) = raw[m][0];
        *reinterpret_cast<vec_t*>(&sG[lr][KV * q]) = gv[m];
      }
    }
  };

  typename M::acc_t acc[S];
#pragma unroll
  for (int s = 0; s < S; ++s) acc[s] = M::zero();
  const int r = lane & 15, g = lane >> 4;
  // slots of this wavefront that hold a sub-tile (an item smaller than its class leaves the rest idle)
  const int slive = it.nsub > w ? (it.nsub - w + W - 1) / W : 0;
  auto slot = [&](int s, T(*sPhi)[RS], T(*sG)[RS]) {
    const vec_t aP = *reinterpret_cast<const vec_t*>(&sPhi[li[s] + r][KV * g]);
    const vec_t bG = *reinterpret_cast<const vec_t*>(&sG[lj[s] + r][KV * g]);
    if constexpr (One) {
#pragma unroll
      for (int t = 0; t < KV; ++t) acc[s] = M::step(aP[t], bG[t], acc[s]);
    } else {
      const vec_t aG = *reinterpret_cast<const vec_t*>(&sG[li[s] + r][KV * g]);
      const vec_t bP = *reinterpret_cast<const vec_t*>(&sPhi[lj[s] + r][KV * g]);
#pragma unroll
      for (int t = 0; t < KV; ++t) acc[s] = M::step(aP[t], bG[t], acc[s]);
#pragma unroll
      for (int t = 0; t < KV; ++t) acc[s] = M::step(aG[t], bP[t], acc[s]);
    }
  };
  if constexpr (sizeof(T) == 8) {
    static_assert((NCH & (NCH - 1)) == 0, "chunks per item: a power of two");
    // Staging without branches, so that the compiler can spread it between the MFMAs of slot 0:
    // G takes all four terms (LDA's gradient potentials and components are zero), tasks beyond
    // the item's rows write rows that no MFMA reads, and chunk NCH re-stages chunk 0 into the
    // buffer no later chunk reads.
    auto store_flat = [&](int c) {
      T(*sPhi)[RS] = sPhi2[c & 1];
      T(*sG)[RS] = sG2[c & 1];
      const int p0 = (c & (NCH - 1)) * KC + KV * q;
      const vec_t w0 = *reinterpret_cast<const vec_t*>(&spot[0][p0]);
      const vec_t w1 = *reinterpret_cast<const vec_t*>(&spot[1][p0]);
      const vec_t w2 = *reinterpret_cast<const vec_t*>(&spot[2][p0]);
      const vec_t w3 = *reinterpret_cast<const vec_t*>(&spot[3][p0]);
#pragma unroll
      for (int m = 0; m < NTASK; ++m) {
        vec_t gv;
#pragma unroll
        for (int e = 0; e < KV; ++e)
          gv[e] = w0[e] * raw[m][0][e] + w1[e] * raw[m][1][e] + w2[e] * raw[m][2][e] + w3[e] * raw[m][3][e];
        const int lr = row_of(tid + NT * m);
        *reinterpret_cast<vec_t*>(&sPhi[lr][KV * q]) = raw[m][0];
        *reinterpret_cast<vec_t*>(&sG[lr][KV * q]) = gv;
      }
    };
    store_flat(0);
    if (NCH > 1) load(1);
    __syncthreads();
    for (int c = 0; c < NCH; ++c) {
      T(*sPhi)[RS] = sPhi2[c & 1];
      T(*sG)[RS] = sG2[c & 1];
      slot(0, sPhi, sG);  // every wavefront (an idle one computes on row 0 and drops the result)
      store_flat(c + 1);
      if (c + 2 < NCH) load(c + 2);
#pragma unroll
      for (int s = 1; s < S; ++s) {
        if (s >= slive) break;  // wavefront-uniform
        slot(s, sPhi, sG);
        // keep one slot's operands live at a time (bounds the register file)
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
    }
  } else {
    store(0);
    __syncthreads();
    for (int c = 0; c < NCH; ++c) {
      T(*sPhi)[RS] = sPhi2[c & 1];
      T(*sG)[RS] = sG2[c & 1];
      if (c + 1 < NCH) load(c + 1);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (s >= slive) break;  // wavefront-uniform
        slot(s, sPhi, sG);
        // keep one slot's operands live at a time (bounds the register file)
        __builtin_amdgcn_sched_barrier(0);
      }
      if (c + 1 < NCH) store(c + 1);
      __syncthreads();
    }
  }

  // store the sub-tiles (block sub-tile (I, J), I <= J; 16 lanes write 16 consecutive values of a row)
  gmem<T>* tb_out = to_global(Tscr + bk.toff);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int t = w + W * s;
    if (t >= it.nsub) continue;
    int i, j;
    decode(t, i, j);
    const int I = it.a0 / 16 + i, J = (diag ? it.a0 : it.b0) / 16 + j;
    gmem<T>* sub = tb_out + fock_row_start(16 * I, npad) + 16 * (J - I) + r;
    const int stride = npad - 16 * I;
#pragma unroll
    for (int e = 0; e < 4; ++e) sub[(int64_t)M::row(lane, e) * stride] = acc[s][e];
  }
}

// One AO row i of the Fock accumulator per workgroup: its entries (the blocks holding AO i, in
// block order) are dealt to groups of Group lanes round-robin; a group adds each entry's
// stored row segment into the workgroup's LDS copy of the row, and the row is written once to
// U[j + n i], j >= i.  Each lane takes an aligned group of four columns (4 Group per step):
// one 16-byte load of their AO indices and one of their stored values, the lanes of a group
// reading one contiguous run of the block's stored row (a block's AO list is padded to
// a multiple of 32 with -1 and its stored row a runs from column 16 (a / 16) to the padded end,
// so an aligned group never leaves either; the columns of the group before the segment start are
// masked).  A group walks its entries' steps as one sequence: while a step's values are added, the
// next step's loads and the entry after it are in flight.  What bounds the kernel is the latency of
// that chain, so short chains (many groups) count: segments hold n_b / 2 columns on average (12 to
// 170), which left most of a wavefront's 64 lanes idle when a whole wavefront took an entry.  Groups
// of 16 against whole wavefronts: (H2O)8/def2-SVP 40 -> 21 us, C20H42/def2-SVP 90 -> 76 us (FP64);
// groups of 32 for blocks of more than 256 AOs on average.  Wavefronts / 32 / 16 lanes in us, FP64 and
// FP32: (H2O)64/def2-TZVP (n_b 337) 1007 / 935 / 992 and 792 / 678 / 703, (H2O)32/def2-TZVP (276)
// 375 / 325 / 337 and 307 / 244 / 241, (H2O)64/def2-SVP (210) 663 / 534 / 529 and 572 / 427 / 392;
// the best order per precision crosses at an n_b of about 200 in FP64 and 300 in FP32.  (The kernel of
// whole wavefronts that broadcast their entries from the lanes took 923 and 681 at (H2O)64, 355 and
// 280 at (H2O)32.)
// Rows longer than the LDS window are done in several passes over the entries.
// Fixed = false: FP64 additions in LDS, which the wavefronts make in an order that varies from run
// to run, so F varies at the rounding level.  Fixed = true: each term x is split into integers,
// x = h 2^-32 + l 2^-72 + e with h = x 2^32 and l = (x - h 2^-32) 2^72 rounded to the nearest
// integer, |l| <= 2^39 and |e| <= 2^-73, and h and l are added into two 64-bit integer sums per
// column; integer sums do not depend on the order, so F is the same bit for bit on every run (and
// the sum is exact up to the e terms).  The rounding adds 1.5 2^20 (1.5 2^52) in FP64, whose unit
// in the last place is then 2^-32 (1), and reads the integer from the bit pattern.  Valid for
// terms of |x| < 2^19 in columns of fewer than 2^23 terms whose absolute values sum to less than
// 2^30.
template <typename T, bool Fixed, int Group>
__global__ __launch_bounds__(64 * kReduceWaves) void fock_reduce_kernel(const RowEnt* __restrict__ ent,
                                                                        const int* __restrict__ row_ptr,
                                                                        const T* __restrict__ Tscr,
                                                                        const int* __restrict__ ao_idx,
                                                                        double* __restrict__ U, int n, int window,
                                                                        const PackSys* __restrict__ pack,
                                                                        ReduceOut out, EnvEnergies env) {
  extern __shared__ unsigned long long racc_u[];  // window (FP64 sums) or 2 window (Fixed: h, then l sums)
  double* racc = reinterpret_cast<double*>(racc_u);
  if (pack) {
    const PackSys& ps = pack[blockIdx.y];
    ent = ps.ent;
    row_ptr = ps.row_ptr;
    Tscr = static_cast<const T*>(ps.T);
    ao_idx = ps.ao_idx;
    U = ps.U;
    n = ps.n;
    if (out.direct) {
      out.F = ps.F;
      out.P = ps.P64;
      out.P32 = out.round ? ps.P32 : nullptr;
      out.round = ps.round;
      out.eblk = ps.eblk;
      out.nxc = ps.nxc;
      out.E = ps.E;
    }
  }
  const int i = blockIdx.x;
  const int tid = threadIdx.x;
  if (i >= n) {  // uniform over the workgroup
    if (i == n && out.direct && out.E) {
      nadd_energy(out.eblk, out.nxc, env, out.E, reinterpret_cast<double*>(racc_u));
    }
    return;
  }
  double c_round = 0.0;
  const gmem<const RowEnt>* entg = to_global(ent);
  const gmem<const T>* Tg = to_global(Tscr);
  const gmem<const int>* idxg = to_global(ao_idx);
  const int e0 = to_global(row_ptr)[i], e1 = to_global(row_ptr)[i + 1];
  for (int w0 = 0; w0 < n - i; w0 += window) {
    const int wl = min(window, n - i - w0);
    for (int k = tid; k < wl; k += 64 * kReduceWaves) {
      if constexpr (Fixed) {
        racc_u[k] = 0;
        racc_u[window + k] = 0;
      } else {
        racc[k] = 0.0;
      }
    }
    __syncthreads();
    // the group's entries e0 + grp + kGroups k; E: the entry of the step in flight, N: the one after it
    constexpr int kGroups = 64 * kReduceWaves / Group;
    const int gl = tid & (Group - 1);
    int k = e0 + tid / Group;
    RowEnt E = {0, 0, 0, 0, 0}, N = {0, 0, 0, 0, 0};
    if (k < e1) E = load_global(entg + k);
    if (k + kGroups < e1) N = load_global(entg + k + kGroups);
    int c = (E.c0 & ~3) + 4 * gl, base = E.c0 & ~3;
    i32x4 gi = {-1, -1, -1, -1};
    T v[4] = {T(0), T(0), T(0), T(0)};
    auto fetch = [&]() {  // the four columns of this lane in the current step, columns outside [c0, c1) masked
      gi = i32x4{-1, -1, -1, -1};
      if (k < e1 && c < E.c1) {
        gi = *reinterpret_cast<const gmem<const i32x4>*>(idxg + E.idx_off + c);
        const gmem<const T>* src = Tg + E.rowbase + c;
        if constexpr (sizeof(T) == 4) {
          const f32x4 f = *reinterpret_cast<const gmem<const f32x4>*>(src);
          v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
        } else {
          const f64x2 f0 = *reinterpret_cast<const gmem<const f64x2>*>(src);
          const f64x2 f1 = *reinterpret_cast<const gmem<const f64x2>*>(src + 2);
          v[0] = f0.x; v[1] = f0.y; v[2] = f1.x; v[3] = f1.y;
        }
      }
    };
    fetch();
    while (__any(k < e1)) {
      // this step's values, then the next step's loads, then the additions
      const i32x4 ga = gi;
      const double x[4] = {(double)v[0], (double)v[1], (double)v[2], (double)v[3]};
      const int lo = E.c0 - c, hi = E.c1 - c;
      base += 4 * Group;
      if (base >= E.c1) {  // the same for the lanes of a group
        k += kGroups;
        E = N;
        if (k + kGroups < e1) N = load_global(entg + k + kGroups);
        base = E.c0 & ~3;
      }
      c = base + 4 * gl;
      fetch();
      const int gg[4] = {ga.x, ga.y, ga.z, ga.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int g = gg[u] - i - w0;
        if (u >= lo && u < hi && g >= 0 && g < wl) {
          if constexpr (Fixed) {
            const double t = x[u] + 0x1.8p20;
            const long long h = __double_as_longlong(t) - __double_as_longlong(0x1.8p20);
            const double rem = x[u] - (t - 0x1.8p20);  // exact, |rem| <= 2^-33
            const long long l = __double_as_longlong(rem * 0x1p72 + 0x1.8p52) - __double_as_longlong(0x1.8p52);
            atomicAdd(racc_u + g, (unsigned long long)h);
            atomicAdd(racc_u + window + g, (unsigned long long)l);
          } else {
            atomicAdd(racc + g, x[u]);
          }
        }
      }
    }
    __syncthreads();
    for (int j = tid; j < wl; j += 64 * kReduceWaves) {
      double f;
      if constexpr (Fixed)
        f = (double)(long long)racc_u[j] * 0x1p-32 + (double)(long long)racc_u[window + j] * 0x1p-72;
      else
        f = racc[j];
      const int64_t lo = (int64_t)(i + w0 + j) + (int64_t)n * i;
      if (out.direct) {
        // both triangles of F, and the row's part of the FP32 rounding term (P is read first: a
        // caller's F may be its P)
        const int64_t up = i + (int64_t)n * (i + w0 + j);
        if (out.P32) {
          c_round += f * (to_global(out.P)[lo] - (double)to_global(out.P32)[lo]);
          if (lo != up) c_round += f * (to_global(out.P)[up] - (double)to_global(out.P32)[up]);
        }
        to_global(out.F)[lo] = f;
        if (lo != up) to_global(out.F)[up] = f;
      } else {
        to_global(U)[lo] = f;
      }
    }
    __syncthreads();
  }
  if (out.direct && out.P32) {
    double* red = reinterpret_cast<double*>(racc_u);  // one per wavefront (the host asks for that much LDS)
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) c_round += __shfl_xor(c_round, m);
    if ((tid & 63) == 0) red[tid >> 6] = c_round;
    __syncthreads();
    if (tid == 0) {
      double s = 0.0;
      for (int v = 0; v < kReduceWaves; ++v) s += red[v];
      out.round[i] = s;
    }
  }
}

__global__ void weight_potential_kernel(int64_t npts, const double* __restrict__ w, const double* __restrict__ v,
                                        const double* __restrict__ g, double* __restrict__ vs,
                                        double* __restrict__ gw) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npts) return;
  vs[q] = w[q] * v[q];
  if (g) {
    gw[q] = w[q] * g[q];
    gw[npts + q] = w[q] * g[npts + q];
    gw[2 * npts + q] = w[q] * g[2 * npts + q];
  }
}

// rho[q] = sum_i list.rho[i][q] in list order (likewise the gradient); rho itself may be listed.
__global__ void sum_densities_kernel(DensityList list, int64_t npts, int want_grad, double* rho, double* grad) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npts) return;
  double r = 0.0;
  for (int i = 0; i < list.n; ++i) r += list.rho[i][q];
  rho[q] = r;
  if (want_grad) {
    for (int c = 0; c < 3; ++c) {
      double g = 0.0;
      for (int i = 0; i < list.n; ++i) g += list.grad[i][c * npts + q];
      grad[c * npts + q] = g;
    }
  }
}

__global__ void copy_kernel(const double4* __restrict__ src, double4* __restrict__ dst, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

__global__ void fill_kernel(double* __restrict__ p, int64_t n, double value) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

// Q = P + P^T, on the diagonal P, of one matrix or of the systems of a pack whose P is their U (P64 into U).
constexpr int kFoldTile = 32;
__global__ __launch_bounds__(256) void fold_kernel(const double* __restrict__ P, double* __restrict__ Q, int n,
                                                   const PackSys* __restrict__ pack) {
  __shared__ double t[kFoldTile][kFoldTile + 1];
  if (pack) {
    const PackSys& ps = pack[blockIdx.z];
    if (ps.P != ps.U) return;
    P = ps.P64;
    Q = ps.U;
    n = ps.n;
  }
  const int i0 = blockIdx.x * kFoldTile, j0 = blockIdx.y * kFoldTile, x = threadIdx.x & 31, y0 = threadIdx.x >> 5;
  if (i0 >= n || j0 >= n) return;  // uniform over the workgroup
  for (int y = y0; y < kFoldTile; y += 8)
    t[y][x] = j0 + x < n && i0 + y < n ? P[(j0 + x) + (int64_t)n * (i0 + y)] : 0.0;
  __syncthreads();
  for (int y = y0; y < kFoldTile; y += 8) {
    const int i = i0 + x, j = j0 + y;
    if (i < n && j < n) {
      const double p = P[i + (int64_t)n * j];
      Q[i + (int64_t)n * j] = i == j ? p : p + t[x][y];
    }
  }
}

__global__ void to_float_kernel(const double* __restrict__ s, float* __restrict__ d, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = (float)s[i];
}

// F = mirror of the lower-triangle accumulator U (or F += it).  With P32 given, each block
// also leaves sum_e F[e] (P[e] - P32[e]) in part[blockIdx.x]: the first-order change of
// E_xc from the FP32-rounded density matrix P32 back to P, since dE_xc/dP = F.
__global__ __launch_bounds__(256) void finalize_kernel(const double* __restrict__ U, double* __restrict__ F, int n,
                                                       int accumulate, const double* __restrict__ P,
                                                       const float* __restrict__ P32, double* __restrict__ part) {
  const int t = threadIdx.x;
  const int64_t e = (int64_t)blockIdx.x * 256 + t;
  double c = 0.0;
  if (e < (int64_t)n * n) {
    const int i = (int)(e % n), j = (int)(e / n);
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    const double u = U[hi + (int64_t)n * lo];
    const double f = accumulate ? F[e] + u : u;
    F[e] = f;
    if (P32) c = f * (P[e] - (double)P32[e]);
  }
  if (!P32) return;  // uniform over the launch
  __shared__ double red[256];
  red[t] = c;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (t < k) red[t] += red[t + k];
    __syncthreads();
  }
  if (t == 0) part[blockIdx.x] = red[0];
}

// sum of x[0..n) and x2[0..n2); mode 0: out = sum; 1: out -= sum
__global__ __launch_bounds__(256) void sum_kernel(const double* __restrict__ x, int64_t n,
                                                  const double* __restrict__ x2, int64_t n2, double* __restrict__ out,
                                                  int mode) {
  __shared__ double red[256];
  const double s = sum_256(x, n, x2, n2, red);
  if (threadIdx.x == 0) out[0] = mode == 0 ? s : out[0] - s;
}

// ---- packed builds: elementwise stages over the systems of a pack (blockIdx.y = system) ----
__global__ void pack_to_float_kernel(const PackSys* __restrict__ pack) {
  const PackSys& ps = pack[blockIdx.y];
  const int64_t nn = (int64_t)ps.n * ps.n;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nn; i += (int64_t)gridDim.x * blockDim.x)
    ps.P32[i] = (float)ps.P64[i];
}

// F = mirror of U; FP32 builds also leave one partial of sum F (P - P32) per workgroup
__global__ __launch_bounds__(256) void pack_finalize_kernel(const PackSys* __restrict__ pack, int fp32) {
  const PackSys& ps = pack[blockIdx.y];
  const int n = ps.n, t = threadIdx.x;
  const int64_t nn = (int64_t)n * n;
  double c = 0.0;
  for (int64_t e = (int64_t)blockIdx.x * 256 + t; e < nn; e += (int64_t)gridDim.x * 256) {
    const int i = (int)(e % n), j = (int)(e / n);
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    const double u = ps.U[hi + (int64_t)n * lo];
    ps.F[e] = u;
    if (fp32) c += u * (ps.P64[e] - (double)ps.P32[e]);
  }
  if (!fp32) return;  // uniform over the launch
  __shared__ double red[256];
  red[t] = c;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (t < k) red[t] += red[t + k];
    __syncthreads();
  }
  if (t == 0) ps.round[blockIdx.x] = red[0];
}

// E_xc of each system: its block energies and nround partials of the FP32 rounding term (one per
// AO row for nround < 0), in a fixed order
__global__ __launch_bounds__(256) void pack_sum_kernel(const PackSys* __restrict__ pack, int nround) {
  const PackSys& ps = pack[blockIdx.x];
  __shared__ double red[256];
  const double s = sum_256(ps.eblk, ps.nxc, ps.round, nround < 0 ? ps.n : nround, red);
  if (threadIdx.x == 0) ps.E[0] = s;
}

inline unsigned grid1d(int64_t n, int bsz) { return (unsigned)((n + bsz - 1) / bsz); }

}  // namespace

void launch_screen(hipStream_t s, const double* pts, int64_t npts, int bs, int nblocks, const DevShell* shells,
                   int nshell, const double* alpha, const double* coef, double radial_thr, int* pos, int* count) {
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(screen_kernel, dim3(nblocks), dim3(64), 0, s, pts, npts, bs, shells, nshell, alpha, coef,
                     radial_thr, pos, count);
}

int row_chunks(int nblocks) { return (nblocks + kRowChunk - 1) / kRowChunk; }

void launch_block_lists(hipStream_t s, const DevBlock* blocks, int nblocks, const DevShell* shells, int nshell, int nao,
                        const int* pos, int* sig_shell, int* sig_pos, int* ao_idx, int* cnt, int* row_ptr,
                        RowEnt* ent) {
  if (nblocks <= 0) return;
  const dim3 chunks(row_chunks(nblocks), (nshell + 255) / 256);
  hipLaunchKernelGGL(block_lists_kernel, dim3(nblocks), dim3(64), 0, s, blocks, shells, nshell, pos, sig_shell, sig_pos,
                     ao_idx);
  hipLaunchKernelGGL(row_count_kernel, chunks, dim3(256), 0, s, pos, nblocks, nshell, cnt);
  hipLaunchKernelGGL(row_offsets_kernel, dim3(1), dim3(1024), 0, s, shells, nshell, (int)chunks.x, nao, cnt, row_ptr);
  hipLaunchKernelGGL(row_entries_kernel, chunks, dim3(256), 0, s, blocks, nblocks, shells, nshell, pos, cnt, row_ptr,
                     ent);
}

void launch_ao_eval(hipStream_t s, const DevBlock* blocks, int nblocks, int max_nshell, const int* sig_shell,
                    const int* sig_pos, const DevShell* shells, const double* alpha, const double* coef, const double* ang,
                    const double* pts, double radial_thr, double exp_thr, int ncomp, double* t64, float* t32) {
  if (nblocks <= 0 || max_nshell <= 0) return;
  hipLaunchKernelGGL(ao_kernel, dim3(nblocks, (max_nshell + kAoShells - 1) / kAoShells), dim3(kTile), 0, s, blocks,
                     sig_shell, sig_pos, shells, alpha, coef, ang, pts, radial_thr, exp_thr, ncomp, t64, t32);
}

template <typename T>
void launch_density_sub(hipStream_t s, const WorkItem* work, int nwork, const DevBlock* blocks, const int* ao_idx,
                        const T* tiles, const T* P, int n, int want_grad, double* part, int64_t npts,
                        const PackSys* pack, const int* nwork_dev, const unsigned char* skip, bool form,
                        bool pairs) {
  if (nwork <= 0) return;
  const DensityArgs<T> arg = {ao_idx, tiles, P, n, want_grad, part, npts};
  const dim3 grid(pairs ? (nwork + 7) / 8 * 16 : nwork);
  const int np = pairs ? nwork : 0;
  if (sizeof(T) == 8 && form)
    hipLaunchKernelGGL((density_sub_kernel<T, sizeof(T) == 8>), grid, dim3(512), 0, s, work, blocks, arg, pack,
                       nwork_dev, skip, np);
  else
    hipLaunchKernelGGL((density_sub_kernel<T, false>), grid, dim3(512), 0, s, work, blocks, arg, pack, nwork_dev,
                       skip, np);
}
template void launch_density_sub<double>(hipStream_t, const WorkItem*, int, const DevBlock*, const int*, const double*,
                                         const double*, int, int, double*, int64_t, const PackSys*, const int*,
                                         const unsigned char*, bool, bool);
template void launch_density_sub<float>(hipStream_t, const WorkItem*, int, const DevBlock*, const int*, const float*,
                                        const float*, int, int, double*, int64_t, const PackSys*, const int*,
                                        const unsigned char*, bool, bool);

// Largest density of block b (128 threads), from the partials of its passes.
__device__ double block_max_density(const DevBlock& bk, int64_t npts, const double* __restrict__ part, double* red) {
  const int t = threadIdx.x;
  double r = 0.0;
  if (t < bk.npts)
    for (int s = 0; s < bk.npass; ++s) r += part[(int64_t)s * 4 * npts + bk.first + t];
  red[t] = r;
  __syncthreads();
  for (int k = 64; k > 0; k >>= 1) {
    if (t < k) red[t] = fmax(red[t], red[t + k]);
    __syncthreads();
  }
  return red[0];
}

// Blocks whose largest density (from the partials of a first pass) exceeds rho_thr have their
// density work items appended to the list, for a second pass.  With a
// mask, only the blocks outside it are tested (the first pass skipped the others) and the listed
// ones join it.
__global__ __launch_bounds__(128) void mark_dense_kernel(const DevBlock* __restrict__ blocks, int64_t npts,
                                                         const double* __restrict__ part, double rho_thr,
                                                         const WorkItem* __restrict__ by_block,
                                                         const int* __restrict__ item0, DenseList list,
                                                         unsigned char* __restrict__ mask) {
  __shared__ double red[128];
  const int b = blockIdx.x, t = threadIdx.x;
  if (mask && mask[b]) return;  // uniform over the workgroup
  const DevBlock bk = blocks[b];
  const bool dense = bk.npass > 0 && block_max_density(bk, npts, part, red) > rho_thr;
  if (t == 0 && dense) {
    const int pos = atomicAdd(list.count, bk.npass);
    for (int k = 0; k < bk.npass; ++k) list.item[pos + k] = by_block[item0[b] + k];
    if (mask) mask[b] = 1;
  }
}

// The density work items of the blocks in the mask, appended to the list.
__global__ __launch_bounds__(64) void list_masked_kernel(const DevBlock* __restrict__ blocks, int nblocks,
                                                         const WorkItem* __restrict__ by_block,
                                                         const int* __restrict__ item0, DenseList list,
                                                         const unsigned char* __restrict__ mask) {
  const int b = blockIdx.x * 64 + threadIdx.x;
  if (b >= nblocks || !mask[b]) return;
  const int np = blocks[b].npass;
  if (np <= 0) return;
  const int pos = atomicAdd(list.count, np);
  for (int k = 0; k < np; ++k) list.item[pos + k] = by_block[item0[b] + k];
}

// After the second pass: a listed block stays in the mask while its density exceeds rho_thr.
__global__ __launch_bounds__(128) void refresh_dense_kernel(const DevBlock* __restrict__ blocks, int64_t npts,
                                                            const double* __restrict__ part, double rho_thr,
                                                            unsigned char* __restrict__ mask) {
  __shared__ double red[128];
  const int b = blockIdx.x;
  if (!mask[b]) return;  // uniform over the workgroup
  const DevBlock bk = blocks[b];
  const bool dense = block_max_density(bk, npts, part, red) > rho_thr;
  if (threadIdx.x == 0) mask[b] = dense ? 1 : 0;
}

__global__ void clear_counts_kernel(int* __restrict__ c, int n) {
  if ((int)threadIdx.x < n) c[threadIdx.x] = 0;
}

__global__ void to_double_kernel(const float* __restrict__ s, double* __restrict__ d, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = (double)s[i];
}

void launch_mark_dense(hipStream_t s, const DevBlock* blocks, int nblocks, int64_t npts, const double* part,
                       double rho_thr, const WorkItem* by_block, const int* item0, const DenseList& list,
                       unsigned char* mask) {
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(clear_counts_kernel, dim3(1), dim3(64), 0, s, list.count, 1);
  hipLaunchKernelGGL(mark_dense_kernel, dim3(nblocks), dim3(128), 0, s, blocks, npts, part, rho_thr, by_block, item0,
                     list, mask);
}

void launch_list_masked(hipStream_t s, const DevBlock* blocks, int nblocks, const WorkItem* by_block,
                        const int* item0, const DenseList& list, const unsigned char* mask) {
  hipLaunchKernelGGL(clear_counts_kernel, dim3(1), dim3(64), 0, s, list.count, 1);
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(list_masked_kernel, dim3((nblocks + 63) / 64), dim3(64), 0, s, blocks, nblocks, by_block, item0,
                     list, mask);
}

void launch_refresh_dense(hipStream_t s, const DevBlock* blocks, int nblocks, int64_t npts, const double* part,
                          double rho_thr, unsigned char* mask) {
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(refresh_dense_kernel, dim3(nblocks), dim3(128), 0, s, blocks, npts, part, rho_thr, mask);
}

void launch_to_double(hipStream_t s, const float* src, double* dst, int64_t n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(to_double_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, dst, n);
}

void launch_reduce_partials(hipStream_t s, const DevBlock* blocks, int bs, int64_t npts, const double* part,
                            int want_grad, double* rho, double* grad, int accumulate) {
  if (npts <= 0) return;
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(grid1d(npts, 256)), dim3(256), 0, s, blocks, bs, npts, part,
                     want_grad, rho, grad, accumulate);
}

void launch_functional(hipStream_t s, int func, int64_t npts, int bs, const double* rho,
                       const double* grad, const DevBlock* blocks, const double* part, const double* w, double* eps,
                       double* v, double* g, double* vs, double* gw, double* e_blk) {
  const int nb = (int)((npts + bs - 1) / bs);
  if (nb <= 0) return;
  hipLaunchKernelGGL(functional_kernel, dim3(nb), dim3(128), 0, s, func, npts, bs, rho, grad, blocks, part, w,
                     eps, v, g, vs, gw, e_blk, (const PackSys*)nullptr);
}

void launch_functional_packed(hipStream_t s, int func, int nblocks, const DevBlock* blocks,
                              const PackSys* pack) {
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(functional_kernel, dim3(nblocks), dim3(128), 0, s, func, (int64_t)0, kTile,
                     (const double*)nullptr, (const double*)nullptr, blocks, (const double*)nullptr,
                     (const double*)nullptr, (double*)nullptr, (double*)nullptr, (double*)nullptr, (double*)nullptr,
                     (double*)nullptr, (double*)nullptr, pack);
}

static unsigned pack_grid(int64_t maxnn) {
  const int64_t g = (maxnn + 255) / 256;
  return (unsigned)(g < 1 ? 1 : g > 1024 ? 1024 : g);
}

__global__ void set_pair_kernel(PackPair pair, PackSys* __restrict__ out) {
  if (threadIdx.x < 2) out[threadIdx.x] = pair.s[threadIdx.x];
}
void launch_set_pair(hipStream_t s, const PackPair& pair, PackSys* out) {
  hipLaunchKernelGGL(set_pair_kernel, dim3(1), dim3(64), 0, s, pair, out);
}

void launch_pack_to_float(hipStream_t s, const PackSys* pack, int nsys, int64_t maxnn) {
  if (nsys <= 0) return;
  hipLaunchKernelGGL(pack_to_float_kernel, dim3(pack_grid(maxnn), nsys), dim3(256), 0, s, pack);
}

void launch_pack_finalize(hipStream_t s, const PackSys* pack, int nsys, int fp32) {
  if (nsys <= 0) return;
  hipLaunchKernelGGL(pack_finalize_kernel, dim3(kPackRoundBlocks, nsys), dim3(256), 0, s, pack, fp32);
}

void launch_pack_sum(hipStream_t s, const PackSys* pack, int nsys, int nround) {
  if (nsys <= 0) return;
  hipLaunchKernelGGL(pack_sum_kernel, dim3(nsys), dim3(256), 0, s, pack, nround);
}

void launch_functional_pol(hipStream_t s, int func, int64_t npts, int bs, const double* ra,
                           const double* ga, const double* rb, const double* gb, const double* w, double* vsa,
                           double* gwa, double* vsb, double* gwb, double* e_blk, const double* ra2,
                           const double* ga2, const double* rb2, const double* gb2, const DevBlock* blocks,
                           const double* part_a, const double* part_b) {
  const int nb = (int)((npts + bs - 1) / bs);
  if (nb <= 0) return;
  hipLaunchKernelGGL(functional_pol_kernel, dim3(nb), dim3(128), 0, s, func, npts, bs, ra, ga, rb, gb, w, vsa,
                     gwa, vsb, gwb, e_blk, ra2, ga2, rb2, gb2, blocks, part_a, part_b);
}

template <typename T>
void launch_fock_sub(hipStream_t s, int shape, const FockItem* work, int nwork, const DevBlock* blocks, const T* tiles,
                     const double* vs, const double* gw, int gga, double thr, T* Tscr, int64_t npts,
                     const PackSys* pack, bool pairs) {
  if (nwork <= 0) return;
  constexpr bool f64 = sizeof(T) == 8;
  const dim3 grid(pairs ? (nwork + 7) / 8 * 16 : nwork);
  const int np = pairs ? nwork : 0;
#define SXC_FOCK_SHAPE(k)                                                                                             \
  if (shape == k) {                                                                                                   \
    constexpr FockShape sh = kFockShape[k];                                                                           \
    if (f64 && !gga)                                                                                                  \
      hipLaunchKernelGGL((fock_sub_kernel<T, sh.waves, sh.rows, sh.slots, f64>), grid, dim3(64 * sh.waves), 0, s,     \
                         work, blocks, tiles, vs, gw, gga, thr, Tscr, npts, pack, np);                                \
    else                                                                                                              \
      hipLaunchKernelGGL((fock_sub_kernel<T, sh.waves, sh.rows, sh.slots, false>), grid, dim3(64 * sh.waves), 0, s,   \
                         work, blocks, tiles, vs, gw, gga, thr, Tscr, npts, pack, np);                                \
    return;                                                                                                           \
  }
  static_assert(kFockShapes == 4, "one case per shape");
  SXC_FOCK_SHAPE(0)
  SXC_FOCK_SHAPE(1)
  SXC_FOCK_SHAPE(2)
  SXC_FOCK_SHAPE(3)
#undef SXC_FOCK_SHAPE
  throw std::runtime_error("launch_fock_sub: unknown workgroup shape");
}
template void launch_fock_sub<double>(hipStream_t, int, const FockItem*, int, const DevBlock*, const double*,
                                      const double*, const double*, int, double, double*, int64_t, const PackSys*,
                                      bool);
template void launch_fock_sub<float>(hipStream_t, int, const FockItem*, int, const DevBlock*, const float*,
                                     const double*, const double*, int, double, float*, int64_t, const PackSys*, bool);

// Row columns per LDS pass of the reduce: kReduceWindow, or less where the device's LDS per
// workgroup cannot hold that many columns of 8 bytes (fixed = false) or 16 bytes (fixed = true).
static int reduce_window_limit(bool fixed) {
  static int cached[2][64] = {};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev < 0 || dev >= 64) dev = 0;
  if (!cached[fixed][dev]) {
    int lds = 65536;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) lds = 65536;
    const int w = lds / (fixed ? 16 : 8);
    cached[fixed][dev] = (w < kReduceWindow ? w : kReduceWindow) / 64 * 64;
  }
  return cached[fixed][dev];
}

template <typename T, bool Fixed>
static void launch_fock_reduce_f(hipStream_t s, const RowEnt* ent, const int* row_ptr, const T* Tscr,
                                 const int* ao_idx, double* U, int n, const PackSys* pack, int nsys, bool wide,
                                 const ReduceOut& out, const EnvEnergies& env) {
  const int lim = reduce_window_limit(Fixed);
  const int window = n < lim ? n : lim;
  size_t lds = (Fixed ? 16 : 8) * (size_t)window;
  // one workgroup more for the energy sum, whose terms need LDS (the rounding term's 16 less)
  const dim3 grid(n + (out.direct && (out.E || pack) ? 1 : 0), nsys);
  if (out.direct) lds = std::max(lds, (256 + kListMax) * sizeof(double));
  if (wide)
    hipLaunchKernelGGL((fock_reduce_kernel<T, Fixed, 32>), grid, dim3(64 * kReduceWaves), lds, s, ent, row_ptr, Tscr,
                       ao_idx, U, n, window, pack, out, env);
  else
    hipLaunchKernelGGL((fock_reduce_kernel<T, Fixed, 16>), grid, dim3(64 * kReduceWaves), lds, s, ent, row_ptr, Tscr,
                       ao_idx, U, n, window, pack, out, env);
}

template <typename T>
void launch_fock_reduce(hipStream_t s, const RowEnt* ent, const int* row_ptr, const T* Tscr, const int* ao_idx,
                        double* U, int n, const PackSys* pack, int nsys, bool fixed, bool wide,
                        const ReduceOut& out, const EnvEnergies& env) {
  if (n <= 0 || nsys <= 0) return;
  if (fixed)
    launch_fock_reduce_f<T, true>(s, ent, row_ptr, Tscr, ao_idx, U, n, pack, nsys, wide, out, env);
  else
    launch_fock_reduce_f<T, false>(s, ent, row_ptr, Tscr, ao_idx, U, n, pack, nsys, wide, out, env);
}
template void launch_fock_reduce<double>(hipStream_t, const RowEnt*, const int*, const double*, const int*, double*,
                                         int, const PackSys*, int, bool, bool, const ReduceOut&,
                                         const EnvEnergies&);
template void launch_fock_reduce<float>(hipStream_t, const RowEnt*, const int*, const float*, const int*, double*,
                                        int, const PackSys*, int, bool, bool, const ReduceOut&,
                                         const EnvEnergies&);

void launch_weight_potential(hipStream_t s, int64_t npts, const double* w, const double* v, const double* g,
                             double* vs, double* gw) {
  if (npts <= 0) return;
  hipLaunchKernelGGL(weight_potential_kernel, dim3(grid1d(npts, 256)), dim3(256), 0, s, npts, w, v, g, vs, gw);
}

void launch_sum_densities(hipStream_t s, const DensityList& list, int64_t npts, int want_grad, double* rho,
                          double* grad) {
  if (npts <= 0) return;
  hipLaunchKernelGGL(sum_densities_kernel, dim3(grid1d(npts, 256)), dim3(256), 0, s, list, npts, want_grad, rho, grad);
}

void launch_nadd_functional(hipStream_t s, int func, int64_t npts, bool potential,
                            const DensityList& sup, const double* rho_act, const double* grad_act,
                            const DensityList& pending, double* const* pending_eblk, const double* w, double* vs,
                            double* gw, double* e_blk) {
  if (npts <= 0 || (!potential && pending.n == 0)) return;
  PendingEnergies pend{};
  pend.dens = pending;
  for (int i = 0; i < pending.n; ++i) pend.eblk[i] = pending_eblk[i];
  hipLaunchKernelGGL(nadd_functional_kernel, dim3(grid1d(npts, kTile), (potential ? 1 : 0) + pending.n), dim3(kTile), 0,
                     s, func, npts, potential ? 0 : 1, sup, rho_act, grad_act, pend, w, vs, gw, e_blk);
}

void launch_nadd_energy(hipStream_t s, const double* e_blk, int64_t n, const EnvEnergies& env, double* out) {
  hipLaunchKernelGGL(nadd_energy_kernel, dim3(1), dim3(256), 0, s, e_blk, n, env, out);
}

void launch_copy(hipStream_t s, const void* src, void* dst, int64_t n32) {
  if (n32 <= 0) return;
  hipLaunchKernelGGL(copy_kernel, dim3(grid1d(n32, 256)), dim3(256), 0, s, (const double4*)src, (double4*)dst, n32);
}

void launch_fill(hipStream_t s, double* p, int64_t n, double value) {
  if (n <= 0) return;
  hipLaunchKernelGGL(fill_kernel, dim3(grid1d(n, 256)), dim3(256), 0, s, p, n, value);
}

void launch_fold(hipStream_t s, const double* P, double* Q, int n, const PackSys* pack, int nsys) {
  if (n <= 0 || nsys <= 0) return;
  const unsigned g = grid1d(n, kFoldTile);
  hipLaunchKernelGGL(fold_kernel, dim3(g, g, nsys), dim3(256), 0, s, P, Q, n, pack);
}

void launch_to_float(hipStream_t s, const double* src, float* dst, int64_t n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(to_float_kernel, dim3(grid1d(n, 256)), dim3(256), 0, s, src, dst, n);
}

void launch_finalize(hipStream_t s, const double* U, double* F, int n, int accumulate, const double* P,
                     const float* P32, double* part) {
  const int64_t nn = (int64_t)n * n;
  if (nn <= 0) return;
  hipLaunchKernelGGL(finalize_kernel, dim3(grid1d(nn, 256)), dim3(256), 0, s, U, F, n, accumulate, P, P32, part);
}

int finalize_blocks(int n) { return (int)grid1d((int64_t)n * n, 256); }

void launch_sum(hipStream_t s, const double* x, int64_t n, double* out, int subtract, const double* x2, int64_t n2) {
  hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(256), 0, s, x, n, x2, n2, out, subtract);
}

}  // namespace sxc
