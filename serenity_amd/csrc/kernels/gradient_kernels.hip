// XC contribution to the nuclear gradient at a fixed grid
// (FuncPotential::getGeomGradients, src/potentials/FuncPotential.cpp:113-239).
//
// For an AO nu on atom A and direction c the reference accumulates, over the
// block's points and the block's AOs mu,
//   grad[A][c] -= 2 P_mu,nu sum_p w v phi_mu d_c phi_nu
//   (GGA)      -= 2 P_mu,nu sum_p w sum_k g_k (phi_mu d_k d_c phi_nu + d_k phi_mu d_c phi_nu).
// With G_mu(p) = w v phi_mu + sum_k w g_k d_k phi_mu and H^c_nu(p) = sum_k w g_k d_k d_c phi_nu
// this is grad[A][c] = -2 sum_{nu on A} a^c_nu with
//   a^c_nu = sum_p (G P)_p,nu d_c phi_nu(p) + (phi P)_p,nu H^c_nu(p),
// i.e. two dense products per block (phi_b P_b and G_b P_b, FP64 matrix cores) and
// column dots against the gradient and Hessian tiles.  Nothing n x n is scattered:
// each work item adds 3 numbers per AO column into a[nu][c].
#include <hip/hip_runtime.h>

#include "mfma.h"
#include "xc_internal.h"

namespace sxc {

namespace {

// Sum over the 16 lanes of a lane group (rotations within the group).
template <int Ctrl>
__device__ __forceinline__ double row_rotate_add(double x) {
  int2 w = __builtin_bit_cast(int2, x), o;
  o.x = __builtin_amdgcn_update_dpp(0, w.x, Ctrl, 0xf, 0xf, false);
  o.y = __builtin_amdgcn_update_dpp(0, w.y, Ctrl, 0xf, 0xf, false);
  return x + __builtin_bit_cast(double, o);
}
__device__ __forceinline__ double row16_sum(double x) {
  x = row_rotate_add<0x128>(x);  // row_ror:8
  x = row_rotate_add<0x124>(x);
  x = row_rotate_add<0x122>(x);
  return row_rotate_add<0x121>(x);
}

constexpr int kGradKC = 16;                // AOs per chunk
constexpr int kGradRS = kGradKC + 2;       // 144-byte LDS rows: the 16 rows of an operand read hit distinct banks
constexpr int kGradRows = 2 * kTile + 16 * kDensMaxS;  // phi, G and P columns

// One workgroup of 16 wavefronts per (block, pass of 16 S columns): wavefront w owns points
// 16 (w % 8) .. + 15 and half w / 8 of the column tiles of both phi P and G P.  What bounds it is the
// FP64 matrix cores, 2 x 2 B n_b ncols operations per pass, and the latency of its loads; one workgroup
// per compute unit (LDS), so the AOs stream in chunks of 16 through two LDS
// buffers with one barrier a chunk: the next chunk is loaded before the chunk's MFMAs and stored
// after them, G formed from the value and gradient tiles on its way.  The accumulators are transposed
// (rows: AO columns, columns: points), so that the column dots read 16 consecutive points of a
// tile row.  At C8H18/def2-TZVP/PBE the kernel takes 0.84 ms (1.00 with 8 wavefronts of all S column
// tiles: 214 registers, two wavefronts per SIMD; 2.57 with 4 wavefronts per 64 columns, one buffer and
// one element per LDS read).  The ten planes of a block and the four staged again per pass come at
// about 3 TB/s, the matrix cores are busy 0.31 ms.
template <int S>
__device__ __forceinline__ void gradient_item(const WorkItem& wk, const DevBlock& bk, const int* __restrict__ ao_idx,
                                              const double* __restrict__ tiles, const double* __restrict__ P, int n,
                                              const double* __restrict__ vs, const double* __restrict__ gw, int gga,
                                              int64_t npts, double* __restrict__ acc,
                                              double (*buf)[kGradRows][kGradRS], double (*spot)[kTile],
                                              double (*red)[16 * kDensMaxS][3]) {
  using M = Mfma<double>;
  constexpr int KC = kGradKC, KV = KC / 4, EV = KC / 8, NP = (16 * S + 63) / 64, HS = (S + 1) / 2;
  typedef double vec_t __attribute__((ext_vector_type(KV)));
  typedef double stage_t __attribute__((ext_vector_type(EV)));
  const int col0 = wk.a, ncols = wk.b;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6) & 7;
  const int c0 = HS * __builtin_amdgcn_readfirstlane(tid >> 9);  // the wavefront's first column tile
  const int r = lane & 15, g = lane >> 4;
  const gmem<const double>* tb = to_global(tiles + bk.tile_off);
  const int64_t cs = (int64_t)bk.npad * kTile;
  const gmem<const int>* idx = to_global(ao_idx + bk.idx_off);
  const gmem<const double>* Pg = to_global(P);
  // staging: point pa, AO pair qa of phi and G; P elements (AO tid % 16, columns tid / 16 + 64 m)
  const int pa = tid & (kTile - 1), qa = tid >> 7, ka = tid & 15;
  double vp = 0.0, gx = 0.0, gy = 0.0, gz = 0.0;
  if (pa < bk.npts) {
    const int64_t q = bk.first + pa;
    vp = to_global(vs)[q];
    if (gga) {
      gx = to_global(gw)[q];
      gy = to_global(gw)[npts + q];
      gz = to_global(gw)[2 * npts + q];
    }
  }
  if (tid < kTile) {
    spot[0][tid] = gx;
    spot[1][tid] = gy;
    spot[2][tid] = gz;
  }
  int nu[NP];
#pragma unroll
  for (int m = 0; m < NP; ++m) {
    const int c = (tid >> 4) + 64 * m;
    nu[m] = c < ncols ? idx[col0 + c] : -1;
  }
  const int kend = (bk.nb + KC - 1) / KC * KC;  // whole chunks: at most npad, whose last AOs are zero
  double ph[EV], dx[EV], dy[EV], dz[EV], rp[NP];
#pragma unroll
  for (int e = 0; e < EV; ++e) dx[e] = dy[e] = dz[e] = 0.0;
  int mu = idx[ka], mu_now = mu;
  auto load = [&](int k0) {
    mu_now = mu;
#pragma unroll
    for (int m = 0; m < NP; ++m) rp[m] = Pg[max(mu, 0) + (int64_t)n * max(nu[m], 0)];
    if (k0 + KC < kend) mu = idx[k0 + KC + ka];  // the next chunk's P addresses depend on no load of it
#pragma unroll
    for (int e = 0; e < EV; ++e) {
      const int64_t o = (int64_t)(k0 + EV * qa + e) * kTile + pa;
      ph[e] = tb[o];
      if (gga) {
        dx[e] = tb[cs + o];
        dy[e] = tb[2 * cs + o];
        dz[e] = tb[3 * cs + o];
      }
    }
  };
  auto store = [&](int b) {
    stage_t f, h;
#pragma unroll
    for (int e = 0; e < EV; ++e) {
      f[e] = ph[e];
      h[e] = vp * ph[e] + gx * dx[e] + gy * dy[e] + gz * dz[e];
    }
    *reinterpret_cast<stage_t*>(&buf[b][pa][EV * qa]) = f;
    *reinterpret_cast<stage_t*>(&buf[b][kTile + pa][EV * qa]) = h;
#pragma unroll
    for (int m = 0; m < NP; ++m) {
      const int c = (tid >> 4) + 64 * m;
      // padding read P[0][0]; a zero for it (a select at the load would wait for it there)
      if (c < 16 * S) buf[b][2 * kTile + c][ka] = mu_now >= 0 && nu[m] >= 0 ? rp[m] : 0.0;
    }
  };
  M::acc_t T[HS], TG[HS];
#pragma unroll
  for (int c = 0; c < HS; ++c) {
    T[c] = M::zero();
    TG[c] = M::zero();
  }
  load(0);
  store(0);
  __syncthreads();
  int b = 0;
  for (int k0 = 0; k0 < kend; k0 += KC, b ^= 1) {
    const bool more = k0 + KC < kend;
    if (more) load(k0 + KC);
    const vec_t af = *reinterpret_cast<const vec_t*>(&buf[b][16 * w + r][KV * g]);
    const vec_t ag = *reinterpret_cast<const vec_t*>(&buf[b][kTile + 16 * w + r][KV * g]);
#pragma unroll
    for (int c = 0; c < HS; ++c) {
      if (c0 + c >= S) break;  // uniform: the last tile of the second half where S is odd
      const vec_t bv = *reinterpret_cast<const vec_t*>(&buf[b][2 * kTile + 16 * (c0 + c) + r][KV * g]);
#pragma unroll
      for (int t = 0; t < KV; ++t) {
        T[c] = M::step(bv[t], af[t], T[c]);
        TG[c] = M::step(bv[t], ag[t], TG[c]);
      }
    }
    if (more) store(b ^ 1);
    __syncthreads();
  }

  // column dots: lane (r, g) holds point 16 w + r of columns 16 c + g + 4 e
  const int p = 16 * w + r;  // rows of points beyond the block are zero in the tiles
  const double wx = spot[0][p], wy = spot[1][p], wz = spot[2][p];
#pragma unroll
  for (int c = 0; c < HS; ++c) {
    if (16 * (c0 + c) >= ncols) break;  // uniform
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int cl = 16 * (c0 + c) + g + 4 * e;
      const gmem<const double>* row = tb + (int64_t)(col0 + cl) * kTile + p;
      const double tg = TG[c][e];
      double ax = tg * row[cs], ay = tg * row[2 * cs], az = tg * row[3 * cs];
      if (gga) {
        const double tv = T[c][e];
        const double hxx = row[4 * cs], hxy = row[5 * cs], hxz = row[6 * cs];
        const double hyy = row[7 * cs], hyz = row[8 * cs], hzz = row[9 * cs];
        ax += tv * (wx * hxx + wy * hxy + wz * hxz);
        ay += tv * (wx * hxy + wy * hyy + wz * hyz);
        az += tv * (wx * hxz + wy * hyz + wz * hzz);
      }
      ax = row16_sum(ax);
      ay = row16_sum(ay);
      az = row16_sum(az);
      if (r == 0) {
        red[w][cl][0] = ax;
        red[w][cl][1] = ay;
        red[w][cl][2] = az;
      }
    }
  }
  __syncthreads();
  if (tid < 3 * ncols) {
    const int cl = tid / 3, c = tid - 3 * cl;
    const int nucol = idx[col0 + cl];
    if (nucol >= 0) {
      double s = 0.0;
#pragma unroll
      for (int v = 0; v < 8; ++v) s += red[v][cl][c];
      atomicAdd(&acc[3 * (int64_t)nucol + c], s);
    }
  }
}

__global__ __launch_bounds__(1024) void gradient_kernel(const WorkItem* __restrict__ work,
                                                       const DevBlock* __restrict__ blocks,
                                                       const int* __restrict__ ao_idx,
                                                       const double* __restrict__ tiles,
                                                       const double* __restrict__ P, int n,
                                                       const double* __restrict__ vs, const double* __restrict__ gw,
                                                       int gga, int64_t npts, double* __restrict__ acc) {
  __shared__ __attribute__((aligned(16))) double buf[2][kGradRows][kGradRS];
  __shared__ double spot[3][kTile];
  __shared__ double red[8][16 * kDensMaxS][3];
  const WorkItem wk = work[blockIdx.x];
  const DevBlock bk = blocks[wk.block];
  static_assert(kDensMaxS == 6 && 3 * 16 * kDensMaxS <= 512, "one case per pass width");
#define SXC_GRAD(S_) \
  case S_:           \
    return gradient_item<S_>(wk, bk, ao_idx, tiles, P, n, vs, gw, gga, npts, acc, buf, spot, red);
  switch ((wk.b + 15) / 16) {
    SXC_GRAD(1)
    SXC_GRAD(2)
    SXC_GRAD(3)
    SXC_GRAD(4)
    SXC_GRAD(5)
    SXC_GRAD(6)
  }
#undef SXC_GRAD
}

// grad[A + natoms c] = -2 sum_{nu : atom(nu) = A} acc[nu][c]: one wavefront per atom, each lane its
// AOs in order, the lanes in a fixed tree.
__global__ __launch_bounds__(64) void gradient_atoms_kernel(const double* __restrict__ acc,
                                                            const int* __restrict__ ao_atom, int n, int natoms,
                                                            double* __restrict__ grad) {
  const int A = blockIdx.x;
  double s[3] = {0.0, 0.0, 0.0};
  for (int nu = threadIdx.x; nu < n; nu += 64)
    if (ao_atom[nu] == A)
      for (int c = 0; c < 3; ++c) s[c] += acc[3 * (int64_t)nu + c];
  for (int c = 0; c < 3; ++c) {
    for (int m = 1; m < 64; m <<= 1) s[c] += __shfl_xor(s[c], m);
    if (threadIdx.x == 0) grad[A + natoms * c] = -2.0 * s[c];
  }
}

}  // namespace

void launch_gradient(hipStream_t s, const WorkItem* work, int nwork, const DevBlock* blocks, const int* ao_idx,
                     const double* tiles, const double* P, int n, const double* vs, const double* gw, int gga,
                     int64_t npts, double* acc) {
  if (nwork <= 0) return;
  hipLaunchKernelGGL(gradient_kernel, dim3(nwork), dim3(1024), 0, s, work, blocks, ao_idx, tiles, P, n, vs, gw, gga,
                     npts, acc);
}

void launch_gradient_atoms(hipStream_t s, const double* acc, const int* ao_atom, int n, int natoms, double* grad) {
  if (natoms <= 0) return;
  hipLaunchKernelGGL(gradient_atoms_kernel, dim3(natoms), dim3(64), 0, s, acc, ao_atom, n, natoms, grad);
}

}  // namespace sxc
