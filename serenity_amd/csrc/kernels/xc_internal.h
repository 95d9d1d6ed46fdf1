// Device-side data layout of the XC Fock build and the kernel launchers shared
// by the C ABI (xc_api.hip) and the kernels (xc_kernels.hip).
//
// HBM layout of the basis-functions-on-grid tiles: the grid is cut into
// blocks of at most 128 consecutive (Hilbert-ordered) points.  Block b keeps
// the n_b AOs that survive Serenity's shell screening, padded to npad (a
// multiple of 32) and stored as ncomp component planes
//   tiles[tile_off + (c * npad + i) * 128 + p],  c = value, d/dx, d/dy, d/dz
// (and, for highest derivative 2, d2/dxx, dxy, dxz, dyy, dyz, dzz),
// i = compact AO index (ao_idx maps it to the global AO, -1 for padding),
// p = point within the block (rows beyond the block's size are zero).  Point
// is the fastest index so a wavefront reads 64 consecutive values.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "functional.h"

namespace sxc {

// Global-memory view of a pointer.  A pointer the compiler cannot trace to a kernel argument (one
// taken from a packed build's per-system table, or selected between such a pointer and an
// argument) is generic to it, and accesses through a generic pointer become flat instructions:
// those count against the LDS counter as well as the vector-memory one, so every wait for an LDS
// read then also waits for all global loads in flight.  Accesses through gmem<T>* are global ones.
template <typename T>
using gmem = __attribute__((address_space(1))) T;
template <typename T>
__device__ __forceinline__ gmem<T>* to_global(T* p) {
  return (gmem<T>*)p;
}
// Vector types for 16-byte global loads through gmem pointers (HIP's float4 and the like are
// classes whose copy constructors take generic references).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
// A struct read through a gmem pointer (structs, too, copy only from generic references), in
// 8-byte words.
template <typename S>
__device__ __forceinline__ S load_global(const gmem<const S>* p) {
  static_assert(sizeof(S) % 8 == 0 && alignof(S) >= 8, "8-byte words");
  S out;
  const gmem<const int64_t>* src = reinterpret_cast<const gmem<const int64_t>*>(p);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(S) / 8); ++k) {
    const int64_t w = src[k];
    __builtin_memcpy(reinterpret_cast<char*>(&out) + 8 * k, &w, 8);
  }
  return out;
}

constexpr int kTile = 128;      // points per tile row (max block size)
constexpr int kAoPad = 32;      // AO padding granularity of a block
constexpr int kMaxL = 6;        // highest angular momentum the AO kernel evaluates

struct DevShell {
  double cx, cy, cz;
  int l, pure, nprim, prim_off;
  int ao_off, nfunc, ang_off, ncart;
};

struct DevBlock {
  int64_t tile_off;   // element offset of the block's tiles
  int64_t toff;       // element offset of the block's Fock sub-tiles in the sub-tile scratch
  int64_t first;      // first grid point
  int npts;           // points in the block (<= 128)
  int nb;             // non-negligible AOs
  int npad;           // nb rounded up to kAoPad
  int idx_off;        // offset into ao_idx
  int shell_off;      // offset into the significant-shell list
  int nshell;         // significant shells
  int npass;          // density column passes (partial rho/grad slots written)
  int sys;            // system of a packed build (index into its PackSys table; 0 otherwise)
};

// Fock sub-tiles of a block: the npad / 16 = nt sub-tile rows and columns of its upper
// triangle, (I, J) with I <= J, in the block's slice of the scratch (DevBlock::toff), stored by
// matrix rows: compact row a (in sub-tile row I = a / 16) holds the columns 16 I .. npad - 1 (from
// its diagonal sub-tile on) contiguously, and the 16 rows of sub-tile row I follow those of the
// rows above, starting at element 256 fock_subtile_index(I, I, nt).  The reduce then reads each
// AO row's segment of a block as one contiguous run.
__host__ __device__ inline int64_t fock_subtile_index(int I, int J, int nt) {
  return (int64_t)I * nt - (int64_t)I * (I - 1) / 2 + (J - I);
}
__host__ __device__ inline int64_t fock_subtile_elems(int npad) {
  const int64_t nt = npad / 16;
  return nt * (nt + 1) / 2 * 256;
}
// element of compact row a, column 16 (a / 16), in the block's slice
__host__ __device__ inline int64_t fock_row_start(int a, int npad) {
  const int I = a / 16;
  return 256 * fock_subtile_index(I, I, npad / 16) + (int64_t)(a % 16) * (npad - 16 * I);
}

// One contribution to a row of the Fock matrix: block `block` holds AO `row` at compact position
// c0, and the compact columns c0 .. c1 - 1 (AOs idx[idx_off + c], in increasing global order)
// carry the values F[row][idx[c]] of the block, column c at element rowbase + c of the scratch
// (rowbase = the block's toff + fock_row_start(c0, npad) - 16 (c0 / 16)).
struct RowEnt {
  int64_t rowbase;
  int c0, c1, idx_off, block;
};

// One system of a packed build: several controllers' builds in one launch per
// stage.  Work items index a merged block list whose entries keep their own
// system's offsets (tile_off, first, idx_off) and name the system in DevBlock::sys.
struct PackSys {
  const void* tiles;    // AO tiles in the contraction precision
  const void* P;        // density matrix in the contraction precision
  const double* P64;    // density matrix (FP64)
  float* P32;           // FP32 copy (FP32 builds)
  const int* ao_idx;
  double* part;         // partial densities
  const double* w;      // grid weights
  double* vs;           // w v
  double* gw;           // w g
  double* U;            // Fock accumulator (lower triangle, written by the row reduce)
  void* T;              // Fock sub-tile scratch (contraction precision)
  const RowEnt* ent;    // row entries of the reduce (sorted by row, then block)
  const int* row_ptr;   // n + 1 offsets into ent
  double* F;            // XC matrix out
  double* eblk;         // per-block energies
  double* round;        // rounding-term partials (FP32)
  double* E;            // E_xc out (device or mapped host memory)
  int64_t npts;
  int n;
  int blk0;             // first merged block of this system
  int nxc;              // 128-point tiles of its grid
  int pad_;
};

// Work item of the sub-tile Fock kernel: the block's AO rows [a0, a0 + na)
// (A side) and [b0, b0 + nb) (B side), multiples of 16.  nb == 0 marks a
// diagonal item (B = A, sub-tiles i <= j).  nsub = 16 x 16 sub-tiles.
struct FockItem {
  int block;
  int a0, na;
  int b0, nb;
  int nsub;
};
constexpr int kFockPanel = 128;       // panel height of blocks split into panel pairs
// Workgroup shapes of the sub-tile kernel: wavefronts, rows an item may stage (576 bytes of LDS each),
// 16 x 16 sub-tiles per wavefront, and the widest block (padded AOs) whose triangle is one item of
// the shape; wider blocks are split into pairs of panels, items of kFockPanelShape.  A compute unit
// holds three workgroups of the first shape and one of the others: an item of few rows waits for its
// loads and barriers most of its time, so several run beside each other (26 potentials of the
// embedding sweep over blocks of up to 64 AOs: 67 -> 34 us each in FP64 with 4 wavefronts instead of
// 16 and a compute unit's whole LDS).  Blocks of 96 to 128 AOs in 8 wavefronts, two per compute unit,
// measured no faster (C20H42/def2-SVP 470 against 431 us): there the matrix cores are the bound.
// The others differ in the slots of a wavefront alone, whose registers every item of a kernel holds.
struct FockShape {
  int waves, rows, slots, npad;
};
constexpr int kFockShapes = 4;
constexpr FockShape kFockShape[kFockShapes] = {{4, 64, 3, 64}, {16, 256, 3, 128}, {16, 256, 4, 160}, {16, 256, 5, 192}};
constexpr int kFockPanelShape = 2;
constexpr bool fock_shapes_fit() {
  for (int k = 0; k < kFockShapes; ++k) {
    const int nt = kFockShape[k].npad / 16;
    if (nt * (nt + 1) / 2 > kFockShape[k].waves * kFockShape[k].slots || kFockShape[k].npad > kFockShape[k].rows)
      return false;
  }
  const int np = kFockPanel / 16;
  const FockShape p = kFockShape[kFockPanelShape];
  return 2 * kFockPanel <= p.rows && np * np <= p.waves * p.slots;
}
static_assert(fock_shapes_fit(), "every item's sub-tiles and rows fit its shape");

// Work item of the density kernel: block, a = first column of the pass,
// b = columns of the pass (multiple of 16), pass = partial-density slot.
struct WorkItem {
  int block, a, b, pass;
};

// ---- launchers (xc_kernels.hip) -------------------------------------------
// pos[b nshell + s]: compact position of shell s in block b, -1 where it is negligible; count[2 b],
// count[2 b + 1]: the block's AOs and significant shells.
void launch_screen(hipStream_t s, const double* pts, int64_t npts, int bs, int nblocks, const DevShell* shells,
                   int nshell, const double* alpha, const double* coef, double radial_thr, int* pos, int* count);
// The blocks' lists (from DevBlock's offsets) and the row entries of the reduce; cnt: scratch of
// row_chunks(nblocks) x nshell.
int row_chunks(int nblocks);
void launch_block_lists(hipStream_t s, const DevBlock* blocks, int nblocks, const DevShell* shells, int nshell, int nao,
                        const int* pos, int* sig_shell, int* sig_pos, int* ao_idx, int* cnt, int* row_ptr,
                        RowEnt* ent);

// max_nshell: the most significant shells of any block
void launch_ao_eval(hipStream_t s, const DevBlock* blocks, int nblocks, int max_nshell, const int* sig_shell,
                    const int* sig_pos,
                    const DevShell* shells, const double* alpha, const double* coef, const double* ang,
                    const double* pts, double radial_thr, double exp_thr, int ncomp, double* tiles64, float* tiles32);

// Sub-tile density kernel: 8 wavefronts per pass of at most 16 kDensMaxS columns.
// Partial densities: part[(pass * 4 + c) * npts + q], c = rho, d/dx, d/dy, d/dz
// (gradient slots hold sum T grad phi without the factor 2).
constexpr int kDensMaxS = 6;
// Mixed precision: blocks whose largest density (bohr^-3) after the FP32 density pass exceeds
// this are contracted again in FP64 (the cores of the heavy atoms, where FP32 rounding of the AO
// values and of phi P gives a bias that does not cancel over the grid).
constexpr double kMixedRhoThreshold = 2.0;
constexpr int kDensIdxLds = 2048;  // AO index lists up to this length are staged in LDS
// With nwork_dev, the launch covers a list filled on the device: only its first *nwork_dev
// items run (nwork is the list's capacity).  form (FP64, no gradient): P is the folded matrix of
// launch_fold, and the density is its quadratic form.
template <typename T>
void launch_density_sub(hipStream_t s, const WorkItem* work, int nwork, const DevBlock* blocks, const int* ao_idx,
                        const T* tiles, const T* P, int n, int want_grad, double* part, int64_t npts,
                        const PackSys* pack = nullptr, const int* nwork_dev = nullptr,
                        const unsigned char* skip = nullptr, bool form = false, bool pairs = false);

// Dense-block refinement of the mixed-precision density: a work list and its device-side count, filled
// by launch_mark_dense.
struct DenseList {
  WorkItem* item;
  int* count;
};
// Clears the count, then appends the density items of every block whose largest density in the
// partials part (one pass per item, 128-point blocks) exceeds rho_thr; by_block holds every block's
// items contiguously from item0[b] (blocks[b].npass of them).
// With a mask (one byte per block: the blocks the first pass skipped because the previous build
// found them dense), only the blocks outside it are tested and the listed ones join it;
// launch_list_masked lists the mask's own blocks (before the first pass, so that their second pass
// can run beside it), and launch_refresh_dense, after the second passes, keeps in the mask only the
// blocks whose density from them still exceeds rho_thr.
void launch_mark_dense(hipStream_t s, const DevBlock* blocks, int nblocks, int64_t npts, const double* part,
                       double rho_thr, const WorkItem* by_block, const int* item0, const DenseList& list,
                       unsigned char* mask = nullptr);
void launch_list_masked(hipStream_t s, const DevBlock* blocks, int nblocks, const WorkItem* by_block,
                        const int* item0, const DenseList& list, const unsigned char* mask);
void launch_refresh_dense(hipStream_t s, const DevBlock* blocks, int nblocks, int64_t npts, const double* part,
                          double rho_thr, unsigned char* mask);
void launch_to_double(hipStream_t s, const float* src, double* dst, int64_t n);

// rho[q] / grad[.][q] from the partials of the block of q (any block size).
void launch_reduce_partials(hipStream_t s, const DevBlock* blocks, int bs, int64_t npts, const double* part,
                            int want_grad, double* rho, double* grad, int accumulate = 0);

// Functional on rho/grad, or (part != nullptr) on the partials of 128-point blocks.
void launch_functional(hipStream_t s, int func, int64_t npts, int bs, const double* rho,
                       const double* grad, const DevBlock* blocks, const double* part, const double* w, double* eps,
                       double* v, double* g, double* vs, double* gw, double* e_blk);
// Functional of a packed build: one 128-point block per workgroup over the merged block list.
void launch_functional_packed(hipStream_t s, int func, int nblocks, const DevBlock* blocks,
                              const PackSys* pack);

// Unrestricted functional: spin densities/gradients (3 x npts each) in; w v_s, w g_s and
// block energies out.
void launch_functional_pol(hipStream_t s, int func, int64_t npts, int bs, const double* ra,
                           const double* ga, const double* rb, const double* gb, const double* w, double* vsa,
                           double* gwa, double* vsb, double* gwb, double* e_blk,
                           const double* ra2 = nullptr, const double* ga2 = nullptr, const double* rb2 = nullptr,
                           const double* gb2 = nullptr, const DevBlock* blocks = nullptr,
                           const double* part_a = nullptr, const double* part_b = nullptr);

// Sub-tile Fock kernel over items of one workgroup shape.
// Each item stores its sub-tiles of phi^T G + G^T phi into the block's scratch slice Tscr + toff
// (zeros when the block-average test skips the block).
template <typename T>
void launch_fock_sub(hipStream_t s, int shape, const FockItem* work, int nwork, const DevBlock* blocks, const T* tiles,
                     const double* vs, const double* gw, int gga, double block_ave_thr, T* Tscr, int64_t npts,
                     const PackSys* pack = nullptr, bool pairs = false);
constexpr int kListMax = 32;  // entries of the lists passed by value (kernel arguments)
// Energies subtracted from a non-additive energy, with the block energies of those still to be summed.
struct EnvEnergies {
  double* e[kListMax];
  const double* eblk[kListMax];
  int n;
};
// U[j + n i] = sum over the row entries of AO i (block order) of the stored sub-tile values at
// columns j >= i, for every i of [0, n): the lower triangle of the Fock accumulator, each element
// written once (its terms meet in LDS in an order that varies from run to run).  Packed:
// blockIdx.y = system, n = the largest n.  16 wavefronts per row: each group's entries form a chain
// of dependent load-add steps, and more wavefronts make shorter chains (with whole wavefronts per
// entry 0.68 ms at (H2O)64/def2-TZVP against 0.86 ms with 8 and 1.40 ms with 4).  wide: blocks hold
// more than 256 AOs on average, so that a row segment (half of them on average) fills the 128
// columns that 32 lanes take at once; else 16 lanes take an entry (both sides: fock_reduce_kernel).
// With out.direct the rows go to both triangles of F instead (no finalize), each row leaves its part of
// the FP32 rounding term sum F (P - P32) in round[row] where P32 is given (packed: where round is
// not null), and one more workgroup sums the block energies into E, less the energies of env (a
// rounding sum, where there is one, is launch_sum's).  For matrices of up to kDirectRows rows: the
// upper triangle's writes go one element per line (n^2 / 2 of them), which costs less than the
// finalize's launch only while they are few.  Whole builds of def2-SVP waters, PBE, direct / not, in us:
// FP32 192 rows 210 / 216, 384 rows 465 / 468, 480 rows 606 / 606, 648 rows 963 / 959; FP64, where the
// energy's launch goes too, 293 / 304, 682 / 692, 894 / 906 and 1452 / 1463.
struct ReduceOut {
  bool direct;
  double* F;
  const double* P;
  const float* P32;
  double* round;
  const double* eblk;
  int nxc;
  double* E;
};
constexpr int kDirectRows = 512;
constexpr int kReduceWaves = 16;
constexpr int kReduceWindow = 8192;  // row columns accumulated in LDS per pass
template <typename T>
void launch_fock_reduce(hipStream_t s, const RowEnt* ent, const int* row_ptr, const T* Tscr, const int* ao_idx,
                        double* U, int n, const PackSys* pack = nullptr, int nsys = 1, bool fixed = false,
                        bool wide = false, const ReduceOut& out = ReduceOut{}, const EnvEnergies& env = EnvEnergies{});
// The two spins of an unrestricted build as a pack of two systems on one controller: launches with pairs
// run each work item once per spin, with entry block.sys + spin of the table.  The table goes to the
// device as a kernel argument, so that a caller's captured build keeps its own.
struct PackPair {
  PackSys s[2];
};
void launch_set_pair(hipStream_t s, const PackPair& pair, PackSys* out);
// Packed elementwise stages over nsys systems (maxnn = largest n^2): P -> FP32,
// F = mirror of U (+ FP32 rounding partials), E = sum of block energies (+ rounding term).
constexpr int kPackRoundBlocks = 512;  // finalize workgroups per system of a packed build
void launch_pack_to_float(hipStream_t s, const PackSys* pack, int nsys, int64_t maxnn);
void launch_pack_finalize(hipStream_t s, const PackSys* pack, int nsys, int fp32);
void launch_pack_sum(hipStream_t s, const PackSys* pack, int nsys, int nround);

// a[nu][c] += sum over the points of a density work item's block of (G P)_p,nu d_c phi_nu +
// (phi P)_p,nu H^c_nu for the item's columns nu (kernels/gradient_kernels.hip); tiles need 4 planes
// (LDA) or 10 (GGA).
void launch_gradient(hipStream_t s, const WorkItem* work, int nwork, const DevBlock* blocks, const int* ao_idx,
                     const double* tiles, const double* P, int n, const double* vs, const double* gw, int gga,
                     int64_t npts, double* acc);
// grad[A + natoms c] = -2 sum_{nu on A} acc[nu][c].
void launch_gradient_atoms(hipStream_t s, const double* acc, const int* ao_atom, int n, int natoms, double* grad);

// ---- density-fitted Coulomb matrix (kernels/coulomb_kernels.hip) ----------
// One significant primitive pair (a of shell A, b of shell B, A >= B) of the orbital basis:
// p = a + b, K = c_a c_b exp(-a b / p |AB|^2), centre P, P - A, P - B; sym = 2 for A > B
// (the pair stands for both orders), 1 for A == B; herm_off: offset of its (L + 1)(L + 2)(L + 3) / 6
// Hermite coefficients (L = l_A + l_B) in the per-pair arrays.
struct JPair {
  int A, B, L, herm_off;
  double sym, p, K;
  double P[3], PA[3], PB[3];
};
constexpr int kJMaxLPrim = 3;                      // orbital shells up to f
constexpr int kJMaxLAux = 4;                       // auxiliary shells up to g
constexpr int kJMaxL = 2 * kJMaxLPrim + kJMaxLAux;
constexpr int kJMaxH = (kJMaxL + 1) * (kJMaxL + 2) * (kJMaxL + 3) / 6;
constexpr int kJMaxHs = (kJMaxLAux + 1) * (kJMaxLAux + 2) * (kJMaxLAux + 3) / 6;
constexpr int kJMaxNcartAux = (kJMaxLAux + 1) * (kJMaxLAux + 2) / 2;
// Boys table: rows at T = 0, 0.1, .. kBoysEnd, each e^-T and F_0 .. F_(kJMaxL + 8).
constexpr double kBoysEnd = 35.0;
constexpr int kBoysPerUnit = 10;
constexpr int kBoysRows = 351;
constexpr int kBoysCols = 1 + kJMaxL + 9;
// Kernels of the pair x auxiliary meetings: L + l up to kJClassTop[0], up to kJClassTop[1], above.
constexpr int kJClasses = 3;
constexpr int kJClassTop[2] = {3, 6};
constexpr int kJGroupL = 3;  // auxiliary classes from this l on share a wavefront's lanes between pairs
// One wavefront's meetings: pairs [q0, q0 + nq) of class L with auxiliary primitives of class l,
// [a0, a0 + na) (step 4) or the na lanes from a0 (step 2).
struct JItem {
  int L, l, q0, nq, a0, na;
};
// Pairs are sorted by L (class L at [pair0[L], pair0[L + 1])), auxiliary primitives by l; herm0 and
// aherm0 are the classes' offsets in the Hermite arrays (D and U: by pair or primitive, then Hermite
// index; V and W: by Hermite index, then pair or primitive).
struct JView {
  const double* pair;  // x, y, z, exponent of every pair
  const double* aux;   // x, y, z, exponent of every auxiliary primitive
  const double* boys;
  int pair0[2 * kJMaxLPrim + 2], aux0[kJMaxLAux + 2];
  int herm0[2 * kJMaxLPrim + 1], aherm0[kJMaxLAux + 1];
};
// Steps 1 and 5: one wavefront's pairs [q0, q0 + nq), of one (l_A, l_B) and of shells with nfa and nfb
// functions, whose angular transforms start at angA and angB; kernels of l_A + l_B <= kJPairTop and above.
struct JPairItem {
  int la, lb, q0, nq, nfa, nfb, angA, angB;
};
constexpr int kJPairClasses = 2;
constexpr int kJPairTop = 3;
void launch_jdens(hipStream_t s, int cls, const JPairItem* items, int nitem, const JPair* pairs, const DevShell* shells,
                  const double* ang, const JView& Jv, const double* P, int n, double* D);
void launch_jrhs(hipStream_t s, int cls, const JItem* items, int nitem, const JView& J, const double* D, double* W);
void launch_jpot(hipStream_t s, int cls, const JItem* items, int nitem, const JView& J, const double* U, double* V);
void launch_jaux_in(hipStream_t s, const JView& J, int naux, const int* prim_shell, const DevShell* aux,
                    const double* prim_coef, const int* cart_off, const double* cc, double* U);
void launch_jaux_out(hipStream_t s, const JView& J, const DevShell* aux, int nshell, const int* shell_prim,
                     const double* prim_coef, const int* cart_off, const double* W, double* bc);
// cc = the Cartesian form of M^-1 b, b the auxiliary AOs of bc, with M = L L^T (L row-major n x n, dinv the
// inverses of its diagonal blocks of kSolveBlock, row-major and zero-padded); b, y: n each.  bad is set
// where b is not finite.
constexpr int kSolveBlock = 64;
void launch_metric_solve(hipStream_t s, const double* L, int n, const double* dinv, const DevShell* aux, int nshell,
                         const double* ang, const int* cart_off, const double* bc, double* b, double* y, double* cc,
                         int* bad);
void launch_jassemble(hipStream_t s, int cls, const JPairItem* items, int nitem, const JPair* pairs,
                      const DevShell* shells, const double* ang, const JView& Jv, const double* V, int n, double* J);

// The device grid build (kernels/grid_kernels.hip): partition weights of every candidate generated
// from the reference grids (keep[c] = w[c] > thr), the cut (exclusive scan of keep into pos, the
// kept points in candidate order), the bounding box (mn, spread) and the Hilbert order.
void launch_partition_gen(hipStream_t s, int type, unsigned smoothing, int natoms, const double* xyz,
                          const double* dist, const double* apair, const double* min_dist, int64_t ncand,
                          const double* ref_xyz, const double* ref_w, const int64_t* ref_off,
                          const int64_t* cand_off, double thr, double* w, int* keep);
size_t grid_scan_temp_bytes(int64_t n);
void launch_cut(hipStream_t s, int natoms, const double* xyz, int64_t ncand, const double* ref_xyz,
                const int64_t* ref_off, const int64_t* cand_off, const double* w, const int* keep, int* pos,
                void* temp, size_t temp_bytes, double* out_xyz, double* out_w);
int bbox_part_count();
void launch_bbox(hipStream_t s, const double* pts, int64_t n, int64_t length, double* part, double* box);
size_t grid_sort_temp_bytes(int64_t n);
void launch_hilbert_order(hipStream_t s, const double* pts, const double* w, int64_t n, const double* box,
                          int64_t length, int64_t* key, int64_t* key_sorted, int64_t* idx, int64_t* order,
                          void* temp, size_t temp_bytes, double* out_pts, double* out_w);

void launch_weight_potential(hipStream_t s, int64_t npts, const double* w, const double* v, const double* g,
                             double* vs, double* gw);
void launch_fill(hipStream_t s, double* p, int64_t n, double value);
void launch_copy(hipStream_t s, const void* src, void* dst, int64_t n32);  // n32 units of 32 bytes

// Up to kListMax densities passed by value (kernel argument).
struct DensityList {
  const double* rho[kListMax];
  const double* grad[kListMax];
  int n;
};
// rho = sum of list.rho[i] in list order; grad likewise (3 x npts each).
void launch_sum_densities(hipStream_t s, const DensityList& list, int64_t npts, int want_grad, double* rho,
                          double* grad);
// w v and w g of v[sum of sup] - v[rho_act] and the block energies of the difference (where the
// potential is wanted); beside it the block energies of the pending densities.
void launch_nadd_functional(hipStream_t s, int func, int64_t npts, bool potential,
                            const DensityList& sup, const double* rho_act, const double* grad_act,
                            const DensityList& pending, double* const* pending_eblk, const double* w, double* vs,
                            double* gw, double* e_blk);
// out = sum of e_blk[0..n) (null: out) minus the listed energies in order (summed first where pending)
void launch_nadd_energy(hipStream_t s, const double* e_blk, int64_t n, const EnvEnergies& env, double* out);
// Q[i, j] = P[i, j] + P[j, i], Q[i, i] = P[i, i] (packed: P64 into U of the systems whose P is U, n the largest)
void launch_fold(hipStream_t s, const double* P, double* Q, int n, const PackSys* pack = nullptr, int nsys = 1);
void launch_to_float(hipStream_t s, const double* src, float* dst, int64_t n);
// F[i + n j] (+)= U[max(i,j) + n min(i,j)] (U holds the lower triangle)
// F = mirror of U (accumulate: F += it); with P32, part[b] = block b's sum of F (P - P32)
// (finalize_blocks(n) partials)
void launch_finalize(hipStream_t s, const double* U, double* F, int n, int accumulate, const double* P = nullptr,
                     const float* P32 = nullptr, double* part = nullptr);
int finalize_blocks(int n);
// *out = sum of x[0..n) and x2[0..n2) (subtract: *out -= that sum)
void launch_sum(hipStream_t s, const double* x, int64_t n, double* out, int subtract = 0, const double* x2 = nullptr,
                int64_t n2 = 0);

}  // namespace sxc
