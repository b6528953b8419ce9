// Launchers of the row kernels (eri_row_impl.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "device_types.hpp"

namespace cqx {

// Row kernels (eri_row_impl.hpp): screening, ERI evaluation and J/K
// digestion of one class pair in one launch, bra pair by bra pair.  A block
// takes a bra pair (a, b) and a chunk of its kets, keeps the rows K(a, :)
// and K(b, :) of every exchange plane in LDS over the columns that the ket
// class reaches, and adds them to the accumulators once.
constexpr int kRowPlanes = 8;  // exchange row planes of a launch
constexpr int kRowJ = 4;       // Coulomb planes of a launch
constexpr int kRowChunk = 1024;  // candidate kets of one work item
struct RowPlane {
  int kind, idx;   // plane idx of the kind's interleaved arrays
  int colwise;     // row r of the plane: element (k, r), else (r, k)
  int mat;         // contraction index (screening mask bit)
  double sign;     // of the element as a row (imaginary part of a Hermitian plane read column-wise: -1)
};
struct RowLaunch {
  int la, lb, lc, ld;
  const PairRec *bra;
  const PairScr *bscr, *kscr;
  const RowKet *ket;
  int nbra, nket, nchunk;       // nchunk: chunks of the longest ket segment
  const int *seg;               // molecule m's kets: [seg[m], seg[m + 1])
  int same_class;
  const double *bra_pn, *ket_pn, *Bg, *Bm, *molmax;
  const long long *mol_boff;
  const int *mol_ns;
  int nmat;
  double thresh;
  int screen;
  double cut32;                 // Schwarz products below go to the FP32 launch (0: none)
  int fp32;
  const PrimPair *prims;
  const PrimC32 *primc32;
  const double *rys, *rys_half;  // the Rys table, and its forms for the row kernels (RysRow)
  const float *rys32_half;
  MolPlanes m0;
  const MolPlanes *mols;
  int nmol;
  int kps[4];
  int width;                    // columns of a row
  const int *colmap;            // [molecule][width]: Cartesian function of a column, -1: none
  int nk;
  RowPlane k[kRowPlanes];
  // Coulomb planes in pair order: plane j, component c, pair i of a class of
  // n pairs at [(j nc + c) n + i]
  int nj;
  int jmat[kRowJ];
  double jcoef[kRowJ];
  const double *jx_bra, *jx_ket;
  double *ja_bra, *ja_ket;
  unsigned long long *count;    // quartets, candidates
  double *prim_sum;
};
// LDS of a row block at most: all a block can have.  One block per CU still
// beats quartet lists: GHF (ps|ps) of (H2O)16 1.41 against 2.04 ms.
constexpr size_t kRowLdsMax = 160 * 1024;
// the LDS one block takes (0: no row kernel for the class, or more than
// kRowLdsMax)
size_t eri_row_lds(int la, int lb, int lc, int ld, int fp32, int nk, int width);
hipError_t launch_eri_row(const RowLaunch &a, hipStream_t s);

}  // namespace cqx
