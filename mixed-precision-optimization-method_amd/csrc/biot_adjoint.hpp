// Device arguments and launchers of the discrete adjoint (biot_adjoint.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "biot_device.hpp"

namespace biot {

// A block of the adjoint passes: ADJ_BX consecutive cells of an x-y plane, the plane's first block
// starting on a 64-cell boundary, in ADJ_BZ planes.  Runs of the update box's own cells left every wave
// two cells off its cache lines; with these the two passes take (us a step, before / after) 329 / 320 at
// 128^3 FP32, 1023 / 1000 at 192^3 FP32, 100 / 92 at 96x80x89 FP16M, 284 / 280 at 110x99x83 FP64.  256
// cells of one plane: 317, 986, 93, 281, and 2 % slower than before at 75^3 (128 x 2: 2 % faster); blocks
// of 512 and blocks that end each axis's loads together, for the rows they share, are slower: the
// passes are bound by the 360 and 265 bytes a cell (FP32) that they move, at 4.1 TB/s.
constexpr uint32_t ADJ_BX = 128, ADJ_BZ = 2;
// Per-grid adjoint arguments.  The forward states of a recomputed segment sit in `slots`
// (state q at slots + q*sb: the fields block, field f at f*fbytes, then the carry blocks at
// coff[0..2]); the adjoint step of segment step q reads state q (after its source) and the
// v, q fields of state q+1.
struct AdjArgs {
  const char *slots;
  uint64_t sb, fbytes, coff[3];
  uint64_t loff;             // offset in a state of the FP16T / FP16C residual arrays (int8, field f at
                             // f*n) or of FP16M's residual records (4 bytes per cell), else 0
  void *lam[NFIELD];         // adjoint wavefields (arithmetic type), storage units
  void *lcarry[3];           // adjoint carries (arithmetic type), forward layout
  // derivative adjoints between the passes (arithmetic type): full arrays of the velocity half's 6
  // (S, Ds of x, y, z) and the stress half's 7 (uxx, uyy, uzz, div w, xy, xz, yz), and per axis the
  // records of the slab's own four (forward carry layout)
  void *gv[6], *gt[7], *gs[3];
  double *grad[NKC];         // dJ/dK in storage units (multiply by the handle's kfac), FP64
  // per-step accumulation of dJ/dK: float partial sums over one checkpoint segment (FP32 and
  // FP16 handles; launch_adjoint_flush adds them into grad and clears them), grad itself on
  // FP64 handles
  void *gacc[NKC];
  // FP32/FP16 handles: the same partial sums packed per cell (float; gpv: K[0..13] of the
  // velocity half step, gpt: K[14..21] of the stress half step, in the 16-byte group layout
  // of biot_packed.hpp); null on FP64 handles
  void *gpv, *gpt;
  const void *k[NKC];        // kernel coefficients (storage type)
  const void *kv, *kt;       // the coefficients packed per cell (storage type, same layout)
  float ks[NKC];             // per-array coefficient scale (16-bit storage), else 1
  const void *prof[3][4];    // e_int, a_int, e_half, a_half per axis (arithmetic type)
  int nx, ny, nz;
  int L[3], R[3];
  int64_t slab[3];
  int64_t sy, sz;
  int blocks, gx, xy0;       // blocks; those of ADJ_BZ planes; the plane cell the first one starts at
  uint32_t nx_rcp;           // ceil(2^32 / nx)
};

// The adjoint sources: a bit per cell tells the thread that updates a cell whether receivers sit
// there, and the cells' sorted list which.
struct InjectArgs {
  const uint32_t *has;       // bit c: cell c holds receivers
  const uint32_t *cells;     // the ncells cells that do, ascending
  const uint32_t *first;     // ncells + 1: their first entries in ids
  const uint32_t *ids;       // receivers by cell
  int ncells;
  int64_t nrec;
  int comp[NFIELD];          // component that records field f, or -1
  float scale[NFIELD];       // storage scale of field f (traces hold scale x stored value)
  const float *src;          // adjoint source [comp][nt][rec]
  int nt;
};

// adjoint of one full step (the stress pass, then the velocity pass) for step it, segment step q,
// with step it's adjoint sources; prec is the storage precision
hipError_t launch_adjoint_step(int prec, int order, const AdjArgs &a, const InjectArgs &j, int q, int it, hipStream_t s);
// grad += packed partial sums, partial sums = 0 over the update box (no-op on FP64 handles,
// which sum into grad)
hipError_t launch_adjoint_flush(int prec, int order, const AdjArgs &a, hipStream_t s);
// J += 1/2 sum (d - obs)^2 (FP64), res = d - obs (res may be null); d is double when
// d_double, else float
hipError_t launch_misfit(const void *d, bool d_double, const float *obs, float *res, int64_t n,
                         double *J, hipStream_t s);

// Batched forms: device tables of per-shot arguments.  block_start[s] is the first block
// of shot s in a grid of 256-thread blocks covering every shot's update box.
struct AdjBatch {
  const AdjArgs *shots;
  const int *block_start;    // nshots + 1
  int nshots, total_blocks;
  const InjectArgs *inject;  // one per shot
};
hipError_t launch_adjoint_step_batch(int prec, int order, const AdjBatch &b, int q, int it, hipStream_t s);
hipError_t launch_adjoint_flush_batch(int prec, int order, const AdjBatch &b, hipStream_t s);

// Chain rule on the device: storage-unit coefficient gradients of one window (grad[k] times
// kfac[k] gives dJ/dK) -> dJ/d(lambda, mu, alpha, M, rho, rho_f), written to (add: added into)
// the model-grid arrays out[6] at the window's position.  One thread owns one model cell, so
// overlapping windows are added by launches that follow one another on a stream.  Parameters
// are the window's.
struct ChainArgs {
  const double *grad[NKC];
  double kfac[NKC];
  const double *par[8];      // lambda mu alpha M rho rhof C1 tphi (window cells)
  double *out[6];            // model grid
  int wx, wy, wz;            // window size
  int x0, y0, z0;            // window origin in the model grid
  int64_t msy, msz;          // model strides
  double dt, Cv, Cp, Hinv;
  int add;
};
hipError_t launch_chain(const ChainArgs &c, hipStream_t s);

// Copies of whole states between live handles and slot buffers, many at once: entry e
// copies bytes[e] from src[e] to dst[e] (all 4-byte aligned).
struct CopyEntry {
  const void *src;
  void *dst;
  uint64_t bytes;
};
hipError_t launch_copy_batch(const CopyEntry *tab, int n, hipStream_t s);

}  // namespace biot
