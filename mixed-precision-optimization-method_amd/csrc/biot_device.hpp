// Device-side data layout of the Biot solver and the launchers of its HIP kernels.
//
// HBM layout (one handle, n = nx*ny*nz cells, x fastest, idx = i + j*nx + k*nx*ny):
//   fields  : 13 arrays of n elements of the storage type (vx vy vz qx qy qz txx tyy tzz txy
//             txz tyz p), one allocation.
//   coefs   : 22 arrays of n elements (the 23 reference arrays minus W3z, which the
//             reference never reads, kernel.cu:220), with 1/dx, the 0.01 kernel constants
//             and the storage scales folded in.
//   carries : C-PML memory, only inside the absorbing slabs.  Per axis, 8 arrays (4 for the
//             velocity half step, 4 for the stress half step) over the slab cells of that
//             axis: x-slab cells (i < Lx or i >= nx-Rx) are packed to ix in [0, Lx+Rx) and
//             stored at ix + (Lx+Rx)*(j + ny*k); y and z likewise.  One folded variable per
//             derivative replaces the reference's (psi, D_prev) pair:
//                 psi_n = c + a D_n,   D <- D + psi_n,   c <- e (psi_n + a D_n)
//             which is algebraically the recursion of kernel.cu:188-196.
//   profiles: per axis e and a = -dt d / 2 at integer and half nodes (1-D, arithmetic type).
//   residuals (FP16C, FP16T): one int8 array per compensated field (FP16C v, tau, p;
//             FP16T tau, p).
//
// Storage modes (enum biot_precision):
//   FP32  fields, coefficients, carries float; arithmetic float.
//   FP16  fields, coefficients and carries binary16 (scaled); arithmetic float.
//   FP16C as FP16, plus an int8 residual r per value of v, tau and p: the value is
//         h + r * ulp(h) / 256 (h the binary16 part), about a 19-bit significand, so the
//         rounding of the leapfrog-integrated fields does not random-walk.
//   FP16T as FP16C with the residual on tau and p only (the velocities plain binary16): the
//         stresses' rounding dominates the binary16 error, and the velocity residuals are
//         a third of FP16C's residual traffic.
//   FP16M v and q binary16 (scaled); tau and p binary16 (scaled) plus a 4-bit residual in
//         units of ulp/16, the binary16 part in the field's own array, the residuals of the
//         seven such fields in one 4-byte record per cell; the medium as per-cell binary16
//         moduli scaled to [-1, 1] (mv: rho, rho_f, C1, C2 in 8 bytes; mt: C, M, lambda_c, H
//         in 8 bytes; mu: 2 bytes), from which the kernels form the staggered averages, the
//         4-cell harmonic means of mu and the 22 coefficients in registers; float C-PML
//         carries.
//   FP64  everything double.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace biot {

enum { NFIELD = 13, NKC = 22, NCARRY = 8 };
enum { PREC_FP32 = 0, PREC_FP16 = 1, PREC_FP64 = 2, PREC_FP16C = 3, PREC_FP16T = 4, PREC_FP16M = 5 };
// fields carrying a residual: FP16C vx vy vz txx tyy tzz txy txz tyz p; FP16T txx .. tyz p
constexpr uint32_t COMP_FIELDS_C = 0x1FC7u, COMP_FIELDS_T = 0x1FC0u;
constexpr uint32_t comp_fields(int prec)
{
  return prec == PREC_FP16C ? COMP_FIELDS_C : (prec == PREC_FP16T || prec == PREC_FP16M) ? COMP_FIELDS_T : 0u;
}
// FP16M: the fields stored as binary16 + residual (txx .. tyz, p): the binary16 part in the
// field's own array, the 4-bit residual in the cell's 4-byte residual record, at nibble
// pk_slot(f) (the record's last nibble is unused)
constexpr uint32_t PK_FIELDS = COMP_FIELDS_T;
constexpr int PK_FIRST = 6, PK_RECORD = 4;
// nibble of field f in the record: the four fields the velocity step differences along x
// (txx, txy, txz, p) in the low half, tyy, tzz, tyz in the high half
constexpr int pk_slot(int f)
{
  return f == 6 ? 0 : f == 9 ? 1 : f == 10 ? 2 : f == 12 ? 3 : f == 7 ? 4 : f == 8 ? 5 : 6;
}
// the kernels take field PK_FIRST's residual pointer as the record base
static_assert(pk_slot(PK_FIRST) == 0, "field PK_FIRST must own nibble 0 of the record");
// ulp(h)/16 from h as a float (exponent below binary16's normal range: the subnormal ulp)
__device__ __forceinline__ float pk_unit(float hf)
{
  const uint32_t e = (__builtin_bit_cast(uint32_t, hf) >> 23) & 0xFFu;
  return __builtin_bit_cast(float, (max(e, 113u) - 14u) << 23);
}
// residual s (0..6) of a record, sign-extended
__device__ __forceinline__ int pk_nib(uint32_t r, int s)
{
  return (int)(r << (28 - 4 * s)) >> 28;
}
// h as a float plus residual n: the value the forward kernels and the adjoint read
__device__ __forceinline__ float pk_join(float hf, int n)
{
  return fmaf((float)n, pk_unit(hf), hf);
}
// kernel coefficient order
enum {
  K_U1X = 0, K_U1Y, K_U1Z, K_U2X, K_U2Y, K_U2Z, K_W1X, K_W1Y, K_W1Z, K_W2X, K_W2Y, K_W2Z,
  K_W3X, K_W3Y,
  K_P1, K_P2, K_S1, K_S2, K_S3, K_SXY, K_SXZ, K_SYZ
};

// FP16M: the constants that turn the stored moduli into kernel coefficients (in the storage
// units of the fields they connect, 1/dx folded in).  Averages along an axis are
// h * (stored(c) + stored(c + axis)); then U1 = cU1 / rho, U2 = kU2 rho_f / rho,
// m = C2 - rho_f^2 / rho, a = aH C1, W1 = (m - a) / (m + a), W2 = cW2 (rho_f / rho) / (m + a),
// W3 = cW3 / (m + a) (main.cpp:447-481); P1 = kP1 C, P2 = kP2 M, S1 = kS1 lambda_c, S2 = kS2 H,
// S3 = kS3 C, Sij = kSh mu_ij (the stored 4-cell harmonic mean, main.cpp:326-337, 483-494), all
// on the stored values.
enum {
  MC_HRHO = 0, MC_HRHOF, MC_HC1, MC_HC2, MC_KU2, MC_CU1, MC_CW2, MC_CW3, MC_AH,
  MC_KP1, MC_KP2, MC_KS1, MC_KS2, MC_KS3, MC_KSH, NMC
};

// Kernel arguments; pointers are type-erased, their element types follow the storage mode.
struct StepArgs {
  void *f[NFIELD];           // field storage
  int8_t *lo[NFIELD];        // FP16C / FP16T residuals (null for other modes / fields)
  const void *k[NKC];        // coefficient arrays (field storage type)
  // the same coefficients packed per cell (storage type): kv holds K[0..13] of the velocity
  // half step, kt K[14..21] of the stress half step, cell c at element c*14 / c*8 (addressed
  // in 64 bits: these arrays may span more than 4 GiB)
  const void *kv, *kt;
  // a medium of few distinct cells (DictArgs): the cell's record, and the records' coefficients
  // (storage type; record r at element 16 r of dv, 8 r of dt); null otherwise
  const uint16_t *ids;
  const void *dv, *dt;
  float ks[NKC];             // per-array scale (binary16 storage), 1 otherwise
  // FP16M: the medium records (mv: 4 binary16 values per cell, mt: 4), the cell shear
  // moduli (mu: binary16) and constants
  const void *mv, *mt, *mu;
  float mc[NMC];
  // per axis: the C-PML carries (carry type) of the slab cells, in two groups of records — the
  // velocity half step's carries 0..3, then the stress half step's 4..7 — each group slab[ax]
  // records of 4 carries: carry m of slab cell o is element (m/4)*4*slab + 4*o + m%4
  void *carry[3];
  int64_t slab[3];           // elements per carry array per axis
  const void *prof[3][4];    // per axis: e_int, a_int, e_half, a_half (arithmetic type)
  int nx, ny, nz;
  int L[3], R[3];            // slab widths
  int64_t sy, sz;            // strides
  int zchunk;
  int gx, gy, gz, ntiles;    // tile grid (x-y tiles of the block shape, z chunks)
  uint64_t sb;               // a run of states: bytes from one to the next
  int xg;                    // consecutive tiles an XCD takes at a time (xcd_run)
  int src[3];                // the source cell (no cell's position: no source)
  int xy0;                   // one-row blocks: the plane cell the first tile starts at
  uint32_t nx_rcp;           // ceil(2^32 / nx)
};

inline size_t field_bytes(int prec) { return prec == PREC_FP64 ? 8 : prec == PREC_FP32 ? 4 : 2; }
// C-PML carries: binary16 in the FP16 policy (all state 16-bit, as the reference stores every
// array in half), float in FP32, FP16C and FP16T, double in FP64
inline size_t carry_bytes(int prec) { return prec == PREC_FP64 ? 8 : prec == PREC_FP16 ? 2 : 4; }

// Host-side launchers (biot_kernels.hip).
struct LaunchShape {
  int bx, by, zchunk;
};
// Workgroup b of a 1-D grid goes to XCD b % 8.  Each XCD takes runs of g consecutive tiles, run
// after run dealt out to the eight in turn, so that the rows neighbouring tiles both read meet in
// one L2 while all XCDs work in the same planes of every array: with one contiguous eighth of the
// tiles each, they streamed from eight places of each of the 30-odd arrays at once.  256^3 FP32,
// velocity + stress, 256-cell tiles of 4 planes: eighths 934 us, runs of 1 tile 886, of 4, 8, 16 and
// 32 tiles 859-862 (8 at 2 planes: 843), of 64 862, of 256 886; 512x512x384 FP32 5.54 ms in eighths,
// 4.88 in runs of 8, FP16M at 16 planes 3.04 and 2.83 ms.  A run is 2048 cells; with few tiles it is
// shorter, for eight runs an XCD.  Grids whose arrays about fit the eight L2s (half a million
// cells) keep contiguous eighths, whose rows meet in one L2 from step to step (64^3 FP32, 200 steps:
// 4.2 ms, in runs 4.5 ms).
inline int xcd_run(int64_t ntiles, int threads, int64_t cells)
{
  if (cells <= (int64_t)1 << 19) return (int)((ntiles + 7) / 8 > 0 ? (ntiles + 7) / 8 : 1);
  const int64_t g = ntiles / 64, most = 2048 / threads;
  return (int)(g < 1 ? 1 : g > most ? most : g);
}
// the slots of one XCD for n tiles in runs of g: local slot m of XCD x is tile xcd_tile(x, m, g)
// (those past n are empty)
inline int64_t xcd_slots(int64_t n, int g) { return (n + 8 * (int64_t)g - 1) / (8 * (int64_t)g) * g; }
__host__ __device__ inline int xcd_tile(int x, int m, int g) { return (m / g * 8 + x) * g + m % g; }
// the tile grid of shape sh over the update box (h cells off every face): rectangles of bx x by
// cells, or for by = 1 runs of bx consecutive cells of the x-y plane, the first starting on a
// 64-cell boundary of the plane
inline void set_tiles(StepArgs &a, LaunchShape sh, int h)
{
  a.zchunk = sh.zchunk;
  a.xy0 = (h * a.nx) & ~63;
  a.nx_rcp = (uint32_t)((((uint64_t)1 << 32) + (uint64_t)a.nx - 1) / (uint64_t)a.nx);
  if (sh.by == 1) {
    a.gx = (int)(((int64_t)(a.ny - h) * a.nx - a.xy0 + sh.bx - 1) / sh.bx);
    a.gy = 1;
  } else {
    a.gx = (a.nx + sh.bx - 1) / sh.bx;
    a.gy = (a.ny + sh.by - 1) / sh.by;
  }
  a.gz = (a.nz - 2 * h + a.zchunk - 1) / a.zchunk;
  a.ntiles = a.gx * a.gy * a.gz;
  a.xg = xcd_run(a.ntiles, sh.bx * sh.by, (int64_t)a.nx * a.ny * a.nz);
}

struct SourceArgs {
  void *f[NFIELD];
  int8_t *lo[NFIELD];
  int64_t cell;
  uint32_t mask;
  const float *wavelet;     // device, one sample per step
  int it;
  int nt_w;                 // wavelet samples
  float inv_scale[NFIELD];  // 1 / storage scale per field
  int outside;              // no half step writes the cell
  uint64_t sb;              // a run of states: bytes from one to the next
  uint64_t ioff, ooff;      // single launches: where the value is read and stored, bytes on
};
struct RecordArgs {
  const void *f[NFIELD];
  const int8_t *lo[NFIELD];
  const int64_t *rec;       // device receiver cells
  int64_t nrec;
  int comp[NFIELD];         // recorded fields, ascending
  int ncomp;
  int c0, c1;               // the components this launch records
  int nvel;                 // components 0..nvel-1 are velocities, the others stresses and p
  float scale[NFIELD];      // storage scale per recorded component
  float *traces;            // device [comp][nt_max][nrec]
  double *traces64;         // same layout in double (FP64 handles), or null
  int *nonfinite;           // device: the first step with a non-finite sample (NONFINITE_NONE:
                            // none so far), or null
  int it, nt_max;
  uint64_t off;             // single launches: the state's place, bytes on
};
// A half step's launch also does the work around it that touches only fields it leaves alone:
// the velocity launch records the stresses and p of the step before, the stress launch the
// velocities of its own step (blocks after the tiles'), and the thread that updates the source
// cell's stresses then adds the next step's source there.  On their own the two were 4.5 us
// launches of a few waves (200 steps of 64^3 FP32 with their outputs: 6.4 ms in four launches a
// step, 5.7 ms in two; 45x38x53 at order 2, 150 steps: 3.8 ms and 3.3 ms).
struct FuseArgs {
  int tile_blocks;          // blocks of the tiles (set by the launcher); the others record
  int record;               // rec holds something to record
  int source;               // src is to be added (stress launch)
  int q;                    // state of a run of states (OOP)
  RecordArgs rec;
  SourceArgs src;
};
// rec (c0, c1 and it set; may be null), src (it set; stress launch; may be null): see FuseArgs;
// q >= 0: out of place, state q of the run of states at the arguments' pointers to state q + 1
hipError_t launch_velocity(int prec, int order, const StepArgs &args, LaunchShape shape, hipStream_t s,
                           const RecordArgs *rec = nullptr, int q = -1);
hipError_t launch_stress(int prec, int order, const StepArgs &args, LaunchShape shape, hipStream_t s,
                         const RecordArgs *rec = nullptr, const SourceArgs *src = nullptr, int q = -1);
// zero values outside the update box of nstates states (loff: the residuals' place in a state)
hipError_t launch_clear_border(int prec, void *slots, int nstates, uint64_t sb, uint64_t loff, int h, int nx, int ny,
                               int nz, hipStream_t s);
// the byte pattern a cleared non-finite flag holds (every byte 0x7F): larger than any step
constexpr int NONFINITE_NONE = 0x7F7F7F7F;
hipError_t launch_source(int prec, const SourceArgs &a, hipStream_t s);

// GPU-side set-up (biot_build.hip), bit-identical to the host builder.
struct MediumArgs {
  const double *Ks, *Kf, *Kb, *mu, *phi, *rhos, *rhof, *eta, *perm;
  double tao, porousm;
  float *out[9];            // M HH H2u C C1 C2 rho rhof mu
};
struct CoefRefArgs {
  const float *mod[9];      // as MediumArgs::out
  float *coef[23];          // the reference arrays (enum biot_coef order)
  int nx, ny, nz;
  float DT, Cv, Cp;
};
struct RefArgs {
  const float *ref[23];     // reference arrays on the device
  int64_t n;
  double H;                 // 1/dx as the kernels hold it
  uint32_t *stats_u32;      // 23 maxima of |ref| (float bits)
  unsigned long long *stats_u64;  // forced q response (double bits)
  void *kout;               // 22 kernel arrays of the storage type
  int scaled;
  double ratio[NKC], inv_ks[NKC];
};
hipError_t launch_moduli(const MediumArgs &m, int64_t n, hipStream_t s);
hipError_t launch_coef_ref(const CoefRefArgs &a, hipStream_t s);
hipError_t launch_ref_stats(const RefArgs &a, hipStream_t s);
hipError_t launch_ref_to_kernel(int prec, const RefArgs &a, hipStream_t s);

// Batched launches over many shots (one grid for all; device-resident argument tables).
struct BatchArgs {
  const StepArgs *shots;    // device, one per shot (gx, gy, gz, zchunk set for the shape)
  const int *tile_start;    // device, nshots + 1 prefix sums of the shots' tile counts
  int nshots, total_tiles;
  int xg;                   // consecutive tiles an XCD takes at a time (xcd_run; set by the launcher)
  int *queue;               // device, 16 ints (zero between launches): per XCD group the tile
                            // counter and the count of finished blocks; null: one block per tile
  // the work around the half step, as FuseArgs per shot: step it[0] + off, the sources of steps
  // below it[1] added by the stress launch (src null: none), the blocks from tile_blocks on
  // recording rec_blocks blocks a shot (rec_blocks 0: none; a step before it[2] is not recorded)
  const SourceArgs *src;
  const RecordArgs *rec;
  const int *it;
  int off, tile_blocks, rec_blocks;
  int64_t cells, state;     // of all the shots' windows: cells, bytes of a state
  int q;                    // >= 0: out of place, as launch_velocity's; one block per tile
};
// blocks: the persistent grid size (a multiple of 8); max_nrec: the most receivers a shot has
// (0: record nothing)
hipError_t launch_step_batch(int prec, int order, bool vel, const BatchArgs &b, LaunchShape sh,
                             int blocks, int64_t max_nrec, hipStream_t s);
// the sources of step it[0] + off (to state q of each shot's run of states, or in place for q < 0);
// the components of step it[0] + off (vel: the velocities too,
// else the stresses and p alone)
hipError_t launch_source_batch(int prec, const SourceArgs *tab, int nshots, const int *it, int off, int q,
                               hipStream_t s);
hipError_t launch_record_batch(int prec, const RecordArgs *tab, int nshots, int64_t max_nrec,
                               bool vel, const int *it, int off, hipStream_t s);
// it[0] += d / it[0] = it[2] = v, it[1] = end on the device (kernels, so they may sit in a
// captured graph)
hipError_t launch_advance(int *it, int d, hipStream_t s);
hipError_t launch_set_counter(int *it, int v, int end, hipStream_t s);
// multiply a stored array by f (lo: its residuals or null); carries use prec of the carry
// type, i.e. pass PREC_FP32 for FP16C/FP16T carries and PREC_FP16 for FP16 carries
hipError_t launch_rescale(int prec, void *p, int8_t *lo, int64_t n, double f, hipStream_t s);
// the same for an FP16M tau or p array of n values (lo: its tagged residual pointer)
hipError_t launch_rescale_pk(void *p, int8_t *lo, int64_t n, double f, hipStream_t s);
// element e of every 4-element record times f[e] (carry groups whose carries scale differently)
hipError_t launch_rescale4(int prec, void *p, int64_t nrec, const double f[4], hipStream_t s);
// the xz slice y = j of one field as float values (stored value times scale): out[k*nx + i]
hipError_t launch_slice_xz(int prec, const void *f, const int8_t *lo, bool comp, double scale, int j, int nx,
                           int ny, int nz, float *out, hipStream_t s);
// per-cell packed copies kv (K[0..13]) and kt (K[14..21]) of the 22 coefficient arrays
// The distinct coefficient records of a medium (biot_build.hip).  Layered and blocky media hold the
// same 22 values in most of their cells: then a cell names its record in 2 bytes instead of streaming
// 88 bytes (FP32) of coefficients a step (256^3 FP32, three layers, velocity + stress: 845 us streamed,
// 680 us with records).  A medium with more than DICT_MAX different cells keeps the streamed arrays
// alone; the scan stops where it finds that many.  A random mix of two rocks, 128 records in no order,
// is still no slower than its streamed arrays (835 us), so the limit is the table's size, not its use:
// 2048 records of 96 bytes (FP32) stay in an L2.
constexpr uint32_t DICT_SLOTS = 4096, DICT_MAX = 2048, DICT_EMPTY = 0xFFFFFFFFu;
struct DictArgs {
  const void *coef;          // 22 * n stored coefficients
  int64_t n;
  uint16_t *ids;             // n
  void *dv, *dt;             // DICT_SLOTS records of 16 and 8 stored values
  uint32_t *slots;           // DICT_SLOTS: a cell with the record's values, or DICT_EMPTY
  uint32_t *state;           // records found less one; 0 once there are too many (both DICT_EMPTY before)
};
hipError_t launch_dict(int prec, const DictArgs &a, hipStream_t s);
hipError_t launch_pack_coef(int prec, const void *soa, void *kv, void *kt, int64_t n, hipStream_t s);
hipError_t launch_record(int prec, const RecordArgs &a, hipStream_t s);

}  // namespace biot
