// The state behind a biot_handle: everything the reference kept in blockInfo
// (common.h:6-133) plus the time-loop state of callCUDAKernel (kernel.cu:1728-1760).
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/biot.h"
#include "biot_adjoint.hpp"
#include "biot_device.hpp"

// Large results to the host: through pinned buffers that a few threads fill and empty in turn.  A
// copy straight to the caller's pages goes at about 9 GB/s where they are new (their first touch is
// the copy's) and 17 GB/s where they are not, to pinned memory at 57 GB/s.  A 128^3 gradient, whose six
// FP64 arrays are 100 MB: 66.2 ms straight, 59.2 ms this way; 8 threads or 4 MB chunks are no faster.
struct ReadBack {
  struct Piece {
    void *dst;
    const void *src;  // device
    size_t bytes;
  };
  static constexpr int THREADS = 4;
  static constexpr size_t CHUNK = (size_t)2 << 20;
  char *pinned = nullptr;  // THREADS chunks, made on the first large read
  ~ReadBack();
  // after the work queued on s; returns with the copies made, false if one failed
  bool read(const std::vector<Piece> &pieces, int device, hipStream_t s);
};

struct biot_handle {
  biot_grid g{};
  int prec = 0;
  size_t esz = 4;    // field / coefficient element bytes
  size_t csz = 4;    // C-PML carry element bytes
  int64_t n = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::string err;

  // device memory
  void *d_fields = nullptr;          // 13 * n elements (FP16M: tau and p as their binary16 parts)
  int8_t *d_lo = nullptr;  // FP16C / FP16T residuals, 13 * n (compensated fields used); FP16M residual records, 4 * n
  void *d_coef = nullptr;            // 22 * n (FP16M: the medium records, 18 bytes per cell)
  void *d_kpack = nullptr;           // the coefficients packed per cell (velocity, then stress block)
  // a medium of few distinct cells, else null: the records' values, the table they were found in and,
  // in the same block, the cells' records (StepArgs)
  void *d_dict = nullptr;
  uint16_t *d_ids = nullptr;
  void *d_carry[3] = {nullptr, nullptr, nullptr};
  float *h_slice = nullptr;          // pinned, nx * nz: the slice of biot_snapshot_xz (made on first use)
  int *d_flag = nullptr;             // first step with a non-finite receiver sample
                                     // (biot::NONFINITE_NONE: none since the last clear)
  void *d_prof[3][4] = {};           // e_int, a_int, e_half, a_half per axis
  int64_t slab[3] = {0, 0, 0};
  int L[3] = {0, 0, 0}, R[3] = {0, 0, 0};
  int64_t device_bytes = 0;

  // host copies
  std::vector<float> coef_ref[BIOT_NCOEF];  // reference representation
  std::vector<float> prof[3][4];            // d, d2, e, e2 per axis (before the x0.01 pack)
  bool have_coef = false;
  float ks[biot::NKC];        // per-coefficient-array scale (binary16 storage)
  double kfac[biot::NKC];     // storage-unit coefficient / physical coefficient, per array
  float fscale[biot::NFIELD]; // per-field storage scale
  // FP16M: the 9 cell moduli the medium records are built from (M HH H2u C C1 C2 rho rhof mu,
  // float, as biot::Moduli) and the constants of the kernels' coefficient formulas
  std::vector<float> mod[9];
  float mc[biot::NMC] = {};

  // source
  std::vector<float> wavelet;
  void *d_wavelet = nullptr;
  int64_t src_cell = 0;
  uint32_t src_mask = 0;
  // receivers
  void *d_rec = nullptr;
  void *d_traces = nullptr;
  double *d_traces64 = nullptr;  // FP64 handles: the traces in double as well
  int64_t nrec = 0;
  std::vector<int64_t> rec_cells;  // host copy
  uint32_t rec_mask = 0;
  int comp[biot::NFIELD] = {};
  int ncomp = 0;
  int nt_max = 0;

  int it = 0;
  double last_ms = 0.0;
  biot::LaunchShape shape{64, 4, 16};

  ~biot_handle();
  void *field_ptr(int f) const;
  // residual array of field f (FP16C / FP16T, stride 1), or for FP16M's tau and p the base of
  // the residual records (stride PK_RECORD) plus the field's nibble (the kernels' runtime
  // loaders read it from the pointer's low 3 bits), or null
  int8_t *lo_ptr(int f) const;
  // where a host copy of field f's residuals starts: FP16M's record base, else lo_ptr(f)
  int8_t *lo_copy_ptr(int f) const { return packed(f) ? d_lo : lo_ptr(f); }
  size_t lo_stride(int f) const { return packed(f) ? biot::PK_RECORD : 1; }
  size_t lo_bytes() const;
  // FP16M keeps tau and p as binary16 + a 4-bit residual: the binary16 part in the field array,
  // the residual in a per-cell record shared by the seven fields
  bool packed(int f) const { return prec == BIOT_FP16M && ((biot::PK_FIELDS >> f) & 1u); }
  size_t fields_bytes() const;
  size_t mt_offset() const { return ((size_t)8 * n + 255) & ~(size_t)255; }  // FP16M stress records
  size_t mu_offset() const { return (mt_offset() + (size_t)8 * n + 255) & ~(size_t)255; }  // FP16M mu
  bool half() const
  {
    return prec == BIOT_FP16 || prec == BIOT_FP16C || prec == BIOT_FP16T || prec == BIOT_FP16M;
  }
  // the arguments over the handle's own arrays, or over the first of a run of states
  void fill_args(biot::StepArgs &a, char *states = nullptr) const;
  int allocate();
  int upload_profiles();
  int upload_coefficients();
  int pack_coefficients();           // d_coef -> d_kpack
  int find_records();                // d_coef -> d_ids, d_dict where the medium has few distinct cells
  void drop_records();
  int build_adjoint_coefs();         // FP16M: d_kpack for the adjoint, from K_last
  int upload_kernel_coefs(const std::vector<double> (&K)[biot::NKC]);
  int upload_from_ref(const float *d_ref);      // 23 reference arrays on the device
  int upload_medium();                          // FP16M: mod -> medium records, mc
  void set_scales(const double amaxK[biot::NKC], double resp);
  int rescale_state(const float old_scale[biot::NFIELD]);

  // inversion parameters (biot_set_params) and the adjoint's buffers
  std::vector<double> par[8];                // lambda mu alpha M rho rhof C1 tphi
  std::vector<double> K_last[biot::NKC];     // kernel coefficients built from par
  std::vector<void *> ckpt;                  // checkpoint states, every ckpt_every steps
  int ckpt_every = 0, ckpt_nt = 0;
  int room_every = 0, room_nt = 0;           // the run the buffers of ckpt were allocated for
  // ckpt_every == 1: ckpt[0] is one block of ckpt_nt + 1 states, state it being step it's
  // state after its source (the last one the state after the run), which the adjoint reads
  // in place of segment recomputation
  void *d_slots = nullptr;                   // segment states (slots_every + 1), zero outside the update box
  int slots_every = 0;
  int slots_seg = -1;                        // the checkpoint segment whose states d_slots holds, or -1
  void *d_lam = nullptr;                     // adjoint fields, carries, derivative adjoints
  double *d_grad = nullptr;                  // 22 FP64 coefficient gradients
  float *d_gpart = nullptr;                  // 22 float per-segment partial sums (not FP64 handles)
  float *d_adjsrc = nullptr;                 // adjoint source traces
  uint32_t *d_inj = nullptr;                 // which cells hold which receivers (InjectArgs)
  int inj_cells = 0;
  double *d_par = nullptr;                   // the 8 parameter arrays of par, for the chain rule
  hipStream_t side = nullptr;                // uploads beside a running sweep (made on first use)
  ReadBack back;
  size_t state_bytes() const;
  size_t state_off(int piece) const;  // 0 fields, 1..3 carries of x, y, z, 4 total
  size_t state_lo_off() const;        // the residual block (lo_bytes())
  void save_state(void *dst);
  void load_state(const void *src);
  void free_adjoint();
  void forget_model();  // drop parameter-built coefficients and every adjoint buffer
  // marks: null, or 3 events per step recorded before velocity, between, after stress;
  // states: null (in place), or a run of nsteps + 1 states, the first given: step s goes from state s,
  // to which its source is added, to state s + 1.  record: false leaves the traces alone.
  int enqueue_steps(int nsteps, hipEvent_t *marks, char *states = nullptr, bool record = true);
  int clear_borders(char *states, int nstates);  // once for new states; on the stream

  // argument blocks shared by the single-grid and batched drivers
  void source_args(biot::SourceArgs &sa, char *states = nullptr) const;
  bool source_outside() const;               // no half step writes the source cell
  void record_args(biot::RecordArgs &ra, char *states = nullptr) const;  // every component
  bool has_source(int step) const { return d_wavelet && src_mask && step < (int)wavelet.size(); }
  // whether a receiver records a stress or p at the source cell that the source changes: it then
  // has to be sampled before the next step's source is added
  bool source_recorded() const;
  // whether the stress launch can add the next step's source (fields it writes, at a cell it
  // updates, not sampled after it)
  bool source_in_stress() const;
  int clear_nonfinite();                     // enqueue a clear of d_flag on the stream
  int check_nonfinite();                     // synchronize; BIOT_ERR_NONFINITE if it was set
  size_t lam_bytes() const;                  // adjoint wavefields, carries, derivative adjoints
  int alloc_slots(int every);                // d_slots
  int alloc_adjoint(int every);              // d_slots (every+1 states; none for 0), d_lam, d_grad, d_adjsrc, d_inj
  int build_inject();                        // d_inj from rec_cells
  void adj_args(biot::AdjArgs &A) const;     // after alloc_adjoint
  // the device copy of par and room for the 6 parameter gradients, for work queued on the stream
  // after the sweep that is queued now
  int chain_buffers(double *&par_dev, double *&out);
  void inject_args(biot::InjectArgs &I) const;
};

// the tile shape of a launch over that many waves a z plane (plane_waves: of one grid)
biot::LaunchShape default_shape(int prec, int64_t plane_waves);
int64_t plane_waves(const biot_grid &g);
// reference arrays -> unscaled kernel coefficients on the host (1/dx and 0.01 folded)
void host_kernel_coefs(double Hinv, const std::vector<float> (&ref)[BIOT_NCOEF],
                       std::vector<double> (&K)[biot::NKC]);
