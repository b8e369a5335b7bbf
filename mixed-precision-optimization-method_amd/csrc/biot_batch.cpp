// Batched shots: many windows of one model advanced together (include/biot.h, biot_batch_*).
//
// Every shot is a grid of its own (a biot_handle: its window of the model, its absorbing
// boundary, source and receivers).  One launch per half step covers the tiles of
// all shots (k_step_batch), the per-shot argument tables live in device memory, and the step
// index comes from a device counter, so a run of steps is captured once into a HIP graph and
// replayed.  The gradient runs the checkpointed forward, the FP64 misfit, the segment
// recompute and the adjoint sweep for all shots at once and adds every shot's parameter
// gradient into one model-grid volume on the device.  The reference has no counterpart.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/biot.h"
#include "biot_adjoint.hpp"
#include "biot_handle.hpp"

using namespace biot;

struct biot_batch {
  biot_batch_config cfg{};
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::string err;
  double last_ms = 0;

  struct Shot {
    biot_handle *h = nullptr;
    int x0, y0, z0;
    std::vector<void *> ckpt;      // checkpoint states
    double *d_par = nullptr;       // the 8 window parameter arrays (chain rule)
    float *d_obs = nullptr;        // observed traces
  };
  std::vector<Shot> shots;

  LaunchShape shape{64, 1, 1};
  int blocks = 8;                  // grid of the batched stencil launches
  bool launch_set = false;         // shape and blocks are the caller's or the autotuner's

  // forward tables
  StepArgs *d_step = nullptr;
  int *d_tiles = nullptr;
  SourceArgs *d_src = nullptr;
  RecordArgs *d_rec = nullptr;
  int *d_it = nullptr;
  int *d_queue = nullptr;          // 16 ints, the persistent grid's work-queue counters
  int total_tiles = 0;
  int64_t cells = 0, state = 0;    // of the shots the tables cover: cells, bytes of a state
  int nactive = 0;                 // shots the current tables cover
  int64_t max_nrec = 0;
  bool fused = false;              // every shot's source and receivers can ride on the half steps
  bool built = false;
  // captured steps
  hipGraphExec_t gexec = nullptr;
  int g_steps = 0;
  bool g_record = false;
  // gradient tables
  AdjArgs *d_adj = nullptr;
  int *d_blocks = nullptr;
  InjectArgs *d_inj = nullptr;
  CopyEntry *d_copy = nullptr;
  StepArgs *d_step_s = nullptr;    // d_step, d_src and d_rec over the segment states
  SourceArgs *d_src_s = nullptr;
  RecordArgs *d_rec_s = nullptr;
  int adj_blocks = 0;
  double *d_gout = nullptr;        // 6 model-grid arrays
  double *d_J = nullptr;
  int groups = 0;                  // shot groups of the last gradient (device memory)
  // the gradient the shots' buffers were allocated for and are kept for (all shots in one group);
  // 0: they are released
  int room_every = 0, room_nt = 0;
  hipStream_t side = nullptr;      // uploads beside the running forward sweep
  ReadBack back;

  ~biot_batch();
  void drop_graph()
  {
    if (gexec) (void)hipGraphExecDestroy(gexec);
    gexec = nullptr;
    g_steps = 0;
  }
  void free_tables();
  void free_gradient();
};

namespace {

int bfail(biot_batch *b, int code, const char *fmt, ...)
{
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  b->err = buf;
  return code;
}

#define BHIP(b, call)                                                                      \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess)                                                                  \
      return bfail((b), BIOT_ERR_HIP, "%s failed: %s", #call, hipGetErrorString(e_));     \
  } while (0)

template <typename T>
void dfree(T *&p)
{
  if (p) (void)hipFree((void *)p);
  p = nullptr;
}

// shot-handle failures carry the handle's message
int hfail(biot_batch *b, biot_handle *h, int rc, const char *what)
{
  const char *m = h ? biot_last_error(h) : nullptr;
  return bfail(b, rc, "%s: %s", what, m && *m ? m : biot_status_string(rc));
}

}  // namespace

void biot_batch::free_tables()
{
  dfree(d_step);
  dfree(d_tiles);
  dfree(d_src);
  dfree(d_rec);
  built = false;
  drop_graph();
}

void biot_batch::free_gradient()
{
  if (stream) (void)hipStreamSynchronize(stream);
  for (auto &s : shots) {
    for (void *p : s.ckpt)
      if (p) (void)hipFree(p);
    s.ckpt.clear();
    dfree(s.d_par);
    dfree(s.d_obs);
    if (s.h) s.h->free_adjoint();
  }
  room_every = room_nt = 0;
  dfree(d_adj);
  dfree(d_blocks);
  dfree(d_inj);
  dfree(d_copy);
  dfree(d_step_s);
  dfree(d_src_s);
  dfree(d_rec_s);
  dfree(d_gout);
  dfree(d_J);
}

biot_batch::~biot_batch()
{
  free_gradient();
  free_tables();
  dfree(d_it);
  dfree(d_queue);
  for (auto &s : shots)
    if (s.h) biot_destroy(s.h);
  if (ev0) (void)hipEventDestroy(ev0);
  if (ev1) (void)hipEventDestroy(ev1);
  if (side) (void)hipStreamDestroy(side);
  if (stream) (void)hipStreamDestroy(stream);
}

// message of the calling thread's last failed biot_batch_create (biot_batch_last_error(NULL))
static thread_local std::string t_batch_create_err;

extern "C" int biot_batch_create(const biot_batch_config *c, biot_batch **out)
{
  t_batch_create_err.clear();
  auto refuse = [](biot_batch *b, int rc, const char *why) {
    delete b;
    t_batch_create_err = why;
    return rc;
  };
  if (!c || !out) return refuse(nullptr, BIOT_ERR_ARG, "config and output pointers are required");
  *out = nullptr;
  if (c->nx < 8 || c->ny < 8 || c->nz < 8)
    return refuse(nullptr, BIOT_ERR_ARG, "the model grid must be at least 8 cells on every axis");
  if (c->order != 2 && c->order != 4) return refuse(nullptr, BIOT_ERR_ARG, "order must be 2 or 4");
  if (c->precision != BIOT_FP32 && c->precision != BIOT_FP16 && c->precision != BIOT_FP16T &&
      c->precision != BIOT_FP16C && c->precision != BIOT_FP16M && c->precision != BIOT_FP64)
    return refuse(nullptr, BIOT_ERR_ARG,
                  "batches run BIOT_FP32, BIOT_FP16, BIOT_FP16T, BIOT_FP16C, BIOT_FP16M or BIOT_FP64");
  if (!(c->dx > 0) || !(c->dt > 0) || c->npml < 0)
    return refuse(nullptr, BIOT_ERR_ARG, "dx and dt must be positive and npml >= 0");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return refuse(nullptr, BIOT_ERR_HIP, "no HIP device");
  if (c->device < 0 || c->device >= ndev) return refuse(nullptr, BIOT_ERR_ARG, "device index out of range");
  biot_batch *b = new biot_batch();
  b->cfg = *c;
  if (hipSetDevice(c->device) != hipSuccess || hipStreamCreate(&b->stream) != hipSuccess ||
      hipEventCreate(&b->ev0) != hipSuccess || hipEventCreate(&b->ev1) != hipSuccess ||
      hipMalloc((void **)&b->d_it, 3 * sizeof(int)) != hipSuccess ||
      hipMalloc((void **)&b->d_queue, 16 * sizeof(int)) != hipSuccess ||
      hipMemset(b->d_queue, 0, 16 * sizeof(int)) != hipSuccess)
    return refuse(b, BIOT_ERR_HIP, "device, stream, event or counter set-up failed");
  *out = b;
  return BIOT_OK;
}

extern "C" int biot_batch_destroy(biot_batch *b)
{
  if (!b) return BIOT_ERR_ARG;
  delete b;
  return BIOT_OK;
}

extern "C" const char *biot_batch_last_error(const biot_batch *b)
{
  return b ? b->err.c_str() : t_batch_create_err.c_str();
}

extern "C" int biot_batch_add_shot(biot_batch *b, const biot_shot *s, const biot_params *p,
                                   const float *wavelet, int32_t nt)
{
  if (!b) return BIOT_ERR_ARG;
  if (!s || !p || !wavelet || nt <= 0) return bfail(b, BIOT_ERR_ARG, "shot, parameters and wavelet required");
  const biot_batch_config &c = b->cfg;
  if (s->x0 < 0 || s->y0 < 0 || s->z0 < 0 || s->nx < 8 || s->ny < 8 || s->nz < 8 ||
      s->x0 + s->nx > c.nx || s->y0 + s->ny > c.ny || s->z0 + s->nz > c.nz)
    return bfail(b, BIOT_ERR_ARG, "window %dx%dx%d at (%d,%d,%d) outside the %dx%dx%d model", s->nx,
                 s->ny, s->nz, s->x0, s->y0, s->z0, c.nx, c.ny, c.nz);
  biot_grid g{};
  g.nx = s->nx;
  g.ny = s->ny;
  g.nz = s->nz;
  g.order = c.order;
  g.precision = c.precision;
  g.npml = c.npml;
  g.dx = c.dx;
  g.dt = c.dt;
  g.pml_v0 = c.pml_v0;
  g.pml_R = c.pml_R;
  g.Cv = c.Cv;
  g.Cp = c.Cp;
  g.device = c.device;
  biot_handle *h = nullptr;
  int rc = biot_create(&g, &h);
  if (rc) return bfail(b, rc, "shot %zu: window grid rejected: %s", b->shots.size(), biot_last_error(nullptr));
  if ((rc = biot_set_params(h, p)) || (rc = biot_set_source(h, s->src_cell, s->src_mask, wavelet, nt)) ||
      (rc = biot_set_receivers(h, s->rec_cells, s->nrec, s->rec_mask, nt))) {
    const int r2 = hfail(b, h, rc, "shot set-up");
    biot_destroy(h);
    return r2;
  }
  biot_batch::Shot sh;
  sh.h = h;
  sh.x0 = s->x0;
  sh.y0 = s->y0;
  sh.z0 = s->z0;
  b->free_gradient();
  b->free_tables();
  b->shots.push_back(sh);
  return BIOT_OK;
}

// New model-grid parameters: each shot's window is cut out and its coefficients rebuilt.
extern "C" int biot_batch_set_model(biot_batch *b, const biot_params *p)
{
  if (!b) return BIOT_ERR_ARG;
  if (!p || !p->lambda || !p->mu || !p->alpha || !p->M || !p->rho || !p->rhof || !p->C1 || !p->tphi)
    return bfail(b, BIOT_ERR_ARG, "every model parameter array is required");
  const double *src[8] = {p->lambda, p->mu, p->alpha, p->M, p->rho, p->rhof, p->C1, p->tphi};
  const int64_t msy = b->cfg.nx, msz = (int64_t)b->cfg.nx * b->cfg.ny;
  b->free_gradient();
  for (size_t i = 0; i < b->shots.size(); ++i) {
    auto &s = b->shots[i];
    biot_handle *h = s.h;
    const int wx = h->g.nx, wy = h->g.ny, wz = h->g.nz;
    std::vector<double> win[8];
    for (int q = 0; q < 8; ++q) {
      win[q].resize((size_t)h->n);
      for (int k = 0; k < wz; ++k)
        for (int j = 0; j < wy; ++j) {
          const double *row = src[q] + (s.x0 + (int64_t)(s.y0 + j) * msy + (int64_t)(s.z0 + k) * msz);
          std::memcpy(win[q].data() + ((int64_t)k * wy + j) * wx, row, (size_t)wx * sizeof(double));
        }
    }
    const biot_params wp{win[0].data(), win[1].data(), win[2].data(), win[3].data(),
                         win[4].data(), win[5].data(), win[6].data(), win[7].data()};
    int rc = biot_set_params(h, &wp);
    if (rc) return hfail(b, h, rc, "shot parameters");
  }
  b->built = false;
  b->drop_graph();
  return BIOT_OK;
}

extern "C" int biot_batch_shot_count(biot_batch *b, int32_t *n)
{
  if (!b || !n) return BIOT_ERR_ARG;
  *n = (int32_t)b->shots.size();
  return BIOT_OK;
}

namespace {

// tile shape and grid for shots [s0, s1) where neither the caller nor the autotuner chose them:
// the shape a single grid of as many waves gets, and one block per tile (a smaller grid that
// takes its tiles from the work queue is 6 % slower over 16 windows of 96-187 cells)
void default_launch(biot_batch *b, int s0, int s1)
{
  int64_t waves = 0, tiles = 0;
  for (int i = s0; i < s1; ++i) waves += plane_waves(b->shots[i].h->g);
  b->shape = default_shape(b->cfg.precision, waves);
  for (int i = s0; i < s1; ++i) {
    StepArgs a;
    b->shots[i].h->fill_args(a);
    set_tiles(a, b->shape, b->cfg.order / 2);
    tiles += a.ntiles;
  }
  b->blocks = (int)((tiles + 7) / 8 * 8);
}

// device tables of the forward launches for the current shape, for shots [s0, s1) (all
// shots when s1 < 0); the tables hold the subset from their first entry
int build_tables(biot_batch *b, int s0 = 0, int s1 = -1)
{
  const bool all = s1 < 0;
  if (all && b->built) return BIOT_OK;
  if (all) s1 = (int)b->shots.size();
  const int S = s1 - s0;
  if (S <= 0) return bfail(b, BIOT_ERR_STATE, "no shots");
  if (!b->launch_set) default_launch(b, s0, s1);
  const int Sall = (int)b->shots.size();
  std::vector<StepArgs> st(S);
  std::vector<int> tiles(S + 1, 0);
  std::vector<SourceArgs> src(S);
  std::vector<RecordArgs> rec(S);
  b->max_nrec = b->cells = b->state = 0;
  b->fused = true;
  const int h2 = b->cfg.order / 2;
  for (int i = 0; i < S; ++i) {
    biot_handle *h = b->shots[s0 + i].h;
    StepArgs &a = st[i];
    h->fill_args(a);
    set_tiles(a, b->shape, h2);
    tiles[i + 1] = tiles[i] + a.ntiles;
    b->cells += h->n;
    b->state += (int64_t)h->state_bytes();
    h->source_args(src[i]);
    h->record_args(rec[i]);
    b->max_nrec = std::max(b->max_nrec, h->nrec);
    b->fused = b->fused && !h->source_recorded() && (!h->src_mask || h->source_in_stress());
  }
  b->total_tiles = tiles[S];
  b->nactive = S;
  if (!b->d_step) {
    BHIP(b, hipMalloc((void **)&b->d_step, Sall * sizeof(StepArgs)));
    BHIP(b, hipMalloc((void **)&b->d_tiles, (Sall + 1) * sizeof(int)));
    BHIP(b, hipMalloc((void **)&b->d_src, Sall * sizeof(SourceArgs)));
    BHIP(b, hipMalloc((void **)&b->d_rec, Sall * sizeof(RecordArgs)));
  }
  BHIP(b, hipMemcpy(b->d_step, st.data(), S * sizeof(StepArgs), hipMemcpyHostToDevice));
  BHIP(b, hipMemcpy(b->d_tiles, tiles.data(), (S + 1) * sizeof(int), hipMemcpyHostToDevice));
  BHIP(b, hipMemcpy(b->d_src, src.data(), S * sizeof(SourceArgs), hipMemcpyHostToDevice));
  BHIP(b, hipMemcpy(b->d_rec, rec.data(), S * sizeof(RecordArgs), hipMemcpyHostToDevice));
  b->built = all;
  if (!all) b->drop_graph();  // a captured graph refers to the full tables
  return BIOT_OK;
}

BatchArgs batch_args(const biot_batch *b)
{
  // a grid smaller than the tile list takes its tiles from the work queue
  int *q = b->blocks < b->total_tiles ? b->d_queue : nullptr;
  BatchArgs a{};
  a.shots = b->d_step;
  a.tile_start = b->d_tiles;
  a.nshots = b->nactive;
  a.total_tiles = b->total_tiles;
  a.cells = b->cells;
  a.state = b->state;
  a.queue = q;
  a.src = b->fused ? b->d_src : nullptr;
  a.rec = b->d_rec;
  a.it = b->d_it;
  a.q = -1;
  return a;
}

// step `off` after the counter's of every shot: velocity, stress, and the source of the next
// step and the recorded samples on them (FuseArgs); where a shot's source or receivers cannot
// ride on the half steps, source and record launches for all.  The first step's source is
// start_steps' launch, the last step's stresses and p are end_steps'.
int enqueue_step(biot_batch *b, bool record, int off)
{
  const int prec = b->cfg.precision, order = b->cfg.order;
  BatchArgs ba = batch_args(b);
  ba.off = off;
  const int64_t rec = record && b->fused ? b->max_nrec : 0;
  if (!b->fused) BHIP(b, launch_source_batch(prec, b->d_src, b->nactive, b->d_it, off, -1, b->stream));
  BHIP(b, launch_step_batch(prec, order, true, ba, b->shape, b->blocks, rec, b->stream));
  BHIP(b, launch_step_batch(prec, order, false, ba, b->shape, b->blocks, rec, b->stream));
  if (record && !b->fused)
    BHIP(b, launch_record_batch(prec, b->d_rec, b->nactive, b->max_nrec, true, b->d_it, off, b->stream));
  return BIOT_OK;
}

// the counter at step `it` of a run of n steps, its first source added
int start_steps(biot_batch *b, int it, int n)
{
  BHIP(b, launch_set_counter(b->d_it, it, it + n, b->stream));
  if (b->fused)
    BHIP(b, launch_source_batch(b->cfg.precision, b->d_src, b->nactive, b->d_it, 0, -1, b->stream));
  return BIOT_OK;
}
// the counter is past the run's last step (off: its distance from the counter)
int end_steps(biot_batch *b, bool record, int off)
{
  if (record && b->fused)
    BHIP(b, launch_record_batch(b->cfg.precision, b->d_rec, b->nactive, b->max_nrec, false, b->d_it, off, b->stream));
  return BIOT_OK;
}

int ensure_graph(biot_batch *b, int steps, bool record)
{
  if (b->gexec && b->g_steps == steps && b->g_record == record) return BIOT_OK;
  b->drop_graph();
  hipGraph_t graph = nullptr;
  BHIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  int rc = BIOT_OK;
  for (int s = 0; s < steps && !rc; ++s) rc = enqueue_step(b, record, s);
  if (!rc && launch_advance(b->d_it, steps, b->stream) != hipSuccess) rc = BIOT_ERR_HIP;
  hipGraph_t g2 = nullptr;
  const hipError_t e = hipStreamEndCapture(b->stream, &g2);
  graph = g2;
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (e != hipSuccess) return bfail(b, BIOT_ERR_HIP, "graph capture: %s", hipGetErrorString(e));
  const hipError_t e2 = hipGraphInstantiate(&b->gexec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e2 != hipSuccess) {
    b->gexec = nullptr;
    return bfail(b, BIOT_ERR_HIP, "graph instantiate: %s", hipGetErrorString(e2));
  }
  b->g_steps = steps;
  b->g_record = record;
  return BIOT_OK;
}

// steps it..it+nt-1: whole graphs, then single steps
int run_steps(biot_batch *b, int it, int nt, int graph_steps, bool record)
{
  int rc = start_steps(b, it, nt);
  if (rc) return rc;
  int done = 0;
  if (graph_steps > 0 && nt >= graph_steps) {
    if ((rc = ensure_graph(b, graph_steps, record))) return rc;
    for (; done + graph_steps <= nt; done += graph_steps) BHIP(b, hipGraphLaunch(b->gexec, b->stream));
  }
  int off = 0;
  for (; done < nt; ++done, ++off)
    if ((rc = enqueue_step(b, record, off))) return rc;
  return end_steps(b, record, off - 1);
}

int reset_all(biot_batch *b)
{
  for (auto &s : b->shots) {
    int rc = biot_reset(s.h);
    if (rc) return hfail(b, s.h, rc, "reset");
  }
  return BIOT_OK;
}

}  // namespace

extern "C" int biot_batch_set_launch(biot_batch *b, int32_t bx, int32_t by, int32_t zchunk, int32_t blocks)
{
  if (!b) return BIOT_ERR_ARG;
  if (bx < 64 || bx % 64 || by < 1 || bx * by > 256 || zchunk < 1 || blocks < 8 || blocks % 8)
    return bfail(b, BIOT_ERR_ARG, "launch %dx%d, zchunk %d, %d blocks not allowed", bx, by, zchunk, blocks);
  b->shape = LaunchShape{bx, by, zchunk};
  b->blocks = blocks;
  b->launch_set = true;
  b->built = false;
  b->drop_graph();
  return BIOT_OK;
}

extern "C" int biot_batch_get_launch(biot_batch *b, int32_t *bx, int32_t *by, int32_t *zchunk, int32_t *blocks)
{
  if (!b || !bx || !by || !zchunk || !blocks) return BIOT_ERR_ARG;
  if (!b->launch_set && !b->shots.empty()) default_launch(b, 0, (int)b->shots.size());
  *bx = b->shape.bx;
  *by = b->shape.by;
  *zchunk = b->shape.zchunk;
  *blocks = b->blocks;
  return BIOT_OK;
}

extern "C" int biot_batch_autotune(biot_batch *b, int32_t trial_steps)
{
  if (!b) return BIOT_ERR_ARG;
  if (trial_steps < 1 || trial_steps > 1000) return bfail(b, BIOT_ERR_ARG, "trial_steps must be 1..1000");
  if (b->shots.empty()) return bfail(b, BIOT_ERR_STATE, "no shots");
  static const int shapes[][2] = {{64, 4}, {64, 2}, {64, 1}, {128, 2}, {128, 1}, {256, 1}};
  static const int chunks[] = {2, 3, 4, 8, 16};
  static const int grids[] = {1024, 2048, 4096, 1 << 30};
  const LaunchShape keep = b->shape;
  const int keep_blocks = b->blocks;
  const bool keep_set = b->launch_set;
  b->launch_set = true;
  LaunchShape best = keep;
  int best_blocks = keep_blocks;
  double best_ms = 1e30;
  int rc = reset_all(b);
  for (auto &sh : shapes)
    for (int zc : chunks)
      for (int gblocks : grids) {
        if (rc) break;
        b->shape = LaunchShape{sh[0], sh[1], zc};
        b->built = false;
        b->drop_graph();
        if ((rc = build_tables(b))) break;
        const int gb = std::min(gblocks, ((b->total_tiles + 7) / 8) * 8);
        if (gblocks == (1 << 30) || gb == gblocks) b->blocks = gb;
        else continue;  // a grid larger than the tile list is the "one block per tile" case
        if ((rc = start_steps(b, 0, trial_steps + 1))) break;
        if ((rc = enqueue_step(b, false, 0))) break;  // warm-up
        float ms = 0;
        if (hipEventRecord(b->ev0, b->stream) != hipSuccess) rc = BIOT_ERR_HIP;
        for (int s = 0; s < trial_steps && !rc; ++s) rc = enqueue_step(b, false, s + 1);
        if (!rc && (hipEventRecord(b->ev1, b->stream) != hipSuccess || hipEventSynchronize(b->ev1) != hipSuccess ||
                    hipEventElapsedTime(&ms, b->ev0, b->ev1) != hipSuccess))
          rc = BIOT_ERR_HIP;
        if (!rc && ms < best_ms) {
          best_ms = ms;
          best = b->shape;
          best_blocks = b->blocks;
        }
      }
  b->shape = rc ? keep : best;
  b->blocks = rc ? keep_blocks : best_blocks;
  b->launch_set = rc ? keep_set : true;
  b->built = false;
  b->drop_graph();
  if (rc) return rc == BIOT_ERR_HIP ? bfail(b, rc, "autotune timing failed") : rc;
  return reset_all(b);
}

extern "C" int biot_batch_forward(biot_batch *b, int32_t nt, int32_t graph_steps)
{
  if (!b) return BIOT_ERR_ARG;
  if (nt <= 0 || graph_steps < 0) return bfail(b, BIOT_ERR_ARG, "nt must be positive, graph_steps >= 0");
  int rc = build_tables(b);
  if (!rc) rc = reset_all(b);
  if (rc) return rc;
  BHIP(b, hipEventRecord(b->ev0, b->stream));
  rc = run_steps(b, 0, nt, graph_steps, true);
  if (rc) return rc;
  BHIP(b, hipEventRecord(b->ev1, b->stream));
  BHIP(b, hipEventSynchronize(b->ev1));
  float ms = 0;
  BHIP(b, hipEventElapsedTime(&ms, b->ev0, b->ev1));
  b->last_ms = ms;
  for (auto &s : b->shots) s.h->it = nt;
  for (size_t i = 0; i < b->shots.size(); ++i)
    if ((rc = b->shots[i].h->check_nonfinite())) {
      char what[32];
      snprintf(what, sizeof what, "shot %d", (int)i);
      return hfail(b, b->shots[i].h, rc, what);
    }
  return BIOT_OK;
}

extern "C" int biot_batch_read_traces(biot_batch *b, int32_t shot, float *out, int64_t count)
{
  if (!b || !out) return BIOT_ERR_ARG;
  if (shot < 0 || shot >= (int)b->shots.size()) return bfail(b, BIOT_ERR_ARG, "no shot %d", shot);
  biot_handle *h = b->shots[shot].h;
  int rc = biot_read_traces(h, out, count);
  return rc ? hfail(b, h, rc, "read traces") : BIOT_OK;
}

extern "C" int biot_batch_shot_handle(biot_batch *b, int32_t shot, biot_handle **h)
{
  if (!b || !h) return BIOT_ERR_ARG;
  if (shot < 0 || shot >= (int)b->shots.size()) return bfail(b, BIOT_ERR_ARG, "no shot %d", shot);
  *h = b->shots[shot].h;
  return BIOT_OK;
}

namespace {

// device bytes the gradient needs for one shot
size_t shot_gradient_bytes(const biot_handle *h, int nseg, int every)
{
  const int64_t m = (int64_t)h->ncomp * h->nt_max * h->nrec;
  return h->state_bytes() * (size_t)(nseg + every + 1) + h->lam_bytes() +
         (size_t)NKC * h->n * (sizeof(double) + (h->prec == BIOT_FP64 ? 0 : sizeof(float))) +
         (h->prec == BIOT_FP16M ? (size_t)NKC * h->n * sizeof(_Float16) : 0) +  // adjoint coefficients
         (size_t)8 * h->n * sizeof(double) +
         (size_t)2 * std::max<int64_t>(m, 1) * sizeof(float);
}

// the gradient of shots [s0, s1): checkpointed forward, misfit, recompute + adjoint, chain
int gradient_group(biot_batch *b, int s0, int s1, int nt, int every, const float *const observed[])
{
  const int S = s1 - s0;
  const int prec = b->cfg.precision, order = b->cfg.order;
  const int nseg = (nt + every - 1) / every;
  const int64_t N = (int64_t)b->cfg.nx * b->cfg.ny * b->cfg.nz;
  int rc = build_tables(b, s0, s1);
  if (rc) return rc;
  for (int i = s0; i < s1; ++i) {
    auto &s = b->shots[i];
    biot_handle *h = s.h;
    if ((rc = h->alloc_adjoint(every))) return hfail(b, h, rc, "adjoint buffers");
    if ((rc = h->build_adjoint_coefs())) return hfail(b, h, rc, "adjoint coefficients");
    while ((int)s.ckpt.size() < nseg) {
      void *p = nullptr;
      if (hipMalloc(&p, h->state_bytes()) != hipSuccess)
        return bfail(b, BIOT_ERR_NOMEM, "checkpoints of shot %d do not fit", i);
      s.ckpt.push_back(p);
    }
    const int64_t m = (int64_t)h->ncomp * h->nt_max * h->nrec;
    if (!s.d_par) BHIP(b, hipMalloc((void **)&s.d_par, (size_t)8 * h->n * sizeof(double)));
    if (!s.d_obs) BHIP(b, hipMalloc((void **)&s.d_obs, (size_t)std::max<int64_t>(m, 1) * sizeof(float)));
  }
  // adjoint / inject tables
  {
    std::vector<AdjArgs> adj(S);
    std::vector<InjectArgs> inj(S);
    std::vector<int> bs(S + 1, 0);
    for (int i = 0; i < S; ++i) {
      b->shots[s0 + i].h->adj_args(adj[i]);
      b->shots[s0 + i].h->inject_args(inj[i]);
      bs[i + 1] = bs[i] + adj[i].blocks;
    }
    b->adj_blocks = bs[S];
    if (!b->d_adj) BHIP(b, hipMalloc((void **)&b->d_adj, S * sizeof(AdjArgs)));
    if (!b->d_blocks) BHIP(b, hipMalloc((void **)&b->d_blocks, (S + 1) * sizeof(int)));
    if (!b->d_inj) BHIP(b, hipMalloc((void **)&b->d_inj, S * sizeof(InjectArgs)));
    BHIP(b, hipMemcpy(b->d_adj, adj.data(), S * sizeof(AdjArgs), hipMemcpyHostToDevice));
    BHIP(b, hipMemcpy(b->d_blocks, bs.data(), (S + 1) * sizeof(int), hipMemcpyHostToDevice));
    BHIP(b, hipMemcpy(b->d_inj, inj.data(), S * sizeof(InjectArgs), hipMemcpyHostToDevice));
    // the half steps' and sources' arguments over the segment states
    std::vector<StepArgs> st(S);
    std::vector<SourceArgs> src(S);
    std::vector<RecordArgs> rec(S);
    for (int i = 0; i < S; ++i) {
      biot_handle *h = b->shots[s0 + i].h;
      h->fill_args(st[i], (char *)h->d_slots);
      set_tiles(st[i], b->shape, order / 2);
      h->source_args(src[i], (char *)h->d_slots);
      h->record_args(rec[i], (char *)h->d_slots);
    }
    if (!b->d_step_s) BHIP(b, hipMalloc((void **)&b->d_step_s, S * sizeof(StepArgs)));
    if (!b->d_src_s) BHIP(b, hipMalloc((void **)&b->d_src_s, S * sizeof(SourceArgs)));
    BHIP(b, hipMemcpy(b->d_step_s, st.data(), S * sizeof(StepArgs), hipMemcpyHostToDevice));
    if (!b->d_rec_s) BHIP(b, hipMalloc((void **)&b->d_rec_s, S * sizeof(RecordArgs)));
    BHIP(b, hipMemcpy(b->d_src_s, src.data(), S * sizeof(SourceArgs), hipMemcpyHostToDevice));
    BHIP(b, hipMemcpy(b->d_rec_s, rec.data(), S * sizeof(RecordArgs), hipMemcpyHostToDevice));
  }
  // copy tables: [save ckpt k] nseg entries of 5 pieces per shot (fields, the three carry blocks,
  // the residuals: 0 bytes on the policies without), [ckpt k to the first segment state] nseg of one,
  // [the last segment's last state to the live arrays] 5 pieces per shot
  constexpr int NP = 5;
  const int per = NP * S;
  {
    std::vector<CopyEntry> tab((size_t)nseg * (per + S) + per);
    for (int i = 0; i < S; ++i) {
      biot_handle *h = b->shots[s0 + i].h;
      char *live[NP] = {(char *)h->d_fields, (char *)h->d_carry[0], (char *)h->d_carry[1], (char *)h->d_carry[2],
                        (char *)h->d_lo};
      const size_t bytes[NP] = {(size_t)NFIELD * h->n * h->esz, (size_t)NCARRY * h->slab[0] * h->csz,
                                (size_t)NCARRY * h->slab[1] * h->csz, (size_t)NCARRY * h->slab[2] * h->csz,
                                h->d_lo ? h->lo_bytes() : 0};
      for (int k = 0; k < nseg; ++k) {
        char *ckpt = (char *)b->shots[s0 + i].ckpt[k];
        for (int p = 0; p < NP; ++p)
          tab[(size_t)k * per + NP * i + p] =
              CopyEntry{live[p], ckpt + (p < 4 ? h->state_off(p) : h->state_lo_off()), bytes[p]};
        tab[(size_t)nseg * per + (size_t)k * S + i] = CopyEntry{ckpt, h->d_slots, h->state_bytes()};
      }
      const char *end = (const char *)h->d_slots + (size_t)(nt - (nseg - 1) * every) * h->state_bytes();
      for (int p = 0; p < NP; ++p)
        tab[(size_t)nseg * (per + S) + NP * i + p] =
            CopyEntry{end + (p < 4 ? h->state_off(p) : h->state_lo_off()), live[p], bytes[p]};
    }
    if (!b->d_copy) BHIP(b, hipMalloc((void **)&b->d_copy, tab.size() * sizeof(CopyEntry)));
    BHIP(b, hipMemcpy(b->d_copy, tab.data(), tab.size() * sizeof(CopyEntry), hipMemcpyHostToDevice));
  }
  auto save_ckpt = [&](int k) { return launch_copy_batch(b->d_copy + (size_t)k * per, per, b->stream); };
  auto load_ckpt = [&](int k) {
    return launch_copy_batch(b->d_copy + (size_t)nseg * per + (size_t)k * S, S, b->stream);
  };
  for (int i = s0; i < s1; ++i) {
    int r = biot_reset(b->shots[i].h);
    if (r) return hfail(b, b->shots[i].h, r, "reset");
  }

  // the steps of a segment from state to state, the first one the checkpoint's; a shot's source that
  // no stress launch can add has every shot's added by launches of their own
  auto segment = [&](int k, int64_t record) -> int {
    const int n0 = k * every, K = std::min(every, nt - n0);
    BHIP(b, load_ckpt(k));
    BHIP(b, launch_set_counter(b->d_it, n0, n0 + K, b->stream));
    for (int q = 0; q < K; ++q) {
      if (q == 0 || !b->fused) BHIP(b, launch_source_batch(prec, b->d_src_s, S, b->d_it, q, q, b->stream));
      BatchArgs ba = batch_args(b);
      ba.shots = b->d_step_s;
      ba.src = b->fused ? b->d_src_s : nullptr;
      ba.rec = b->d_rec_s;
      ba.off = ba.q = q;
      BHIP(b, launch_step_batch(prec, order, true, ba, b->shape, b->blocks, record, b->stream));
      BHIP(b, launch_step_batch(prec, order, false, ba, b->shape, b->blocks, record, b->stream));
    }
    return BIOT_OK;
  };
  // ---- forward with checkpoints; the last segment through the segment states, where the sweep finds
  // them (all shots' receivers have to ride on the half steps for that)
  const bool hold = b->fused;
  for (int k = 0; k < nseg; ++k) {
    BHIP(b, save_ckpt(k));
    if (hold && k == nseg - 1) {
      if ((rc = segment(k, b->max_nrec))) return rc;
      BHIP(b, launch_copy_batch(b->d_copy + (size_t)nseg * (per + S), per, b->stream));
      rc = end_steps(b, true, nt - k * every - 1);
    } else {
      rc = run_steps(b, k * every, std::min(every, nt - k * every), 0, true);
    }
    if (rc) return rc;
  }
  // the window parameters and the observed traces go up while the forward sweep runs
  if (!b->side) BHIP(b, hipStreamCreate(&b->side));
  for (int i = s0; i < s1; ++i) {
    auto &s = b->shots[i];
    const int64_t m = (int64_t)s.h->ncomp * s.h->nt_max * s.h->nrec;
    for (int q = 0; q < 8; ++q)
      BHIP(b, hipMemcpyAsync(s.d_par + (size_t)q * s.h->n, s.h->par[q].data(), (size_t)s.h->n * sizeof(double),
                             hipMemcpyHostToDevice, b->side));
    BHIP(b, hipMemcpyAsync(s.d_obs, observed[i], (size_t)m * sizeof(float), hipMemcpyHostToDevice, b->side));
  }
  BHIP(b, hipStreamSynchronize(b->side));
  // ---- FP64 misfit per shot; the residual is the adjoint source
  for (int i = s0; i < s1; ++i) {
    biot_handle *h = b->shots[i].h;
    const int64_t m = (int64_t)h->ncomp * h->nt_max * h->nrec;
    const bool dbl = h->d_traces64 != nullptr;
    BHIP(b, launch_misfit(dbl ? (const void *)h->d_traces64 : h->d_traces, dbl, b->shots[i].d_obs,
                          h->d_adjsrc, m, b->d_J, b->stream));
    BHIP(b, hipMemsetAsync(h->d_lam, 0, h->lam_bytes(), b->stream));
    BHIP(b, hipMemsetAsync(h->d_grad, 0, (size_t)NKC * h->n * sizeof(double), b->stream));
    if (h->d_gpart) BHIP(b, hipMemsetAsync(h->d_gpart, 0, (size_t)NKC * h->n * sizeof(float), b->stream));
  }
  // ---- segment recompute and adjoint sweep, all shots of the group per launch
  const AdjBatch ab{b->d_adj, b->d_blocks, S, b->adj_blocks, b->d_inj};
  for (int k = nseg - 1; k >= 0; --k) {
    const int n0 = k * every, K = std::min(every, nt - n0);
    if (!(hold && k == nseg - 1))
      if ((rc = segment(k, 0))) return rc;
    for (int it = n0 + K - 1; it >= n0; --it) BHIP(b, launch_adjoint_step_batch(prec, order, ab, it - n0, it, b->stream));
    BHIP(b, launch_adjoint_flush_batch(prec, order, ab, b->stream));
  }
  // ---- chain rule per shot into the model-grid gradient
  for (int i = s0; i < s1; ++i) {
    auto &s = b->shots[i];
    biot_handle *h = s.h;
    ChainArgs c{};
    for (int k = 0; k < NKC; ++k) {
      c.grad[k] = h->d_grad + (size_t)k * h->n;
      c.kfac[k] = h->kfac[k];
    }
    for (int q = 0; q < 8; ++q) c.par[q] = s.d_par + (size_t)q * h->n;
    for (int q = 0; q < 6; ++q) c.out[q] = b->d_gout + (size_t)q * N;
    c.wx = h->g.nx;
    c.wy = h->g.ny;
    c.wz = h->g.nz;
    c.x0 = s.x0;
    c.y0 = s.y0;
    c.z0 = s.z0;
    c.msy = b->cfg.nx;
    c.msz = (int64_t)b->cfg.nx * b->cfg.ny;
    c.dt = b->cfg.dt;
    c.Cv = b->cfg.Cv;
    c.Cp = b->cfg.Cp;
    c.Hinv = (double)(1.0f / b->cfg.dx);
    c.add = 1;
    BHIP(b, launch_chain(c, b->stream));
  }
  for (int i = s0; i < s1; ++i) b->shots[i].h->it = nt;
  return BIOT_OK;
}

// releases the per-shot gradient buffers of shots [s0, s1) and the group tables
void free_group(biot_batch *b, int s0, int s1)
{
  (void)hipStreamSynchronize(b->stream);
  for (int i = s0; i < s1; ++i) {
    auto &s = b->shots[i];
    for (void *p : s.ckpt)
      if (p) (void)hipFree(p);
    s.ckpt.clear();
    dfree(s.d_par);
    dfree(s.d_obs);
    s.h->free_adjoint();
  }
  b->room_every = b->room_nt = 0;
  dfree(b->d_adj);
  dfree(b->d_blocks);
  dfree(b->d_inj);
  dfree(b->d_copy);
  dfree(b->d_step_s);
  dfree(b->d_src_s);
  dfree(b->d_rec_s);
}

}  // namespace

extern "C" int biot_batch_gradient(biot_batch *b, int32_t nt, int32_t every, const float *const observed[],
                                   double *J, double *const grad[6])
{
  if (!b) return BIOT_ERR_ARG;
  if (!observed || !J || !grad) return bfail(b, BIOT_ERR_ARG, "observed, J and grad are required");
  for (int q = 0; q < 6; ++q)
    if (!grad[q]) return bfail(b, BIOT_ERR_ARG, "grad[%d] is null", q);
  const int S = (int)b->shots.size();
  if (S == 0) return bfail(b, BIOT_ERR_STATE, "no shots");
  if (nt <= 0 || every <= 0) return bfail(b, BIOT_ERR_ARG, "nt and every must be positive");
  for (int i = 0; i < S; ++i) {
    if (!observed[i]) return bfail(b, BIOT_ERR_ARG, "observed[%d] is null", i);
    if (b->shots[i].h->nt_max < nt) return bfail(b, BIOT_ERR_ARG, "shot %d records fewer than nt steps", i);
    if (b->shots[i].h->src_mask & 0x3Fu)
      return bfail(b, BIOT_ERR_ARG, "shot %d: the adjoint path supports sources on stresses and pressure only", i);
  }
  const int nseg = (nt + every - 1) / every;
  const int64_t N = (int64_t)b->cfg.nx * b->cfg.ny * b->cfg.nz;
  // The buffers of a gradient of all shots in one group serve the next one with the same steps and
  // checkpoints, if they hold at most an eighth of the device's memory; new shots, a new model and
  // biot_batch_release release them, and a shot's own handle does where it is given another source,
  // receivers, parameters or checkpointed run.  Reserving and releasing them took half of the 17 ms
  // that a gradient of 4 windows of 36-73 cells spent around its 25 ms on the GPU.
  bool room = b->room_every == every && b->room_nt == nt;
  for (int i = 0; i < S && room; ++i) {
    const biot_handle *h = b->shots[i].h;
    room = h->d_slots && h->slots_every == every && h->d_lam && h->d_grad && h->d_adjsrc && h->d_inj && h->ckpt.empty();
  }
  size_t free_b = 0, total_b = 0, held = 0;
  if (!room) {
    b->free_gradient();
    BHIP(b, hipMalloc((void **)&b->d_gout, (size_t)6 * N * sizeof(double)));
    BHIP(b, hipMalloc((void **)&b->d_J, sizeof(double)));
    BHIP(b, hipMemGetInfo(&free_b, &total_b));
  }
  // shots go in groups that fit the free device memory (one group when they all fit)
  const size_t budget = (size_t)((double)free_b * 0.9);
  std::vector<std::pair<int, int>> groups;
  if (room) groups.emplace_back(0, S);
  for (int i = 0; i < S && !room;) {
    size_t used = 0;
    int j = i;
    while (j < S) {
      const size_t need = shot_gradient_bytes(b->shots[j].h, nseg, every);
      if (j > i && used + need > budget) break;
      used += need;
      ++j;
    }
    groups.emplace_back(i, j);
    held += used;
    i = j;
  }
  const bool keep = room || (groups.size() == 1 && held <= total_b / 8);
  BHIP(b, hipMemsetAsync(b->d_gout, 0, (size_t)6 * N * sizeof(double), b->stream));
  BHIP(b, hipMemsetAsync(b->d_J, 0, sizeof(double), b->stream));
  BHIP(b, hipEventRecord(b->ev0, b->stream));
  int rc = BIOT_OK;
  for (auto &g : groups) {
    rc = gradient_group(b, g.first, g.second, nt, every, observed);
    if (rc || !keep) free_group(b, g.first, g.second);
    if (rc) break;
  }
  b->built = false;
  if (rc) return rc;
  if (keep) b->room_every = every, b->room_nt = nt;
  BHIP(b, hipEventRecord(b->ev1, b->stream));
  BHIP(b, hipEventSynchronize(b->ev1));
  float ms = 0;
  BHIP(b, hipEventElapsedTime(&ms, b->ev0, b->ev1));
  b->last_ms = ms;
  b->groups = (int)groups.size();
  BHIP(b, hipMemcpy(J, b->d_J, sizeof(double), hipMemcpyDeviceToHost));
  std::vector<ReadBack::Piece> pieces;
  for (int q = 0; q < 6; ++q) pieces.push_back({grad[q], b->d_gout + (size_t)q * N, (size_t)N * sizeof(double)});
  if (!b->back.read(pieces, b->cfg.device, b->stream)) return bfail(b, BIOT_ERR_HIP, "reading the gradients failed");
  return BIOT_OK;
}

extern "C" int biot_batch_gradient_groups(biot_batch *b, int32_t *groups)
{
  if (!b || !groups) return BIOT_ERR_ARG;
  *groups = b->groups;
  return BIOT_OK;
}

extern "C" int biot_batch_last_ms(biot_batch *b, double *ms)
{
  if (!b || !ms) return BIOT_ERR_ARG;
  *ms = b->last_ms;
  return BIOT_OK;
}

extern "C" int biot_batch_release(biot_batch *b)
{
  if (!b) return BIOT_ERR_ARG;
  b->free_gradient();
  return BIOT_OK;
}
