// Batched numeric assembly of libgdx: many independent problems (uneven
// sizes and partitions) assembled by one graph launch.
//
//   gdx_batch_add       problems after their symbolic phase, on one context
//   gdx_batch_autotune  sets every 3D diffusion problem's matrix kernel to the
//                       pair-lattice kernel and times nothing: 3D Q2 64^3 0.42 ms
//                       against 0.79 (z-marching) and 0.63 (per tile); Q1
//                       131 x 97 x 75 0.050 ms against 0.45 (z-marching)
//   gdx_batch_capture   records every problem's numeric launches (coefficient,
//                       RHS and matrix kernels; no memsets) into one hipGraph:
//                       the diffusion problems on the uniform box go together,
//                       the tiles of all of them in one launch (and their
//                       coefficients in two); the others are independent
//                       branches, spread over kBranches streams (largest first,
//                       each to the branch with the least work), forked from
//                       and joined back into the context's stream
//   gdx_batch_launch    replays it on the context's stream
//
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "gdx_internal.h"

struct gdx_batch {
  gdx_ctx *ctx = nullptr;
  std::vector<gdx_problem *> probs;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  // the diffusion problems on the uniform box, together in a few launches
  gdx::LatticeBatch *lattice = nullptr;
  gdx::CoefBatch *coef = nullptr;
  // tables of dropped graphs, not yet freed
  std::vector<gdx::LatticeBatch *> old_lattice;
  std::vector<gdx::CoefBatch *> old_coef;
  // capture-time fork/join streams and events (default priority)
  std::vector<hipStream_t> side;
  std::vector<hipEvent_t> ev;  // [0] fork, [1..] joins
};

namespace {

// branches of the batch graph: the context's stream plus kBranches - 1 side
// streams (the device runs at most 4 hardware queues per process by default)
constexpr int kBranches = 4;

int ensure_branches(gdx_batch *b) {
  while ((int)b->side.size() < kBranches - 1) {
    hipStream_t s;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return GDX_ERR_HIP;
    b->side.push_back(s);
  }
  while ((int)b->ev.size() < kBranches) {
    hipEvent_t e;
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return GDX_ERR_HIP;
    b->ev.push_back(e);
  }
  return GDX_OK;
}

void free_branches(gdx_batch *b) {
  for (hipStream_t s : b->side) (void)hipStreamDestroy(s);
  for (hipEvent_t e : b->ev) (void)hipEventDestroy(e);
  b->side.clear();
  b->ev.clear();
}

int fail(int code, const char *msg) {
  gdx::set_error(msg);
  return code;
}

void drop_graph(gdx_batch *b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
  if (b->lattice) b->old_lattice.push_back(b->lattice);
  if (b->coef) b->old_coef.push_back(b->coef);
  b->lattice = nullptr;
  b->coef = nullptr;
  if (b->old_lattice.empty() && b->old_coef.empty()) return;
  // a replay in flight reads the tables; while a caller captures the stream it can
  // neither be waited for nor memory freed, and they stay until the next time
  if (b->ctx) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(b->ctx->stream, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone)
      return;
    (void)hipStreamSynchronize(b->ctx->stream);
  }
  for (gdx::LatticeBatch *t : b->old_lattice) gdx::lattice_batch_free(t);
  for (gdx::CoefBatch *t : b->old_coef) gdx::coef_batch_free(t);
  b->old_lattice.clear();
  b->old_coef.clear();
}

}  // namespace

extern "C" {

int gdx_batch_create(gdx_ctx *ctx, gdx_batch **out) {
  if (!ctx || !out) return fail(GDX_ERR_ARG, "NULL argument");
  *out = new (std::nothrow) gdx_batch;
  if (!*out) return fail(GDX_ERR_ALLOC, "host allocation failed");
  (*out)->ctx = ctx;
  ctx->batches.push_back(*out);
  return GDX_OK;
}

int gdx_batch_add(gdx_batch *b, gdx_problem *p) {
  if (!b || !p) return fail(GDX_ERR_ARG, "NULL argument");
  if (!b->ctx) return fail(GDX_ERR_STATE, "the batch's context was finalized");
  if (p->ctx != b->ctx) return fail(GDX_ERR_ARG, "the problem belongs to another context");
  if (!p->symbolic_done) return fail(GDX_ERR_STATE, "gdx_symbolic has not run");
  if (std::find(b->probs.begin(), b->probs.end(), p) != b->probs.end())
    return fail(GDX_ERR_ARG, "the problem is already in the batch");
  drop_graph(b);
  b->probs.push_back(p);
  return GDX_OK;
}

int gdx_batch_autotune(gdx_batch *b, int32_t reps, int32_t *chosen) {
  if (!b || reps < 1 || reps > 100) return fail(GDX_ERR_ARG, "invalid argument");
  if (!b->ctx) return fail(GDX_ERR_STATE, "the batch's context was finalized");
  if (hipSetDevice(b->ctx->device) != hipSuccess) return fail(GDX_ERR_HIP, "hipSetDevice failed");
  drop_graph(b);
  int rc = GDX_OK;
  for (size_t i = 0; i < b->probs.size() && !rc; ++i) {
    gdx_problem *p = b->probs[i];
    p->precision = GDX_PREC_FP64;  // the choice is made for (and applies to) the FP64 form
    p->hbm_patterns = false;       // and for the tiles' usual pattern placement
    if (p->D == 3 && p->desc.op_kind == GDX_OP_DIFFUSION) rc = gdx::set_kernel_variant(p, 2, 0);
    if (chosen) chosen[i] = p->kvariant3d == 0 ? p->tileR[2] : -p->kvariant3d;
  }
  if (rc) gdx::set_error("autotuning failed");
  return rc;
}

int gdx_batch_capture(gdx_batch *b) {
  if (!b) return fail(GDX_ERR_ARG, "NULL argument");
  if (!b->ctx) return fail(GDX_ERR_STATE, "the batch's context was finalized");
  if (b->probs.empty()) return fail(GDX_ERR_STATE, "the batch is empty");
  if (hipSetDevice(b->ctx->device) != hipSuccess) return fail(GDX_ERR_HIP, "hipSetDevice failed");
  hipStream_t st = b->ctx->stream;
  drop_graph(b);
  if (hipStreamSynchronize(st) != hipSuccess) return fail(GDX_ERR_HIP, "stream failed");
  if (ensure_branches(b)) return fail(GDX_ERR_HIP, "stream or event creation failed");
  // the diffusion problems of the pair-lattice kernel go together, on the first branch
  std::vector<gdx_problem *> lat, points, rest;
  double lat_work = 0.0;
  for (gdx_problem *p : b->probs) {
    if (p->desc.op_kind != GDX_OP_DIFFUSION || p->mapped || !gdx::lattice_used(p)) {
      rest.push_back(p);
      continue;
    }
    lat.push_back(p);
    if (gdx::points_used(p)) points.push_back(p);
    lat_work += (double)p->nnz_total;
  }
  if ((!lat.empty() && gdx::lattice_batch_build(lat, &b->lattice)) ||
      (!points.empty() && gdx::coef_batch_build(points, &b->coef))) {
    drop_graph(b);
    return fail(GDX_ERR_ALLOC, "the batch's tables do not fit in device memory");
  }
  // the others: largest first, each to the least loaded branch (work = stored values);
  // within a branch they keep the batch order
  const int nb = std::max(1, std::min<int>(kBranches, (int)rest.size() + (lat.empty() ? 0 : 1)));
  std::vector<size_t> order(rest.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(),
                   [&](size_t x, size_t y) { return rest[x]->nnz_total > rest[y]->nnz_total; });
  std::vector<int> branch(rest.size(), 0);
  std::vector<double> load(nb, 0.0);
  load[0] = lat_work;
  for (size_t i : order) {
    const int k = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    branch[i] = k;
    load[k] += (double)rest[i]->nnz_total + 1.0;
  }
  auto stream_of = [&](int k) { return k == 0 ? st : b->side[k - 1]; };
  if (hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) != hipSuccess)
    return fail(GDX_ERR_HIP, "hipStreamBeginCapture failed");
  int rc = GDX_OK;
  if (hipEventRecord(b->ev[0], st) != hipSuccess) rc = GDX_ERR_HIP;
  for (int k = 1; k < nb && !rc; ++k)
    if (hipStreamWaitEvent(stream_of(k), b->ev[0], 0) != hipSuccess) rc = GDX_ERR_HIP;
  if (!rc && b->coef) rc = gdx::coef_batch_launch(b->coef, st);
  for (size_t i = 0; i < points.size() && !rc; ++i) rc = gdx::launch_rhs(points[i], st);
  if (!rc && b->lattice) rc = gdx::lattice_batch_launch(b->lattice, st);
  for (size_t i = 0; i < rest.size() && !rc; ++i) rc = gdx::numeric_launches(rest[i], stream_of(branch[i]));
  // join every side branch that was forked, also after a failed launch, so the capture can end
  for (int k = 1; k < nb; ++k)
    if (hipEventRecord(b->ev[k], stream_of(k)) != hipSuccess || hipStreamWaitEvent(st, b->ev[k], 0) != hipSuccess)
      rc = rc ? rc : GDX_ERR_HIP;
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(st, &g);
  if (rc || e != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    drop_graph(b);
    return fail(rc ? rc : GDX_ERR_HIP, "graph capture failed");
  }
  b->graph = g;
  if (hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0) != hipSuccess) {
    drop_graph(b);
    return fail(GDX_ERR_HIP, "hipGraphInstantiate failed");
  }
  return GDX_OK;
}

int gdx_batch_launch(gdx_batch *b) {
  if (!b) return fail(GDX_ERR_ARG, "NULL argument");
  if (!b->ctx) return fail(GDX_ERR_STATE, "the batch's context was finalized");
  if (!b->exec) return fail(GDX_ERR_STATE, "gdx_batch_capture has not run since the batch changed");
  if (hipSetDevice(b->ctx->device) != hipSuccess) return fail(GDX_ERR_HIP, "hipSetDevice failed");
  return hipGraphLaunch(b->exec, b->ctx->stream) == hipSuccess ? GDX_OK : fail(GDX_ERR_HIP, "hipGraphLaunch failed");
}

int gdx_batch_destroy(gdx_batch *b) {
  if (!b) return fail(GDX_ERR_ARG, "NULL argument");
  if (gdx_ctx *ctx = b->ctx) {
    gdx::release_batch_device(b);
    gdx::unregister(ctx->batches, b);
  }
  delete b;
  return GDX_OK;
}

}  // extern "C"

namespace gdx {
void release_batch_device(gdx_batch *b) {
  if (!b->ctx) return;
  (void)hipSetDevice(b->ctx->device);
  (void)hipStreamSynchronize(b->ctx->stream);
  drop_graph(b);
  free_branches(b);
  b->probs.clear();
  b->ctx = nullptr;
}
void batch_invalidate_problem(gdx_ctx *ctx, gdx_problem *p) {
  for (gdx_batch *b : ctx->batches)
    if (std::find(b->probs.begin(), b->probs.end(), p) != b->probs.end()) drop_graph(b);
}
void batch_forget_problem(gdx_ctx *ctx, gdx_problem *p) {
  for (gdx_batch *b : ctx->batches)
    for (size_t i = 0; i < b->probs.size(); ++i)
      if (b->probs[i] == p) {
        drop_graph(b);
        b->probs.erase(b->probs.begin() + i);
        break;
      }
}
}  // namespace gdx
