// Skeleton drivers: allocate the temporaries a skeleton needs, marshal its
// arguments, pick the launch shape and enqueue the kernel(s).
//
// These are the roles of executeOp / foldCore / foldSegOp / scanCore /
// permuteOp / stencilOp in CUDA/Execute.hs:264-450, of the argument
// marshalling at :823-909,930-982 and of the launch arithmetic in
// CUDA/Analysis/Launch.hs:42-172 -- re-derived for 64-lane wavefronts, 256
// compute units and single-pass kernels (one launch where the reference needs
// two or three).
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "skeleton.hpp"

using acc::fail;

namespace {

// Kernel arguments in launch order.  Every argument of these kernels is at
// most 8 bytes, so each gets one 8-byte slot whose address is handed to HIP.
// What the driver that is running on this thread launches for: the instance's entry name (for the launch trace) and,
// for an instance built with ACC_FLAG_GUARDED, the address of the guard word that every one of its kernels takes as
// its last parameter (0: no loop).
struct Running {
  const char *entry = "";
  bool dump_exec = false;     // the context was created under ACC_HIP_DEBUG=dump-exec
  bool guarded = false;
  uint64_t guard = 0;
};
thread_local Running t_run;

class Args {
 public:
  void i64(int64_t v) { push(&v, sizeof(v)); }
  void u32(uint32_t v) { push(&v, sizeof(v)); }
  void i32(int32_t v) { push(&v, sizeof(v)); }
  void ptr(uint64_t v) { push(&v, sizeof(v)); }
  size_t count() const { return count_; }
  // the arguments as HIP wants them, the guard's address appended for a guarded instance
  void **data()
  {
    if (t_run.guarded && !guard_pushed_) {
      ptr(t_run.guard);
      guard_pushed_ = true;
    }
    return data_without_guard();
  }
  // (for a launch whose last arguments are not 8-byte slots: the caller appends them, then the guard)
  void **data_without_guard()
  {
    uint64_t *slot = count_ <= FEW ? few_ : many_.data();
    void **ptr = few_ptrs_;
    if (count_ > FEW) {
      many_ptrs_.resize(count_);
      ptr = many_ptrs_.data();
    }
    for (size_t k = 0; k < count_; ++k) ptr[k] = slot + k;
    return ptr;
  }

 private:
  void push(const void *p, size_t n)
  {
    uint64_t s = 0;
    std::memcpy(&s, p, n);
    if (count_ < FEW) {
      few_[count_++] = s;
      return;
    }
    if (count_ == FEW) many_.assign(few_, few_ + FEW);
    many_.push_back(s);
    ++count_;
  }
  // (in place as far as any but the longest lists go: a call's host side is a few microseconds, and as long as a small
  // array's whole call)
  static constexpr size_t FEW = 40;
  size_t count_ = 0;
  uint64_t few_[FEW];
  void *few_ptrs_[FEW];
  std::vector<uint64_t> many_;
  std::vector<void *> many_ptrs_;
  bool guard_pushed_ = false;
};

// Every kernel launch of the drivers.  ACC_HIP_DEBUG=dump-exec prints one line per launch -- entry<<<grid, block,
// lds>>> and the time on the device -- as the reference's -ddump-exec does (Debug.hs:41-76, hooked at
// Execute.hs:975-982); timing a launch means waiting for it, so the trace serialises the stream.
// acc_trace_start .. acc_trace_stop on a thread: an event before and one behind every launch it makes
struct Trace {
  bool on = false;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> spans;
};
thread_local Trace t_trace;

hipError_t launch_kernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned lds,
                         hipStream_t st, void **args, void **extra)
{
  if (t_trace.on) {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    const bool timed = hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess && hipEventRecord(e0, st) == hipSuccess;
    const hipError_t rc = hipModuleLaunchKernel(f, gx, gy, gz, bx, by, bz, lds, st, args, extra);
    if (timed && rc == hipSuccess && hipEventRecord(e1, st) == hipSuccess) {
      t_trace.spans.emplace_back(e0, e1);
    } else {
      if (e0) (void)hipEventDestroy(e0);
      if (e1) (void)hipEventDestroy(e1);
    }
    return rc;
  }
  if (!t_run.dump_exec) return hipModuleLaunchKernel(f, gx, gy, gz, bx, by, bz, lds, st, args, extra);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  const bool timed = hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess && hipEventRecord(e0, st) == hipSuccess;
  const hipError_t rc = hipModuleLaunchKernel(f, gx, gy, gz, bx, by, bz, lds, st, args, extra);
  float ms = -1.0f;
  if (timed && rc == hipSuccess && hipEventRecord(e1, st) == hipSuccess && hipEventSynchronize(e1) == hipSuccess)
    (void)hipEventElapsedTime(&ms, e0, e1);
  const char *name = hipKernelNameRef(f);
  std::fprintf(stderr, "[acc-hip exec] %s: %s<<<%u, %u, %u>>> gpu: %.3f ms%s\n", t_run.entry, name ? name : "?", gx, bx, lds, ms,
               rc == hipSuccess ? "" : " FAILED");
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipGetLastError();
  return rc;
}

int64_t array_size(const acc_array &a)
{
  int64_t n = 1;
  for (int d = 0; d < a.rank; ++d) n *= a.shape[d];
  return n;
}

bool aligned16(uint64_t p) { return (p & 15u) == 0; }

// free array variables first, in Gamma order; per array the extents outermost
// first, then the component pointers highest component first
// (CodeGen/Base.hs:344-357, Execute.hs:835-836,946-951)
int push_env(const acc_skel_s *s, const acc_array *env, Args *args, bool *aligned)
{
  const std::vector<acc::EnvSig> &sig = s->spec.env;
  if (!sig.empty() && !env) return fail(ACC_ERR_INVALID, "%s: env arrays missing", s->entry.c_str());
  for (size_t k = 0; k < sig.size(); ++k) {
    const acc_array &a = env[k];
    if (a.rank != sig[k].rank || a.ncomp != sig[k].ncomp)
      return fail(ACC_ERR_INVALID, "%s: env array %zu has rank %d / %d components, the kernel was built for %d / %d",
                  s->entry.c_str(), k, a.rank, a.ncomp, sig[k].rank, sig[k].ncomp);
    int64_t n = 1;
    for (int d = 0; d < a.rank; ++d) {
      if (a.shape[d] < 0) return fail(ACC_ERR_INVALID, "%s: env array %zu has a negative extent", s->entry.c_str(), k);
      n *= a.shape[d];
      args->i64(a.shape[d]);
    }
    for (int c = a.ncomp - 1; c >= 0; --c) {
      if (!a.ptr[c] && n > 0) return fail(ACC_ERR_INVALID, "%s: env array %zu component %d is NULL", s->entry.c_str(), k, c);
      if (!aligned16(a.ptr[c])) *aligned = false;
      args->ptr(a.ptr[c]);
    }
  }
  return ACC_OK;
}

int check_out(const acc_skel_s *s, const acc_array *out, int rank, const char *what, int ncomp)
{
  if (!out) return fail(ACC_ERR_INVALID, "%s: %s array missing", s->entry.c_str(), what);
  if (out->rank != rank) return fail(ACC_ERR_INVALID, "%s: %s array has rank %d, expected %d", s->entry.c_str(), what, out->rank, rank);
  if (out->ncomp != ncomp)
    return fail(ncomp == 1 ? ACC_ERR_UNSUPPORTED : ACC_ERR_INVALID, "%s: %s array has %d components, the kernel was built for %d",
                s->entry.c_str(), what, out->ncomp, ncomp);
  for (int d = 0; d < rank; ++d)
    if (out->shape[d] < 0) return fail(ACC_ERR_INVALID, "%s: %s array has a negative extent", s->entry.c_str(), what);
  for (int c = 0; c < ncomp; ++c)
    if (!out->ptr[c] && array_size(*out) > 0) return fail(ACC_ERR_INVALID, "%s: %s array is NULL", s->entry.c_str(), what);
  return ACC_OK;
}

// an array of the skeleton's element type: one component, or the tuple's
int check_out(const acc_skel_s *s, const acc_array *out, int rank, const char *what) { return check_out(s, out, rank, what, s->ncomp()); }

// the component pointers of a result array, highest component first; NULL array = that many null pointers
void push_ptrs(const acc_array *a, int ncomp, Args *args, bool *aligned)
{
  for (int c = ncomp - 1; c >= 0; --c) {
    const uint64_t p = a ? a->ptr[c] : 0;
    if (a && !aligned16(p)) *aligned = false;
    args->ptr(p);
  }
}

void push_out(const acc_array &out, Args *args, bool *aligned)
{
  for (int d = 0; d < out.rank; ++d) args->i64(out.shape[d]);
  push_ptrs(&out, out.ncomp, args, aligned);
}

// whether a result shares memory with one of the free array variables
bool out_in_env(const acc_skel_s *s, const acc_array *env, const acc_array &out)
{
  const std::vector<acc::EnvSig> &sig = s->spec.env;
  const uint64_t n_out = static_cast<uint64_t>(array_size(out));
  for (size_t k = 0; k < sig.size(); ++k) {
    const uint64_t n = static_cast<uint64_t>(array_size(env[k]));
    for (int c = 0; c < env[k].ncomp; ++c)
      for (int o = 0; o < out.ncomp; ++o) {
        const uint64_t bytes = n * (uint64_t)acc::type_size(sig[k].type[c]);
        const uint64_t bytes_out = n_out * (s->spec.comp_types.empty() ? s->spec.elt_size : acc::type_size(s->spec.comp_types[out.ncomp - 1 - o]));
        if (env[k].ptr[c] < out.ptr[o] + bytes_out && out.ptr[o] < env[k].ptr[c] + bytes) return true;
      }
  }
  return false;
}

int launch(acc_skel_s *s, int variant, int64_t grid, size_t dyn_lds, hipStream_t stream, Args *args)
{
  if (grid < 1 || grid > 0x7fffffffLL) return fail(ACC_ERR_INVALID, "%s: grid of %lld blocks", s->entry.c_str(), (long long)grid);
  ACC_TRY(s->ensure_variant(variant));
  ACC_TRY(s->ctx->make_current());
  ACC_HIP_TRY(launch_kernel(s->variants[variant].fn, static_cast<unsigned>(grid), 1, 1,
                                    static_cast<unsigned>(s->variants[variant].block), 1, 1, static_cast<unsigned>(dyn_lds), stream,
                                    args->data(), nullptr));
  return ACC_OK;
}

// For the length of one driver call: what Args::data() and launch_kernel read (see Running).  A stream under a guard
// only takes instances whose kernels look at it.
struct RunScope {
  Running saved;
  int rc = ACC_OK;
  RunScope(acc_skel_s *s, hipStream_t st) : saved(t_run)
  {
    t_run.entry = s->entry.c_str();
    t_run.dump_exec = s->ctx->dump_exec;
    t_run.guarded = s->spec.guarded;
    t_run.guard = 0;
    const uint64_t g = s->ctx->guard_of(st);
    if (g && !s->spec.guarded)
      rc = fail(ACC_ERR_INVALID, "%s: the stream is under a guard (acc_stream_set_guard) and this instance was created without ACC_FLAG_GUARDED",
                s->entry.c_str());
    else
      t_run.guard = g;
  }
  ~RunScope() { t_run = saved; }
  RunScope(const RunScope &) = delete;
  RunScope &operator=(const RunScope &) = delete;
};
#define ACC_RUN_SCOPE(s, st)                          \
  RunScope run_scope__((s), (st));                    \
  if (run_scope__.rc != ACC_OK) return run_scope__.rc

bool kind_is(const acc_skel_s *s, std::initializer_list<int> kinds)
{
  return std::find(kinds.begin(), kinds.end(), s->spec.kind) != kinds.end();
}

size_t round256(size_t n) { return (n + 255) & ~size_t(255); }

// resident-grid cap: compute units x workgroups per unit (Launch.hs:51-55)
int64_t resident(const acc_skel_s *s, int variant) { return (int64_t)s->ctx->props.multiProcessorCount * s->variants[variant].blocks_per_cu; }

}  // namespace

extern "C" {

int acc_trace_start(acc_context ctx)
{
  if (!ctx) return fail(ACC_ERR_INVALID, "acc_trace_start: NULL context");
  if (t_trace.on) return fail(ACC_ERR_INVALID, "acc_trace_start: this thread is tracing already");
  t_trace.on = true;
  return ACC_OK;
}

int acc_trace_stop(acc_context ctx, int32_t *launches, double *gpu_ms)
{
  if (!ctx) return fail(ACC_ERR_INVALID, "acc_trace_stop: NULL context");
  if (!t_trace.on) return fail(ACC_ERR_INVALID, "acc_trace_stop: this thread is not tracing");
  t_trace.on = false;
  int rc = ctx->make_current();
  double total = 0.0;
  int32_t count = 0;
  for (auto &span : t_trace.spans) {
    float ms = 0.0f;
    if (rc == ACC_OK) {
      hipError_t e = hipEventSynchronize(span.second);
      if (e == hipSuccess) e = hipEventElapsedTime(&ms, span.first, span.second);
      if (e != hipSuccess) rc = acc::fail_hip(e, "acc_trace_stop");
    }
    total += ms;
    ++count;
    (void)hipEventDestroy(span.first);
    (void)hipEventDestroy(span.second);
  }
  t_trace.spans.clear();
  if (launches) *launches = count;
  if (gpu_ms) *gpu_ms = total;
  return rc;
}

int acc_exec_map(acc_skel s, const acc_array *env, const acc_array *out, acc_stream stream)
{
  if (!s) return fail(ACC_ERR_INVALID, "acc_exec_map: NULL skeleton");
  ACC_RUN_SCOPE(s, static_cast<hipStream_t>(stream));
  if (!kind_is(s, {ACC_SKEL_MAP, ACC_SKEL_GENERATE, ACC_SKEL_TRANSFORM})) return fail(ACC_ERR_INVALID, "acc_exec_map: skeleton is '%s'", s->entry.c_str());
  ACC_TRY(check_out(s, out, s->spec.out_rank, "result"));
  Args args;
  bool aligned = true;
  ACC_TRY(push_env(s, env, &args, &aligned));
  push_out(*out, &args, &aligned);
  const int64_t n = array_size(*out);
  if (n == 0) return ACC_OK;
  int v = aligned ? 0 : 1;
  // A result of a few columns or rows leaves most of every tile outside it (a transpose of 2^23 x 2 either way:
  // 170 us in tiles, 23-34 in runs): such a call takes variants 2 and 3, the same map in runs.  (A result of 2^20 rows
  // of 8 / 16 / 24 / 32 columns: 45 / 56 / 100 / 44 us in tiles, 10 / 20 / 40 / 41 in runs, and 29 against 52 for 33
  // columns.  Of 6 / 8 / 12 / 16 rows of 2^20 columns: 41 / 41 / 43 / 43 in tiles, 17 / 31 / 82 / 151 in runs.)
  const bool in_tiles = s->spec.map_tiled && out->shape[s->spec.out_rank - 1] >= s->knobs.map_tiled_min_w &&
                        out->shape[s->spec.out_rank - 1 - s->spec.map_tile_dim] >= s->knobs.map_tiled_min_h;
  if (s->spec.map_tiled && !in_tiles) v += 2;
  ACC_TRY(s->ensure_variant(v));
  if (in_tiles) {
    // a wave per tile of 32 x 32 elements of the innermost dimension and the second innermost one, or the one that
    // ACC_FLAG_TILE_DIM names, as skel_map.h arranges them in a workgroup
    const int rank = s->spec.out_rank;
    const int64_t side = 8 * (int64_t)s->spec.map_tile_block, esz = std::max(1, s->spec.elt_size);
    const int64_t w = out->shape[rank - 1], h = out->shape[rank - 1 - s->spec.map_tile_dim];
    const int64_t waves = s->variants[v].block / 64;
    bool whole = (w * esz) % 128 == 0;
    for (int c = 0; c < out->ncomp; ++c) whole = whole && out->ptr[c] % 128 == 0;
    // A result in place of an operand takes the form for whole lines whatever its rows are, the one that evaluates every
    // element once: in the others workgroups evaluate their neighbours' columns too, and lanes beyond the result its last row or
    // column, which by then may hold what has been written -- no index any more, for instance.  (It is the slower one where
    // rows are no whole lines: a matrix plus another one transposed, in place, us as pieces or lines / so: 1001 x 999 Float32
    // 4.6 / 6.3, 12000 x 501 16.2 / 16.9, 5003 x 3001 32.3 / 37.1, 8191^2 161.9 / 161.1, 7001 x 2500 Float64 71 / 91.)
    whole = whole || out_in_env(s, env, *out);
    const bool strips = whole && n == w * h && n * esz >= acc::map_strips_from;
    // Results of no whole lines, or that begin amid one, go out in lines from 28 MB on, about what the L2s hold together (us as
    // they stand / in lines, operands that the memory-side cache does not hold: 5003 x 3001 Float32 33.3 / 28.8, 8191^2 148 / 104,
    // 3891 x 2048 17.9 / 15.8, 7001 x 2500 Float64 77 / 60, with another operand read along the rows 3001 x 2999 29.4 / 27.6, 5003 x
    // 3001 47 / 43; but 1001 x 999 4.6 / 5.6, 1500 x 1501 with another operand 8.5 / 10.3, thirty planes of 400 x 501 14.8 / 16.5).
    // Lines have a third of the elements (of 8 bytes a seventh) evaluated twice, which is in the way where they take more than
    // the memory does.  How much that is is told by the size of the kernel, straight through as it is: up to 16 KB of code, 40
    // of 8-byte elements.  5003 x 3001 transposed, code of the lines / as it stands / in lines, Float32: e^x 7.7 KB 33.2 / 30.0, a
    // polynomial of degree 24 14.5 KB 33.8 / 31.6, of 32 17.6 KB 34.1 / 36.1, of 64 29.9 KB 45.1 / 56.3, x^1.7 31.0 KB 50.9 / 68.0;
    // Float64: degree 32 23.0 KB 67.1 / 58.9, sin 36.3 KB 102 / 92, x^1.7 46.9 KB 95 / 105, degree 64 60.8 KB 94 / 111; Int32: degree 32 13.6 KB 33.8 / 32.7,
    // 64 21.9 KB 37.9 / 48.8.  (On the wrong side are tanh of Float32, short branches, 11.6 KB 48.5 / 52.5, and a Float64 polynomial of degree 48, 34.9 KB 68.5 / 76.8.)
    const bool in_lines = s->spec.map_lines && !whole && n * esz >= s->knobs.map_lines_from_mb * ((int64_t)1 << 20) &&
                          !s->spec.map_loops && s->variants[v].lines_code <= (esz == 8 ? 40 : 16) * (size_t)1024;
    const int64_t down = h <= side || in_lines ? 1 : (strips ? waves : (waves % 2 == 0 && !whole ? 2 : 1));
    const int64_t columns = waves / down * side - (in_lines ? 128 / esz : 0);
    const int64_t groups = ((w + columns - 1) / columns) * ((h + down * side - 1) / (down * side)) * (n / (w * h));
    const int64_t grid = std::min<int64_t>(groups, (int64_t)1 << 22);
    if (whole) return launch(s, v, grid, 0, static_cast<hipStream_t>(stream), &args);
    ACC_TRY(s->ctx->make_current());
    ACC_HIP_TRY(launch_kernel(in_lines ? s->variants[v].fn_lines : s->variants[v].fn_pieces, static_cast<unsigned>(grid), 1, 1,
                              static_cast<unsigned>(s->variants[v].block), 1, 1, 0, static_cast<hipStream_t>(stream), args.data(), nullptr));
    return ACC_OK;
  }
  // streaming with no reuse: one short-lived workgroup per tile keeps the most loads in flight
  const int64_t grid = acc_launch_grid(n, s->elements_per_block(), resident(s, v), s->knobs.map_oversub);
  return launch(s, v, grid, 0, static_cast<hipStream_t>(stream), &args);
}

namespace {

// The segmented fold over `nseg` segments holding `n` elements in all; `args` holds the kernel parameters up to and
// including the segment description (offsets, or rows and row length).
//   short segments: a lane per segment over chunks staged in LDS (skel_foldseg.h);
//   long ones (on average: the lengths themselves are on the device) would serialise on that lane, so a wave, or
//   from `foldseg.block_team_len` a workgroup, takes one segment at a time;
//   fewer long segments than the device has room for teams: every segment is cut into `split` pieces, a team
//   each, and a second launch joins the pieces in order.
// Very long segments among the others (skel_foldseg.h, ACC_GIANTS).  Variants 4 to 7 of a segmented fold hand such a
// segment over to a second launch, at a cost to sources that have none; so an instance takes them once a look at its
// segment lengths has found such a segment -- a small kernel behind calls number 1, 2, 4, 8 ... of the instance, which
// says so in a word of host memory -- and once they are compiled, which happens in the background meanwhile.
// `foldseg.giants`: 2 this, 1 always, 0 never.
struct GiantsPlan {
  bool hand_over = false;      // this call takes variant `lv + 4`
  bool look = false;           // this call is followed by the look at the segment lengths
};

int plan_giants(acc_skel_s *s, int lv, GiantsPlan *plan)
{
  plan->hand_over = s->knobs.foldseg_giants == 1;
  if (s->knobs.foldseg_giants != 2 || s->hint_slot < 0) return ACC_OK;
  // (the word is the device's to write, at any time: read as such)
  if (!s->met_giants.load(std::memory_order_relaxed) &&
      __atomic_load_n(const_cast<uint32_t *>(s->ctx->status_host) + acc::STATUS_WORDS + s->hint_slot, __ATOMIC_RELAXED) != 0)
    s->met_giants.store(true, std::memory_order_relaxed);
  if (s->met_giants.load(std::memory_order_relaxed)) {
    ACC_TRY(s->start_variant(lv + 4));
    plan->hand_over = s->variant_compiled(lv + 4);
  } else {
    const unsigned call = s->seg_calls.fetch_add(1, std::memory_order_relaxed) + 1;
    plan->look = (call & (call - 1)) == 0;
  }
  return ACC_OK;
}

// the look: the parameters of the fold's own kernel (`common`, a guard's address behind them) and the word's address
int launch_probe(acc_skel_s *s, int lv, Args *common, int64_t nseg, hipStream_t st)
{
  (void)common->data();
  common->ptr(s->ctx->status_dev + (uint64_t)(acc::STATUS_WORDS + s->hint_slot) * sizeof(uint32_t));
  const int64_t lookers = std::min<int64_t>((nseg + s->spec.block - 1) / s->spec.block, (int64_t)s->ctx->props.multiProcessorCount * 8);
  hipError_t e = launch_kernel(s->variants[lv].fn_sweep, static_cast<unsigned>(lookers), 1, 1, static_cast<unsigned>(s->spec.block), 1, 1, 0, st,
                               common->data_without_guard(), nullptr);
  return e == hipSuccess ? ACC_OK : acc::fail_hip(e, "hipModuleLaunchKernel(segmented fold, probe)");
}

// the table of jobs: head, 32 jobs of 8 words and 16 ticket counters 32 words apart, then values of tagged words -- two
// for every piece of 4 chunks the source has, and one a job
int acquire_jobs(acc_skel_s *s, int lv, int64_t n, hipStream_t st, acc::ScratchRef *jobs)
{
  const int64_t piece = (int64_t)std::max(1, s->knobs.foldseg_giant_chunks) * (int64_t)((lv & 2) ? s->spec.chunk_long : s->spec.chunk);
  const size_t words_a_value = ((size_t)s->spec.elt_size + 3) / 4;
  const size_t bytes = (8 + 32 * (8 + 16 * 32) + (2 * (size_t)(n / piece + 2) + 32) * words_a_value) * 8;
  return s->ctx->scratch_acquire(bytes, st, acc::SCRATCH_FLAGS, jobs);
}

// the second launch, which takes what the first has entered in the table: `common` with the table behind it
int launch_sweep(acc_skel_s *s, int lv, Args *common, const acc::ScratchRef &jobs, hipStream_t st)
{
  common->ptr(reinterpret_cast<uint64_t>(jobs.ptr));
  common->u32(jobs.epoch);
  common->ptr(s->ctx->status_dev);
  const int64_t sweepers = (int64_t)s->ctx->props.multiProcessorCount * std::max(1, std::min(s->knobs.foldseg_sweep_per_cu, 2048 / s->spec.block));
  hipError_t e = launch_kernel(s->variants[lv].fn_sweep, static_cast<unsigned>(sweepers), 1, 1, static_cast<unsigned>(s->spec.block), 1, 1, 0, st,
                               common->data(), nullptr);
  return e == hipSuccess ? ACC_OK : acc::fail_hip(e, "hipModuleLaunchKernel(segmented fold, sweep)");
}

// Segments a workgroup: one for each of its lanes, or a half, a quarter, an eighth of them, the least that leaves it more
// than 1024 elements.  A workgroup goes through its chunks one after the other, a round trip or, of a gather, two each, and
// more of them run side by side (us with a lane each / so: rows of 64, 1000 of them 15.4 / 4.4, 67352 of 83 24.6 / 7.9,
// 8000 of 100 29.9 / 7.7; sparse matrices of 1000 rows of 64 21.0 / 5.1, 18251 of 95 33 / 13).  Once there are more than
// eight for a compute unit, which is what it holds, every chunk counts whether it is full or not.  Then no more of them in
// all than a lane a segment would make, or, where every workgroup has a single one, of no gathers, and so nothing to wait
// for in between, a third more: 359769 rows of 20 take 8.2 us in two chunks a workgroup of 128, in one of 64, half full, 10.6,
// and 9.3 in two of 256; 765249 of 10, one chunk either way, 9.0 in workgroups of 256 and 11.8 of 128; 300000 of 50 18.0 in
// five chunks of 256, 18.9 in two of 64 (rows of a matrix 13.6 / 15.5); but 200000 of 70 21.0 in six and 14.6 in one of 32,
// 524287 of 40 21.4 in four and 17.3 in one of 64.  (Sparse matrices: 250000 rows of 33 43.6 in three of 256, 46.6 in one of
// 64; 262143 of 64 84 in three of 128, 92 in one of 32.)  And no more workgroups than 32 for a compute unit, 20 where
// elements are gathered: 10^6 rows of 30, 61 of them, 27.3 and 25.9 in 256, the sparse matrix of 524287 rows of 40, 32 of
// them, 109.3 and 102.7 in 128.
int64_t segments_a_workgroup(const acc_skel_s *s, int lv, int64_t nseg, int64_t avg)
{
  const int64_t lanes = s->spec.block, chunk = (lv & 2) ? s->spec.chunk_long : s->spec.chunk;
  const int64_t spread = s->knobs.foldseg_spread * s->ctx->props.multiProcessorCount;
  const bool streams = s->spec.get_streams;
  auto chunks = [&](int64_t own) { return (own * avg + chunk - 1) / chunk; };
  for (int64_t own = lanes / 8; own < lanes; own *= 2) {
    if (2 * own * avg <= s->knobs.foldseg_spread_min || 4 * nseg > (streams ? 8 : 5) * own * spread) continue;
    const int64_t in_all = chunks(own) * (lanes / own);
    if (2 * nseg <= own * spread || 100 * in_all <= (streams && chunks(own) == 1 ? 134 : 115) * chunks(lanes)) return own;
  }
  return lanes;
}

// `args`: the parameters every kernel of the template begins with (free arrays, result, segments).  `giants`: the
// segments are a vector's (the kernels of rows and of arrays of rank > 1 know no table).
int launch_segmented(acc_skel_s *s, int v, Args *args, const acc_array *env, const acc_array *out, int64_t nseg, int64_t n,
                     hipStream_t st, bool giants = false)
{
  const int64_t avg = n / nseg;
  if (avg < s->knobs.foldseg_wave_team_len) {
    // Segments of 8 elements or more on average stage half as much again at a time (variants 2 and 3 of the
    // instance, built when first wanted): 2^25 elements in segments of 8 / 32 / 100 on average 36 / 31 / 51 us
    // -> 32 / 27 / 40; shorter segments lose by it (rows of 4: 46 -> 49 us), and so keep the shorter chunk.
    int lv = v;
    if (avg >= s->knobs.foldseg_long_from && s->spec.chunk_long > s->spec.chunk) {
      lv = v + 2;
      ACC_TRY(s->ensure_variant(lv));
    }
    GiantsPlan plan;
    if (giants) ACC_TRY(plan_giants(s, lv, &plan));
    const int64_t own = segments_a_workgroup(s, lv, nseg, avg);
    if (!plan.hand_over) {
      const int64_t grid = acc_launch_grid(nseg, own, resident(s, lv), s->knobs.foldseg_oversub);
      int rc = launch(s, lv, grid, 0, st, args);
      if (rc == ACC_OK && plan.look) rc = launch_probe(s, lv, args, nseg, st);
      return rc;
    }
    lv += 4;
    ACC_TRY(s->ensure_variant(lv));
    const int64_t grid = acc_launch_grid(nseg, own, resident(s, lv), s->knobs.foldseg_oversub);
    acc::ScratchRef jobs;
    ACC_TRY(acquire_jobs(s, lv, n, st, &jobs));
    Args first = *args;
    first.ptr(reinterpret_cast<uint64_t>(jobs.ptr));
    first.u32(jobs.epoch);
    first.ptr(s->ctx->status_dev);
    int rc = launch(s, lv, grid, 0, st, &first);
    if (rc == ACC_OK) rc = launch_sweep(s, lv, args, jobs, st);
    s->ctx->scratch_release(jobs, st);
    return rc;
  }
  // teams: a workgroup (1) from `foldseg.block_team_len`, a row of 16 lanes (2) below `foldseg.row_team_below`, else a wave (0)
  const int block_team = avg >= s->knobs.foldseg_block_team_len ? 1 : (avg < s->knobs.foldseg_row_team_below ? 2 : 0);
  const int64_t cus = s->ctx->props.multiProcessorCount;
  const int64_t team_lanes = block_team == 1 ? s->spec.block : (block_team == 2 ? 16 : 64);
  const int64_t room = cus * (2048 / team_lanes);                    // teams the device holds at once
  const int64_t min_piece = team_lanes * 64;                          // a piece keeps its team busy for a while
  int64_t split = 1;
  if (nseg * 2 <= room) split = std::max<int64_t>(1, std::min<int64_t>({room / nseg, avg / min_piece, s->knobs.foldseg_max_split}));
  // (segments that are all cut into pieces are not looked at, and none is handed over)
  GiantsPlan plan;
  if (giants && split == 1) ACC_TRY(plan_giants(s, v, &plan));
  const int tv = plan.hand_over ? v + 4 : v;
  if (plan.hand_over) ACC_TRY(s->ensure_variant(tv));
  acc::ScratchRef blk, jobs;
  uint64_t part = 0, part_ok = 0;
  if (split > 1) {
    const size_t pieces = (size_t)(nseg * split);
    const size_t ok_off = round256(pieces * s->spec.elt_size);
    ACC_TRY(s->ctx->scratch_acquire(ok_off + pieces * 4, st, acc::SCRATCH_FOLD, &blk));
    part = reinterpret_cast<uint64_t>(blk.ptr);
    part_ok = part + ok_off;
  }
  if (plan.hand_over) {
    const int rj = acquire_jobs(s, tv, n, st, &jobs);
    if (rj != ACC_OK) { s->ctx->scratch_release(blk, st); return rj; }
  }
  Args team = *args;
  team.i32(block_team);
  team.i64(split);
  team.ptr(part);
  team.ptr(part_ok);
  if (plan.hand_over) {
    team.ptr(reinterpret_cast<uint64_t>(jobs.ptr));
    team.u32(jobs.epoch);
    team.ptr(s->ctx->status_dev);
  }
  const int64_t per_block = block_team == 1 ? 1 : s->spec.block / team_lanes;
  const int64_t tgrid = acc_launch_grid(nseg * split, per_block, cus, 2048 / s->spec.block);
  int rc = s->ctx->make_current();
  if (rc == ACC_OK) {
    hipError_t e = launch_kernel(s->variants[tv].fn_finish, static_cast<unsigned>(tgrid), 1, 1,
                                         static_cast<unsigned>(s->spec.block), 1, 1, 0, st, team.data(), nullptr);
    if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(segmented fold, team)");
  }
  if (rc == ACC_OK && split > 1) {
    Args join;
    bool al = true;
    rc = push_env(s, env, &join, &al);
    join.i64(nseg);
    push_ptrs(out, out->ncomp, &join, &al);
    join.i64(split);
    join.ptr(part);
    join.ptr(part_ok);
    if (rc == ACC_OK) {
      const int64_t waves = s->spec.block / 64;
      const int64_t jgrid = (nseg + waves - 1) / waves;          // a wave per segment
      hipError_t e = launch_kernel(s->variants[v].fn_fill, static_cast<unsigned>(jgrid), 1, 1,
                                           static_cast<unsigned>(s->spec.block), 1, 1, 0, st, join.data(), nullptr);
      if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(segmented fold, join)");
    }
  }
  if (rc == ACC_OK && plan.hand_over) rc = launch_sweep(s, tv, args, jobs, st);
  if (rc == ACC_OK && plan.look) rc = launch_probe(s, v, args, nseg, st);
  s->ctx->scratch_release(blk, st);
  if (plan.hand_over) s->ctx->scratch_release(jobs, st);
  return rc;
}

// A fold along the innermost dimension whose element function reads neighbouring addresses where the ROW moves by one
// (ACC_FLAG_TILED: the fold of a transposed matrix, a matrix product written as a fold): neighbouring rows in
// neighbouring lanes (<entry>_across) -- a team of lanes along such a row asks for 64 cache lines with every load (sums
// down the columns of 4096 x 4096 Int32: 0.9 ms).  With fewer rows than the device has lanes the rows are cut into
// pieces of at least `fold.across_min_piece` elements: as many as a workgroup has room for beside one another (`subs`),
// and `split` times that, joined in order by <entry>_join, until there is a workgroup for every compute unit (two, of
// lanes with one row each).  Neither more nor in between: 312 workgroups, 56 units with two of them, take 19.9 us for the
// columns of 20000 x 1000, 256 take 18.3 and 512 18.9.  Below 4096 rows a lane takes several (1000 rows 18.3 us against
// 22.0 with one, 4096 rows 15.3 and 14.6; the product of two 128 x 128 matrices, 16384 rows, 12 and 7: there several
// rows read one element of the left operand each).
int launch_across(acc_skel_s *s, int v, Args *args, const acc_array *env, const acc_array *out, int64_t rows, int64_t inner, hipStream_t st)
{
  const int64_t cus = s->ctx->props.multiProcessorCount, block = s->spec.block;
  const int64_t wide = rows < s->knobs.fold_across_wide_below ? acc::across_rows(s->spec) : 1, lanes = (rows + wide - 1) / wide;
  const int64_t pieces = rows < cus * 2048 ? inner / std::max(1, s->knobs.fold_across_min_piece) : 1;
  // lanes side by side: a wave's worth or, of rows that are not cut, a workgroup's; spread evenly over the workgroups
  const int64_t most = pieces > 1 ? 64 : block, chunks = (lanes + most - 1) / most, chunk = (lanes + chunks - 1) / chunks;
  const int64_t subs = std::max<int64_t>(1, std::min(block / chunk, pieces));
  const int64_t split = std::max<int64_t>(1, std::min<int64_t>({(wide > 1 ? 1 : 2) * cus / chunks, pieces / subs, s->knobs.foldseg_max_split}));
  acc::ScratchRef blk;
  uint64_t part = 0, part_ok = 0;
  if (split > 1) {
    const size_t pieces = (size_t)(rows * split);
    const size_t ok_off = round256(pieces * s->spec.elt_size);
    ACC_TRY(s->ctx->scratch_acquire(ok_off + pieces * 4, st, acc::SCRATCH_FOLD, &blk));
    part = reinterpret_cast<uint64_t>(blk.ptr);
    part_ok = part + ok_off;
  }
  Args first = *args;
  first.i64(split);
  first.ptr(part);
  first.ptr(part_ok);
  first.i32(static_cast<int32_t>(chunk));
  first.i32(static_cast<int32_t>(subs));
  const int64_t grid = std::min<int64_t>(chunks * split, (int64_t)1 << 22);
  int rc = s->ctx->make_current();
  if (rc == ACC_OK) {
    hipError_t e = launch_kernel(wide > 1 ? s->variants[v].fn_across_wide : s->variants[v].fn_across, static_cast<unsigned>(grid), 1, 1, static_cast<unsigned>(s->spec.block), 1, 1, 0, st,
                                 first.data(), nullptr);
    if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(fold, a lane a row)");
  }
  if (rc == ACC_OK && split > 1) {
    Args join;
    bool al = true;
    rc = push_env(s, env, &join, &al);
    join.i64(rows);
    push_ptrs(out, out->ncomp, &join, &al);
    join.i64(split);
    join.ptr(part);
    join.ptr(part_ok);
    if (rc == ACC_OK) {
      const int64_t waves = s->spec.block / 64;
      hipError_t e = launch_kernel(s->variants[v].fn_fill, static_cast<unsigned>((rows + waves - 1) / waves), 1, 1,
                                   static_cast<unsigned>(s->spec.block), 1, 1, 0, st, join.data(), nullptr);
      if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(fold, join)");
    }
  }
  s->ctx->scratch_release(blk, st);
  return rc;
}

}  // namespace

int acc_exec_fold(acc_skel s, const acc_array *env, int32_t in_rank, const int64_t *in_shape, const acc_array *out, acc_stream stream)
{
  if (!s) return fail(ACC_ERR_INVALID, "acc_exec_fold: NULL skeleton");
  ACC_RUN_SCOPE(s, static_cast<hipStream_t>(stream));
  if (!kind_is(s, {ACC_SKEL_FOLD, ACC_SKEL_FOLD1})) return fail(ACC_ERR_INVALID, "acc_exec_fold: skeleton is '%s'", s->entry.c_str());
  if (in_rank != s->spec.out_rank + 1 || !in_shape) return fail(ACC_ERR_INVALID, "%s: input rank %d, kernel was built for %d", s->entry.c_str(), in_rank, s->spec.out_rank + 1);
  ACC_TRY(check_out(s, out, s->spec.out_rank, "result"));
  for (int d = 0; d < in_rank; ++d)
    if (in_shape[d] < 0) return fail(ACC_ERR_INVALID, "%s: negative input extent", s->entry.c_str());
  int64_t inner = in_shape[in_rank - 1];
  // fold1 of an empty innermost dimension: Execute.hs:282-285
  if (inner == 0 && !s->spec.has_seed) return fail(ACC_ERR_INVALID, "%s: empty array", s->entry.c_str());
  // empty outer extents count as 1 in the result of a seeded fold: Execute.hs:287-289.  (The reference then runs its
  // kernel over rows that do not exist; here such a result is the seed in every position, as for rows without
  // elements, and a fold1 over no rows has nothing to do.)
  int64_t rows = 1;
  bool no_rows = false;
  for (int d = 0; d + 1 < in_rank; ++d) {
    rows *= std::max<int64_t>(1, in_shape[d]);
    no_rows = no_rows || in_shape[d] == 0;
  }
  if (no_rows) {
    if (!s->spec.has_seed) return ACC_OK;
    inner = 0;
  }
  if (array_size(*out) < rows && !(in_rank == 1)) return fail(ACC_ERR_INVALID, "%s: result holds %lld elements, %lld needed", s->entry.c_str(), (long long)array_size(*out), (long long)rows);

  hipStream_t st = static_cast<hipStream_t>(stream);
  Args args;
  bool aligned = true;
  ACC_TRY(push_env(s, env, &args, &aligned));
  const int v = aligned ? 0 : 1;
  ACC_TRY(s->ensure_variant(v));

  if (s->spec.out_rank > 0) {      // along the innermost dimension: a segmented fold over rows of one length
    args.i64(rows);
    push_ptrs(out, out->ncomp, &args, &aligned);
    args.i64(rows);
    args.i64(inner);
    if (inner == 0) {
      // rows without elements: every result is the seed; the one-lane-per-row entry does that
      const int64_t grid = acc_launch_grid(rows, s->spec.block, resident(s, v), 1 << 20);
      return launch(s, v, grid, 0, st, &args);
    }
    if (inner <= std::min(16, s->knobs.fold_rows_max)) {
      // short rows: a lane reads its row straight from memory (skel_foldseg.h, _rows)
      const int64_t r = inner == 1 ? 4 : (inner == 2 ? 2 : 1), u = r * inner >= 16 ? 1 : 16 / (r * inner);   // as the kernel's R and U
      const int64_t grid = acc_launch_grid(rows, s->spec.block * r * u, resident(s, v), s->knobs.foldseg_oversub);
      hipError_t e = launch_kernel(s->variants[v].fn_rows, static_cast<unsigned>(grid), 1, 1, static_cast<unsigned>(s->spec.block), 1, 1,
                                           0, st, args.data(), nullptr);
      return e == hipSuccess ? ACC_OK : acc::fail_hip(e, "hipModuleLaunchKernel(fold, short rows)");
    }
    if (s->spec.fold_across)
      return launch_across(s, v, &args, env, out, rows, inner, st);
    return launch_segmented(s, v, &args, env, out, rows, rows * inner, st);
  }

  const int64_t n = inner;
  const int64_t tile = s->elements_per_block();
  int64_t grid = acc_launch_grid(n, tile, s->ctx->props.multiProcessorCount,
                                 std::min(s->variants[v].blocks_per_cu, s->knobs.fold_blocks_per_cu));
  const bool single = s->spec.fold_single;       // as generated into the kernel
  if (grid == 1) {                 // a lone block finishes the job itself
    push_ptrs(out, out->ncomp, &args, &aligned);
    args.i64(n);
    args.ptr(0);
    if (single) { args.u32(0); args.ptr(s->ctx->status_dev); }
    return launch(s, v, 1, 0, st, &args);
  }
  if (single) {
    // one launch: every block leaves its partial result in 64-bit words that carry the launch's epoch in their
    // upper half, and the last block collects them (skel_fold.h).  Every word of the scratch block is only ever
    // written in that form, so words of earlier launches, whatever their grid or element type, read as "not yet".
    const size_t words = (s->spec.elt_size + 3) / 4;
    acc::ScratchRef blk;
    ACC_TRY(s->ctx->scratch_acquire((size_t)grid * words * 8, st, acc::SCRATCH_FLAGS, &blk));
    push_ptrs(out, out->ncomp, &args, &aligned);
    args.i64(n);
    args.ptr(reinterpret_cast<uint64_t>(blk.ptr));
    args.u32(blk.epoch);
    args.ptr(s->ctx->status_dev);
    int rc = launch(s, v, grid, 0, st, &args);
    s->ctx->scratch_release(blk, st);
    return rc;
  }
  // one partial per block, then a single-block launch folds them: foldRec, Execute.hs:304-315,
  // always exactly one level deep because the first grid never exceeds what is resident
  acc::ScratchRef blk;
  ACC_TRY(s->ctx->scratch_acquire((size_t)grid * s->spec.elt_size, st, acc::SCRATCH_FOLD, &blk));
  const uint64_t partials = reinterpret_cast<uint64_t>(blk.ptr);
  push_ptrs(out, out->ncomp, &args, &aligned);
  args.i64(n);
  args.ptr(partials);
  int rc = launch(s, v, grid, 0, st, &args);
  if (rc == ACC_OK) {
    Args fin;
    bool al = true;
    rc = push_env(s, env, &fin, &al);
    push_ptrs(out, out->ncomp, &fin, &al);
    fin.ptr(partials);
    fin.i64(grid);
    if (rc == ACC_OK) {
      hipError_t e = launch_kernel(s->variants[v].fn_finish, 1, 1, 1, static_cast<unsigned>(s->spec.block), 1, 1, 0, st, fin.data(), nullptr);
      if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(fold finish)");
    }
  }
  s->ctx->scratch_release(blk, st);
  return rc;
}

int acc_exec_foldseg_nd(acc_skel s, const acc_array *env, int32_t in_rank, const int64_t *in_shape, const acc_array *offsets,
                        const acc_array *out, acc_stream stream)
{
  if (!s) return fail(ACC_ERR_INVALID, "acc_exec_foldseg: NULL skeleton");
  ACC_RUN_SCOPE(s, static_cast<hipStream_t>(stream));
  if (!kind_is(s, {ACC_SKEL_FOLDSEG, ACC_SKEL_FOLD1SEG})) return fail(ACC_ERR_INVALID, "acc_exec_foldseg: skeleton is '%s'", s->entry.c_str());
  const int rank = std::max(1, s->spec.out_rank);        // of the input and of the result alike
  if (in_rank != rank || !in_shape) return fail(ACC_ERR_INVALID, "%s: input rank %d, kernel was built for %d", s->entry.c_str(), in_rank, rank);
  ACC_TRY(check_out(s, offsets, 1, "segment offsets", 1));
  ACC_TRY(check_out(s, out, rank, "result"));
  int64_t rows = 1;
  for (int d = 0; d < rank; ++d) {
    if (in_shape[d] < 0) return fail(ACC_ERR_INVALID, "%s: negative input extent", s->entry.c_str());
    if (d + 1 < rank) rows *= in_shape[d];
  }
  const int64_t inner = in_shape[rank - 1];
  // the offsets vector is one longer than the number of segments of a row: Execute.hs:320-324;
  // the result is  sh :. number of segments  for an input  sh :. inner
  const int64_t per_row = offsets->shape[0] - 1;
  if (per_row <= 0 || rows == 0) return ACC_OK;
  for (int d = 0; d + 1 < rank; ++d)
    if (out->shape[d] != in_shape[d]) return fail(ACC_ERR_INVALID, "%s: the result's outer extents differ from the input's", s->entry.c_str());
  if (out->shape[rank - 1] < per_row)
    return fail(ACC_ERR_INVALID, "%s: result holds %lld segments a row, %lld needed", s->entry.c_str(), (long long)out->shape[rank - 1], (long long)per_row);
  if (rank > 1 && out->shape[rank - 1] != per_row)
    return fail(ACC_ERR_INVALID, "%s: the result's rows must be exactly the %lld segments long", s->entry.c_str(), (long long)per_row);
  const int64_t nseg = rows * per_row, n = rows * inner;
  Args args;
  bool aligned = true;
  ACC_TRY(push_env(s, env, &args, &aligned));
  args.i64(nseg);
  push_ptrs(out, out->ncomp, &args, &aligned);
  args.i64(n);
  args.ptr(offsets->ptr[0]);
  if (rank > 1) {        // segments restart in every outer row: CodeGen/Reduction.hs:473-474
    args.i64(inner);
    args.i64(per_row);
  }
  const int v = aligned ? 0 : 1;
  ACC_TRY(s->ensure_variant(v));
  return launch_segmented(s, v, &args, env, out, nseg, n, static_cast<hipStream_t>(stream), rank == 1);
}

int acc_exec_foldseg(acc_skel s, const acc_array *env, int64_t n, const acc_array *offsets, const acc_array *out, acc_stream stream)
{
  if (s && std::max(1, s->spec.out_rank) != 1)
    return fail(ACC_ERR_INVALID, "acc_exec_foldseg: the kernel was built for rank %d: use acc_exec_foldseg_nd", s->spec.out_rank);
  return acc_exec_foldseg_nd(s, env, 1, &n, offsets, out, stream);
}

namespace {

// A variant that makes what another one of the instance makes too: whether it is there, or can be had now (a stream under
// capture is no place to load a module).  Where it cannot be built the call goes on with the other.
bool may_build(hipStream_t st)
{
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &capture) != hipSuccess) {
    (void)hipGetLastError();      // (answered by the other form: no later call is to find this error)
    return false;
  }
  return capture == hipStreamCaptureStatusNone;
}
bool may_take(acc_skel s, int v, hipStream_t st) { return s->variant_ready(v) || (may_build(st) && s->ensure_variant(v) == ACC_OK); }

// scanOp / scan1Op / scan'Op / scanCore, Execute.hs:328-392, as ONE launch.  `noalloc`: the tile descriptors live in
// the library's file-scope device array instead of a block of the context's pool, and nothing may be allocated,
// compiled or loaded on the way.
int scan_core(acc_skel s, const acc_array *env, int64_t n, const acc_array *out, const acc_array *total, acc_stream stream,
              const bool noalloc, const char *who)
{
  if (!s) return fail(ACC_ERR_INVALID, "%s: NULL skeleton", who);
  ACC_RUN_SCOPE(s, static_cast<hipStream_t>(stream));
  if (!kind_is(s, {ACC_SKEL_SCANL, ACC_SKEL_SCANL1, ACC_SKEL_SCANLP, ACC_SKEL_SCANR, ACC_SKEL_SCANR1, ACC_SKEL_SCANRP}))
    return fail(ACC_ERR_INVALID, "%s: skeleton is '%s'", who, s->entry.c_str());
  if (n < 0) return fail(ACC_ERR_INVALID, "%s: negative input extent", s->entry.c_str());
  ACC_TRY(check_out(s, out, 1, "result"));
  const int kind = s->spec.kind;
  const bool plus_one = (kind == ACC_SKEL_SCANL || kind == ACC_SKEL_SCANR);     // Execute.hs:328-339
  const bool primed = (kind == ACC_SKEL_SCANLP || kind == ACC_SKEL_SCANRP);     // Execute.hs:352-362
  if (out->shape[0] < n + (plus_one ? 1 : 0))
    return fail(ACC_ERR_INVALID, "%s: result holds %lld elements, %lld needed", s->entry.c_str(), (long long)out->shape[0], (long long)(n + (plus_one ? 1 : 0)));
  if (primed) ACC_TRY(check_out(s, total, 0, "total"));
  if (n == 0 && !plus_one && !primed) return ACC_OK;       // scanl1 / scanr1 of nothing is nothing

  hipStream_t st = static_cast<hipStream_t>(stream);
  Args args;
  bool aligned = true;
  ACC_TRY(push_env(s, env, &args, &aligned));
  push_out(*out, &args, &aligned);
  {
    bool ignore = true;      // a scalar's alignment decides nothing
    push_ptrs(primed ? total : nullptr, s->ncomp(), &args, &ignore);
  }
  args.i64(n);

  // An array of up to 12 MB takes the small-tile variant (4 rows a lane instead of 32): a workgroup runs through the
  // instructions of all the rows of its tile whether the array fills them or not, and a small array spread over few
  // large tiles leaves most of the device idle (Int32: 1024 elements 10.6 us -> 4.4, 2^18 8.6 -> 4.1, 2^21 10.0 ->
  // 8.1, 3 M + 3 14.8 -> 9.3; at 2^22 the two are level, 11.7 and 11.2, and so are 2^21 Float64, 12.0 and 13.2).
  const bool small = s->spec.scan_small_rows > 0 &&
                     n * (int64_t)s->spec.elt_size <= (int64_t)s->knobs.scan_small_below_kb * 1024;
  // Above that and up to 48 MB: tiles of 12 rows a lane.  Of 32 rows there are fewer tiles than two for a compute unit,
  // each a long way from its first load to its last store; of 4 so many that the chain of their totals takes longer than
  // the data (us with 4 / 8 / 12 / 16 / 32 rows: Int32 4 M 11.3 / 9.9 / 10.9 / 10.9 / 14.3, 6 M 14.6 / 12.1 / 11.7 / 12.7 /
  // 15.4, 12 M 29.5 / 20.2 / 18.8 / 18.6 / 21.0, 16 M 36.4 / 28.1 / 30.1 / 24.7 / 23.9; Float64 3 M 18.6 / 14.1 / 13.0 /
  // 13.9 / 16.0).  The variant is loaded together with the large tile's (acc_skel_s::ensure_variant).
  const bool mid = !small && s->spec.scan_mid_rows > 0 && s->knobs.scan_small_below_kb > 0 &&
                   n * (int64_t)s->spec.elt_size <= (int64_t)s->knobs.scan_mid_below_kb * 1024;
  const int v = (aligned ? 0 : 1) + (small ? 2 : mid ? 4 : 0);
  if (noalloc) {
    // building a variant compiles and loads a module: not here
    if (!s->variant_ready(v))
      return fail(ACC_ERR_INVALID, "%s: the %s %s-tile variant of this instance is not loaded yet; run acc_exec_scan once on operands of the same alignment and of %s %d KB first",
                  who, aligned ? "aligned" : "unaligned", small ? "small" : "large", small ? "at most" : "more than", s->knobs.scan_small_below_kb);
  } else {
    ACC_TRY(s->ensure_variant(v));
  }
  const int block = s->variants[v].block;
  const int64_t tile = (int64_t)block * s->variants[v].rows * s->vec();
  const int64_t tiles = (n + tile - 1) / tile;
  const int64_t grid = std::max<int64_t>(1, tiles);     // one workgroup per tile, in dispatch order
  const int64_t ndesc = std::max<int64_t>(1, tiles);
  const size_t esz = s->spec.elt_size;
  // one descriptor per tile: 64-bit words {flag, 4 bytes of the value}, `desc_stride` words apart
  // (more when the element needs more words)
  const size_t words = std::max<size_t>((esz + 3) / 4, (size_t)s->spec.scan_desc_stride);
  const size_t off_d0 = 256, off_d1 = 256, off_d2 = 256;
  const size_t bytes = 256 + round256((size_t)ndesc * 8 * words);
  if (noalloc) {
    if (tiles > ACC_NOALLOC_MAX_TILES)
      return fail(ACC_ERR_INVALID, "%s: %lld elements are %lld tiles of %lld, more than the %d the scratch array has descriptors for",
                  who, (long long)n, (long long)tiles, (long long)tile, ACC_NOALLOC_MAX_TILES);
    ACC_TRY(s->ctx->make_current());
    void *nbase = nullptr;
    uint32_t nepoch = 0;
    ACC_TRY(acc::noalloc_scan_state(s->ctx->device, bytes, st, &nbase, &nepoch));
    char *b = static_cast<char *>(nbase);
    args.ptr(reinterpret_cast<uint64_t>(b + off_d0));
    args.ptr(reinterpret_cast<uint64_t>(b + off_d1));
    args.ptr(reinterpret_cast<uint64_t>(b + off_d2));
    args.u32(nepoch);
    args.i64(tiles);
    args.ptr(s->ctx->status_dev);
    if (grid < 1 || grid > 0x7fffffffLL) return fail(ACC_ERR_INVALID, "%s: grid of %lld blocks", who, (long long)grid);
    ACC_HIP_TRY(launch_kernel(s->variants[v].fn, static_cast<unsigned>(grid), 1, 1, static_cast<unsigned>(block), 1, 1,
                                      0, st, args.data(), nullptr));
    return ACC_OK;
  }
  // A scan with more tiles than the device holds at once does not share the device with another such scan: tiles of
  // one could fill a compute die waiting for a tile that another die, full of waiting tiles of the other, has no
  // room for.  (Not under `noalloc`: calls through that entry that overlap on one device are excluded as it is.)
  const bool big = grid > resident(s, v);
  if (big) ACC_TRY(acc::scan_order_before(s->ctx->device, st));
  acc::ScratchRef blk;
  {
    const int arc = s->ctx->scratch_acquire(bytes, st, acc::SCRATCH_SCAN, &blk);
    if (arc != ACC_OK) {
      if (big) acc::scan_order_after(s->ctx->device);
      return arc;
    }
  }
  const uint32_t epoch = blk.epoch;
  char *base = static_cast<char *>(blk.ptr);
  if (s->spec.scan_ticket) (void)hipMemsetAsync(base + 64, 0, 4, st);      // (measurement knob scan.ticket: the counter tiles are drawn from)
  args.ptr(reinterpret_cast<uint64_t>(base + off_d0));
  args.ptr(reinterpret_cast<uint64_t>(base + off_d1));
  args.ptr(reinterpret_cast<uint64_t>(base + off_d2));
  args.u32(epoch);
  args.i64(tiles);
  args.ptr(s->ctx->status_dev);
  const int rc = launch(s, v, grid, 0, st, &args);
  if (big) acc::scan_order_after(s->ctx->device);
  s->ctx->scratch_release(blk, st);
  return rc;
}

}  // namespace

int acc_exec_scan(acc_skel s, const acc_array *env, int64_t n, const acc_array *out, const acc_array *total, acc_stream stream)
{
  return scan_core(s, env, n, out, total, stream, false, "acc_exec_scan");
}

int acc_exec_scan_noalloc(acc_skel s, const acc_array *env, int64_t n, const acc_array *out, const acc_array *total, acc_stream stream)
{
  return scan_core(s, env, n, out, total, stream, true, "acc_exec_scan_noalloc");
}

namespace {

// `permute const`, the combination that is the new value (skel_scatter.h): the defaults go to the result, the sources
// are stored over them.
int permute_const(acc_skel_s *s, const acc_array *env, int64_t n_src, const acc_array &defaults, const acc_array &out, bool copy_defaults, hipStream_t st)
{
  Args args;
  bool aligned = true;
  ACC_TRY(push_env(s, env, &args, &aligned));
  push_out(out, &args, &aligned);
  const int v = aligned ? 0 : 1;
  ACC_TRY(s->ensure_variant(v));
  const acc::Variant &var = s->variants[v];
  const int64_t ntarget = array_size(out);
  bool ignore = true;
  if (n_src <= acc::SCATTER_SMALL && ntarget <= acc::SCATTER_SMALL) {
    push_ptrs(&defaults, s->ncomp(), &args, &ignore);
    args.i32(copy_defaults ? 1 : 0);
    args.i64(n_src);
    ACC_HIP_TRY(launch_kernel(var.fn_finish, 1, 1, 1, 1024, 1, 1, 0, st, args.data(), nullptr));
    return ACC_OK;
  }
  if (copy_defaults) {
    Args f;
    push_ptrs(&out, s->ncomp(), &f, &ignore);
    push_ptrs(&defaults, s->ncomp(), &f, &ignore);
    f.i64(ntarget);
    const int64_t pieces = (ntarget * s->spec.vec_size + 15) / 16;      // 16 bytes a lane
    const int64_t grid = std::min<int64_t>((pieces + 255) / 256, (int64_t)1 << 20);
    ACC_HIP_TRY(launch_kernel(var.fn_fill, static_cast<unsigned>(grid), 1, 1, 256, 1, 1, 0, st, f.data(), nullptr));
  }
  acc::ScratchRef winner;
  const bool claimed = s->ncomp() > 1 || s->spec.elt_size > 8;           // as ACC_CLAIMED
  if (claimed) ACC_TRY(s->ctx->scratch_acquire((size_t)ntarget * 4, st, acc::SCRATCH_FOLD, &winner));
  // indices in `winner` are 32 bits wide: a longer source goes piece by piece, the later ones over the earlier
  int rc = ACC_OK;
  for (int64_t first = 0; first < n_src && rc == ACC_OK; first += (int64_t)1 << 32) {
    const int64_t past = std::min<int64_t>(n_src, first + ((int64_t)1 << 32));
    const int64_t tile = (int64_t)s->spec.block * s->spec.unroll;
    const unsigned grid = static_cast<unsigned>((past - first + tile - 1) / tile);
    Args piece = args;
    piece.i64(first);
    piece.i64(past);
    piece.ptr(reinterpret_cast<uint64_t>(winner.ptr));
    for (hipFunction_t fn : {claimed ? var.fn_claim : nullptr, var.fn}) {
      if (!fn || rc != ACC_OK) continue;
      hipError_t e = launch_kernel(fn, grid, 1, 1, static_cast<unsigned>(s->spec.block), 1, 1, 0, st, piece.data(), nullptr);
      if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(permute const)");
    }
  }
  s->ctx->scratch_release(winner, st);
  return rc;
}

}  // namespace

int acc_exec_permute(acc_skel s, const acc_array *env, int64_t n_src, const acc_array *defaults, const acc_array *out, acc_stream stream)
{
  if (!s) return fail(ACC_ERR_INVALID, "acc_exec_permute: NULL skeleton");
  ACC_RUN_SCOPE(s, static_cast<hipStream_t>(stream));
  if (!kind_is(s, {ACC_SKEL_PERMUTE})) return fail(ACC_ERR_INVALID, "acc_exec_permute: skeleton is '%s'", s->entry.c_str());
  if (n_src < 0) return fail(ACC_ERR_INVALID, "permute: negative source extent");
  ACC_TRY(check_out(s, out, s->spec.out_rank, "result"));
  ACC_TRY(check_out(s, defaults, s->spec.out_rank, "defaults"));
  for (int d = 0; d < out->rank; ++d)
    if (defaults->shape[d] != out->shape[d]) return fail(ACC_ERR_INVALID, "permute: defaults and result differ in shape");
  const int64_t ntarget = array_size(*out);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const size_t esz = s->spec.elt_size;
  ACC_TRY(s->ctx->make_current());
  // the result starts as a copy of the defaults: Execute.hs:401-406
  const bool copy_defaults = ntarget > 0 && defaults->ptr[0] != out->ptr[0];
  auto plain_copy = [&]() -> int {
    if (!copy_defaults) return ACC_OK;
    const int nc = s->ncomp();
    for (int c = 0; c < nc; ++c) {
      const size_t csz = nc == 1 ? esz : (size_t)acc::type_size(s->spec.comp_types[nc - 1 - c]);
      if (t_run.guard)      // under a loop's guard the copy, too, must not happen once the loop has ended
        ACC_TRY(acc::guarded_copy(out->ptr[c], defaults->ptr[c], (size_t)ntarget * csz, t_run.guard, st));
      else
        ACC_HIP_TRY(hipMemcpyAsync(reinterpret_cast<void *>(out->ptr[c]), reinterpret_cast<void *>(defaults->ptr[c]), (size_t)ntarget * csz, hipMemcpyDeviceToDevice, st));
    }
    return ACC_OK;
  };
  if (n_src == 0 || ntarget == 0) return plain_copy();
  if (s->spec.permute_replace) return permute_const(s, env, n_src, *defaults, *out, copy_defaults, st);

  // A combination without an atomic instruction of its own on few targets: compare-and-swap loops on the result
  // meet on those few addresses (16 M Float32 `max` updates on 1000 targets: 16.6 ms), the tables in LDS of the
  // locked template do not (74 us).  Such a skeleton carries that template as its variants 2 and 3.
  const int64_t lds_all = std::min<int64_t>((int64_t)s->ctx->props.sharedMemPerBlock, s->knobs.permute_lds_bytes);
  // targets per table in LDS (value + state word each), and how many such windows the targets need
  const int64_t lds_cap = std::max<int64_t>(1, (lds_all - 16) / ((int64_t)esz + 4));
  const int64_t lds_windows = (ntarget + lds_cap - 1) / lds_cap;
  const bool lds_table_fits = lds_windows <= s->knobs.permute_lock_max_windows &&
                              n_src >= s->knobs.permute_lock_lds_min_ratio * ntarget;
  // (Floating-point addition has an LDS atomic, but it runs at a fifth of the integer one's rate -- 16 M updates on
  // 1000 targets: 95 us against 63 us through the tables -- so between 48 and 6144 targets it goes the same way.
  // Below, the tables' locks are what lanes meet on (16 targets 149 us against 93, one target 2.1 ms against 0.12);
  // above, a table holds half the targets an array of plain values does and the passes over the source multiply
  // (16 384 targets 123 us against 102, 131 072: 407 against 107).)
  const bool fp_add = s->spec.combine_hint == ACC_COMBINE_ADD && (s->spec.elt_type == "float" || s->spec.elt_type == "double") &&
                      ntarget >= s->knobs.permute_fp_tables_from && ntarget <= s->knobs.permute_fp_tables_to;
  const bool generic_few = !s->spec.permute_locked && (s->spec.combine_hint == ACC_COMBINE_GENERIC || fp_add) && lds_table_fits &&
                           s->knobs.permute_generic_lds != 0;
  if (s->spec.permute_locked || generic_few) {
    // elements no atomic covers: a lock per target (the reference's lock array, Execute.hs:402-405)
    ACC_TRY(plain_copy());
    Args largs;
    bool al = true;
    ACC_TRY(push_env(s, env, &largs, &al));
    push_out(*out, &largs, &al);
    largs.i64(n_src);
    const int lv = (al ? 0 : 1) + (s->spec.permute_locked ? 0 : 2);
    ACC_TRY(s->ensure_variant(lv));
    acc::ScratchRef lblk;
    ACC_TRY(s->ctx->scratch_acquire((size_t)ntarget * 4 + 256, st, acc::SCRATCH_LOCKS, &lblk));
    // the locks start 256 bytes in
    largs.ptr(reinterpret_cast<uint64_t>(lblk.ptr) + 256);
    // Lanes in flight are kept to a few per target: every failed attempt on a lock is an atomic that queues in front
    // of the holder's own accesses, and with hundreds of lanes waiting per lock the device's whole atomic rate goes
    // into failed attempts (1000 targets: 12 M updates/s with every compute unit full, 20 times that with 32 lanes
    // per target).
    const int64_t lanes = std::max<int64_t>(64, ntarget * s->knobs.permute_lock_lanes_per_target);
    int64_t lgrid = std::min(acc_launch_grid(n_src, s->spec.block, s->ctx->props.multiProcessorCount, 8),
                             (lanes + s->spec.block - 1) / s->spec.block);
    // With few targets every workgroup combines in a table of its own in LDS (value + state word per target),
    // leaves it as a row of a table in memory, and a second launch folds the rows into the result: no global lock.
    const int64_t lds_budget = lds_all;
    int32_t lds_bins = 0, lds_copies = 1, win_blocks = 1;
    int64_t lds_need = 0;
    acc::ScratchRef dblk;
    uint64_t dump_val = 0, dump_ok = 0;
    if (lds_table_fits) {
      // windows of equal size; a single window that is small is kept once per wave, within a quarter of the LDS so
      // that several workgroups still fit
      lds_bins = static_cast<int32_t>((ntarget + lds_windows - 1) / lds_windows);
      auto lds_for = [&](int64_t copies) { return (((int64_t)lds_bins * copies * (int64_t)esz + 15) & ~int64_t(15)) + (int64_t)lds_bins * copies * 4; };
      const int64_t waves = s->spec.block / 64;
      while (lds_windows == 1 && lds_copies * 2 <= waves &&
             lds_for(lds_copies * 2) <= std::min<int64_t>(lds_budget, s->knobs.permute_lock_copies_bytes)) lds_copies *= 2;
      lds_need = lds_for(lds_copies);
      int bpc = 0;
      hipError_t oe = hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, s->variants[lv].fn, s->spec.block, (size_t)lds_need);
      if (oe != hipSuccess || bpc < 1) { (void)hipGetLastError(); bpc = 1; }
      // the device full of workgroups, shared out between the windows, as long as their rows stay within
      // `permute.lock_table_mbytes`
      const int64_t row_bytes = (int64_t)lds_bins * ((int64_t)esz + 4);
      const int64_t row_cap = std::max<int64_t>(lds_windows, ((int64_t)s->knobs.permute_lock_table_mbytes << 20) / row_bytes);
      const int64_t blocks = std::max<int64_t>(lds_windows, std::min<int64_t>(
          lds_windows * acc_launch_grid(n_src, s->spec.block, s->ctx->props.multiProcessorCount, bpc), std::min<int64_t>((int64_t)s->ctx->props.multiProcessorCount * bpc, row_cap)));
      win_blocks = static_cast<int32_t>(std::max<int64_t>(1, blocks / lds_windows));
      lgrid = lds_windows * win_blocks;
      const size_t ok_off = round256((size_t)(lgrid * lds_bins) * esz);
      const int arc = s->ctx->scratch_acquire(ok_off + (size_t)(lgrid * lds_bins) * 4, st, acc::SCRATCH_FOLD, &dblk);
      if (arc != ACC_OK) { s->ctx->scratch_release(lblk, st); return arc; }
      dump_val = reinterpret_cast<uint64_t>(dblk.ptr);
      dump_ok = dump_val + ok_off;
    }
    largs.i32(lds_bins);
    largs.i32(lds_copies);
    largs.ptr(dump_val);
    largs.ptr(dump_ok);
    largs.i32(win_blocks);
    largs.ptr(s->ctx->status_dev);
    int lrc = launch(s, lv, lgrid, lds_bins ? (size_t)lds_need : 0, st, &largs);
    if (lrc == ACC_OK && lds_bins) {
      Args j;
      bool jal = true;
      lrc = push_env(s, env, &j, &jal);
      push_out(*out, &j, &jal);
      j.ptr(dump_val);
      j.ptr(dump_ok);
      j.i32(win_blocks);
      j.i32(lds_bins);
      j.i64(ntarget);
      if (lrc == ACC_OK) {
        hipError_t je = launch_kernel(s->variants[lv].fn_finish, static_cast<unsigned>((ntarget + 3) / 4), 1, 1, 256, 1, 1, 0, st,
                                              j.data(), nullptr);
        if (je != hipSuccess) lrc = acc::fail_hip(je, "hipModuleLaunchKernel(permute_join)");
      }
    }
    s->ctx->scratch_release(dblk, st);
    s->ctx->scratch_release(lblk, st);
    return lrc;
  }

  Args args;
  bool aligned = true;
  ACC_TRY(push_env(s, env, &args, &aligned));
  push_out(*out, &args, &aligned);
  args.i64(n_src);

  // Integer addition on more targets than one LDS table of whole elements holds, but no more than one of 16-bit
  // counts does (65536 Int32 or Int64 targets in 128 KB): one pass over the source instead of one per window.  Also
  // from `permute.narrow_from` targets that whole elements would still hold: a single copy of such a table is what
  // all sixteen waves add to, and the smaller one does better (2^24 keys into 16 384 / 40 960 targets: 25.2 / 31.4
  // -> 22.8 / 27.0 us).
  const bool int_add = s->spec.combine_hint == ACC_COMBINE_ADD &&
                       (s->spec.elt_type == "Int32" || s->spec.elt_type == "Word32" || s->spec.elt_type == "Int64" || s->spec.elt_type == "Word64");
  // Only where the source is spelt as a small constant -- the counting idiom, `permute (+) zeros bin ones` -- since any
  // other addend would go to the result one device-scope atomic at a time (`permute.narrow=2` takes every source).
  const int narrow = s->knobs.permute_narrow;
  if (int_add && ntarget > std::min<int64_t>(s->knobs.permute_narrow_from, lds_all / (int64_t)esz) && ((ntarget + 1) / 2) * 4 <= lds_all && n_src >= 4 * ntarget &&
      (narrow == 2 || (narrow == 1 && s->spec.get_small_constant))) {
    const int nv = (aligned ? 0 : 1) + 6;
    ACC_TRY(s->ensure_variant(nv));
    // A source spelt as a small constant never adds to the result directly: its corrections go to a table of carries
    // (all zero between launches: the merge clears what it reads) and the merge writes  defaults + carries + rows,
    // so nothing has to be in the result beforehand and the copy of the defaults is not a launch of its own.  Any
    // other source (`permute.narrow=2`) may hold addends the table does not take; those go to the result, which must
    // then hold the defaults before the main kernel starts.
    const bool direct_adds = !s->spec.get_small_constant;
    if (direct_adds && copy_defaults) {
      Args f;
      f.ptr(0);
      f.i64(0);
      f.ptr(out->ptr[0]);
      f.ptr(defaults->ptr[0]);
      f.i64(ntarget);
      const int64_t fill_grid = std::min<int64_t>((ntarget + 255) / 256, 8 * (int64_t)s->ctx->props.multiProcessorCount);
      hipError_t fe = launch_kernel(s->variants[nv].fn_fill, static_cast<unsigned>(fill_grid), 1, 1, 256, 1, 1, 0, st, f.data(), nullptr);
      if (fe != hipSuccess) return acc::fail_hip(fe, "hipModuleLaunchKernel(permute_fill, narrow counts)");
    }
    const int64_t nwords = (ntarget + 1) / 2;
    const size_t nlds = (size_t)nwords * 4;
    // a workgroup a compute unit, whatever room a small table leaves for others: every one is a row that the merge reads (18 754
    // targets, 3.5 M / 67 M sources: 11.7 + 11.5 us / 50.2 + 8.2 with as many as there is room for, 8.6 + 4.6 / 49.6 + 4.8
    // so; 20 M on 30 000 targets 21.3 + 6.9 / 18.0 + 4.8)
    const int64_t cus_n = s->ctx->props.multiProcessorCount;
    const int64_t ngrid = acc_launch_grid(n_src, s->elements_per_block(), cus_n, 1);
    acc::ScratchRef nblk, cblk;
    ACC_TRY(s->ctx->scratch_acquire((size_t)ntarget * esz, st, acc::SCRATCH_CARRY, &cblk));
    const int64_t nd = (nwords + 1) / 2;             // words a workgroup's row of 8-bit counts takes
    int nrc = s->ctx->scratch_acquire((size_t)(ngrid * nd) * 4, st, acc::SCRATCH_FOLD, &nblk);
    if (nrc != ACC_OK) { s->ctx->scratch_release(cblk, st); return nrc; }
    const uint64_t ndump = reinterpret_cast<uint64_t>(nblk.ptr), ncarry = reinterpret_cast<uint64_t>(cblk.ptr);
    args.i32(static_cast<int32_t>(ntarget));
    args.i32(1);
    args.ptr(ndump);
    args.ptr(ncarry);
    args.ptr(s->ctx->status_dev);
    nrc = launch(s, nv, ngrid, nlds, st, &args);
    const bool main_launched = nrc == ACC_OK;
    if (nrc == ACC_OK) {
      Args m;
      bool mal = true;
      nrc = push_env(s, env, &m, &mal);
      push_out(*out, &m, &mal);
      m.ptr(ndump);
      m.i64(nwords);
      m.i32(static_cast<int32_t>(ngrid));
      m.i64(ntarget);
      m.ptr(ncarry);
      m.ptr(direct_adds ? out->ptr[0] : defaults->ptr[0]);
      if (nrc == ACC_OK) {
        // a workgroup per 64 words of a row, each of its waves its share of the rows
        const unsigned merge_threads = 64u * static_cast<unsigned>(s->spec.merge_waves);
        hipError_t me = launch_kernel(s->variants[nv].fn_finish, static_cast<unsigned>((nd + 63) / 64), 1, 1, merge_threads, 1, 1, 0, st,
                                      m.data(), nullptr);
        if (me != hipSuccess) nrc = acc::fail_hip(me, "hipModuleLaunchKernel(permute_merge, narrow counts)");
      }
    }
    // (the merge clears the carries it reads: if the main kernel went out and the merge did not, they stay behind)
    if (nrc != ACC_OK && main_launched) s->ctx->scratch_mark_dirty(cblk);
    s->ctx->scratch_release(cblk, st);
    s->ctx->scratch_release(nblk, st);
    return nrc;
  }

  // A hinted combination on more targets than two LDS tables hold: windows of targets, each with its share of the
  // workgroups, which walk the whole source (skel_permute.h).  Up to `permute.max_windows` passes are cheaper than
  // a device-scope atomic per element (27 G/s for the whole device).
  if (s->spec.combine_hint != ACC_COMBINE_GENERIC) {
    const int64_t wcap = std::max<int64_t>(1, lds_all / (int64_t)esz);
    int win_log = 0;                                       // a power of two of windows: targets are dealt out modulo it
    while (((ntarget + ((int64_t)1 << win_log) - 1) >> win_log) > wcap) ++win_log;
    const int64_t windows = (int64_t)1 << win_log;
    if (windows >= s->knobs.permute_windows_from && windows <= s->knobs.permute_max_windows && n_src >= 4 * ntarget) {
      const int wv = (aligned ? 0 : 1) + 4;
      ACC_TRY(s->ensure_variant(wv));
      ACC_TRY(plain_copy());
      const int64_t wbins = (ntarget + windows - 1) >> win_log;
      const size_t wlds = (size_t)wbins * esz;
      int bpc = 0;
      hipError_t oe = hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, s->variants[wv].fn, s->spec.block, wlds);
      if (oe != hipSuccess || bpc < 1) { (void)hipGetLastError(); bpc = 1; }
      const int64_t cus_w = s->ctx->props.multiProcessorCount;
      const int64_t win_blocks = std::max<int64_t>(1, std::min<int64_t>(cus_w * bpc / windows,
                                                                         acc_launch_grid(n_src, s->elements_per_block(), cus_w, bpc)));
      const int64_t wgrid = windows * win_blocks;
      acc::ScratchRef wblk;
      ACC_TRY(s->ctx->scratch_acquire((size_t)(wgrid * wbins) * esz, st, acc::SCRATCH_FOLD, &wblk));
      const uint64_t wdump = reinterpret_cast<uint64_t>(wblk.ptr);
      args.i32(static_cast<int32_t>(wbins));
      args.i32(1);
      args.ptr(wdump);
      args.ptr(0);
      args.i32(static_cast<int32_t>(win_blocks));
      args.i32(win_log);
      int wrc = launch(s, wv, wgrid, wlds, st, &args);
      if (wrc == ACC_OK) {
        struct MergeJob { uint64_t dump; int64_t stride, first, cols; int32_t nrows, slices, window_log; };
        const int64_t columns = (ntarget + 255) / 256;
        const int64_t slices = std::max<int64_t>(1, std::min<int64_t>(win_blocks, (2 * cus_w + columns - 1) / columns));
        MergeJob ja = {wdump, wbins, 0, ntarget, static_cast<int32_t>(win_blocks), static_cast<int32_t>(slices), win_log};
        MergeJob jb = {0, 0, 0, 0, 0, 1, -1};
        int32_t blocks_a32 = static_cast<int32_t>(columns * slices);
        Args m;
        bool mal = true;
        wrc = push_env(s, env, &m, &mal);
        push_out(*out, &m, &mal);
        void **mslots = m.data_without_guard();
        std::vector<void *> margs(mslots, mslots + m.count());
        margs.push_back(&ja);
        margs.push_back(&blocks_a32);
        margs.push_back(&jb);
        uint64_t mguard = t_run.guard;
        if (t_run.guarded) margs.push_back(&mguard);
        if (wrc == ACC_OK) {
          hipError_t me = launch_kernel(s->variants[wv].fn_finish, static_cast<unsigned>(blocks_a32), 1, 1, 256, 1, 1, 0, st,
                                                margs.data(), nullptr);
          if (me != hipSuccess) wrc = acc::fail_hip(me, "hipModuleLaunchKernel(permute_merge, windows)");
        }
      }
      s->ctx->scratch_release(wblk, st);
      return wrc;
    }
  }

  const int v = aligned ? 0 : 1;
  ACC_TRY(s->ensure_variant(v));

  // privatise target indices [0, bins) in LDS when the combine has a hardware
  // atomic and an identity; small targets get one copy per wave to spread
  // same-address traffic
  const int cus = s->ctx->props.multiProcessorCount;
  int64_t bins = 0, copies = 1;
  if (s->spec.combine_hint != ACC_COMBINE_GENERIC) {
    const int64_t budget = std::min<int64_t>((int64_t)s->ctx->props.sharedMemPerBlock, s->knobs.permute_lds_bytes) - s->variants[v].static_lds;
    const int64_t cap = std::max<int64_t>(0, budget / (int64_t)esz);
    bins = std::min(ntarget, cap);
    if (bins == ntarget && bins > 0) copies = std::max<int64_t>(1, std::min<int64_t>(s->spec.block / 64, cap / bins));
    copies = std::min<int64_t>(copies, s->knobs.permute_max_copies);
  }
  const size_t lds = (size_t)(bins * copies) * esz;
  int bpc = 0;
  hipError_t e = hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, s->variants[v].fn, s->spec.block, lds);
  if (e != hipSuccess || bpc < 1) { (void)hipGetLastError(); bpc = 1; }
  const int64_t grid = acc_launch_grid(n_src, s->elements_per_block(), cus, std::min(bpc, s->knobs.permute_max_blocks_per_cu));

  // How the privatised part leaves the blocks: atomics while they are few, otherwise a table of
  // per-block bins folded by a second kernel.
  // Targets beyond the LDS window would be hit with device-scope atomics, the slowest operation on
  // the machine.  While a row of the whole target stays well inside one XCD's L2, the workgroups of
  // each XCD share such a row instead, and the rows are folded into the result afterwards.
  constexpr int64_t XCD_ROWS = 16;                 // what the kernel's XCC_ID field can name
  const bool far_rows = bins > 0 && bins < ntarget &&
                        ntarget * (int64_t)esz <= (int64_t)s->knobs.permute_xcd_row_kbytes << 10;
  const bool table = bins > 0 && grid * bins > s->knobs.permute_atomic_flush_max;
  const size_t far_bytes = far_rows ? (size_t)(XCD_ROWS * ntarget) * esz : 0;
  const size_t dump_bytes = table ? (size_t)(grid * bins) * esz : 0;
  acc::ScratchRef blk;
  uint64_t far = 0, dump = 0;
  if (far_rows || table) {
    ACC_TRY(s->ctx->scratch_acquire(far_bytes + dump_bytes, st, acc::SCRATCH_FOLD, &blk));
    const uint64_t base = reinterpret_cast<uint64_t>(blk.ptr);
    if (far_rows) far = base;
    if (table) dump = base + far_bytes;
  }
  // Where every target has its bin in LDS and the bins leave by atomics, the result's first contents -- the defaults --
  // are copied by workgroup 0 of the main kernel while the others read the source, and a word in scratch memory
  // ({epoch, 1}, as the fold's partial results are tagged) tells them when their atomics may follow: one launch.
  const bool inline_fill = copy_defaults && !far_rows && !table && bins == ntarget && bins > 0 && n_src > 0 &&
                           s->knobs.permute_inline_fill != 0;
  acc::ScratchRef rblk;
  if (inline_fill) {
    const int arc = s->ctx->scratch_acquire(256, st, acc::SCRATCH_FLAGS, &rblk);
    if (arc != ACC_OK) { s->ctx->scratch_release(blk, st); return arc; }
  }
  int rc = ACC_OK;
  if (far_rows) {                       // one launch: identity into the XCD rows, defaults into the result
    Args f;
    f.ptr(far);
    f.i64(XCD_ROWS * ntarget);
    f.ptr(out->ptr[0]);
    f.ptr(defaults->ptr[0]);
    f.i64(copy_defaults ? ntarget : 0);
    const int64_t fill_grid = std::min<int64_t>((XCD_ROWS * ntarget + 255) / 256, 8 * (int64_t)cus);
    e = launch_kernel(s->variants[v].fn_fill, static_cast<unsigned>(fill_grid), 1, 1, 256, 1, 1, 0, st, f.data(), nullptr);
    if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(permute_fill)");
  } else if (copy_defaults && !inline_fill) {   // the defaults by the same kernel: a runtime copy of 1 KB takes 4 us, this launch 2
    Args f;
    f.ptr(0);
    f.i64(0);
    f.ptr(out->ptr[0]);
    f.ptr(defaults->ptr[0]);
    f.i64(ntarget);
    const int64_t fill_grid = std::min<int64_t>((ntarget + 255) / 256, 8 * (int64_t)cus);
    e = launch_kernel(s->variants[v].fn_fill, static_cast<unsigned>(fill_grid), 1, 1, 256, 1, 1, 0, st, f.data(), nullptr);
    if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(permute_fill, defaults)");
  }
  args.i32(static_cast<int32_t>(bins));
  args.i32(static_cast<int32_t>(copies));
  args.ptr(dump);
  args.ptr(far);
  args.ptr(inline_fill ? defaults->ptr[0] : 0);
  args.ptr(reinterpret_cast<uint64_t>(rblk.ptr));
  args.u32(rblk.epoch);
  args.ptr(s->ctx->status_dev);
  if (rc == ACC_OK) rc = launch(s, v, grid, lds, st, &args);
  if (inline_fill) s->ctx->scratch_release(rblk, st);
  if (rc == ACC_OK && (table || far_rows)) {
    // the tables are folded into the result by one launch: the per-block window rows, the per-XCD rows
    struct MergeJob { uint64_t dump; int64_t stride, first, cols; int32_t nrows, slices, window_log; };
    auto job = [&](uint64_t tbl, int64_t stride, int64_t first, int64_t cols, int64_t rows, int64_t *blocks) {
      // enough workgroups to fill the machine: columns x row slices
      const int64_t columns = (cols + 255) / 256;
      const int64_t slices = std::max<int64_t>(1, std::min<int64_t>(rows, (2 * cus + columns - 1) / columns));
      *blocks = columns * slices;
      return MergeJob{tbl, stride, first, cols, static_cast<int32_t>(rows), static_cast<int32_t>(slices), -1};
    };
    int64_t blocks_a = 0, blocks_b = 0;
    MergeJob ja = {0, 0, 0, 0, 0, 1, -1}, jb = {0, 0, 0, 0, 0, 1, -1};
    if (table) ja = job(dump, bins, 0, bins, grid, &blocks_a);
    if (far_rows) jb = job(far, ntarget, bins, ntarget - bins, XCD_ROWS, &blocks_b);
    Args m;
    bool al = true;
    rc = push_env(s, env, &m, &al);
    push_out(*out, &m, &al);
    int32_t blocks_a32 = static_cast<int32_t>(blocks_a);
    void **mslots = m.data_without_guard();
    std::vector<void *> margs(mslots, mslots + m.count());
    margs.push_back(&ja);
    margs.push_back(&blocks_a32);
    margs.push_back(&jb);
    uint64_t mguard = t_run.guard;
    if (t_run.guarded) margs.push_back(&mguard);
    if (rc == ACC_OK) {
      e = launch_kernel(s->variants[v].fn_finish, static_cast<unsigned>(blocks_a + blocks_b), 1, 1, 256, 1, 1, 0, st, margs.data(), nullptr);
      if (e != hipSuccess) rc = acc::fail_hip(e, "hipModuleLaunchKernel(permute_merge)");
    }
  }
  s->ctx->scratch_release(blk, st);
  return rc;
}

// Whether a volume that could go by the vectors of whole planes (skel_stencil_flat.h) is better off in strips that walk through
// many planes: `both` the bytes of an element of source and result.  us in strips / by vectors, 7 and 27 points Float32, then
// 7 and 27 points Float64 of half the columns or other sizes as given:
//   - By vectors what the memory-side cache holds a good part of (200 x 512 x 512 55 / 50, 127 / 62; 60 x 1024 x 1024 64 / 61,
//     118 / 74; Float64 50 x 512 x 1024 53 / 52, 89 / 58), and rows that leave much of a strip outside the array (400^3 Float64
//     244 / 218, 356 / 228; 418 x 418 x 600 220 / 169, 252 / 183; 250 x 900 x 900 377 / 346, 375 / 371).
//   - Rows of whole strips: in strips from 768 MB on (512^3 194 / 222, 203 / 234; 50 x 1000 x 1024 Float64 145 / 172, 178 / 192),
//     and from 512 MB on where planes lie far apart: a result that reads few rows from planes of 2 MB on (150 x 512 x 1024
//     108 / 134, 75 x 1024 x 1024 100 / 130; Float64 170 x 512 x 512 136 / 149, 75 x 512 x 1024 101 / 137; but 360 x 512 x 512
//     158 / 150), one that reads many from 2^19 elements and 576 MB on (180 x 512 x 1024 153 / 178, 75 x 1024 x 1024 144 / 165,
//     Float64 75 x 512 x 1024 144 / 161; but 130 x 512 x 1024 133 / 105, 170 x 512 x 512 Float64 196 / 164).
//   - Rows of nearly whole strips (a twentieth outside at most) in strips from 512 MB and planes of 3.5 MB on: Float64 that
//     reads few rows (45 x 1000 x 1000 134 / 153, 300 x 700 x 760 501 / 560, 500 x 640 x 1000 983 / 1143; with 27 points 164 / 167,
//     632 / 610, 1186 / 1208: left), Float32 that reads many (90 x 1000 x 1000 158 / 167, 200 x 1200 x 1000 415 / 459, 1000^3 1658 /
//     1816), and Float32 that reads few up to planes of 6 MB (135 / 149, 407 / 416, 1647 / 1718; but 150 x 1500 x 2040 966 / 846,
//     100 x 3000 x 2500 1427 / 1353).  Smaller planes go either way (510^3 222 / 219, 228 / 233; 600 x 512 x 500 279 / 251, 337 /
//     263; 600 x 400 x 1000 396 / 415, 406 / 442; 300 x 700 x 760 271 / 260, 331 / 288).
static bool volume_in_strips(const acc_skel_s *s, int64_t w, int64_t h, int64_t planes, int64_t both)
{
  const int64_t half = (int64_t)32 * s->spec.svec, halves = (w + half - 1) / half;
  const int64_t covered = half * (halves <= 3 ? halves : (halves + 1) / 2 * 2);        // columns of all strips (half ones up to three)
  const int64_t kb = w * h * both / 1024 * planes, plane_kb = w * h * both / 2048;
  const bool few = s->spec.flat_prefetch >= s->spec.flat_planes, wide = both >= 16;
  if (kb <= 512 * 1024) return false;
  if (w % (2 * half) == 0) return kb > 768 * 1024 || (few ? plane_kb >= 2048 : kb > 576 * 1024 && w * h >= (1 << 19));
  return (covered - w) * 20 <= covered && plane_kb >= 3584 && (few ? wide || plane_kb <= 6144 : !wide);
}

// `in2` is the second source of a stencil2, NULL for a stencil
static int stencil_once(acc_skel s, const acc_array *env, const acc_array *in, const acc_array *in2, const acc_array *out, hipStream_t st)
{
  ACC_RUN_SCOPE(s, st);
  const int rank = s->spec.out_rank;
  Args args;
  bool aligned = true;
  ACC_TRY(push_env(s, env, &args, &aligned));
  push_out(*out, &args, &aligned);
  const int64_t w = out->shape[rank - 1];
  const int64_t h = rank >= 2 ? out->shape[rank - 2] : 1;
  const int64_t planes = rank == 3 ? out->shape[0] : 1;
  // rows start on 16-byte boundaries only if the row pitch allows it: of every component of a source
  auto row_aligned = [&](const acc_array &a, const std::vector<std::string> &comps) {
    const int nc = (int)comps.size();
    for (int c = 0; c < nc; ++c) {
      const size_t esz = acc::type_size(comps[nc - 1 - c]);          // component c is the (nc - 1 - c)-th in writing order
      if (!aligned16(a.ptr[c]) || (a.shape[rank - 1] * (int64_t)esz) % 16 != 0) return false;
    }
    return true;
  };
  // (of a tuple result: the rows of every component's array)
  const int ncomp = s->ncomp();
  for (int c = 0; c < ncomp; ++c) {
    const int64_t csz = ncomp == 1 ? (int64_t)s->spec.elt_size : (int64_t)acc::type_size(s->spec.comp_types[ncomp - 1 - c]);
    if ((w * csz) % 16 != 0) aligned = false;
  }
  if (!row_aligned(*in, s->spec.stencil_in_comps)) aligned = false;
  if (in2) {      // each source with its extents (Stencil.hs:146-152)
    if (!row_aligned(*in2, s->spec.stencil_in2_comps)) aligned = false;
    bool ignore = true;
    push_out(*in, &args, &ignore);
    push_out(*in2, &args, &ignore);
  } else {
    bool ignore = true;
    push_ptrs(in, in->ncomp, &args, &ignore);
  }
  if (array_size(*out) == 0) return ACC_OK;
  // An array of a few columns leaves nearly every lane of a strip outside it (3 x 3 on 2^24 x 3: 1.9 ms, 7 points on
  // 2^22 x 2 x 2 and 2^24 x 1 x 1: 0.76 and 2.8 ms): variants 6 and 7 of the instance, an element a thread as for the
  // stencils that strips cannot take, run at 2.8 (2-D) and 2.1 TB/s (3-D) whatever the shape, which is more than the
  // strips reach up to 36 columns in 2-D (2^20 rows of 28 / 33: 117 / 119 us in strips, 84 / 98 so; 2^19 of 40: 60
  // either way) and 16 in 3-D (2^17 x 8 x 16: 74 against 65; 2^14 x 32 x 32: 51 against 65).
  const bool thin = !s->spec.stencil_nd && ((rank == 2 && w <= s->knobs.stencil_thin_2d) || (rank == 3 && w <= s->knobs.stencil_thin_3d));
  if (s->spec.stencil_nd || thin) {
    // an element of the result a thread (skel_stencil_nd.h); the kernel takes the strips' `walk` and ignores it
    args.i32(0);
    const int v = (aligned ? 0 : 1) + (thin ? 6 : 0);
    ACC_TRY(s->ensure_variant(v));
    const int64_t grid = acc_launch_grid(array_size(*out), s->spec.block, resident(s, v), s->knobs.map_oversub);
    return launch(s, v, grid, 0, st, &args);
  }
  // A volume takes variants 8 and 9, lanes over the vectors of a whole plane, where the instance has them
  // (skel_stencil_flat.h) and volume_in_strips does not say otherwise.
  if (s->spec.flat_planes > 0 && s->knobs.stencil_flat != 0 && w >= s->spec.svec &&
      (s->knobs.stencil_flat == 2 || !volume_in_strips(s, w, h, planes, s->spec.elt_size + acc::type_size(s->spec.stencil_in_comps[0])))) {
    const int64_t deep = s->spec.flat_planes, per_block = s->spec.block / 64;
    const int64_t owned = s->spec.reach_x == 1 ? 62 : 64;          // lanes that store: the others hand over columns
    const int64_t per_plane = (((w + s->spec.svec - 1) / s->spec.svec) * h + owned - 1) / owned, runs = (planes + deep - 1) / deep;
    // the kernel counts lanes and waves in 32 bits, and bytes within a plane of source and result
    const int64_t widest = std::max(s->spec.elt_size, 8);
    const int v = (aligned ? 0 : 1) + 8;
    if (w * h * widest < ((int64_t)1 << 32) && planes < ((int64_t)1 << 30) && per_plane * 8 < ((int64_t)1 << 30) && (per_plane + 40) * planes < ((int64_t)1 << 30) &&
        may_take(s, v, st)) {
      args.i32(0);
      // every die an eighth of every plane, or one after the other: as the kernel numbers them
      const int64_t grid = per_plane >= 8 * acc::flat_spread ? 8 * (((per_plane + 7) / 8 + per_block - 1) / per_block) * runs : (per_plane * runs + per_block - 1) / per_block;
      return launch(s, v, grid, 0, st, &args);
    }
  }
  // one wave per strip of 256 columns x tile_h rows
  // (for 2-D the waves of a workgroup are stacked vertically, so the row count is rounded up to whole groups)
  const int64_t waves = s->spec.block / 64;
  // An array narrower than half a strip (a quarter) takes the variant with half (a quarter) of the columns a lane,
  // where the stencil's reach allows: the lanes of a strip that lie outside the array do nothing.
  int narrow = 0;
  while (narrow < s->knobs.stencil_narrow_max && (s->spec.svec >> (narrow + 1)) >= std::max(1, s->spec.reach_x) &&
         w <= (int64_t)64 * (s->spec.svec >> (narrow + 1)))
    ++narrow;
  // Strips that walk through planes are bound by the instructions of a strip, whatever its share of columns inside the
  // array: one and a half strips' width is taken as three strips of half the width, not as two of the whole one
  // (200 x 200 x 300: 35.3 -> 27.4 us), and less than one strip's width as two of half the width, not as one that the
  // edge of the array cuts (150^3: 17.0 -> 13.3 us).  (In 2-D the columns a last strip produces a second time cost
  // next to nothing.)
  if (narrow == 0 && s->spec.zmarch && (s->spec.svec >> 1) >= std::max(1, s->spec.reach_x) && s->knobs.stencil_half_strips != 0) {
    const int64_t halves = (w + 32 * s->spec.svec - 1) / (32 * s->spec.svec);
    if (halves == 3 || (halves == 2 && w < 64 * s->spec.svec)) narrow = 1;
  }
  const int64_t tile_w = (int64_t)64 * (s->spec.svec >> narrow);
  const int64_t strips_x = (w + tile_w - 1) / tile_w;
  int64_t bands = (h + s->spec.tile_h - 1) / s->spec.tile_h;
  if (rank == 2 && s->knobs.stencil_stack) bands = (bands + waves - 1) / waves * waves;
  int64_t zbands = (planes + s->spec.tile_z - 1) / s->spec.tile_z;             // tile_z result planes per strip
  int64_t walk = s->spec.tile_h;
  if (s->spec.zmarch) {                  // strips tile_z rows tall that walk through tile_h planes
    bands = (h + s->spec.tile_z - 1) / s->spec.tile_z;
    // ... or through fewer, halving down to 4, until there are three strips for every compute unit: a volume of
    // 256^3 has 256 strips of 64 planes, a wave for every fourth SIMD (44.1 us; 23.4 with 1024 strips of 16 planes,
    // although each reads 2 rz planes beyond its own; 128 x 128 x 256: 40.5 us -> 6.6 at 4 planes a strip).
    const int64_t enough = (int64_t)s->knobs.stencil_strips_per_cu * s->ctx->props.multiProcessorCount;
    const int64_t shortest = std::max(1, std::min(s->knobs.stencil_walk_min, s->spec.tile_h));
    while (walk / 2 >= shortest && strips_x * bands * ((planes + walk - 1) / walk) < enough) walk /= 2;
    zbands = (planes + walk - 1) / walk;
  }
  args.i32(static_cast<int32_t>(walk));
  return launch(s, (aligned ? 0 : 1) + 2 * narrow, (strips_x * bands * zbands + waves - 1) / waves, 0, st, &args);
}

// Two, three or four applications of a stencil in one launch (skel_stencil_pair.h): the waves' columns, rows and number, where
// the instance and the shape allow; false if not.
struct ManyPlan { int64_t walk, waves; };
static bool plan_many(const acc_skel_s *s, int levels, const acc_array *out, ManyPlan *plan)
{
  if (!s->spec.pair_form || s->knobs.stencil_pair == 0 || array_size(*out) == 0) return false;
  // lanes at either side of a strip whose columns go wrong, and the columns of a strip (as the kernel has them)
  const int64_t svec = s->spec.svec, outer = s->spec.reach_x > 0 ? (levels + svec - 1) / svec : 1, owned = (64 - 2 * outer) * svec;
  const int64_t w = out->shape[1], h = out->shape[0];
  if ((w != owned && w < owned + outer * svec) || h < 3 || w >= (1 << 30) || h >= (1 << 30)) return false;
  const int64_t strips = (w + owned - 1) / owned;
  // rows a wave walks through: 28, or fewer, down to 4, as long as that leaves a compute unit fewer than eight waves (the
  // rows above and below are read and worked out for every walk anew: 3000 x 3000 Float32 in 28 / 20 / 12 / 8 rows 24.5 /
  // 22.4 / 25.0 / 23.3 us for four applications, 1024 x 1024 in 16 / 8 / 4 rows 14.2 / 9.9 / 9.2, 300 x 300 13.5 / 9.1 / 6.3)
  plan->walk = s->knobs.stencil_pair_walk;
  if (plan->walk <= 0) plan->walk = std::max<int64_t>(4, std::min<int64_t>(28, h * strips / (8 * (int64_t)s->ctx->props.multiProcessorCount)));
  plan->waves = strips * ((h + plan->walk - 1) / plan->walk);
  return plan->waves < (1 << 30);
}

// ... and the launch; false, with nothing done, where a form is not there and cannot be had.
static bool stencil_many(acc_skel s, int levels, const acc_array *env, const acc_array *in, const acc_array *out, hipStream_t st, int *rc)
{
  ManyPlan plan;
  if (!plan_many(s, levels, out, &plan)) return false;
  const int64_t w = out->shape[1], esz = s->spec.elt_size;
  // the forms for four, three and two are compiled at the same time and loaded together, four the last: which of them a call
  // finds does not hang on what was called before
  const int four = 10 + ((aligned16(in->ptr[0]) && aligned16(out->ptr[0]) && w * esz % 16 == 0) ? 0 : 1), v = four + 2 * (4 - levels);
  if (!s->variant_ready(four)) {
    if (!may_build(st)) return false;
    for (int k = four; k < four + 6; k += 2)
      if (s->start_variant(k) != ACC_OK) return false;
    for (int k = four + 4; k >= four; k -= 2)
      if (s->ensure_variant(k) != ACC_OK) return false;
  }
  *rc = [&]() -> int {
    ACC_RUN_SCOPE(s, st);
    Args args;
    bool aligned = true;
    ACC_TRY(push_env(s, env, &args, &aligned));
    push_out(*out, &args, &aligned);
    push_ptrs(in, in->ncomp, &args, &aligned);
    args.i32(static_cast<int32_t>(plan.walk));
    const int64_t per_block = s->spec.block / 64, grid = (plan.waves + per_block - 1) / per_block;
    ACC_TRY(s->ctx->make_current());
    const acc::Variant &var = s->variants[v];
    ACC_HIP_TRY(launch_kernel(var.fn, static_cast<unsigned>(grid), 1, 1, static_cast<unsigned>(var.block), 1, 1, 0, st, args.data(), nullptr));
    return ACC_OK;
  }();
  return true;
}

// What a launch of one, two, three and four applications takes, in twentieths of one by itself (entry 0 is not used).  3 x 3, us
// one / two / three / four: small arrays, where launches count, 500 x 500 Float32 3.2 / 4.8 / 5.8 / 7.2, 768 x 768 Float64 4.3 /
// 6.4 / 7.7 / 9.1; such that the memory-side cache holds both, where one application by itself writes past it, 3000 x 3000
// Float32 15.9 / 16.2 / 20.9 / 27.1, Float64 27.1 / 22.3 / 25.9 / 33.2, 4096 x 4096 Float64 45.6 / 35.6 / 42.8 / 54.2; and larger
// ones, 8192 x 8192 88 / 110 / 111 / 116, Float64 176 / 225 / 217 / 218.  A call of five, as 2 2 1 and as 3 1 1: 12.6 / 12.3,
// 16.6 / 17.2; 45.8 / 50.8, 68 / 77, 108 / 123; 305 / 272, 620 / 563.  Of six, as 2 2 1 1 and as 3 1 1 1, either side of the
// lower line: 1500 x 1500 Float32 33.9 / 31.7, 2048 x 2048 37.4 / 39.8; of the upper one: 4096 x 4096 Float64 160 / 176, 6000 x
// 6000 Float32 219 / 202.
static const int32_t *stencil_costs(const acc_skel_s *s, const acc_array *out)
{
  static const int32_t small[5] = {0, 20, 31, 37, 44}, held[5] = {0, 20, 19, 23, 30}, large[5] = {0, 20, 25, 25, 27};
  const int64_t bytes = array_size(*out) * (int64_t)s->spec.elt_size;
  return bytes < ((int64_t)12 << 20) ? small : bytes <= ((int64_t)128 << 20) ? held : large;
}

// How many launches of four, three and two applications a call of `iters` makes (left[4], left[3] and left[2]; the rest go one by
// one): as leaves every result where one a launch would, so an even number of fours and twos together -- the arrays then have
// changed places as often; a three changes them as three single ones do -- and at least one application by itself at the
// end, whose source is then the result before the last.  Of these splits the one that takes least.  (Strips of two columns a
// lane are wider for two applications than for three or four: what the rows are too short for is not among them.)
static void stencil_split(const acc_skel_s *s, const acc_array *out, int32_t iters, int32_t left[5])
{
  const int32_t *cost = stencil_costs(s, out);
  const int64_t many = std::max(iters, 1) - 1;
  ManyPlan plan;
  const bool threes = plan_many(s, 3, out, &plan), twos = plan_many(s, 2, out, &plan);
  const int64_t most = plan_many(s, 4, out, &plan) ? many / 4 : 0;
  int64_t least = -1;
  for (int64_t four = most; four >= 0 && four > most - 8; --four)
    for (int64_t two = four & 1; two <= (twos ? 3 : 0) && 4 * four + 2 * two <= many; two += 2) {
      const int64_t rest = many - 4 * four - 2 * two, three = threes ? rest / 3 : 0, one = rest - 3 * three;
      const int64_t all = four * cost[4] + three * cost[3] + two * cost[2] + one * cost[1];
      if (least >= 0 && all >= least) continue;
      least = all;
      left[4] = static_cast<int32_t>(four);
      left[3] = static_cast<int32_t>(three);
      left[2] = static_cast<int32_t>(two);
    }
}

static int stencil_check(acc_skel s, const acc_array *in, const acc_array *out)
{
  if (!s) return fail(ACC_ERR_INVALID, "acc_exec_stencil: NULL skeleton");
  if (!kind_is(s, {ACC_SKEL_STENCIL})) return fail(ACC_ERR_INVALID, "acc_exec_stencil: skeleton is '%s'", s->entry.c_str());
  ACC_TRY(check_out(s, out, s->spec.out_rank, "result"));
  ACC_TRY(check_out(s, in, s->spec.out_rank, "source", (int)s->spec.stencil_in_comps.size()));
  for (int d = 0; d < out->rank; ++d)
    if (in->shape[d] != out->shape[d]) return fail(ACC_ERR_INVALID, "stencil: source and result differ in shape");
  for (int ci = 0; ci < in->ncomp && array_size(*out) > 0; ++ci)
    for (int co = 0; co < out->ncomp; ++co)
      if (in->ptr[ci] == out->ptr[co]) return fail(ACC_ERR_INVALID, "stencil: source and result must not alias");
  return ACC_OK;
}

int acc_exec_stencil(acc_skel s, const acc_array *env, const acc_array *in, const acc_array *out, acc_stream stream)
{
  ACC_TRY(stencil_check(s, in, out));
  return stencil_once(s, env, in, nullptr, out, static_cast<hipStream_t>(stream));
}

int acc_exec_stencil2(acc_skel s, const acc_array *env, const acc_array *in1, const acc_array *in2, const acc_array *out, acc_stream stream)
{
  if (!s) return fail(ACC_ERR_INVALID, "acc_exec_stencil2: NULL skeleton");
  if (!kind_is(s, {ACC_SKEL_STENCIL2})) return fail(ACC_ERR_INVALID, "acc_exec_stencil2: skeleton is '%s'", s->entry.c_str());
  ACC_TRY(check_out(s, out, s->spec.out_rank, "result"));
  ACC_TRY(check_out(s, in1, s->spec.out_rank, "first source", (int)s->spec.stencil_in_comps.size()));
  ACC_TRY(check_out(s, in2, s->spec.out_rank, "second source", (int)s->spec.stencil_in2_comps.size()));
  for (int d = 0; d < out->rank; ++d)
    if (out->shape[d] > std::min(in1->shape[d], in2->shape[d]))
      return fail(ACC_ERR_INVALID, "stencil2: the result is larger than the intersection of the sources' extents");
  for (const acc_array *in : {in1, in2})
    for (int ci = 0; ci < in->ncomp && array_size(*out) > 0; ++ci)
      for (int co = 0; co < out->ncomp; ++co)
        if (in->ptr[ci] == out->ptr[co]) return fail(ACC_ERR_INVALID, "stencil2: a source and the result must not alias");
  return stencil_once(s, env, in1, in2, out, static_cast<hipStream_t>(stream));
}

int acc_exec_stencil_iterate(acc_skel s, const acc_array *env, const acc_array *a, const acc_array *b, int32_t iters, acc_stream stream, int32_t *result_in_b)
{
  ACC_TRY(stencil_check(s, a, b));
  if (iters < 0) return fail(ACC_ERR_INVALID, "stencil: negative iteration count");
  const acc_array *src = a, *dst = b;
  int32_t left[5] = {0, 0, 0, 0, 0};
  stencil_split(s, b, iters, left);
  for (int32_t i = 0; i < iters;) {
    const int32_t levels = left[4] > 0 ? 4 : left[3] > 0 ? 3 : left[2] > 0 ? 2 : 1;
    int rc = ACC_OK;
    if (levels > 1 && !stencil_many(s, levels, env, src, dst, static_cast<hipStream_t>(stream), &rc)) {
      left[4] = left[3] = left[2] = 0;   // (never after the first: what one launch has taken the others find there)
      continue;
    }
    if (levels == 1) rc = stencil_once(s, env, src, nullptr, dst, static_cast<hipStream_t>(stream));
    ACC_TRY(rc);
    i += levels;
    --left[levels];
    std::swap(src, dst);
  }
  if (result_in_b) *result_in_b = (iters & 1);
  return ACC_OK;
}

}  // extern "C"
