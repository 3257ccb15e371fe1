// The layer's host path: one call per autograd node.  Allocates every output and workspace with
// torch's caching allocator, enqueues the kernels of libmomoe_hip.so on the current stream and
// records the autograd nodes.  It is native because a call makes a dozen launches: driven from
// Python (a wrapper, an allocation or two and a foreign-function call per launch) the host needed
// 84 us for a forward and 240 us for a training step of any size, longer than the GPU works on a
// decode call or on a small step.
//
// Nothing here synchronises with the device (unless the caller asks for the routing check): every
// launch is sized from static upper bounds and the routing-dependent tile list lives in device
// memory.
#include <ATen/autocast_mode.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>
#include <torch/library.h>

#include <atomic>
#include <mutex>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/momoe_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- launch timing (kernel_timer in _hip.py): an event pair around every library call ---------
struct TimedCall {
  std::string name;
  hipEvent_t begin, end;
};
std::mutex g_timing_mutex;
std::atomic<bool> g_timing{false};  // read by every thread that launches; a stale read only skips a record
std::vector<TimedCall> g_calls;

void timing_start() { g_timing.store(true, std::memory_order_relaxed); }
void timing_stop() { g_timing.store(false, std::memory_order_relaxed); }
// durations in ms of the calls recorded so far; the device must be idle
std::vector<std::pair<std::string, double>> timing_take() {
  std::lock_guard<std::mutex> lock(g_timing_mutex);
  std::vector<std::pair<std::string, double>> out;
  for (auto& c : g_calls) {
    float ms = 0.0f;
    const bool ok = hipEventElapsedTime(&ms, c.begin, c.end) == hipSuccess;
    (void)hipEventDestroy(c.begin);
    (void)hipEventDestroy(c.end);
    if (ok) out.emplace_back(c.name, (double)ms);
  }
  g_calls.clear();
  return out;
}

// fn(), with an event pair around it on `st` while launches are timed
template <class Fn>
auto timed(const char* name, hipStream_t st, Fn fn) {
  if (!g_timing.load(std::memory_order_relaxed)) return fn();
  TimedCall t{name, nullptr, nullptr};
  const bool begun = hipEventCreate(&t.begin) == hipSuccess && hipEventCreate(&t.end) == hipSuccess &&
                     hipEventRecord(t.begin, st) == hipSuccess;
  auto result = fn();
  if (begun && hipEventRecord(t.end, st) == hipSuccess) {
    std::lock_guard<std::mutex> lock(g_timing_mutex);
    g_calls.push_back(std::move(t));
  } else {
    if (t.begin) (void)hipEventDestroy(t.begin);
    if (t.end) (void)hipEventDestroy(t.end);
  }
  return result;
}

template <class Fn, class... Args>
void call(const char* name, hipStream_t st, Fn fn, Args... args) {
  const int code = timed(name, st, [&] { return fn(args..., (void*)st); });
  TORCH_CHECK(code == MOMOE_OK, name, " failed: status ", code, " (", momoe_status_string(code), ")");
}
#define MOMOE_CALL(fn, st, ...) call(#fn, st, fn, __VA_ARGS__)

hipStream_t stream_of(const at::Device& dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

Tensor empty_bf16(at::IntArrayRef size, const at::Device& dev) {
  return at::empty(size, at::TensorOptions().dtype(at::kBFloat16).device(dev));
}
Tensor empty_i32(int64_t n, const at::Device& dev) {
  return at::empty({n}, at::TensorOptions().dtype(at::kInt).device(dev));
}
Tensor empty_f32(at::IntArrayRef size, const at::Device& dev) {
  return at::empty(size, at::TensorOptions().dtype(at::kFloat).device(dev));
}

// Buffers that live no longer than the call: pieces of one allocation where they are few bytes in all, since an
// allocation takes the host a microsecond and a small call is as long as its host work (in us of the host, a forward of 7 tokens
// with its router 37.2 -> 34.8, the backward of 128 tokens 88 -> 81); allocations of their own, given back as soon as they are
// done with, where their size counts.  The line is torch's own between small allocations and large ones; forwards in a row below
// it, us, in several -> in one: 7 tokens, D = 256, H = 128, N = 16, K = 2 19.8 -> 18.2; 128, 512, 128, 32, 2 21.9 -> 21.6; 150, 512, 128, 48, 4
// 22.3 -> 22.1; 300, 512, 256, 16, 2 25.9 -> 25.4; 200, 256, 256, 96, 4 26.7 -> 26.6; 400, 384, 128, 64, 2 24.2 -> 24.1.
class Transients {
  const at::Device dev_;
  Tensor block_;
  int64_t used_ = 0;
  static int64_t up(int64_t bytes) { return (bytes + 255) & ~(int64_t)255; }

 public:
  Transients(const at::Device& dev, std::initializer_list<int64_t> sizes) : dev_(dev) {
    constexpr int64_t kMost = 1 << 20;
    int64_t all = 0;
    for (int64_t bytes : sizes) all += bytes <= kMost ? up(bytes) : 2 * kMost;
    if (all <= kMost) block_ = bytes_of(all);
  }
  Tensor bytes_of(int64_t bytes) const { return at::empty({bytes}, at::TensorOptions().dtype(at::kByte).device(dev_)); }
  // the next of those sizes; `own` holds it if it is an allocation of its own
  void* take(int64_t bytes, Tensor& own) {
    if (!block_.defined()) return (own = bytes_of(bytes)).data_ptr();
    TORCH_INTERNAL_ASSERT(used_ + bytes <= block_.numel());
    void* const p = (char*)block_.data_ptr() + used_;
    used_ += up(bytes);
    return p;
  }
};

// A Python exception of the given type, raised when the binding returns
[[noreturn]] void throw_python(PyObject* type, const std::string& what) {
  py::gil_scoped_acquire gil;
  PyErr_SetString(type, what.c_str());
  throw py::error_already_set();
}

// Whether a call has to go through its autograd function.  A forward-mode tangent counts: the
// function refuses it, where the plain forward would drop it without a word.
bool wants_autograd(std::initializer_list<const Tensor*> inputs) {
  bool any = false;
  for (const Tensor* t : inputs)
    any = any || (at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(/*level=*/0).defined();
  return any;
}

// A call under torch.jit.trace, made again through the operator momoe::`name` (TORCH_LIBRARY
// below), whose kernel is the calling function itself: the tracer records operators that pass
// the dispatcher.  Of a plain call it would see the allocations only and record a graph that
// returns unwritten memory.
template <class Result, class... Args>
Result call_recorded(const char* name, Args... args) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Result(Args...)>().call(
      std::forward<Args>(args)...);
}

// A tensor that a backward hands to kernels by pointer, as the forward saved it.  A saved-tensor hook
// may have put any other in its place: one on the host, of another type or shorter would be read
// past its end on the device.  `packed`: contiguous and on a 16-byte boundary.
const Tensor& as_saved(const Tensor& t, const char* name, const at::Device& dev, at::ScalarType type,
                       at::IntArrayRef sizes, bool packed = true) {
  TORCH_CHECK(t.defined() && t.device() == dev && t.scalar_type() == type && t.sizes() == sizes &&
                  (!packed || (t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0)),
              "backward: the saved tensor ", name, " came back from its hook as something else than ", type, " ", sizes,
              " on ", dev, packed ? ", contiguous" : "");
  return t;
}

// ---- experts -----------------------------------------------------------------------------------
// What the index build leaves for the rest of the forward and for the backward, in one allocation:
// [cumsums N+1 | idx Msum | inv Msum | tile table | table of tiles of at most 256 rows], every part
// on a 16-byte boundary.  The parts are found again from the sizes alone.
struct Index {
  int64_t M, N, K, tile_rows;
  bool with_rc;  // with the second table; the first one is then of the library's choice
  int64_t off_idx, off_inv, off_table, off_rc, ints;
  Index(int64_t M_, int64_t N_, int64_t K_, int64_t tile_rows_, bool with_rc_)
      : M(M_), N(N_), K(K_), tile_rows(tile_rows_), with_rc(with_rc_) {
    auto up = [](int64_t n) { return (n + 3) & ~(int64_t)3; };
    off_idx = up(N + 1);
    off_inv = off_idx + up(M * K);
    off_table = off_inv + up(M * K);
    off_rc = off_table + up(momoe_tile_table_ints(M, N, K, (int)tile_rows));
    ints = off_rc + (with_rc ? up(momoe_tile_table_ints(M, N, K, MOMOE_RECOMPUTE_TILE_ROWS)) : 0);
  }
  int32_t* base = nullptr;
  int32_t* cumsums() const { return base; }
  int32_t* idx() const { return base + off_idx; }
  int32_t* inv() const { return base + off_inv; }
  int32_t* table() const { return base + off_table; }
  int32_t* table_rc() const { return with_rc ? base + off_rc : nullptr; }
  // the one that suits a GEMM of `cols` output columns
  int32_t* table_for(int64_t cols, int64_t contraction) const {
    return with_rc && momoe_gemm_tile_rows(M * K, N, cols, contraction) != 0 ? table_rc() : table();
  }
};

struct Forward {
  Tensor y, sizes;                     // results
  Tensor x, W1, W2, s, index, ab_save; // for the backward
};

Forward experts_forward(const Tensor& x_BSD, const Tensor& Wl1, const Tensor& Wl2, const Tensor& mask_NM,
                        const Tensor& s_NM, int64_t K, int64_t msave, bool want_rc, int64_t tile_rows,
                        bool check) {
  const at::Device dev = Wl1.device();
  const int64_t B = x_BSD.size(0), S = x_BSD.size(1), D = x_BSD.size(2), M = B * S;
  const int64_t N = Wl1.size(0), H = Wl1.size(2) / 2, msum = M * K;
  const c10::DeviceGuard guard(dev);
  const hipStream_t st = stream_of(dev);
  Forward f;
  f.x = x_BSD.reshape({M, D}).to(dev, at::kBFloat16).contiguous();
  f.W1 = Wl1.to(at::kBFloat16).contiguous();
  f.W2 = Wl2.to(at::kBFloat16).contiguous();
  const Tensor mask = mask_NM.to(dev, at::kInt);
  f.s = s_NM.to(dev, at::kFloat);
  TORCH_CHECK(mask.dim() == 2 && mask.size(0) == N && mask.size(1) == M, "mask_NM must be [", N, ", ", M, "]");
  TORCH_CHECK(f.s.dim() == 2 && f.s.size(0) == N && f.s.size(1) == M, "s_NM must be [", N, ", ", M, "]");

  Index ib(M, N, K, tile_rows, want_rc);
  f.index = empty_i32(ib.ints, dev);
  ib.base = f.index.data_ptr<int32_t>();
  f.sizes = at::empty({N}, at::TensorOptions().dtype(at::kLong).device(dev));
  const int64_t ws_bytes = momoe_index_workspace_bytes(M, N);
  // only the build itself needs these: its panel counts, the slot of every pair, and the counter
  // of tokens with another number of experts than K, which starts from zero if it is to be read
  const int64_t scratch_bytes = (4 + ((msum + 3) & ~(int64_t)3) + (ws_bytes + 3) / 4) * 4;
  Transients transients(dev, {scratch_bytes, msum * H * 2, msum * D * 2});
  Tensor counter, scratch, h_own, ys_own;
  int32_t* const build = (int32_t*)transients.take(scratch_bytes, scratch);
  int32_t* violations = build;
  if (check) {
    counter = at::zeros({4}, at::TensorOptions().dtype(at::kInt).device(dev));
    violations = counter.data_ptr<int32_t>();
  }
  MOMOE_CALL(momoe_index_build, st, mask.data_ptr<int32_t>(), mask.stride(0), mask.stride(1), M, N, K,
             f.sizes.data_ptr<int64_t>(), ib.cumsums(), ib.idx(), build + 4, ib.inv(), ib.table(),
             (int)tile_rows, ib.table_rc(), (void*)(build + 4 + ((msum + 3) & ~(int64_t)3)), ws_bytes,
             violations);

  if (msave > 0) f.ab_save = empty_bf16({msave, 2 * H}, dev);
  // h in blocks of 32 hidden columns, [H/32][Msum][32]: the layout the down projection reads
  void* const h = transients.take(msum * H * 2, h_own);
  MOMOE_CALL(momoe_lin1_swiglu_fwd, st, f.x.data_ptr(), f.W1.data_ptr(), ib.idx(), ib.table_for(2 * H, D), h,
             msave > 0 ? f.ab_save.data_ptr() : nullptr, (int64_t)0, msave, M, D, H, N, msum);
  void* const ys = transients.take(msum * D * 2, ys_own);
  MOMOE_CALL(momoe_lin2_scale_fwd, st, h, f.W2.data_ptr(), f.s.data_ptr<float>(), f.s.stride(0),
             f.s.stride(1), ib.idx(), ib.table_for(D, H), ys, M, D, H, N, msum);
  h_own.reset();
  f.y = empty_bf16({B, S, D}, dev);
  MOMOE_CALL(momoe_combine, st, ys, ib.inv(), f.y.data_ptr(), M, D, K, msum);
  if (check) {
    const int v = counter.narrow(0, 0, 1).item<int32_t>();
    TORCH_CHECK(v == 0, "mask_NM: ", v, " tokens do not have exactly K = ", K,
                " experts (or the mask holds more than M*K pairs)");
  }
  if (x_BSD.device() != dev) f.y = f.y.to(x_BSD.device());
  return f;
}

// Tile height left to the library (tile_rows = 0): one table of 256 rows if that suits all these GEMMs (output
// columns, contraction), else the library's choice, and that one next to it if any wants it.
void choose_tables(std::initializer_list<std::pair<int64_t, int64_t>> gemms, int64_t msum, int64_t N, int64_t& tile_rows,
                   bool& with_rc) {
  if (tile_rows != 0) {
    with_rc = false;
    return;
  }
  bool all = true;
  for (const auto& g : gemms) {
    const bool short_tiles = momoe_gemm_tile_rows(msum, N, g.first, g.second) != 0;
    all = all && short_tiles;
    with_rc = with_rc || short_tiles;
  }
  if (!all) return;
  tile_rows = MOMOE_RECOMPUTE_TILE_ROWS;
  with_rc = false;
}

struct ExpertsFn : torch::autograd::Function<ExpertsFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& W1, const Tensor& W2,
                               const Tensor& mask, const Tensor& s, int64_t K, int64_t msave, int64_t tile_rows,
                               bool check) {
    // the recomputing GEMM's tiles have at most 256 rows
    bool want_rc = msave < x.size(0) * x.size(1) * K;
    const int64_t D = W1.size(1), H = W2.size(1);
    choose_tables({{2 * H, D}, {D, H}, {H, D}, {D, 2 * H}}, x.size(0) * x.size(1) * K, W1.size(0), tile_rows, want_rc);
    Forward f = experts_forward(x, W1, W2, mask, s, K, msave, want_rc, tile_rows, check);
    // (one entry: each takes the host 0.3 us to make and 0.2 to find)
    ctx->saved_data["call"] = std::vector<int64_t>{K, msave, tile_rows, want_rc, f.W1.device().index(), f.W1.size(1), f.W2.size(0), f.W2.size(1)};
    ctx->save_for_backward({f.x, f.s, f.W1, f.W2, f.index, f.ab_save});
    ctx->mark_non_differentiable({f.sizes});
    ctx->set_materialize_grads(false);
    return {f.y, f.sizes};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const std::vector<int64_t> call_of = ctx->saved_data["call"].toIntVector();
    const int64_t K = call_of[0], msave = call_of[1], tile_rows = call_of[2], D = call_of[5], N = call_of[6], H = call_of[7];
    const bool need_x = ctx->needs_input_grad(0), need_w1 = ctx->needs_input_grad(1),
               need_w2 = ctx->needs_input_grad(2), need_s = ctx->needs_input_grad(4);
    variable_list out(9);
    if (!grads[0].defined()) return out;
    const at::Device dev(at::kCUDA, (at::DeviceIndex)call_of[4]), gdev = grads[0].device();
    const int64_t B = grads[0].size(0), S = grads[0].size(1), M = B * S, msum = M * K;
    Index ib(M, N, K, tile_rows, call_of[3] != 0);
    const variable_list saved = ctx->get_saved_variables();
    const Tensor& x = as_saved(saved[0], "x", dev, at::kBFloat16, {M, D});
    const Tensor& s = as_saved(saved[1], "s", dev, at::kFloat, {N, M}, /*packed=*/false);
    const Tensor& W1 = as_saved(saved[2], "Wl1", dev, at::kBFloat16, {N, D, 2 * H});
    const Tensor& W2 = as_saved(saved[3], "Wl2", dev, at::kBFloat16, {N, H, D});
    ib.base = as_saved(saved[4], "index", dev, at::kInt, {ib.ints}).data_ptr<int32_t>();
    const Tensor& ab_save = saved[5];
    if (msave > 0) as_saved(ab_save, "a|b", dev, at::kBFloat16, {msave, 2 * H});
    const c10::DeviceGuard guard(dev);
    const hipStream_t st = stream_of(dev);
    const Tensor Gy = grads[0].reshape({M, D}).to(dev, at::kBFloat16).contiguous();

    // dL/dh before the gate weight, in sorted order
    // few tiles and no row saved: made on the way by the launch that needs it
    const bool joined = msave == 0 && momoe_dgrad_h_lin1_bwd_fits(M, D, H, N, msum) != 0;
    const int64_t u_bytes = msum * H * 2, gz_bytes = 2 * u_bytes, hst_bytes = momoe_padded_rows(msum, N) * H * 2;
    const int64_t nparts = momoe_gs_parts(H, N, msum), parts_bytes = nparts * msum * 4, gxs_bytes = need_x ? msum * D * 2 : 0;
    // scratch for the weight gradients of experts with many rows: what the library can use, but no
    // more than u occupied (just freed, so the peak does not move)
    auto scratch_bytes = [&](bool need, int64_t X, int64_t Y) {
      return need ? std::min(u_bytes, momoe_wgrad_workspace_bytes(N, X, Y, msum)) : 0;
    };
    // small: both weight gradients and dL/dx in one launch
    const bool tail = need_w1 && need_w2 && need_x && momoe_backward_tail_fits(M, D, H, N, msum) != 0;
    const int64_t ws2_bytes = scratch_bytes(need_w2 && !tail, H, D), ws1_bytes = scratch_bytes(need_w1 && !tail, D, 2 * H);
    Transients transients(dev, {u_bytes, gz_bytes, hst_bytes, parts_bytes, ws2_bytes, ws1_bytes, gxs_bytes});
    Tensor u_own, gz_own, hst_own, parts_own;
    void* const u = transients.take(u_bytes, u_own);
    if (!joined) MOMOE_CALL(momoe_dgrad_h, st, Gy.data_ptr(), W2.data_ptr(), ib.idx(), ib.table_for(H, D), u, M, D, H, N, msum);
    // SwiGLU backward: rows with saved a|b read them; the others recompute a|b = x.Wl1 and consume
    // them straight from the GEMM's accumulators.
    // G_a|G_b in blocks of 32 columns, [2H/32][Msum][32]: the layout dL/dx contracts over
    void* const gz = transients.take(gz_bytes, gz_own);
    // s*h in groups of 32 padded sorted rows, feature-major inside a group: the layout the Wl2
    // gradient reads fastest
    void* const hst = transients.take(hst_bytes, hst_own);
    float* const gs_part = (float*)transients.take(parts_bytes, parts_own);
    if (msave > 0)
      MOMOE_CALL(momoe_swiglu_bwd_saved, st, ab_save.data_ptr(), u, s.data_ptr<float>(), s.stride(0),
                 s.stride(1), ib.idx(), ib.cumsums(), msave, gz, hst, H,
                 gs_part, nparts, M, H, N, msum);
    if (msave < msum) {
      // the recomputing GEMM takes no taller tiles: a table of its own where another height was given
      Tensor own;
      const int32_t* table_rc = ib.with_rc ? ib.table_rc() : ib.table();
      if (tile_rows != 0 && tile_rows != MOMOE_RECOMPUTE_TILE_ROWS) {
        own = empty_i32(momoe_tile_table_ints(M, N, K, MOMOE_RECOMPUTE_TILE_ROWS), dev);
        MOMOE_CALL(momoe_tile_table_build, st, ib.cumsums(), N, msum, MOMOE_RECOMPUTE_TILE_ROWS,
                   own.data_ptr<int32_t>());
        table_rc = own.data_ptr<int32_t>();
      }
      if (joined)
        MOMOE_CALL(momoe_dgrad_h_lin1_bwd, st, Gy.data_ptr(), W2.data_ptr(), x.data_ptr(), W1.data_ptr(), (const int32_t*)ib.idx(),
                   table_rc, (const float*)s.data_ptr<float>(), s.stride(0), s.stride(1), u, gz, hst, H, gs_part, nparts, M, D, H, N, msum);
      else
        call("momoe_lin1_swiglu_bwd", st, momoe_lin1_swiglu_bwd_parts, x.data_ptr(), W1.data_ptr(), ib.idx(), table_rc,
           u, s.data_ptr<float>(), s.stride(0), s.stride(1), msave, gz, hst, H,
           gs_part, nparts, M, D, H, N, msum);
    }
    u_own.reset();
    float* gs_tail = nullptr;
    if (need_s) {
      // in the layout of s, where autograd keeps it without a copy
      if (s.stride(0) == 1 && s.stride(1) == N) {
        out[4] = at::empty_strided({N, M}, {1, N}, at::TensorOptions().dtype(at::kFloat).device(dev));
        if (tail)
          gs_tail = out[4].data_ptr<float>();
        else
          call("momoe_gs_scatter", st, momoe_gs_scatter_tokens, gs_part, nparts, (const int32_t*)ib.idx(),
               (const int32_t*)ib.cumsums(), out[4].data_ptr<float>(), M, N, msum);
      } else {
        out[4] = empty_f32({N, M}, dev);
        MOMOE_CALL(momoe_gs_scatter, st, gs_part, nparts, ib.idx(), ib.cumsums(),
                   out[4].data_ptr<float>(), M, N, msum);
      }
    }
    if (!tail) parts_own.reset();
    // (what the joined launch reads and writes is all there at once: the peak is the weight gradients, gz, s*h, the partial sums and
    // gxs, where one launch after the other has dL/dx in the place of s*h: 11.6 MiB more at 700 tokens, D = 2048, H = 768, N = 128,
    // K = 8, and always less than the 64 MiB of momoe_backward_tail_fits)
    if (need_w2) out[2] = at::empty_like(W2);
    if (need_w1 && tail) out[1] = at::empty_like(W1);
    Tensor gxs_own;
    void* gxs = nullptr;
    if (tail) {
      gxs = transients.take(gxs_bytes, gxs_own);
      MOMOE_CALL(momoe_backward_tail, st, hst, H, Gy.data_ptr(), x.data_ptr(), gz, W1.data_ptr(), (const int32_t*)ib.idx(),
                 (const int32_t*)ib.cumsums(), (const int32_t*)ib.table_for(D, 2 * H), out[2].data_ptr(), out[1].data_ptr(), gxs,
                 (const float*)gs_part, nparts, gs_tail, M, D, H, N, msum);
      parts_own.reset();
      gz_own.reset();
    }
    if (need_w2 && !tail) {
      Tensor ws_own;
      void* const ws = ws2_bytes > 0 ? transients.take(ws2_bytes, ws_own) : nullptr;
      MOMOE_CALL(momoe_wgrad, st, hst, H, MOMOE_LAYOUT_TRANSPOSED, (const int32_t*)nullptr, Gy.data_ptr(),
                 D, MOMOE_LAYOUT_ROWS, (const int32_t*)ib.idx(), ib.cumsums(), out[2].data_ptr(), M, N, H, D, msum,
                 ws, ws2_bytes);
    }
    hst_own.reset();
    if (need_w1 && !tail) {
      out[1] = at::empty_like(W1);
      Tensor ws_own;
      void* const ws = ws1_bytes > 0 ? transients.take(ws1_bytes, ws_own) : nullptr;
      MOMOE_CALL(momoe_wgrad, st, x.data_ptr(), D, MOMOE_LAYOUT_ROWS, (const int32_t*)ib.idx(), gz, msum,
                 MOMOE_LAYOUT_KBLOCKED, (const int32_t*)nullptr, ib.cumsums(), out[1].data_ptr(), M, N, D, 2 * H, msum,
                 ws, ws1_bytes);
    }
    if (need_x) {
      if (!tail) {
        gxs = transients.take(gxs_bytes, gxs_own);
        MOMOE_CALL(momoe_dgrad_x, st, gz, W1.data_ptr(), ib.table_for(D, 2 * H), gxs, M, D, H, N, msum);
      }
      Tensor Gx = empty_bf16({B, S, D}, dev);
      MOMOE_CALL(momoe_combine, st, gxs, ib.inv(), Gx.data_ptr(), M, D, K, msum);
      out[0] = gdev == dev ? Gx : Gx.to(gdev);
    }
    return out;
  }
};

std::tuple<Tensor, Tensor> experts(const Tensor& x, const Tensor& W1, const Tensor& W2, const Tensor& mask,
                                   const Tensor& s, int64_t K, double save_percent, int64_t tile_rows, bool check) {
  if (torch::jit::tracer::isTracing())
    return call_recorded<std::tuple<Tensor, Tensor>, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                         const Tensor&, int64_t, double, int64_t, bool>("momoe::experts", x, W1, W2, mask, s, K,
                                                                        save_percent, tile_rows, check);
  if (W1.device() != W2.device())
    throw_python(PyExc_AssertionError, "All weights must be on the same device, but got: Wl1_ND2H.device = " +
                                    W1.device().str() + ", Wl2_NHD.device = " + W2.device().str());
  TORCH_CHECK(W1.is_cuda(), "MoMoE weights must live on the GPU: there is no CPU compute path");
  if (x.dim() != 3 || W1.dim() != 3 || W2.dim() != 3 || W1.size(1) != x.size(2) || W2.size(0) != W1.size(0) ||
      W2.size(1) != W1.size(2) / 2 || W2.size(2) != x.size(2))
    throw_python(PyExc_AssertionError, "x_BSD [B,S,D], Wl1_ND2H [N,D,2H] and Wl2_NHD [N,H,D] do not fit together");
  const int64_t msum = x.size(0) * x.size(1) * K;
  if (!wants_autograd({&x, &W1, &W2, &s})) {  // nothing is kept for a backward that cannot happen
    bool with_rc = false;
    choose_tables({{2 * W2.size(1), W1.size(1)}, {W1.size(1), W2.size(1)}}, msum, W1.size(0), tile_rows, with_rc);
    Forward f = experts_forward(x, W1, W2, mask, s, K, 0, with_rc, tile_rows, check);
    return {f.y, f.sizes};
  }
  // the Wl1 gradient addresses the eight 32-column blocks of a gz tile with 32-bit byte offsets
  // (momoe_wgrad, k-blocked operand): say so now rather than in the backward
  TORCH_CHECK(!W1.requires_grad() || 8 * msum * 64 < (1ll << 32),
              "MoMoE backward supports fewer than 8388608 (token, expert) pairs per call, got ", msum,
              ": split the batch");
  const int64_t msave = (int64_t)((double)msum * save_percent / 100.0);  // momoe/momoe.py:251
  variable_list r = ExpertsFn::apply(x, W1, W2, mask, s, K, msave, tile_rows, check);
  return {r[0], r[1]};
}

// ---- router ------------------------------------------------------------------------------------
struct Routed {
  Tensor x_MD, mask, s_MN, p_sel, norms;
};
Routed router_forward(const Tensor& x_BSD, const Tensor& Wg, const Tensor& biases, int64_t N, int64_t K, int64_t Ks) {
  const at::Device dev = Wg.device();
  const int64_t D = x_BSD.size(2), M = x_BSD.size(0) * x_BSD.size(1);
  const c10::DeviceGuard guard(dev);
  Routed r;
  r.x_MD = x_BSD.reshape({M, D}).to(dev, at::kBFloat16);
  // Few tokens: the product in the library's kernel, whose launch alone takes the host 18 us
  const int64_t ws_bytes = momoe_gate_router_workspace_bytes(M, D, N);
  const auto aligned = [](const Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; };
  const bool own = ws_bytes >= 0 && !at::autocast::is_autocast_enabled(at::kCUDA) && Wg.dim() == 2 && Wg.size(0) == D &&
                   Wg.size(1) == N && Wg.is_contiguous() && aligned(Wg) && aligned(r.x_MD) && r.x_MD.stride(1) == 1 &&
                   r.x_MD.stride(0) >= D && r.x_MD.stride(0) % 8 == 0;
  // Other products come first of all: the GPU has work while the host allocates
  Tensor logits;
  if (!own) {
    // autocast may give the product another type than its operands'; the kernel reads two of them
    logits = at::mm(r.x_MD, Wg).contiguous();
    if (logits.scalar_type() != at::kBFloat16 && logits.scalar_type() != at::kFloat)
      throw_python(PyExc_AssertionError, std::string("the gate logits must be bfloat16 or float32, got ") +
                                             c10::toString(logits.scalar_type()));
    TORCH_CHECK(logits.size(1) == N, "Wg_DN must have N = ", N, " columns");
  }
  const Tensor bias = biases.to(dev, at::kFloat).contiguous();
  TORCH_CHECK(bias.numel() == N, "biases_N must have N = ", N, " elements");
  r.mask = at::empty({N, M}, at::TensorOptions().dtype(at::kInt).device(dev));
  r.s_MN = empty_f32({M, N}, dev);
  r.p_sel = empty_f32({M, N}, dev);
  r.norms = empty_f32({2, M}, dev);  // per token: sum over the selected, over the shared experts
  float* norms = r.norms.data_ptr<float>();
  const hipStream_t st = stream_of(dev);
  if (own) {
    const Tensor ws = empty_f32({ws_bytes / 4}, dev);
    MOMOE_CALL(momoe_gate_router_fwd, st, r.x_MD.data_ptr(), r.x_MD.stride(0), Wg.data_ptr(), bias.data_ptr<float>(), M, D, N, K,
               Ks, r.mask.data_ptr<int32_t>(), r.s_MN.data_ptr<float>(), r.p_sel.data_ptr<float>(), norms, norms + M,
               ws.data_ptr(), ws_bytes);
    return r;
  }
  MOMOE_CALL(momoe_router_fwd, st, logits.data_ptr(), logits.scalar_type() == at::kFloat, bias.data_ptr<float>(), M, N, K, Ks,
             r.mask.data_ptr<int32_t>(), r.s_MN.data_ptr<float>(), r.p_sel.data_ptr<float>(), norms, norms + M);
  return r;
}

// x^T . G_logits [D, N].  (The library's product has few tiles and one long contraction for each, and takes the host 18 us where
// two launches take 8: 300 tokens, D = 512, N = 64 9.0 us of the GPU against 9.6; 1024, 1024, 32 9.3, 8.9; 2000, 1120, 48 19.6, 9.4;
// 8192, 2048, 128 60, 22.)  The own kernel's partial sums are D * N at the least, written and read for each range of tokens:
// it takes more than 2^18 results only from a token for 1024 of them on, and up to 2^20, where the library's tiles
// fill the chip.  Us, 300 tokens, D = 2048, N = 128 10.3, 11.6; 1000, 2048, 256 14.7, 15.9; 4096, 2048, 256 29.9, 21.3;
// 4096, 2048, 512 31.3, 30.3; past the line 300, 2048, 256 9.2, 12.8; 1000, 2048, 512 15.4, 21.9; 4096, 4096, 512 38.5, 47.1; 8192,
// 8192, 512 91, 147 (though 32768, 4096, 512 302, 276).  And the library's where autograd records it.
Tensor gate_gradient(const Tensor& x, const Tensor& G_logit) {
  const int64_t M = x.size(0), D = x.size(1), N = G_logit.size(1);
  const int64_t bytes = momoe_gate_wgrad_workspace_bytes(M, D, N);
  const bool sizes = bytes >= 0 && (D * N <= 1 << 18 || (D * N <= 1 << 20 && D * N <= 1024 * M));
  const bool rows = x.stride(1) == 1 && x.stride(0) >= D && x.stride(0) % 8 == 0 && (uintptr_t)x.data_ptr() % 16 == 0;
  if (!sizes || !rows || at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA)) return at::mm(x.t(), G_logit);
  const Tensor out = empty_bf16({D, N}, x.device()), ws = empty_f32({bytes / 4}, x.device());
  MOMOE_CALL(momoe_gate_wgrad, stream_of(x.device()), x.data_ptr(), x.stride(0), G_logit.data_ptr(), out.data_ptr(), M, D, N,
             ws.data_ptr(), bytes);
  return out;
}

// G_x + G_logits . Wg^T [M, D]; G_x may be undefined.  (The library copies G_x in front of its product, and takes the host 14 us
// more.)  The own kernel reloads both operands for every 32 experts and waits for each: with more than 128 experts it takes
// products of up to 2^31 terms.  In a graph, us, the library's -> own: 8192 tokens, D = 2048, N = 128 32.4 -> 26.1; 32768, 4096, 128
// 232 -> 198; 1000, 1024, 256 9.9 -> 12.3; 8192, 1024, 256 25.8 -> 22.9; 4096, 1024, 512 20.4 -> 20.8; 1000, 2048, 512 14.2 -> 19.7;
// past the line 4096, 2048, 512 29.7 -> 36.6; 8192, 2048, 256 35.3 -> 39.7; 32768, 4096, 512 299 -> 511.
Tensor gate_input_gradient(const Tensor& G_x, const Tensor& G_logit, const Tensor& Wg) {
  const int64_t M = G_logit.size(0), N = G_logit.size(1), D = Wg.size(0);
  const auto packed = [](const Tensor& t) { return t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0; };
  const bool sizes = momoe_gate_wgrad_workspace_bytes(M, D, N) >= 0 && M < 65535 * 128 && (N <= 128 || M * D * N <= (1ll << 31));
  if (!sizes || !packed(Wg) || (G_x.defined() && !packed(G_x)) || at::GradMode::is_enabled() ||
      at::autocast::is_autocast_enabled(at::kCUDA))
    return G_x.defined() ? at::addmm(G_x, G_logit, Wg.t()) : at::mm(G_logit, Wg.t());
  const Tensor out = empty_bf16({M, D}, G_logit.device());
  MOMOE_CALL(momoe_gate_dgrad, stream_of(G_logit.device()), G_logit.data_ptr(), Wg.data_ptr(),
             G_x.defined() ? (const void*)G_x.data_ptr() : nullptr, out.data_ptr(), M, D, N);
  return out;
}

struct RouterFn : torch::autograd::Function<RouterFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& Wg, const Tensor& biases,
                               int64_t N, int64_t K, int64_t Ks) {
    Routed r = router_forward(x, Wg, biases, N, K, Ks);
    ctx->save_for_backward({r.x_MD, Wg, r.mask, r.p_sel, r.s_MN, r.norms});
    ctx->saved_data["call"] = std::vector<int64_t>{Ks, N, Wg.device().index(), x.size(0), x.size(1), x.size(2)};
    ctx->mark_non_differentiable({r.mask});
    ctx->set_materialize_grads(false);
    return {x, r.mask, r.s_MN.t()};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const std::vector<int64_t> call_of = ctx->saved_data["call"].toIntVector();
    const at::Device dev(at::kCUDA, (at::DeviceIndex)call_of[2]);
    const int64_t Ks = call_of[0], N = call_of[1], M = call_of[3] * call_of[4], D = call_of[5];
    const Tensor& x = as_saved(saved[0], "x", dev, at::kBFloat16, {M, D}, /*packed=*/false);
    const Tensor& Wg = as_saved(saved[1], "Wg", dev, at::kBFloat16, {D, N}, /*packed=*/false);
    const Tensor& mask = as_saved(saved[2], "mask", dev, at::kInt, {N, M});
    const Tensor& p_sel = as_saved(saved[3], "p", dev, at::kFloat, {M, N});
    const Tensor& s_MN = as_saved(saved[4], "s", dev, at::kFloat, {M, N});
    const Tensor& norms = as_saved(saved[5], "norms", dev, at::kFloat, {2, M});
    const bool need_x = ctx->needs_input_grad(0), need_wg = ctx->needs_input_grad(1);
    const c10::DeviceGuard guard(dev);
    variable_list out(6);
    const Tensor &G_x_BSD = grads[0], &G_s_NM = grads[2];
    Tensor G_x;
    if (G_x_BSD.defined()) G_x = G_x_BSD.reshape({M, D}).to(dev, at::kBFloat16);
    if (G_s_NM.defined()) {
      const Tensor G_s = G_s_NM.to(dev, at::kFloat);
      const Tensor G_logit = empty_bf16({M, N}, dev);
      const float* nrm = norms.data_ptr<float>();
      MOMOE_CALL(momoe_router_bwd, stream_of(dev), G_s.data_ptr<float>(), G_s.stride(0), G_s.stride(1),
                 p_sel.data_ptr<float>(), s_MN.data_ptr<float>(), nrm, nrm + M, mask.data_ptr<int32_t>(), M, N,
                 Ks, G_logit.data_ptr());
      if (need_x) G_x = gate_input_gradient(G_x, G_logit, Wg);
      if (need_wg) out[1] = gate_gradient(x, G_logit);
    } else if (need_wg) {
      out[1] = at::zeros_like(Wg);
    }
    if (need_x && G_x.defined()) out[0] = G_x.reshape({call_of[3], call_of[4], D});
    return out;
  }
};

std::tuple<Tensor, Tensor, Tensor> router(const Tensor& x, const Tensor& Wg, const Tensor& biases, int64_t N, int64_t K,
                                          int64_t Ks) {
  if (torch::jit::tracer::isTracing())
    return call_recorded<std::tuple<Tensor, Tensor, Tensor>, const Tensor&, const Tensor&, const Tensor&, int64_t,
                         int64_t, int64_t>("momoe::router", x, Wg, biases, N, K, Ks);
  if (Wg.scalar_type() != at::kBFloat16) throw_python(PyExc_AssertionError, "Wg_DN must be of type torch.bfloat16");
  TORCH_CHECK(Wg.is_cuda(), "TopKRouter weights must live on the GPU: there is no CPU compute path");
  TORCH_CHECK(x.dim() == 3, "x_BSD must be [B, S, D]");
  if (!wants_autograd({&x, &Wg})) {
    Routed r = router_forward(x, Wg, biases, N, K, Ks);
    return {x, r.mask, r.s_MN.t()};
  }
  variable_list r = RouterFn::apply(x, Wg, biases, N, K, Ks);
  return {r[0], r[1], r[2]};
}

// biases += rate * sign(c_avg - sizes), in place, in fp32
void bias_update(Tensor biases, const Tensor& sizes, double c_avg, double rate) {
  const c10::DeviceGuard guard(biases.device());
  MOMOE_CALL(momoe_bias_update, stream_of(biases.device()), sizes.data_ptr<int64_t>(), (float)c_avg, (float)rate,
             biases.numel(), biases.data_ptr<float>());
  biases.unsafeGetTensorImpl()->bump_version();
}

}  // namespace

// The operators of a traced call.  A graph keeps the integers and flags it was traced with, the sizes
// are those of the tensors it is run on.
TORCH_LIBRARY(momoe, m) {
  m.def("experts(Tensor x_BSD, Tensor Wl1_ND2H, Tensor Wl2_NHD, Tensor mask_NM, Tensor s_NM, int K, "
        "float save_percent, int tile_rows, bool check) -> (Tensor, Tensor)",
        torch::dispatch(c10::DispatchKey::CompositeImplicitAutograd, TORCH_FN(experts)));
  m.def("router(Tensor(a) x_BSD, Tensor Wg_DN, Tensor biases_N, int N, int K, int Ks) -> (Tensor(a), Tensor, Tensor)",
        torch::dispatch(c10::DispatchKey::CompositeImplicitAutograd, TORCH_FN(router)));
}

PYBIND11_MODULE(_layer, m) {
  m.def("experts", &experts, py::call_guard<py::gil_scoped_release>());
  m.def("router", &router, py::call_guard<py::gil_scoped_release>());
  m.def("bias_update", &bias_update, py::call_guard<py::gil_scoped_release>());
  m.def("timing_start", &timing_start);
  m.def("timing_stop", &timing_stop);
  m.def("timing_take", &timing_take);
  // a library call made from Python, recorded like those made here
  m.def("timed", [](const std::string& name, uintptr_t stream, const py::function& fn) {
    return timed(name.c_str(), (hipStream_t)stream, [&] { return py::object(fn()); });
  });
}
