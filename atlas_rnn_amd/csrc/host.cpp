// host.cpp - the host path of the package in native code: argument checks, allocations, the calls into
// libatlas_mem.so and the autograd nodes, as the extension module atlas_rnn_amd._host.
//
// Why: a pass over a small or medium problem was bound by the host, not by its kernels. The Python
// path (operand checks, ctypes structures and one Python autograd node per operator, whose backward
// takes the interpreter lock on the engine's thread) issued a decode step in 29 us against 4.6 us of
// kernel, a training step in 155 - 260 us against 100 of kernels and a cell step in 760 - 1040 us
// against 695.
//
// Every function here takes what the kernels take and returns None for anything else (other shapes,
// devices or types): the Python callers then pad, split or raise. The nodes keep their tensors with
// save_for_backward (saved-tensor hooks and version checks apply) and refuse functorch transforms and
// forward-mode differentiation, as autograd functions without those rules do. torch.jit.trace cannot see
// into them: functional._native records a call as a Python node, and an entry reached by the trace itself
// raises (it would be recorded as the allocation of its outputs).
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <dlfcn.h>

#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/atlas_mem.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
typedef std::optional<Tensor> OptTensor;

// ---------------------------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------------------------
// libatlas_mem.so's entry points, looked up in the library that the Python package has loaded (bind): one
// library serves both, also where a program has chosen another file than the one beside this module.
#define ATLAS_LIBRARY(X) \
  X(atlas_block_merge) X(atlas_block_parts) X(atlas_block_split) X(atlas_heads_bwd) X(atlas_heads_fwd) \
  X(atlas_linear_batch) X(atlas_linear_wgrad_batch) X(atlas_linear_wgrad_batch_workspace_bytes) X(atlas_mem_bwd) \
  X(atlas_mem_bwd_workspace_bytes) X(atlas_mem_fwd) X(atlas_mem_infer) X(atlas_mem_saved_bytes) X(atlas_mem_step) \
  X(atlas_mem_strerror) X(atlas_mem_validate) X(atlas_omega_chain_bwd) X(atlas_omega_chain_fwd_keep) \
  X(atlas_omega_chain_workspace_bytes) X(atlas_partials_sum) X(atlas_prologue_bwd) X(atlas_prologue_fwd) \
  X(atlas_prologue_num_workgroups) X(atlas_replicas) X(atlas_tensor_map_bwd_sym) X(atlas_tensor_map_fwd_sym) \
  X(atlas_tensor_map_symmetrize)
struct Library {
#define ATLAS_FIELD(name) decltype(&::name) name;
  ATLAS_LIBRARY(ATLAS_FIELD)
#undef ATLAS_FIELD
  std::string path;
};
std::atomic<const Library*> bound{nullptr};

void bind(const std::string& path) {
  static std::mutex mu;
  static std::map<std::string, Library> known;   // never dropped: a backward may still be running on one
  std::lock_guard<std::mutex> lk(mu);
  auto it = known.find(path);
  if (it == known.end()) {
    void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(h, "cannot load ", path, ": ", dlerror());
    Library l{};
#define ATLAS_FIND(name)                                        \
  l.name = reinterpret_cast<decltype(&::name)>(dlsym(h, #name)); \
  TORCH_CHECK(l.name, path, " has no " #name);
    ATLAS_LIBRARY(ATLAS_FIND)
#undef ATLAS_FIND
    l.path = path;
    it = known.emplace(path, std::move(l)).first;
  }
  bound.store(&it->second, std::memory_order_release);
}
const Library& lib() {
  const Library* l = bound.load(std::memory_order_acquire);
  TORCH_CHECK(l, "no library is bound: call through atlas_rnn_amd");
  return *l;
}

void check(int status, const char* what) {
  TORCH_CHECK(status == ATLAS_MEM_OK, what, " failed: ", lib().atlas_mem_strerror(status), " (status ", status, ")");
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool kernel_dtype(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }
int dt_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? ATLAS_DT_BF16 : ATLAS_DT_F32; }

// a tensor's address as the kernels' argument types (null: absent)
struct CPtr {
  const void* p;
  operator const void*() const { return p; }
  operator const float*() const { return static_cast<const float*>(p); }
};
struct MPtr {
  void* p;
  operator void*() const { return p; }
  operator float*() const { return static_cast<float*>(p); }
};
CPtr ptr(const Tensor& t) { return {t.defined() ? t.const_data_ptr() : nullptr}; }
MPtr mptr(const Tensor& t) { return {t.defined() ? t.mutable_data_ptr() : nullptr}; }
const float* fptr(const Tensor& t) { return ptr(t); }
float* mfptr(const Tensor& t) { return mptr(t); }

Tensor get(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }

// contiguous with a 16-byte aligned start (the C ABI rejects other pointers)
Tensor aligned(const Tensor& t) {
  if (!t.defined()) return t;
  Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.const_data_ptr()) % 16 == 0 ? c : c.clone();
}
Tensor canon(const Tensor& t, at::ScalarType dt) {
  if (!t.defined()) return t;
  return aligned(t.scalar_type() == dt ? t : t.to(dt));
}
Tensor like(const Tensor& t) { return t.defined() ? at::empty(t.sizes(), t.options().requires_grad(false)) : Tensor(); }
Tensor f32(const Tensor& ref, at::IntArrayRef sizes) {
  return at::empty(sizes, ref.options().dtype(at::kFloat).requires_grad(false));
}
Tensor plain(const Tensor& ref, at::IntArrayRef sizes) { return at::empty(sizes, ref.options().requires_grad(false)); }
// a workspace of at least `bytes` bytes, as fp32
Tensor scratch(const Tensor& ref, int64_t bytes) { return f32(ref, {(std::max<int64_t>(bytes, 16) + 3) / 4}); }

// ---------------------------------------------------------------------------------------------
// the recurrence (atlas_pytorch/rnn_memory.py:300-406, :605-730)
// ---------------------------------------------------------------------------------------------
struct RecOut {
  Tensor y, S_T, Z_T, buf;
};

atlas_mem_fwd_args fwd_args(const Tensor& k, const Tensor& q, const Tensor& v, const Tensor& lr, const Tensor& decay,
                            const Tensor& beta, const Tensor& gate, const Tensor& S_ref, const Tensor& S0,
                            const Tensor& Z0, const Tensor& buf, const RecOut& o) {
  atlas_mem_fwd_args a{};
  a.k = ptr(k); a.q = ptr(q); a.v = ptr(v); a.lr = ptr(lr); a.decay = ptr(decay); a.beta = ptr(beta);
  a.gate = ptr(gate); a.S_ref = fptr(S_ref); a.S0 = fptr(S0); a.Z0 = fptr(Z0); a.buffer_in = fptr(buf);
  a.y = mptr(o.y); a.S_T = mfptr(o.S_T); a.Z_T = mfptr(o.Z_T); a.buffer_out = mfptr(o.buf);
  return a;
}

RecOut rec_outputs(const atlas_mem_problem& p, const Tensor& k) {
  RecOut o;
  o.y = plain(k, {p.bh, p.seq_len, p.d_v});
  o.S_T = f32(k, {p.bh, p.d_v, p.d_k});
  if (p.momentum) o.Z_T = f32(k, {p.bh, p.d_v, p.d_k});
  if (p.window > 1) o.buf = f32(k, {p.bh, p.window - 1, p.d_v, p.d_k});
  return o;
}

// y, S_T, [Z_T], [buffer_out] = recurrence(...): every tensor canonical (contiguous, 16-byte aligned, the
// operands of one dtype, the states fp32)
struct RecurrenceFn : public Function<RecurrenceFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& k, const Tensor& q, const Tensor& v, const Tensor& lr,
                               const Tensor& decay, const OptTensor& beta, const OptTensor& gate, const Tensor& S_ref,
                               const Tensor& S0, const OptTensor& Z0, const OptTensor& buf,
                               const atlas_mem_problem& prob, bool infer) {
    // outputs a loss does not use get no gradient tensor (a missing one counts as zero)
    ctx->set_materialize_grads(false);
    const RecOut o = rec_outputs(prob, k);
    const Tensor saved = scratch(k, (int64_t)lib().atlas_mem_saved_bytes(&prob));
    const atlas_mem_fwd_args a = fwd_args(k, q, v, lr, decay, get(beta), get(gate), S_ref, S0, get(Z0), get(buf), o);
    if (infer) {   // no input asks for a gradient: nothing for a backward is formed or kept
      check(lib().atlas_mem_infer(&prob, &a, mfptr(saved), stream_of(k)), "atlas_mem_fwd");
      variable_list out{o.y, o.S_T};
      if (o.Z_T.defined()) out.push_back(o.Z_T);
      if (o.buf.defined()) out.push_back(o.buf);
      return out;
    }
    check(lib().atlas_mem_fwd(&prob, &a, mfptr(saved), stream_of(k)), "atlas_mem_fwd");
    ctx->save_for_backward({k, q, v, lr, decay, get(beta), get(gate), S_ref, S0, get(Z0), get(buf), saved});
    ctx->saved_data["prob"] = std::string(reinterpret_cast<const char*>(&prob), sizeof(prob));
    variable_list out{o.y, o.S_T};
    if (o.Z_T.defined()) out.push_back(o.Z_T);
    if (o.buf.defined()) out.push_back(o.buf);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const variable_list s = ctx->get_saved_variables();
    const std::string& bytes = ctx->saved_data["prob"].toStringRef();
    atlas_mem_problem prob;
    std::memcpy(&prob, bytes.data(), sizeof(prob));
    const Tensor &k = s[0], &q = s[1], &v = s[2], &lr = s[3], &decay = s[4], &beta = s[5], &gate = s[6], &S_ref = s[7],
                 &S0 = s[8], &Z0 = s[9], &buf = s[10], &saved = s[11];
    c10::DeviceGuard guard(k.device());
    size_t i = 0;
    const Tensor dy = canon(g[i++], k.scalar_type()), dS_T = canon(g[i++], at::kFloat);
    const Tensor dZ_T = prob.momentum ? canon(g[i++], at::kFloat) : Tensor();
    const Tensor dbuf_out = prob.window > 1 ? canon(g[i++], at::kFloat) : Tensor();
    const Tensor dk = like(k), dq = like(q), dv = like(v), dlr = like(lr), dd = like(decay), db = like(beta),
                 dg = like(gate), dbuf = like(buf);
    const Tensor dS_ref = like(S_ref), dS0 = like(S0), dZ0 = prob.momentum ? like(S0) : Tensor();
    const size_t ws_bytes = lib().atlas_mem_bwd_workspace_bytes(&prob);
    const Tensor ws = scratch(k, (int64_t)ws_bytes);
    atlas_mem_bwd_args a{};
    a.k = ptr(k); a.q = ptr(q); a.v = ptr(v); a.lr = ptr(lr); a.decay = ptr(decay); a.beta = ptr(beta);
    a.gate = ptr(gate); a.S_ref = fptr(S_ref); a.S0 = fptr(S0); a.Z0 = fptr(Z0); a.buffer_in = fptr(buf);
    a.dy = ptr(dy); a.dS_T = fptr(dS_T); a.dZ_T = fptr(dZ_T); a.dbuffer_out = fptr(dbuf_out);
    a.dk = mptr(dk); a.dq = mptr(dq); a.dv = mptr(dv); a.dlr = mptr(dlr); a.ddecay = mptr(dd); a.dbeta = mptr(db);
    a.dgate = mptr(dg); a.dS_ref = mfptr(dS_ref); a.dS0 = mfptr(dS0); a.dZ0 = mfptr(dZ0); a.dbuffer_in = mfptr(dbuf);
    check(lib().atlas_mem_bwd(&prob, &a, fptr(saved), mptr(ws), ws_bytes, stream_of(k)), "atlas_mem_bwd");
    return {dk, dq, dv, dlr, dd, db, dg, dS_ref, dS0, Z0.defined() ? dZ0 : Tensor(), dbuf, Tensor(), Tensor()};
  }
};

bool shape_is(const Tensor& t, at::IntArrayRef want) { return !t.defined() || t.sizes() == want; }

// memory_recurrence on the kernels, or nullopt: operands they do not take as they are. map_degree > 1:
// the elementwise polynomial map.
std::optional<RecOut> recurrence_or_none(const Tensor& k, const Tensor& q, const Tensor& v, const Tensor& lr,
                                         const Tensor& decay, const Tensor& beta, const Tensor& gate, Tensor S_ref,
                                         Tensor S0, Tensor Z0, Tensor buf, int64_t window, int64_t map_degree,
                                         std::optional<int64_t> clamp_every, int64_t clamp_final) {
  if (k.dim() != 3 || v.dim() != 3 || !k.is_cuda()) return std::nullopt;
  const int64_t bh = k.size(0), T = k.size(1), dk = k.size(2), dv = v.size(2);
  if (dk != dv || (dk != 32 && dk != 64) || window < 1 || window > 64 || bh < 1 || T < 1 || bh > INT32_MAX ||
      T > INT32_MAX || map_degree < INT32_MIN || map_degree > INT32_MAX || clamp_final < 0 || clamp_final > 1)
    return std::nullopt;
  int gate_mode = ATLAS_GATE_NONE;
  if (gate.defined()) {
    if (gate.dim() != 2 && gate.dim() != 3) return std::nullopt;
    gate_mode = gate.dim() == 2 ? ATLAS_GATE_TOKEN : ATLAS_GATE_LAG;
    if (gate.dim() == 2 ? !shape_is(gate, {bh, T}) : !shape_is(gate, {bh, T, window})) return std::nullopt;
  }
  if (!shape_is(q, {bh, T, dk}) || !shape_is(v, {bh, T, dv}) || !shape_is(lr, {bh, T}) || !shape_is(decay, {bh, T}) ||
      !shape_is(beta, {bh, T}) || !shape_is(S_ref, {bh, dv, dk}) || !shape_is(S0, {bh, dv, dk}) ||
      !shape_is(Z0, {bh, dv, dk}) || (window > 1 && !shape_is(buf, {bh, window - 1, dv, dk})))
    return std::nullopt;
  for (const Tensor* t : std::initializer_list<const Tensor*>{&q, &v, &lr, &decay, &beta, &gate, &S_ref, &S0, &Z0, &buf})
    if (t->defined() && t->device() != k.device()) return std::nullopt;
  if (clamp_every.has_value() && (*clamp_every < 0 || *clamp_every > INT32_MAX)) {
    if (*clamp_every < 0) return std::nullopt;
    clamp_every = std::nullopt;   // past any T: no clamp point before the last token
  }
  if (clamp_every.has_value() && *clamp_every >= T) clamp_every = std::nullopt;
  const at::ScalarType dt = kernel_dtype(k.scalar_type()) ? k.scalar_type() : at::kFloat;
  const bool elementwise = map_degree > 1;
  atlas_mem_problem p{};
  p.abi_version = ATLAS_MEM_ABI_VERSION;
  p.bh = (int)bh; p.seq_len = (int)T; p.d_k = (int)dk; p.d_v = (int)dv; p.window = (int)window;
  p.momentum = beta.defined();
  p.gate_mode = gate_mode;
  p.map_mode = elementwise ? ATLAS_MAP_ELEMENTWISE : ATLAS_MAP_OFF;
  p.map_degree = elementwise ? (int)map_degree : 1;
  if (window == 1) buf = Tensor();
  if (!p.momentum) Z0 = Tensor();
  p.has_buffer = buf.defined();
  p.clamp_every = (int)clamp_every.value_or(0);
  p.clamp_final = (int)clamp_final;
  p.dtype = dt == at::kBFloat16 ? ATLAS_DT_BF16 : ATLAS_DT_F32;
  if (lib().atlas_mem_validate(&p) != ATLAS_MEM_OK) return std::nullopt;
  c10::DeviceGuard guard(k.device());
  const Tensor kc = canon(k, dt), qc = canon(q, dt), vc = canon(v, dt), lc = canon(lr, dt), dc = canon(decay, dt),
               bc = canon(beta, dt), gc = canon(gate, dt);
  if (!S0.defined()) S0 = at::zeros({bh, dv, dk}, k.options().dtype(at::kFloat).requires_grad(false));
  const Tensor S0c = canon(S0, at::kFloat);
  const Tensor Src = !S_ref.defined() || S_ref.is_same(S0) ? S0c : canon(S_ref, at::kFloat);
  const Tensor Zc = canon(Z0, at::kFloat), Bc = canon(buf, at::kFloat);
  RecOut o;
  bool grad = false;
  if (at::GradMode::is_enabled())
    for (const Tensor* t : {&kc, &qc, &vc, &lc, &dc, &bc, &gc, &Src, &S0c, &Zc, &Bc})
      grad = grad || (t->defined() && t->requires_grad());
  if (T == 1 && !grad) {
    bool tangent = false;   // (a forward-mode tangent: the node refuses it)
    for (const Tensor* t : {&kc, &qc, &vc, &lc, &dc, &bc, &gc, &Src, &S0c, &Zc, &Bc})
      tangent = tangent || (t->defined() && t->_fw_grad(0).defined());
    if (!tangent) {   // decode: one launch, no saved buffer (rnn_transformer.py:863-900 through the cell at T = 1)
      o = rec_outputs(p, kc);
      const atlas_mem_fwd_args a = fwd_args(kc, qc, vc, lc, dc, bc, gc, Src, S0c, Zc, Bc, o);
      check(lib().atlas_mem_step(&p, &a, stream_of(kc)), "atlas_mem_step");
      return o;
    }
  }
  const variable_list out = RecurrenceFn::apply(kc, qc, vc, lc, dc, opt(bc), opt(gc), Src, S0c, opt(Zc), opt(Bc), p,
                                                !grad);
  size_t i = 0;
  o.y = out[i++];
  o.S_T = out[i++];
  if (p.momentum) o.Z_T = out[i++];
  if (p.window > 1) o.buf = out[i++];
  return o;
}

// y, S_T, Z_T, buffer_out (None: absent)
typedef std::tuple<Tensor, Tensor, OptTensor, OptTensor> Four;

std::optional<Four> recurrence(const Tensor& k, const Tensor& q, const Tensor& v, const Tensor& lr, const Tensor& decay,
                               const OptTensor& beta, const OptTensor& gate, const OptTensor& S_ref, const OptTensor& S0,
                               const OptTensor& Z0, const OptTensor& buffer, int64_t window, int64_t map_degree,
                               std::optional<int64_t> clamp_every, int64_t clamp_final) {
  const std::optional<RecOut> o = recurrence_or_none(k, q, v, lr, decay, get(beta), get(gate), get(S_ref), get(S0), get(Z0),
                                                     get(buffer), window, map_degree, clamp_every, clamp_final);
  if (!o.has_value()) return std::nullopt;
  return Four{o->y, o->S_T, opt(o->Z_T), opt(o->buf)};
}

// ---------------------------------------------------------------------------------------------
// the tensor feature map (rnn_memory.py:125-130)
// ---------------------------------------------------------------------------------------------
std::tuple<Tensor, Tensor> symmetrized(const Tensor& proj, int64_t d, at::ScalarType dt) {
  TORCH_CHECK_VALUE(proj.dim() == 2 && d >= 1 && proj.size(0) == d + d * d, "the projection must be [d + d*d, m] for d = ", d,
                    ", got ", proj.sizes());
  const Tensor p = aligned(proj.detach().to(dt));
  const int64_t m = p.size(1);
  const Tensor ps = like(p), pst = plain(p, {m, p.size(0)});
  check(lib().atlas_tensor_map_symmetrize(dt_code(p), (int)d, (int)m, ptr(p), mptr(ps), mptr(pst), stream_of(p)),
        "atlas_tensor_map_symmetrize");
  return {ps, pst};
}

// x [n, d] -> phi [n, m] on the symmetrised tables (ps [d + d d, m], pst its transpose)
struct TensorMapFn : public Function<TensorMapFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& ps, const Tensor& pst, int64_t degree) {
    const int64_t n = x.size(0), d = x.size(1), m = ps.size(1);
    const Tensor out = plain(x, {n, m}), pre = degree > 1 ? plain(x, {n, m}) : Tensor();
    check(lib().atlas_tensor_map_fwd_sym(dt_code(x), n, (int)d, (int)m, (int)degree, ptr(x), ptr(pst), mptr(out), mptr(pre),
                                   stream_of(x)), "atlas_tensor_map_fwd_sym");
    ctx->save_for_backward({x, ps, pre});
    ctx->saved_data["degree"] = degree;
    return {out};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &ps = s[1], &pre = s[2];
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    c10::DeviceGuard guard(x.device());
    const Tensor dout = canon(g[0], x.scalar_type()), dx = like(x);
    check(lib().atlas_tensor_map_bwd_sym(dt_code(x), x.size(0), (int)x.size(1), (int)ps.size(1),
                                   (int)ctx->saved_data["degree"].toInt(), ptr(x), ptr(ps), ptr(pre), ptr(dout), mptr(dx),
                                   stream_of(x)), "atlas_tensor_map_bwd_sym");
    return {dx, Tensor(), Tensor(), Tensor()};
  }
};

// operands checked by the caller (functional.tensor_feature_map)
Tensor tensor_map(const Tensor& x, const Tensor& proj, int64_t degree, const OptTensor& ps, const OptTensor& pst) {
  c10::DeviceGuard guard(x.device());
  const int64_t d = x.size(-1), m = proj.size(-1);
  const Tensor x2 = aligned(x.dim() == 2 ? x : x.reshape({-1, d}));
  Tensor a = get(ps), b = get(pst);
  if (!a.defined()) std::tie(a, b) = symmetrized(proj, d, x.scalar_type());
  const Tensor out = TensorMapFn::apply(x2, a, b, degree)[0];
  if (x.dim() == 2) return out;
  std::vector<int64_t> sizes = x.sizes().vec();
  sizes.back() = m;
  return out.reshape(sizes);
}

// ---------------------------------------------------------------------------------------------
// 64 x 64 state blocks for head sizes above 64 or d_k != d_v (functional.block_recurrence)
// ---------------------------------------------------------------------------------------------
constexpr int64_t kBlock = 64;
enum { kReplicate = 0, kReplicaSum = 1 };

// one launch per dtype and four arrays: nrep copies stacked along the first axis, or their sum
variable_list replicas(int op, int64_t nrep, at::TensorList in) {
  TORCH_CHECK_VALUE(nrep >= 1, "the number of replicas must be at least 1, got ", nrep);
  variable_list xs, outs;
  for (const Tensor& t : in) xs.push_back(t.contiguous());
  for (const Tensor& x : xs) {
    TORCH_CHECK(x.is_cuda() && kernel_dtype(x.scalar_type()), "replicas: fp32 or bf16 GPU tensors, got ", x.scalar_type());
    TORCH_CHECK_VALUE(op == kReplicate || x.size(0) % nrep == 0, "replica sum: first axis ", x.size(0),
                      " is not a multiple of ", nrep, " replicas");
    std::vector<int64_t> sizes = x.sizes().vec();
    sizes[0] = op == kReplicate ? sizes[0] * nrep : sizes[0] / nrep;
    outs.push_back(plain(x, sizes));
  }
  for (at::ScalarType dt : {at::kBFloat16, at::kFloat}) {
    int64_t n[4];
    const void* src[4];
    void* dst[4];
    int cnt = 0;
    for (size_t i = 0; i <= xs.size(); ++i) {
      if (i < xs.size() && xs[i].scalar_type() == dt) {
        n[cnt] = (op == kReplicate ? xs[i] : outs[i]).numel();
        src[cnt] = ptr(xs[i]);
        dst[cnt++] = mptr(outs[i]);
      }
      if (cnt > 0 && (cnt == 4 || i == xs.size())) {
        check(lib().atlas_replicas(op == kReplicate ? ATLAS_REPLICATE : ATLAS_REPLICA_SUM,
                             dt == at::kBFloat16 ? ATLAS_DT_BF16 : ATLAS_DT_F32, cnt, (int)nrep, n, src, dst,
                             stream_of(xs[0])), "atlas_replicas");
        cnt = 0;
      }
    }
  }
  return outs;
}

template <int OP>
struct ReplicaFn : public Function<ReplicaFn<OP>> {
  static variable_list forward(AutogradContext* ctx, int64_t nrep, at::TensorList xs) {
    ctx->saved_data["nrep"] = nrep;
    return replicas(OP, nrep, xs);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    c10::DeviceGuard guard(g[0].device());
    variable_list out = replicas(OP == kReplicate ? kReplicaSum : kReplicate, ctx->saved_data["nrep"].toInt(), g);
    out.insert(out.begin(), Tensor());
    return out;
  }
};
variable_list replicate(int64_t nrep, const variable_list& xs) {
  return ReplicaFn<kReplicate>::apply(nrep, at::TensorList(xs));
}
variable_list replica_sum(int64_t nrep, const variable_list& xs) {
  return ReplicaFn<kReplicaSum>::apply(nrep, at::TensorList(xs));
}

// phi, psi [BH, T, Dk], v [BH, T, Dv], S_ref [BH, Dv, Dk] -> phi_b, psi_b, nv_b [NB BH, T, 64]
// with nv = v - S_ref phi, block r = (i * Dk/64 + j) * BH + bh
struct BlockSplitFn : public Function<BlockSplitFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& phi, const Tensor& psi, const Tensor& v,
                               const Tensor& S_ref) {
    ctx->set_materialize_grads(false);
    const int64_t bh = phi.size(0), T = phi.size(1), dk = phi.size(2), dv = v.size(2);
    const int64_t nb = (dk / kBlock) * (dv / kBlock);
    const Tensor a = plain(phi, {nb * bh, T, kBlock}), b = like(a), c = like(a);
    check(lib().atlas_block_split(dt_code(phi), (int)bh, (int)T, (int)dk, (int)dv, ptr(phi), ptr(psi), ptr(v), fptr(S_ref),
                            mptr(a), mptr(b), mptr(c), stream_of(phi)), "atlas_block_split");
    ctx->save_for_backward({phi, S_ref});
    ctx->saved_data["dv"] = dv;
    return {a, b, c};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &phi = s[0], &S_ref = s[1];
    c10::DeviceGuard guard(phi.device());
    const int64_t bh = phi.size(0), T = phi.size(1), dk = phi.size(2), dv = ctx->saved_data["dv"].toInt();
    Tensor d[3];
    for (int i = 0; i < 3; ++i)
      d[i] = g[i].defined() ? canon(g[i], phi.scalar_type())
                            : at::zeros({(dk / kBlock) * (dv / kBlock) * bh, T, kBlock}, phi.options());
    const Tensor dphi = like(phi), dpsi = like(phi), dvv = plain(phi, {bh, T, dv});
    const Tensor parts = f32(phi, {bh, lib().atlas_block_parts((int)T), dv, dk});
    check(lib().atlas_block_merge(dt_code(phi), (int)bh, (int)T, (int)dk, (int)dv, ptr(phi), fptr(S_ref), ptr(d[0]), ptr(d[1]),
                            ptr(d[2]), mptr(dphi), mptr(dpsi), mptr(dvv), mfptr(parts), stream_of(phi)),
          "atlas_block_merge");
    return {dphi, dpsi, dvv, parts.sum(1)};
  }
};

std::tuple<Tensor, Tensor, Tensor> block_split(const Tensor& phi, const Tensor& psi, const Tensor& v, const Tensor& S_ref) {
  TORCH_CHECK(phi.is_cuda() && kernel_dtype(phi.scalar_type()), "block_split takes fp32 or bf16 GPU tensors");
  c10::DeviceGuard guard(phi.device());
  const at::ScalarType dt = phi.scalar_type();
  const variable_list o = BlockSplitFn::apply(aligned(phi), canon(psi, dt), canon(v, dt), canon(S_ref, at::kFloat));
  return {o[0], o[1], o[2]};
}

// ---------------------------------------------------------------------------------------------
// linear layers
// ---------------------------------------------------------------------------------------------
int64_t rows_of(const Tensor& t) { return t.numel() / std::max<int64_t>(t.size(-1), 1); }

// up to four products over the same rows in one launch: NT y = x W^T, NN dx = dy W; torch's for other
// dtypes, or sizes that are not multiples of 8
variable_list products(int layout, const variable_list& acts, const variable_list& weights) {
  TORCH_CHECK_VALUE(!acts.empty() && acts.size() == weights.size(), "products of ", acts.size(), " activations with ",
                    weights.size(), " weights");
  const int64_t m = rows_of(acts[0]);
  bool ok = acts.size() <= 4;
  for (size_t i = 0; i < acts.size(); ++i)
    ok = ok && acts[i].scalar_type() == at::kBFloat16 && weights[i].scalar_type() == at::kBFloat16 &&
         acts[i].size(-1) % 8 == 0 && weights[i].size(0) % 8 == 0 && weights[i].size(1) % 8 == 0 && rows_of(acts[i]) == m;
  variable_list outs;
  if (!ok) {
    for (size_t i = 0; i < acts.size(); ++i)
      outs.push_back(layout == ATLAS_GEMM_NT ? at::linear(acts[i], weights[i]) : at::matmul(acts[i], weights[i]));
    return outs;
  }
  for (size_t i = 0; i < acts.size(); ++i)   // the kernel reads what the sizes say, on the current device
    TORCH_CHECK(weights[i].dim() == 2 && weights[i].size(layout == ATLAS_GEMM_NT ? 1 : 0) == acts[i].size(-1) &&
                    acts[i].device() == acts[0].device() && weights[i].device() == acts[0].device(),
                "the products' operands do not fit: ", acts[i].sizes(), " on ", acts[i].device(), " and ",
                weights[i].sizes(), " on ", weights[i].device());
  TORCH_CHECK(acts[0].is_cuda(), "the bf16 products run on ROCm GPU tensors only");
  variable_list a, w;
  int ns[4], ks[4];
  const void *ap[4], *wp[4];
  void* op[4];
  for (size_t i = 0; i < acts.size(); ++i) {
    a.push_back(aligned(acts[i]));
    w.push_back(aligned(weights[i]));
    ns[i] = (int)w[i].size(layout == ATLAS_GEMM_NT ? 0 : 1);
    ks[i] = (int)a[i].size(-1);
    std::vector<int64_t> sizes = a[i].sizes().vec();
    sizes.back() = ns[i];
    outs.push_back(plain(a[i], sizes));
    ap[i] = ptr(a[i]);
    wp[i] = ptr(w[i]);
    op[i] = mptr(outs[i]);
  }
  check(lib().atlas_linear_batch(layout, (int)acts.size(), m, ns, ks, ap, wp, op, stream_of(a[0])), "atlas_linear_batch");
  return outs;
}

// dW = dy^T x over every leading axis, for each (dy, x) pair: bf16 pairs over the same tokens in one
// launch (csrc/wgrad.hip); others torch's product over token slices
variable_list wgrads(const variable_list& dys_in, const variable_list& xs_in, at::ScalarType dt) {
  TORCH_CHECK_VALUE(!dys_in.empty() && dys_in.size() == xs_in.size(), "weight gradients of ", dys_in.size(), " and ",
                    xs_in.size(), " activations");
  variable_list dys, xs, out;
  for (size_t i = 0; i < dys_in.size(); ++i) {
    dys.push_back(dys_in[i].reshape({-1, dys_in[i].size(-1)}));
    xs.push_back(xs_in[i].reshape({-1, xs_in[i].size(-1)}));
  }
  const int64_t n = dys[0].size(0);
  bool ok = kernel_dtype(dt) && dys.size() <= 4;
  for (size_t i = 0; i < dys.size(); ++i)
    ok = ok && dys[i].scalar_type() == at::kBFloat16 && xs[i].scalar_type() == at::kBFloat16 && dys[i].size(1) % 8 == 0 &&
         xs[i].size(1) % 8 == 0 && dys[i].size(0) == n && xs[i].size(0) == n;
  if (ok) {
    for (size_t i = 0; i < dys.size(); ++i)
      TORCH_CHECK(dys[i].device() == dys[0].device() && xs[i].device() == dys[0].device(),
                  "the weight gradients' operands are on more than one device");
    TORCH_CHECK(dys[0].is_cuda(), "the bf16 weight gradients run on ROCm GPU tensors only");
    int os[4], is[4];
    const void *dp[4], *xp[4];
    void* wp[4];
    const int cnt = (int)dys.size();
    for (int i = 0; i < cnt; ++i) {
      dys[i] = aligned(dys[i]);
      xs[i] = aligned(xs[i]);
      os[i] = (int)dys[i].size(1);
      is[i] = (int)xs[i].size(1);
      out.push_back(at::empty({os[i], is[i]}, dys[i].options().dtype(dt).requires_grad(false)));
      dp[i] = ptr(dys[i]);
      xp[i] = ptr(xs[i]);
      wp[i] = mptr(out[i]);
    }
    const int64_t bytes = lib().atlas_linear_wgrad_batch_workspace_bytes(cnt, n, os, is);
    const Tensor ws = scratch(dys[0], bytes);
    check(lib().atlas_linear_wgrad_batch(dt == at::kBFloat16 ? ATLAS_DT_BF16 : ATLAS_DT_F32, cnt, n, os, is, dp, xp, wp, mptr(ws),
                                   bytes, stream_of(dys[0])), "atlas_linear_wgrad_batch");
    return out;
  }
  for (size_t i = 0; i < dys.size(); ++i) {
    const int64_t o = dys[i].size(1), ni = xs[i].size(1);
    int64_t S = 1;
    for (int64_t c : {2, 4, 8})
      if (n % c == 0 && n / c >= 1024) S = c;
    if (S == 1) {
      out.push_back(at::matmul(dys[i].t(), xs[i]).to(dt));
      continue;
    }
    const Tensor a = dys[i].reshape({S, n / S, o}).transpose(1, 2).contiguous();   // both operands row-major
    out.push_back(at::bmm(a, xs[i].reshape({S, n / S, ni}).contiguous()).to(at::kFloat).sum(0).to(dt));
  }
  return out;
}

struct LinearFn : public Function<LinearFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
    ctx->save_for_backward({x, w});
    ctx->saved_data["need_x"] = x.requires_grad();
    ctx->saved_data["need_w"] = w.requires_grad();
    return products(ATLAS_GEMM_NT, {x}, {w});
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const variable_list s = ctx->get_saved_variables();
    c10::DeviceGuard guard(s[0].device());
    Tensor dx, dw;
    if (ctx->saved_data["need_x"].toBool()) dx = products(ATLAS_GEMM_NN, {g[0]}, {s[1]})[0];
    if (ctx->saved_data["need_w"].toBool()) dw = wgrads({g[0]}, {s[0]}, s[1].scalar_type())[0];
    return {dx, dw};
  }
};
Tensor linear(const Tensor& x, const Tensor& w) { return LinearFn::apply(x, w)[0]; }

// ---------------------------------------------------------------------------------------------
// the cell prologue (rnn_memory.py:567-653) as one node
// ---------------------------------------------------------------------------------------------
struct Partial {   // partial sums [rows, ..] fp32 -> their sum over the rows, in dt, of `sizes`
  Tensor parts;
  at::ScalarType dt;
  std::vector<int64_t> sizes;
};
variable_list sum_partials(const std::vector<Partial>& items) {
  constexpr int kMax = 16;
  TORCH_CHECK(!items.empty() && items.size() <= kMax, "sum_partials: ", items.size(), " items");
  int cols[kMax], dts[kMax];
  const float* src[kMax];
  void* dst[kMax];
  variable_list outs, keep;
  for (size_t i = 0; i < items.size(); ++i) {
    keep.push_back(aligned(items[i].parts));
    cols[i] = (int)(keep[i].numel() / keep[i].size(0));
    dts[i] = items[i].dt == at::kBFloat16 ? ATLAS_DT_BF16 : ATLAS_DT_F32;
    outs.push_back(at::empty(items[i].sizes, keep[i].options().dtype(items[i].dt)));
    src[i] = ptr(keep[i]);
    dst[i] = mptr(outs[i]);
  }
  check(lib().atlas_partials_sum((int)items.size(), (int)keep[0].size(0), cols, src, dst, dts, stream_of(keep[0])),
        "atlas_partials_sum");
  return outs;
}

struct PrologueDims {
  int64_t conv_k, heads, d;
  double eps;
};

// inputs: x, norm weight, three conv weights (conv_k > 1), three projections, up to four gate weights and
// biases, the two head-norm gammas. Outputs: xn, q, k, v, then one [(B H), T] tensor per gate head.
struct CellPrologueFn : public Function<CellPrologueFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& norm_w, const OptTensor& wq,
                               const OptTensor& wk, const OptTensor& wv, const Tensor& Wq, const Tensor& Wk,
                               const Tensor& Wv, const OptTensor& g0, const OptTensor& g1, const OptTensor& g2,
                               const OptTensor& g3, const OptTensor& b0, const OptTensor& b1, const OptTensor& b2,
                               const OptTensor& b3, const OptTensor& qg_in, const OptTensor& kg_in,
                               const PrologueDims& dims) {
    ctx->set_materialize_grads(false);
    const Tensor x = aligned(x_in);
    const int64_t B = x.size(0), T = x.size(1), dim = x.size(2), K = dims.conv_k, H = dims.heads, d = dims.d;
    const bool conv = K > 1;
    const int dt = dt_code(x);
    void* st = stream_of(x);
    Tensor xn = like(x), qi, ki, vi, taps[3];
    const Tensor inv = f32(x, {B, T});
    if (conv) {
      qi = like(x);
      ki = like(x);
      vi = like(x);
      const OptTensor* w[3] = {&wq, &wk, &wv};
      for (int i = 0; i < 3; ++i) taps[i] = aligned((*w[i])->reshape({dim, K}));
    }
    check(lib().atlas_prologue_fwd(dt, (int)B, (int)T, (int)dim, (int)K, (float)dims.eps, ptr(x), ptr(norm_w), ptr(taps[0]),
                             ptr(taps[1]), ptr(taps[2]), mptr(xn), mptr(qi), mptr(ki), mptr(vi), mptr(inv), st),
          "atlas_prologue_fwd");
    if (!conv) qi = ki = vi = xn;
    variable_list gw, gb;
    std::vector<int64_t> rows;
    for (const OptTensor* t : {&g0, &g1, &g2, &g3})
      if (t->has_value()) {
        gw.push_back(**t);
        rows.push_back((*t)->size(0));
      }
    for (const OptTensor* t : {&b0, &b1, &b2, &b3})
      if (t->has_value()) gb.push_back(**t);
    const Tensor Wg = gw.empty() ? Tensor() : aligned(gw.size() == 1 ? gw[0] : at::cat(gw));
    const Tensor bg = gb.empty() ? Tensor() : aligned(gb.size() == 1 ? gb[0] : at::cat(gb));
    variable_list acts{qi, ki, vi}, ws{Wq, Wk, Wv};
    if (Wg.defined()) {
      acts.push_back(xn);
      ws.push_back(Wg);
    }
    variable_list p = products(ATLAS_GEMM_NT, acts, ws);
    for (Tensor& t : p) t = aligned(t);
    const int64_t nG = bg.defined() ? bg.numel() / H : 0;
    const Tensor qg = qg_in.has_value() ? aligned(qg_in->reshape({H, d})) : Tensor();
    const Tensor kg = kg_in.has_value() ? aligned(kg_in->reshape({H, d})) : Tensor();
    const Tensor q = plain(x, {B * H, T, d}), k = like(q), v = like(q);
    const Tensor gates = nG ? plain(x, {nG, B * H, T}) : Tensor();
    check(lib().atlas_heads_fwd(dt, (int)B, (int)T, (int)H, (int)d, (int)nG, ptr(p[0]), ptr(p[1]), ptr(p[2]),
                          nG ? ptr(p[3]).p : nullptr, ptr(qg), ptr(kg), ptr(bg), mptr(q), mptr(k), mptr(v), mptr(gates), st),
          "atlas_heads_fwd");
    ctx->save_for_backward({x, norm_w, taps[0], taps[1], taps[2], inv, qi, ki, vi, xn, Wq, Wk, Wv, Wg, p[0], p[1], qg, kg,
                            gates});
    ctx->saved_data["dims"] = std::vector<int64_t>{K, H, d, nG};
    ctx->saved_data["rows"] = rows;
    ctx->saved_data["wshape"] = conv ? wq->sizes().vec() : std::vector<int64_t>{};
    ctx->saved_data["gshape"] = qg.defined() ? qg_in->sizes().vec() : std::vector<int64_t>{};
    ctx->saved_data["bdt"] = (int64_t)(bg.defined() ? bg.scalar_type() : x.scalar_type());
    ctx->saved_data["slots"] = std::vector<int64_t>{g0.has_value(), g1.has_value(), g2.has_value(), g3.has_value(),
                                                    b0.has_value(), b1.has_value(), b2.has_value(), b3.has_value()};
    ctx->saved_data["brows"] = [&] {
      std::vector<int64_t> r;
      for (const Tensor& t : gb) r.push_back(t.size(0));
      return r;
    }();
    variable_list out{xn, q, k, v};
    for (int64_t i = 0; i < nG; ++i) out.push_back(gates.select(0, i));
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &norm_w = s[1], &tq = s[2], &tk = s[3], &tv = s[4], &inv = s[5], &qi = s[6], &ki = s[7],
                 &vi = s[8], &xn = s[9], &Wq = s[10], &Wk = s[11], &Wv = s[12], &Wg = s[13], &ql = s[14], &kl = s[15],
                 &qg = s[16], &kg = s[17], &gates = s[18];
    c10::DeviceGuard guard(x.device());
    const std::vector<int64_t> dims = ctx->saved_data["dims"].toIntVector();
    const int64_t K = dims[0], H = dims[1], d = dims[2], nG = dims[3];
    const int64_t B = x.size(0), T = x.size(1), dim = x.size(2);
    const bool conv = K > 1, norm = qg.defined();
    const int dt = dt_code(x);
    void* st = stream_of(x);
    auto or_zero = [&](const Tensor& t, at::IntArrayRef sizes) {
      return t.defined() ? canon(t, x.scalar_type()) : at::zeros(sizes, x.options().requires_grad(false));
    };
    // ---- heads
    const Tensor dq = or_zero(g[1], {B * H, T, d}), dk = or_zero(g[2], {B * H, T, d}), dv = or_zero(g[3], {B * H, T, d});
    Tensor dg;
    if (nG) {
      variable_list parts;
      for (int64_t i = 0; i < nG; ++i) parts.push_back(or_zero(g[4 + i], {B * H, T}));
      dg = at::stack(parts);
    }
    const int64_t nwg = lib().atlas_prologue_num_workgroups((int)B, (int)T);
    const Tensor dql = like(ql), dkl = like(kl), dvl = like(ql);
    const Tensor dzl = nG ? plain(x, {B, T, nG * H}) : Tensor();
    const Tensor dqg = norm ? f32(x, {nwg, H, d}) : Tensor(), dkg = norm ? f32(x, {nwg, H, d}) : Tensor();
    const Tensor dbias = nG ? f32(x, {nwg, nG * H}) : Tensor();
    check(lib().atlas_heads_bwd(dt, (int)B, (int)T, (int)H, (int)d, (int)nG, ptr(ql), ptr(kl), ptr(qg), ptr(kg), ptr(gates),
                          ptr(dq), ptr(dk), ptr(dv), ptr(dg), mptr(dql), mptr(dkl), mptr(dvl), mptr(dzl), mptr(dqg),
                          mptr(dkg), mptr(dbias), st), "atlas_heads_bwd");
    // ---- projections
    variable_list acts{dql, dkl, dvl}, ws{Wq, Wk, Wv}, ins{qi, ki, vi};
    if (Wg.defined()) {
      acts.push_back(dzl);
      ws.push_back(Wg);
      ins.push_back(xn);
    }
    const variable_list di = products(ATLAS_GEMM_NN, acts, ws);
    const variable_list dw = wgrads(acts, ins, Wq.scalar_type());
    Tensor dsum = g[0];
    if (Wg.defined()) dsum = dsum.defined() ? dsum + di[3] : di[3];
    // ---- norm and convolutions
    Tensor dci[3];
    if (conv) {
      for (int i = 0; i < 3; ++i) dci[i] = canon(di[i], x.scalar_type());
    } else {
      const Tensor t = di[0] + di[1] + di[2];
      dsum = dsum.defined() ? t + dsum : t;
    }
    const Tensor dxn = or_zero(dsum, x.sizes());
    const Tensor dx = like(x), dnw = f32(x, {nwg, dim}), dcv = conv ? f32(x, {nwg, 3, dim, K}) : Tensor();
    check(lib().atlas_prologue_bwd(dt, (int)B, (int)T, (int)dim, (int)K, ptr(x), ptr(norm_w), ptr(tq), ptr(tk), ptr(tv), ptr(inv),
                             ptr(dxn), ptr(dci[0]), ptr(dci[1]), ptr(dci[2]), mptr(dx), mptr(dnw), mptr(dcv), st),
          "atlas_prologue_bwd");
    // ---- every parameter gradient of the two kernels from their partials, in one launch
    std::vector<Partial> parts{{dnw, norm_w.scalar_type(), norm_w.sizes().vec()}};
    std::vector<int64_t> wshape = ctx->saved_data["wshape"].toIntVector();
    if (conv) {
      wshape.insert(wshape.begin(), 3);
      parts.push_back({dcv, x.scalar_type(), wshape});
    }
    const std::vector<int64_t> gshape = ctx->saved_data["gshape"].toIntVector();
    if (norm) {
      parts.push_back({dqg, qg.scalar_type(), gshape});
      parts.push_back({dkg, kg.scalar_type(), gshape});
    }
    if (nG) parts.push_back({dbias, (at::ScalarType)ctx->saved_data["bdt"].toInt(), {nG * H}});
    const variable_list sums = sum_partials(parts);
    size_t i = 1;
    variable_list out(19);
    out[0] = dx;
    out[1] = sums[0];
    if (conv) {
      const Tensor t = sums[i++];
      for (int j = 0; j < 3; ++j) out[2 + j] = t.select(0, j);
    }
    for (int j = 0; j < 3; ++j) out[5 + j] = dw[j];
    if (norm) {
      out[16] = sums[i++];
      out[17] = sums[i++];
    }
    const std::vector<int64_t> slots = ctx->saved_data["slots"].toIntVector();
    const std::vector<int64_t> rows = ctx->saved_data["rows"].toIntVector(), brows = ctx->saved_data["brows"].toIntVector();
    int64_t at_w = 0, at_b = 0;
    size_t wi = 0, bi = 0;
    for (int j = 0; j < 4; ++j) {
      if (slots[j]) {
        out[8 + j] = dw[3].narrow(0, at_w, rows[wi]);
        at_w += rows[wi++];
      }
      if (slots[4 + j]) {
        out[12 + j] = sums[i].narrow(0, at_b, brows[bi]);
        at_b += brows[bi++];
      }
    }
    return out;
  }
};

variable_list cell_prologue(const Tensor& x, const Tensor& norm_weight, double eps, const variable_list& convs,
                            const variable_list& projs, variable_list gw, variable_list gb, const OptTensor& q_gamma,
                            const OptTensor& k_gamma, int64_t heads, int64_t dim_head) {
  // every list is indexed by position below, and the kernels read what the sizes here say
  TORCH_CHECK_VALUE(x.dim() == 3 && kernel_dtype(x.scalar_type()), "x must be an fp32 or bf16 tensor [B, T, dim]");
  TORCH_CHECK_VALUE(convs.empty() || convs.size() == 3, "conv_weights must be three (q, k, v), got ", convs.size());
  TORCH_CHECK_VALUE(projs.size() >= 3, "proj_weights must be three (q, k, v), got ", projs.size());
  TORCH_CHECK_VALUE(gw.empty() == gb.empty(), "gate_weights and gate_biases must both be given, got ", gw.size(), " and ",
                    gb.size());
  const int64_t dim = x.size(2), inner = heads * dim_head;
  TORCH_CHECK_VALUE(heads >= 1 && dim_head >= 1 && norm_weight.numel() == dim, "norm_weight must hold dim = ", dim,
                    " values, got ", norm_weight.sizes());
  for (int i = 0; i < 3; ++i)
    TORCH_CHECK_VALUE(projs[i].sizes() == at::IntArrayRef({inner, dim}), "proj_weights must be [", inner, ", ", dim,
                      "] (heads * dim_head, dim), got ", projs[i].sizes());
  int64_t gate_rows = 0, bias_rows = 0;
  for (const Tensor& t : gw) {
    TORCH_CHECK_VALUE(t.dim() == 2 && t.size(1) == dim, "gate_weights must be [heads, dim = ", dim, "], got ", t.sizes());
    gate_rows += t.size(0);
  }
  for (const Tensor& t : gb) bias_rows += t.numel();
  TORCH_CHECK_VALUE(gate_rows == bias_rows && gate_rows % heads == 0, "the gates have ", gate_rows, " weight rows and ",
                    bias_rows, " biases for ", heads, " heads");
  auto on_device = [&](const Tensor& t) { return t.device() == x.device(); };
  bool fits = x.is_cuda() && on_device(norm_weight) && (!q_gamma.has_value() || on_device(*q_gamma)) &&
              (!k_gamma.has_value() || on_device(*k_gamma));
  for (const variable_list* l : {&convs, &projs, (const variable_list*)&gw, (const variable_list*)&gb})
    for (const Tensor& t : *l) fits = fits && on_device(t);
  TORCH_CHECK(fits, "the cell prologue runs on ROCm GPU tensors of one device only");
  c10::DeviceGuard guard(x.device());
  const at::ScalarType dt = x.scalar_type();
  auto cast = [&](const Tensor& t) { return t.scalar_type() == dt ? t : t.to(dt); };
  auto ocast = [&](const OptTensor& t) { return t.has_value() ? OptTensor(cast(*t)) : OptTensor(); };
  for (Tensor& t : gw) t = cast(t);
  for (Tensor& t : gb) t = cast(t);
  if (gw.size() > 4 || gb.size() != gw.size()) {   // the biases may come in another split than the weights
    gw = {at::cat(gw)};
    gb = {at::cat(gb)};
  }
  OptTensor g[4], b[4], c[3];
  for (size_t i = 0; i < gw.size(); ++i) {
    g[i] = gw[i];
    b[i] = gb[i];
  }
  int64_t conv_k = convs.empty() ? 0 : convs[0].size(-1);
  if (conv_k > 1) {
    for (int i = 0; i < 3; ++i) c[i] = cast(convs[i]);
  } else {
    conv_k = 0;
  }
  const PrologueDims dims{conv_k, heads, dim_head, eps};
  return CellPrologueFn::apply(x, cast(norm_weight).contiguous(), c[0], c[1], c[2], cast(projs[0]), cast(projs[1]),
                               cast(projs[2]), g[0], g[1], g[2], g[3], b[0], b[1], b[2], b[3], ocast(q_gamma),
                               ocast(k_gamma), dims);
}

// ---------------------------------------------------------------------------------------------
// the Omega weight-update chain (omega.py:254-322): every tensor of surprise's dtype, surprise [BH, n, P]
// ---------------------------------------------------------------------------------------------
struct OmegaChainFn : public Function<OmegaChainFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& s, const Tensor& decay, const Tensor& last,
                               const OptTensor& am_, const OptTensor& lm_, const OptTensor& gate_, const OptTensor& buf_,
                               int64_t window, bool grad) {
    ctx->set_materialize_grads(false);
    const Tensor am = get(am_), lm = get(lm_), gate = get(gate_), buf = get(buf_);
    const int64_t BH = s.size(0), n = s.size(1), p = s.size(2), O = am.defined() ? am.size(0) : 0;
    const Tensor update = plain(s, {BH, n + 1, p}), moms = O && grad ? plain(s, {O, BH, n, p}) : Tensor();
    const Tensor next_lm = O ? plain(s, {O, BH, p}) : Tensor(), next_buf = window > 1 ? plain(s, {BH, window - 1, p}) : Tensor();
    // the backward has its own copies of the updates and the decays, so that the caller may edit the returned
    // and the given ones in place before it (a second write of the updates: 91.4 -> 93.6 us forward and backward at 16 x 64 x 8192 fp32)
    const Tensor kept = grad ? like(update) : Tensor(), kept_decay = grad ? like(decay) : Tensor();
    check(lib().atlas_omega_chain_fwd_keep(dt_code(s), BH, n, p, (int)O, (int)window, ptr(s), ptr(decay), ptr(last), ptr(am),
                                     ptr(lm), ptr(gate), ptr(buf), mptr(update), mptr(moms), mptr(next_lm), mptr(next_buf),
                                     mptr(kept), mptr(kept_decay), stream_of(s)),
          "atlas_omega_chain_fwd");
    if (grad) {   // (only the gradient of a gate on the surprises themselves reads them)
      const bool dgate = gate.defined() && gate.requires_grad();
      ctx->save_for_backward({!O && dgate ? s : Tensor(), kept_decay, am, lm, gate, kept, moms});
      ctx->saved_data["dgate"] = dgate;
      ctx->saved_data["window"] = window;
      ctx->saved_data["has_buf"] = buf.defined();
    }
    variable_list out{update};
    if (O) out.push_back(next_lm);
    if (window > 1) out.push_back(next_buf);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const variable_list sv = ctx->get_saved_variables();
    const Tensor &s = sv[0], &decay = sv[1], &am = sv[2], &lm = sv[3], &gate = sv[4], &update = sv[5], &moms = sv[6];
    c10::DeviceGuard guard(update.device());
    const int64_t BH = update.size(0), n = update.size(1) - 1, p = update.size(2), O = am.defined() ? am.size(0) : 0;
    const int64_t e = ctx->saved_data["window"].toInt();
    size_t i = 1;
    const Tensor dup = aligned(g[0]), dlm = O ? aligned(g[i++]) : Tensor(), dbo = e > 1 ? aligned(g[i++]) : Tensor();
    const Tensor ds = plain(update, {BH, n, p}), dd = like(decay), dam = like(am), dlm0 = like(lm),
                 dlast = plain(update, {BH, p});
    const Tensor dg = ctx->saved_data["dgate"].toBool() ? like(gate) : Tensor();
    const Tensor dbuf = ctx->saved_data["has_buf"].toBool() ? plain(update, {BH, e - 1, p}) : Tensor();
    const int64_t bytes = lib().atlas_omega_chain_workspace_bytes(BH, n, p, (int)O);
    const Tensor ws = scratch(update, bytes);
    check(lib().atlas_omega_chain_bwd(dt_code(update), BH, n, p, (int)O, (int)e, ptr(s), ptr(decay), ptr(am), ptr(lm), ptr(gate),
                                ptr(update), ptr(moms), ptr(dup), ptr(dlm), ptr(dbo), mptr(ds), mptr(dd), mptr(dlast),
                                mptr(dam), mptr(dlm0), mptr(dg), mptr(dbuf), mptr(ws), bytes, stream_of(update)),
          "atlas_omega_chain_bwd");
    return {ds, dd, dlast, dam, dlm0, dg, dbuf, Tensor(), Tensor()};
  }
};

// None where the fused kernels do not apply: one dtype (fp32 or bf16) on one GPU for the surprises and
// the scalars, at most two momentum orders and a window of at most 16 (both are held in registers),
// and sizes inside their index ranges.
std::optional<Four> omega_chain(const Tensor& s, const Tensor& decay, const Tensor& last, const OptTensor& am,
                                const OptTensor& lm, const OptTensor& gate, int64_t window, const OptTensor& buf) {
  const at::ScalarType dt = s.scalar_type();
  if (!kernel_dtype(dt) || !s.is_cuda() || window < 1 || window > 16 || s.dim() < 2 || s.numel() == 0) return std::nullopt;
  const int64_t BH = s.size(0), n = s.size(1), p = s.numel() / (BH * n), O = am.has_value() ? am->size(0) : 0;
  if ((am.has_value() && (O < 1 || O > 2 || !lm.has_value())) || BH > 65535 || n > (1 << 24) || p > ((int64_t)1 << 31))
    return std::nullopt;
  bool grad = false;
  auto ok = [&](const Tensor& t, bool scalar) {
    grad = grad || t.requires_grad();
    return t.device() == s.device() && (!scalar || t.scalar_type() == dt);
  };
  auto ook = [&](const OptTensor& t, bool scalar) { return !t.has_value() || ok(*t, scalar); };
  if (!ok(s, true) || !ok(decay, true) || !ok(last, false) || !ook(am, true) || !ook(lm, false) || !ook(gate, true) ||
      !ook(buf, false))
    return std::nullopt;
  c10::DeviceGuard guard(s.device());
  // views only where the shape differs: each is a node of the autograd graph
  auto shaped = [](const Tensor& t, at::IntArrayRef sizes) { return t.sizes() == sizes ? t : t.reshape(sizes); };
  auto flat = [&](const Tensor& t, at::IntArrayRef sizes) { return canon(shaped(t, sizes), dt); };
  const std::vector<int64_t> param(s.sizes().begin() + 2, s.sizes().end());
  auto full = [&](const Tensor& t, std::vector<int64_t> sizes) {
    sizes.insert(sizes.end(), param.begin(), param.end());
    return shaped(t, sizes);
  };
  const variable_list out = OmegaChainFn::apply(
      flat(s, {BH, n, p}), shaped(decay, {BH, n}).contiguous(), flat(last, {BH, p}),
      am.has_value() ? OptTensor(shaped(*am, {O, BH, n}).contiguous()) : OptTensor(),
      O ? OptTensor(flat(*lm, {O, BH, p})) : OptTensor(),
      gate.has_value() ? OptTensor(shaped(*gate, {BH, n}).contiguous()) : OptTensor(),
      buf.has_value() && window > 1 ? OptTensor(flat(*buf, {BH, window - 1, p})) : OptTensor(), window,
      grad && at::GradMode::is_enabled());
  const Tensor update = full(out[0], {BH, n + 1});
  size_t i = 1;
  const Tensor lm1 = O ? full(out[i++], {O, BH}) : Tensor(), buf1 = window > 1 ? full(out[i++], {BH, window - 1}) : Tensor();
  return Four{update, update.select(1, n), opt(lm1), opt(buf1)};
}

// an entry point of the module: refused while torch.jit.trace records, other Python threads run meanwhile
template <typename R, typename... A>
auto entry(R (*f)(A...)) {
  return [f](A... a) -> R {
    TORCH_CHECK(!torch::jit::tracer::isTracing(), "the native operators are not traced: call them through atlas_rnn_amd");
    py::gil_scoped_release threads;
    return f(std::forward<A>(a)...);
  };
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("bind", &bind);
  m.def("library", [] { return lib().path; });
  m.def("recurrence", entry(&recurrence));
  m.def("tensor_map", entry(&tensor_map));
  m.def("symmetrized", entry(&symmetrized));
  m.def("block_split", entry(&block_split));
  m.def("replicate", entry(&replicate));
  m.def("replica_sum", entry(&replica_sum));
  m.def("products", entry(&products));
  m.def("wgrads", entry(&wgrads));
  m.def("linear", entry(&linear));
  m.def("cell_prologue", entry(&cell_prologue));
  m.def("omega_chain", entry(&omega_chain));
}
