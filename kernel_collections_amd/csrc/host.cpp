// Native host layer of the decode and score calls: checks, split choice, scratch and every launch of one call behind a single
// Python call.  A decode step of a short context is 10 - 20 us of kernels; marshalled through ctypes, launch by launch, the same
// call cost 28 us (plain GQA, two launches) to 102 us (prefix + tail, six) of host time and was bound by it.
//
// Each function takes the operands as the public wrapper got them and returns its result, or None when an operand is not
// what it serves as it is (a shape the wrapper asserts on, a layout that has to be copied first): the wrapper then goes through its
// general path, which raises or copies.  No state but a per-thread table of split counts, which depend on sizes alone.
//
// The C ABI of libxkv_hip.so is called through the addresses of the library that the Python binding loaded (init).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cstdint>
#include <stdexcept>

#include "../../include/xkv_hip.h"
#include "head_rows.h"
#include "merge_rule.h"
#include "recon_groups.h"

namespace {

// ---- the kernels' library ------------------------------------------------------------------------------------------
#define XKV_SYMBOLS(X)                                                                                              \
  X(xkv_error_string) X(xkv_absorb_q) X(xkv_blockdiag_q) X(xkv_latent_stage1) X(xkv_softmax_pv_stage1) X(xkv_recon_stage1) \
  X(xkv_recon_workspace_bytes) X(xkv_merge_stage2) X(xkv_plan_splits)
// newer than the version they are in, with xkv_softmax_pv_stage1 over value rows of 128 and 192 and more than 32 heads: over a library
// without them (joined() false) a call takes the launches that it has
#define XKV_OPTIONAL_SYMBOLS(X) X(xkv_absorb_q_tail) X(xkv_merge_stage2_tail)
#define XKV_DECLARE(name) decltype(&name) p_##name = nullptr;
XKV_SYMBOLS(XKV_DECLARE)
XKV_OPTIONAL_SYMBOLS(XKV_DECLARE)
#undef XKV_DECLARE

bool joined() { return p_xkv_absorb_q_tail && p_xkv_merge_stage2_tail; }

struct CallError : std::runtime_error { using std::runtime_error::runtime_error; };
void check(int rc, const char* what) {
  if (rc != XKV_OK)
    throw CallError(std::string(what) + " failed: " + p_xkv_error_string(rc) + " (code " + std::to_string(rc) + ")");
}

struct Decline {};                       // an operand this layer does not serve as it is
inline void need(bool ok) { if (!ok) throw Decline(); }

inline int cdiv(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

// ---- splits ----------------------------------------------------------------------------------------------------------
int num_cus(int device) {
  static std::array<std::atomic<int>, 64> cache{};
  if (device < 0 || device >= 64) throw CallError("device index out of range");
  int n = cache[device].load(std::memory_order_relaxed);
  if (!n) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0)
      throw CallError("cannot read the number of compute units");
    cache[device].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Number of KV splits for a stage 1 that keeps `per_cu` workgroups on a CU: the count whose slowest CU is done first when every
// workgroup costs its tiles plus a start of about four (launch, query and factor loads, first tile).  A count just past a
// whole number of rounds would leave the chip idle behind a nearly empty last one (batch 3 x 8 kv heads: 11 splits are 264
// workgroups, two rounds on 256 CUs; 10 are one), and 160 workgroups (batch 20) are one round of a chip that is two thirds full
// where 480 are two full ones.
int balanced_splits(int64_t batch, int groups, int64_t kv_len, int tile, int per_cu, int cus) {
  const int64_t blocks = (kv_len + 31) / 32;   // split lengths are multiples of 32 tokens, and the length counts in those alone
  // a decode loop has another length at every token: it finds its count here for 32 steps, and the search for the next (a few
  // microseconds) looks at every length of a split once, not at every number of splits
  struct Entry { int64_t batch = -1, blocks = 0; int groups = 0, tile = 0, per_cu = 0, cus = 0, splits = 0; };
  static thread_local std::array<Entry, 256> table;
  size_t h = (size_t)(batch * 1000003 + blocks) * 31 + groups * 7 + tile * 131 + per_cu;
  Entry& e = table[(h ^ (h >> 8) ^ (h >> 17)) & 255];
  if (e.batch == batch && e.blocks == blocks && e.groups == groups && e.tile == tile && e.per_cu == per_cu && e.cus == cus) return e.splits;
  constexpr int XCDS = 8, START = 4;
  const int64_t most = std::min<int64_t>(blocks, 4LL * per_cu * cus);
  int64_t best = 1, best_cost = INT64_MAX, seen = 0;
  for (int64_t want = 1, per; want <= most; want = per > 1 ? (blocks + per - 2) / (per - 1) : most + 1) {
    per = (blocks + want - 1) / want;
    const int64_t live = (blocks + per - 1) / per;   // splits that hold tokens
    if (live == seen) continue;
    seen = live;
    // clusters of `groups` workgroups (one (sequence, split)) go round-robin over the XCDs, each with cus / XCDS CUs of its own
    const int64_t slots = (int64_t)per_cu * (cus / XCDS);
    const int64_t rounds = ((batch * live + XCDS - 1) / XCDS * groups + slots - 1) / slots;
    const int64_t cost = rounds * ((32 * per + tile - 1) / tile + START);
    if (cost < best_cost) { best = live; best_cost = cost; }
    if (rounds > 2 && batch * live * groups > 8LL * per_cu * cus) break;   // finer only adds starts
  }
  e = Entry{batch, blocks, groups, tile, per_cu, cus, (int)best};
  return (int)best;
}

int head_groups(int64_t hq) {            // smallest number of equal head groups of at most 32
  need(hq > 0);
  int g = cdiv(hq, 32);
  while (hq % g) ++g;
  return g;
}

// ---- operands --------------------------------------------------------------------------------------------------------
typedef const at::Tensor& Ten;

int code16(Ten t) {
  const auto d = t.scalar_type();
  need(d == at::kBFloat16 || d == at::kHalf);
  return d == at::kBFloat16 ? XKV_BF16 : XKV_F16;
}
int code_any(Ten t) { return t.scalar_type() == at::kFloat ? XKV_F32 : code16(t); }

// unit stride on the feature axis, every other stride a multiple of 8 elements, 16-byte base
bool rows(Ten t) {
  const auto st = t.strides();
  const int64_t n = t.dim();
  if (st[n - 1] != 1 || (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15)) return false;
  for (int64_t i = 0; i + 1 < n; ++i)
    if (st[i] & 7) return false;
  return true;
}
bool packed_q(Ten t) { return t.is_contiguous() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
xkv_kv_operand kv(Ten t, int64_t sh, int64_t dim) { return {t.data_ptr(), t.stride(0), t.stride(1), sh, (int)dim}; }
constexpr xkv_kv_operand NO_KV = {nullptr, 0, 0, 0, 0};
constexpr xkv_q_operand NO_Q = {nullptr, 0};

// One call: its device, stream, operand type, and one scratch buffer cut into 256-byte-aligned pieces.
struct Call {
  c10::DeviceGuard guard;
  int device, cus, dt;
  void* stream;
  at::TensorOptions opts;
  at::Tensor scratch;
  int64_t used = 0;
  Call(Ten q) : guard(q.device()), device(q.device().index()), cus(num_cus(device)), dt(code16(q)),
                stream(c10::hip::getCurrentHIPStream(device).stream()), opts(q.options()) {}
  int64_t plan(int64_t bytes) { const int64_t at = used; used += (bytes + 255) & ~(int64_t)255; return at; }
  void alloc() { scratch = at::empty({used}, opts.dtype(at::kByte)); }
  bool try_alloc() {   // false: no room for it
    try {
      alloc();
    } catch (const c10::OutOfMemoryError&) {
      return false;
    }
    return true;
  }
  template <typename T> T* get(int64_t at) const { return reinterpret_cast<T*>(reinterpret_cast<char*>(scratch.data_ptr()) + at); }
};
inline void same(Ten q, std::initializer_list<const at::Tensor*> ts) {   // same 16-bit type, same device
  need(q.is_cuda());
  for (const at::Tensor* t : ts) need(t->is_cuda() && t->device() == q.device() && t->scalar_type() == q.scalar_type());
}

// Splits of one stage 1 + merge: a count for every sequence, or a packed plan on the device for a ragged batch.  S: splits that a
// sequence may have; n: what the C entry points take as max_splits (S, or the jobs of the plan).
struct Splits {
  int S, cap;
  const int32_t* lens;
  int32_t* plan;
  int jobs = 0;
  int n() const { return jobs ? jobs : S; }
  int64_t rows(int64_t batch, int64_t hq) const { return hq * (jobs ? jobs : batch * S); }   // partial rows of the whole call
};

// Shortest split, in tokens: 128, where a job's start (about 5 us) is a third of its time, or less for a batch too short to fill the
// device at that.  u: the split at which it is filled once, or half of it where the merged rows are up-projected (every split adds a
// partial row to that merge).  The register-staged kernel goes down to its tile of 64.
int split_floor(int64_t batch, int groups, int64_t kv_len, int per_cu, int cus, bool up) {
  const int64_t slots = (int64_t)per_cu * cus / (up ? 2 : 1), u = (batch * kv_len * groups + slots - 1) / slots;
  if (per_cu > 1) return u <= 64 ? 64 : 128;
  return (int)std::clamp<int64_t>((u + 31) / 32 * 32, up ? 64 : 32, 128);
}
// Jobs that a ragged batch is cut into at most: one per workgroup the chip holds, or as many whole rounds as make two a sequence.  With
// no more jobs than sequences none is cut, and the longest one is the call: 64 sequences, one of 8000 tokens among short ones, 64 heads
// on 8 kv heads (64 jobs a round) 250 us, with two rounds 40; all of 1000 .. 8000 tokens 299 and 269.  Three or more jobs a sequence
// gain up to 15 % on evenly spread lengths and lose as much on a long one among short ones.
int ragged_target(int64_t batch, int groups, int per_cu, int cus) {
  const int64_t round = std::max(1, per_cu * cus / groups);
  return (int)(round * ((2 * batch + round - 1) / round));
}

// A ragged batch: planned on the device so that it is cut into at most ragged_target() jobs, no job shorter than
// `floor` tokens or a 256th of the longest sequence.  Its partial rows are packed: as many as there are jobs, or sequences, whatever the
// lengths (64 sequences of up to 32K tokens, 32 heads, value rank 512: 17 MB; one row per sequence and possible split would be 1.07 GB).
struct Ragged { int target; int64_t at; };
Ragged ragged(Call& c, Splits& s, int64_t batch, int groups, int64_t kv_len, int floor, int per_cu) {
  s.cap = std::max<int64_t>(floor, (cdiv(kv_len, 256) + 31) / 32 * 32);
  s.S = cdiv(kv_len, s.cap);
  // a workgroup per CU even if all are as long: the floor is the plan, without the 4 us of the planning kernel in front of the scan
  if (batch * s.S * groups <= c.cus) return {0, 0};
  const int target = ragged_target(batch, groups, per_cu, c.cus);
  s.jobs = std::max<int64_t>(target, batch);
  return {target, c.plan((3 + 2 * (int64_t)s.jobs + batch) * 4)};
}
void write_plan(const Call& c, Splits& s, const Ragged& r, int64_t batch) {
  if (!s.jobs) return;
  s.plan = c.get<int32_t>(r.at);
  check(p_xkv_plan_splits(s.lens, nullptr, batch, s.jobs, s.cap, r.target, s.plan, c.stream), "xkv_plan_splits");
}

// ---- merge (with or without the up-projection by vB [b, hkv, dv, d_out]) ------------------------------------------------
struct Up { const void* p; int64_t sb, sh, sr; int d_out, dtype, hkv; };
bool rows_first(int S, int64_t hq, const Up& up, int64_t dv, int64_t batch) { return xkv::merge_rows_first(S, hq, up.hkv, dv, batch, up.d_out); }
int64_t rows_bytes(int64_t batch, int64_t hq, int64_t dv) { return batch * hq * (dv + 1) * 4; }

void merge(const Call& c, const float* partial, const float* lse, void* out, int64_t sOb, int64_t sOh, int out_dtype, const Up* up,
           int64_t rows_at, const Splits& s, int64_t batch, int64_t hq, int64_t kv_len, int64_t dv, float* lse_out = nullptr,
           int64_t sLb = 0, int64_t sLh = 0) {
  if (!up) {
    check(p_xkv_merge_stage2(partial, lse, out, nullptr, 0, 0, 0, 0, XKV_BF16, nullptr, s.lens, batch, hq, hq, kv_len, s.n(), s.cap,
                             s.plan, dv, sOb, sOh, out_dtype, lse_out, sLb, sLh, c.stream), "xkv_merge_stage2");
    return;
  }
  if (rows_first(s.S, hq, *up, dv, batch)) {   // many splits: merge the rows first, spread over the chip, then one row per head
    float* mid = c.get<float>(rows_at);
    float* mid_lse = lse_out ? lse_out : mid + batch * hq * dv;
    if (!lse_out) { sLb = hq; sLh = 1; }
    check(p_xkv_merge_stage2(partial, lse, mid, nullptr, 0, 0, 0, 0, XKV_BF16, nullptr, s.lens, batch, hq, hq, kv_len, s.n(), s.cap,
                             s.plan, dv, hq * dv, dv, XKV_F32, mid_lse, sLb, sLh, c.stream), "xkv_merge_stage2");
    // a single row's log-sum-exp is not read
    check(p_xkv_merge_stage2(mid, mid_lse, out, up->p, up->sb, up->sh, up->sr, up->d_out, up->dtype, nullptr, nullptr, batch, hq, up->hkv,
                             32, 1, 0, nullptr, dv, sOb, sOh, out_dtype, nullptr, 0, 0, c.stream), "xkv_merge_stage2");
    return;
  }
  check(p_xkv_merge_stage2(partial, lse, out, up->p, up->sb, up->sh, up->sr, up->d_out, up->dtype, nullptr, s.lens, batch, hq, up->hkv,
                           kv_len, s.n(), s.cap, s.plan, dv, sOb, sOh, out_dtype, lse_out, sLb, sLh, c.stream), "xkv_merge_stage2");
}

Up up_of(Ten vB, int64_t hq, int dt) {
  need(rows(vB) && vB.size(3) <= 512 && vB.size(3) % 8 == 0);
  Up u{vB.data_ptr(), vB.stride(0), vB.stride(1), vB.stride(2), (int)vB.size(3), dt, (int)vB.size(1)};
  if (u.hkv == 1 && hq > 32) { u.hkv = head_groups(hq); u.sh = 0; }   // the kernel serves at most 32 query heads per kv head
  need(hq / u.hkv <= 32);
  return u;
}

// ---- arguments -------------------------------------------------------------------------------------------------------
Ten T(PyObject* o) {
  need(THPVariable_Check(o));
  return THPVariable_Unpack(o);
}
float F(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); throw Decline(); }
  return (float)v;
}
int64_t I(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); throw Decline(); }
  return v;
}
at::Tensor lens_of(PyObject* o, Ten q, int64_t batch) {   // undefined: one length
  if (o == Py_None) return at::Tensor();
  Ten l = T(o);
  need(l.is_cuda() && l.device() == q.device() && l.scalar_type() == at::kInt && l.dim() == 1 && l.numel() == batch && l.is_contiguous());
  return l;
}

template <typename Fn> PyObject* guarded(Py_ssize_t n, Py_ssize_t want, Fn fn) {
  if (n != want) { PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n); return nullptr; }
  try {
    return fn();
  } catch (const Decline&) {
    Py_RETURN_NONE;
  } catch (...) {   // as torch's own bindings raise it: an allocator that ran out of memory as torch.OutOfMemoryError
    if (!PyErr_Occurred()) torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}
inline PyObject* give(PyObject* o) { Py_INCREF(o); return o; }
// What a call does once its arguments are C++ values.  Other Python threads run meanwhile: an allocator that has to free its cache
// waits for the device, and a host function that Python put on a stream needs the interpreter to finish.
template <typename Fn> void without_gil(Fn fn) {
  struct Released {
    PyThreadState* state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  fn();
}

// ---- shared pieces of the factorised calls -----------------------------------------------------------------------------
// Absorbed query q~ = q . B^T as a high + low pair [b, hq, rank]
void absorb(const Call& c, const void* q, Ten B, void* hi, void* lo, int64_t batch, int64_t hq, int64_t d, int64_t rank) {
  int64_t hkv = B.size(1), sh = B.stride(1);
  if (hkv == 1 && hq > 32) { hkv = head_groups(hq); sh = 0; }
  check(p_xkv_absorb_q(q, B.data_ptr(), hi, lo, batch, hq, hkv, d, rank, B.stride(0), sh, B.stride(2), c.dt, c.stream), "xkv_absorb_q");
}
bool ring_rank(int64_t r) { return r == 512 || r == 384 || r == 256; }
// absorbed scans that the LDS-ring kernel serves: key rank 192 only beside values of a ring rank of their own, or for scores (rv 0)
bool ring_scan(int64_t r, int64_t rv) { return ring_rank(r) || (r == 192 && (rv == 0 || ring_rank(rv))); }
// an absorbed scan over `rank`-wide rows: the LDS-ring kernel (one workgroup per CU) at ranks 256 .. 512, else the register-staged one
int scan_splits(const Call& c, int64_t batch, int groups, int64_t kv_len, bool ring) {
  return balanced_splits(batch, groups, kv_len, ring ? 32 : 64, ring ? 1 : 2, c.cus);
}

// nope_decode(q [b,hq,d], kA [b,L,r], kB [b,hkv,r,d], vA [b,L,rv], vB [b,hkv,rv,dv], o, sm_scale, lens | None) -> o | None
PyObject* nope_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 8, [&]() -> PyObject* {
    Ten q = T(a[0]), kA = T(a[1]), kB = T(a[2]), vA = T(a[3]), vB = T(a[4]), o = T(a[5]);
    const float scale = F(a[6]);
    same(q, {&kA, &kB, &vA, &vB});
    need(o.is_cuda() && o.device() == q.device());
    need(q.dim() == 3 && kA.dim() == 3 && kB.dim() == 4 && vA.dim() == 3 && vB.dim() == 4 && o.dim() == 3);
    const int64_t b = q.size(0), hq = q.size(1), d = q.size(2), L = kA.size(1), r = kA.size(2), hkv = kB.size(1), rv = vA.size(2);
    need(b > 0 && L > 0 && hkv > 0 && kA.size(0) == b && kB.size(0) == b && vA.size(0) == b && vB.size(0) == b && vA.size(1) == L && vB.size(1) == hkv);
    need(kB.size(2) == r && kB.size(3) == d && vB.size(2) == rv && hq % hkv == 0 && r % 32 == 0 && rv % 64 == 0 && rv <= 512 && d <= 512 && d % 8 == 0);
    need(packed_q(q) && rows(kA) && rows(kB) && rows(vA) && o.stride(2) == 1 && o.size(0) == b && o.size(1) == hq && o.size(2) == vB.size(3));
    need(hkv == 1 || hq / hkv <= 32);
    const at::Tensor lens = lens_of(a[7], q, b);
    without_gil([&] {
      Call c(q);
      const Up up = up_of(vB, hq, c.dt);
      const int groups = head_groups(hq), odt = code_any(o);
      Ragged rg{};
      Splits s{0, 0, nullptr, nullptr};
      const int per_cu = ring_scan(r, rv) ? 1 : 2;
      const bool planned = lens.defined() && b > 1;   // one sequence is cut into the splits of the longest it may be
      if (planned) rg = ragged(c, s, b, groups, L, split_floor(b, groups, L, per_cu, c.cus, true), per_cu);
      else s.S = scan_splits(c, b, groups, L, ring_scan(r, rv));
      if (lens.defined()) s.lens = lens.data_ptr<int32_t>();
      const int64_t hi = c.plan(b * hq * r * 2), lo = c.plan(b * hq * r * 2), part = c.plan(s.rows(b, hq) * rv * 4), lse = c.plan(s.rows(b, hq) * 4);
      const int64_t mid = c.plan(rows_first(s.S, hq, up, rv, b) ? rows_bytes(b, hq, rv) : 0);
      c.alloc();
      if (planned) write_plan(c, s, rg, b);
      absorb(c, q.data_ptr(), kB, c.get<void>(hi), c.get<void>(lo), b, hq, d, r);
      check(p_xkv_latent_stage1({c.get<void>(hi), (int)r}, c.get<void>(lo), NO_Q, kv(kA, 0, r), NO_KV, kv(vA, 0, rv), c.get<float>(part),
                                c.get<float>(lse), nullptr, 0, nullptr, s.lens, b, hq, groups, L, s.n(), s.cap, s.plan, scale, 0.f, c.dt,
                                c.stream), "xkv_latent_stage1");
      merge(c, c.get<float>(part), c.get<float>(lse), o.data_ptr(), o.stride(0), o.stride(1), odt, &up, mid, s, b, hq, L, rv);
    });
    return give(a[5]);
  });
}

// nope_scores(q [b,hq,1,d], A [b,L,r], B [b,hkv,r,d], sm_scale, fp32_out) -> [b,hq,1,L] | None
PyObject* nope_scores(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 5, [&]() -> PyObject* {
    Ten q = T(a[0]), A = T(a[1]), B = T(a[2]);
    const float scale = F(a[3]);
    const bool f32 = I(a[4]);
    same(q, {&A, &B});
    need(q.dim() == 4 && A.dim() == 3 && B.dim() == 4 && q.size(2) == 1);
    const int64_t b = q.size(0), hq = q.size(1), d = q.size(3), L = A.size(1), r = A.size(2), hkv = B.size(1);
    need(b > 0 && L > 0 && hkv > 0 && A.size(0) == b && B.size(0) == b && B.size(2) == r && B.size(3) == d && hq % hkv == 0 && r % 32 == 0);
    need(d <= 512 && d % 8 == 0 && packed_q(q) && rows(A) && rows(B) && (hkv == 1 || hq / hkv <= 32));
    at::Tensor out;
    without_gil([&] {
      Call c(q);
      const int groups = head_groups(hq), S = scan_splits(c, b, groups, L, ring_scan(r, 0));
      const int64_t hi = c.plan(b * hq * r * 2), lo = c.plan(b * hq * r * 2);
      c.alloc();
      out = at::empty({b, hq, 1, L}, f32 ? c.opts.dtype(at::kFloat) : c.opts);
      absorb(c, q.data_ptr(), B, c.get<void>(hi), c.get<void>(lo), b, hq, d, r);
      check(p_xkv_latent_stage1({c.get<void>(hi), (int)r}, c.get<void>(lo), NO_Q, kv(A, 0, r), NO_KV, NO_KV, nullptr, nullptr, out.data_ptr(),
                                f32 ? XKV_F32 : c.dt, nullptr, nullptr, b, hq, groups, L, S, 0, nullptr, scale, 0.f, c.dt, c.stream),
            "xkv_latent_stage1");
    });
    return THPVariable_Wrap(out);
  });
}

void recon(const Call& c, Ten q, Ten kA, Ten kB, const at::Tensor* vA, float* partial, float* lse, void* scores, int scores_dtype, int S,
           bool grouped, int64_t b, int64_t hq, int64_t hkv, int64_t L, float scale, const float* inv, int64_t pos, void* ws, int64_t ws_bytes,
           const int32_t* lens = nullptr) {
  check(p_xkv_recon_stage1(q.data_ptr(), kv(kA, 0, kA.size(2)), kB.data_ptr(), kB.stride(0), kB.stride(1), kB.stride(2),
                           vA ? kv(*vA, 0, vA->size(2)) : NO_KV, partial, lse, scores, scores_dtype, nullptr, lens, b, hq, hkv, L, S,
                           scale, grouped ? XKV_ROPE_GROUPED : 1, inv, pos, nullptr, 0, ws, ws_bytes, c.dt, c.stream), "xkv_recon_stage1");
}
void rope_operands(Ten q, int64_t hq, int64_t d, Ten kA, Ten kB, Ten inv) {
  const int64_t b = q.size(0), hkv = kB.size(1), r = kA.size(2);
  need(b > 0 && kA.size(1) > 0 && hkv > 0 && kA.size(0) == b && kB.size(0) == b && kB.size(2) == r && kB.size(3) == d && d == 128);
  need(hq % hkv == 0 && hq / hkv <= 16 && r % 32 == 0 && r <= 512 && packed_q(q) && rows(kA) && kB.stride(3) == 1);
  need(inv.is_cuda() && inv.device() == q.device() && inv.scalar_type() == at::kFloat && inv.numel() == 64 && inv.is_contiguous());
}
// recon_scores_kernel: four tiles of 16 tokens a step (two beyond rank 256), one workgroup per CU; otherwise the kernels that hold a kv
// head's factor in registers keep one, the generic kernel two or three.
// what recon_scores_kernel alone runs, of the operands that this layer takes
bool scores_alone(Ten kB, int64_t r, int64_t G) { return rows(kB) && (r <= 224 ? G <= 16 : (r == 320 || r == 448) && G <= 8); }
// Several kv heads a workgroup (recon_heads_impl.h) where that leaves enough workgroups: the splits, or 0
int heads_splits(bool packets, int64_t b, int64_t hkv, int64_t G, int64_t L, int64_t r, bool scores, int cus) {
  const int nh = packets ? xkv::recon_heads(r, hkv, G, scores) : 0;
  if (!nh || b * hkv * L < xkv::recon_heads_work(r, hkv)) return 0;
  const int S = balanced_splits(b, hkv / nh, L, 32, 1, cus);
  return b * (hkv / nh) * S >= xkv::RECON_HEADS_WORKGROUPS ? S : 0;
}
struct ReconSplits { int S; bool grouped; };   // grouped: cut for several kv heads a workgroup
ReconSplits score_splits(const Call& c, Ten kB, int64_t b, int64_t hkv, int64_t G, int64_t L, int64_t r) {
  if (const int S = heads_splits(rows(kB), b, hkv, G, L, r, true, c.cus)) return {S, true};
  if (scores_alone(kB, r, G) || xkv::recon_scores_pays(r, hkv, G, b * L))
    return {balanced_splits(b, hkv, L, r <= 256 ? 64 : 32, 1, c.cus), false};
  const bool resident = ring_rank(r) && G <= 8;
  return {balanced_splits(b, hkv, L, 32, resident || r > 256 ? 1 : r > 128 ? 2 : 3, c.cus), false};
}
// Scores and P.A in one kernel: one workgroup per CU; two only where the generic kernel, instantiated for the rank, does without a value
// tile of its own (us at one / two / three workgroups a CU, batch 1, 32 heads on 8, 9000 tokens: rank 64 32 / 42 / 50, rank 128 28 / 26 / 34,
// rank 192 31 / 29 / 33, rank 192 with values of its own 34 / 45 / 47).
int decode_splits(int64_t b, int64_t hkv, int64_t L, int64_t r, bool shared, int cus) {
  return balanced_splits(b, hkv, L, 32, shared && (r == 128 || r == 192) ? 2 : 1, cus);
}

// rope_decode(q [b,hq,128], kA, kB, vA, vB, o, sm_scale, inv_freq, pos_offset, two_pass) -> o | None
PyObject* rope_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 10, [&]() -> PyObject* {
    Ten q = T(a[0]), kA = T(a[1]), kB = T(a[2]), vA = T(a[3]), vB = T(a[4]), o = T(a[5]), inv = T(a[7]);
    const float scale = F(a[6]);
    const int64_t pos = I(a[8]);
    const bool may_two_pass = I(a[9]);
    same(q, {&kA, &kB, &vA, &vB});
    need(o.is_cuda() && o.device() == q.device());
    need(q.dim() == 3 && kA.dim() == 3 && kB.dim() == 4 && vA.dim() == 3 && vB.dim() == 4 && o.dim() == 3);
    const int64_t b = q.size(0), hq = q.size(1), L = kA.size(1), r = kA.size(2), hkv = kB.size(1), rv = vA.size(2);
    rope_operands(q, hq, q.size(2), kA, kB, inv);
    need(vA.size(0) == b && vA.size(1) == L && vB.size(0) == b && vB.size(1) == hkv && vB.size(2) == rv && rv % 64 == 0 && rv <= 512 && rows(vA));
    need(o.stride(2) == 1 && o.size(0) == b && o.size(1) == hq && o.size(2) == vB.size(3));
    without_gil([&] {
      Call c(q);
      const Up up = up_of(vB, hq, c.dt);
      const int odt = code_any(o);
      const bool shared = vA.data_ptr() == kA.data_ptr() && vA.sizes() == kA.sizes() && vA.strides() == kA.strides();
      const int64_t ws_bytes = p_xkv_recon_workspace_bytes(b, hkv, r, kB.stride(0)), ws = c.plan(ws_bytes);
      const float* invp = inv.data_ptr<float>();
      Splits s{0, 0, nullptr, nullptr};
      // over one basis that kernel is ahead of two passes too, and as exact (rank 256, 52000 tokens 51.0 / 44.7, 65536 57.5 / 50.4, 131072 90.0 / 79.1, 16 x 32768 283 / 256 us)
      const int S_heads = shared ? heads_splits(rows(kB), b, hkv, hq / hkv, L, r, false, c.cus) : 0;
      if (may_two_pass && !S_heads && (scores_alone(kB, r, hq / hkv) || (ring_rank(r) && hq / hkv <= 8)) && (joined() || hq <= 32) &&
          (ring_rank(rv) || (joined() && shared && (rv == 192 || rv == 128)))) {
        // scores first, then softmax and P.v_A in one stream for all heads.  The second pass reads the
        // scores in 16-byte packets, so their rows are whole packets: at another length the kernels get the padded one as the row's
        // and the true one as every sequence's (one fill, about 2 us).
        // Where there is no room for the scores, one kernel, which needs none.
        const int64_t row = (L + 3) / 4 * 4, one_kernel = c.used;
        at::Tensor lens;
        if (row != L) {
          lens = at::full({b}, L, c.opts.dtype(at::kInt));
          s.lens = lens.data_ptr<int32_t>();
        }
        s.S = scan_splits(c, b, head_groups(hq), L, true);
        const int64_t sc = c.plan(b * hq * row * 4), part = c.plan(s.rows(b, hq) * rv * 4), lse = c.plan(s.rows(b, hq) * 4);
        const int64_t mid = c.plan(rows_first(s.S, hq, up, rv, b) ? rows_bytes(b, hq, rv) : 0);
        if (c.try_alloc()) {
          const ReconSplits scores = score_splits(c, kB, b, hkv, hq / hkv, L, r);
          recon(c, q, kA, kB, nullptr, nullptr, nullptr, c.get<void>(sc), XKV_F32, scores.S, scores.grouped, b, hq, hkv, row, scale,
                invp, pos, ws_bytes ? c.get<void>(ws) : nullptr, ws_bytes, s.lens);
          check(p_xkv_softmax_pv_stage1(c.get<float>(sc), kv(vA, 0, rv), c.get<float>(part), c.get<float>(lse), nullptr, s.lens, b, hq, row, s.S,
                                        0, nullptr, c.dt, c.stream), "xkv_softmax_pv_stage1");
          merge(c, c.get<float>(part), c.get<float>(lse), o.data_ptr(), o.stride(0), o.stride(1), odt, &up, mid, s, b, hq, row, rv);
          return;
        }
        c.used = one_kernel;
        s.lens = nullptr;
      }
      s.S = S_heads ? S_heads : decode_splits(b, hkv, L, r, shared, c.cus);
      const int64_t part = c.plan(s.rows(b, hq) * rv * 4), lse = c.plan(s.rows(b, hq) * 4);
      const int64_t mid = c.plan(rows_first(s.S, hq, up, rv, b) ? rows_bytes(b, hq, rv) : 0);
      c.alloc();
      recon(c, q, kA, kB, &vA, c.get<float>(part), c.get<float>(lse), nullptr, 0, s.S, S_heads > 0, b, hq, hkv, L, scale, invp, pos,
            ws_bytes ? c.get<void>(ws) : nullptr, ws_bytes);
      merge(c, c.get<float>(part), c.get<float>(lse), o.data_ptr(), o.stride(0), o.stride(1), odt, &up, mid, s, b, hq, L, rv);
    });
    return give(a[5]);
  });
}

// rope_scores(q [b,hq,1,128], A, B, sm_scale, inv_freq, pos_offset, fp32_out) -> [b,hq,1,L] | None
PyObject* rope_scores(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 7, [&]() -> PyObject* {
    Ten q = T(a[0]), A = T(a[1]), B = T(a[2]), inv = T(a[4]);
    const float scale = F(a[3]);
    const int64_t pos = I(a[5]);
    const bool f32 = I(a[6]);
    same(q, {&A, &B});
    need(q.dim() == 4 && A.dim() == 3 && B.dim() == 4 && q.size(2) == 1);
    const int64_t b = q.size(0), hq = q.size(1), L = A.size(1), r = A.size(2), hkv = B.size(1);
    rope_operands(q, hq, q.size(3), A, B, inv);
    at::Tensor out;
    without_gil([&] {
      Call c(q);
      const int64_t ws_bytes = p_xkv_recon_workspace_bytes(b, hkv, r, B.stride(0)), ws = c.plan(ws_bytes);
      if (ws_bytes) c.alloc();
      out = at::empty({b, hq, 1, L}, f32 ? c.opts.dtype(at::kFloat) : c.opts);
      const ReconSplits s = score_splits(c, B, b, hkv, hq / hkv, L, r);
      recon(c, q, A, B, nullptr, nullptr, nullptr, out.data_ptr(), f32 ? XKV_F32 : c.dt, s.S, s.grouped, b, hq, hkv, L,
            scale, inv.data_ptr<float>(), pos, ws_bytes ? c.get<void>(ws) : nullptr, ws_bytes);
    });
    return THPVariable_Wrap(out);
  });
}

// gqa(q [b,hq,d], k [b,L,hkv,d], v | vA [b,L,rv], None | vB, o, sm_scale, lens | None, floor_wide, floor) -> o | None
PyObject* gqa(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 9, [&]() -> PyObject* {
    Ten q = T(a[0]), k = T(a[1]), v = T(a[2]), o = T(a[4]);
    const bool fact = a[3] != Py_None;
    const float scale = F(a[5]);
    const int floor_wide = I(a[7]), floor_head = I(a[8]);
    same(q, {&k, &v});
    need(o.is_cuda() && o.device() == q.device());
    need(q.dim() == 3 && k.dim() == 4 && v.dim() == (fact ? 3 : 4) && o.dim() == 3);
    const int64_t b = q.size(0), hq = q.size(1), d = q.size(2), L = k.size(1), hkv = k.size(2), dv = v.size(-1);
    need(b > 0 && L > 0 && hkv > 0 && k.size(0) == b && k.size(3) == d && v.size(0) == b && v.size(1) == L && hq % hkv == 0 && hq / hkv <= 32);
    need(d % 32 == 0 && dv % 64 == 0 && dv <= 512 && packed_q(q) && rows(k) && rows(v) && o.stride(2) == 1 && o.size(0) == b && o.size(1) == hq);
    if (!fact) need(v.size(2) == hkv && dv == d && o.size(2) == dv);
    const at::Tensor lens = lens_of(a[6], q, b);
    Ten vB = fact ? T(a[3]) : v;
    without_gil([&] {
      Call c(q);
      const int odt = code_any(o);
      Up up{};
      if (fact) {
        same(q, {&vB});
        need(vB.dim() == 4 && vB.size(0) == b && vB.size(1) == hkv && vB.size(2) == dv && o.size(2) == vB.size(3));
        up = up_of(vB, hq, c.dt);
      }
      // 2, 4 or 8 kv heads of 128 side by side in a token row: stage 1 serves every head of a split from one workgroup, one per CU
      const bool rows128 = (hkv == 8 || hkv == 4 || hkv == 2) && d == 128 && hq <= 32 && k.stride(2) == d && k.stride(1) >= hkv * d;
      const bool planned = lens.defined() && b > 1;   // one sequence is cut into the splits of the longest it may be
      const bool in_row = rows128 && (fact ? ring_rank(dv) && v.stride(1) >= dv
                                           : v.stride(2) == d && v.stride(1) >= hkv * d && xkv::head_rows_pay(hkv, hq, b, L, planned, false));
      // 512-wide token rows of other heads beside 512-wide value rows: the same form, against a block-diagonal query
      const bool wide4 = !in_row && fact && hkv * d == 512 && dv == 512 && hq <= 32 && k.stride(2) == d;
      const bool wide = in_row || wide4;
      const int per_cu = wide ? 1 : 2, groups = wide ? 1 : (int)hkv, longest_floor = wide ? floor_wide : floor_head;
      need(longest_floor > 0);
      int floor = split_floor(b, groups, L, per_cu, c.cus, fact);
      if (in_row && !fact) floor = xkv::head_rows_floor(hkv, b * L, floor);
      floor = std::min(longest_floor, floor);
      Ragged rg{};
      Splits s{0, 0, nullptr, nullptr};
      if (planned) rg = ragged(c, s, b, groups, L, floor, per_cu);
      else s.S = std::min(balanced_splits(b, groups, L, 32, per_cu, c.cus), cdiv(L, floor));
      if (lens.defined()) s.lens = lens.data_ptr<int32_t>();
      const int64_t part = c.plan(s.rows(b, hq) * dv * 4), lse = c.plan(s.rows(b, hq) * 4), bd = c.plan(wide4 ? b * hq * 512 * 2 : 0);
      const int64_t mid = c.plan(fact && rows_first(s.S, hq, up, dv, b) ? rows_bytes(b, hq, dv) : 0);
      c.alloc();
      if (planned) write_plan(c, s, rg, b);
      const void* qp = q.data_ptr();
      if (wide4) {
        check(p_xkv_blockdiag_q(qp, c.get<void>(bd), b, hq, hkv, d, c.dt, c.stream), "xkv_blockdiag_q");
        qp = c.get<void>(bd);
      }
      check(p_xkv_latent_stage1({qp, wide4 ? 512 : (int)d}, nullptr, NO_Q, wide4 ? kv(k, 0, 512) : kv(k, k.stride(2), d), NO_KV,
                                kv(v, fact ? 0 : v.stride(2), dv), c.get<float>(part), c.get<float>(lse), nullptr, 0, nullptr, s.lens, b, hq,
                                wide4 ? 1 : hkv, L, s.n(), s.cap, s.plan, scale, 0.f, c.dt, c.stream), "xkv_latent_stage1");
      merge(c, c.get<float>(part), c.get<float>(lse), o.data_ptr(), o.stride(0), o.stride(1), odt, fact ? &up : nullptr, mid, s, b, hq, L, dv);
    });
    return give(a[4]);
  });
}

// mla(q_nope [b,H,w], q_rope [b,H,e], kv [b,L,1,r], None | kv_B [b,1,r,w], k_rope [b,L,1,e], sm_scale) -> [b,H,w] | None
PyObject* mla(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 6, [&]() -> PyObject* {
    Ten qn = T(a[0]), qr = T(a[1]), C = T(a[2]), R = T(a[4]);
    const bool fact = a[3] != Py_None;
    const float scale = F(a[5]);
    same(qn, {&qr, &C, &R});
    need(qn.dim() == 3 && qr.dim() == 3 && C.dim() == 4 && R.dim() == 4 && C.size(2) == 1 && R.size(2) == 1);
    const int64_t b = qn.size(0), hq = qn.size(1), w = qn.size(2), e = qr.size(2), L = C.size(1), r = C.size(3);
    need(b > 0 && L > 0 && hq > 0 && C.size(0) == b && R.size(0) == b && R.size(1) == L && qr.size(0) == b && qr.size(1) == hq && R.size(3) == e);
    need(r % 64 == 0 && r <= 512 && e % 32 == 0 && e > 0 && e <= 128 && packed_q(qn) && packed_q(qr) && rows(C) && rows(R));
    Ten B = fact ? T(a[3]) : C;
    at::Tensor o;
    without_gil([&] {
      Call c(qn);
      Up up{};
      if (fact) {
        same(qn, {&B});
        need(B.dim() == 4 && B.size(0) == b && B.size(1) == 1 && B.size(2) == r && B.size(3) == w && w % 8 == 0 && w <= 512 && rows(B));
        up = up_of(B, hq, c.dt);
      } else {
        need(w == r);
      }
      const int groups = head_groups(hq);
      Splits s{scan_splits(c, b, groups, L, e == 64 && (r == 512 || (fact && ring_rank(r)))), 0, nullptr, nullptr};
      const int64_t hi = c.plan(fact ? b * hq * r * 2 : 0), lo = c.plan(fact ? b * hq * r * 2 : 0);
      const int64_t part = c.plan(s.rows(b, hq) * r * 4), lse = c.plan(s.rows(b, hq) * 4);
      const int64_t mid = c.plan(fact && rows_first(s.S, hq, up, r, b) ? rows_bytes(b, hq, r) : 0);
      c.alloc();
      o = at::empty({b, hq, w}, c.opts);
      const void *q_hi = qn.data_ptr(), *q_lo = nullptr;
      if (fact) {
        absorb(c, q_hi, B, c.get<void>(hi), c.get<void>(lo), b, hq, w, r);
        q_hi = c.get<void>(hi);
        q_lo = c.get<void>(lo);
      }
      check(p_xkv_latent_stage1({q_hi, (int)r}, q_lo, {qr.data_ptr(), (int)e}, kv(C, 0, r), kv(R, 0, e), kv(C, 0, r), c.get<float>(part),
                                c.get<float>(lse), nullptr, 0, nullptr, nullptr, b, hq, groups, L, s.S, 0, nullptr, scale, 0.f, c.dt, c.stream),
            "xkv_latent_stage1");
      merge(c, c.get<float>(part), c.get<float>(lse), o.data_ptr(), hq * w, w, c.dt, fact ? &up : nullptr, mid, s, b, hq, L, r);
    });
    return THPVariable_Wrap(o);
  });
}

// prefix_tail(q [b,H,w], kA, kB [b,1,r,w], vA, vB [b,1,rv,w], k_tail [b,Lt,1,w], v_tail, sm_scale, logit_cap) -> [b,H,w] | None
PyObject* prefix_tail(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 9, [&]() -> PyObject* {
    Ten q = T(a[0]), kA = T(a[1]), kB = T(a[2]), vA = T(a[3]), vB = T(a[4]), kT = T(a[5]), vT = T(a[6]);
    const float scale = F(a[7]), logit_cap = F(a[8]);
    same(q, {&kA, &kB, &vA, &vB, &kT, &vT});
    need(q.dim() == 3 && kA.dim() == 3 && kB.dim() == 4 && vA.dim() == 3 && vB.dim() == 4 && kT.dim() == 4 && vT.dim() == 4);
    const int64_t b = q.size(0), hq = q.size(1), w = q.size(2), L = kA.size(1), r = kA.size(2), rv = vA.size(2), Lt = kT.size(1);
    need(b > 0 && L > 0 && Lt > 0 && kB.size(1) == 1 && vB.size(1) == 1 && kT.size(2) == 1 && vT.size(2) == 1);
    need(kA.size(0) == b && kB.size(0) == b && vA.size(0) == b && vB.size(0) == b && kT.size(0) == b && vT.size(0) == b && vA.size(1) == L && vT.size(1) == Lt);
    need(kB.size(2) == r && kB.size(3) == w && vB.size(2) == rv && kT.size(3) == w && w != 576 && w != 288 && vB.size(3) == vT.size(3));
    const int64_t dv = vT.size(3);
    need(r % 32 == 0 && rv % 64 == 0 && rv <= 512 && w % 32 == 0 && w <= 512 && dv % 64 == 0 && dv <= 512);
    need(packed_q(q) && rows(kA) && rows(kB) && rows(vA) && rows(kT) && rows(vT));
    at::Tensor o;
    without_gil([&] {
      Call c(q);
      const Up up = up_of(vB, hq, c.dt);
      const int groups = head_groups(hq);
      const bool shared = vA.data_ptr() == kA.data_ptr() && vA.strides() == kA.strides() && rv == r;
      Splits s1{scan_splits(c, b, groups, L, ring_rank(r)), 0, nullptr, nullptr};
      // the tail: as many splits as it has 32-token blocks, up to 32 of equal numbers of them.  In launches of its own at most four, every one of
      // them live; a cap states the count, because the rows are one more: row 0 is the merged, up-projected prefix with its log-sum-exp
      const bool join = joined();
      const int blocks = cdiv(Lt, 32), per = cdiv(blocks, join ? 32 : 4), S2 = cdiv(blocks, per), rows2 = S2 + (join ? 0 : 1);
      const bool first = xkv::merge_tail_rows_first(s1.S, hq, up.hkv, rv);
      const int64_t hi = c.plan(b * hq * r * 2), lo = c.plan(b * hq * r * 2), part1 = c.plan(b * hq * s1.S * rv * 4), lse1 = c.plan(b * hq * s1.S * 4);
      const int64_t mid = c.plan((join ? first : rows_first(s1.S, hq, up, rv, b)) ? rows_bytes(b, hq, rv) : 0), part2 = c.plan(b * hq * rows2 * dv * 4), lse2 = c.plan(b * hq * rows2 * 4);
      c.alloc();
      o = at::empty({b, hq, dv}, c.opts);
      // the query absorbed and the tail attended to in one launch: neither depends on the other
      if (!join) absorb(c, q.data_ptr(), kB, c.get<void>(hi), c.get<void>(lo), b, hq, w, r);
      else check(p_xkv_absorb_q_tail(q.data_ptr(), kB.data_ptr(), c.get<void>(hi), c.get<void>(lo), b, hq, groups, w, r, kB.stride(0), 0, kB.stride(2),
                                kv(kT, 0, w), kv(vT, 0, dv), Lt, S2, c.get<float>(part2), c.get<float>(lse2), scale, logit_cap, c.dt, c.stream),
            "xkv_absorb_q_tail");
      check(p_xkv_latent_stage1({c.get<void>(hi), (int)r}, c.get<void>(lo), NO_Q, kv(kA, 0, r), NO_KV, shared ? kv(kA, 0, r) : kv(vA, 0, rv),
                                c.get<float>(part1), c.get<float>(lse1), nullptr, 0, nullptr, nullptr, b, hq, groups, L, s1.S, 0, nullptr, scale,
                                logit_cap, c.dt, c.stream), "xkv_latent_stage1");
      if (!join) {
        float *pf = c.get<float>(part2), *lf = c.get<float>(lse2);
        merge(c, c.get<float>(part1), c.get<float>(lse1), pf, hq * rows2 * dv, rows2 * dv, XKV_F32, &up, mid, s1, b, hq, L, rv, lf, hq * rows2, rows2);
        check(p_xkv_latent_stage1({q.data_ptr(), (int)w}, nullptr, NO_Q, kv(kT, 0, w), NO_KV, kv(vT, 0, dv), pf + dv, lf + 1, nullptr, 0, nullptr,
                                  nullptr, b, hq, groups, Lt, rows2, 32 * per, nullptr, scale, logit_cap, c.dt, c.stream), "xkv_latent_stage1");
        merge(c, pf, lf, o.data_ptr(), hq * dv, dv, c.dt, nullptr, 0, {rows2, 0, nullptr, nullptr}, b, hq, 32 * rows2, dv);   // every row live
        return;
      }
      const float *rows = c.get<float>(part1), *rows_lse = c.get<float>(lse1);
      int n_rows = s1.S, len = L;
      if (first) {   // many splits: merged by the whole chip, then one row per head
        float* m = c.get<float>(mid);
        check(p_xkv_merge_stage2(rows, rows_lse, m, nullptr, 0, 0, 0, 0, XKV_BF16, nullptr, nullptr, b, hq, hq, L, s1.S, 0, nullptr, rv, hq * rv, rv,
                                 XKV_F32, m + b * hq * rv, hq, 1, c.stream), "xkv_merge_stage2");
        rows = m; rows_lse = m + b * hq * rv; n_rows = 1; len = 32;
      }
      check(p_xkv_merge_stage2_tail(rows, rows_lse, o.data_ptr(), up.p, up.sb, up.sh, up.sr, up.d_out, c.dt, b, hq, up.hkv, len, n_rows, rv,
                                    c.get<float>(part2), c.get<float>(lse2), S2, hq * dv, dv, c.stream), "xkv_merge_stage2_tail");
    });
    return THPVariable_Wrap(o);
  });
}

// decode_splits(batch, kv heads, kv_len, rank, shared, cus) -> int
PyObject* py_decode_splits(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 6, [&]() -> PyObject* { return PyLong_FromLong(decode_splits(I(a[0]), I(a[1]), I(a[2]), I(a[3]), I(a[4]), I(a[5]))); });
}

// head_rows(heads, hq, batch, kv_len, ragged) -> bool and head_rows_floor(heads, tokens, floor) -> int (head_rows.h)
PyObject* py_head_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 5, [&]() -> PyObject* { return PyBool_FromLong(xkv::head_rows_pay(I(a[0]), I(a[1]), I(a[2]), I(a[3]), I(a[4]), false)); });
}
PyObject* py_head_rows_floor(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 3, [&]() -> PyObject* { return PyLong_FromLong(xkv::head_rows_floor(I(a[0]), I(a[1]), I(a[2]))); });
}
// recon_scores_pays(rank, kv heads, heads per kv head, tokens) -> bool (recon_groups.h)
PyObject* py_recon_scores_pays(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject* { return PyBool_FromLong(xkv::recon_scores_pays(I(a[0]), I(a[1]), I(a[2]), I(a[3]))); });
}
// merge_rows_first(splits, heads, kv heads, width, batch, columns) -> bool (merge_rule.h)
PyObject* py_merge_rows_first(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 6, [&]() -> PyObject* { return PyBool_FromLong(xkv::merge_rows_first(I(a[0]), I(a[1]), I(a[2]), I(a[3]), I(a[4]), I(a[5]))); });
}
// split_floor(batch, groups, kv_len, per_cu, cus, up) -> int
PyObject* py_split_floor(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 6, [&]() -> PyObject* { return PyLong_FromLong(split_floor(I(a[0]), I(a[1]), I(a[2]), I(a[3]), I(a[4]), I(a[5]))); });
}

// ragged_target(batch, groups, per_cu, cus) -> int
PyObject* py_ragged_target(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject* { return PyLong_FromLong(ragged_target(I(a[0]), I(a[1]), I(a[2]), I(a[3]))); });
}

// balanced_splits(batch, groups, kv_len, tile, per_cu, cus) -> int
PyObject* py_balanced_splits(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 6, [&]() -> PyObject* {
    return PyLong_FromLong(balanced_splits(I(a[0]), I(a[1]), I(a[2]), I(a[3]), I(a[4]), I(a[5])));
  });
}

// init(path of libxkv_hip.so): the library is loaded already; take the addresses of its entry points
PyObject* init(PyObject*, PyObject* path) {
  const char* p = PyUnicode_AsUTF8(path);
  if (!p) return nullptr;
  void* h = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  if (!h) { PyErr_Format(PyExc_RuntimeError, "cannot load %s: %s", p, dlerror()); return nullptr; }
  const auto version = reinterpret_cast<decltype(&xkv_abi_version)>(dlsym(h, "xkv_abi_version"));
  if (!version || version() != XKV_ABI_VERSION) {
    PyErr_Format(PyExc_RuntimeError, "%s has ABI %d, the native host layer is built for %d; rebuild", p, version ? version() : 0, XKV_ABI_VERSION);
    return nullptr;
  }
#define XKV_RESOLVE(name)                                                                  \
  p_##name = reinterpret_cast<decltype(p_##name)>(dlsym(h, #name));                        \
  if (!p_##name) { PyErr_Format(PyExc_RuntimeError, "%s has no " #name, p); return nullptr; }
  XKV_SYMBOLS(XKV_RESOLVE)
#undef XKV_RESOLVE
#define XKV_RESOLVE(name) p_##name = reinterpret_cast<decltype(p_##name)>(dlsym(h, #name));
  XKV_OPTIONAL_SYMBOLS(XKV_RESOLVE)
#undef XKV_RESOLVE
  Py_RETURN_NONE;
}

#define XKV_FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"init", init, METH_O, nullptr},       XKV_FAST("balanced_splits", py_balanced_splits), XKV_FAST("nope_decode", nope_decode), XKV_FAST("ragged_target", py_ragged_target),
    XKV_FAST("split_floor", py_split_floor), XKV_FAST("decode_splits", py_decode_splits), XKV_FAST("head_rows", py_head_rows),
    XKV_FAST("head_rows_floor", py_head_rows_floor), XKV_FAST("recon_scores_pays", py_recon_scores_pays),
    XKV_FAST("merge_rows_first", py_merge_rows_first),
    XKV_FAST("nope_scores", nope_scores),  XKV_FAST("rope_decode", rope_decode),            XKV_FAST("rope_scores", rope_scores),
    XKV_FAST("gqa", gqa),                  XKV_FAST("mla", mla),                            XKV_FAST("prefix_tail", prefix_tail),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_xkv_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__xkv_host(void) { return PyModule_Create(&module); }
