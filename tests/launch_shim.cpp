// The entry points that the native host layer calls, in front of libxkv_hip.so (tests load this in the library's place): each one
// counts the calls made with the Python interpreter locked and, when poisoning is on, fills the LDS of the whole device before a
// stage-1 launch.  shim_recon_splits: the splits that the last reconstructing launch was given.
#include <dlfcn.h>

#include "../include/xkv_hip.h"

static void* real_lib;
static int (*gil_held)();
extern "C" {
int shim_launches, shim_stage1, shim_locked_calls, shim_poison, shim_poisoned, shim_recon_splits;
int shim_init(const char* path) {
  real_lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  gil_held = (int (*)())dlsym(RTLD_DEFAULT, "PyGILState_Check");
  return real_lib && gil_held ? 0 : -1;
}
}

template <typename F> static F* real(const char* name) { return (F*)dlsym(real_lib, name); }
static void before(bool stage1, void* stream) {
  ++shim_launches;
  if (gil_held()) ++shim_locked_calls;
  if (!stage1) return;
  ++shim_stage1;
  if (shim_poison && real<decltype(xkv_poison_lds)>("xkv_poison_lds")(0x7FFF7FFF, nullptr, stream) == 0)   // a NaN as fp16, bf16 and fp32
    ++shim_poisoned;
}
#define FORWARD(name, stage1, params, args) \
  extern "C" int name params { before(stage1, stream); return real<decltype(name)>(#name) args; }

extern "C" int xkv_abi_version(void) { return real<decltype(xkv_abi_version)>("xkv_abi_version")(); }
extern "C" const char* xkv_error_string(int code) { return real<decltype(xkv_error_string)>("xkv_error_string")(code); }
extern "C" int64_t xkv_recon_workspace_bytes(int b, int hkv, int r, int64_t s) {
  return real<decltype(xkv_recon_workspace_bytes)>("xkv_recon_workspace_bytes")(b, hkv, r, s);
}
FORWARD(xkv_absorb_q, false, (const void* q, const void* B, void* hi, void* lo, int b, int hq, int hkv, int d, int r, int64_t s0, int64_t s1,
                              int64_t s2, int dt, void* stream), (q, B, hi, lo, b, hq, hkv, d, r, s0, s1, s2, dt, stream))
FORWARD(xkv_blockdiag_q, false, (const void* q, void* out, int b, int hq, int hkv, int d, int dt, void* stream), (q, out, b, hq, hkv, d, dt, stream))
FORWARD(xkv_plan_splits, false, (const int32_t* kl, const int32_t* ns, int b, int S, int fl, int target, int32_t* plan, void* stream),
        (kl, ns, b, S, fl, target, plan, stream))
FORWARD(xkv_latent_stage1, true, (xkv_q_operand qn, const void* lo, xkv_q_operand qr, xkv_kv_operand C, xkv_kv_operand R, xkv_kv_operand V,
                                  float* part, float* lse, void* sc, int sdt, const int32_t* ns, const int32_t* kl, int b, int hq, int g, int L,
                                  int S, int cap, const int32_t* plan, float scale, float lc, int dt, void* stream),
        (qn, lo, qr, C, R, V, part, lse, sc, sdt, ns, kl, b, hq, g, L, S, cap, plan, scale, lc, dt, stream))
FORWARD(xkv_softmax_pv_stage1, true, (const float* sc, xkv_kv_operand V, float* part, float* lse, const int32_t* ns, const int32_t* kl, int b,
                                      int hq, int L, int S, int cap, const int32_t* plan, int dt, void* stream),
        (sc, V, part, lse, ns, kl, b, hq, L, S, cap, plan, dt, stream))
FORWARD(xkv_recon_stage1, true, (const void* q, xkv_kv_operand A, const void* B, int64_t s0, int64_t s1, int64_t s2, xkv_kv_operand V, float* part,
                                 float* lse, void* sc, int sdt, const int32_t* ns, const int32_t* kl, int b, int hq, int hkv, int L, int S,
                                 float scale, int rope, const float* inv, int64_t pos, const void* tab, int64_t st, void* ws, int64_t wb, int dt,
                                 void* stream),
        (q, A, B, s0, s1, s2, V, part, lse, sc, sdt, ns, kl, b, hq, hkv, L, shim_recon_splits = S, scale, rope, inv, pos, tab, st, ws, wb, dt, stream))
FORWARD(xkv_merge_stage2, false, (const float* part, const float* lse, void* out, const void* vB, int64_t v0, int64_t v1, int64_t v2, int d, int vdt,
                                  const int32_t* ns, const int32_t* kl, int b, int hq, int hkv, int L, int S, int cap, const int32_t* plan, int dv,
                                  int64_t o0, int64_t o1, int odt, float* lo, int64_t l0, int64_t l1, void* stream),
        (part, lse, out, vB, v0, v1, v2, d, vdt, ns, kl, b, hq, hkv, L, S, cap, plan, dv, o0, o1, odt, lo, l0, l1, stream))
