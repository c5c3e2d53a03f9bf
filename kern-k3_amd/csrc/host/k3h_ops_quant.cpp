// Typed wrappers: per-tensor fp8 pair (manifest op quant_fp8_tensor,
// k3-tp4-prefill-16k.json:407194: amax then apply, both grid (2048), block 256).
#include "k3h_internal.h"

namespace {
const char* quant_key(int v2) { return v2 ? "k3_quant_fp8_pair_v2" : "k3_quant_fp8_pair"; }
// k3h_quant_fp8_once (one launch that keeps most of x on the chip between the passes): one
// workgroup per CU, the manifest's nb only.
constexpr int kOnceNb = 2048, kOnceGrid = 256, kOnceBlock = 1024;
// below, its fixed cost exceeds the second read of x (back to back over three sets 20.8 ->
// 18.7 us at n = 25 M, 18.0 -> 17.8 at 21 M)
constexpr int kOnceMinN = 24 << 20;
// How long a workgroup waits for the others' partials before it takes the missing ones
// itself, in ticks of the 100 MHz clock: twice the undisturbed meeting (4 us), and an eighth
// of the reading time, by which the workgroups' ends differ (at n = 537 M 414 us; 450 with 8
// us for every n).  Longer only costs the call whose workgroups are kept out (beside a
// one-wave kernel at n = 25 M: 54 us at 8 us, 77 at 30).
int once_spin_ticks(int n) { return 800 + (n >> 18); }
bool quant_args_ok(const void* x, int n, const void* partials, int nb) {
  return n >= 0 && nb >= 1 && nb <= 65535 && k3h_okp(x, 16) && k3h_okp(partials, 4);
}
}  // namespace

extern "C" {

K3H_API int k3h_quant_fp8_amax(k3h_ctx_t ctx, void* stream, int v2, const void* x, int n,
                               float* partials, int nb) {
  if (!ctx || !quant_args_ok(x, n, partials, nb)) return K3H_EINVAL;
  K3hArgs a;
  a.ptr(x).i32(n).ptr(partials);
  return k3h_run(ctx, quant_key(v2), v2 ? "kern_quant_fp8_amax_v2" : "kern_quant_fp8_amax",
                 (uint32_t)nb, 1, 1, 256, stream, a);
}

K3H_API int k3h_quant_fp8_apply(k3h_ctx_t ctx, void* stream, int v2, const void* x, void* y,
                                int n, const float* partials, int nb, float* scale_out) {
  if (!ctx || !quant_args_ok(x, n, partials, nb) || !k3h_okp(y, 8)) return K3H_EINVAL;
  if (scale_out && !k3h_aligned(scale_out, 4)) return K3H_EINVAL;
  K3hArgs a;
  a.ptr(x).ptr(y).i32(n).ptr(partials).i32(nb).ptr(scale_out);
  return k3h_run(ctx, quant_key(v2), v2 ? "kern_quant_fp8_apply_v2" : "kern_quant_fp8_apply",
                 (uint32_t)nb, 1, 1, 256, stream, a);
}

K3H_API int k3h_quant_fp8_tensor(k3h_ctx_t ctx, void* stream, int v2, const void* x, void* y,
                                 float* scale_out, float* partials, int n, int nb) {
  if (!ctx || !quant_args_ok(x, n, partials, nb) || !k3h_okp(y, 8) ||
      (scale_out && !k3h_aligned(scale_out, 4)))
    return K3H_EINVAL;
  if (v2 && nb == kOnceNb && n >= kOnceMinN) {
    int hold = 0;
    const int rc = k3h_ctx_resident(ctx, quant_key(1), "k3h_quant_fp8_once", kOnceBlock, &hold);
    if (rc != K3H_OK) return rc;
    if (hold >= kOnceGrid) {  // the whole grid at once, as the wait for the partials assumes
      K3hArgs m;
      m.ptr(partials);
      const int r = k3h_run(ctx, quant_key(1), "k3h_quant_fp8_mark", kOnceNb / kOnceBlock, 1, 1,
                            kOnceBlock, stream, m);
      if (r != K3H_OK) return r;
      K3hArgs a;
      a.ptr(x).ptr(y).i32(n).ptr(partials).ptr(scale_out).i32(once_spin_ticks(n));
      return k3h_run(ctx, quant_key(1), "k3h_quant_fp8_once", kOnceGrid, 1, 1, kOnceBlock, stream, a);
    }
  }
  const int r = k3h_quant_fp8_amax(ctx, stream, v2, x, n, partials, nb);
  if (r != K3H_OK) return r;
  return k3h_quant_fp8_apply(ctx, stream, v2, x, y, n, partials, nb, scale_out);
}

}  // extern "C"
