// The MoE layer's forward and backward as one call each: the entry points of
// abacus_moe.h in the order of moe.py:60-86 and its autograd, on buffers carved
// out of a few allocations (LayerPlan).  At small batches the layer's time is the
// host's: with one foreign call and some twenty allocations per direction less, an
// fp32 layer of 256 tokens, forward + backward, went 356 -> 228 us (same host).
#include "common.h"

namespace {

// The plan's int64 fields, in the order of abacus_amd/moe.py's _PLAN_FIELDS.
// Offsets are bytes into the named buffer; -1: absent.
struct LayerPlan {
  int64_t T, D, E, K, M, ld, dtype;
  int64_t decode;  // 1: small batch without gradients (abacus_experts_decode_fwd)
  // route buffer (kept with the module's routing record)
  int64_t logits, weights, indices, counts, offsets, pos, perm;
  // keep buffer (saved for the backward)
  int64_t idx, score, wt, gate_pad, up_pad, xp, gate, up, h, y;
  // forward scratch
  int64_t hist, base, ws, ws_bytes;
  // backward scratch
  int64_t dy, dlogit, dgate, dup, dxp, ctr, bws, bws_bytes, partial;
};

char* at(void* base, int64_t off) { return off < 0 ? nullptr : (char*)base + off; }
const char* at(const void* base, int64_t off) { return off < 0 ? nullptr : (const char*)base + off; }

#define RUN(call)            \
  do {                       \
    const int rc_ = (call);  \
    if (rc_) return rc_;     \
  } while (0)

}  // namespace

extern "C" int64_t abacus_layer_plan_fields(void) { return sizeof(LayerPlan) / sizeof(int64_t); }

extern "C" int abacus_layer_fwd(const int64_t* plan, const void* x, const void* w_DE, const void* w_gate,
                                const void* w_up, const void* w_down, void* bias, double route_scale,
                                double bias_speed, int update_bias, void* route, void* keep, void* scratch, void* out,
                                void* s) {
  ABACUS_CHECK_ARG(plan && route && keep && scratch && out, "layer_fwd: null buffer");
  const LayerPlan& p = *reinterpret_cast<const LayerPlan*>(plan);
  const int64_t R = p.T * p.K;
  const int dt = (int)p.dtype;
  int32_t* idx = (int32_t*)at(keep, p.idx);
  int32_t* hist = (int32_t*)at(scratch, p.hist);
  int32_t* offsets = (int32_t*)at(route, p.offsets);
  int32_t* pos = (int32_t*)at(route, p.pos);
  void* weights = at(route, p.weights);
  char *xp = at(keep, p.xp), *h = at(keep, p.h), *y = at(keep, p.y);
  RUN(abacus_moe_router_fwd(x, w_DE, bias, p.T, p.D, p.E, p.K, route_scale, dt, at(route, p.logits), weights,
                            (int64_t*)at(route, p.indices), idx, at(keep, p.score), hist, at(keep, p.wt), s));
  RUN(abacus_moe_dispatch(hist, x, idx, p.T, p.D, p.E, p.K, update_bias ? bias : nullptr,
                          update_bias ? bias_speed : 0.0, dt, (int32_t*)at(route, p.counts), offsets, pos,
                          (int32_t*)at(route, p.perm), xp, (int32_t*)at(scratch, p.base), s));
  if (p.decode) {
    RUN(abacus_experts_decode_fwd(xp, w_gate, w_up, w_down, offsets, R, p.D, p.M, p.E, dt, p.ld, h, y,
                                  at(scratch, p.ws), p.ws_bytes, s));
  } else {
    if (p.gate_pad >= 0) {
      RUN(abacus_experts_pad_columns(w_gate, p.E * p.D, p.M, p.ld, at(keep, p.gate_pad), s));
      RUN(abacus_experts_pad_columns(w_up, p.E * p.D, p.M, p.ld, at(keep, p.up_pad), s));
      w_gate = at(keep, p.gate_pad);
      w_up = at(keep, p.up_pad);
    }
    RUN(abacus_moe_gateup_fwd(xp, w_gate, w_up, offsets, R, p.D, p.ld, p.E, dt, at(keep, p.gate), at(keep, p.up), h, s));
    if (p.ld != p.M)
      RUN(abacus_experts_down_fwd(h, w_down, offsets, R, p.M, p.ld, p.D, p.E, y, at(scratch, p.ws), p.ws_bytes, s));
    else
      RUN(abacus_moe_down_fwd(h, w_down, offsets, R, p.M, p.D, p.E, dt, y, at(scratch, p.ws), p.ws_bytes, s));
  }
  return abacus_moe_combine_fwd(y, weights, idx, pos, p.T, p.D, p.K, dt, out, s);
}

extern "C" int abacus_layer_bwd(const int64_t* plan, const void* x, const void* w_DE, const void* w_gate,
                                const void* w_up, const void* w_down, double route_scale, const void* route,
                                const void* keep, const void* dout, void* scratch, void* dx, void* dw_DE,
                                void* dw_gate, void* dw_up, void* dw_down, void* s) {
  ABACUS_CHECK_ARG(plan && route && keep && dout && scratch, "layer_bwd: null buffer");
  ABACUS_CHECK_ARG(!dw_gate == !dw_up, "layer_bwd: dw_gate and dw_up come together");
  const LayerPlan& p = *reinterpret_cast<const LayerPlan*>(plan);
  const int64_t R = p.T * p.K;
  const int dt = (int)p.dtype;
  const int32_t* idx = (const int32_t*)at(keep, p.idx);
  const int32_t* offsets = (const int32_t*)at(route, p.offsets);
  const int32_t* pos = (const int32_t*)at(route, p.pos);
  const char *xp = at(keep, p.xp), *gate = at(keep, p.gate), *up = at(keep, p.up), *h = at(keep, p.h);
  char *dy = at(scratch, p.dy), *dgate = at(scratch, p.dgate), *dup = at(scratch, p.dup), *dxp = at(scratch, p.dxp);
  float* dlogit = (float*)at(scratch, p.dlogit);
  int32_t* ctr = (int32_t*)at(scratch, p.ctr);
  RUN(abacus_moe_combine_bwd(dout, at(keep, p.y), at(route, p.weights), at(keep, p.score), pos, p.T, p.D, p.K,
                             route_scale, dt, dy, dlogit, s));
  const bool pitched = p.ld != p.M;
  if (pitched) {
    w_gate = at(keep, p.gate_pad);
    w_up = at(keep, p.up_pad);
    RUN(abacus_experts_down_bwd(dy, w_down, gate, up, h, offsets, R, p.M, p.ld, p.D, p.E, dgate, dup, dw_down, ctr, s));
  } else if (dw_down) {
    RUN(abacus_moe_down_bwd(dy, w_down, gate, up, h, offsets, R, p.M, p.D, p.E, dt, dgate, dup, dw_down, ctr, s));
  } else {
    RUN(abacus_moe_down_bwd_dgrad(dy, w_down, gate, up, offsets, R, p.M, p.D, p.E, dt, dgate, dup, s));
  }
  const bool want_x = dx != nullptr, want_w = dw_gate != nullptr;
  if ((want_x || want_w) && pitched) {
    RUN(abacus_experts_gateup_bwd(dgate, dup, w_gate, w_up, xp, offsets, R, p.D, p.M, p.ld, p.E, dt, want_x ? dxp : nullptr,
                                  dw_gate, dw_up, ctr, at(scratch, p.bws), p.bws_bytes, s));
  } else if (want_x && want_w && p.bws_bytes > 0) {
    RUN(abacus_experts_gateup_bwd(dgate, dup, w_gate, w_up, xp, offsets, R, p.D, p.M, p.ld, p.E, dt, dxp, dw_gate, dw_up,
                                  ctr, at(scratch, p.bws), p.bws_bytes, s));
  } else if (want_x && want_w) {
    RUN(abacus_moe_gateup_bwd(dgate, dup, w_gate, w_up, xp, offsets, R, p.D, p.M, p.E, dt, dxp, dw_gate, dw_up, ctr, s));
  } else if (want_x) {
    RUN(abacus_moe_gateup_bwd_dgrad(dgate, dup, w_gate, w_up, offsets, R, p.D, p.M, p.E, dt, dxp, s));
  } else if (want_w) {
    RUN(abacus_moe_gateup_bwd_wgrad(xp, dgate, dup, offsets, R, p.D, p.M, p.E, dt, dw_gate, dw_up, ctr, s));
  }
  if (dx)  // (w_DE = NULL: wt holds the forward's transposed router weights)
    RUN(abacus_moe_unpermute_bwd(dxp, dlogit, idx, pos, nullptr, const_cast<char*>(at(keep, p.wt)), p.T, p.D, p.E, p.K,
                                 dt, dx, s));
  if (dw_DE)
    RUN(abacus_moe_router_wgrad(x, dlogit, idx, p.T, p.D, p.E, p.K, dt, (float*)at(scratch, p.partial), dw_DE, s));
  return 0;
}
