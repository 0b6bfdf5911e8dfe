// A whole forward or backward of the layer in one call: the launches of the
// staged entry points, in order, on one stream. A small layer is bound by the
// host between its launches (a single-token forward launches four kernels,
// 30 us of GPU time; issued one entry point at a time from Python they took
// 60 us of host time, from one call 30).
#include "common.h"

namespace {

// Carves 256-byte aligned pieces from a scratch buffer.
struct Carver {
  char* base;
  size_t used = 0;
  template <class T>
  T* take(size_t bytes) {
    T* p = reinterpret_cast<T*>(base + used);
    used += mm_align_up(bytes, 256);
    return p;
  }
};

struct ForwardScratch {
  int32_t *counts, *offsets, *send_route, *send_token, *route_to_send;
  float* weight_perm;
  void* tiles;
  size_t tiles_bytes;
  uint16_t *act, *y;
  void* route_ws;
  size_t route_ws_bytes, bytes;

  // keep_tables: the tables, tile lists and act are the caller's
  ForwardScratch(void* base, int64_t R, int E, int hidden, int inter, bool keep_tables) {
    Carver c{static_cast<char*>(base)};
    tiles_bytes = mm_tile_lists_bytes(R, E);
    route_ws_bytes = mm_route_workspace_bytes(R, E);
    y = c.take<uint16_t>(static_cast<size_t>(R) * hidden * 2);
    route_ws = c.take<void>(route_ws_bytes);
    counts = offsets = send_route = send_token = route_to_send = nullptr;
    weight_perm = nullptr;
    tiles = nullptr;
    act = nullptr;
    if (!keep_tables) {
      const size_t r = static_cast<size_t>(R) * 4;
      counts = c.take<int32_t>(static_cast<size_t>(E) * 4);
      offsets = c.take<int32_t>(static_cast<size_t>(E + 1) * 4);
      send_route = c.take<int32_t>(r);
      send_token = c.take<int32_t>(r);
      route_to_send = c.take<int32_t>(r);
      weight_perm = c.take<float>(r);
      tiles = c.take<void>(tiles_bytes);
      act = c.take<uint16_t>(static_cast<size_t>(R) * inter * 2);
    }
    bytes = c.used;
  }
};

bool layer_sizes_ok(int64_t tokens, int32_t top_k, int32_t num_experts, int32_t hidden, int32_t inter) {
  return tokens >= 0 && top_k > 0 && top_k <= 64 && num_experts > 0 && hidden > 0 && inter > 0 &&
         tokens < (int64_t(1) << 31) / top_k;
}

}  // namespace

extern "C" size_t mm_moe_forward_scratch_bytes(int64_t tokens, int32_t top_k, int32_t num_experts, int32_t hidden,
                                               int32_t inter, int32_t keep_tables) {
  if (!layer_sizes_ok(tokens, top_k, num_experts, hidden, inter)) return 0;
  return ForwardScratch(nullptr, tokens * top_k, num_experts, hidden, inter, keep_tables != 0).bytes;
}

extern "C" int mm_moe_forward(const uint16_t* x, const int32_t* selected, const float* routing_weights,
                              const uint16_t* w1, const uint16_t* w2, int64_t w2_se, int64_t w2_sh, int64_t w2_sf,
                              int64_t tokens, int32_t top_k, int32_t num_experts, int32_t hidden, int32_t inter,
                              int32_t act_kind, float situ_beta, float situ_linear_beta, float clamp_limit,
                              int32_t* counts, int32_t* offsets, int32_t* send_route, int32_t* send_token,
                              int32_t* route_to_send, float* weight_perm, void* tiles, size_t tiles_bytes,
                              uint16_t* act, void* fc1_out, int32_t fc1_format, float* fc1_scale, uint16_t* out,
                              void* scratch, size_t scratch_bytes, mm_stream_t stream) {
  MM_CHECK_ARG(layer_sizes_ok(tokens, top_k, num_experts, hidden, inter), "mm_moe_forward: bad sizes");
  const int64_t R = tokens * top_k;
  const bool keep = counts != nullptr;
  MM_CHECK_ARG(keep ? (offsets && send_route && send_token && route_to_send && weight_perm && tiles && act)
                    : !(offsets || send_route || send_token || route_to_send || weight_perm || tiles || act || fc1_out),
               "mm_moe_forward: the tables, tile lists and act are given together or not at all");
  ForwardScratch s(scratch, R, num_experts, hidden, inter, keep);
  if (!scratch || scratch_bytes < s.bytes) {
    mm_set_error("mm_moe_forward: scratch needs %zu bytes", s.bytes);
    return MM_E_WS;
  }
  if (tokens == 0) return MM_OK;
  if (!keep) {
    counts = s.counts;
    offsets = s.offsets;
    send_route = s.send_route;
    send_token = s.send_token;
    route_to_send = s.route_to_send;
    weight_perm = s.weight_perm;
    tiles = s.tiles;
    tiles_bytes = s.tiles_bytes;
    act = s.act;
  }
  int rc = mm_route_tiles(selected, R, top_k, num_experts, routing_weights, counts, offsets, send_route, send_token,
                          route_to_send, weight_perm, tiles, tiles_bytes, s.route_ws, s.route_ws_bytes, stream);
  if (rc) return rc;
  rc = mm_fc1_swiglu_tiles(x, hidden, send_token, w1, offsets, weight_perm, num_experts, R, hidden, inter, act_kind,
                           situ_beta, situ_linear_beta, clamp_limit, act, fc1_out, fc1_format, fc1_scale, tiles,
                           tiles_bytes, stream);
  if (rc) return rc;
  rc = mm_grouped_gemm_tiles(act, inter, nullptr, w2, w2_se, w2_sh, w2_sf, offsets, num_experts, R, hidden, inter,
                             s.y, hidden, tiles, tiles_bytes, stream);
  if (rc) return rc;
  return mm_combine(s.y, hidden, route_to_send, tokens, top_k, hidden, out, hidden, stream);
}

extern "C" int mm_moe_backward(const uint16_t* dy, const uint16_t* x, const uint16_t* w1, const uint16_t* w2,
                               int64_t w2_se, int64_t w2_sh, int64_t w2_sf, int64_t tokens, int32_t top_k,
                               int32_t num_experts, int32_t hidden, int32_t inter, int32_t act_kind, float situ_beta,
                               float situ_linear_beta, float clamp_limit, const int32_t* offsets,
                               const int32_t* send_token, const int32_t* route_to_send, const float* weight_perm,
                               const void* tiles, size_t tiles_bytes, const void* fc1_out, int32_t fc1_format,
                               const float* fc1_scale, uint16_t* act, int32_t recompute_act, uint16_t* grad_act,
                               uint16_t* dab, uint16_t* dscale, uint16_t* grad_fc2, uint16_t* dx,
                               uint16_t* grad_hidden, float* grad_rw, uint16_t* grad_gate_up, mm_stream_t stream) {
  MM_CHECK_ARG(layer_sizes_ok(tokens, top_k, num_experts, hidden, inter) && tokens > 0, "mm_moe_backward: bad sizes");
  const int64_t R = tokens * top_k;
  const int E = num_experts, two_i = 2 * inter;
  int rc = mm_grouped_gemm_tiles(dy, hidden, send_token, w2, w2_se, w2_sf, w2_sh, offsets, E, R, inter, hidden,
                                 grad_act, inter, tiles, tiles_bytes, stream);
  if (rc) return rc;
  rc = mm_swiglu_bwd(grad_act, inter, fc1_out, two_i, fc1_format, fc1_scale, weight_perm, offsets, E, R, inter,
                     act_kind, situ_beta, situ_linear_beta, clamp_limit, dab, dscale, stream);
  if (rc) return rc;
  if (recompute_act) {
    rc = mm_gated_act(fc1_out, two_i, fc1_format, fc1_scale, weight_perm, offsets, E, R, inter, act_kind, situ_beta,
                      situ_linear_beta, clamp_limit, act, inter, stream);
    if (rc) return rc;
  }
  rc = mm_grouped_wgrad(dy, hidden, send_token, act, inter, nullptr, offsets, E, R, hidden, inter, grad_fc2, nullptr,
                        0, stream);
  if (rc) return rc;
  rc = mm_grouped_gemm_tiles(dab, two_i, nullptr, w1, static_cast<int64_t>(hidden) * two_i, two_i, 1, offsets, E, R,
                             hidden, two_i, dx, hidden, tiles, tiles_bytes, stream);
  if (rc) return rc;
  rc = mm_combine_bwd(dx, hidden, route_to_send, tokens, top_k, hidden, grad_hidden, hidden, dscale, grad_rw, stream);
  if (rc) return rc;
  return mm_grouped_wgrad(x, hidden, send_token, dab, two_i, nullptr, offsets, E, R, hidden, two_i, grad_gate_up,
                          nullptr, 0, stream);
}
