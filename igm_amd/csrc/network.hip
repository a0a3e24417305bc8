// The emulator's passes as one call each: the launches of all layers, from the
// host code next to them.  A call per layer from Python costs 5 to 10 us of
// host time, which is what a pass over a small grid then took: 100 x 100, 10
// launches of 60 us in all, 160 us a pass; now 75.
#include "conv_common.hpp"

using namespace igm;

namespace {
constexpr int64_t kW3x3 = 9 * kC * kC;  // weights of a 3x3 layer
}

extern "C" {

int igm_cnn_fwd(int32_t nl, const float* f0, const float* f1, const float* f2, const float* f3, const float* f4,
                int64_t fb, int64_t fr, int64_t fc, const int32_t* extents, int32_t B, int32_t H, int32_t W,
                const float* w, const int64_t* offs, const void* fwd, const void* head, int32_t cout, void* acts,
                int32_t keep, float* Y, void* stream) {
  IGM_CHECK_ARG(w && offs && head && acts && Y && (nl < 2 || fwd), "null pointer");
  IGM_CHECK_ARG(nl >= 1 && B >= 1 && H >= 1 && W >= 1, "bad sizes");
  const int64_t size = (int64_t)B * H * W * kC;
  const auto act = [&](int i) { return (bf16*)acts + (keep ? i : i & 1) * size; };
  const auto wt = [&](int l) { return (const bf16*)fwd + (l - 1) * kW3x3; };
  const auto bias = [&](int l) { return w + offs[2 * l + 1]; };
  if (const int rc = igm_conv_in_fwd(f0, f1, f2, f3, f4, fb, fr, fc, extents, B, H, W, w + offs[0], bias(0), act(0),
                                     stream))
    return rc;
  int i = 0;  // activations so far
  for (int l = 1; l < nl; ++i) {
    if (l + 1 == nl)  // with the output layer; the activations are stored for a backward pass only
      return igm_conv3x3_head_fwd_bf16(act(i), wt(l), bias(l), head, bias(nl), extents, B, H, W, cout,
                                       keep ? act(i + 1) : nullptr, Y, stream);
    if (keep) {
      if (const int rc = igm_conv3x3_fwd_bf16(act(i), wt(l), bias(l), extents, B, H, W, act(i + 1), stream)) return rc;
      l += 1;
    } else {  // two layers in one launch: the one between them is not stored
      if (const int rc = igm_conv3x3_pair_fwd_bf16(act(i), wt(l), bias(l), wt(l + 1), bias(l + 1), extents, B, H, W,
                                                   act(i + 1), stream))
        return rc;
      l += 2;
    }
  }
  return igm_conv1x1_head_fwd(act(i), head, bias(nl), extents, B, H, W, cout, Y, stream);
}

int igm_cnn_bwd(int32_t nl, const float* dY, const void* const* acts, const float* f0, const float* f1,
                const float* f2, const float* f3, const float* f4, int64_t fb, int64_t fr, int64_t fc,
                const int32_t* extents, int32_t B, int32_t H, int32_t W, const float* w, const int64_t* offs,
                const void* dgr, int32_t cout, int32_t nblocks_in, int32_t nblocks_3x3, int32_t nblocks_head,
                float* part_in, float* part_3x3, float* part_head, int32_t accumulate, void* dz0, void* dz1,
                float* input_grad, void* stream) {
  IGM_CHECK_ARG(acts && w && offs && dz0 && dz1 && (nl < 2 || (dgr && part_3x3)), "null pointer");
  IGM_CHECK_ARG(nl >= 1 && B >= 1 && H >= 1 && W >= 1, "bad sizes");
  void *dz = dz0, *below = dz1;
  if (const int rc = igm_conv1x1_head_bwd(dY, acts[nl - 1], w + offs[2 * nl], extents, B, H, W, cout, dz, below, stream))
    return rc;
  if (const int rc = igm_conv_wgrad_partials_bf16(1, acts[nl - 1], below, extents, B, H, W, nblocks_head, part_head,
                                                  accumulate, stream))
    return rc;
  for (int l = nl - 1; l > 0; --l) {
    float* part = part_3x3 + (l - 1) * igm_wgrad_workspace_floats(9, nblocks_3x3);
    if (const int rc = igm_conv3x3_bwd_bf16(acts[l - 1], dz, (const bf16*)dgr + (l - 1) * kW3x3, extents, B, H, W,
                                            nblocks_3x3, part, accumulate, below, stream))
      return rc;
    void* t = dz;
    dz = below;
    below = t;
  }
  if (const int rc = igm_conv_in_wgrad_partials(f0, f1, f2, f3, f4, fb, fr, fc, extents, B, H, W, dz, nblocks_in,
                                                part_in, accumulate, stream))
    return rc;
  if (input_grad == nullptr) return 0;
  return igm_conv_in_dgrad(dz, w + offs[0], extents, B, H, W, input_grad, stream);
}

}  // extern "C"
