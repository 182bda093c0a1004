// The routers' choice for one row, by one wave.
#pragma once

#include "mx_common.h"

namespace mx {

enum { kRouteSoftmaxTop = 0, kRouteSigmoid = 1, kRouteSoftmaxAll = 2 };     // corr: the selection bias of the last

// A lane an expert (at most 64), z its logit: every lane finds its expert's place in the order (ties to the lower index) by
// comparing with all others, so no choice waits for the one before.  idx, wts: the row's `top`.
__device__ __forceinline__ void choose_in_lanes(int* __restrict__ idx, float* __restrict__ wts, float z,
                                                const float* __restrict__ corr, int experts, int top, int mode, float scale,
                                                int groups, int keep, int lane) {
  const bool on = lane < experts;
  if (!on) z = -INFINITY;
  // ch: what the choice goes by; p: the softmax over all
  float p = 0.f, ch = z;
  if (mode == kRouteSoftmaxAll) {
    const float top_z = ft::wave_max(z);
    p = on ? expf(z - top_z) : 0.f;
    p = p / ft::wave_sum(p);
    ch = on ? p + corr[lane] : -INFINITY;
  }
  if (!(ch == ch)) ch = -INFINITY;          // (the order must hold every expert once)
  auto at = [&](float v, int e) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), e)); };
  if (keep < groups) {
    const int gsz = experts / groups, g = lane / gsz;
    float score = -INFINITY;
    for (int o = 0, e = 0; o < groups; ++o) {
      float a = -INFINITY, b = -INFINITY;    // the two largest of group o
      for (int j = 0; j < gsz; ++j, ++e) {
        const float v = at(ch, e);
        b = v > a ? a : fmaxf(b, v);
        a = fmaxf(a, v);
      }
      if (mode != kRouteSoftmaxAll) a = sigmoidf_(a) + (gsz > 1 ? sigmoidf_(b) : 0.f);
      score = o == g ? a : score;
    }
    int better_groups = 0;
    for (int o = 0; o < groups; ++o) {
      const float v = at(score, o * gsz);
      better_groups += v > score || (v == score && o < g);
    }
    if (better_groups >= keep) ch = -INFINITY;
  }
  int place = 0;
  for (int e = 0; e < experts; ++e) {
    const float v = at(ch, e);
    place += v > ch || (v == ch && e < lane);
  }
  const bool chosen = on && place < top;
  float w = p;
  if (mode != kRouteSoftmaxAll) {
    const float first = ft::wave_max(chosen ? ch : -INFINITY);
    w = !chosen ? 0.f : mode == kRouteSigmoid ? sigmoidf_(ch) : expf(ch - first);
    w = w / (ft::wave_sum(w) + (mode == kRouteSigmoid ? 1e-20f : 0.f)) * scale;
  }
  if (chosen) {
    idx[place] = lane;
    wts[place] = w;
  }
}

}  // namespace mx
