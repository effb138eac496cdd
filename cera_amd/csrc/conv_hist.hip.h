// History of a layer's input convolutions, for the kernels that add it up.
#pragma once
#include "sigmoid_attn.h"

// of the token at `pos`: taps 0 .. taps-2 against rows pos - taps + 1 .. pos - 1.  i: channel, those of the second convolution behind the first's
__device__ __forceinline__ void conv_hist_body(const ConvRing& ring, const ConvHist& h, uint32_t pos, uint32_t i) {
    const float* const w = i < ring.width ? h.wa : h.wb;
    const uint32_t c = i < ring.width ? i : i - ring.width;
    if (!w || c >= ring.width) return;
    float s = 0.0f;
    for (uint32_t j = 0; j + 1 < h.taps; ++j) {
        const uint32_t back = h.taps - 1 - j;
        if (back <= pos) s = fmaf(w[static_cast<uint64_t>(j) * ring.width + c], ring.rows[static_cast<uint64_t>((pos - back) & (ring.depth - 1)) * ring.ld + c], s);
    }
    (i < ring.width ? h.a : h.b)[c] = s;
}
