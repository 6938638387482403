// The rotary embedding applied behind a per-head norm, forward and backward, on rows held in registers.
#pragma once

#include "norm_device.h"

namespace ttn {

// ---- rotary embedding behind the norm -----------------------------------------
// The attention caller rotates the normalised query and key right after the per-head norm
// (teletron/models/dit/dit_attention.py:266-273, :435-443) with the real-pair form of
// diffusers' apply_rotary_emb: for tokens below `tokens`
//     out = cast(float(y) * cos + float(rotate_pairs(y)) * sin),   rotate_pairs(y)[2i, 2i+1] = (-y[2i+1], y[2i])
// with cos, sin fp32 tables [tokens, C]; each product and the sum are rounded to fp32, the result
// once to the element type.  Pairs are adjacent, so both halves sit in one lane's 16-byte piece.
struct NoRope {
    static constexpr bool kOn = false;
};
struct RopeTable {
    static constexpr bool kOn = true;
    const float *cos, *sin;  // [tokens, C] fp32, row = token index
    int64_t tokens;          // rows of the view at sequence index >= tokens are left unrotated
};

template <int VEC>
__device__ __forceinline__ void load_fp32_run(float (&dst)[VEC], const float *p) {
#pragma unroll
    for (int i = 0; i < VEC / 4; ++i) {
        const u32x4 t = load16(reinterpret_cast<const u32x4 *>(p) + i);  // cached: every head reuses the row
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[4 * i + j] = as_f32(t[j]);
    }
}

// One row's share of the tables in registers: lane l holds the VEC columns of each of its CHUNKS pieces.
template <bool ON, int CHUNKS, int VEC>
struct RopeRows {};
template <int CHUNKS, int VEC>
struct RopeRows<true, CHUNKS, VEC> {
    float c[CHUNKS][VEC], s[CHUNKS][VEC];
    bool on;  // this lane's row is rotated (a row that exists, at a token index below rope.tokens)
    __device__ __forceinline__ void fetch(const RopeTable &rope, bool ok, int64_t seq, int C, int l, int LANES) {
        on = ok && seq < rope.tokens;
        if (on) {
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k) {
                const int64_t col0 = seq * C + (k * LANES + l) * VEC;
                load_fp32_run<VEC>(c[k], rope.cos + col0);
                load_fp32_run<VEC>(s[k], rope.sin + col0);
            }
        }
    }
};

// y -> y*cos + rotate_pairs(y)*sin in fp32 (y already rounded to the element type)
template <int VEC>
__device__ __forceinline__ void rotate_pairs_forward(float (&v)[VEC], const float (&c)[VEC], const float (&s)[VEC]) {
#pragma unroll
    for (int j = 0; j < VEC; j += 2) {
        const float a = v[j], b = v[j + 1];
        v[j] = a * c[j] - b * s[j];
        v[j + 1] = b * c[j + 1] + a * s[j + 1];
    }
}

// The gradient of the rotation as autograd forms it: g*cos and g*sin are each cast to the element
// type (the two branches of x.float() and rotate_pairs(x).float()), the latter routed back through
// the pair swap, and the two contributions are added in the element type.
template <typename E, int VEC>
__device__ __forceinline__ void rotate_pairs_backward(float (&g)[VEC], const float (&c)[VEC], const float (&s)[VEC]) {
    float direct[VEC], swapped[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
        direct[j] = g[j] * c[j];
        swapped[j] = g[j] * s[j];
    }
    E::round(direct);
    E::round(swapped);
#pragma unroll
    for (int j = 0; j < VEC; j += 2) {
        g[j] = direct[j] + swapped[j + 1];
        g[j + 1] = direct[j + 1] - swapped[j];
    }
    E::round(g);
}

}  // namespace ttn
