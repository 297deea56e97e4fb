#pragma once
// A Gaussian's record as the compositing kernels stage it in LDS, the tests that leave an entry of a
// tile's list out of the compositing passes, and the one that sends an entry to their general path.  In
// a header of its own, and callable on the host as well, so that the tests can be checked against brute
// force over a tile's pixels without a GPU.
#include <cstdint>

#include <xyz_autodiff/detail/config.cuh>
#include <xyz_autodiff/operations/math.cuh>

#include "splat.cuh"

namespace xad_splat {

using namespace xyz_autodiff;

constexpr float kHalfLog2e = 0.72134752044448170368f;  // log2(e) / 2

struct alignas(16) Staged {
    float cx, cy, a_s, b2_s;          // centre; a' and 2b'
    float c_s, alpha0, a, b;          // c'; sigmoid(opacity); inverse covariance as stored
    float red, green, blue, c;        // colour; inverse covariance
};
static_assert(sizeof(Staged) == 48, "Staged must be three float4");

XAD_INLINE Staged stage_record(const Record* __restrict__ records, std::uint32_t g) {
    const float4* src = reinterpret_cast<const float4*>(records + g);
    const float4 v0 = src[0], v1 = src[1], v2 = src[2];
    Staged s;
    s.cx = v0.x;
    s.cy = v0.y;
    s.a = v0.z;
    s.b = v0.w;
    s.c = v1.x;
    s.red = v1.y;
    s.green = v1.z;
    s.blue = v1.w;
    s.alpha0 = v2.x;
    s.a_s = -kHalfLog2e * s.a;
    s.b2_s = -2.f * kHalfLog2e * s.b;
    s.c_s = -kHalfLog2e * s.c;
    return s;
}

// List entries that cannot be seen from a tile.  The binning rectangle is the 3-sigma box of the
// Gaussian's own axes-aligned extent, so a rotated, elongated Gaussian is listed in corner tiles that
// its ellipse never comes near (about a fifth of all pairs when scales span 0.5 to 40 pixels).  Such
// an entry is recognised when its record is staged: the minimum of q over the tile's pixel centres
// is bounded from below by the minimum over their bounding box, which for a convex quadratic whose
// centre lies outside the box is attained on one of the four edges.  If even there alpha stays below
// kNegligibleAlpha, the entry is left out of the compositing loop: it would change a pixel by less than
// 1e-8 (an fp32 ulp of 0.5 is 6e-8).  The backward pass asks about a whole tile, the forward pass about
// the half that a wavefront walks (see negligible_in_part() for what keeps the two together).  Lists and
// pair counts are not affected.  Comparisons with NaN are false, so an odd record is kept.
constexpr float kNegligibleAlpha = 1e-8f;

// over the pixels from (left, top) on, kTile of them across and `high` down
XAD_INLINE bool negligible_in_rectangle(const Staged& s, float left, float top, int high) {
    const float x0 = left - s.cx, x1 = x0 + static_cast<float>(kTile - 1);
    const float y0 = top - s.cy, y1 = y0 + static_cast<float>(high - 1);
    float q_min = 0.f;
    if (!(x0 <= 0.f && x1 >= 0.f && y0 <= 0.f && y1 >= 0.f)) {
        const float x_of_y = -s.b / s.a, y_of_x = -s.b / s.c;  // where q is least along a line
        auto along_x = [&](float y) {  // min over x in [x0, x1] of a x^2 + 2 b x y + c y^2
            const float x = __builtin_fminf(__builtin_fmaxf(x_of_y * y, x0), x1);
            return ::fmaf(::fmaf(s.a, x, 2.f * s.b * y), x, s.c * y * y);
        };
        auto along_y = [&](float x) {
            const float y = __builtin_fminf(__builtin_fmaxf(y_of_x * x, y0), y1);
            return ::fmaf(::fmaf(s.c, y, 2.f * s.b * x), y, s.a * x * x);
        };
        q_min = __builtin_fminf(__builtin_fminf(along_x(y0), along_x(y1)), __builtin_fminf(along_y(x0), along_y(x1)));
    }
    return s.alpha0 * math::fp32::exp2_raw(-kHalfLog2e * q_min) < kNegligibleAlpha;
}

XAD_INLINE bool negligible_in_tile(const Staged& s, float tile_x, float tile_y) {
    return negligible_in_rectangle(s, tile_x, tile_y, kTile);
}

// Entries for which the compositing loops have to make sure of two things themselves.  For all others
//   - alpha stays below kAlphaMax at every pixel: alpha0 does by a margin, and q cannot come out negative by more
//     than rounding.  (q >= (1 - |b| / sqrt(ac)) (a dx^2 + c dy^2), the rounding of its three terms is at most
//     5e-7 (a dx^2 + c dy^2), and 1 - |b| / sqrt(ac) >= (ac - b^2) / 2ac > 5e-6);
//   - a pixel whose x is kFarAway gets alpha = 0: there a dx^2 >= 1e-9 1e36, and neither 2 |b dx dy| <=
//     2 sqrt(ac) 1e18 |dy| nor c dy^2 comes near it (|dy| < 1.1e6: images are at most 32767 tiles high).
// Comparisons with NaN are false, so an odd record is taken with care.
// An entry that needs care sends its pair to the general path.  Where nearly all do, opacity logits ~ N(6, 1), a step of
// 200 000 Gaussians at 2048 x 2048 takes 635 us (forward 157, backward 400), of 10 000 at 512 x 512 111 us; loops without
// the distinction, every pixel's compares and selects in every trip, took 668 (195, 393) and 137.
constexpr float kFarAway = 1e18f;

XAD_INLINE bool ill_shaped(const Staged& s) {
    const float ac = s.a * s.c;
    return !(s.a >= 1e-9f && s.a <= 1e9f && s.c >= 1e-9f && s.c <= 1e9f && ac - s.b * s.b >= 1e-5f * ac && s.cx >= -1e6f &&
             s.cx <= 1e6f && s.cy >= -5e5f && s.cy <= 5e5f);
}
XAD_INLINE bool needs_care(const Staged& s) { return !(s.alpha0 <= 0.98f) || ill_shaped(s); }

// What the forward walk of one part of a tile (`high` rows from part_y on) leaves out.  The backward walk takes whole tiles
// and leaves out what negligible_in_tile() says, and the two must not disagree about an entry that changes a pixel: one that
// only the forward pass composited stays in the transmittance that the backward pass starts from, for every entry in front
// of it.  For an entry of good shape they cannot: the rounding of q is at most 1e-6 (a dx^2 + c dy^2), a fifth of q, so one
// that either test leaves out has an alpha below 1e-8^(1/1.44) = 3e-6 at every pixel in question.  Of long thin Gaussians q
// can cancel to nothing but rounding (0.3 x 3000 pixels: one in 2000 near pairs came out up to 0.99 in one test only);
// about those both passes ask for the tile, and get the same answer.
XAD_INLINE bool negligible_in_part(const Staged& s, float tile_x, float tile_y, float part_y, int high) {
    const bool whole = ill_shaped(s);
    return negligible_in_rectangle(s, tile_x, whole ? tile_y : part_y, whole ? kTile : high);
}

}  // namespace xad_splat
