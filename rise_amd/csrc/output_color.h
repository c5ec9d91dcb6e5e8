// output_color.h -- the output stage's per-pixel colour pipeline, compiled for
// host and device: film XYZ -> linear Rec.709 (with the reference's gamut
// clip) -> exposure and display transform (LDR formats) -> output colour
// space -> clamp and integerize.  Double precision throughout, in the
// reference's operation order, so that quantized bytes match its writers.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#ifndef RISE_HD
#define RISE_HD __host__ __device__
#endif

namespace rise_hip {
namespace out {

struct P2 {
    double x, y;
};

constexpr double kNearZero = 1e-12;

// LineIntersection2D (Utilities/Color/ColorUtils.cpp:150-175).
RISE_HD inline bool line_intersection(P2 a0, P2 a1, P2 b0, P2 b1, P2& out)
{
    const double denom = (b1.y - b0.y) * (a1.x - a0.x) - (b1.x - b0.x) * (a1.y - a0.y);
    if (denom > -kNearZero && denom < kNearZero) return false;
    const double ua = ((b1.x - b0.x) * (a0.y - b0.y) - (b1.y - b0.y) * (a0.x - b0.x)) / denom;
    out.x = a0.x + ua * (a1.x - a0.x);
    out.y = a0.y + ua * (a1.y - a0.y);
    return true;
}

// IsPointOnLineSegment (:198-205): the x-parameter strictly inside (0, 1).
RISE_HD inline bool on_segment(P2 s, P2 e, P2 p)
{
    const double v = (p.x - s.x) / (e.x - s.x);
    return v >= kNearZero && v <= 1.0 - kNearZero;
}

// ClipAgainstGamutEdge (:207-222).
RISE_HD inline bool clip_edge(P2 c, P2 a, P2 b, P2 w, P2& out)
{
    if (!line_intersection(w, c, a, b, out)) return false;
    if (!on_segment(a, b, out)) return false;
    if (on_segment(w, out, c)) {
        out = c;
        return true;
    }
    return on_segment(w, c, out);
}

constexpr P2 kRed{0.640, 0.330}, kGreen{0.300, 0.600}, kBlue{0.150, 0.060}, kWhite{0.3127, 0.3290};

// Where a chromaticity moves to (false: nowhere), by the edges in order.
RISE_HD inline bool clip_chromaticity(P2 c, P2& hit)
{
    return clip_edge(c, kRed, kGreen, kWhite, hit) || clip_edge(c, kRed, kBlue, kWhite, hit) ||
           clip_edge(c, kBlue, kGreen, kWhite, hit);
}

// The same with one edge's divisions instead of up to three edges': the sector
// between two vertices, seen from the white point, holds the only edge that c's
// ray can meet; the others' lines meet it behind the white point, which
// clip_edge refuses.  c too near a sector's border, the vertical through the
// white point or infinity for rounding to be ruled out is left to
// clip_chromaticity.  The edge's expressions are those of clip_edge, so the
// result is the same to the bit; no edge takes a NaN.
RISE_HD inline bool clip_chromaticity_quick(P2 c, P2& hit)
{
    if (c.x != c.x || c.y != c.y) return false;
    const double dx = c.x - kWhite.x, dy = c.y - kWhite.y;
    const double tr = (kRed.x - kWhite.x) * dy - (kRed.y - kWhite.y) * dx;
    const double tg = (kGreen.x - kWhite.x) * dy - (kGreen.y - kWhite.y) * dx;
    const double tb = (kBlue.x - kWhite.x) * dy - (kBlue.y - kWhite.y) * dx;
    const double eps = 1e-7;
    const bool clear = fabs(tr) > eps && fabs(tg) > eps && fabs(tb) > eps && fabs(dx) > 1e-6 && fabs(dx) < 4.0 &&
                       fabs(dy) < 4.0;
    if (!clear) return clip_chromaticity(c, hit);
    const bool rg = tr > 0.0 && tg < 0.0, bg = tg > 0.0 && tb < 0.0;  // else red-blue
    const P2 a{bg ? kBlue.x : kRed.x, bg ? kBlue.y : kRed.y};
    const P2 b{rg || bg ? kGreen.x : kBlue.x, rg || bg ? kGreen.y : kBlue.y};
    return clip_edge(c, a, b, kWhite, hit);
}

// MoveXYZIntoRec709RGBGamut + XYZtoRec709RGB (ColorUtils.cpp:351-363,
// Color.cpp:214-220): chromaticities outside the Rec.709 triangle move
// toward the white point onto its edge (red-green, red-blue, blue-green
// tried in that order), luminance kept; then the XYZ -> Rec.709 matrix.
template <bool QUICK = false>
RISE_HD inline void xyz_to_rec709(double X, double Y, double Z, double rgb[3])
{
    const double ovs = 1.0 / (X + Y + Z);
    const P2 c{X * ovs, Y * ovs};
    P2 hit{0.0, 0.0};
    if (QUICK ? clip_chromaticity_quick(c, hit) : clip_chromaticity(c, hit)) {
        const double prod = (1.0 / hit.y) * Y;
        X = prod * hit.x;
        Z = prod * (1 - hit.x - hit.y);
    }
    rgb[0] = 3.240479 * X + -1.537150 * Y + -0.498535 * Z;
    rgb[1] = -0.969256 * X + 1.875992 * Y + 0.041556 * Z;
    rgb[2] = 0.055648 * X + -0.204043 * Y + 1.057311 * Z;
}

// Display transforms (Rendering/DisplayTransform.h): non-finite and
// non-positive inputs are 0.
RISE_HD inline double sanitise(double x) { return ((x - x) == 0.0 && x > 0.0) ? x : 0.0; }  // x - x: NaN unless finite

RISE_HD inline double clamp01(double y) { return fmin(fmax(y, 0.0), 1.0); }

RISE_HD inline double display_curve(int dt, double x)
{
    const double s = sanitise(x);
    switch (dt) {
    case 0:  // none
        return s;
    case 1:  // Reinhard
        return s / (1.0 + s);
    case 3: {  // AgX (scalar sigmoid in log10)
        const double lx = log10(s + 1e-10);
        return clamp01(0.5 + 0.5 * tanh(1.0 * (lx - 0.0)));
    }
    case 4: {  // Hable, white point 11.2
        auto curve = [](double v) {
            const double A = 0.15, B = 0.50, C = 0.10, D = 0.20, E = 0.02, F = 0.30;
            return ((v * (A * v + C * B) + D * E) / (v * (A * v + B) + D * F)) - E / F;
        };
        return clamp01(curve(s * 2.0) / curve(11.2));
    }
    case 2:  // ACES (Narkowicz fit), also the fallback of unknown values
    default: {
        const double num = s * (2.51 * s + 0.03);
        const double den = s * (2.43 * s + 0.59) + 0.14;
        return clamp01(num / den);
    }
    }
}

// SRGBTransferFunction (ColorUtils.cpp:20-31).
RISE_HD inline double srgb_oetf(double x)
{
    if (x == 0) return 0;
    if (x <= 0.003040247678) return 12.92 * x;
    return 1.055 * pow(x, 1.0 / 2.4) - 0.055;
}

struct Params {
    int color_space;    // 0 linear Rec.709, 1 sRGB
    int display;        // display transform (applied when `tone` is set)
    int tone;           // LDR with a display transform or exposure: DisplayTransformWriter
    double exposure;    // 2^EV
};

// The pixel as the writer sees it before integerizing, RISEPel after the
// optional DisplayTransformWriter, but for the output colour space's curve.
template <bool QUICK>
RISE_HD inline void pixel_linear(const Params& p, float fx, float fy, float fz, double out[3])
{
    xyz_to_rec709<QUICK>((double)fx, (double)fy, (double)fz, out);
    if (p.tone)
        for (int k = 0; k < 3; ++k) out[k] = display_curve(p.display, out[k] * p.exposure);
}

// Color_Template::Integerize (Color_Template.h:129-134): clamp to [0, 1],
// scale, truncate.
template <class T>
RISE_HD inline T integerize(double v, double maxv)
{
    if (v > 1.0) v = 1.0;
    if (v < 0.0) v = 0.0;
    return (T)(v * maxv);
}

// integerize(srgb_oetf(x), maxv) without the 64-bit power function, which is
// 60% of the output stage's instructions: x^(1/2.4) from 32-bit log2 and exp2
// (relative error e below 1e-6, 7e-7 by their error bounds) and one Newton step
// of y^12 = x^5 in 64 bits, whose error is 5.5 e^2 < 6e-12.  Where that could
// change the truncated value (v within 1e-10 of the scale of a whole number)
// the power function decides.
template <class T>
RISE_HD inline T integerize_srgb(double x, double maxv)
{
    if (x <= 0.003040247678) return integerize<T>(12.92 * x, maxv);  // 0 at 0
    if (x == 1.0) return integerize<T>(1.055 * 1.0 - 0.055, maxv);
    if (x > 1.01) return integerize<T>(1.0, maxv);
    const double y = (double)exp2f(log2f((float)x) * (float)(1.0 / 2.4));
    const double x2 = x * x, y2 = y * y, y4 = y2 * y2, y12 = y4 * y4 * y4;
    const double root = y + y * (double)((float)(x2 * x2 * x - y12) / (12.0f * (float)y12));
    const double v = (1.055 * root - 0.055) * maxv, g = 1e-10 * maxv;
    if (floor(v - g) == floor(v + g)) return integerize<T>(1.055 * root - 0.055, maxv);
    return integerize<T>(srgb_oetf(x), maxv);  // also NaN
}

// HDRWriter::WriteHDRPixelToBuffer (RasterImages/HDRWriter.h:37-58): shared
// exponent of the largest channel, mantissas scaled by 255.9999.
RISE_HD inline void rgbe(const double c[3], uint8_t out[4])
{
    double v = c[0] > c[1] ? (c[0] > c[2] ? c[0] : c[2]) : (c[1] > c[2] ? c[1] : c[2]);
    if (v < 1e-32) {
        out[0] = out[1] = out[2] = out[3] = 0;
        return;
    }
    int e;
    v = frexp(v, &e) * 255.9999 / v;
    out[0] = (uint8_t)(c[0] < 0 ? 0 : c[0] * v);
    out[1] = (uint8_t)(c[1] < 0 ? 0 : c[1] * v);
    out[2] = (uint8_t)(c[2] < 0 ? 0 : c[2] * v);
    out[3] = (uint8_t)(e + 128);
}

}  // namespace out
}  // namespace rise_hip
