// Which strips of a tile a list entry is filed for: shared by the kernel that emits the
// (Gaussian, tile) instances, which decides it, and the blend kernels, which rely on it.
//
// Most (pixel, Gaussian) visits of the reference loop (K/cuda_rasterizer_hgs/forward.cu:338-372,
// K = rasterization_kernels/diff-gaussian-rasterization-half-gaussian) end at "alpha < 1/255" or at
// the half-Gaussian box test.  Three conservative tests remove such visits a whole 16x4 strip at a
// time without changing any result:
//  * alpha >= 1/255 needs power >= -ln(255 * opacity); with that floor (minus a margin) above
//    zero no pixel can pass;
//  * power >= floor is an ellipse around the Gaussian's centre; an entry whose ellipse (first its
//    bounding box, then the ellipse itself) misses the strip's rectangle is not filed;
//  * the world-space ray sample is affine in the pixel, so its range over a strip follows from the
//    strip's corner coordinates: an entry whose strip lies entirely outside the submodel box is not
//    filed, one whose strip lies entirely inside skips the per-pixel box test.
// All three only drop work that the exact evaluation would have skipped too.
#pragma once
#include "rgs_device.h"

namespace rgs {

__device__ __forceinline__ float wave_uniform(float v)
{
	return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// What the half-Gaussian test needs besides the pixel: rows 0..2 of the inverse projection
// (column-major 4x4, m[c][r] = element (r, c)) and the submodel box.  Read once per wavefront
// into scalar registers; the test itself runs for every blended sample.
struct BoxFrame {
	float m[4][3];
	float3 lo, hi;
	float tanx, tany;
};

// A pointer to what no kernel writes while it is read: such loads go through the scalar unit, straight into scalar registers.
typedef const __attribute__((address_space(4))) float* ConstantFloats;
__device__ __forceinline__ ConstantFloats constant_floats(const float* p) { return (ConstantFloats)(uintptr_t)p; }

__device__ __forceinline__ BoxFrame load_box_frame(const float* projinv, const float* range_low, const float* range_up, float tanx, float tany)
{
	BoxFrame b;
	const ConstantFloats m = constant_floats(projinv), lo = constant_floats(range_low), hi = constant_floats(range_up);
#pragma unroll
	for (int c = 0; c < 4; c++)
#pragma unroll
		for (int r = 0; r < 3; r++)
			b.m[c][r] = m[4 * c + r];
	b.lo = float3{lo[0], lo[1], lo[2]};
	b.hi = float3{hi[0], hi[1], hi[2]};
	b.tanx = tanx;
	b.tany = tany;
	return b;
}

// What the tests need of a Gaussian's 64-byte blend record: (pixel x, pixel y, exponent floor, clip w),
// the conic (xx, xy, yy) and the half extents of the alpha >= 1/255 ellipse's bounding box.
struct FiledGeometry {
	float4 geom;
	float4 conic;
	float2 half;
};

// NDC of the middle of a tile's 16 columns or rows of pixels (pix_to_ndc with the division replaced by the reciprocal image size: it
// only feeds the conservative range test, which has room for the last bit).
__device__ __forceinline__ float tile_middle_ndc(int tile, int pixels)
{
	return (float)((2.0 * ((double)(tile * kTile) + 7.5) + 1.0) * (1.0 / (double)pixels) - 1.0);
}

// How far the first and last pixel centres lie from the middle, in NDC: of a tile's columns, of its rows and of a strip's rows; and a
// strip's middle from the next one's.
struct NdcSteps {
	float tile_x, tile_y, strip_y, strips;
};
__device__ __forceinline__ NdcSteps ndc_steps(int W, int H)
{
	return NdcSteps{15.f / (float)W, 15.f / (float)H, 3.f / (float)H, 8.f / (float)H};
}

// The part of the tests that depends on the Gaussian and the frame but not on the tile, computed
// once per Gaussian.  The ray sample at the Gaussian's clip w is affine in the pixel's NDC
// coordinates, p_k = A_k nx + B_k ny + C_k per world coordinate k, so over a rectangle of pixels it lies within
// |A_k| and |B_k| times the half extents of its value in the middle; the box tolerance is taken from the magnitudes of the terms, not
// of the result, so that it also covers the rounding of this regrouped evaluation when the terms
// cancel.
struct StripTests {
	float gx, gy, hx, hy;
	float a, b, c, limit;   // conic; -2 floor
	float rc;               // 1 / c
	float A[3], B[3], C[3], tol[3];
	uint32_t flags;         // bit 0: the conic is an ellipse; bit 1: no pixel can reach alpha >= 1/255
	uint32_t pad;
};

__device__ __forceinline__ StripTests prepare_strip_tests(const FiledGeometry& e, const BoxFrame& box)
{
#pragma clang fp contract(off)
	StripTests t;
	t.gx = e.geom.x; t.gy = e.geom.y; t.hx = e.half.x; t.hy = e.half.y;
	const float floor = e.geom.z, w = e.geom.w;
	t.a = e.conic.x; t.b = e.conic.y; t.c = e.conic.z;
	t.limit = -2.f * floor;
	// hardware reciprocals and square roots (one unit in the last place) here and below: these values only place the
	// bounds of conservative tests, whose margins are three orders of magnitude wider, and a correctly rounded division
	// or square root costs ten instructions where these cost one
	t.rc = __builtin_amdgcn_rcpf(t.c);
	const bool ellipse = (t.a > 0.f) && (t.c > 0.f) && (t.a * t.c - t.b * t.b > 0.f);
	t.flags = (ellipse ? 1u : 0u) | ((floor > 0.f) ? 2u : 0u);  // floor > 0: even power = 0 gives alpha < 1/255
	t.pad = 0u;
	const float wp = w + 0.0000001f;
	const float sx = wp * box.tanx, sy = wp * box.tany;
#pragma unroll
	for (int k = 0; k < 3; k++) {
		const float m2w = box.m[2][k] * w;
		t.A[k] = box.m[0][k] * sx;
		t.B[k] = box.m[1][k] * sy;
		t.C[k] = m2w + box.m[3][k];
		t.tol[k] = 1e-4f * fmaxf((fabsf(t.A[k]) + fabsf(t.B[k])) + (fabsf(m2w) + fabsf(box.m[3][k])), 1.f);
	}
	return t;
}

// The decisions for the four strips of the tile whose first pixel is (x0, y0): bit s of the result =
// the entry is filed for strip s, bit 4 + s = that strip lies inside the box.  nx, ny = NDC of the tile's middle.
__device__ __forceinline__ uint32_t strips_filed_for(const StripTests& t, float x0, float y0, float nx, float ny, const NdcSteps& steps,
                                                     const BoxFrame& box)
{
#pragma clang fp contract(off)
	if (t.flags & 2u)
		return 0u;
	if ((t.gx + t.hx < x0) || (t.gx - t.hx > x0 + 15.f))
		return 0u;
	const float a = t.a, b = t.b, c = t.c;
	const bool ellipse = (t.flags & 1u) != 0u;
	const float dxl = t.gx - (x0 + 15.f), dxh = t.gx - x0;

	// Per world coordinate the ray sample's value in the middle of the tile's columns and its reach over them, the tolerance on
	// top; then the box test for the whole tile (of which the strips are parts).  Most Gaussians are far from their submodel's
	// faces, and a tile that lies inside the box needs no test per strip.  (Middle and reach take 30 instructions where the ends of
	// both ranges took 66.  The key duplication is bound by the issue of these tests: with that, the strips' answers without branches
	// and the ellipse's with fused products it went from 148 to 126 us for two submodels of 2.8 M, 735 to 624 at 5185x3359.)
	const float lov[3] = {box.lo.x, box.lo.y, box.lo.z}, hiv[3] = {box.hi.x, box.hi.y, box.hi.z};
	float middle[3], reach[3];
	bool tile_inside = true, tile_outside = false;
#pragma unroll
	for (int k = 0; k < 3; k++) {
		middle[k] = __builtin_fmaf(t.A[k], nx, t.C[k]);
		reach[k] = __builtin_fmaf(fabsf(t.A[k]), steps.tile_x, t.tol[k]);
		const float m = __builtin_fmaf(t.B[k], ny, middle[k]), r = __builtin_fmaf(fabsf(t.B[k]), steps.tile_y, reach[k]);
		tile_inside = tile_inside & (m - r > lov[k]) & (m + r < hiv[k]);
		tile_outside = tile_outside | (m + r < lov[k]) | (m - r > hiv[k]);
	}
	if (tile_outside)
		return 0u;

	// The rows the ellipse q(d) = a dx^2 + 2 b dx dy + c dy^2 <= limit reaches over the tile's 16 columns, once for the four
	// strips (d = centre - pixel, so dx runs over [dxl, dxh]).  For a given dx the ellipse holds the dy between
	// (-b dx -+ sqrt(c limit - det dx^2)) / c; the upper end is concave in dx and the lower convex, so over an interval
	// of dx each is extreme at the ellipse's own extreme point (dy = +-Y at dx = -+b Y / a, Y = sqrt(a limit / det)) if
	// that lies inside the interval, at one of its ends otherwise.  The limit gets room for the rounding
	// of q (relative to its largest terms over the tile), and the rows a margin of a hundredth of a pixel.
	float dy_low = -INFINITY, dy_high = INFINITY;
	if (ellipse) {
		const float dy_first = t.gy - y0, dy_last = t.gy - (y0 + 15.f);
		const float largest = a * fmaxf(dxl * dxl, dxh * dxh) + c * fmaxf(dy_first * dy_first, dy_last * dy_last);
		const float limit = t.limit + __builtin_fmaf(1e-5f, largest, __builtin_fmaf(1e-4f, t.limit, 1e-3f));
		const float det = a * c - b * b;
		const float room = limit * __builtin_amdgcn_rcpf(det), c_limit = c * limit;
		const float X = __builtin_amdgcn_sqrtf(c * room), Y = __builtin_amdgcn_sqrtf(a * room);
		const float dl = fmaxf(dxl, -X), dh = fminf(dxh, X);
		if (dl > dh)
			return 0u;  // the columns lie beside the ellipse
		const float sl = __builtin_amdgcn_sqrtf(fmaxf(__builtin_fmaf(-det * dl, dl, c_limit), 0.f)),
		            sh = __builtin_amdgcn_sqrtf(fmaxf(__builtin_fmaf(-det * dh, dh, c_limit), 0.f));
		const float bY = b * Y, first = a * dl, last = a * dh;  // a times: the dx of the ellipse's lowest dy (that of its highest is its negative), the ends
		const float top = fmaxf(__builtin_fmaf(-b, dl, sl), __builtin_fmaf(-b, dh, sh)) * t.rc;
		const float bottom = fminf(__builtin_fmaf(-b, dl, -sl), __builtin_fmaf(-b, dh, -sh)) * t.rc;
		const float margin = __builtin_fmaf(1e-5f, Y, 1e-2f);
		dy_high = ((!(-bY < first) & !(-bY > last)) ? Y : top) + margin;
		dy_low = ((!(bY < first) & !(bY > last)) ? -Y : bottom) - margin;
	}
	// Which strips the entry reaches, without a branch: all four are answered by two comparisons each and lane masks (four against each of
	// the ends, with their differences, took 19 instructions more: 621 -> 606 us at 5185x3359, 185 -> 181 for four calls at 1600x1036).  Of a
	// tile inside the box that is all.
	uint32_t bits = 0;
	const float cy = t.gy - y0;
	const float top = fminf(cy + t.hy, cy - dy_low), bottom = fmaxf(cy - t.hy, cy - dy_high);  // the last and first row it reaches, from y0
#pragma unroll
	for (int s = 0; s < 4; s++) {
		const bool beside = (top < (float)(4 * s)) | (bottom > (float)(4 * s + 3));
		bits |= beside ? 0u : 0x11u << s;
	}
	if (!tile_inside) {
#pragma unroll
		for (int s = 0; s < 4; s++) {
			const float strip_ny = __builtin_fmaf((float)s - 1.5f, steps.strips, ny);
			bool inside = true, outside = false;
#pragma unroll
			for (int k = 0; k < 3; k++) {
				const float m = __builtin_fmaf(t.B[k], strip_ny, middle[k]), r = __builtin_fmaf(fabsf(t.B[k]), steps.strip_y, reach[k]);
				inside = inside & (m - r > lov[k]) & (m + r < hiv[k]);
				outside = outside | (m + r < lov[k]) | (m - r > hiv[k]);
			}
			// a NaN can set neither flag, which leaves the decision to the per-pixel test
			bits &= outside ? ~(0x11u << s) : inside ? ~0u : ~(0x10u << s);
		}
	}
	return bits;
}

}  // namespace rgs
