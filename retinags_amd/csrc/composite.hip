// Front-to-back compositing of K partial images (RGB, depth, accumulated alpha), forward
// and backward, one pixel per thread, one pass over every input plane.
// Restates parallel_utils/basic_parallel_trainer/result_aggregator.py:244-259:
//   T_0 = 1, T_k = prod_{j<k} (1 - alpha_j)
//   image = sum_k T_k image_k + bg T_K,  depth = sum_k T_k depth_k,  alpha = 1 - T_K
// The inputs arrive already in compositing order.
#include "rgs_kernels.h"

namespace rgs {

// Whether the rasterizer listed nothing for a layer in the 16x4 pixels around this one.  There, on a black background, the layer is
// zero in all of its planes, and they need no reads: a frame's submodels each cover a part of the image (four submodels
// at 5185x3359, two thirds of their strips empty: forward 364 -> 180 us, backward 444 -> 350; 24.7 -> 18.7 and 38.4 -> 29.7 at 1600x1036).
struct StripPlace {
	size_t strip;
	bool black;
};
__device__ __forceinline__ StripPlace strip_of_pixel(const CompositeArgs& a, size_t p)
{
	const uint32_t y = (uint32_t)p / (uint32_t)a.W, x = (uint32_t)p - y * (uint32_t)a.W;
	const uint32_t tile = (y >> 4) * (((uint32_t)a.W + 15u) >> 4) + (x >> 4);
	return StripPlace{4 * (size_t)tile + ((y & 15u) >> 2), a.layer_bg[0] == 0.f && a.layer_bg[1] == 0.f && a.layer_bg[2] == 0.f};
}
// Bits of the layers from k0 on, kLayers of them at most, that have something there.
template <int kLayers>
__device__ __forceinline__ uint32_t layers_with_entries(const CompositeArgs& a, const StripPlace& at, int k0)
{
	uint32_t count[kLayers], mask = 0u;
#pragma unroll
	for (int q = 0; q < kLayers; q++) {
		count[q] = 1u;
		if (k0 + q < a.K && a.strips[k0 + q] && at.black)
			count[q] = a.strips[k0 + q][at.strip];
	}
#pragma unroll
	for (int q = 0; q < kLayers; q++)
		mask |= count[q] != 0u ? 1u << q : 0u;
	return mask;
}

// kStrips: some layers bring their strips' counts.
template <bool kStrips>
__global__ __launch_bounds__(256) void composite_forward_kernel(CompositeArgs a)
{
	const size_t n = (size_t)a.H * a.W;
	const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
	if (p >= n)
		return;
	StripPlace at = {};
	if (kStrips)
		at = strip_of_pixel(a, p);
	float T = 1.f, r = 0.f, g = 0.f, b = 0.f, d = 0.f;
	// kAhead layers' planes are asked for together: one layer at a time, the kernel waited for memory once per layer with five
	// requests on their way (12 layers at 1920x1080: 140 -> 128 us, 4.2 TB/s; four pixels per thread with 16-byte loads: 132)
	constexpr int kAhead = 4;
	for (int k0 = 0; k0 < a.K; k0 += kAhead) {
		float v[kAhead][5] = {};
		const uint32_t filled = kStrips ? layers_with_entries<kAhead>(a, at, k0) : ~0u;
#pragma unroll
		for (int q = 0; q < kAhead; q++)
			if (k0 + q < a.K && (!kStrips || ((filled >> q) & 1u))) {
				const float* img = a.images[k0 + q];
				v[q][0] = img[p];
				v[q][1] = img[n + p];
				v[q][2] = img[2 * n + p];
				v[q][3] = a.depths[k0 + q][p];
				v[q][4] = a.alphas[k0 + q][p];
			}
#pragma unroll
		for (int q = 0; q < kAhead; q++)
			if (k0 + q < a.K) {
				r += T * v[q][0];
				g += T * v[q][1];
				b += T * v[q][2];
				d += T * v[q][3];
				T = T * (1.f - v[q][4]);
			}
	}
	float bg0 = 0.f, bg1 = 0.f, bg2 = 0.f;
	if (a.bg) {
		bg0 = a.bg[0];
		bg1 = a.bg[1];
		bg2 = a.bg[2];
	}
	a.out_image[p] = r + bg0 * T;
	a.out_image[n + p] = g + bg1 * T;
	a.out_image[2 * n + p] = b + bg2 * T;
	a.out_depth[p] = d;
	a.out_alpha[p] = 1.f - T;
}

// dL/dimage_k = T_k g, dL/ddepth_k = T_k g_d, dL/dalpha_k = -T_k R_k with
// R_{K-1} = <bg, g> - g_a and R_{k-1} = <image_k, g> + depth_k g_d + (1 - alpha_k) R_k.
// No division, so alpha_k = 1 is handled exactly.  T_k and alpha_k are kept per thread for the
// back-to-front sweep: in registers when the number of layers is at most kLayers (the loops are unrolled over kLayers
// and guarded by K, so the arrays are indexed by constants), otherwise (kLayers = 0) in an array indexed at run time,
// which the compiler places in scratch memory: every value then goes out to memory and comes back.
// kDepth: there is a gradient of the composited depth.  Without one the layers' depths are not read and their gradients
// (zero) are written only where the caller has planes for them; the kernel is bound by memory, and both are planes of K
// (12 layers at 1920x1080: 168 -> 135 us, 6 TB/s).
template <int kLayers, bool kDepth, bool kStrips>
__global__ __launch_bounds__(256) void composite_backward_kernel(CompositeArgs a)
{
	const size_t n = (size_t)a.H * a.W;
	const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
	if (p >= n)
		return;
	constexpr int kHeld = kLayers > 0 ? kLayers : kMaxComposite;
	float Tk[kHeld], alpha[kHeld];
	float T = 1.f;
	StripPlace at = {};
	uint32_t filled = ~0u;
	if (kStrips) {
		at = strip_of_pixel(a, p);
		if constexpr (kLayers > 0)
			filled = layers_with_entries<kLayers>(a, at, 0);
	}
	auto has = [&](int k) { return !kStrips || (kLayers > 0 ? (filled >> k) & 1u : layers_with_entries<1>(a, at, k)) != 0u; };
	if (kLayers > 0) {
#pragma unroll
		for (int k = 0; k < kLayers; k++)
			if (k < a.K) {
				alpha[k] = has(k) ? a.alphas[k][p] : 0.f;
				Tk[k] = T;
				T = T * (1.f - alpha[k]);
			}
	} else {
		for (int k = 0; k < a.K; k++) {
			alpha[k] = has(k) ? a.alphas[k][p] : 0.f;
			Tk[k] = T;
			T = T * (1.f - alpha[k]);
		}
	}
	const float gr = a.g_image[p], gg = a.g_image[n + p], gb = a.g_image[2 * n + p];
	const float gd = kDepth ? a.g_depth[p] : 0.f;
	const float ga = a.g_alpha ? a.g_alpha[p] : 0.f;
	float R = -ga;
	if (a.bg)
		R += a.bg[0] * gr + a.bg[1] * gg + a.bg[2] * gb;
	auto layer = [&](int k, float t, float alpha_k) {
		float* di = a.d_images[k];
		di[p] = t * gr;
		di[n + p] = t * gg;
		di[2 * n + p] = t * gb;
		if (kDepth || a.d_depths[k])
			a.d_depths[k][p] = t * gd;
		a.d_alphas[k][p] = -(t * R);
		float c0 = 0.f, c1 = 0.f, c2 = 0.f, depth = 0.f;
		if (has(k)) {
			const float* img = a.images[k];
			c0 = img[p];
			c1 = img[n + p];
			c2 = img[2 * n + p];
			if (kDepth)
				depth = a.depths[k][p];
		}
		const float colour = c0 * gr + c1 * gg + c2 * gb;
		R = (kDepth ? colour + depth * gd : colour) + (1.f - alpha_k) * R;
	};
	if (kLayers > 0) {
#pragma unroll
		for (int k = kLayers - 1; k >= 0; k--)
			if (k < a.K)
				layer(k, Tk[k], alpha[k]);
	} else {
		for (int k = a.K - 1; k >= 0; k--)
			layer(k, Tk[k], alpha[k]);
	}
}

void launch_composite_forward(const CompositeArgs& a, hipStream_t s)
{
	const size_t n = (size_t)a.H * a.W;
	stage_mark("composite_forward", s);
	const dim3 grid((unsigned)((n + 255) / 256));
	if (a.layer_bg)
		hipLaunchKernelGGL(composite_forward_kernel<true>, grid, dim3(256), 0, s, a);
	else
		hipLaunchKernelGGL(composite_forward_kernel<false>, grid, dim3(256), 0, s, a);
}

template <bool kDepth, bool kStrips>
static void launch_composite_backward_as(const CompositeArgs& a, hipStream_t s)
{
	const size_t n = (size_t)a.H * a.W;
	const dim3 grid((unsigned)((n + 255) / 256));
	if (a.K <= 4)
		hipLaunchKernelGGL((composite_backward_kernel<4, kDepth, kStrips>), grid, dim3(256), 0, s, a);
	else if (a.K <= 16)
		hipLaunchKernelGGL((composite_backward_kernel<16, kDepth, kStrips>), grid, dim3(256), 0, s, a);
	else
		hipLaunchKernelGGL((composite_backward_kernel<0, kDepth, kStrips>), grid, dim3(256), 0, s, a);
}

void launch_composite_backward(const CompositeArgs& a, hipStream_t s)
{
	stage_mark("composite_backward", s);
	if (a.g_depth && a.layer_bg)
		launch_composite_backward_as<true, true>(a, s);
	else if (a.g_depth)
		launch_composite_backward_as<true, false>(a, s);
	else if (a.layer_bg)
		launch_composite_backward_as<false, true>(a, s);
	else
		launch_composite_backward_as<false, false>(a, s);
}

}  // namespace rgs
