// The two steps either side of the renderer in a training iteration: the image loss
// (1 - lambda) L1 + lambda (1 - SSIM) with its gradient, and the Adam update of the parameters.
//
// SSIM (utils/loss_utils.py:39-63): five zero-padded 11x11 Gaussian-window (sigma 1.5) means per
// pixel and channel, of x, y, x^2, y^2 and xy, then
//   f = (2 mu1 mu2 + C1)(2 s12 + C2) / ((mu1^2 + mu2^2 + C1)(s11 + s22 + C2)),  C1 = 0.01^2, C2 = 0.03^2.
// The window is an outer product, so each mean is a row pass followed by a column pass.  A
// workgroup produces a 32x16 tile of one channel: the 42x26 pixels it needs go to LDS once, the
// row pass leaves 5 x 26 x 32 partial means in LDS, the column pass finishes them, and the
// per-pixel SSIM and |x - y| are summed per workgroup (a second kernel adds the partial sums in a
// fixed order, so the loss is reproducible).  For the backward the same kernel stores three
// derivative maps per pixel,
//   a = df/dmu1,  b = df/dE[x^2] = -f / B2,  c = df/dE[xy] = 2 A1 / (B1 B2),
// and the gradient is their windowed means: dL/dx(q) = W*a (q) + 2 x(q) W*b (q) + y(q) W*c (q),
// which the backward kernel computes with the same two passes.  Bound by HBM (44 bytes per pixel
// and channel over both kernels) and by LDS reads.
//
// Activation (scene/gaussian_nn_module.py:373-394): what a submodel's renderer and neighbours see
// is exp of the stored scales, sigmoid of the stored opacities, the normalised quaternions and the
// two SH parameter tensors joined: one flat pass forward and one backward.
//
// Adam (torch.optim.Adam as the reference configures it, scene/gaussian_nn_module.py:429-444:
// eps 1e-15, no weight decay, no amsgrad): one pass over parameter, gradient and both moments.
#include "rgs_device.h"
#include "rgs_kernels.h"

namespace rgs {

namespace {

constexpr int kLossTileW = 32, kLossTileH = 16;
constexpr int kHalo = 5, kTaps = 11;
constexpr int kRegionW = kLossTileW + 2 * kHalo, kRegionH = kLossTileH + 2 * kHalo;
constexpr int kRowRun = 4;   // columns a thread takes in the row pass (26 x 8 runs for 256 threads)
constexpr int kColRun = 2;   // rows a thread takes in the column pass (8 x 32 runs)
static_assert(kRegionH * (kLossTileW / kRowRun) <= 256 && (kLossTileH / kColRun) * kLossTileW == 256, "pass shapes");

__device__ __forceinline__ float block256_sum(float v, float* lds)
{
	v = wave_sum_to_lane63(v);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	if (lane == 63)
		lds[wave] = v;
	__syncthreads();
	const float total = lds[0] + lds[1] + lds[2] + lds[3];
	__syncthreads();
	return total;
}

// Workgroups are dealt to the 8 XCDs in turn, and each XCD has its own L2.  Workgroup b therefore
// takes tile (b % 8) * ceil(tiles / 8) + b / 8 of the row-major (channel, tile row, tile column)
// order: an XCD gets a contiguous band of tiles, and the halo a tile shares with its neighbours is
// fetched from memory once per band instead of once per tile.
struct LossTile {
	int channel, tx, ty;
	uint32_t linear;
	bool valid;
};

__device__ __forceinline__ LossTile loss_tile_of_block(const LossArgs& a)
{
	const uint32_t tiles_x = (a.W + kLossTileW - 1) / kLossTileW, tiles_y = (a.H + kLossTileH - 1) / kLossTileH;
	const uint32_t total = tiles_x * tiles_y * (uint32_t)a.C;
	const uint32_t per_xcd = (total + 7) / 8;
	LossTile t;
	t.linear = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
	t.valid = blockIdx.x / 8 < per_xcd && t.linear < total;
	const uint32_t in_plane = t.linear % (tiles_x * tiles_y);
	t.channel = (int)(t.linear / (tiles_x * tiles_y));
	t.ty = (int)(in_plane / tiles_x);
	t.tx = (int)(in_plane % tiles_x);
	return t;
}

__global__ __launch_bounds__(256) void ssim_forward_kernel(LossArgs a)
{
	__shared__ float sx[kRegionH][kRegionW + 1];
	__shared__ float sy[kRegionH][kRegionW + 1];
	__shared__ float rows[5][kRegionH][kLossTileW + 1];
	__shared__ float red[4];
	const int tid = threadIdx.x;
	const LossTile tile = loss_tile_of_block(a);
	if (!tile.valid)
		return;
	const size_t plane = (size_t)tile.channel * a.H * a.W;
	const int x0 = tile.tx * kLossTileW - kHalo, y0 = tile.ty * kLossTileH - kHalo;
	for (int i = tid; i < kRegionH * kRegionW; i += 256) {
		const int r = i / kRegionW, c = i % kRegionW;
		const int gx = x0 + c, gy = y0 + r;
		const bool inside = gx >= 0 && gx < a.W && gy >= 0 && gy < a.H;
		const size_t at = plane + (size_t)gy * a.W + gx;
		sx[r][c] = inside ? a.x[at] : 0.f;
		sy[r][c] = inside ? a.y[at] : 0.f;
	}
	__syncthreads();
	// row pass: a thread takes 4 neighbouring columns of one row, so 14 pixels of each image
	// feed 4 x 5 sums (28 LDS reads instead of 88)
	if (tid < kRegionH * (kLossTileW / kRowRun)) {
		const int r = tid / (kLossTileW / kRowRun), c0 = kRowRun * (tid % (kLossTileW / kRowRun));
		float u[kTaps + kRowRun - 1], v[kTaps + kRowRun - 1];
#pragma unroll
		for (int k = 0; k < kTaps + kRowRun - 1; k++) {
			u[k] = sx[r][c0 + k];
			v[k] = sy[r][c0 + k];
		}
#pragma unroll
		for (int o = 0; o < kRowRun; o++) {
			float m1 = 0.f, m2 = 0.f, xx = 0.f, yy = 0.f, xy = 0.f;
#pragma unroll
			for (int k = 0; k < kTaps; k++) {
				const float w = a.w[k];
				m1 += w * u[o + k];
				m2 += w * v[o + k];
				xx += w * (u[o + k] * u[o + k]);
				yy += w * (v[o + k] * v[o + k]);
				xy += w * (u[o + k] * v[o + k]);
			}
			rows[0][r][c0 + o] = m1; rows[1][r][c0 + o] = m2; rows[2][r][c0 + o] = xx; rows[3][r][c0 + o] = yy;
			rows[4][r][c0 + o] = xy;
		}
	}
	__syncthreads();
	float ssim_sum = 0.f, l1_sum = 0.f;
	// column pass: a thread takes kColRun rows of one column
	float part[5][kTaps + kColRun - 1];
	const int col = tid % kLossTileW, row0 = kColRun * (tid / kLossTileW);
#pragma unroll
	for (int q = 0; q < 5; q++)
#pragma unroll
		for (int k = 0; k < kTaps + kColRun - 1; k++)
			part[q][k] = rows[q][row0 + k][col];
#pragma unroll
	for (int o = 0; o < kColRun; o++) {
		const int r = row0 + o, c = col;
		const int gx = x0 + kHalo + c, gy = y0 + kHalo + r;
		if (gx >= a.W || gy >= a.H)
			continue;
		float m1 = 0.f, m2 = 0.f, xx = 0.f, yy = 0.f, xy = 0.f;
#pragma unroll
		for (int k = 0; k < kTaps; k++) {
			const float w = a.w[k];
			m1 += w * part[0][o + k];
			m2 += w * part[1][o + k];
			xx += w * part[2][o + k];
			yy += w * part[3][o + k];
			xy += w * part[4][o + k];
		}
		const float C1 = 0.01f * 0.01f, C2 = 0.03f * 0.03f;
		const float m11 = m1 * m1, m22 = m2 * m2, m12 = m1 * m2;
		const float s11 = xx - m11, s22 = yy - m22, s12 = xy - m12;
		const float A1 = 2.f * m12 + C1, A2 = 2.f * s12 + C2, B1 = m11 + m22 + C1, B2 = s11 + s22 + C2;
		const float inv = 1.f / (B1 * B2);
		const float f = A1 * A2 * inv;
		ssim_sum += f;
		l1_sum += fabsf(sx[r + kHalo][c + kHalo] - sy[r + kHalo][c + kHalo]);
		if (a.maps) {
			const size_t n = (size_t)a.C * a.H * a.W;
			const size_t at = plane + (size_t)gy * a.W + gx;
			a.maps[at] = 2.f * m2 * (A2 - A1) * inv - 2.f * m1 * f * (1.f / B1 - 1.f / B2);
			a.maps[n + at] = -f / B2;
			a.maps[2 * n + at] = 2.f * A1 * inv;
		}
	}
	ssim_sum = block256_sum(ssim_sum, red);
	l1_sum = block256_sum(l1_sum, red);
	if (tid == 0) {
		a.partial[2 * (size_t)tile.linear] = ssim_sum;
		a.partial[2 * (size_t)tile.linear + 1] = l1_sum;
	}
}

// One workgroup: the partial sums in index order (double accumulators), then the three results.
__global__ __launch_bounds__(256) void loss_finish_kernel(LossArgs a, uint32_t blocks)
{
	__shared__ double red[2][256];
	double s = 0.0, l = 0.0;
	for (uint32_t i = threadIdx.x; i < blocks; i += 256) {
		s += (double)a.partial[2 * i];
		l += (double)a.partial[2 * i + 1];
	}
	red[0][threadIdx.x] = s;
	red[1][threadIdx.x] = l;
	__syncthreads();
	for (int step = 128; step > 0; step >>= 1) {
		if ((int)threadIdx.x < step) {
			red[0][threadIdx.x] += red[0][threadIdx.x + step];
			red[1][threadIdx.x] += red[1][threadIdx.x + step];
		}
		__syncthreads();
	}
	if (threadIdx.x == 0) {
		const double n = (double)a.C * a.H * a.W;
		const float ssim = (float)(red[0][0] / n), l1 = (float)(red[1][0] / n);
		a.out[0] = (1.0f - a.lambda) * l1 + a.lambda * (1.0f - ssim);
		a.out[1] = l1;
		a.out[2] = ssim;
	}
}

__global__ __launch_bounds__(256) void ssim_backward_kernel(LossArgs a)
{
	__shared__ float sm[3][kRegionH][kRegionW + 1];
	__shared__ float rows[3][kRegionH][kLossTileW + 1];
	const int tid = threadIdx.x;
	const size_t n = (size_t)a.C * a.H * a.W;
	const LossTile tile = loss_tile_of_block(a);
	if (!tile.valid)
		return;
	const size_t plane = (size_t)tile.channel * a.H * a.W;
	const int x0 = tile.tx * kLossTileW - kHalo, y0 = tile.ty * kLossTileH - kHalo;
	for (int i = tid; i < kRegionH * kRegionW; i += 256) {
		const int r = i / kRegionW, c = i % kRegionW;
		const int gx = x0 + c, gy = y0 + r;
		const bool inside = gx >= 0 && gx < a.W && gy >= 0 && gy < a.H;
		const size_t at = plane + (size_t)gy * a.W + gx;
		sm[0][r][c] = inside ? a.maps[at] : 0.f;
		sm[1][r][c] = inside ? a.maps[n + at] : 0.f;
		sm[2][r][c] = inside ? a.maps[2 * n + at] : 0.f;
	}
	__syncthreads();
	if (tid < kRegionH * (kLossTileW / kRowRun)) {
		const int r = tid / (kLossTileW / kRowRun), c0 = kRowRun * (tid % (kLossTileW / kRowRun));
#pragma unroll
		for (int q = 0; q < 3; q++) {
			float u[kTaps + kRowRun - 1];
#pragma unroll
			for (int k = 0; k < kTaps + kRowRun - 1; k++)
				u[k] = sm[q][r][c0 + k];
#pragma unroll
			for (int o = 0; o < kRowRun; o++) {
				float acc = 0.f;
#pragma unroll
				for (int k = 0; k < kTaps; k++)
					acc += a.w[k] * u[o + k];
				rows[q][r][c0 + o] = acc;
			}
		}
	}
	__syncthreads();
	const float upstream = a.grad_loss ? a.grad_loss[0] : 1.0f;
	const float l1_scale = upstream * (1.0f - a.lambda) / (float)n, ssim_scale = -upstream * a.lambda / (float)n;
	float part[3][kTaps + kColRun - 1];
	const int col = tid % kLossTileW, row0 = kColRun * (tid / kLossTileW);
#pragma unroll
	for (int q = 0; q < 3; q++)
#pragma unroll
		for (int k = 0; k < kTaps + kColRun - 1; k++)
			part[q][k] = rows[q][row0 + k][col];
#pragma unroll
	for (int o = 0; o < kColRun; o++) {
		const int r = row0 + o, c = col;
		const int gx = x0 + kHalo + c, gy = y0 + kHalo + r;
		if (gx >= a.W || gy >= a.H)
			continue;
		float ca = 0.f, cb = 0.f, cc = 0.f;
#pragma unroll
		for (int k = 0; k < kTaps; k++) {
			const float w = a.w[k];
			ca += w * part[0][o + k];
			cb += w * part[1][o + k];
			cc += w * part[2][o + k];
		}
		const size_t at = plane + (size_t)gy * a.W + gx;
		const float x = a.x[at], y = a.y[at];
		const float d = x - y;
		const float sign = d > 0.f ? 1.f : (d < 0.f ? -1.f : 0.f);
		a.d_image[at] = l1_scale * sign + ssim_scale * (ca + 2.f * x * cb + y * cc);
	}
}

// torch.optim.Adam's single-tensor update, in its order of operations:
//   m = b1 m + (1 - b1) g;  v = b2 v + (1 - b2) g g;
//   p = p - (lr / (1 - b1^t)) * m / (sqrt(v) / sqrt(1 - b2^t) + eps)
// One launch updates every tensor of a parameter-group list; a workgroup takes kAdamBlock
// consecutive elements of one tensor.  Bound by memory, 28 bytes per element, none of which another kernel reads soon:
// streaming accesses leave the caches to the others and run at 5.7 instead of 4.9 TB/s (168 M floats: 965 us with plain accesses,
// 844 with the loads streaming, 828 with the stores as well; from 3.6 M floats on, the smallest tried, no slower).
constexpr int kAdamBlock = 4096;

__device__ __forceinline__ void adam_one(float& p, float g, float& m, float& v, const AdamTensor& t, const AdamArgs& a)
{
	m = m * a.beta1 + g * a.one_minus_beta1;
	v = v * a.beta2 + (g * g) * a.one_minus_beta2;
	const float denom = sqrtf(v) / t.bias2_sqrt + a.eps;
	p = p - t.step_size * (m / denom);
}

__global__ __launch_bounds__(256) void adam_step_kernel(AdamArgs a)
{
	int k = 0;
	while (k + 1 < a.tensors && blockIdx.x >= a.t[k + 1].block0)
		k++;
	const AdamTensor& t = a.t[k];
	const size_t base = (size_t)(blockIdx.x - t.block0) * kAdamBlock;
#pragma unroll
	for (int it = 0; it < kAdamBlock / 1024; it++) {
		const size_t i = base + (size_t)it * 1024 + threadIdx.x * 4;
		if (i >= t.n)
			break;
		if (i + 4 <= t.n && t.by_16_bytes) {
			float4 p = load_streaming(reinterpret_cast<const float4*>(t.param + i));
			const float4 g = load_streaming(reinterpret_cast<const float4*>(t.grad + i));
			float4 m = load_streaming(reinterpret_cast<const float4*>(t.exp_avg + i));
			float4 v = load_streaming(reinterpret_cast<const float4*>(t.exp_avg_sq + i));
			adam_one(p.x, g.x, m.x, v.x, t, a);
			adam_one(p.y, g.y, m.y, v.y, t, a);
			adam_one(p.z, g.z, m.z, v.z, t, a);
			adam_one(p.w, g.w, m.w, v.w, t, a);
			store_streaming(reinterpret_cast<float4*>(t.param + i), p);
			store_streaming(reinterpret_cast<float4*>(t.exp_avg + i), m);
			store_streaming(reinterpret_cast<float4*>(t.exp_avg_sq + i), v);
		} else {
			for (size_t j = i; j < t.n && j < i + 4; j++) {
				float p = t.param[j], m = t.exp_avg[j], v = t.exp_avg_sq[j];
				adam_one(p, t.grad[j], m, v, t, a);
				t.param[j] = p;
				t.exp_avg[j] = m;
				t.exp_avg_sq[j] = v;
			}
		}
	}
}

// Both activation kernels are flat passes over four arrays; a workgroup works on one of them (its part is the same for all
// its threads) and reads and writes 16 bytes per lane.  The SH rows are the one place where that takes care: a row of the joined
// tensor is 3 floats of one source followed by 3 * rest of the other.  A workgroup takes kActRows whole rows, whose floats are
// consecutive in all three tensors, and joins (or splits) them in LDS, where the shift by a row's 3 floats is 4-byte accesses.
// Bound by memory, 4 bytes read and 4 written per float.  With 4-byte accesses on the side of the two tensors, the form that is
// left for more coefficients than kActMaxRest and for arrays that do not start at a multiple of 16 bytes, 2.8 M Gaussians of 16
// coefficients took 268 us forward and 348 backward; now 220 and 240.
constexpr int kActUnits = 1024;   // 16-byte units per workgroup: 4 per thread
constexpr int kActRows = 128;     // SH rows per workgroup: six workgroups' rows fit a CU's LDS
constexpr int kActMaxRest = 15;
static_assert(kActRows % 4 == 0, "a workgroup's rows begin at a multiple of 16 bytes in each of the tensors");

__host__ __device__ inline uint32_t blocks_of(size_t units, size_t per_block) { return (uint32_t)((units + per_block - 1) / per_block); }

struct ActParts {
	uint32_t sh_blocks, rot_blocks, scale_blocks, opacity_blocks;
	uint32_t rest_reciprocal;  // 0: the SH rows go by 4-byte accesses, kActUnits per workgroup; otherwise kActRows rows per workgroup
};

// f / (3 rest) is (f * reciprocal) >> 20 for every float f of a workgroup's rows: the excess of the reciprocal over 2^20 / d,
// less than 1, adds f / 2^20 < 1 / d to the quotient.
static_assert((size_t)kActRows * 3 * kActMaxRest * 3 * kActMaxRest < (1u << 20), "exact division");

inline ActParts act_parts(int n, int rest, bool sh_by_16_bytes)
{
	const size_t sh_floats = 3 * (size_t)(1 + rest);
	ActParts p;
	const bool by_rows = sh_by_16_bytes && rest >= 1 && rest <= kActMaxRest;
	p.rest_reciprocal = by_rows ? ((1u << 20) + 3 * (uint32_t)rest - 1) / (3 * (uint32_t)rest) : 0u;
	p.sh_blocks = by_rows ? blocks_of((size_t)n, kActRows) : blocks_of(((size_t)n * sh_floats + 3) / 4, kActUnits);
	p.rot_blocks = blocks_of((size_t)n, kActUnits);
	p.scale_blocks = blocks_of(((size_t)n * 3 + 3) / 4, kActUnits);
	p.opacity_blocks = blocks_of(((size_t)n + 3) / 4, kActUnits);
	return p;
}

// Unit u (floats [4u, 4u+4)) of `total` floats that start at a multiple of 16 bytes.
__device__ __forceinline__ float4 read_unit(const float* __restrict__ in, uint32_t u, uint32_t total)
{
	if (4 * u + 4 <= total)
		return load_streaming(reinterpret_cast<const float4*>(in) + u);
	float4 v = {0.f, 0.f, 0.f, 0.f};
	if (4 * u < total)
		v.x = in[4 * u];
	if (4 * u + 1 < total)
		v.y = in[4 * u + 1];
	if (4 * u + 2 < total)
		v.z = in[4 * u + 2];
	return v;
}
__device__ __forceinline__ void write_unit(float* __restrict__ out, uint32_t u, uint32_t total, const float4 v)
{
	if (4 * u + 4 <= total) {
		store_streaming(reinterpret_cast<float4*>(out) + u, v);
		return;
	}
	if (4 * u < total)
		out[4 * u] = v.x;
	if (4 * u + 1 < total)
		out[4 * u + 1] = v.y;
	if (4 * u + 2 < total)
		out[4 * u + 2] = v.z;
}

// Where float f of a workgroup's dc or rest floats (floats_per_row of a row) lies among its joined rows.
struct JoinedPlace {
	uint32_t at, left;  // left: floats of the row from this one on
};
__device__ __forceinline__ JoinedPlace joined_place(uint32_t f, uint32_t floats_per_row, uint32_t reciprocal, uint32_t sh_floats, uint32_t shift)
{
	const uint32_t row = (f * reciprocal) >> 20, col = f - row * floats_per_row;
	return JoinedPlace{row * sh_floats + shift + col, floats_per_row - col};
}

constexpr uint32_t kThirds = ((1u << 20) + 2) / 3;  // the reciprocal of a row of dc

constexpr int kActRestTurns = (kActRows * 3 * kActMaxRest / 4 + 255) / 256, kActRowTurns = (kActRows * 3 * (1 + kActMaxRest) / 4 + 255) / 256;

// Rows [first, first + rows) of dc and rest joined into shs.
__device__ __forceinline__ void join_rows(const ActivateArgs& a, uint32_t reciprocal, size_t first, uint32_t rows, float* joined)
{
	const uint32_t tid = threadIdx.x, rest_floats = 3u * (uint32_t)a.rest, sh_floats = rest_floats + 3u;
	const uint32_t rest_total = rows * rest_floats, dc_total = 3u * rows, total = rows * sh_floats;
	const float* rest = a.features_rest + first * rest_floats;
	float4 v[kActRestTurns], d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
	for (int t = 0; t < kActRestTurns; t++)
		if (4 * (256 * t + tid) < rest_total)
			v[t] = read_unit(rest, 256 * t + tid, rest_total);
	if (4 * tid < dc_total)
		d = read_unit(a.features_dc + first * 3, tid, dc_total);
	auto place = [&](uint32_t f, uint32_t end, uint32_t floats_per_row, uint32_t recip, uint32_t shift, const float4 q) {
		const JoinedPlace p = joined_place(f, floats_per_row, recip, sh_floats, shift);
		const uint32_t gap = sh_floats - floats_per_row;  // between a row's last float and the next row's first
		const float x[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
		for (uint32_t k = 0; k < 4; k++)
			if (f + k < end)
				joined[p.at + k + (k >= p.left ? gap : 0u) + (k >= p.left + floats_per_row ? gap : 0u)] = x[k];
	};
#pragma unroll
	for (int t = 0; t < kActRestTurns; t++)
		place(4 * (256 * t + tid), rest_total, rest_floats, reciprocal, 3u, v[t]);
	place(4 * tid, dc_total, 3u, kThirds, 0u, d);
	__syncthreads();
	float* out = a.shs + first * sh_floats;
#pragma unroll
	for (int t = 0; t < kActRowTurns; t++) {
		const uint32_t u = 256 * t + tid;
		if (4 * u < total)
			write_unit(out, u, total, reinterpret_cast<const float4*>(joined)[u]);
	}
}

// ... and the gradient of those rows split.
__device__ __forceinline__ void split_rows(const ActivateBackwardArgs& a, uint32_t reciprocal, size_t first, uint32_t rows, float* joined)
{
	const uint32_t tid = threadIdx.x, rest_floats = 3u * (uint32_t)a.rest, sh_floats = rest_floats + 3u;
	const uint32_t rest_total = rows * rest_floats, dc_total = 3u * rows, total = rows * sh_floats;
	const float* in = a.g_shs + first * sh_floats;
	float4 v[kActRowTurns];
#pragma unroll
	for (int t = 0; t < kActRowTurns; t++)
		if (4 * (256 * t + tid) < total)
			v[t] = read_unit(in, 256 * t + tid, total);
#pragma unroll
	for (int t = 0; t < kActRowTurns; t++)
		if (4 * (256 * t + tid) < total)
			reinterpret_cast<float4*>(joined)[256 * t + tid] = v[t];
	__syncthreads();
	auto pick = [&](uint32_t f, uint32_t end, uint32_t floats_per_row, uint32_t recip, uint32_t shift) {
		const JoinedPlace p = joined_place(f, floats_per_row, recip, sh_floats, shift);
		const uint32_t gap = sh_floats - floats_per_row;
		float x[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
		for (uint32_t k = 0; k < 4; k++)
			if (f + k < end)
				x[k] = joined[p.at + k + (k >= p.left ? gap : 0u) + (k >= p.left + floats_per_row ? gap : 0u)];
		return float4{x[0], x[1], x[2], x[3]};
	};
#pragma unroll
	for (int t = 0; t < kActRestTurns; t++) {
		const uint32_t u = 256 * t + tid;
		if (4 * u < rest_total)
			write_unit(a.d_features_rest + first * rest_floats, u, rest_total, pick(4 * u, rest_total, rest_floats, reciprocal, 3u));
	}
	if (4 * tid < dc_total)
		write_unit(a.d_features_dc + first * 3, tid, dc_total, pick(4 * tid, dc_total, 3u, kThirds, 0u));
}

// Four 16-byte units of a flat array of `total` floats per thread, element by element where the array ends; f(value, other): `other`
// is the element of a second array (null: 0).
template <typename F>
__device__ __forceinline__ void flat_units(uint32_t block, size_t total, const float* __restrict__ in, const float* __restrict__ other,
                                           float* __restrict__ out, F f)
{
	constexpr int kTurns = kActUnits / 256;
	float4 v[kTurns], o[kTurns];
	const size_t u0 = (size_t)block * kActUnits + threadIdx.x;
#pragma unroll
	for (int t = 0; t < kTurns; t++)
		if (4 * (u0 + 256 * t) + 4 <= total) {
			v[t] = load_streaming(reinterpret_cast<const float4*>(in) + u0 + 256 * t);
			o[t] = other ? load_streaming(reinterpret_cast<const float4*>(other) + u0 + 256 * t) : float4{0.f, 0.f, 0.f, 0.f};
		}
#pragma unroll
	for (int t = 0; t < kTurns; t++) {
		const size_t u = u0 + 256 * t;
		if (4 * u + 4 <= total)
			store_streaming(reinterpret_cast<float4*>(out) + u,
			                float4{f(v[t].x, o[t].x), f(v[t].y, o[t].y), f(v[t].z, o[t].z), f(v[t].w, o[t].w)});
		else
			for (size_t k = 4 * u; k < total; k++)
				out[k] = f(in[k], other ? other[k] : 0.f);
	}
}

// The length that a quaternion is divided by (that of torch.nn.functional.normalize).  The order of the sum is written out: left to the compiler it
// differs from kernel to kernel, and a last bit of a rotation is 1e-4 of the gradient of a scene's worst conditioned Gaussian.
__device__ __forceinline__ float quaternion_length(const float4 q)
{
	return fmaxf(sqrtf(__builtin_fmaf(q.w, q.w, __builtin_fmaf(q.z, q.z, __builtin_fmaf(q.x, q.x, q.y * q.y)))), 1e-12f);
}

// kActUnits quaternions per workgroup: made unit ones, and the gradient through that.
__device__ __forceinline__ void unit_quaternions(uint32_t block, size_t n, const float* __restrict__ from, float* __restrict__ to)
{
	constexpr int kTurns = kActUnits / 256;
	const size_t i0 = (size_t)block * kActUnits + threadIdx.x;
	float4 v[kTurns];
#pragma unroll
	for (int t = 0; t < kTurns; t++)
		if (i0 + 256 * t < n)
			v[t] = load_streaming(reinterpret_cast<const float4*>(from) + i0 + 256 * t);
#pragma unroll
	for (int t = 0; t < kTurns; t++)
		if (i0 + 256 * t < n) {
			const float4 q = v[t];
			const float len = quaternion_length(q);
			store_streaming(reinterpret_cast<float4*>(to) + i0 + 256 * t, float4{q.x / len, q.y / len, q.z / len, q.w / len});
		}
}
__device__ __forceinline__ void unit_quaternions_backward(uint32_t block, size_t n, const float* __restrict__ from, const float* __restrict__ grad,
                                                          float* __restrict__ to)
{
	constexpr int kTurns = kActUnits / 256;
	const size_t i0 = (size_t)block * kActUnits + threadIdx.x;
	float4 v[kTurns], w[kTurns];
#pragma unroll
	for (int t = 0; t < kTurns; t++)
		if (i0 + 256 * t < n) {
			v[t] = load_streaming(reinterpret_cast<const float4*>(from) + i0 + 256 * t);
			w[t] = load_streaming(reinterpret_cast<const float4*>(grad) + i0 + 256 * t);
		}
#pragma unroll
	for (int t = 0; t < kTurns; t++)
		if (i0 + 256 * t < n) {
			// d/dq of q / |q|: (g - u (u . g)) / |q| with u = q / |q|
			const float4 q = v[t], g = w[t];
			const float len = quaternion_length(q);
			const float u0 = q.x / len, u1 = q.y / len, u2 = q.z / len, u3 = q.w / len;
			const float along = __builtin_fmaf(u3, g.w, __builtin_fmaf(u2, g.z, __builtin_fmaf(u0, g.x, u1 * g.y)));
			store_streaming(reinterpret_cast<float4*>(to) + i0 + 256 * t,
			                float4{(g.x - u0 * along) / len, (g.y - u1 * along) / len, (g.z - u2 * along) / len,
			                       (g.w - u3 * along) / len});
		}
}

__device__ __forceinline__ float activated_scale(float v) { return expf(v); }
__device__ __forceinline__ float activated_opacity(float v) { return 1.0f / (1.0f + expf(-v)); }

// Scales, rotations, opacities and the zeros of the screen-space placeholder of every stored model of a frame (blockIdx.y), in units as above.
__global__ __launch_bounds__(256) void activate_many_kernel(Batch<ActivateJob> batch)
{
	const ActivateJob& j = batch.job[blockIdx.y];
	const size_t n = (size_t)j.n;
	uint32_t block = blockIdx.x;
	const uint32_t rot_blocks = blocks_of(n, kActUnits), scale_blocks = blocks_of((3 * n + 3) / 4, kActUnits),
	               opacity_blocks = blocks_of((n + 3) / 4, kActUnits);
	if (block < rot_blocks) {
		unit_quaternions(block, n, j.rotation, j.rotations);
		return;
	}
	block -= rot_blocks;
	if (block < scale_blocks) {
		flat_units(block, 3 * n, j.scaling, nullptr, j.scales, [](float v, float) { return activated_scale(v); });
		return;
	}
	block -= scale_blocks;
	if (block < opacity_blocks) {
		flat_units(block, n, j.opacity, nullptr, j.opacities, [](float v, float) { return activated_opacity(v); });
		return;
	}
	block -= opacity_blocks;
	const size_t floats = 3 * (size_t)j.zero_rows;
#pragma unroll
	for (int t = 0; t < kActUnits / 256; t++) {
		const size_t at = 4 * ((size_t)block * kActUnits + 256 * t + threadIdx.x);
		if (at + 4 <= floats)
			*reinterpret_cast<float4*>(j.means2D + at) = float4{0.f, 0.f, 0.f, 0.f};
		else
			for (size_t k = at; k < floats; k++)
				j.means2D[k] = 0.f;
	}
}

__global__ __launch_bounds__(256) void activate_many_backward_kernel(Batch<ActivateBackwardJob> batch)
{
	const ActivateBackwardJob& j = batch.job[blockIdx.y];
	const size_t n = (size_t)j.n;
	uint32_t block = blockIdx.x;
	const uint32_t rot_blocks = blocks_of(n, kActUnits), scale_blocks = blocks_of((3 * n + 3) / 4, kActUnits),
	               opacity_blocks = blocks_of((n + 3) / 4, kActUnits);
	if (block < rot_blocks) {
		unit_quaternions_backward(block, n, j.rotation, j.g_rotations, j.d_rotation);
		return;
	}
	block -= rot_blocks;
	if (block < scale_blocks) {
		flat_units(block, 3 * n, j.g_scales, j.scales, j.d_scaling, [](float g, float s) { return g * s; });
		return;
	}
	block -= scale_blocks;
	if (block < opacity_blocks) {
		flat_units(block, n, j.g_opacities, j.opacities, j.d_opacity, [](float g, float o) { return g * (o * (1.0f - o)); });
		return;
	}
	block -= opacity_blocks;
	float x[kActUnits / 256], y[kActUnits / 256];
	const size_t i0 = (size_t)block * kActUnits + threadIdx.x;
#pragma unroll
	for (int t = 0; t < kActUnits / 256; t++)
		if (i0 + 256 * t < n) {
			x[t] = j.g_means2D[3 * (i0 + 256 * t)];
			y[t] = j.g_means2D[3 * (i0 + 256 * t) + 1];
		}
#pragma unroll
	for (int t = 0; t < kActUnits / 256; t++)
		if (i0 + 256 * t < n)
			j.d_meta[i0 + 256 * t] = sqrtf(x[t] * x[t] + y[t] * y[t]);
}

__global__ __launch_bounds__(256) void activate_forward_kernel(ActivateArgs a, ActParts parts)
{
	__shared__ __attribute__((aligned(16))) float joined[kActRows * 3 * (1 + kActMaxRest)];
	uint32_t block = blockIdx.x;
	const size_t n = (size_t)a.n;
	if (block < parts.sh_blocks) {
		if (parts.rest_reciprocal != 0u) {
			const size_t first = (size_t)block * kActRows;
			join_rows(a, parts.rest_reciprocal, first, (uint32_t)min((size_t)kActRows, n - first), joined);
			return;
		}
		const size_t sh_floats = 3 * (size_t)(1 + a.rest), rest_floats = 3 * (size_t)a.rest, total = n * sh_floats;
		for (int it = 0; it < kActUnits / 256; it++) {
			const size_t u = (size_t)block * kActUnits + it * 256 + threadIdx.x;
			if (4 * u >= total)
				break;
			float v[4];
#pragma unroll
			for (int k = 0; k < 4; k++) {
				const size_t at = 4 * u + k;
				if (at < total) {
					const size_t row = at / sh_floats, col = at - row * sh_floats;
					v[k] = col < 3 ? a.features_dc[3 * row + col] : a.features_rest[rest_floats * row + (col - 3)];
				} else {
					v[k] = 0.f;
				}
			}
			if (4 * u + 4 <= total)
				reinterpret_cast<float4*>(a.shs)[u] = float4{v[0], v[1], v[2], v[3]};
			else
				for (size_t k = 4 * u; k < total; k++)
					a.shs[k] = v[k - 4 * u];
		}
		return;
	}
	block -= parts.sh_blocks;
	if (block < parts.rot_blocks) {
		unit_quaternions(block, n, a.rotation, a.rotations);
		return;
	}
	block -= parts.rot_blocks;
	if (block < parts.scale_blocks) {
		flat_units(block, 3 * n, a.scaling, nullptr, a.scales, [](float v, float) { return activated_scale(v); });
		return;
	}
	block -= parts.scale_blocks;
	flat_units(block, n, a.opacity, nullptr, a.opacities, [](float v, float) { return activated_opacity(v); });
}

__global__ __launch_bounds__(256) void activate_backward_kernel(ActivateBackwardArgs a, ActParts parts)
{
	__shared__ __attribute__((aligned(16))) float joined[kActRows * 3 * (1 + kActMaxRest)];
	uint32_t block = blockIdx.x;
	const size_t n = (size_t)a.n;
	if (block < parts.sh_blocks) {
		if (!a.g_shs)
			return;
		if (parts.rest_reciprocal != 0u) {
			const size_t first = (size_t)block * kActRows;
			split_rows(a, parts.rest_reciprocal, first, (uint32_t)min((size_t)kActRows, n - first), joined);
			return;
		}
		const size_t sh_floats = 3 * (size_t)(1 + a.rest), rest_floats = 3 * (size_t)a.rest, total = n * sh_floats;
		for (int it = 0; it < kActUnits / 256; it++) {
			const size_t u = (size_t)block * kActUnits + it * 256 + threadIdx.x;
			if (4 * u >= total)
				break;
			float v[4] = {0.f, 0.f, 0.f, 0.f};
			if (4 * u + 4 <= total) {
				const float4 g = reinterpret_cast<const float4*>(a.g_shs)[u];
				v[0] = g.x; v[1] = g.y; v[2] = g.z; v[3] = g.w;
			} else {
				for (size_t k = 4 * u; k < total; k++)
					v[k - 4 * u] = a.g_shs[k];
			}
#pragma unroll
			for (int k = 0; k < 4; k++) {
				const size_t at = 4 * u + k;
				if (at < total) {
					const size_t row = at / sh_floats, col = at - row * sh_floats;
					if (col < 3)
						a.d_features_dc[3 * row + col] = v[k];
					else
						a.d_features_rest[rest_floats * row + (col - 3)] = v[k];
				}
			}
		}
		return;
	}
	block -= parts.sh_blocks;
	if (block < parts.rot_blocks) {
		if (!a.g_rotations)
			return;
		unit_quaternions_backward(block, n, a.rotation, a.g_rotations, a.d_rotation);
		return;
	}
	block -= parts.rot_blocks;
	if (block < parts.scale_blocks) {
		if (a.g_scales)
			flat_units(block, 3 * n, a.g_scales, a.scales, a.d_scaling, [](float g, float s) { return g * s; });
		return;
	}
	block -= parts.scale_blocks;
	if (a.g_opacities)
		flat_units(block, n, a.g_opacities, a.opacities, a.d_opacity, [](float g, float o) { return g * (o * (1.0f - o)); });
}

}  // namespace

void launch_activate_forward(const ActivateArgs& a, hipStream_t s)
{
	stage_mark("activate_forward", s);
	if (a.n <= 0)
		return;
	const ActParts p = act_parts(a.n, a.rest, a.features_by_16_bytes);
	hipLaunchKernelGGL(activate_forward_kernel, dim3(p.sh_blocks + p.rot_blocks + p.scale_blocks + p.opacity_blocks), dim3(256),
	                   0, s, a, p);
}

void launch_activate_backward(const ActivateBackwardArgs& a, hipStream_t s)
{
	stage_mark("activate_backward", s);
	if (a.n <= 0)
		return;
	const ActParts p = act_parts(a.n, a.rest, a.features_by_16_bytes);
	hipLaunchKernelGGL(activate_backward_kernel, dim3(p.sh_blocks + p.rot_blocks + p.scale_blocks + p.opacity_blocks), dim3(256),
	                   0, s, a, p);
}

void launch_activate_many(const ActivateJob* jobs, int count, hipStream_t s)
{
	stage_mark("activate_forward", s);
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<ActivateJob> b;
		uint32_t most = 0;
		for (int k = 0; k < nj; k++) {
			const ActivateJob& j = b.job[k] = jobs[at + k];
			const size_t n = (size_t)j.n;
			const uint32_t blocks = blocks_of(n, kActUnits) + blocks_of((3 * n + 3) / 4, kActUnits) + blocks_of((n + 3) / 4, kActUnits) +
			                        blocks_of((3 * (size_t)j.zero_rows + 3) / 4, kActUnits);
			most = blocks > most ? blocks : most;
		}
		if (most)
			hipLaunchKernelGGL(activate_many_kernel, dim3(most, (unsigned)nj), dim3(256), 0, s, b);
	}
}

void launch_activate_many_backward(const ActivateBackwardJob* jobs, int count, hipStream_t s)
{
	stage_mark("activate_backward", s);
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<ActivateBackwardJob> b;
		uint32_t most = 0;
		for (int k = 0; k < nj; k++) {
			const size_t n = (size_t)(b.job[k] = jobs[at + k]).n;
			const uint32_t blocks = 2 * blocks_of(n, kActUnits) + blocks_of((3 * n + 3) / 4, kActUnits) + blocks_of((n + 3) / 4, kActUnits);
			most = blocks > most ? blocks : most;
		}
		if (most)
			hipLaunchKernelGGL(activate_many_backward_kernel, dim3(most, (unsigned)nj), dim3(256), 0, s, b);
	}
}

uint32_t loss_blocks(int C, int H, int W)
{
	return (uint32_t)(((W + kLossTileW - 1) / kLossTileW) * ((H + kLossTileH - 1) / kLossTileH) * C);
}

void launch_l1_ssim_forward(const LossArgs& a, hipStream_t s)
{
	stage_mark("l1_ssim_forward", s);
	const uint32_t grid = 8 * ((loss_blocks(a.C, a.H, a.W) + 7) / 8);
	hipLaunchKernelGGL(ssim_forward_kernel, dim3(grid), dim3(256), 0, s, a);
	hipLaunchKernelGGL(loss_finish_kernel, dim3(1), dim3(256), 0, s, a, loss_blocks(a.C, a.H, a.W));
}

void launch_l1_ssim_backward(const LossArgs& a, hipStream_t s)
{
	stage_mark("l1_ssim_backward", s);
	const uint32_t grid = 8 * ((loss_blocks(a.C, a.H, a.W) + 7) / 8);
	hipLaunchKernelGGL(ssim_backward_kernel, dim3(grid), dim3(256), 0, s, a);
}

uint32_t adam_blocks_for(size_t n)
{
	return (uint32_t)((n + kAdamBlock - 1) / kAdamBlock);
}

void launch_adam_step(const AdamArgs& a, uint32_t blocks, hipStream_t s)
{
	stage_mark("adam_step", s);
	if (blocks)
		hipLaunchKernelGGL(adam_step_kernel, dim3(blocks), dim3(256), 0, s, a);
}

}  // namespace rgs
