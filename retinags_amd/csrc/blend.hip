// Per-tile alpha blending, forward and backward.  A 16x16 tile is four strips of 16x4 pixels;
// a wavefront owns one strip, one pixel per lane, and every strip is a workgroup of its own
// (strips end at very different times, and a wave slot should not idle until its tile's longest
// strip is done); the backward takes the longest strips first.
//
// Compiled with -ffp-contract=off: every per-pixel decision (power > 0, alpha < 1/255,
// the half-Gaussian box test, T(1-alpha) < 1e-4) is evaluated with the unfused
// single-precision expressions of K/cuda_rasterizer_hgs/forward.cu:338-392
// (K = rasterization_kernels/diff-gaussian-rasterization-half-gaussian), so a pixel
// can only differ from that evaluation through the last bits of exp() (exp_of_exponent below).
//
// Blending front to back gives a strip no parallelism beyond its 64 pixels, but deciding which
// entries of a tile's list can matter to a strip needs no order at all.  So the work is split:
// the kernel that emits the (Gaussian, tile) instances decides for each of them which of the
// tile's four strips it can matter to (strip_filing.h) and sends that along with the tile key
// through the sort; a placing kernel turns the sorted bits into one list per strip (the list
// positions that matter to it, in list order); the blend kernels then walk only those, in chunks
// of 64 (lane l takes entry l of the chunk; the next chunk's records, the ids of the one after and
// the positions of the one after that are already in flight while the current chunk is
// processed).  With many small Gaussians a tile's list runs to tens of thousands of entries of
// which a strip needs a few thousand at most.  The backward walks the same filed lists, up to the
// last entry any pixel blended.  The forward narrows a step further: of each chunk it packs, per
// 8-pixel-wide half of the strip, the entries whose ellipse reaches that half, and the lanes of
// each half walk their own packed entries side by side (as many steps as the longer of the two).
//
// (Inside the walk the floor power >= -ln(255 * opacity), which alpha >= 1/255 needs and the packing uses, is not looked at
// again: skipping a group of four entries that no live lane reaches, before exp() is evaluated, costs more than it saves where
// most visited entries blend somewhere.  Without the test and with it (in a build for five wavefronts per SIMD, since it needs
// registers that six do not leave), us: 287 and 300 at 1600x1036 with 5.6 M Gaussians, 1847 and 1919 at 5185x3359, 158 and 168
// for the view of a city; but 924 and 896 for the scene of 62.9 M Gaussians, where one visit in twenty blends.)
#include "rgs_kernels.h"
#include "strip_filing.h"
#include "tile_order.h"

namespace rgs {

struct PixelRay {
	float ndc_x, ndc_y;  // pixel centre in NDC
};

// NDC of a strip's pixel columns and rows, in LDS: only chunks that straddle a face of the box use them, and in registers
// they would cost the walks of all others two.
struct StripRays {
	float x[16], y[4];
};
__device__ __forceinline__ void stage_rays(StripRays& r, const float2 pixf, const BlendArgs& a, int lane)
{
	int W = a.W, H = a.H;
	asm volatile("" : "+s"(W), "+s"(H));  // (converted here each time: four registers held from strip to strip otherwise)
	r.x[lane & 15] = pix_to_ndc(pixf.x, W);  // (four lanes write the same value)
	r.y[lane >> 4] = pix_to_ndc(pixf.y, H);
}
__device__ __forceinline__ PixelRay ray_of(const StripRays& r)
{
	const int lane = threadIdx.x & 63;
	return PixelRay{r.x[lane & 15], r.y[lane >> 4]};
}

__device__ __forceinline__ PixelRay ray_of(const PixelRay& r) { return r; }

__device__ __forceinline__ BoxFrame load_box_frame(const BlendArgs& a)
{
	return load_box_frame(a.projinv, a.range_low, a.range_up, a.tanfovx, a.tanfovy);
}

// World-space point of the pixel's ray at clip-w `w`, tested against the submodel box
// (low, up] (K/cuda_rasterizer_hgs/forward.cu:360-372).  True when the sample is clipped.
__device__ __forceinline__ bool clipped_by_box(const PixelRay& ray, float w, const BoxFrame& b)
{
	const float3 ph = {ray.ndc_x * (w + 0.0000001f) * b.tanx, ray.ndc_y * (w + 0.0000001f) * b.tany, w};
	const float wx = b.m[0][0] * ph.x + b.m[1][0] * ph.y + b.m[2][0] * ph.z + b.m[3][0];
	const float wy = b.m[0][1] * ph.x + b.m[1][1] * ph.y + b.m[2][1] * ph.z + b.m[3][1];
	const float wz = b.m[0][2] * ph.x + b.m[1][2] * ph.y + b.m[2][2] * ph.z + b.m[3][2];
	return (wx <= b.lo.x) || (wx > b.hi.x) || (wy <= b.lo.y) || (wy > b.hi.y) || (wz <= b.lo.z) || (wz > b.hi.z);
}

// The clip w, all positive, between which clipped_by_box() lets a sample of a pixel's ray pass: at none outside of
// [from, to], at all inside of (from_sure, to_sure).  The ray sample's world coordinates are affine in clip w, slope w +
// offset, so each face of the box bounds w on one side; slope and offset get room for the rounding of the exact test (about
// seven roundings of half a unit each, relative to the terms and not to their possibly cancelling sum) and of this one.
// Four comparisons with it replace the exact test, which is as long as all the rest of a visit, for nearly every sample.
struct BoxSpan {
	float from, to, from_sure, to_sure;
};

__device__ __forceinline__ BoxSpan w_inside_box(const PixelRay& ray, const BoxFrame& b)
{
	const float rx = ray.ndc_x * b.tanx, ry = ray.ndc_y * b.tany;
	const float lo[3] = {b.lo.x, b.lo.y, b.lo.z}, hi[3] = {b.hi.x, b.hi.y, b.hi.z};
	BoxSpan s = {0.f, INFINITY, 0.f, INFINITY};
#pragma unroll
	for (int k = 0; k < 3; k++) {
		const float t0 = b.m[0][k] * rx, t1 = b.m[1][k] * ry, t2 = b.m[2][k], offset = b.m[3][k];
		const float slope = t0 + t1 + t2, room = 2e-6f * (fabsf(t0) + fabsf(t1) + fabsf(t2));
		const float room_offset = 2e-6f * fabsf(offset) + 2e-7f * (fabsf(t0) + fabsf(t1));  // (and for the exact test's w + 1e-7)
		// slope w > lo - offset and, mirrored, -slope w > -(hi - offset)
#pragma unroll
		for (int side = 0; side < 2; side++) {
			const float rise = side ? -slope : slope, need = side ? offset - hi[k] : lo[k] - offset;
			const float rise_p = rise + room, rise_s = rise - room;
			const float at_p = (need - room_offset) * __builtin_amdgcn_rcpf(rise_p);
			const float at_s = (need + room_offset) * __builtin_amdgcn_rcpf(rise_s);
			s.from = fmaxf(s.from, rise_p > 0.f ? at_p : 0.f);
			s.to = fminf(s.to, rise_p < 0.f ? at_p : INFINITY);
			s.from_sure = fmaxf(s.from_sure, rise_s > 0.f ? at_s : rise_s < 0.f ? 0.f : INFINITY);
			s.to_sure = fminf(s.to_sure, rise_s < 0.f ? at_s : INFINITY);
		}
	}
	return BoxSpan{s.from * 0.9999f, s.to * 1.0001f, s.from_sure * 1.0001f, s.to_sure * 0.9999f};
}

// The lanes among `lanes` whose sample at clip w the box does not clip (a NaN, which marks an entry that has the whole
// strip inside the box: all of them).
template <typename Rays>
__device__ __forceinline__ uint64_t lanes_inside_box(uint64_t lanes, float w, const BoxSpan& s, const Rays& rays, const BlendArgs& a)
{
	lanes &= ~(lanes_where(w < s.from) | lanes_where(w > s.to));
	const uint64_t unsure = lanes & (lanes_where(w <= s.from_sure) | lanes_where(w >= s.to_sure));
	if (unsure != 0ull)
		lanes &= ~lanes_where(clipped_by_box(ray_of(rays), w, load_box_frame(a)));
	return lanes;
}
// The same for the entries of a group: their comparisons stand together and one branch is for all of them.  (A branch per entry waits for
// its comparisons each time, and the walks that last longest are those along a face of the box: forward of four submodels of 5.6 M, a call
// each, 435 -> 410 us; in one launch 254 -> 247; 62.9 M 730 -> 716.  The backward, which has more to do between them, gained nothing.)
template <int kEntries, typename Rays>
__device__ __forceinline__ void keep_lanes_inside_box(uint64_t (&mask)[kEntries], const float (&w)[kEntries], const BoxSpan& s, const Rays& rays, const BlendArgs& a)
{
	uint64_t unsure[kEntries], any = 0ull;
#pragma unroll
	for (int i = 0; i < kEntries; i++) {
		mask[i] &= ~(lanes_where(w[i] < s.from) | lanes_where(w[i] > s.to));
		unsure[i] = mask[i] & (lanes_where(w[i] <= s.from_sure) | lanes_where(w[i] >= s.to_sure));
		any |= unsure[i];
	}
	if (any != 0ull)
#pragma unroll
		for (int i = 0; i < kEntries; i++)
			if (unsure[i] != 0ull)
				mask[i] &= ~lanes_where(clipped_by_box(ray_of(rays), w[i], load_box_frame(a)));
}
// The same by the exact test alone, where some entry of the chunk lies at a clip w that is not positive.
template <typename Rays>
__device__ __forceinline__ uint64_t lanes_inside_box(uint64_t lanes, float w, const Rays& rays, const BlendArgs& a)
{
	return lanes & ~lanes_where(clipped_by_box(ray_of(rays), w, load_box_frame(a)));
}
// How a chunk's samples are tested against the box: not at all (it has the strip inside for every entry), by spans, exactly.
enum BoxTest { kBoxNone, kBoxSpans, kBoxExact };

// exp(x) for the exponents of the blend (-6 < x <= 0 where the result is used): 2^(x log2 e) on the hardware exp2 unit.
// The product's rounding (half a unit in the last place of a number below 8) and the unit's own leave the result within
// four units in the last place, the class of a library expf; the decisions taken on it (alpha against 1/255, the
// transmittance against 1e-4) agree with an exact evaluation except within a few 1e-7 of their thresholds.  Forward
// and backward use the same function, so they take the same per-pixel decisions.
__device__ __forceinline__ float exp_of_exponent(float x)
{
	return __builtin_amdgcn_exp2f(x * 1.44269502e+0f);
}

// Launch-order classes of the backward's strips, by the number of entries they have to walk.
constexpr int kStripClasses = 256;
constexpr uint32_t kEmptyClass = kStripClasses;  // of the strips without entries: the last ones of an order
__device__ __forceinline__ uint32_t strip_class(uint32_t filed) { return filed == 0u ? kEmptyClass : 255u - min(filed >> 3, 255u); }
// Words of strip_classes behind the counters and cursors of the two orders (1: the forward's, 0: the backward's).
constexpr int kStripTail = 4 * kStripClasses;
constexpr int strip_empty_word(int forward) { return kStripTail + 2 * forward; }  // how many strips are empty; behind it the placement cursor
constexpr int kStripLongWord = kStripTail + 4;   // how many strips at the front of the backward's order four wavefronts walk
constexpr int kStripTotalWord = kStripTail + 5;  // the entries of all strips that the backward walks (where two kernels order them)
static_assert(kStripTotalWord < kRangeTailWords, "the words lie behind the ranges");

constexpr int kPerLane = 1;             // list entries per lane and step (2 was measured slower)
constexpr int kChunk = 64 * kPerLane;   // list entries a wavefront takes per step

// What the backward reads of a record: it takes the forward's word for which entries matter.
struct LoadedRecord {
	float4 geom, conic, cd;
	uint32_t id;
};

__device__ __forceinline__ LoadedRecord load_record(const BlendArgs& a, uint32_t id, bool in_range)
{
	LoadedRecord e;
	id = min(id, a.gaussians - 1u);  // (a list that is not this frame's must not lead outside the records)
	e.id = id;
	if (in_range) {
		const float4* rec = a.record + 4 * (size_t)id;
		e.geom = rec[0];
		e.conic = rec[1];
		e.cd = rec[2];
	} else {
		e.geom = float4{0.f, 0.f, INFINITY, 0.f};
		e.conic = float4{0.f, 0.f, 0.f, 0.f};
		e.cd = float4{0.f, 0.f, 0.f, 0.f};
	}
	return e;
}

__device__ __forceinline__ float exponent_of(const float4 g, const float4 co, const float2 pixf, float2& d)
{
	d = float2{g.x - pixf.x, g.y - pixf.y};
	return -0.5f * (co.x * d.x * d.x + co.z * d.y * d.y) - co.y * d.x * d.y;
}

// The blend kernels stage a conic as (-xx / 2, -xy, -yy / 2, opacity): scaling by a power of two and negation commute
// with rounding, so the exponent below has the very bits of exponent_of() on the conic as stored, one multiplication less
// per pixel and entry.
__device__ __forceinline__ float4 staged_conic(const float4 co) { return float4{-0.5f * co.x, -co.y, -0.5f * co.z, co.w}; }
__device__ __forceinline__ float exponent_of_staged(const float4 g, const float4 sc, const float2 pixf)
{
	const float dx = g.x - pixf.x, dy = g.y - pixf.y;
	return (sc.x * dx * dx + sc.z * dy * dy) + sc.y * dx * dy;
}

__device__ __forceinline__ float exponent_of_staged(const float4 centre_conic, float conic_yy, const float2 pixf)
{
	const float dx = centre_conic.x - pixf.x, dy = centre_conic.y - pixf.y;
	return (centre_conic.z * dx * dx + conic_yy * dy * dy) + centre_conic.w * dx * dy;
}

// ---- filing ------------------------------------------------------------------------------------
// The sorted keys carry, above the tile, one bit per strip the entry is filed for and one per strip
// that lies inside the box (key_strips).  A workgroup takes kFileGroup consecutive positions of the
// sorted list, whichever tiles they belong to, four neighbouring positions per thread.  An entry's rank
// in its strip's list is the number of filed entries of its tile before it: those inside the workgroup
// follow from a prefix count over the workgroup (per thread in LDS, four strips packed 16 bits each),
// taken at the entry and at the place where its tile begins; those in earlier workgroups (only the
// tile of the workgroup's first entry can have any) are the sum, over the workgroups since that tile
// began, of what each filed for the tile of its LAST entry, which the tile-range kernel has left in
// file_tail.  The thread that holds a tile's last entry also writes the strips' totals.

// Counts of the four strips packed in two words, 16 bits each (a workgroup files at most kFileGroup per strip).
__device__ __forceinline__ uint2 packed_strip_bits(uint32_t bits)
{
	return uint2{(bits & 1u) | ((bits & 2u) << 15), ((bits >> 2) & 1u) | ((bits & 8u) << 13)};
}

struct FileStage {
	uint2 before[kFileBlock];   // entries filed by the threads before this one
	uint16_t bits[kFileBlock];  // the filed bits of the thread's four positions, four bits each
	uint2 wave_total[4];
	uint32_t carry[4][4];       // [wave][strip] partial sums of the earlier workgroups' counts
};

// Entries filed at positions [0, i) of the workgroup.
__device__ __forceinline__ uint2 filed_before(const FileStage& st, uint32_t i)
{
	const uint32_t t = i >> 2, q = i & 3u;
	uint2 n = st.before[t];
	const uint32_t bits = st.bits[t];
#pragma unroll
	for (uint32_t k = 0; k < 3; k++)
		if (k < q) {
			const uint2 c = packed_strip_bits((bits >> (4 * k)) & 0xFu);
			n.x += c.x;
			n.y += c.y;
		}
	return n;
}

__global__ __launch_bounds__(kFileBlock) void strip_file_place_kernel(BlendBatch batch)
{
	__shared__ FileStage st;
	const BlendArgs& a = batch.job[blockIdx.y];
	const uint32_t capacity = a.capacity;
	const uint32_t first = blockIdx.x * (uint32_t)kFileGroup;
	if (first >= capacity)
		return;
	// A workgroup lives as long as its chain of reads: the keys (there is room for `capacity`, whatever they hold), the statuses and the
	// count are asked for together (71 M entries 262 -> 255 us, 42 M 132 -> 127).
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const uint32_t pos0 = first + 4u * (uint32_t)tid;
	uint32_t key[4] = {0u, 0u, 0u, 0u};
	if (pos0 + 3u < capacity) {
		const uint4 k4 = *reinterpret_cast<const uint4*>(a.tile_keys + pos0);
		key[0] = k4.x; key[1] = k4.y; key[2] = k4.z; key[3] = k4.w;
	} else {
#pragma unroll
		for (int q = 0; q < 4; q++)
			if (pos0 + (uint32_t)q < capacity)
				key[q] = a.tile_keys[pos0 + q];
	}
	const uint32_t first_key = a.tile_keys[first];
	const uint32_t gave_up = (a.sort_status ? *a.sort_status : 0u) | (a.order_status ? *a.order_status : 0u);
	const uint32_t R = a.count_device ? min(capacity, *a.count_device) : capacity;
	// after a sort that gave up the list is not sorted and the tile ranges are empty: nothing to place
	if (first >= R || gave_up != 0u)
		return;
	uint2 range[4];
	uint32_t filed[4];
	uint2 own = {0u, 0u};
	uint32_t all = 0;
#pragma unroll
	for (int q = 0; q < 4; q++) {
		const bool valid = pos0 + (uint32_t)q < R;
		range[q] = valid ? a.ranges[key_tile(key[q])] : uint2{0u, 0u};
		filed[q] = valid ? (key_strips(key[q]) & 0xFu) : 0u;
		const uint2 c = packed_strip_bits(filed[q]);
		own.x += c.x;
		own.y += c.y;
		all |= filed[q] << (4 * q);
	}
	const uint2 inc = {wave_inclusive_scan_u32(own.x), wave_inclusive_scan_u32(own.y)};
	if (lane == 63)
		st.wave_total[wave] = inc;
	st.bits[tid] = (uint16_t)all;
	// what the tile of this workgroup's first entry filed in the workgroups before this one
	{
		const uint32_t begin0 = a.ranges[key_tile(first_key)].x;
		uint4 sum = {0u, 0u, 0u, 0u};
		if (begin0 < first)
			for (uint32_t g = begin0 / (uint32_t)kFileGroup + (uint32_t)tid; g < blockIdx.x; g += kFileBlock) {
				const uint4 t = a.file_tail[g];
				sum.x += t.x; sum.y += t.y; sum.z += t.z; sum.w += t.w;
			}
		uint32_t v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
		for (int s = 0; s < 4; s++) {
			const uint32_t tot = wave_inclusive_scan_u32(v[s]);
			if (lane == 63)
				st.carry[wave][s] = tot;
		}
	}
	__syncthreads();
	uint2 mine = {inc.x - own.x, inc.y - own.y};  // filed before this thread's first position
#pragma unroll
	for (int w = 0; w < 3; w++)
		if (w < wave) {
			mine.x += st.wave_total[w].x;
			mine.y += st.wave_total[w].y;
		}
	st.before[tid] = mine;
	__syncthreads();
	uint32_t carry[4];
#pragma unroll
	for (int s = 0; s < 4; s++)
		carry[s] = st.carry[0][s] + st.carry[1][s] + st.carry[2][s] + st.carry[3][s];

	uint32_t begin_of = 0xFFFFFFFFu;  // the tile start the last `from` was taken at
	uint2 from = {0u, 0u};
#pragma unroll
	for (int q = 0; q < 4; q++) {
		const uint32_t pos = pos0 + (uint32_t)q;
		if (pos < R) {
			const uint2 r = range[q];
			const bool continues = r.x < first;  // the tile began in an earlier workgroup
			const uint32_t begin = max(r.x, first) - first;
			if (begin != begin_of) {
				from = begin == 0u ? uint2{0u, 0u} : filed_before(st, begin);
				begin_of = begin;
			}
			const uint32_t n = r.y - r.x, e = pos - r.x, bits = key_strips(key[q]);
			uint32_t* lists = a.strip_lists + 4 * (size_t)r.x;
			const uint32_t at[4] = {mine.x & 0xFFFFu, mine.x >> 16, mine.y & 0xFFFFu, mine.y >> 16};
			const uint32_t base[4] = {from.x & 0xFFFFu, from.x >> 16, from.y & 0xFFFFu, from.y >> 16};
			uint32_t rank[4];
#pragma unroll
			for (int s = 0; s < 4; s++) {
				rank[s] = (continues ? carry[s] : 0u) + at[s] - base[s];
				if ((bits >> s) & 1u)
					lists[(size_t)s * n + rank[s]] = e | (((bits >> (4 + s)) & 1u) ? 0x80000000u : 0u);
			}
			if (pos + 1u == r.y) {  // the tile's last entry: its ranks plus itself are the strips' totals
				uint4 total = {rank[0] + (bits & 1u), rank[1] + ((bits >> 1) & 1u), rank[2] + ((bits >> 2) & 1u),
				               rank[3] + ((bits >> 3) & 1u)};
				reinterpret_cast<uint4*>(a.strip_total)[key_tile(key[q])] = total;
			}
		}
		const uint2 c = packed_strip_bits(filed[q]);
		mine.x += c.x;
		mine.y += c.y;
	}
}

// ---- forward (K/cuda_rasterizer_hgs/forward.cu:263-405) ---------------------------------------

struct ForwardPixel {
	// Transmittance in front of the next entry, at least 1e-4, of a pixel that takes further entries; that of a finished
	// pixel (the reference's done flag) with its sign turned, so that one register says both: a product with it stays
	// below the threshold and nothing blends any more.
	float T;
	float C0, C1, C2, weight, D;
	uint32_t last_filed;  // the last entry blended, counted in entries filed for the strip (1-based; 0: none)
	int last_slot;        // the same within the chunk being walked, as a packed slot of the pixel's half (-1: none)
};

// (In the order in which a walk reads them: 16 bytes, 8 or 16, 16 per entry.  With the record's own order, of which the walk skips two
// words, the compiler made four reads of the first eight, 20 per group of four entries instead of 10; with plain_entry: forward blend
// 270 -> 258 us at 1600x1036 and 5.6 M Gaussians, 1 609 -> 1 500 at 5185x3359, 44 -> 39 for 100 000 Gaussians at 512x512.)
struct ForwardSlot {
	float4 centre_conic;  // pixel x, pixel y, staged conic -xx / 2, -xy
	float4 rest;          // staged conic -yy / 2, opacity, clip w (NaN: strip inside the box), unused
	float4 cd;            // r, g, b, view depth: what only a blended sample uses
};

struct ForwardStage {  // one per workgroup (a single wavefront)
	// The chunk's entries once per 8-pixel-wide half of the strip they can reach, each half's packed to the front, so
	// that a step's reads are at addresses known when the step begins (and from one base):
	ForwardSlot slots[2 * kChunk + 1];  // of half h from h (kChunk + 1) on: one apart, or both halves' reads would meet in the same banks
	__device__ __forceinline__ ForwardSlot* slot(int half) { return slots + half * (kChunk + 1); }
	__device__ __forceinline__ const ForwardSlot* slot(int half) const { return slots + half * (kChunk + 1); }
	uint8_t entry[2][kChunk];     // which entry of the chunk a packed slot holds
	StripRays rays;
};

// Adds a sample to the pixels of `lanes`: one product alpha T (`weight`) and a fused multiply-add per channel instead
// of the reference's two products and an add each (forward.cu:378-385); the sums feed no decision, the images are compared
// by tolerance.  Under a lane mask, so that a colour that is not finite reaches the pixels that blend it and no others;
// written out because the compiler puts a branch around every masked region, and four taken branches per group of
// entries cost a wavefront that is alone on its SIMD more than the additions do.  (Lanes that are not active around it stay so.)
__device__ __forceinline__ void blend_sample(ForwardPixel& p, uint64_t lanes, float weight, const float4 cd, int slot)
{
	uint64_t active;
	asm("s_and_saveexec_b64 %[active], %[lanes]\n\t"
	    "v_fmac_f32 %[c0], %[r], %[w]\n\t"
	    "v_fmac_f32 %[c1], %[g], %[w]\n\t"
	    "v_fmac_f32 %[c2], %[b], %[w]\n\t"
	    "v_fmac_f32 %[d], %[z], %[w]\n\t"
	    "v_add_f32 %[sum], %[sum], %[w]\n\t"
	    "v_mov_b32 %[last], %[slot]\n\t"
	    "s_mov_b64 exec, %[active]"
	    : [c0] "+v"(p.C0), [c1] "+v"(p.C1), [c2] "+v"(p.C2), [d] "+v"(p.D), [sum] "+v"(p.weight), [last] "+v"(p.last_slot),
	      [active] "=&s"(active)
	    : [lanes] "s"(lanes), [w] "v"(weight), [r] "v"(cd.x), [g] "v"(cd.y), [b] "v"(cd.z), [z] "v"(cd.w), [slot] "s"(slot)
	    : "scc");
}

// Four neighbouring slots of the pixel's half.  Alpha of all four first, by every lane, with the decisions kept as lane
// masks in scalar registers; then the transmittances, one entry after the other, without a branch: an entry that a pixel
// does not take has alpha 0 there, and one that finishes it (T (1 - alpha) < 1e-4) is not blended and turns T's sign.
// Instructions that only some entries need are few (most visited entries blend somewhere), while a branch per entry
// had the wavefront wait for its scalar masks four times a group: a walk alone on its SIMD advanced at 280 cycles per
// entry, two and a half times what issuing its instructions takes.
struct FourEntries {
	float power[4], clip_w[4], opacity[4], alpha[4];
	uint64_t mask[4];
};

// What four slots hold, read ahead of its use: left to itself the compiler puts each read in front of the entry that
// needs it, and a wavefront that is alone on its SIMD then waits for LDS four times.
template <BoxTest kBox>
__device__ __forceinline__ void read_four(const ForwardSlot* slot, float4 (&centre_conic)[4], float4 (&rest)[4])
{
#pragma unroll
	for (int i = 0; i < 4; i++) {
		centre_conic[i] = slot[i].centre_conic;
		if (kBox == kBoxNone) {
			const float2 v = *reinterpret_cast<const float2*>(&slot[i].rest);
			rest[i] = float4{v.x, v.y, 0.f, 0.f};
		} else {
			rest[i] = slot[i].rest;
		}
	}
}

// Whether an entry's exponent is certainly not positive and its alpha below 0.99 in every pixel, so that a walk of such
// entries alone needs neither of the two comparisons.  Of the exponent's three terms (A + B) + C, A and B not positive, C is at most
// sqrt(1 - 1e-5) (|A| + |B|), which leaves 5e-6 (|A| + |B|); six roundings take 4e-7 of it.  False for a NaN.
__device__ __forceinline__ bool plain_entry(const LoadedRecord& r)
{
	const float ca = r.conic.x, cb = r.conic.y, cc = r.conic.z;
	return ca > 1e-20f && cc > 1e-20f && cb * cb <= 0.99999f * (ca * cc) && r.conic.w <= 0.989f && fabsf(r.geom.x) < 1e9f && fabsf(r.geom.y) < 1e9f;
}

// Alphas, zero where the pixel does not take the entry, and the masks of those that do (as far as exponent, alpha and box decide).
// (Each mask from single comparisons, with a negation so that a NaN is kept, as in the exact loop: a comparison's result is
// the mask; that of a combined flag is formed through a register.)
template <BoxTest kBox, bool kPlain>
__device__ __forceinline__ void forward_alphas(FourEntries& e, uint64_t live, const StripRays& rays, const BoxSpan& span, const BlendArgs& a)
{
#pragma unroll
	for (int i = 0; i < 4; i++) {
		const float alpha = e.opacity[i] * exp_of_exponent(e.power[i]);
		e.alpha[i] = kPlain ? alpha : fminf(0.99f, alpha);
		e.mask[i] = lanes_where(!(e.alpha[i] < 1.0f / 255.0f));
		if (!kPlain)
			e.mask[i] &= lanes_where(!(e.power[i] > 0.0f));
	}
	if (kBox == kBoxSpans) {
#pragma unroll
		for (int i = 0; i < 4; i++)
			e.mask[i] &= live;
		keep_lanes_inside_box(e.mask, e.clip_w, span, rays, a);
	}
	if (kBox == kBoxExact)
#pragma unroll
		for (int i = 0; i < 4; i++)
			e.mask[i] = lanes_inside_box(e.mask[i] & live, e.clip_w[i], rays, a);
#pragma unroll
	for (int i = 0; i < 4; i++)
		e.alpha[i] = __builtin_amdgcn_inverse_ballot_w64(e.mask[i]) ? e.alpha[i] : 0.f;
}

__device__ __forceinline__ void forward_blend(ForwardPixel& p, const float* alpha, uint64_t* mask, const float4* cd, int slot)
{
	float weight[4];
#pragma unroll
	for (int i = 0; i < 4; i++) {
		const float test_T = p.T * (1 - alpha[i]);
		const bool ok = !(test_T < 0.0001f);
		weight[i] = alpha[i] * p.T;
		p.T = ok ? test_T : -fabsf(p.T);
		mask[i] &= lanes_where(ok);
	}
#pragma unroll
	for (int i = 0; i < 4; i++)
		blend_sample(p, mask[i], weight[i], cd[i], slot + i);
}

template <BoxTest kBox, bool kPlain>
__device__ __forceinline__ void forward_group(ForwardPixel& p, uint64_t& live, const StripRays& rays, const ForwardSlot* slot, int k,
                                              const float2 pixf, const BoxSpan& span, const BlendArgs& a)
{
	FourEntries e;
	float4 centre_conic[4], rest[4];
	read_four<kBox>(slot, centre_conic, rest);
	__builtin_amdgcn_sched_barrier(0);
#pragma unroll
	for (int i = 0; i < 4; i++) {
		e.power[i] = exponent_of_staged(centre_conic[i], rest[i].x, pixf);
		e.opacity[i] = rest[i].y;
		e.clip_w[i] = rest[i].z;
	}
	// the entries' colours are asked for ahead of the exponentials and used behind the transmittances
	float4 cd[4];
#pragma unroll
	for (int i = 0; i < 4; i++)
		cd[i] = slot[i].cd;
	__builtin_amdgcn_sched_barrier(0);
	forward_alphas<kBox, kPlain>(e, live, rays, span, a);
	forward_blend(p, e.alpha, e.mask, cd, k);
	live = lanes_where(p.T > 0.f);
}

// The packed slots of a chunk, as many as the longer half has, or until no pixel takes any more.
template <BoxTest kBox, bool kPlain>
__device__ __forceinline__ void forward_chunk(ForwardPixel& p, uint64_t& live, const ForwardStage& st, int half, int steps,
                                              const float2 pixf, const BoxSpan& span, const BlendArgs& a)
{
	for (int k = 0; k < steps && live != 0ull; k += 4)
		forward_group<kBox, kPlain>(p, live, st.rays, st.slot(half) + k, k, pixf, span, a);
}

// Number of set bits of a ballot below the calling lane.
__device__ __forceinline__ uint32_t lanes_below(uint64_t ballot)
{
	return __builtin_amdgcn_mbcnt_hi((uint32_t)(ballot >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ballot, 0u));
}

// Bounding box (first and last column, first and last row, relative to the strip's first pixel) of the live pixels in
// the half of the strip that starts at column `column` (0 or 8); one that nothing reaches if there are none.
__device__ __forceinline__ float4 live_box(uint64_t live, int column)
{
	const uint64_t mine = (live >> column) & 0x00FF00FF00FF00FFull;
	if (mine == 0ull)
		return float4{INFINITY, -INFINITY, INFINITY, -INFINITY};
	uint32_t columns = (uint32_t)mine | (uint32_t)(mine >> 32);
	columns = (columns | (columns >> 16)) & 0xFFu;
	return float4{(float)(column + __builtin_ctz(columns)), (float)(column + 31 - __builtin_clz(columns)),
	              (float)(__builtin_ctzll(mine) >> 4), (float)((63 - __builtin_clzll(mine)) >> 4)};
}

// Per 8-pixel-wide half of the strip (columns: bit 3 of the lane), the largest of its lanes' values, which are not negative
// (non-negative floats compare like their bits).
__device__ __forceinline__ uint2 half_max_u32(uint32_t v)
{
	int x = (int)v;
	x = max(x, __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, true));   // quad_perm:[1,0,3,2]
	x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, true));   // quad_perm:[2,3,0,1]
	x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, true));  // row_half_mirror: the other quad of the eight
	int m[2];
#pragma unroll
	for (int h = 0; h < 2; h++)
		m[h] = max(max(__builtin_amdgcn_readlane(x, 8 * h), __builtin_amdgcn_readlane(x, 8 * h + 16)),
		           max(__builtin_amdgcn_readlane(x, 8 * h + 32), __builtin_amdgcn_readlane(x, 8 * h + 48)));
	return uint2{(uint32_t)m[0], (uint32_t)m[1]};
}

// Bounds on clip w between which, per half, some pixel that still takes entries can have its sample inside the box.
struct HalfSpan {
	float from[2], to[2];
};
__device__ __forceinline__ HalfSpan live_w_span(bool takes, const BoxSpan& span)
{
	takes = takes && !(span.from > span.to);
	// (the smallest entering w through its complement in the order of the bits)
	const uint2 to = half_max_u32(takes ? __float_as_uint(fmaxf(span.to, 0.f)) : 0u),
	            from_c = half_max_u32(takes ? 0x7F800000u - __float_as_uint(span.from) : 0u);
	return HalfSpan{{__uint_as_float(0x7F800000u - from_c.x), __uint_as_float(0x7F800000u - from_c.y)},
	                {__uint_as_float(to.x), __uint_as_float(to.y)}};
}

// Takes the entries that no live pixel can have inside the box out of a chunk whose entries straddle one of its faces in
// the strip, all of them at a positive clip w.
__device__ __forceinline__ void prune_by_box(bool straddles, bool takes, float w, const BoxSpan& span, bool& left, bool& right)
{
	const HalfSpan h = live_w_span(takes, span);
	if (straddles) {
		left = left && !(w > h.to[0]) && !(w < h.from[0]);
		right = right && !(w > h.to[1]) && !(w < h.from[1]);
	}
}

// In which 8-pixel-wide halves of the strip (first pixel x0, ya) an entry's ellipse power >= floor can reach a pixel that
// still takes entries, by the bounding boxes of the ellipse and of each half's live pixels.  The ellipse's half extents are
// sqrt(limit c / (a c - b^2)) in x and sqrt(limit a / (a c - b^2)) in y with limit = -2 floor, here with room for the
// rounding of the exponent the pixels evaluate (relative to its largest terms over the strip) and of the determinant.  An
// entry outside that box would pass the floor test in none of those pixels, so leaving it out of the half's walk changes no
// result.  (The rows matter as much as the columns: a ground plane at a grazing angle is made of flat ellipses, and a row
// of pixels just above the horizon, which nothing fills, kept its strip walking thousands of entries that only its finished
// rows could see.)
struct EllipseBox {
	float dx, dy, reach_x, reach_y;  // centre relative to the strip's first pixel, half extents
};
__device__ __forceinline__ EllipseBox ellipse_box(const LoadedRecord& r, float x0, float ya)
{
	const float ca = r.conic.x, cb = r.conic.y, cc = r.conic.z;
	const float dxa = r.geom.x - x0, dya = r.geom.y - ya;
	const float limit = -2.f * r.geom.z;
	const float far_x = fmaxf(fabsf(dxa), fabsf(dxa - 15.f)), far_y = fmaxf(fabsf(dya), fabsf(dya - 3.f));
	const float allowed = limit + (1e-3f + 1e-4f * limit + 1e-5f * (ca * far_x * far_x + cc * far_y * far_y));
	const float det = ca * cc - cb * cb - 1e-6f * ca * cc;
	EllipseBox b = {dxa, dya, INFINITY, INFINITY};
	if ((ca > 0.f) && (cc > 0.f) && (det > 0.f)) {
		const float scale = allowed * __builtin_amdgcn_rcpf(det);
		b.reach_x = __builtin_amdgcn_sqrtf(scale * cc) * 1.001f + 0.01f;
		b.reach_y = __builtin_amdgcn_sqrtf(scale * ca) * 1.001f + 0.01f;
	}
	return b;
}
// box: first and last column, first and last row, relative to the strip's first pixel.  (A NaN, as of a Gaussian whose floor is,
// excludes nothing.)
__device__ __forceinline__ bool reaches(const EllipseBox& e, const float4 box)
{
	return !(e.dx + e.reach_x < box.x) && !(e.dx - e.reach_x > box.y) && !(e.dy + e.reach_y < box.z) && !(e.dy - e.reach_y > box.w);
}

constexpr uint32_t kNone = 0xFFFFFFFFu, kPosition = 0x7FFFFFFFu;  // of a filed entry: none, and its list position

// Files an entry in slot `at` of a half.
__device__ __forceinline__ void stage_slot(ForwardStage& st, int half, uint32_t at, const LoadedRecord& r, uint32_t pos, int entry)
{
	float w = r.geom.w;
	int nan = 0x7FC00000;
	asm volatile("" : "+v"(nan));  // (made here each time rather than held through the walk)
	if (pos & 0x80000000u)
		w = __int_as_float(nan);  // the strip lies inside the box: no per-pixel test
	const float4 conic = staged_conic(r.conic);
	ForwardSlot& slot = st.slot(half)[at];
	slot.centre_conic = float4{r.geom.x, r.geom.y, conic.x, conic.y};
	slot.rest = float4{conic.z, conic.w, w, 0.f};
	slot.cd = r.cd;
	st.entry[half][at] = (uint8_t)entry;
}

// A slot that no pixel takes: opacity 0.
__device__ __forceinline__ void stage_nothing(ForwardStage& st, int half, uint32_t at)
{
	float zero = 0.f;
	asm volatile("" : "+v"(zero));  // (made here each time: four registers held through the walk otherwise)
	st.slot(half)[at].centre_conic = float4{zero, zero, zero, zero};
	st.slot(half)[at].rest = float4{zero, zero, zero, zero};
}

// What a strip's walk leaves: how many of the filed entries the backward has to walk (up to the last one some pixel
// blended), and the images.  px, py: the lane's pixel.
__device__ __forceinline__ void forward_finish(const BlendArgs& a, uint32_t strip_id, const ForwardPixel& p, uint32_t filed,
                                               const uint32_t* filed_list, uint32_t px, uint32_t py, int lane)
{
	const uint32_t upto = filed != 0u ? wave_max_u32(p.last_filed) : 0u;  // (zero for a pixel outside the image)
	if (lane == 0)
		a.strip_filed[strip_id] = upto;
	if (px < (uint32_t)a.W && py < (uint32_t)a.H) {
		const uint32_t pix_id = (uint32_t)a.W * py + px;
		const size_t plane = (size_t)a.H * a.W;
		// the reference's n_contrib: the 1-based position in the tile's list of the last entry the pixel blended
		a.n_contrib[pix_id] = p.last_filed != 0u ? (filed_list[p.last_filed - 1u] & kPosition) + 1u : 0u;
		a.out_color[pix_id] = p.C0 + fabsf(p.T) * a.bg[0];
		a.out_color[plane + pix_id] = p.C1 + fabsf(p.T) * a.bg[1];
		a.out_color[2 * plane + pix_id] = p.C2 + fabsf(p.T) * a.bg[2];
		a.out_alpha[pix_id] = p.weight;
		a.out_depth[pix_id] = p.D;
	}
}

// Word i of an array that is the same for every lane, by its distance in bytes (i below 2^30): an address of 64 bits takes two registers.
__device__ __forceinline__ uint32_t word_at(const uint32_t* words, uint32_t i)
{
	return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(words) + 4u * i);
}

// The first chunk from entry `at` on that holds an entry which some pixel that still takes entries may have inside the box, or one whose strip lies
// inside it or whose clip w is not positive; `filed` if there is none.  A pixel whose ray has left the box (or enters it behind everything) stays
// unfinished, and its strip walks on to the end of its list: of the 232 chunks of one such list of 62.9 M Gaussians 206 held nothing for any
// pixel, at 2.2 us each (records, ellipses and packing, beside five other wavefronts), and the launch waited for it.  Here eight chunks at a
// time are looked at for their clip w alone.  Forward blend, us: 62.9 M 713 -> 641, four submodels of 5.6 M with a call each 413 -> 374, a view
// of a city 137 -> 133 (four chunks at a time 638, 380, 133; sixteen 672, 387, 144).
constexpr int kScanned = 8;
__device__ __forceinline__ uint32_t next_within_spans(const BlendArgs& a, const uint32_t* list, const uint32_t* filed_list, uint32_t at, uint32_t filed,
                                                      const HalfSpan& h, int lane)
{
	for (; at < filed; at += 64u * kScanned) {
		uint32_t pos[kScanned], id[kScanned];
		float w[kScanned];
#pragma unroll
		for (int q = 0; q < kScanned; q++) {
			const uint32_t e = at + 64u * (uint32_t)q + (uint32_t)lane;
			pos[q] = e < filed ? word_at(filed_list, e) : kNone;
		}
#pragma unroll
		for (int q = 0; q < kScanned; q++)
			id[q] = pos[q] != kNone ? min(word_at(list, pos[q] & kPosition), a.gaussians - 1u) : 0u;
#pragma unroll
		for (int q = 0; q < kScanned; q++)
			w[q] = a.record[4 * (size_t)id[q]].w;
#pragma unroll
		for (int q = 0; q < kScanned; q++) {
			const bool within = (!(w[q] > h.to[0]) && !(w[q] < h.from[0])) || (!(w[q] > h.to[1]) && !(w[q] < h.from[1]));
			if (lanes_where(pos[q] != kNone && (within || (pos[q] & 0x80000000u) != 0u || !(w[q] > 0.f))) != 0ull)
				return at + 64u * (uint32_t)q;
		}
	}
	return filed;
}

// One strip by one wavefront.
__device__ __forceinline__ void forward_strip(const BlendArgs& a, uint32_t strip_id, ForwardStage& st, int lane)
{
	const int tile = (int)(strip_id >> 2), wave = (int)(strip_id & 3u);  // wave: which strip of the tile
	const uint2 range = a.ranges[tile];
	const uint32_t n = range.y - range.x;
	const int tx = tile % a.grid_x, ty = tile / a.grid_x;
	const uint32_t px = tx * kTile + (lane & 15), py = ty * kTile + wave * 4 + (lane >> 4);
	const bool inside = px < (uint32_t)a.W && py < (uint32_t)a.H;
	const float2 pixf = {(float)px, (float)py};

	ForwardPixel p = {inside ? 1.0f : -1.0f, 0.f, 0.f, 0.f, 0.f, 0.f, 0u, -1};
	uint64_t live = lanes_where(inside);
	// the entries filed for this strip, in list order: list position, bit 31 = strip inside the box
	const uint32_t filed = a.strip_total[strip_id];
	if (filed != 0u && live != 0ull) {
		stage_rays(st.rays, pixf, a, lane);
		const uint32_t* list = a.point_list + range.x;
		const uint32_t* filed_list = a.strip_lists + 4 * (size_t)range.x + (size_t)wave * n;
		// Lane l of the chunk that starts at filed entry `first` takes entry first + l: its list
		// position (and box flag), through that the Gaussian's index, through that its record.
		// Three chunks are in flight: the records of the next one, the indices of the one after,
		// the positions of the one after that.
		uint32_t lane_here = (uint32_t)lane;
		asm volatile("" : "+v"(lane_here));  // (what follows from it is not held from strip to strip)
		uint32_t pos_cur = lane_here < filed ? word_at(filed_list, lane_here) : kNone;
		uint32_t pos_next = 64u + lane_here < filed ? word_at(filed_list, 64u + lane_here) : kNone;
		uint32_t pos_after = 128u + lane_here < filed ? word_at(filed_list, 128u + lane_here) : kNone;
		LoadedRecord cur = load_record(a, pos_cur != kNone ? word_at(list, pos_cur & kPosition) : 0u, pos_cur != kNone);
		uint32_t id_next = pos_next != kNone ? word_at(list, pos_next & kPosition) : 0u;

		const float x0 = wave_uniform((float)(tx * kTile)), ya = wave_uniform((float)(ty * kTile + wave * 4));
		// Where an entry straddles a face of the box, the pixel's span is worked out once, at the first such chunk: a strip
		// with a pixel that stays unfinished walks hundreds of chunks that hold nothing for it, and with the span (150 instructions
		// and the box from memory) formed twice in each, as once, such a walk took 3.9 us a chunk (62.9 M Gaussians: 232 chunks).
		BoxSpan span = {0.f, 0.f, 0.f, 0.f};
		bool have_span = false;
		for (uint32_t first = 0; first < filed && live != 0ull; first += 64) {
			const int count = (int)min(filed - first, 64u);
			// what follows from the lane's number is worked out per chunk: held through the walk it costs half a dozen registers
			int l = lane;
			asm volatile("" : "+v"(l));
			const int half = (l >> 3) & 1;
			const float4 box_l = live_box(live, 0), box_r = live_box(live, 8);
			bool left = false, right = false;
			if (l < count) {
				const EllipseBox e = ellipse_box(cur, x0, ya);
				left = reaches(e, box_l);
				right = reaches(e, box_r);
			}
			// Entries whose sample the box clips in every pixel of a half that still takes entries are left out too: a
			// pixel whose ray has left the box, or enters it behind everything, stays unfinished for good, and a strip with
			// one such pixel walked its list to the end (at 1600x1036 and 5.6 M Gaussians, a camera that looks along a
			// plane between submodels: one that blends none of its last 2 800 entries walked 3 387; 0.54 ms of launch).
			const bool straddles = l < count && (pos_cur & 0x80000000u) == 0u;
			const BoxTest box = lanes_where(straddles) == 0ull ? kBoxNone : lanes_where(straddles && !(cur.geom.w > 0.f)) == 0ull ? kBoxSpans : kBoxExact;
			if (box == kBoxSpans) {
				if (!have_span) {
					span = w_inside_box(ray_of(st.rays), load_box_frame(a));
					have_span = true;
				}
				prune_by_box(straddles, p.T > 0.f, cur.geom.w, span, left, right);
			}
			const uint64_t in_left = lanes_where(left), in_right = lanes_where(right);
			const bool plain = box == kBoxNone && lanes_where((left || right) && !plain_entry(cur)) == 0ull;
			const int n_left = __popcll(in_left), n_right = __popcll(in_right);
			const int steps = max(n_left, n_right), padded = (steps + 3) & ~3;
			if (left)
				stage_slot(st, 0, lanes_below(in_left), cur, pos_cur, l);
			if (right)
				stage_slot(st, 1, lanes_below(in_right), cur, pos_cur, l);
			// both halves are walked for `padded` slots: the rest get entries that nothing takes
			if (l >= n_left && l < padded)
				stage_nothing(st, 0, (uint32_t)l);
			if (l >= n_right && l < padded)
				stage_nothing(st, 1, (uint32_t)l);
			__builtin_amdgcn_wave_barrier();
			// the chunk is in LDS now: its registers take the next chunk's records, loaded during the walk
			cur = load_record(a, id_next, pos_next != kNone);
			pos_cur = pos_next;
			pos_next = pos_after;
			id_next = pos_next != kNone ? word_at(list, pos_next & kPosition) : 0u;
			const uint32_t e3 = first + 192 + (uint32_t)l;
			pos_after = e3 < filed ? word_at(filed_list, e3) : kNone;

			if (plain)
				forward_chunk<kBoxNone, true>(p, live, st, half, steps, pixf, span, a);
			else if (box == kBoxNone)
				forward_chunk<kBoxNone, false>(p, live, st, half, steps, pixf, span, a);
			else if (box == kBoxSpans)
				forward_chunk<kBoxSpans, false>(p, live, st, half, steps, pixf, span, a);
			else
				forward_chunk<kBoxExact, false>(p, live, st, half, steps, pixf, span, a);
			if (p.last_slot >= 0)
				p.last_filed = first + st.entry[half][p.last_slot] + 1u;
			p.last_slot = -1;
			__builtin_amdgcn_wave_barrier();
			if (steps == 0 && box == kBoxSpans) {
				// the chunk held nothing for any pixel: on to the next one that may
				int m = lane;
				asm volatile("" : "+v"(m));
				const uint32_t at = next_within_spans(a, list, filed_list, first + 64u, filed, live_w_span(p.T > 0.f, span), m);
				first = at - 64u;
				pos_cur = at + (uint32_t)m < filed ? word_at(filed_list, at + (uint32_t)m) : kNone;
				pos_next = at + 64u + (uint32_t)m < filed ? word_at(filed_list, at + 64u + (uint32_t)m) : kNone;
				pos_after = at + 128u + (uint32_t)m < filed ? word_at(filed_list, at + 128u + (uint32_t)m) : kNone;
				cur = load_record(a, pos_cur != kNone ? word_at(list, pos_cur & kPosition) : 0u, pos_cur != kNone);
				id_next = pos_next != kNone ? word_at(list, pos_next & kPosition) : 0u;
			}
		}
	}
	// (the pixel's place is worked out again, from the lane's number as the hardware counts it: kept from the start it would
	// hold a register through the whole walk, one more than the kernel's wavefronts per SIMD leave it)
	const int lane_again = (int)lanes_below(~0ull);
	forward_finish(a, strip_id, p, filed, a.strip_lists + 4 * (size_t)range.x + (size_t)wave * n, tx * kTile + (lane_again & 15),
	               ty * kTile + wave * 4 + (lane_again >> 4), lane_again);
}

// ---- a walk shared by four wavefronts ------------------------------------------------------------
// A wavefront alone on its SIMD advances four entries in 1 200 cycles, of which it issues in 430: the rest is the latency of
// one chain of LDS reads, dependent instructions and masks.  A launch with fewer strips than fill that time lasts as long as
// its longest walk.  There (see blend_shared) a strip is walked by four wavefronts, one per quarter of 8x2 pixels, and each takes
// four entries at a time: lane 4 p + e is pixel p's view of entry e, so that one exponential, one comparison serves
// four entries.  What depends on order is kept bit for bit: the transmittances in front of the four entries are the same products
// in the same order, taken by three multiplications inside each quad of lanes, and lane c of a quad adds channel c of
// the four samples one after the other.  In all it is twice the work.  (The backward shared in the same way adds to each Gaussian's row
// four times as often, and additions to one address take 12 ns each: 5 000 Gaussians at 512x512 took 303 us a pass for 200.)
constexpr uint32_t kSharedList = 64;  // entries from which a strip is worth four wavefronts (24 to 128 measure the same, 192 up to 3 us more)

template <int Ctrl>
__device__ __forceinline__ float quad_move(float v)
{
	return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), Ctrl, 0xF, 0xF, true));
}
// Lane e of a quad: start times (plus) the f of lanes 0 to e - 1, in that order.
__device__ __forceinline__ float product_in_front(float start, float f, int e)
{
	const float shifted = quad_move<0x90>(f);                      // quad_perm:[0,0,1,2]
	const float in_front = e == 0 ? 1.f : shifted;
	return start * quad_move<0x54>(in_front) * quad_move<0xA0>(in_front) * quad_move<0xC0>(in_front);  // [0,1,1,1], [0,0,2,2], [0,0,0,3]
}

struct QuarterPlace {
	int tile, strip, column, row;  // the quarter's first pixel relative to the strip's
	uint32_t px, py;               // the lane's pixel
	bool inside;
};
__device__ __forceinline__ QuarterPlace quarter_place(const BlendArgs& a, uint32_t strip_id, int quarter, int lane)
{
	QuarterPlace q;
	q.tile = (int)(strip_id >> 2);
	q.strip = (int)(strip_id & 3u);
	q.column = 8 * (quarter & 1);
	q.row = 2 * (quarter >> 1);
	q.px = (uint32_t)(q.tile % a.grid_x * kTile + q.column + ((lane >> 2) & 7));
	q.py = (uint32_t)(q.tile / a.grid_x * kTile + 4 * q.strip + q.row + (lane >> 5));
	q.inside = q.px < (uint32_t)a.W && q.py < (uint32_t)a.H;
	return q;
}

struct QuarterPixel {
	float T;        // transmittance in front of the next entry (of a finished pixel: in front of the entry that finished it)
	float C;        // lane c: channel c (r, g, b, depth)
	float weight;
	int last_slot;  // the last of the lane's entries that the pixel blended, as a packed slot of the chunk (-1: none)
};

// The four entries of slots k to k + 3.  odd_colours: some colour of the chunk is not finite, so that one which is not blended
// must not be multiplied by its weight, zero.
__device__ __forceinline__ void quarter_group(QuarterPixel& p, uint64_t& live, const ForwardSlot* slots, int k, int lane,
                                              const float2 pixf, BoxTest box, const BoxSpan& span, const PixelRay& ray, bool odd_colours,
                                              const BlendArgs& a)
{
	const int e = lane & 3;
	const float4 centre_conic = slots[k + e].centre_conic, rest = slots[k + e].rest;
	float colour[4];
#pragma unroll
	for (int i = 0; i < 4; i++)
		colour[i] = reinterpret_cast<const float*>(&slots[k + i].cd)[e];
	__builtin_amdgcn_sched_barrier(0);
	const float power = exponent_of_staged(centre_conic, rest.x, pixf);
	float alpha = fminf(0.99f, rest.y * exp_of_exponent(power));
	uint64_t mask = live & lanes_where(!(power > 0.0f)) & lanes_where(!(alpha < 1.0f / 255.0f));
	if (box == kBoxSpans)
		mask = lanes_inside_box(mask, rest.z, span, ray, a);
	else if (box == kBoxExact)
		mask = lanes_inside_box(mask, rest.z, ray, a);
	alpha = __builtin_amdgcn_inverse_ballot_w64(mask) ? alpha : 0.f;
	const float beyond = 1 - alpha;
	const float T = product_in_front(p.T, beyond, e), test_T = T * beyond;
	const bool ok = !(test_T < 0.0001f);            // (false for every entry behind one for which it is)
	const uint64_t passed = lanes_where(ok);
	const float weight = ok ? alpha * T : 0.f;
	p.last_slot = __builtin_amdgcn_inverse_ballot_w64(mask & passed) ? k + e : p.last_slot;
	// in front of the next group: behind the last entry that passed
	float t = ok ? test_T : p.T;
	t = fminf(t, quad_move<0xB1>(t));     // quad_perm:[1,0,3,2]
	p.T = fminf(t, quad_move<0x4E>(t));   // quad_perm:[2,3,0,1]
	const uint64_t through = (passed >> 3) & 0x1111111111111111ull;  // pixels that entry 3 has passed
	live &= (through << 4) - through;
	const float w[4] = {quad_move<0x00>(weight), quad_move<0x55>(weight), quad_move<0xAA>(weight), quad_move<0xFF>(weight)};
#pragma unroll
	for (int i = 0; i < 4; i++)
		p.weight += w[i];
	if (!odd_colours) {
#pragma unroll
		for (int i = 0; i < 4; i++)
			p.C = __builtin_fmaf(w[i], colour[i], p.C);
	} else {
#pragma unroll
		for (int i = 0; i < 4; i++)
			p.C = w[i] != 0.f ? __builtin_fmaf(w[i], colour[i], p.C) : p.C;  // (the weight of a blended sample is not zero)
	}
}

// Bounding box of a quarter's live pixels, relative to the strip's first pixel.
__device__ __forceinline__ float4 quarter_box(uint64_t live, const QuarterPlace& q)
{
	const uint32_t upper = (uint32_t)live & 0x11111111u, lower = (uint32_t)(live >> 32) & 0x11111111u, columns = upper | lower;
	return float4{(float)(q.column + (__builtin_ctz(columns) >> 2)), (float)(q.column + ((31 - __builtin_clz(columns)) >> 2)),
	              (float)(q.row + (upper == 0u ? 1 : 0)), (float)(q.row + (lower == 0u ? 0 : 1))};
}

__device__ __forceinline__ void forward_quarter(const BlendArgs& a, uint32_t strip_id, uint32_t filed, int quarter, ForwardStage& st, int lane)
{
	const QuarterPlace q = quarter_place(a, strip_id, quarter, lane);
	const uint2 range = a.ranges[q.tile];
	const uint32_t n = range.y - range.x;
	const int e = lane & 3;
	const float2 pixf = {(float)q.px, (float)q.py};
	uint64_t live = lanes_where(q.inside);
	if (live == 0ull)
		return;
	const PixelRay ray = {pix_to_ndc(pixf.x, a.W), pix_to_ndc(pixf.y, a.H)};
	const float x0 = wave_uniform((float)(q.tile % a.grid_x * kTile)), ya = wave_uniform((float)(q.tile / a.grid_x * kTile + 4 * q.strip));
	const uint32_t* list = a.point_list + range.x;
	const uint32_t* filed_list = a.strip_lists + 4 * (size_t)range.x + (size_t)q.strip * n;
	QuarterPixel p = {1.f, 0.f, 0.f, -1};
	uint32_t last_filed = 0u;
	BoxSpan span = {0.f, 0.f, 0.f, 0.f};
	bool have_span = false;
	// (chunks as in forward_strip)
	uint32_t pos_cur = (uint32_t)lane < filed ? filed_list[lane] : kNone;
	uint32_t pos_next = (uint32_t)(64 + lane) < filed ? filed_list[64 + lane] : kNone;
	uint32_t pos_after = (uint32_t)(128 + lane) < filed ? filed_list[128 + lane] : kNone;
	LoadedRecord cur = load_record(a, pos_cur != kNone ? list[pos_cur & kPosition] : 0u, pos_cur != kNone);
	uint32_t id_next = pos_next != kNone ? list[pos_next & kPosition] : 0u;
	for (uint32_t first = 0; first < filed && live != 0ull; first += 64) {
		const int count = (int)min(filed - first, 64u);
		bool reached = lane < count && reaches(ellipse_box(cur, x0, ya), quarter_box(live, q));
		const bool straddles = lane < count && (pos_cur & 0x80000000u) == 0u;
		const BoxTest box = lanes_where(straddles) == 0ull ? kBoxNone : lanes_where(straddles && !(cur.geom.w > 0.f)) == 0ull ? kBoxSpans : kBoxExact;
		if (box == kBoxSpans) {
			if (!have_span) {
				span = w_inside_box(ray, load_box_frame(a));
				have_span = true;
			}
			// entries that the box clips in every live pixel (as prune_by_box, over the quarter)
			const bool takes = __builtin_amdgcn_inverse_ballot_w64(live) && !(span.from > span.to);
			const float to = __uint_as_float(wave_max_u32(takes ? __float_as_uint(fmaxf(span.to, 0.f)) : 0u));
			const float from = __uint_as_float(0x7F800000u - wave_max_u32(takes ? 0x7F800000u - __float_as_uint(span.from) : 0u));
			if (straddles)
				reached = reached && !(cur.geom.w > to) && !(cur.geom.w < from);
		}
		const uint64_t in = lanes_where(reached);
		const int steps = __popcll(in);
		// (a sum that is not finite names a colour that is not; one of finite colours may overflow, which only costs time)
		const bool odd_colours = lanes_where(reached && !(fabsf(cur.cd.x + cur.cd.y + cur.cd.z + cur.cd.w) < INFINITY)) != 0ull;
		if (reached)
			stage_slot(st, 0, lanes_below(in), cur, pos_cur, lane);
		if (lane < 3) {  // up to a multiple of four
			stage_nothing(st, 0, (uint32_t)(steps + lane));
			st.slots[steps + lane].cd = float4{0.f, 0.f, 0.f, 0.f};
		}
		__builtin_amdgcn_wave_barrier();
		cur = load_record(a, id_next, pos_next != kNone);
		pos_cur = pos_next;
		pos_next = pos_after;
		id_next = pos_next != kNone ? list[pos_next & kPosition] : 0u;
		const uint32_t e3 = first + 192 + (uint32_t)lane;
		pos_after = e3 < filed ? filed_list[e3] : kNone;
		for (int k = 0; k < steps && live != 0ull; k += 4)
			quarter_group(p, live, st.slots, k, lane, pixf, box, span, ray, odd_colours, a);
		if (p.last_slot >= 0)
			last_filed = first + st.entry[0][p.last_slot] + 1u;
		p.last_slot = -1;
		__builtin_amdgcn_wave_barrier();
	}
	const uint32_t upto = wave_max_u32(last_filed);
	if (lane == 0 && upto != 0u)
		atomicMax(&a.strip_filed[strip_id], upto);  // (zero before the launch)
	last_filed = max(last_filed, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)last_filed, 0xB1, 0xF, 0xF, true));
	last_filed = max(last_filed, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)last_filed, 0x4E, 0xF, 0xF, true));
	if (q.inside) {
		const uint32_t pix_id = (uint32_t)a.W * q.py + q.px;
		const size_t plane = (size_t)a.H * a.W;
		if (e < 3)
			a.out_color[e * plane + pix_id] = p.C + p.T * a.bg[e];
		else
			a.out_depth[pix_id] = p.C;
		if (e == 0)
			a.out_alpha[pix_id] = p.weight;
		if (e == 1)
			a.n_contrib[pix_id] = last_filed != 0u ? (filed_list[last_filed - 1u] & kPosition) + 1u : 0u;
	}
}

// The place in the order of a workgroup's first, second ... strip.
__device__ __forceinline__ uint32_t turn_of_workgroup(uint32_t number, uint32_t turn, uint32_t workgroups)
{
	return turn * workgroups + ((turn & 1u) != 0u ? workgroups - 1u - number : number);
}

// Strips without entries, at most 64 of them: background, and nothing for the backward to walk.
__device__ __forceinline__ void forward_empty(const BlendArgs& a, const uint32_t* order, uint32_t count, int lane)
{
	const uint32_t mine = (uint32_t)lane < count ? order[lane] : 0u;
	const size_t plane = (size_t)a.H * a.W;
	const float r = a.bg[0], g = a.bg[1], b = a.bg[2];
	for (uint32_t k = 0; k < count; k++) {
		const uint32_t strip_id = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)k), tile = strip_id >> 2;
		const uint32_t px = (tile % (uint32_t)a.grid_x) * kTile + (lane & 15), py = (tile / (uint32_t)a.grid_x) * kTile + 4u * (strip_id & 3u) + (lane >> 4);
		if (lane == 0)
			a.strip_filed[strip_id] = 0u;
		if (px < (uint32_t)a.W && py < (uint32_t)a.H) {
			const uint32_t pix_id = (uint32_t)a.W * py + px;
			a.n_contrib[pix_id] = 0u;
			a.out_color[pix_id] = r;
			a.out_color[plane + pix_id] = g;
			a.out_color[2 * plane + pix_id] = b;
			a.out_alpha[pix_id] = 0.f;
			a.out_depth[pix_id] = 0.f;
		}
	}
}

template <bool kShared>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6, 6))) void blend_forward_kernel(BlendBatch batch)
{
	__shared__ ForwardStage st;
	// The jobs of a batch (the submodels of a frame) take turns, each handing out its strips longest
	// list first: a long strip that starts late is what a launch waits for, and with several jobs in one
	// launch there is other work to run beside the longest strips of each.  Most strips of a large image are empty
	// in most jobs, and workgroups are launched at about one per nanosecond, so a job has batch.workgroups of them, a
	// share of its strips: strips with entries beyond that number are second turns, the last of them that of the workgroup
	// with the longest first one.  The empty ones are dealt out evenly and come first: their stores leave while the walk goes on.
	const BlendArgs& a = batch.job[blockIdx.x % (uint32_t)batch.count];
	const int lane = threadIdx.x;
	const uint32_t number = blockIdx.x / (uint32_t)batch.count, workgroups = batch.workgroups;
	uint32_t strip_id = a.strip_order_forward[min(number, batch.strips - 1u)];  // (asked for beside the number of empty ones)
	const uint32_t none = min(a.strip_classes[strip_empty_word(1)], batch.strips), filled = batch.strips - none;
	const uint32_t share = (none + workgroups - 1u) / workgroups;
	for (uint32_t first = number * share, end = min(first + share, none); first < end; first += 64u)
		forward_empty(a, a.strip_order_forward + filled + first, min(64u, end - first), lane);
	if (kShared) {
		// four neighbouring workgroups per strip
		if (number / 4u >= filled)
			return;
		strip_id = a.strip_order_forward[number / 4u];
		const uint32_t entries = a.strip_total[strip_id];
		if (entries >= kSharedList)
			forward_quarter(a, strip_id, entries, (int)(number & 3u), st, lane);
		else if ((number & 3u) == ((number >> 3) & 3u))  // (not always the same of the four: they lie on different XCDs)
			forward_strip(a, strip_id, st, lane);
		return;
	}
	for (uint32_t at = number, turn = 0; at < filled;) {
		forward_strip(a, strip_id, st, lane);
		at = turn_of_workgroup(number, ++turn, workgroups);
		if (at < filled)
			strip_id = a.strip_order_forward[at];
	}
}

// Work accounting: the reference loop taken literally, one list entry at a time with no
// filter, counting over all pixels the entries visited by a live pixel (A), those with
// power <= 0 (B), with alpha >= 1/255 (C), inside the box (D), blended (E), and B, C and A
// restricted to entries up to each pixel's last blended one (the backward's share).
__global__ __launch_bounds__(256) void blend_count_kernel(BlendArgs a)
{
	__shared__ float4 s_geom[256];
	__shared__ float4 s_conic[256];

	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int tile = tile_of_block((int)blockIdx.x, a.grid_x, a.grid_y);
	if (tile < 0)
		return;
	const int tx = tile % a.grid_x, ty = tile / a.grid_x;
	const uint32_t px = tx * kTile + (lane & 15), py = ty * kTile + wave * 4 + (lane >> 4);
	const bool inside = px < (uint32_t)a.W && py < (uint32_t)a.H;
	const float2 pixf = {(float)px, (float)py};
	const PixelRay ray = {pix_to_ndc(pixf.x, a.W), pix_to_ndc(pixf.y, a.H)};
	const BoxFrame box = load_box_frame(a);
	const uint2 range = a.ranges[tile];
	const int rounds = (int)((range.y - range.x + 255) / 256);
	int todo = (int)(range.y - range.x);

	bool done = !inside;
	float T = 1.0f;
	uint32_t nA = 0, nB = 0, nC = 0, nD = 0, nE = 0, nA_last = 0, nB_last = 0, nC_last = 0;
	for (int i = 0; i < rounds; i++, todo -= 256) {
		__syncthreads();
		const uint32_t src = range.x + (uint32_t)i * 256 + tid;
		if (src < range.y) {
			const uint32_t id = a.point_list[src];
			const float4 r0 = a.record[4 * (size_t)id];
			s_geom[tid] = float4{r0.x, r0.y, 0.f, r0.w};
			s_conic[tid] = a.record[4 * (size_t)id + 1];
		}
		__syncthreads();
		const int count = todo < 256 ? todo : 256;
		for (int j = 0; !done && j < count; j++) {
			const float4 g = s_geom[j];
			const float4 co = s_conic[j];
			float2 d;
			const float power = exponent_of(g, co, pixf, d);
			nA++;
			if (power > 0.0f)
				continue;
			nB++;
			const float alpha = fminf(0.99f, co.w * expf(power));
			if (alpha < 1.0f / 255.0f)
				continue;
			nC++;
			if (clipped_by_box(ray, g.w, box))
				continue;
			nD++;
			const float test_T = T * (1 - alpha);
			if (test_T < 0.0001f) {
				done = true;
				continue;
			}
			nE++;
			nA_last = nA;
			nB_last = nB;
			nC_last = nC;
			T = test_T;
		}
	}
	const uint32_t c[8] = {nA, nB, nC, nD, nE, nB_last, nC_last, nA_last};
#pragma unroll
	for (int q = 0; q < 8; q++) {
		const uint32_t tot = wave_inclusive_scan_u32(c[q]);
		if (lane == 63)
			atomicAdd(reinterpret_cast<unsigned long long*>(a.counters) + q, (unsigned long long)tot);
	}
}

// ---- backward (K/cuda_rasterizer_hgs/backward.cu:415-622) ---------------------------------------
// Each wavefront walks, back to front, the entries the forward filed for its strip, starting at
// the last one that any of its 64 pixels blended, eight entries at a time.  The pass is split in two so
// that no cross-lane reduction is needed per entry:
//  * pixel-parallel part (lane = pixel, as in the forward): the per-pixel recurrences of the
//    reference loop give, for an entry, two numbers per pixel: u = G dL/dalpha-term and
//    aT = alpha T.  They are parked in one LDS row per entry.
//  * entry-parallel part (lane = (entry, strip row, half of the row)):
//    each lane sweeps 8 pixels and accumulates sum u, sum u dx, sum u dx^2 and
//    sum aT g_{r,g,b,depth}; dy is constant along a strip row, so the y moments follow from
//    those; three exchanges inside each group of eight lanes finish the sums, and the group adds its
//    entry's ten sums into the Gaussian's row of `sums`, eight neighbouring columns in one atomic
//    instruction and the last two in another.
// All ten sums of the reference (mean2D x/y, conic xx/xy/yy, opacity, colour r/g/b, depth)
// are linear in u and aT, which is what makes the split possible.
// (The sums as one product of the eight entries' sixteen rows with a 64 x 10 matrix of pixel moments and upstream
// gradients, sixteen 16x16x4 matrix instructions in fp32, were built and measured: 0.60 -> 0.66 ms at 1600x1036 with
// 5.6 M Gaussians.  The fp32 matrix instructions take their time from the vector instructions of the SIMD's other
// wavefronts, and 512 cycles per eight entries is more than the sweep needs; bf16 ones, which would not, need three
// terms per factor for the same precision, and splitting them costs what the sweep does.)

constexpr int kRows = 8;      // entries per entry-parallel part
// Pixel p of the strip sits in column p + (p >> 4) of a row of kRowStride (u, alpha T) pairs: the LDS has 32 banks of 4
// bytes, an 8-byte access is served 16 lanes at a time, and with these numbers neither the per-pixel writes nor
// the per-(entry, strip row, half row) reads below hit a bank twice within such a group.
constexpr int kRowStride = 68;
__device__ __forceinline__ int row_column(int pixel) { return pixel + (pixel >> 4); }

struct BackwardPixel {
	float T;
	float behind;  // what lies behind the entry being visited, weighted with the upstream gradient: see backward_rows
	float g_r, g_g, g_b, g_depth, g_alpha;
};

// An LDS address in a register of its own: left to itself the compiler folds a member's place in the stage into every
// access, where it exceeds what two-address accesses can encode, and adds it anew for each of them.
typedef float Pair __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) Pair LdsPair;
__device__ __forceinline__ LdsPair* lds_base(float2* p)
{
	LdsPair* at = (LdsPair*)p;
	asm volatile("" : "+v"(at));
	return at;
}

// Zeros in two neighbouring registers by one instruction (volatile: copies of a shared pair would take two).
__device__ __forceinline__ Pair zero_pair()
{
	Pair z;
	asm volatile("v_mov_b64 %0, 0" : "=v"(z));
	return z;
}

struct BackwardChunk {  // each what one read of the walk takes; + padding up to a multiple of eight entries
	float4 centre_conic[kChunk + kRows - 1];  // pixel x, pixel y, staged conic -xx / 2, -xy
	float4 rest[kChunk + kRows - 1];          // staged conic -yy / 2, opacity, clip w, 0-based position in the tile list (as bits)
	float4 cd[kChunk + kRows - 1];
	uint32_t sum_row[kChunk + kRows - 1];  // where the Gaussian's row of `sums` begins, in 16 bytes
};

struct BackwardStage {  // wave-private
	BackwardChunk chunk;
	float2 u_at[kRows * kRowStride];  // [row][row_column(pixel)]: (u, alpha T)
	float g_depth[72];                // upstream gradient of the depth image by pixel, eight of nine words
	StripRays rays;
};

struct StripFrame {
	float x0, y0;            // first pixel of the strip
	float ddelx_dx, ddely_dy;
};

template <int DppCtrl>
__device__ __forceinline__ float dpp_exchange_add(float v)
{
	const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), DppCtrl, 0xF, 0xF, true);
	return v + __builtin_bit_cast(float, moved);
}

// What a lane needs in the entry-parallel part whatever the entries, held for the whole walk: the upstream colour gradients of
// the eight pixels that it sweeps, their place in its entry's row, and the columns of `sums` that it adds to (of row 0).
struct Sweep {
	float r[8], g[8], b[8];   // (those of the depth image, where there are any, stay in LDS: BackwardStage::g_depth)
	LdsPair* row;
	float *column_low, *column_high;  // for entries 0-3 and for entries 4-7 of a pass
};

// Which entries of a pass some pixel blended: entries 0-3 and entries 4-7, 16 lanes each, a row of the wavefront per entry.
struct Blended {
	uint64_t low, high;
};

// Entry-parallel part for the eight entries staged from slot0 on.  A 16-lane row of the wavefront serves two entries, e in
// its low eight lanes and e + 4 in its high eight; lane (h = (lane >> 1) & 3, half = lane & 1) of the eight
// sums the entry's row over the 8 pixels of one half of strip row h; the eight lanes of an entry then add up what
// they hold (three exchanges inside their group of eight) and the entry's ten sums go into the Gaussian's
// row of `sums` with one atomic instruction: the entry's own lanes add columns 0-7, two lanes of the other eight of
// the 16-lane row add columns 8 and 9, so a first instruction serves entries 0-3 and a second one entries 4-7.
// (Adding columns 0-7 of all eight entries first and columns 8-9 after them, which needs no exchange between the
// groups, had every request of the second instruction hit a cache line that one of the first was still at work on:
// measured, that second instruction cost eight times what the first did, a fifth of the kernel's time.)
// The x moments are summed pixel by pixel about the entry's centre.  About the lane's first pixel, with constants for factors and
// moved to the centre once, they take 15 vector instructions fewer per pass, and the kernel 4 us less at 1600x1036 with
// 5.6 M Gaussians (532 for 536) and 39 at 5185x3359 (2855 for 2894), but terms of up to 49 u cancel to one of the Gaussian's
// own extent squared: for a Gaussian of half a pixel, the usual one of a dense scene, the sum for the conic's xx is then 7.7e-6
// off (relative L2 against 64 bits) and that for the mean's x 4.9e-7; this way both are 1.3e-7, as the sums in y.
// No instruction here only moves or repeats: one base address per LDS region, sums that start from the first pixel's terms, exchanges
// folded into their additions, rows of `sums` addressed by one shifted addition (50 vector instructions fewer per pass of eight
// entries; the kernel 555 -> 520 us at 1600x1036, 2935 -> 2885 at 5185x3359 when that was done, with the moments about the
// first pixel).
// kDepth: a gradient arrived for the depth image (without one, the usual case of a loss on the colour image alone, the
// terms it multiplies are left out: the depth column of `sums` stays zero).
template <bool kDepth>
__device__ __forceinline__ void sum_rows(const BackwardChunk& st, const float* g_depth, int slot0, const Blended& blended, const Sweep& sweep,
                                         const StripFrame& f, int lane)
{
#pragma clang fp contract(fast)
	__builtin_amdgcn_wave_barrier();
	const int upper = (lane >> 3) & 1;  // which eight of the 16-lane row
	const int e = (lane >> 4) + 4 * upper, h = (lane >> 1) & 3, half = lane & 1, j = lane & 7;
	const int slot = slot0 + e;
	const float4 centre = st.centre_conic[slot];
	const float dx_first = centre.x - (f.x0 + (float)(8 * half)), dy = centre.y - (f.y0 + (float)h);
	// (the first pixel's terms start the sums: added to zeros they would take six instructions)
	Pair ua = sweep.row[0];
	float s0 = ua.x, sx = ua.x * dx_first, sxx = sx * dx_first;
	float cr = ua.y * sweep.r[0], cg = ua.y * sweep.g[0], cb = ua.y * sweep.b[0];
	float cdp = kDepth ? ua.y * g_depth[9 * (lane & 7)] : 0.f;
#pragma unroll
	for (int step = 1; step < 8; step++) {
		ua = sweep.row[step];
		const float dx = dx_first - (float)step, t = ua.x * dx;
		s0 += ua.x;
		sx += t;
		sxx += t * dx;
		cr += ua.y * sweep.r[step];
		cg += ua.y * sweep.g[step];
		cb += ua.y * sweep.b[step];
		if (kDepth)
			cdp += ua.y * g_depth[9 * (lane & 7) + step];
	}
	// the two halves of the strip row first (dy is theirs in common), then the four strip rows
	float w[7] = {s0, sx, sxx, cr, cg, cb, cdp};
#pragma unroll
	for (int q = 0; q < (kDepth ? 7 : 6); q++)
		w[q] = dpp_exchange_add<0xB1>(w[q]);  // quad_perm:[1,0,3,2]
	float v[10] = {w[0], w[1], dy * w[0], w[2], dy * w[1], dy * dy * w[0], w[3], w[4], w[5], w[6]};
#pragma unroll
	for (int q = 0; q < (kDepth ? 10 : 9); q++) {
		v[q] = dpp_exchange_add<0x4E>(v[q]);   // quad_perm:[2,3,0,1]
		v[q] = dpp_exchange_add<0x141>(v[q]);  // row_half_mirror: the other quad of the eight
	}
	// (every lane forms all five products and then picks its own: a handful of multiplications more than the one or two
	// a lane needs, but no branch per column and no wait for the conic inside one)
	const float2 rest = *reinterpret_cast<const float2*>(&st.rest[slot]);
	const float4 co = float4{centre.z, centre.w, rest.x, rest.y};  // the staged conic: -xx / 2, -xy, -yy / 2, opacity
	const uint32_t sum_row = st.sum_row[slot];
	const float S0 = v[0], Sx = v[1], Sy = v[2], Sxx = v[3], Sxy = v[4], Syy = v[5];
	const float half_w = -0.5f * co.w;
	const float m0 = co.w * f.ddelx_dx * (2.f * co.x * Sx + co.y * Sy), m1 = co.w * f.ddely_dy * (2.f * co.z * Sy + co.y * Sx);
	const float k0 = half_w * Sxx, k1 = half_w * Sxy, k3 = half_w * Syy;
	// lane j of the eight holds column j of the row, lanes 0 and 1 also columns 8 and 9: see SumCol
	// (picked bit by bit of j: a chain of comparisons becomes a switch)
	const bool j0 = (j & 1) != 0, j1 = (j & 2) != 0, j2 = (j & 4) != 0;
	const float c01 = j0 ? m1 : m0, c23 = j0 ? k1 : k0, c45 = j0 ? S0 : k3, c67 = j0 ? v[7] : v[6];
	const float c03 = j1 ? c23 : c01, c47 = j1 ? c67 : c45;
	const float c89 = j0 ? (kDepth ? v[9] : 0.f) : v[8];
	const float first = j2 ? c47 : c03, second = !j1 && !j2 ? c89 : 0.f;
	// columns 8 and 9 and the Gaussian's row go to the same lanes of the other eight of the 16-lane row (row_ror:8)
	const float second_there = __builtin_bit_cast(
		float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, second), 0x128, 0xF, 0xF, true));
	const uint32_t row_there = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)sum_row, 0x128, 0xF, 0xF, true);
	// Entries 0-3: their own (lower) lanes add columns 0-7, the upper lanes columns 8 and 9 for them; then entries 4-7 the
	// other way round.  Which entries some pixel blended is asked here alone (an entry that none blends, as the slots behind the
	// last one, has zeros in its row, which an upstream gradient that is not finite would turn into NaN): with a branch around
	// the choices above, the compiler moves the last additions of the exchanges into it and their lane moves stay outside as
	// instructions of their own.
	const float low = upper ? second_there : first, high = upper ? first : second_there;
	float* at_low = reinterpret_cast<float*>(reinterpret_cast<char*>(sweep.column_low) + ((uint64_t)(upper ? row_there : sum_row) << 4));
	float* at_high = reinterpret_cast<float*>(reinterpret_cast<char*>(sweep.column_high) + ((uint64_t)(upper ? sum_row : row_there) << 4));
	if (__builtin_amdgcn_inverse_ballot_w64(blended.low) && low != 0.f)
		unsafeAtomicAdd(at_low, low);
	if (__builtin_amdgcn_inverse_ballot_w64(blended.high) && high != 0.f)
		unsafeAtomicAdd(at_high, high);
	__builtin_amdgcn_wave_barrier();
}

// Pixel-parallel part for the four entries staged from slot k on: first what needs no other entry, then the recurrences.
// kVisit: which comparisons the chunk's entries need (three of 29 vector instructions per entry; with an entry's words in
// the order of their reads 2 775 -> 2 740 us at 5185x3359, 64.5 -> 63 for 100 000 Gaussians at 512x512).
enum Visit { kVisitAll, kVisitPlain, kVisitPlainReached };  // plain: see plain_entry; reached: every pixel blended an entry behind the chunk
struct VisitedEntries {
	float alpha[4], G[4], inv[4], weighted[4];
	uint64_t mask[4];  // the pixels that blended the entry
};
template <bool kDepth, BoxTest kBox, Visit kVisit>
__device__ __forceinline__ void backward_visit(VisitedEntries& v, const BackwardPixel& p, uint32_t last_contributor, const BackwardChunk& st, int k,
                                               const StripRays& rays, const float2 pixf, const BoxSpan& span, const BlendArgs& a)
{
	float power[4], clip_w[4], opacity[4];
	float (&alpha)[4] = v.alpha, (&G)[4] = v.G, (&inv)[4] = v.inv, (&weighted)[4] = v.weighted;
	uint64_t (&mask)[4] = v.mask;
#pragma unroll
	for (int i = 0; i < 4; i++) {
		const float4 centre_conic = st.centre_conic[k + i], rest = st.rest[k + i];
		power[i] = exponent_of_staged(centre_conic, rest.x, pixf);
		opacity[i] = rest.y;
		clip_w[i] = rest.z;
		// (each mask from single comparisons: a comparison's result is the mask; nearly every walked entry is blended
		// by some pixel, so the exponent's floor, which would spare an exponential now and then, is not looked at)
		mask[i] = ~0ull;
		if (kVisit != kVisitPlainReached)
			mask[i] = lanes_where(__float_as_uint(rest.w) < last_contributor);
		if (kVisit == kVisitAll)
			mask[i] &= lanes_where(!(power[i] > 0.0f));
	}
	// the entries' colours are asked for ahead of the exponentials
	float4 cd[4];
#pragma unroll
	for (int i = 0; i < 4; i++)
		cd[i] = st.cd[k + i];
	__builtin_amdgcn_sched_barrier(0);
#pragma unroll
	for (int i = 0; i < 4; i++) {
		G[i] = exp_of_exponent(power[i]);
		alpha[i] = kVisit == kVisitAll ? fminf(0.99f, opacity[i] * G[i]) : opacity[i] * G[i];
		mask[i] &= lanes_where(!(alpha[i] < 1.0f / 255.0f));
		if (kBox == kBoxSpans)
			mask[i] = lanes_inside_box(mask[i], clip_w[i], span, rays, a);
		if (kBox == kBoxExact)
			mask[i] = lanes_inside_box(mask[i], clip_w[i], rays, a);
		// From here on nothing feeds a decision: gradients are compared by tolerance, so the divisions use the hardware
		// reciprocal.
		inv[i] = __builtin_amdgcn_rcpf(1.f - alpha[i]);
		weighted[i] = __builtin_fmaf(cd[i].x, p.g_r, __builtin_fmaf(cd[i].y, p.g_g, __builtin_fmaf(cd[i].z, p.g_b, p.g_alpha)));
		if (kDepth)
			weighted[i] = __builtin_fmaf(cd[i].w, p.g_depth, weighted[i]);
	}
}

// `rows`: the pixel's place in the first of the four entries' rows.  Returns, as sum_rows asks for it (16 lanes per entry), which of them
// any pixel blended.
__device__ __forceinline__ uint64_t backward_rows(BackwardPixel& p, const VisitedEntries& v, LdsPair* rows)
{
	// The pixel's outputs are sums over its blended entries j of w_j (colour_j, depth_j, 1) with w_j = alpha_j T_j,
	// T_j the product of (1 - alpha_k) over the entries in front, plus T_final times the background.  Their
	// derivative with respect to alpha_i is T_i (colour_i, depth_i, 1) minus (the sum over the entries behind i +
	// T_final background) / (1 - alpha_i).  The reference carries that sum per channel and per unit of transmittance
	// (K/cuda_rasterizer_hgs/backward.cu:568-599: accum_rec = last_alpha * last_color + (1 - last_alpha) * accum_rec,
	// and the background term apart); only its product with the upstream gradient is needed, so one number per
	// pixel does for all channels: `behind` = sum over the entries behind of w_j <g, (colour_j, depth_j, 1)> +
	// T_final <g, background>, started with the latter.
	// Under the mask of the pixels that blend the entry, written out: the compiler would put a branch around each of the
	// four (the mask's move is also the instruction that has to lie between a reciprocal and the first use of it).
#pragma unroll
	for (int i = 0; i < 4; i++) {
		float dL_dopa;
		Pair z = zero_pair();
		float u = z.x, aT = z.y;
		uint64_t active;
		asm("s_and_saveexec_b64 %[active], %[lanes]\n\t"
		    "v_mul_f32 %[T], %[T], %[inv]\n\t"
		    "v_mul_f32 %[d], %[behind], %[inv]\n\t"
		    "v_mul_f32 %[aT], %[alpha], %[T]\n\t"
		    "v_fma_f32 %[d], %[weighted], %[T], -%[d]\n\t"
		    "v_fmac_f32 %[behind], %[aT], %[weighted]\n\t"
		    "v_mul_f32 %[u], %[G], %[d]\n\t"
		    "s_mov_b64 exec, %[active]"
		    : [T] "+v"(p.T), [behind] "+v"(p.behind), [aT] "+v"(aT), [u] "+v"(u), [d] "=&v"(dL_dopa), [active] "=&s"(active)
		    : [lanes] "s"(v.mask[i]), [inv] "v"(v.inv[i]), [alpha] "v"(v.alpha[i]), [weighted] "v"(v.weighted[i]), [G] "v"(v.G[i])
		    : "scc");
		rows[i * kRowStride] = Pair{u, aT};
	}
	uint64_t blended = 0ull;
#pragma unroll
	for (int i = 0; i < 4; i++)
		blended |= v.mask[i] != 0ull ? 0xFFFFull << (16 * i) : 0ull;
	return blended;
}

// The entries of a chunk, eight at a time.
template <bool kDepth, BoxTest kBox, Visit kVisit>
__device__ __forceinline__ void backward_chunk(BackwardPixel& p, uint32_t last_contributor, const BackwardStage& st, int count,
                                               LdsPair* const (&rows)[2], const float2 pixf, const BoxSpan& span, const Sweep& sweep,
                                               const StripFrame& frame, int lane, const BlendArgs& a)
{
	for (int k = 0; k < count; k += kRows) {
		VisitedEntries v;
		Blended blended;
		backward_visit<kDepth, kBox, kVisit>(v, p, last_contributor, st.chunk, k, st.rays, pixf, span, a);
		blended.low = backward_rows(p, v, rows[0]);
		backward_visit<kDepth, kBox, kVisit>(v, p, last_contributor, st.chunk, k + 4, st.rays, pixf, span, a);
		blended.high = backward_rows(p, v, rows[1]);
		if ((blended.low | blended.high) != 0ull)
			sum_rows<kDepth>(st.chunk, st.g_depth, k, blended, sweep, frame, lane);
	}
}

// Files a chunk's entry of this lane, and behind the last one entries up to a multiple of eight that lie behind every pixel's last one.
__device__ __forceinline__ void stage_backward(BackwardChunk& st, const LoadedRecord& cur, uint32_t pos_cur, int count, int lane)
{
	if (lane < count) {
		const float w = (pos_cur & 0x80000000u) ? __int_as_float(0x7FC00000) : cur.geom.w;  // (the strip lies inside the box: no per-pixel test)
		const float4 conic = staged_conic(cur.conic);
		st.centre_conic[lane] = float4{cur.geom.x, cur.geom.y, conic.x, conic.y};
		st.rest[lane] = float4{conic.z, conic.w, w, __uint_as_float(pos_cur & kPosition)};
		st.cd[lane] = cur.cd;
		st.sum_row[lane] = kSumCols / 4 * cur.id;  // (32 bits hold it: a thousand million Gaussians' gradients fit no device)
	}
	if (lane < kRows - 1) {
		st.centre_conic[count + lane] = float4{0.f, 0.f, 0.f, 0.f};
		st.rest[count + lane] = float4{0.f, 0.f, 0.f, __uint_as_float(0xFFFFFFFFu)};
		st.cd[count + lane] = float4{0.f, 0.f, 0.f, 0.f};
		st.sum_row[count + lane] = 0u;
	}
}

template <bool kDepth>
__device__ __forceinline__ void backward_strip(const BlendArgs& a, uint32_t strip_id, BackwardStage& st, int lane)
{
	const int tile = (int)(strip_id >> 2), wave = (int)(strip_id & 3u);  // wave: which strip of the tile
	uint2 range = a.ranges[tile];
	range.y = min(range.y, a.capacity);
	range.x = min(range.x, range.y);
	const int tx = tile % a.grid_x, ty = tile / a.grid_x;
	const uint32_t px = tx * kTile + (lane & 15), py = ty * kTile + wave * 4 + (lane >> 4);
	const bool inside = px < (uint32_t)a.W && py < (uint32_t)a.H;
	const uint32_t pix_id = (uint32_t)a.W * py + px;
	const float2 pixf = {(float)px, (float)py};
	const size_t plane = (size_t)a.H * a.W;
	const float strip_x0 = (float)(tx * kTile), strip_y0 = (float)(ty * kTile + wave * 4);
	const StripFrame frame = {strip_x0, strip_y0, (float)(0.5 * a.W), (float)(0.5 * a.H)};

	// The forward blend has written down which entries of the tile's list matter to this strip
	// (its conservative filters, not repeated here), up to the last one that any pixel blended.
	const uint32_t n = range.y - range.x;
	const uint32_t filed = min(a.strip_filed[strip_id], n);
	if (filed == 0u)
		return;
	const uint32_t last_contributor = inside ? a.n_contrib[pix_id] : 0u;

	BackwardPixel p;
	const float T_final = inside ? (1 - a.out_alpha[pix_id]) : 0.f;
	p.T = T_final;
	p.g_r = p.g_g = p.g_b = p.g_depth = p.g_alpha = 0.f;
	if (inside) {
		p.g_r = a.dL_dpix[pix_id];
		p.g_g = a.dL_dpix[plane + pix_id];
		p.g_b = a.dL_dpix[2 * plane + pix_id];
		p.g_depth = a.dL_dpix_depth ? a.dL_dpix_depth[pix_id] : 0.f;  // absent: no gradient came in
		p.g_alpha = a.dL_dalpha ? a.dL_dalpha[pix_id] : 0.f;
	}
	p.behind = T_final * ((0.f + a.bg[0] * p.g_r + a.bg[1] * p.g_g) + a.bg[2] * p.g_b);

	stage_rays(st.rays, pixf, a, lane);
	Sweep sweep;
	{
		const int upper = (lane >> 3) & 1, e = (lane >> 4) + 4 * upper, h = (lane >> 1) & 3, j = lane & 7;
		sweep.row = lds_base(st.u_at + e * kRowStride + row_column(h * 16 + 8 * (lane & 1)));
		sweep.column_low = a.sums + (upper ? 8 + j : j);
		sweep.column_high = a.sums + (upper ? j : 8 + j);
		float4* by_pixel = st.chunk.centre_conic;  // (not in use yet)
		by_pixel[lane] = float4{p.g_r, p.g_g, p.g_b, 0.f};
		if (kDepth)
			st.g_depth[lane + (lane >> 3)] = p.g_depth;
		__builtin_amdgcn_wave_barrier();
#pragma unroll
		for (int s = 0; s < 8; s++) {
			const float4 g = by_pixel[8 * (lane & 7) + s];  // pixels of strip row (lane >> 1) & 3, half lane & 1
			sweep.r[s] = g.x;
			sweep.g[s] = g.y;
			sweep.b[s] = g.z;
		}
		__builtin_amdgcn_wave_barrier();
	}

	LdsPair* const rows[2] = {lds_base(st.u_at + row_column(lane)), lds_base(st.u_at + 4 * kRowStride + row_column(lane))};

	// Lane l of the chunk that starts `first` entries from the back takes filed entry
	// filed-1-first-l: its list position (and box flag), through that the Gaussian's index,
	// through that its record.  Three chunks are in flight: the records of the next one, the
	// indices of the one after, the positions of the one after that.
	const uint32_t* list = a.point_list + range.x;
	const uint32_t* filed_list = a.strip_lists + 4 * (size_t)range.x + (size_t)wave * n;
	uint32_t pos_cur = (uint32_t)lane < filed ? filed_list[filed - 1 - lane] : kNone;
	uint32_t pos_next = (uint32_t)(64 + lane) < filed ? filed_list[filed - 1 - (64 + lane)] : kNone;
	uint32_t pos_after = (uint32_t)(128 + lane) < filed ? filed_list[filed - 1 - (128 + lane)] : kNone;
	LoadedRecord cur = load_record(a, pos_cur != kNone ? list[min(pos_cur & kPosition, n - 1u)] : 0u, pos_cur != kNone);
	uint32_t id_next = pos_next != kNone ? list[min(pos_next & kPosition, n - 1u)] : 0u;

	BoxSpan span;  // of the pixel, from the first chunk that straddles a face of the box on
	bool have_span = false;
	for (uint32_t first = 0; first < filed; first += 64) {
		const int count = (int)min(filed - first, 64u);
		stage_backward(st.chunk, cur, pos_cur, count, lane);
		const bool straddles = lane < count && (pos_cur & 0x80000000u) == 0u;
		const bool boxed = lanes_where(straddles) != 0ull, all_in_front = lanes_where(straddles && !(cur.geom.w > 0.f)) == 0ull;
		// (lane 0 holds the chunk's entry that lies furthest back; the padding's opacity is 0)
		const bool plain = lanes_where(lane < count && !plain_entry(cur)) == 0ull;
		const bool reached = lanes_where((uint32_t)__builtin_amdgcn_readfirstlane((int)(pos_cur & kPosition)) >= last_contributor) == 0ull;
		__builtin_amdgcn_wave_barrier();
		// the chunk is in LDS now: its registers take the next chunk's records, loaded during the walk
		cur = load_record(a, id_next, pos_next != kNone);
		pos_cur = pos_next;
		pos_next = pos_after;
		id_next = pos_next != kNone ? list[min(pos_next & kPosition, n - 1u)] : 0u;
		const uint32_t e3 = first + 192 + (uint32_t)lane;
		pos_after = e3 < filed ? filed_list[filed - 1 - e3] : kNone;

		// (few strips straddle a face of their box: their chunks run copies of the loop that have the test)
		if (boxed && all_in_front) {
			if (kDepth || !have_span) {  // (with the depth terms no registers are left to hold it)
				span = w_inside_box(ray_of(st.rays), load_box_frame(a));
				have_span = true;
			}
			backward_chunk<kDepth, kBoxSpans, kVisitAll>(p, last_contributor, st, count, rows, pixf, span, sweep, frame, lane, a);
		} else if (boxed) {
			backward_chunk<kDepth, kBoxExact, kVisitAll>(p, last_contributor, st, count, rows, pixf, span, sweep, frame, lane, a);
		} else if (plain && reached) {
			backward_chunk<kDepth, kBoxNone, kVisitPlainReached>(p, last_contributor, st, count, rows, pixf, span, sweep, frame, lane, a);
		} else if (plain) {
			backward_chunk<kDepth, kBoxNone, kVisitPlain>(p, last_contributor, st, count, rows, pixf, span, sweep, frame, lane, a);
		} else {
			backward_chunk<kDepth, kBoxNone, kVisitAll>(p, last_contributor, st, count, rows, pixf, span, sweep, frame, lane, a);
		}
		__builtin_amdgcn_wave_barrier();
	}
}

template <bool kDepth>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 4))) void blend_backward_kernel(BlendBatch batch)
{
	__shared__ BackwardStage st;
	// the jobs of the batch take turns; each hands out its strips with the most entries first: a long
	// strip that starts late is what the whole launch waits for (workgroups and their turns as in blend_forward_kernel; a strip
	// without entries to walk needs nothing)
	const BlendArgs& a = batch.job[blockIdx.x % (uint32_t)batch.count];
	const uint32_t number = blockIdx.x / (uint32_t)batch.count;
	uint32_t strip_id = a.strip_order[number];
	const uint32_t filled = batch.strips - min(a.strip_classes[strip_empty_word(0)], batch.strips);
	for (uint32_t at = number, turn = 0; at < filled;) {
		// What the forward left in the workspaces (the strips' order, the tiles' ranges, the lists, the walk lengths) comes
		// back through the caller's hands: every index taken from it is held inside the arrays' bounds, so that a
		// workspace that is not the forward's (stale, or another frame's) gives wrong gradients and no stray access.
		int lane = threadIdx.x;
		asm volatile("" : "+v"(lane));  // (what follows from it is worked out per turn: held from the first on, it costs registers)
		backward_strip<kDepth>(a, min(strip_id, batch.strips - 1u), st, lane);
		at = turn_of_workgroup(number, ++turn, batch.workgroups);
		if (at < filled)
			strip_id = a.strip_order[at];
	}
}

// ---- a backward walk shared by four wavefronts -------------------------------------------------
// A wavefront alone on its SIMD takes 0.2 us per entry, twice what issuing its instructions takes and far more than a
// strip's share where the chip is full, so a launch of few strips lasts as long as its longest walks.  There (see long_strip_classes) four
// wavefronts walk a strip, a pass of eight entries each in turn.  What needs no other entry (exponentials, alphas, reciprocals, colours
// against the upstream gradient) and the sums over the pixels run side by side; transmittance and `behind` of the 64 pixels are
// handed from pass to pass through LDS, and only three instructions per entry lie between taking and passing them on.  They and what
// follows are the operations of one wavefront's walk on the same operands in the same order (factors of an entry that a pixel did not blend are made 1, 0
// and 0, which leaves both as they are), and as many additions go to each Gaussian's row.  (Shared by pixels instead, as the forward's
// walk, four times as many do, and additions to one address take 12 ns each.  Eight wavefronts: 67 to 75 us for 100 000 Gaussians at
// 512x512, four 50, two 44; but two 112 for 61 000 Gaussians of two submodels at 397x251, four 72.)
// Chunks are staged in turn as well, two ahead of their use, in kStagedChunks buffers.  The wavefronts of a workgroup run at the same
// time and every word that one waits for is written by one that waits for earlier passes alone; the waits are bounded all the same.
constexpr int kSharedWaves = 4;
constexpr int kStagedChunks = 4;
enum ChunkKind : uint32_t { kChunkSpans, kChunkExact, kChunkReached, kChunkPlain, kChunkAll };  // which copy of the loop a chunk runs
constexpr int kSharedPolls = 1 << 20;

struct SharedStage {
	BackwardChunk chunk[kStagedChunks];
	float2 u_at[kSharedWaves][kRows * kRowStride];
	float2 carry[64];     // per pixel: transmittance and `behind`, as the pass before left them
	float g_depth[72];
	StripRays rays;
	uint32_t turn;                    // the pass that may take `carry`
	uint32_t staged[kStagedChunks];   // one more than the chunk that a buffer holds
	uint32_t kind[kStagedChunks];
	uint32_t walked[kSharedWaves];          // chunks that a wavefront is done with
};

// Waits until a word that another wavefront of the workgroup counts up has reached `value`.  (A wavefront's LDS accesses are served in
// order, so what the writer stored ahead of the word is there when the word is; the empty assembly keeps the compiler to that order.)
__device__ __forceinline__ void wait_for(const uint32_t* word, uint32_t value)
{
	for (int polls = 0; polls < kSharedPolls; polls++) {
		const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
		if ((int)(v - value) >= 0)
			break;
		__builtin_amdgcn_s_sleep(0);
	}
	asm volatile("" ::: "memory");
}
__device__ __forceinline__ void publish(uint32_t* word, uint32_t value, int lane)
{
	asm volatile("" ::: "memory");
	if (lane == 0)
		__hip_atomic_store(word, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
	asm volatile("" ::: "memory");
}

// The pixel's transmittance and `behind` once it is the turn of `pass`, read with the word that says so.
__device__ __forceinline__ float2 wait_for_carry(const uint32_t& turn, const float2& carry, uint32_t pass)
{
	float2 c;
	for (int polls = 0; polls < kSharedPolls; polls++) {
		const uint32_t v = __hip_atomic_load(&turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
		asm volatile("" ::: "memory");
		c = carry;
		asm volatile("" ::: "memory");
		if ((uint32_t)__builtin_amdgcn_readfirstlane((int)v) == pass)
			break;
	}
	return c;
}

template <bool kDepth, BoxTest kBox, Visit kVisit>
__device__ __forceinline__ void backward_chunk_shared(BackwardPixel& p, uint32_t last_contributor, SharedStage& st, int buffer, uint32_t first_pass,
                                                      int count, LdsPair* const (&rows)[2], const float2 pixf, const BoxSpan& span, const Sweep& sweep,
                                                      const StripFrame& frame, int lane, int wave, const BlendArgs& a)
{
	const BackwardChunk& chunk = st.chunk[buffer];
	for (int k = kRows * wave; k < count; k += kRows * kSharedWaves) {
		VisitedEntries v[2];
		backward_visit<kDepth, kBox, kVisit>(v[0], p, last_contributor, chunk, k, st.rays, pixf, span, a);
		backward_visit<kDepth, kBox, kVisit>(v[1], p, last_contributor, chunk, k + 4, st.rays, pixf, span, a);
		Blended blended = {0ull, 0ull};
#pragma unroll
		for (int i = 0; i < 8; i++) {
			VisitedEntries& e = v[i >> 2];
			const bool took = __builtin_amdgcn_inverse_ballot_w64(e.mask[i & 3]);
			e.inv[i & 3] = took ? e.inv[i & 3] : 1.f;
			e.alpha[i & 3] = took ? e.alpha[i & 3] : 0.f;
			e.weighted[i & 3] = took ? e.weighted[i & 3] : 0.f;
			uint64_t& b = i < 4 ? blended.low : blended.high;
			b |= e.mask[i & 3] != 0ull ? 0xFFFFull << (16 * (i & 3)) : 0ull;
		}
		const uint32_t pass = first_pass + (uint32_t)k / kRows;
		const float2 carry = wait_for_carry(st.turn, st.carry[lane], pass);
		{
			float T = carry.x, behind = carry.y;
#pragma unroll
			for (int i = 0; i < 8; i++) {
				const VisitedEntries& e = v[i >> 2];
				T *= e.inv[i & 3];
				behind = __builtin_fmaf(e.alpha[i & 3] * T, e.weighted[i & 3], behind);
			}
			st.carry[lane] = float2{T, behind};
		}
		publish(&st.turn, pass + 1u, lane);
		{
			// (once more, with what it gives each entry: kept from above it would take 24 registers)
			float T = carry.x, behind = carry.y;
			asm volatile("" : "+v"(T), "+v"(behind));
#pragma unroll
			for (int i = 0; i < 8; i++) {
				const VisitedEntries& e = v[i >> 2];
				T *= e.inv[i & 3];
				const float past = behind * e.inv[i & 3], aT = e.alpha[i & 3] * T, d = __builtin_fmaf(e.weighted[i & 3], T, -past);
				behind = __builtin_fmaf(aT, e.weighted[i & 3], behind);
				// (a transmittance that is not finite stays out of the rows of entries that the pixel did not blend)
				const bool took = __builtin_amdgcn_inverse_ballot_w64(e.mask[i & 3]);
				rows[i >> 2][(i & 3) * kRowStride] = Pair{took ? e.G[i & 3] * d : 0.f, took ? aT : 0.f};
			}
		}
		if ((blended.low | blended.high) != 0ull)
			sum_rows<kDepth>(chunk, st.g_depth, k, blended, sweep, frame, lane);
	}
}

template <bool kDepth>
__device__ __forceinline__ void backward_strip_shared(const BlendArgs& a, uint32_t strip_id, SharedStage& st, int lane, int wave)
{
	const int tile = (int)(strip_id >> 2), strip = (int)(strip_id & 3u);
	uint2 range = a.ranges[tile];
	range.y = min(range.y, a.capacity);
	range.x = min(range.x, range.y);
	const int tx = tile % a.grid_x, ty = tile / a.grid_x;
	const uint32_t px = tx * kTile + (lane & 15), py = ty * kTile + strip * 4 + (lane >> 4);
	const bool inside = px < (uint32_t)a.W && py < (uint32_t)a.H;
	const uint32_t pix_id = (uint32_t)a.W * py + px;
	const float2 pixf = {(float)px, (float)py};
	const size_t plane = (size_t)a.H * a.W;
	const StripFrame frame = {(float)(tx * kTile), (float)(ty * kTile + strip * 4), (float)(0.5 * a.W), (float)(0.5 * a.H)};
	const uint32_t n = range.y - range.x;
	const uint32_t filed = min(a.strip_filed[strip_id], n);
	if (filed == 0u)  // (the same for every wavefront)
		return;
	const uint32_t last_contributor = inside ? a.n_contrib[pix_id] : 0u;

	// the wavefront's own chunks, every kSharedWaves-th
	const uint32_t* list = a.point_list + range.x;
	const uint32_t* filed_list = a.strip_lists + 4 * (size_t)range.x + (size_t)strip * n;
	auto position = [&](uint32_t chunk) {
		const uint32_t e = 64u * chunk + (uint32_t)lane;
		return e < filed ? filed_list[filed - 1u - e] : kNone;
	};
	auto index_of = [&](uint32_t pos) { return pos != kNone ? list[min(pos & kPosition, n - 1u)] : 0u; };
	uint32_t next_chunk = (uint32_t)wave;
	uint32_t pos_cur = position(next_chunk), pos_next = position(next_chunk + kSharedWaves), pos_after = position(next_chunk + 2 * kSharedWaves);
	LoadedRecord cur = load_record(a, index_of(pos_cur), pos_cur != kNone);
	uint32_t id_next = index_of(pos_next);

	BackwardPixel p;
	const float T_final = inside ? (1 - a.out_alpha[pix_id]) : 0.f;
	p.T = T_final;
	p.g_r = p.g_g = p.g_b = p.g_depth = p.g_alpha = 0.f;
	if (inside) {
		p.g_r = a.dL_dpix[pix_id];
		p.g_g = a.dL_dpix[plane + pix_id];
		p.g_b = a.dL_dpix[2 * plane + pix_id];
		p.g_depth = a.dL_dpix_depth ? a.dL_dpix_depth[pix_id] : 0.f;
		p.g_alpha = a.dL_dalpha ? a.dL_dalpha[pix_id] : 0.f;
	}
	p.behind = T_final * ((0.f + a.bg[0] * p.g_r + a.bg[1] * p.g_g) + a.bg[2] * p.g_b);

	float4* by_pixel = reinterpret_cast<float4*>(st.u_at[0]);  // (not in use yet)
	if (wave == 0) {
		stage_rays(st.rays, pixf, a, lane);
		by_pixel[lane] = float4{p.g_r, p.g_g, p.g_b, 0.f};
		st.carry[lane] = float2{p.T, p.behind};
		if (kDepth)
			st.g_depth[lane + (lane >> 3)] = p.g_depth;
		if (lane == 0)
			st.turn = 0u;
		if (lane < kStagedChunks)
			st.staged[lane] = 0u;
		if (lane < kSharedWaves)
			st.walked[lane] = 0u;
	}
	__syncthreads();
	Sweep sweep;
	{
		const int upper = (lane >> 3) & 1, e = (lane >> 4) + 4 * upper, h = (lane >> 1) & 3, j = lane & 7;
		sweep.row = lds_base(st.u_at[wave] + e * kRowStride + row_column(h * 16 + 8 * (lane & 1)));
		sweep.column_low = a.sums + (upper ? 8 + j : j);
		sweep.column_high = a.sums + (upper ? j : 8 + j);
#pragma unroll
		for (int s = 0; s < 8; s++) {
			const float4 g = by_pixel[8 * (lane & 7) + s];
			sweep.r[s] = g.x;
			sweep.g[s] = g.y;
			sweep.b[s] = g.z;
		}
	}
	__syncthreads();
	LdsPair* const rows[2] = {lds_base(st.u_at[wave] + row_column(lane)), lds_base(st.u_at[wave] + 4 * kRowStride + row_column(lane))};

	const uint32_t chunks = (filed + 63u) / 64u;
	auto stage = [&]() {
		const uint32_t buffer = next_chunk % kStagedChunks;
		const int count = (int)min(filed - 64u * next_chunk, 64u);
		stage_backward(st.chunk[buffer], cur, pos_cur, count, lane);
		const bool straddles = lane < count && (pos_cur & 0x80000000u) == 0u;
		const bool boxed = lanes_where(straddles) != 0ull, all_in_front = lanes_where(straddles && !(cur.geom.w > 0.f)) == 0ull;
		const bool plain = lanes_where(lane < count && !plain_entry(cur)) == 0ull;
		const bool reached = lanes_where((uint32_t)__builtin_amdgcn_readfirstlane((int)(pos_cur & kPosition)) >= last_contributor) == 0ull;
		const uint32_t kind = boxed ? (all_in_front ? kChunkSpans : kChunkExact) : plain ? (reached ? kChunkReached : kChunkPlain) : kChunkAll;
		if (lane == 0)
			st.kind[buffer] = kind;
		publish(&st.staged[buffer], next_chunk + 1u, lane);
		next_chunk += kSharedWaves;
		cur = load_record(a, id_next, pos_next != kNone);
		pos_cur = pos_next;
		pos_next = pos_after;
		id_next = index_of(pos_next);
		pos_after = position(next_chunk + 2 * kSharedWaves);
	};
	if (next_chunk < min(chunks, 2u))
		stage();

	BoxSpan span;
	bool have_span = false;
	for (uint32_t c = 0; c < chunks; c++) {
		if (next_chunk == c + 2u && next_chunk < chunks) {
			// its buffer held chunk c - 2
#pragma unroll
			for (int w = 0; w < kSharedWaves; w++)
				if (c >= 2u)
					wait_for(&st.walked[w], c - 1u);
			stage();
		}
		const int buffer = (int)(c % kStagedChunks);
		wait_for(&st.staged[buffer], c + 1u);
		const uint32_t kind = (uint32_t)__builtin_amdgcn_readfirstlane((int)st.kind[buffer]);
		const int count = (int)min(filed - 64u * c, 64u);
		if (kind == kChunkSpans) {
			if (kDepth || !have_span) {
				span = w_inside_box(ray_of(st.rays), load_box_frame(a));
				have_span = true;
			}
			backward_chunk_shared<kDepth, kBoxSpans, kVisitAll>(p, last_contributor, st, buffer, 8u * c, count, rows, pixf, span, sweep, frame, lane, wave, a);
		} else if (kind == kChunkExact) {
			backward_chunk_shared<kDepth, kBoxExact, kVisitAll>(p, last_contributor, st, buffer, 8u * c, count, rows, pixf, span, sweep, frame, lane, wave, a);
		} else if (kind == kChunkReached) {
			backward_chunk_shared<kDepth, kBoxNone, kVisitPlainReached>(p, last_contributor, st, buffer, 8u * c, count, rows, pixf, span, sweep, frame, lane, wave, a);
		} else if (kind == kChunkPlain) {
			backward_chunk_shared<kDepth, kBoxNone, kVisitPlain>(p, last_contributor, st, buffer, 8u * c, count, rows, pixf, span, sweep, frame, lane, wave, a);
		} else {
			backward_chunk_shared<kDepth, kBoxNone, kVisitAll>(p, last_contributor, st, buffer, 8u * c, count, rows, pixf, span, sweep, frame, lane, wave, a);
		}
		publish(&st.walked[wave], c + 1u, lane);
	}
}

// Launches of few strips: the longest walks by a workgroup each, of the others one per wavefront (neighbours in the order, so they end at
// about the same time).  Three wavefronts per SIMD: what the shared walk holds fits 168 registers, and the others run as fast as with four.
template <bool kDepth>
__global__ __launch_bounds__(64 * kSharedWaves) __attribute__((amdgpu_waves_per_eu(3, 3))) void blend_backward_shared_kernel(BlendBatch batch)
{
	__shared__ union Stages {
		SharedStage shared;
		BackwardStage alone[kSharedWaves];
		__device__ Stages() {}
	} st;
	const BlendArgs& a = batch.job[blockIdx.x % (uint32_t)batch.count];
	const uint32_t number = blockIdx.x / (uint32_t)batch.count;
	const uint32_t filled = batch.strips - min(a.strip_classes[strip_empty_word(0)], batch.strips);
	const uint32_t longer = min(a.strip_classes[kStripLongWord], filled), items = longer + (filled - longer + kSharedWaves - 1u) / kSharedWaves;
	const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	for (uint32_t at = number, turn = 0; at < items; at = turn_of_workgroup(number, ++turn, batch.workgroups)) {
		int lane = (int)(threadIdx.x & 63u);
		asm volatile("" : "+v"(lane));
		if (at < longer) {
			backward_strip_shared<kDepth>(a, min(a.strip_order[at], batch.strips - 1u), st.shared, lane, wave);
			__syncthreads();  // the stage is the next strip's
		} else {
			const uint32_t mine = longer + kSharedWaves * (at - longer) + (uint32_t)wave;
			if (mine < filled)
				backward_strip<kDepth>(a, min(a.strip_order[mine], batch.strips - 1u), st.alone[wave], lane);
		}
	}
}

// Strips by decreasing number of entries to walk, in kStripClasses classes of 8 (longer ones share
// the first class); the order inside a class is whatever the atomics give, which is all a
// launch order needs; the strips without any come last.  Two small kernels: count the strips of every class, then place them; one
// launch of each serves every job of a batch (blockIdx.y).  Both aggregate in LDS first: most
// strips fall into one class (nothing to walk), and thousands of global atomics on one word would
// take longer than the blend itself.  What bounds them is the additions of all workgroups to the same few counters, so a
// workgroup takes kOrderStrips strips, four per thread, and the lanes with empty strips (often most of a wavefront) add to their
// LDS counter as one
// (5185x3359, both kernels and both orders: 92 us with a strip per thread, 31 now; 1600x1036: 19 and 20).
constexpr uint32_t kOrderStrips = 1024;

// How many classes, the longest ones, hold strips whose backward walk is shared by four wavefronts: those that one wavefront would be busy
// with for 0.85 of the time that all the launch's entries take the chip (0.2 us per entry alone, 0.094 ns where every SIMD has four
// walks), the entries of all jobs estimated from the job's own.  Backward blend in us, kernel of single wavefronts and this one by that
// fraction (none shared, 2, 1, 0.82, 0.5, 0.35): 61 000 Gaussians of two submodels at 397x251 177, 179, 81, 71, 74, 74, 78; 100 000 at 512x512
// 62, 64, 50, 53, 52, 48, 48; four submodels at 648x420 147, 148, 145, 143, 143, 162, 172; a call on each of four submodels at 1600x1036
// 607, 592, 594, 568, 556, 589, 633; 333 000 at 1013x761 107, 106, 104, 102, 100, 110, 144.
constexpr float kLongWalk = 0.85f * 0.094e-3f / 0.2f;
__device__ __forceinline__ uint32_t long_strip_classes(uint32_t entries, float share)
{
	const float bound = fmaxf(share * (float)entries, 64.f);
	return bound < 2048.f ? strip_class((uint32_t)bound) : 0u;
}

// The calling lane's place among its workgroup's strips of class c (all lanes come here).
__device__ __forceinline__ uint32_t count_in_class(uint32_t* s_count, uint32_t c, bool valid)
{
	const uint64_t last = lanes_where(valid && c == kEmptyClass);
	uint32_t rank = 0;
	if (valid && c != kEmptyClass)
		rank = atomicAdd(&s_count[c], 1u);
	if (last != 0ull) {
		uint32_t base = 0;
		if (lanes_below(~0ull) == 0u)
			base = atomicAdd(&s_count[kEmptyClass], (uint32_t)__popcll(last));
		base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
		if (valid && c == kEmptyClass)
			rank = base + lanes_below(last);
	}
	return rank;
}

struct StripOrderJob {
	const uint32_t* length;  // per strip
	uint32_t* classes;       // kStripClasses counters and as many placement cursors, zero beforehand
	uint32_t* empty;         // how many strips are empty, and their placement cursor, zero beforehand
	uint32_t* order;
	uint32_t* clear;         // per strip, set to zero (may be null)
	uint32_t* longer;        // receives how many strips are long ones (see long_strip_classes; may be null); behind it a word for the sum of lengths, zero beforehand
};
struct StripOrderBatch {
	StripOrderJob job[kMaxBlendBatch];
	uint32_t strips;
	float long_share;  // of all entries: a walk of more is a long one
};

__global__ __launch_bounds__(256) void strip_count_kernel(StripOrderBatch batch)
{
	__shared__ uint32_t s_count[kStripClasses + 1];
	const StripOrderJob& j = batch.job[blockIdx.y];
	s_count[threadIdx.x] = 0;
	if (threadIdx.x == 0)
		s_count[kEmptyClass] = 0;
	__syncthreads();
	uint32_t length[kOrderStrips / 256];
#pragma unroll
	for (uint32_t q = 0; q < kOrderStrips / 256; q++) {
		const uint32_t k = blockIdx.x * kOrderStrips + 256 * q + threadIdx.x;
		length[q] = k < batch.strips ? j.length[k] : 0u;
	}
#pragma unroll
	for (uint32_t q = 0; q < kOrderStrips / 256; q++)
		count_in_class(s_count, strip_class(length[q]), blockIdx.x * kOrderStrips + 256 * q + threadIdx.x < batch.strips);
	__syncthreads();
	if (s_count[threadIdx.x] != 0u)
		atomicAdd(&j.classes[threadIdx.x], s_count[threadIdx.x]);
	if (threadIdx.x == 0 && s_count[kEmptyClass] != 0u)
		atomicAdd(&j.empty[0], s_count[kEmptyClass]);
	if (j.longer) {
		const uint32_t sum = wave_inclusive_scan_u32(length[0] + length[1] + length[2] + length[3]);
		if ((threadIdx.x & 63) == 63 && sum != 0u)
			atomicAdd(&j.longer[1], sum);
	}
}

__global__ __launch_bounds__(256) void strip_place_kernel(StripOrderBatch batch)
{
	__shared__ uint32_t s_count[kStripClasses + 1];  // strips of this block per class, then where they go
	__shared__ uint32_t s_scan[8];
	const StripOrderJob& j = batch.job[blockIdx.y];
	s_count[threadIdx.x] = 0;
	if (threadIdx.x == 0)
		s_count[kEmptyClass] = 0;
	__syncthreads();
	const uint32_t in_class = j.classes[threadIdx.x];
	uint32_t c[kOrderStrips / 256], rank[kOrderStrips / 256];
#pragma unroll
	for (uint32_t q = 0; q < kOrderStrips / 256; q++) {
		const uint32_t k = blockIdx.x * kOrderStrips + 256 * q + threadIdx.x;
		c[q] = strip_class(k < batch.strips ? j.length[k] : 0u);
	}
#pragma unroll
	for (uint32_t q = 0; q < kOrderStrips / 256; q++)
		rank[q] = count_in_class(s_count, c[q], blockIdx.x * kOrderStrips + 256 * q + threadIdx.x < batch.strips);
	__syncthreads();
	uint32_t total;
	const uint32_t start = block256_exclusive_scan_u32(in_class, s_scan, total);
	if (j.longer && blockIdx.x == 0 && threadIdx.x == long_strip_classes(j.longer[1], batch.long_share))
		j.longer[0] = start;
	const uint32_t mine = s_count[threadIdx.x];
	__syncthreads();
	s_count[threadIdx.x] = start + (mine != 0u ? atomicAdd(&j.classes[kStripClasses + threadIdx.x], mine) : 0u);
	if (threadIdx.x == 0)
		s_count[kEmptyClass] = total + (s_count[kEmptyClass] != 0u ? atomicAdd(&j.empty[1], s_count[kEmptyClass]) : 0u);
	__syncthreads();
#pragma unroll
	for (uint32_t q = 0; q < kOrderStrips / 256; q++) {
		const uint32_t k = blockIdx.x * kOrderStrips + 256 * q + threadIdx.x;
		if (k < batch.strips) {
			j.order[s_count[c[q]] + rank[q]] = k;
			if (j.clear)
				j.clear[k] = 0u;
		}
	}
}

// The same for up to kOrderAtOnce strips, in one kernel: one workgroup has them all.  Two kernels of 3.2 and 3.3 us become one of 3.5 at
// 320 strips, 3.7 and 3.7 one of 4.5 at 4 096, 4.5 and 4.1 one of 7.6 at 12 288, each with a launch less; at 20 800 the two are the
// faster ones (9.8 us; 14 for one workgroup).
constexpr uint32_t kOrderAtOnce = 16384;
__global__ __launch_bounds__(1024) void strip_order_kernel(StripOrderBatch batch)
{
	constexpr uint32_t kPerThread = kOrderAtOnce / 1024;
	__shared__ uint32_t s_count[kStripClasses + 1];
	__shared__ uint32_t s_scan[16];
	__shared__ uint32_t s_total;
	const StripOrderJob& j = batch.job[blockIdx.x];
	const uint32_t tid = threadIdx.x, strips = batch.strips;
	uint32_t c[kPerThread], rank[kPerThread], sum = 0;
#pragma unroll
	for (uint32_t q = 0; q < kPerThread; q++) {
		c[q] = 1024 * q + tid < strips ? j.length[1024 * q + tid] : 0u;
		sum += c[q];
	}
	if (tid <= kStripClasses)
		s_count[tid] = 0;
	if (tid == 0)
		s_total = 0;
	__syncthreads();
	if (j.longer) {
		sum = wave_inclusive_scan_u32(sum);
		if ((tid & 63) == 63)
			atomicAdd(&s_total, sum);
	}
#pragma unroll
	for (uint32_t q = 0; q < kPerThread; q++)
		if (1024 * q < strips) {
			c[q] = strip_class(c[q]);
			rank[q] = count_in_class(s_count, c[q], 1024 * q + tid < strips);
		}
	__syncthreads();
	uint32_t total;
	const uint32_t start = block_exclusive_scan_u32<16>(tid < kStripClasses ? s_count[tid] : 0u, s_scan, total);
	if (tid == 0)
		*j.empty = s_count[kEmptyClass];
	if (j.longer && tid == long_strip_classes(s_total, batch.long_share))
		j.longer[0] = start;
	__syncthreads();
	if (tid <= kStripClasses)
		s_count[tid] = start;  // (of the empty class: all the others)
	__syncthreads();
#pragma unroll
	for (uint32_t q = 0; q < kPerThread; q++) {
		const uint32_t k = 1024 * q + tid;
		if (k < strips) {
			j.order[s_count[c[q]] + rank[q]] = k;
			if (j.clear)
				j.clear[k] = 0u;
		}
	}
}

// which: 0 = the forward's order (by the entries filed), 1 = the backward's (by the entries up to the last one blended)
static void launch_strip_order(const BlendArgs* jobs, int count, int which, hipStream_t s)
{
	StripOrderBatch b;
	b.strips = (uint32_t)(4 * jobs[0].grid_x * jobs[0].grid_y);
	b.long_share = kLongWalk * (float)count;
	for (int k = 0; k < count; k++) {
		b.job[k].length = which == 0 ? jobs[k].strip_total : jobs[k].strip_filed;
		b.job[k].classes = jobs[k].strip_classes + (which == 0 ? 2 * kStripClasses : 0);
		b.job[k].clear = which == 0 ? jobs[k].strip_filed : nullptr;  // (the wavefronts that share a strip take the largest of theirs)
		b.job[k].empty = jobs[k].strip_classes + strip_empty_word(which == 0 ? 1 : 0);
		b.job[k].longer = which == 0 ? nullptr : jobs[k].strip_classes + kStripLongWord;
		b.job[k].order = which == 0 ? jobs[k].strip_order_forward : jobs[k].strip_order;
	}
	if (b.strips <= kOrderAtOnce) {
		hipLaunchKernelGGL(strip_order_kernel, dim3((unsigned)count), dim3(1024), 0, s, b);
		return;
	}
	const dim3 grid((b.strips + kOrderStrips - 1) / kOrderStrips, (unsigned)count);
	hipLaunchKernelGGL(strip_count_kernel, grid, dim3(256), 0, s, b);
	hipLaunchKernelGGL(strip_place_kernel, grid, dim3(256), 0, s, b);
}

void launch_blend_count(const BlendArgs& a, hipStream_t s)
{
	stage_mark("blend_count", s);
	hipLaunchKernelGGL(blend_count_kernel, dim3(tile_order_blocks(a.grid_x, a.grid_y)), dim3(256), 0, s, a);
}

void launch_strip_filing(const BlendArgs* jobs, int count, hipStream_t s)
{
	stage_mark("strip_filing", s);
	for (int at = 0; at < count; at += kMaxBlendBatch) {
		BlendBatch batch;
		batch.count = 0;
		uint32_t most = 0;
		for (int k = at; k < count && k < at + kMaxBlendBatch; k++)
			if (jobs[k].capacity != 0u) {
				batch.job[batch.count++] = jobs[k];
				most = jobs[k].capacity > most ? jobs[k].capacity : most;
			}
		if (batch.count)
			hipLaunchKernelGGL(strip_file_place_kernel, dim3((most + kFileGroup - 1) / kFileGroup, (unsigned)batch.count),
			                   dim3(kFileBlock), 0, s, batch);
	}
}

// Workgroups of a job in a blend launch (see blend_forward_kernel): one per strip up to kStripWorkgroups of all jobs together,
// beyond that half as many as strips.  Forward and backward in us with one per strip, half and a quarter as many, all with the
// empty strips dealt out: 104 000 strips of which 28 700 have entries (1600x1036, 4 jobs) 281 + 542, 278 + 539, 286 + 554;
// 1 094 000 strips (5185x3359) 1 735 + 2 889, 1 612 + 2 773, 1 600 + 2 770; 130 560 of which 36 800 (view of a city) 157, 145, 151.
// Where all strips nearly fit the chip at once, second turns only lengthen the launch (12 288 strips at 1013x761: 59 -> 64).
constexpr unsigned kStripWorkgroups = 32768;
static unsigned blend_workgroups(unsigned strips, int jobs)
{
	return (size_t)strips * (size_t)jobs <= kStripWorkgroups ? strips : (strips + 1) / 2;
}

// Whether a launch's strips are shared by four wavefronts each: up to 4 strips per SIMD of the chip, of all jobs together.  Forward blend
// in us, one and four wavefronts per strip: 320 strips 28.9 and 22.8 (4 000 Gaussians), 52 and 36 (60 000); 1 900 strips 28.7 and 26.2,
// 51.7 and 39.7; 3 200 strips of two submodels, with walks that the box leaves unfinished, 123 and 62; 4 096 strips 27.8 and 27.8 (5 000
// Gaussians), 39.7 and 36.7, 53.3 and 49.9; a call with 4 400 to 10 000 strips is 7 to 30 us slower, a frame with 17 700 by 37.
constexpr unsigned kSharedStrips = 4096;
static bool blend_shared(unsigned strips, int jobs) { return (size_t)strips * (size_t)jobs <= kSharedStrips; }

// All jobs share the image size (they are the submodels of one frame, or a single call).
void launch_blend_forward(const BlendArgs* jobs, int count, hipStream_t s)
{
	const unsigned strips = (unsigned)(4 * jobs[0].grid_x * jobs[0].grid_y);
	for (int at = 0; at < count; at += kMaxBlendBatch) {
		BlendBatch batch;
		batch.count = count - at < kMaxBlendBatch ? count - at : kMaxBlendBatch;
		for (int k = 0; k < batch.count; k++)
			batch.job[k] = jobs[at + k];
		stage_mark("strip_order", s);
		launch_strip_order(jobs + at, batch.count, 0, s);
		stage_mark("blend_forward", s);
		batch.strips = strips;
		const bool shared = blend_shared(strips, batch.count);
		batch.workgroups = shared ? 4 * strips : blend_workgroups(strips, batch.count);
		const dim3 grid(batch.workgroups * (unsigned)batch.count);
		if (shared)
			hipLaunchKernelGGL(blend_forward_kernel<true>, grid, dim3(64), 0, s, batch);
		else
			hipLaunchKernelGGL(blend_forward_kernel<false>, grid, dim3(64), 0, s, batch);
		// the order in which the backward will take the strips
		stage_mark("strip_order", s);
		launch_strip_order(jobs + at, batch.count, 1, s);
	}
}

void launch_blend_backward(const BlendArgs* jobs, int count, hipStream_t s)
{
	const unsigned strips = (unsigned)(4 * jobs[0].grid_x * jobs[0].grid_y);
	stage_mark("blend_backward", s);
	for (int at = 0; at < count; at += kMaxBlendBatch) {
		BlendBatch batch;
		batch.count = count - at < kMaxBlendBatch ? count - at : kMaxBlendBatch;
		for (int k = 0; k < batch.count; k++)
			batch.job[k] = jobs[at + k];
		batch.strips = strips;
		bool depth = false;  // does any job of the batch bring a gradient of the depth image?
		for (int k = 0; k < batch.count; k++)
			depth = depth || batch.job[k].dL_dpix_depth != nullptr;
		const unsigned jobs = (unsigned)batch.count;
		if ((size_t)strips * jobs <= kStripWorkgroups) {
			// (with more strips than that, few walks are long against the launch: 517 us for 1600x1036 and four submodels, 550 by this kernel)
			batch.workgroups = (strips + kSharedWaves - 1) / kSharedWaves + 1024u / jobs;
			const dim3 grid(batch.workgroups * jobs), threads(64 * kSharedWaves);
			if (depth)
				hipLaunchKernelGGL(blend_backward_shared_kernel<true>, grid, threads, 0, s, batch);
			else
				hipLaunchKernelGGL(blend_backward_shared_kernel<false>, grid, threads, 0, s, batch);
			continue;
		}
		batch.workgroups = blend_workgroups(strips, batch.count);
		const dim3 grid(batch.workgroups * jobs);
		if (depth)
			hipLaunchKernelGGL(blend_backward_kernel<true>, grid, dim3(64), 0, s, batch);
		else
			hipLaunchKernelGGL(blend_backward_kernel<false>, grid, dim3(64), 0, s, batch);
	}
}

}  // namespace rgs
