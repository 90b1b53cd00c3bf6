// Binning stages: offset scans, depth order of the Gaussians, tile-key duplication, stable
// radix sorts and per-tile range extraction.  All integer work; results are bit-exact by
// construction.  K = rasterization_kernels/diff-gaussian-rasterization-half-gaussian.
//
// The reference sorts R (Gaussian, tile) instances by the 64-bit key (tile << 32) | depth bits
// with a stable sort (K/cuda_rasterizer_hgs/rasterizer_impl.cu:300-317): 6 passes over 12-byte
// pairs at 6 500 tiles.  The same permutation is produced here in two cheaper steps:
//   1. the P Gaussians are sorted by their depth bits (stable, so equal depths stay in index
//      order), 4 passes over P 8-byte pairs;
//   2. instances are emitted in that order with the tile as a 32-bit key and sorted by it
//      (stable, so every tile keeps depth order, ties in index order), ceil(log2(tiles)/8)
//      passes over R 8-byte pairs.
// A stable sort by (tile, depth) of instances emitted in index order and a stable sort by tile
// of instances emitted in (depth, index) order give the same list: within a tile both order by
// depth and break ties by Gaussian index (a Gaussian touches a tile at most once).
#include "rgs_kernels.h"
#include "strip_filing.h"

#include <atomic>

namespace rgs {

// ---- prefix sums ---------------------------------------------------------------------------
// Replaces cub::DeviceScan::InclusiveSum at K/cuda_rasterizer_hgs/rasterizer_impl.cu:283
// with three small kernels: per-256 block totals, one single-block scan of those totals,
// and a per-block scan that adds the block's base.  On the rasterizer path the block totals
// come from the kernel that produces the values (the forward preprocess, the gather of the
// depth order), so only the last two run there.

// In all three kernels a non-null n_device overrides n (the launch is then sized for an upper bound).
__global__ __launch_bounds__(256) void block_totals_kernel(const uint32_t* __restrict__ in, size_t n,
                                                            const uint32_t* __restrict__ n_device,
                                                            uint32_t* __restrict__ totals)
{
	__shared__ uint32_t lds[8];
	if (n_device)
		n = *n_device;
	const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
	const uint32_t v = i < n ? in[i] : 0u;
	uint32_t total;
	(void)block256_exclusive_scan_u32(v, lds, total);
	if (threadIdx.x == 0)
		totals[blockIdx.x] = total;
}

// In-place exclusive scan of `data[0..n)` by one block of 1024 threads; the grand total goes
// to *total_out and *total_copy (if non-null).  Block 1, if launched, does the same for a second
// array of the same length.  blockIdx.y selects the job.
struct BlockScanJob {
	uint32_t* data;
	size_t n;
	const uint32_t* n_device;  // if non-null: the number of elements behind the entries, `per_entry` of them to an entry
	uint32_t per_entry;
	uint32_t* total_out;
	uint32_t* total_copy;
	uint32_t* data_b;
	uint32_t* total_out_b;
};

// Many elements, up to what fits, pass through LDS: read and written in lines, summed there by the thread whose elements they are.  (In
// memory a thread's elements lie apart from its neighbours', and each step of its run waits for 64 lines: 27 000 elements of each of
// four jobs 14.6 us, now 8.2; 21 000 at most of twelve 25.8 and 9.8; 5 500 5.5, and 6.4 by way of LDS.)
constexpr uint32_t kScanInLds = 32768, kScanFromLds = 8192;

__global__ __launch_bounds__(1024) void single_block_exclusive_scan_kernel(Batch<BlockScanJob> batch)
{
	__shared__ uint32_t wave_tot[16];
	__shared__ uint32_t s_data[kScanInLds];
	const BlockScanJob& j = batch.job[blockIdx.y];
	uint32_t* data = j.data;
	size_t n = j.n;
	const uint32_t* n_device = j.n_device;
	uint32_t* total_out = j.total_out;
	uint32_t* total_copy = j.total_copy;
	if (blockIdx.x == 1) {
		data = j.data_b;
		total_out = j.total_out_b;
		total_copy = nullptr;
	}
	if (!data)
		return;
	if (n_device)
		n = ((size_t)*n_device + j.per_entry - 1) / j.per_entry;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const bool in_lds = n >= kScanFromLds && n <= kScanInLds;
	const size_t chunk = ((n + 1023) / 1024) | 1;  // (odd: the threads' elements lie in different banks)
	const size_t lo = min((size_t)tid * chunk, n);
	const size_t hi = lo + chunk < n ? lo + chunk : n;
	uint32_t* from = data;
	if (in_lds) {
#pragma unroll 8
		for (uint32_t i = (uint32_t)tid; i < (uint32_t)n; i += 1024)
			s_data[i] = data[i];
		__syncthreads();
		from = s_data;
	}
	uint32_t sum = 0;
	for (size_t i = lo; i < hi; i++)
		sum += from[i];
	const uint32_t inc = wave_inclusive_scan_u32(sum);
	if (lane == 63)
		wave_tot[wave] = inc;
	__syncthreads();
	uint32_t base = 0, total = 0;
#pragma unroll
	for (int w = 0; w < 16; w++) {
		const uint32_t s = wave_tot[w];
		if (w < wave)
			base += s;
		total += s;
	}
	if (tid == 0 && total_copy)
		__hip_atomic_store(total_copy, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);  // (host memory: the host waits for this word)
	uint32_t run = base + inc - sum;
	for (size_t i = lo; i < hi; i++) {
		const uint32_t v = from[i];
		from[i] = run;
		run += v;
	}
	if (in_lds) {
		__syncthreads();
		for (uint32_t i = (uint32_t)tid; i < (uint32_t)n; i += 1024)
			data[i] = s_data[i];
	}
	if (tid == 0 && total_out)
		*total_out = total;
}

struct BlockInclusiveJob {
	const uint32_t* in;
	const uint32_t* block_base;
	size_t n;
	const uint32_t* n_device;
	uint32_t* out;
	uint32_t* first_of_block;  // may be null; see DuplicateJob
	uint32_t first_of_block_words;
	// non-zero: block_base holds the totals of the workgroups' elements, not yet scanned: a workgroup adds up those
	// ahead of its own itself (for a few thousand workgroups at most, which saves the launch that scans them)
	uint32_t base_from_totals;
};

// kPer consecutive elements per thread; with kPer = 4 `in` and `out` are 16-byte aligned and moved 16 bytes at a time.
constexpr int kScanGroup = 1024;  // elements per workgroup of the four-per-thread kernels of the depth order
template <int kPer>
__global__ __launch_bounds__(256) void block_inclusive_scan_kernel(Batch<BlockInclusiveJob> batch)
{
	__shared__ uint32_t lds[8];
	constexpr size_t kGroup = 256 * (size_t)kPer;
	const BlockInclusiveJob& j = batch.job[blockIdx.y];
	const uint32_t* __restrict__ in = j.in;
	const uint32_t* __restrict__ block_base = j.block_base;
	uint32_t* __restrict__ out = j.out;
	size_t n = j.n;
	if (j.n_device)
		n = *j.n_device;
	if ((size_t)blockIdx.x * kGroup >= n)
		return;
	const size_t i0 = (size_t)blockIdx.x * kGroup + (size_t)kPer * threadIdx.x;
	uint32_t v[kPer];
	const bool whole = i0 + kPer <= n;
	bool loaded = false;
	if constexpr (kPer == 4) {
		if (whole) {
			const uint4 v4 = *reinterpret_cast<const uint4*>(in + i0);
			v[0] = v4.x; v[1] = v4.y; v[2] = v4.z; v[3] = v4.w;
			loaded = true;
		}
	}
	if (!loaded) {
#pragma unroll
		for (int q = 0; q < kPer; q++)
			v[q] = i0 + q < n ? in[i0 + q] : 0u;
	}
	uint32_t sum = 0;
#pragma unroll
	for (int q = 0; q < kPer; q++)
		sum += v[q];
	uint32_t total;
	uint32_t base = 0;
	if (j.base_from_totals) {
		uint32_t ahead = 0;
		for (uint32_t b = threadIdx.x; b < blockIdx.x; b += 256)
			ahead += block_base[b];
		(void)block256_exclusive_scan_u32(ahead, lds, base);
	} else {
		base = block_base[blockIdx.x];
	}
	uint32_t run = base + block256_exclusive_scan_u32(sum, lds, total);
	uint32_t end[kPer];
#pragma unroll
	for (int q = 0; q < kPer; q++) {
		const uint32_t begin = run;
		run += v[q];
		end[q] = run;
		if (j.first_of_block && i0 + q < n) {
			// element i covers positions [begin, end): it is where every workgroup of the key duplication starts whose
			// first position, a multiple of kDupPositions, lies among them
			for (uint32_t b = (begin + (uint32_t)kDupPositions - 1u) / (uint32_t)kDupPositions;
			     b < j.first_of_block_words && (uint64_t)b * (uint64_t)kDupPositions < (uint64_t)run; b++)
				j.first_of_block[b] = (uint32_t)(i0 + q);
		}
	}
	bool stored = false;
	if constexpr (kPer == 4) {
		if (whole) {
			*reinterpret_cast<uint4*>(out + i0) = uint4{end[0], end[1], end[2], end[3]};
			stored = true;
		}
	}
	if (!stored) {
#pragma unroll
		for (int q = 0; q < kPer; q++)
			if (i0 + q < n)
				out[i0 + q] = end[q];
	}
}

size_t scan_temp_words(size_t n)
{
	return (n + 255) / 256 + 1;
}

static void inclusive_sum(const uint32_t* in, uint32_t* out, size_t n, const uint32_t* n_device, uint32_t* temp,
                          hipStream_t s)
{
	const size_t nb = (n + 255) / 256;
	hipLaunchKernelGGL(block_totals_kernel, dim3((unsigned)nb), dim3(256), 0, s, in, n, n_device, temp);
	Batch<BlockScanJob> scan = {};
	scan.job[0] = BlockScanJob{temp, nb, n_device, 256u, nullptr, nullptr, nullptr, nullptr};
	hipLaunchKernelGGL(single_block_exclusive_scan_kernel, dim3(1), dim3(1024), 0, s, scan);
	Batch<BlockInclusiveJob> inc = {};
	inc.job[0] = BlockInclusiveJob{in, temp, n, n_device, out, nullptr, 0u, 0u};
	hipLaunchKernelGGL(block_inclusive_scan_kernel<1>, dim3((unsigned)nb), dim3(256), 0, s, inc);
}

void launch_inclusive_sum(const uint32_t* in, uint32_t* out, size_t n, uint32_t* temp, const char* stage,
                          hipStream_t s)
{
	if (n == 0)
		return;
	if (stage)
		stage_mark(stage, s);
	inclusive_sum(in, out, n, nullptr, temp, s);
}

void launch_totals_from_block_sums(const TotalsJob* jobs, int count, hipStream_t s)
{
	stage_mark("offset_scan", s);
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<BlockScanJob> b = {};
		for (int k = 0; k < nj; k++) {
			const TotalsJob& t = jobs[at + k];
			b.job[k] = BlockScanJob{t.block_sums, ((size_t)t.P + 255) / 256, nullptr, 256u, t.total_out, t.total_copy, t.block_visible,
			                        t.visible_count};
		}
		hipLaunchKernelGGL(single_block_exclusive_scan_kernel, dim3(2, (unsigned)nj), dim3(1024), 0, s, b);
	}
}

// ---- depth order and key duplication (K/cuda_rasterizer_hgs/rasterizer_impl.cu:70-111) -------

// Keys of the depth sort.  A rendered Gaussian's depth exceeds 0.2, so its bit pattern, which orders like the value,
// lies above that of 0.125: the sort looks at bits - kDepthKeyBase, whose low kDepthKeyBits bits (three 9-bit digits)
// tell every depth below 8192 apart.  Should a key have bits above those (a depth of 8192 or more), the kernel that
// writes the keys says so in the sort's scratch and a fourth pass over the remaining bits runs; otherwise that pass
// returns at once.  Either way the order is that of the full 32 bits.
constexpr uint32_t kDepthKeyBase = 0x3E000000u;
constexpr int kDepthKeyBits = 27;
constexpr int kDepthPasses = 3;                 // of 9 bits each, plus the one on demand
constexpr uint32_t kSortExtraPass = 2057;       // word of the sort scratch's header: non-zero = the fourth pass is needed

// The values of the depth sort carry the Gaussian's tile count above its index, so that the pass that ends the sort
// can write the counts in depth order itself (a gather of its own over the sorted indices cost as much as a pass).
// A count that does not fit is stored as all ones and looked up by that pass.
__host__ __device__ inline uint32_t depth_index_bits(uint32_t P)
{
	uint32_t bits = 1;
	while (bits < 31u && (P - 1u) >> bits)
		bits++;
	return bits;
}

// (depth key, index and tile count) pairs of the Gaussians that touch a tile, compacted in index order: the
// group of Gaussians [kScanGroup b, kScanGroup (b + 1)), four neighbouring ones per thread, is written
// from visible_base[4 b] on (the bases are per 256 Gaussians).  A workgroup takes every gridDim.x-th group and
// counts the digits of the keys it writes on the way: at the end it adds its counts to a copy of the digit counts
// the sort of these pairs starts from (see kDigitCopies; cleared beforehand), which saves that sort its own pass over the keys.
__global__ __launch_bounds__(256) void depth_pairs_kernel(Batch<DepthOrderJob> batch)
{
	__shared__ uint32_t lds[8];
	__shared__ uint32_t s_hist[kDepthPasses][512];
	__shared__ uint32_t s_top[32];   // digit of the pass on demand; value 0 is not counted here but derived
	const DepthOrderJob& j = batch.job[blockIdx.y];
	const size_t P = (size_t)j.P;
	if ((size_t)blockIdx.x * kScanGroup >= P)
		return;
	const float* __restrict__ depths = j.depths;
	const uint32_t* __restrict__ tiles_touched = j.tiles_touched;
	const uint32_t* __restrict__ visible_base = j.block_visible;
	uint32_t* __restrict__ keys = j.keys_a;
	uint32_t* __restrict__ values = j.vals_a;
	const uint32_t index_bits = depth_index_bits((uint32_t)j.P), cap = 0xFFFFFFFFu >> index_bits;
#pragma unroll
	for (int p = 0; p < kDepthPasses; p++) {
		s_hist[p][threadIdx.x] = 0u;
		s_hist[p][256 + threadIdx.x] = 0u;
	}
	if (threadIdx.x < 32)
		s_top[threadIdx.x] = 0u;
	__syncthreads();
	uint32_t written = 0;
	// How many of a group's Gaussians are listed is known ahead of it.  Where neighbours in memory are neighbours in the scene most
	// groups have none (a city stored along a space-filling curve, 5 % in view: 39.5 -> 29 us; 62.9 M Gaussians in random order
	// 124 -> 101; both before the digit counts had copies), so a workgroup with many groups looks for those that have some, 64 at a
	// time; one with few would only wait for the answer.
	const size_t blocks = (P + 255) / 256, groups = (P + kScanGroup - 1) / kScanGroup;
	const bool many = groups > 4 * (size_t)gridDim.x;
	auto listed_up_to = [&](size_t group) { return 4 * group < blocks ? visible_base[4 * group] : *j.visible_count; };
	for (size_t ahead = blockIdx.x; ahead < groups; ahead += 64 * (size_t)gridDim.x) {
		const size_t looked_at = ahead + (size_t)(threadIdx.x & 63) * gridDim.x;
		uint32_t base = 0u;
		bool some = looked_at < groups;
		if (some) {
			base = listed_up_to(looked_at);
			if (many)
				some = base != listed_up_to(looked_at + 1);
		}
		for (uint64_t todo = lanes_where(some); todo != 0ull; todo &= todo - 1ull) {  // (the same in every wavefront of the workgroup)
			const int which = __builtin_ctzll(todo);
			const size_t group = ahead + (size_t)which * gridDim.x;
			const size_t idx0 = group * kScanGroup + 4 * (size_t)threadIdx.x;
			// the depth of a Gaussian that touches no tile is stored as 0, that of one that does exceeds 0.2: the
			// depths alone say which ones are listed
			float depth[4] = {0.f, 0.f, 0.f, 0.f};
			uint32_t count[4] = {0u, 0u, 0u, 0u};
			if (idx0 + 4 <= P) {
				const float4 d4 = *reinterpret_cast<const float4*>(depths + idx0);
				const uint4 c4 = *reinterpret_cast<const uint4*>(tiles_touched + idx0);
				depth[0] = d4.x; depth[1] = d4.y; depth[2] = d4.z; depth[3] = d4.w;
				count[0] = c4.x; count[1] = c4.y; count[2] = c4.z; count[3] = c4.w;
			} else {
#pragma unroll
				for (int q = 0; q < 4; q++)
					if (idx0 + q < P) {
						depth[q] = depths[idx0 + q];
						count[q] = tiles_touched[idx0 + q];
					}
			}
			uint32_t mine = 0;
#pragma unroll
			for (int q = 0; q < 4; q++)
				mine += __float_as_uint(depth[q]) != 0u ? 1u : 0u;
			uint32_t total;
			uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)base, which) + block256_exclusive_scan_u32(mine, lds, total);
			written += mine;
#pragma unroll
			for (int q = 0; q < 4; q++)
				if (__float_as_uint(depth[q]) != 0u) {
					const uint32_t key = __float_as_uint(depth[q]) - kDepthKeyBase;
					keys[at] = key;
					values[at] = (uint32_t)(idx0 + q) | (min(count[q], cap) << index_bits);
					at++;
#pragma unroll
					for (int p = 0; p < kDepthPasses; p++)
						atomicAdd(&s_hist[p][(key >> (9 * p)) & 511u], 1u);
					if (key >> kDepthKeyBits)
						atomicAdd(&s_top[key >> kDepthKeyBits], 1u);
				}
		}
	}
	__syncthreads();
	uint32_t* digits = j.digits + (blockIdx.x & (j.digit_copies - 1u)) * kDigitWords;
#pragma unroll
	for (int p = 0; p < kDepthPasses; p++)
#pragma unroll
		for (int h = 0; h < 2; h++) {
			const uint32_t c = s_hist[p][256 * h + threadIdx.x];
			if (c)
				atomicAdd(&digits[512 * p + 256 * h + threadIdx.x], c);
		}
	// the digit of the pass on demand: value 0 takes every key that was not counted under another value
	uint32_t all_written;
	(void)block256_exclusive_scan_u32(written, lds, all_written);
	if (threadIdx.x < 32) {
		uint32_t c = s_top[threadIdx.x];
		if (threadIdx.x == 0) {
			uint32_t others = 0;
			for (int v = 1; v < 32; v++)
				others += s_top[v];
			c = all_written - others;
			if (others)
				atomicOr(&j.sort_temp[kSortExtraPass], 1u);
		}
		if (c)
			atomicAdd(&digits[512 * kDepthPasses + threadIdx.x], c);
	}
}

// The sum of every kScanGroup of the tile counts in depth order (the first level of the scan that follows), a wavefront per group, without
// a barrier; the count of them is on the device.  The wavefronts that are resident together take all groups: with a workgroup per group
// most had none (62.9 M Gaussians, a third listed: 28 -> 13 us).
__global__ __launch_bounds__(256) void order_totals_kernel(Batch<DepthOrderJob> batch)
{
	static_assert(kScanGroup == 1024, "16 counts per lane");
	const DepthOrderJob& j = batch.job[blockIdx.y];
	// what the key duplication will count the digits of its tiles into
	for (int w = (int)(blockIdx.x * 256 + threadIdx.x); w < (int)j.digit_copies * kDigitWords / 4; w += (int)gridDim.x * 256)
		reinterpret_cast<uint4*>(j.digits)[w] = uint4{0u, 0u, 0u, 0u};
	const size_t n = min((size_t)*j.visible_count, (size_t)j.P);
	const uint32_t* __restrict__ in = j.tiles_in_order;
	const int lane = threadIdx.x & 63;
	for (size_t group = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6); group * kScanGroup < n; group += (size_t)gridDim.x * 4) {
		const size_t k0 = group * kScanGroup + 4 * (size_t)lane;
		uint4 v[4];
#pragma unroll
		for (int q = 0; q < 4; q++)
			v[q] = k0 + 256 * q + 4 <= n ? *reinterpret_cast<const uint4*>(in + k0 + 256 * q) : uint4{0u, 0u, 0u, 0u};
		uint32_t sum = 0;
#pragma unroll
		for (int q = 0; q < 4; q++)
			sum += v[q].x + v[q].y + v[q].z + v[q].w;
		// the lane that holds the last counts, up to three of them
		if (n - group * kScanGroup < kScanGroup && n > (n & ~(size_t)3) && (size_t)lane == (n >> 2 & 63))
			for (size_t k = n & ~(size_t)3; k < n; k++)
				sum += in[k];
		sum = wave_inclusive_scan_u32(sum);
		if (lane == 63)
			j.scan_temp[group] = sum;
	}
}

// Instances of the Gaussians in depth order, tiles row by row like the reference, at the offsets
// of the scan taken in that same order.  The work is dealt out by output position, not by Gaussian:
// a workgroup writes runs of kDupPositions consecutive instances, whichever Gaussians they belong to (one
// that covers thousands of tiles is shared by several runs, a thousand that cover one tile
// each are taken by one).  It takes the first Gaussian of a run from the table the offset scan has filled
// (beyond that table, from a 64-ary search over the inclusive offsets), stages the offsets and indices of
// the Gaussians of the run in LDS 256 at a time
// and lets every thread find the Gaussian of its output position by how many of those 256 have begun
// up to it, read that Gaussian's 64-byte record, and take the tile from the position inside the
// record's rectangle; stores are contiguous.  The thread also decides which of the
// tile's four strips the instance can matter to (strip_filing.h) and puts those bits above the
// tile in the key: the sort only looks at the tile bits, so they travel with the instance for free.
// On the way the workgroup counts the digits of the tiles it writes (what the sort's passes start from:
// the sort then has no pass of its own over the keys) and it clears the sort's scratch and the tile ranges.
// `order` is the output of a sort: should that sort ever have given up, its entries may be anything, so
// they are clamped to the P Gaussians there are (the tile ranges then stay empty and nothing reads the result).
struct DuplicateStage {
	uint32_t end[256];     // inclusive offset of each staged Gaussian
	uint32_t index[256];
	__align__(16) uint32_t begins[2][8];  // bit per position of a run: a staged Gaussian's instances begin there (two: one is cleared while the other is read)
};

// Floats of LDS for the NDC tables of a grid of tiles: one per tile column, one per tile row.
static inline size_t ndc_table_floats(int gx, int gy)
{
	return (size_t)gx + (size_t)gy;
}
constexpr size_t kNdcTableMaxFloats = 8192;  // larger grids compute the coordinates per instance

__global__ __launch_bounds__(256) void duplicate_with_keys_kernel(Batch<DuplicateJob> batch, int gx, int gy, int ndc_in_lds)
{
	__shared__ DuplicateStage st;
	__shared__ uint32_t s_first;
	constexpr int kTileDigitWords = 4 * 512;  // one digit of up to 11 bits, or up to three of 9 (tiles have at most 24 bits)
	__shared__ uint32_t s_digits[kTileDigitWords];  // digit counts of the tiles this workgroup writes
	extern __shared__ __align__(16) float s_ndc[];  // NDC of the middle of every tile column, then of every tile row
	const DuplicateJob& job = batch.job[blockIdx.y];
	const uint32_t P = (uint32_t)job.P;
	const uint32_t* __restrict__ visible_count = job.visible_count;
	const uint32_t* __restrict__ order = job.order;
	const uint32_t* __restrict__ offsets = job.offsets;
	const FilingArgs& filing = job.filing;
	uint32_t* __restrict__ keys = job.keys;
	uint32_t* __restrict__ values = job.values;
	const uint32_t capacity = job.capacity;
	uint32_t* __restrict__ clear = job.clear;
	const size_t clear_words = job.clear_words;
	const int tid = threadIdx.x, lane = tid & 63;
	// the scratch of the sort that follows is cleared here, which saves a launch
	for (size_t w = (size_t)blockIdx.x * 256 + tid; w < clear_words; w += (size_t)gridDim.x * 256)
		clear[w] = 0u;
	for (size_t w = (size_t)blockIdx.x * 256 + tid; w < job.also_clear_words; w += (size_t)gridDim.x * 256)
		job.also_clear[w] = 0u;
	const uint32_t n = min(*visible_count, P);
	const uint32_t total = *job.total;
	if (n == 0u)
		return;
	const uint32_t limit = min(total, capacity);  // positions beyond the room the caller gave are dropped
	if (blockIdx.x * (uint32_t)kDupPositions >= limit)
		return;
	const int digit_bits = sort_max_digit_bits_u32(job.end_bit);
	const int passes = sort_passes(job.end_bit, digit_bits);
	for (int w = tid; w < kTileDigitWords; w += 256)
		s_digits[w] = 0u;
	if (tid < 16)
		st.begins[tid >> 3][tid & 7] = 0u;
	int which = 0;

	if (ndc_in_lds) {
		for (int c = tid; c < gx; c += 256)
			s_ndc[c] = tile_middle_ndc(c, filing.W);
		for (int r = tid; r < gy; r += 256)
			s_ndc[gx + r] = tile_middle_ndc(r, filing.H);
	}
	const NdcSteps steps = ndc_steps(filing.W, filing.H);
	const BoxFrame box = load_box_frame(filing.projinv, filing.range_low, filing.range_up, filing.tanfovx, filing.tanfovy);

	// A workgroup takes every gridDim.x-th run of kDupPositions positions: the tables above are set up once, and the
	// digit counts of many runs leave with one atomic add per digit.  What a run needs first (the Gaussian its
	// positions begin at, from the table the offset scan has filled, and the offsets and indices of the 256 Gaussians
	// from there on: a run of 256 positions cannot span more, every listed Gaussian having an instance) is asked for
	// one run ahead, so that these two dependent reads are under way while the previous run is worked on.
	const uint32_t table_runs = (uint32_t)dup_first_words((size_t)P);
	uint32_t ahead_end = 0, ahead_index = 0, ahead_begin = 0;
	bool ahead = false;  // the same for every thread of the workgroup
	auto ask_for = [&](uint32_t r) {
		const uint32_t f = min(job.first_of_block[r], n - 1u);
		const uint32_t g = f + (uint32_t)tid;
		ahead_end = g < n ? offsets[g] : total;
		ahead_index = g < n ? min(order[g], P - 1u) : 0u;
		ahead_begin = f == 0u ? 0u : offsets[f - 1];
		ahead = true;
	};
	if (blockIdx.x < table_runs)
		ask_for(blockIdx.x);
	for (uint32_t run = blockIdx.x; (uint64_t)run * kDupPositions < (uint64_t)limit; run += gridDim.x) {
		const uint32_t start = run * (uint32_t)kDupPositions;
		const uint32_t stop = min(start + (uint32_t)kDupPositions, limit);
		__syncthreads();  // the previous run is done with s_first and the staged Gaussians; the tables are written
		uint32_t staged_begin, own_end;
		if (ahead) {
			own_end = ahead_end;
			st.index[tid] = ahead_index;
			staged_begin = ahead_begin;
		} else {
			// beyond the table (more than 16 instances per Gaussian on average): the first Gaussian whose inclusive offset
			// exceeds `start` by a 64-ary search of the first wavefront
			if (tid < 64) {
				uint32_t lo = 0, hi = n;  // the answer lies in [lo, hi]
				while (lo < hi) {
					const uint32_t step = (hi - lo + 63u) / 64u;
					const uint32_t probe = lo + (uint32_t)lane * step;
					const bool below = probe < hi && offsets[probe] <= start;
					const uint32_t c = (uint32_t)__popcll(lanes_where(below));  // the predicate is monotone: the first c probes hold
					if (c == 0u) {
						hi = lo;
					} else {
						const uint32_t last_true = lo + (c - 1u) * step;
						lo = last_true + 1u;
						hi = min(last_true + step, hi);
					}
				}
				if (lane == 0)
					s_first = min(lo, n - 1u);
			}
			__syncthreads();
			const uint32_t g0 = s_first, g = g0 + (uint32_t)tid;
			own_end = g < n ? offsets[g] : total;
			st.index[tid] = g < n ? min(order[g], P - 1u) : 0u;
			staged_begin = g0 == 0u ? 0u : offsets[g0 - 1];
		}
		st.end[tid] = own_end;
		const uint32_t next_begins = own_end - start;
		if (next_begins - 1u < 255u)
			atomicOr(&st.begins[which][next_begins >> 5], 1u << (next_begins & 31u));
		__syncthreads();
		ahead = false;
		if (tid < 8)
			st.begins[which ^ 1][tid] = 0u;
		if ((uint64_t)(run + gridDim.x) * kDupPositions < (uint64_t)limit && run + gridDim.x < table_runs)
			ask_for(run + gridDim.x);

		{
			const uint32_t staged_end = st.end[255];
			const uint32_t from = max(start, staged_begin), to = min(stop, staged_end);
			// Up to kDupPositions / 256 positions per thread.  First all of them find their Gaussian and ask for its
			// record (pixel centre, conic, extents, radius: everything else follows from those), then each is finished:
			// the records of a thread arrive together, not one wait after another.
			constexpr int kPerThread = kDupPositions / 256;
			static_assert(kPerThread == 1, "a bit per thread");
			// The staged Gaussian of a position: as many as have begun up to it since the run's first (every listed one has an instance).
			// One read of the bits and a count where a binary search took eight reads in LDS, each after the one before: 611 -> 587 us for
			// 62.9 M Gaussians, where most have an instance or two; nothing where they have many.
			const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
			uint32_t begun = 0, own_lo = 0, own_hi = 0;
			{
				const uint4 m0 = *reinterpret_cast<const uint4*>(&st.begins[which][0]), m1 = *reinterpret_cast<const uint4*>(&st.begins[which][4]);
				const uint32_t m[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
				which ^= 1;
#pragma unroll
				for (int w = 0; w < 4; w++) {
					const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)m[2 * w]), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)m[2 * w + 1]);
					begun += w < wave ? (uint32_t)(__popc(lo) + __popc(hi)) : 0u;
					own_lo = w == wave ? lo : own_lo;
					own_hi = w == wave ? hi : own_hi;
				}
				// (a lane counts the bits below its own: its own bit is shifted down to be one of them)
				begun += own_lo & 1u;
				own_lo = own_lo >> 1 | own_hi << 31;
				own_hi >>= 1;
			}
			uint32_t first[kPerThread], index[kPerThread];
			float4 r0[kPerThread], r1[kPerThread], r3[kPerThread];
#pragma unroll
			for (int q = 0; q < kPerThread; q++) {
				const uint32_t pos = from + (uint32_t)tid + 256u * (uint32_t)q;
				first[q] = 0u;
				index[q] = 0u;
				if (pos < to) {
					const int lo = (int)(begun + __builtin_amdgcn_mbcnt_hi(own_hi, __builtin_amdgcn_mbcnt_lo(own_lo, 0u)));
					first[q] = lo == 0 ? staged_begin : min(st.end[lo - 1], pos);
					index[q] = st.index[lo];
					const float4* rec = filing.record + 4 * (size_t)index[q];
					r0[q] = rec[0];
					r1[q] = rec[1];
					r3[q] = rec[3];
				}
			}
			uint32_t tile_of[kPerThread];
#pragma unroll
			for (int q = 0; q < kPerThread; q++) {
				const uint32_t pos = from + (uint32_t)tid + 256u * (uint32_t)q;
				tile_of[q] = 0xFFFFFFFFu;
				if (pos >= to)
					continue;
				const TileRect rc = tile_rect(r0[q].x, r0[q].y, __float_as_int(r3[q].z), gx, gy);
				const uint32_t t = pos - first[q], w = max(rc.x1 - rc.x0, 1u);
				// t / w through the reciprocal in single precision (both are below 2^24, so exact as floats; the quotient
				// is off by one at most, which the remainder shows): a third of the instructions of the integer division
				uint32_t row = (uint32_t)((float)t * __builtin_amdgcn_rcpf((float)w));
				int col = (int)(t - __umul24(row, w));
				if (col < 0) {
					row--;
					col += (int)w;
				} else if (col >= (int)w) {
					row++;
					col -= (int)w;
				}
				const int tx = (int)rc.x0 + col, ty = (int)(rc.y0 + row);
				const uint32_t tile = (uint32_t)ty * (uint32_t)gx + (uint32_t)tx;
				float nx, ny;
				if (ndc_in_lds) {
					nx = s_ndc[tx];
					ny = s_ndc[gx + ty];
				} else {
					nx = tile_middle_ndc(tx, filing.W);
					ny = tile_middle_ndc(ty, filing.H);
				}
				const StripTests tests = prepare_strip_tests(FiledGeometry{r0[q], r1[q], float2{r3[q].x, r3[q].y}}, box);
				const uint32_t strips = strips_filed_for(tests, (float)(tx * kTile), (float)(ty * kTile), nx, ny, steps, box);
				keys[pos] = tile | (strips << kKeyTileBits);
				values[pos] = index[q];
				tile_of[q] = tile;
			}
			// the digits of the tiles just written, for the sort (every lane comes here: the narrow digits are counted by ballot)
#pragma unroll
			for (int q = 0; q < kPerThread; q++) {
				const bool have = tile_of[q] != 0xFFFFFFFFu;
				for (int p = 0; p < passes; p++) {
					const int shift = sort_digit_shift(job.end_bit, p, digit_bits);
					const int bits = sort_digit_bits(job.end_bit, p, digit_bits);
					const uint32_t d = (tile_of[q] >> shift) & ((1u << bits) - 1u);
					if (bits <= 2) {
						// a digit of one or two bits: every lane would add to one of a few words, one after the other
						for (uint32_t v = 0; v < (1u << bits); v++) {
							const uint32_t c = (uint32_t)__popcll(lanes_where(have && d == v));
							if (lane == 0 && c != 0u)
								atomicAdd(&s_digits[512 * p + v], c);
						}
					} else if (have) {
						atomicAdd(&s_digits[512 * p + d], 1u);
					}
				}
			}
		}
	}
	__syncthreads();
	for (int w = tid; w < (passes == 1 ? 1 << job.end_bit : 512 * passes); w += 256) {
		const uint32_t c = s_digits[w];
		if (c)
			atomicAdd(&job.tile_digits[(blockIdx.x & (job.digit_copies - 1u)) * kDigitWords + w], c);
	}
}

void launch_duplicate_with_keys(const DuplicateJob* jobs, int count, int grid_x, int grid_y, hipStream_t s)
{
	stage_mark("duplicate_with_keys", s);
	const size_t table = ndc_table_floats(grid_x, grid_y);
	const int ndc_in_lds = table <= kNdcTableMaxFloats ? 1 : 0;
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<DuplicateJob> b = {};
		size_t blocks = 1;
		for (int k = 0; k < nj; k++) {
			b.job[k] = jobs[at + k];
			// sized for the positions there is room for; at least enough workgroups to clear the sort's scratch at a decent rate
			const size_t need = max((size_t)(b.job[k].capacity + kDupPositions - 1) / kDupPositions,
			                        min((b.job[k].clear_words + 4095) / 4096, (size_t)1024));
			blocks = need > blocks ? need : blocks;
		}
		// every workgroup ends with an atomic add per digit into its job's counts: enough of them to fill the GPU several
		// times over, each over many runs of positions, rather than one per run.  (Half and twice as many: 16.6 and 14.9 us for 12.4 at
		// 100 000 Gaussians, 44 and 50 for 45 in the city, 691 and 595 for 610 in the scene of 62.9 M.)
		const size_t most = nj >= 8 ? 512 : nj >= 4 ? 4096 / (size_t)nj : 1024;
		blocks = blocks < most ? blocks : most;
		hipLaunchKernelGGL(duplicate_with_keys_kernel, dim3((unsigned)blocks, (unsigned)nj), dim3(256),
		                   ndc_in_lds ? table * sizeof(float) : 0, s, b, grid_x, grid_y, ndc_in_lds);
	}
}

// ---- radix sort -------------------------------------------------------------------------------
// Replaces cub::DeviceRadixSort::SortPairs at K/cuda_rasterizer_hgs/rasterizer_impl.cu:312-317:
// a stable least-significant-digit sort of (key, u32 value) pairs on key bits [0, end_bit), in the one-sweep form:
// the digit histogram of every pass is built while the keys are written (or, for the stand-alone entry points, by one
// kernel that reads them once), then each pass is a single kernel whose blocks take tiles of
// kSortThreads * kItems pairs in arrival order, rank them in LDS, obtain their global digit offsets from
// the blocks before them through a chained look-back over per-tile status words, and scatter.
// Element order inside a tile is (wave, round, lane); ranking preserves it, and tiles are
// ordered by their id, so every pass is stable.  A digit has up to kBits bits (template parameter): 7 to 11 for 32-bit
// keys (sort_max_digit_bits_u32), 8 for 64-bit keys, whose tiles of pairs fill the LDS.
//
// Scratch layout (u32 words), B = 2^kBits:
//   [0, 2048)      digit histograms, B words per pass, where the job names no digit_counts (every block of a pass scans its counts itself)
//   [2048, 2056)   tile counter of each pass
//   [2056]         status: non-zero if a look-back ever gave up waiting (never expected)
//   [2057]         depth sort only: non-zero if its pass on demand is needed (kSortExtraPass)
//   [kSortHeader + pass * B * tiles + tile * B + digit]  look-back words

constexpr uint32_t kSortCounters = 2048;
constexpr uint32_t kSortStatus = 2056;
constexpr uint32_t kFlagAggregate = 1u << 30;  // word holds this tile's own digit count
constexpr uint32_t kFlagInclusive = 2u << 30;  // word holds the count of this and all earlier tiles
constexpr uint32_t kValueMask = (1u << 30) - 1u;
constexpr int kLookbackSpinLimit = 1 << 18;
constexpr int kLookBatch = 4;  // earlier tiles a look-back reads at once (1, 2 and 8 to 32 were measured slower)

// How many times a look-back polls a word that has not been published yet before it gives up.
// A negative value makes every look-back give up at once: the way a test drives the give-up
// path from the host (every kernel still runs to its end).
static std::atomic<int> g_lookback_spin_limit{kLookbackSpinLimit};

void set_lookback_spin_limit(int polls)
{
	g_lookback_spin_limit.store(polls == 0 ? kLookbackSpinLimit : polls);
}

template <typename KeyT>
__device__ __forceinline__ uint32_t digit_of(KeyT key, int shift, uint32_t mask)
{
	return (uint32_t)(key >> shift) & mask;
}

// Only the stand-alone sort entry points run this (64-bit keys, digits of kDigitBitsU64 bits).
template <typename KeyT>
__global__ __launch_bounds__(256) void sort_digit_histogram_kernel(Batch<SortJob<KeyT>> batch, int passes, int end_bit)
{
	constexpr int kMaxPasses = 8;
	__shared__ uint32_t s_hist[kMaxPasses][256];
	const SortJob<KeyT>& j = batch.job[blockIdx.y];
	const KeyT* __restrict__ keys = j.keys_in;
	size_t n = j.n;
	const uint32_t* __restrict__ n_device = j.n_device;
	uint32_t* __restrict__ hist = j.temp;
	uint32_t* __restrict__ clear = j.also_clear;
	const size_t clear_words = j.also_clear_words;
	for (size_t w = (size_t)blockIdx.x * 256 + threadIdx.x; w < clear_words; w += (size_t)gridDim.x * 256)
		clear[w] = 0u;  // an array that a later kernel of the same stream wants cleared
	if (n_device)
		n = min(n, (size_t)*n_device);
#pragma unroll
	for (int p = 0; p < kMaxPasses; p++)
		s_hist[p][threadIdx.x] = 0;
	__syncthreads();
	// four keys per thread and round, requested together: one key at a time the loop waits for
	// memory once per key and the kernel takes as long as a pass of the sort
	const size_t threads = (size_t)gridDim.x * 256;
	for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < n; k += 4 * threads) {
		KeyT key[4];
#pragma unroll
		for (int q = 0; q < 4; q++)
			key[q] = k + q * threads < n ? keys[k + q * threads] : (KeyT)0;
#pragma unroll
		for (int q = 0; q < 4; q++) {
			if (k + q * threads >= n)
				break;
			for (int p = 0; p < passes; p++) {
				const int shift = sort_digit_shift(end_bit, p, kDigitBitsU64);
				const int bits = sort_digit_bits(end_bit, p, kDigitBitsU64);
				const uint32_t d = digit_of(key[q], shift, (1u << bits) - 1u);
				if (bits <= 2) {
					// a digit of one or two bits: every lane would add to one of a few words, one after the
					// other; count the lanes of each value instead
					for (uint32_t v = 0; v < (1u << bits); v++) {
						const uint32_t c = (uint32_t)__popcll(lanes_where(d == v));
						if ((threadIdx.x & 63) == 0 && c != 0u)
							atomicAdd(&s_hist[p][v], c);
					}
				} else {
					atomicAdd(&s_hist[p][d], 1u);
				}
			}
		}
	}
	__syncthreads();
	for (int p = 0; p < passes; p++) {
		const uint32_t c = s_hist[p][threadIdx.x];
		if (c)
			atomicAdd(&hist[p * 256 + threadIdx.x], c);
	}
}

// What a pass does with its output:
//   kPassPlain        keys and values to the other buffer pair;
//   kPassEndsUnless   depth sort, third pass: if the scratch says that a fourth pass is needed, as kPassPlain; otherwise the
//                     sort ends here and the values are taken apart (Gaussian index to final_index, its tile count to
//                     final_count, see SortJob);
//   kPassOnDemand     depth sort, fourth pass: returns at once unless the scratch says it is needed; ends the sort.
enum SortPassKind { kPassPlain = 0, kPassEndsUnless = 1, kPassOnDemand = 2 };

// Per-wave digit counts fit 16 bits (a wavefront ranks kSortItems * 64 keys), and so does a digit's place inside a tile.
template <int kBits>
struct SortCounts {
	uint16_t digit_base[1 << kBits];                  // exclusive prefix over digits within the tile
	__align__(8) uint32_t global_base[1 << kBits];    // where this tile's run of each digit starts globally
};

// How many wavefronts stand by to fill the gaps of the others' phases (loads, ranking, look-back, stores) and how long the runs are
// that a tile writes set the pace of a pass: sixteen wavefronts per tile, 32 per CU with up to eight pairs per lane (64
// registers; the counts of the ranking lie where the tile's keys go afterwards), 16 with sixteen.  A lane keeps three registers per pair
// from phase to phase (key, value, rank): with the parts of the ranks and the digits' addresses kept too, eight pairs per lane spilled
// to memory, ahead of the ranking, and sixteen took 119 registers instead of 89 (per pass, us: instances of two submodels of 2.8 M
// 64 -> 58, of two at 5185x3359 378 -> 328, of one of 2.8 M in training 45 -> 42, its depths 20 -> 17).
template <typename KeyT, int kBits, int kKind, int kItems>
__global__ __launch_bounds__(kSortThreads) __attribute__((amdgpu_waves_per_eu(sizeof(KeyT) == 4 && kItems <= 8 && kBits <= 10 ? 8 : 4))) void sort_onesweep_kernel(
	Batch<SortJob<KeyT>> batch, int pass, int shift, uint32_t mask, int spin_limit)
{
	constexpr int kBins = 1 << kBits;
	constexpr int kWaves = kSortThreads / 64, kBlock = kSortThreads * kItems;
	// A thread owns one digit value, or two neighbouring ones whose counts and look-back words it handles as halves of one number.
	constexpr int kOwn = kBins > kSortThreads ? 2 : 1;
	static_assert(kBins <= 2 * kSortThreads, "a thread owns at most two digit values");
	typedef std::conditional_t<kOwn == 2, uint64_t, uint32_t> Word;
	constexpr Word kBoth = kOwn == 2 ? (Word)0x100000001ull : (Word)1u;
	constexpr Word kAggregates = kFlagAggregate * kBoth, kInclusives = kFlagInclusive * kBoth, kValues = kValueMask * kBoth;
	const SortJob<KeyT>& j = batch.job[blockIdx.y];
	// the passes ping-pong between the two buffer pairs, starting in -> out
	const KeyT* __restrict__ keys_in = (pass & 1) ? j.keys_out : j.keys_in;
	const uint32_t* __restrict__ vals_in = (pass & 1) ? j.vals_out : j.vals_in;
	KeyT* __restrict__ keys_out = (pass & 1) ? j.keys_in : j.keys_out;
	uint32_t* __restrict__ vals_out = (pass & 1) ? j.vals_in : j.vals_out;
	const uint32_t* __restrict__ n_device = j.n_device;
	const size_t job_tiles = (j.n + kBlock - 1) / kBlock;
	uint32_t n = (uint32_t)j.n;  // (fewer than 2^30: the look-back words hold no more)
	if (n_device)  // (no kernel writes it meanwhile: read by the scalar unit)
		n = (uint32_t)min(j.n, (size_t)*(const __attribute__((address_space(4))) uint32_t*)(uintptr_t)n_device);
	// The launch is sized for the job with the most tiles, and for an upper bound of n: as many workgroups take a tile as there are
	// tiles, the others leave at once.  (Most of a depth sort's, which is launched for all Gaussians: 25 -> 22 us per pass for three
	// submodels of a city, a twentieth of 27 M in view, when they no longer took a ticket first.)
	if (blockIdx.x >= (n + (uint32_t)kBlock - 1u) / (uint32_t)kBlock)
		return;
	bool ends_here = false;
	if (kKind != kPassPlain) {
		const bool extra = j.temp[kSortExtraPass] != 0u;
		if (kKind == kPassOnDemand && !extra)
			return;
		ends_here = kKind == kPassOnDemand || !extra;
	}
	// the digit counts of a pass: 512 words apart for 32-bit keys whatever the digit width, 256 for 64-bit keys
	constexpr int kCountStride = sizeof(KeyT) == 4 ? 512 : 256;
	const uint32_t* __restrict__ digit_count = (j.digit_counts ? j.digit_counts : j.temp) + pass * kCountStride;
	uint32_t* __restrict__ lookback = j.temp + kSortHeader + (size_t)pass * kBins * job_tiles;
	uint32_t* __restrict__ tile_counter = j.temp + kSortCounters + pass;
	uint32_t* __restrict__ status = j.temp + kSortStatus;
	constexpr int kCountKeys = kWaves * kBins * (int)sizeof(uint16_t) / (int)sizeof(KeyT);  // the room that the counts take
	__shared__ __align__(16) KeyT s_keys[kBlock > kCountKeys ? kBlock : kCountKeys];
	__shared__ uint32_t s_vals[kBlock];
	__shared__ SortCounts<kBits> sc;
	__shared__ uint32_t s_scan[kWaves];
	// per-wave digit counts, then their exclusive prefix over waves; the keys take their place when all have been read
	uint16_t (*const wave_hist)[kBins] = reinterpret_cast<uint16_t (*)[kBins]>(s_keys);
	static_assert(sizeof(s_keys) >= kWaves * kBins * sizeof(uint16_t), "the counts fit where the keys go");
	__shared__ uint32_t s_tile;

	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const bool owns = tid < kBins;
	const int own = tid * kOwn;  // the first digit value that the thread owns
	// Tiles are handed out in arrival order, so every tile a block waits for below belongs to
	// a block that is already running.
	if (tid == 0)
		s_tile = atomicAdd(tile_counter, 1u);
#pragma unroll
	for (int w = 0; w < kWaves * kBins / 2 / kSortThreads; w++)
		reinterpret_cast<uint32_t*>(s_keys)[w * kSortThreads + tid] = 0u;
	__syncthreads();
	const uint32_t tile = s_tile;
	const uint32_t block_base = tile * (uint32_t)kBlock;
	const uint32_t wave_base = block_base + (uint32_t)wave * (kItems * 64);

	KeyT key[kItems];
	uint32_t val[kItems];
	uint32_t rank[kItems];
	// Behind the data a tile is filled up with keys of ones: the last digit value, and after every pair in the tile that has it.
	if (block_base + (uint32_t)kBlock <= n) {
		const KeyT* const keys_at = keys_in + wave_base;
		const uint32_t* const vals_at = vals_in + wave_base;
#pragma unroll
		for (int i = 0; i < kItems; i++) {
			key[i] = keys_at[i * 64 + lane];
			val[i] = vals_at[i * 64 + lane];
		}
	} else {
#pragma unroll
		for (int i = 0; i < kItems; i++) {
			const uint32_t k = wave_base + (uint32_t)(i * 64 + lane);
			const bool ok = k < n;
			key[i] = ok ? keys_in[k] : (KeyT)~(KeyT)0;
			val[i] = ok ? vals_in[k] : 0u;
		}
	}

#pragma unroll
	for (int i = 0; i < kItems; i++) {
		const uint32_t d = digit_of(key[i], shift, mask);
		// The lanes with this lane's digit: a vote per bit, taken as it is or inverted by a mask made of the lane's own bit, four vector
		// instructions per bit instead of nine (which kept the SIMDs busy for 60 % of a pass: 78 -> 71 us for the instances of
		// 5.6 M Gaussians at 1600x1036).
		uint32_t same_lo = ~0u, same_hi = ~0u;
#pragma unroll
		for (int b = 0; b < kBits; b++) {
			int bit = (int)(d << (31 - b)) >> 31;
			asm("" : "+v"(bit));  // (or the compiler forms the bit a second time for the vote)
			const uint64_t vote = lanes_where(bit != 0);
			// same & ~(vote ^ bit), one instruction
			same_lo = (uint32_t)__builtin_amdgcn_bitop3_b32((int)same_lo, (int)(uint32_t)vote, bit, 0x90);
			same_hi = (uint32_t)__builtin_amdgcn_bitop3_b32((int)same_hi, (int)(uint32_t)(vote >> 32), bit, 0x90);
		}
		const uint32_t below = __builtin_amdgcn_mbcnt_hi(same_hi, __builtin_amdgcn_mbcnt_lo(same_lo, 0u));
		// every lane reads its digit's count (lanes of one digit the same word), then the first of each digit's lanes adds theirs:
		// a wavefront's LDS accesses are served in order
		const uint32_t prior = wave_hist[wave][d];
		if (below == 0u)
			wave_hist[wave][d] = (uint16_t)(prior + (uint32_t)__popc(same_lo) + (uint32_t)__popc(same_hi));
		rank[i] = prior + below;
		asm volatile("" : "+v"(rank[i]), "+v"(key[i]));  // (the sum is made here, and the digit taken from the key again later)
		__builtin_amdgcn_wave_barrier();
	}
	// the counts of the thread's digit value in all tiles, needed once this tile's are published
	Word totals[kDigitCopies] = {};
	if (owns) {
		totals[0] = *reinterpret_cast<const Word*>(digit_count + own);
		if (j.digit_copies > 1u)
#pragma unroll
			for (int c = 1; c < kDigitCopies; c++)
				totals[c] = *reinterpret_cast<const Word*>(digit_count + c * kDigitWords + own);
	}
	__syncthreads();

	// For the digit values that a thread owns: prefix over the waves, publish the tile's counts.
	const uint32_t valid = min(n - block_base, (uint32_t)kBlock);
	// (by its distance in bytes, below 2^32: an address of 64 bits takes its registers through the whole kernel)
	auto word_of = [&](uint32_t t) { return reinterpret_cast<Word*>(reinterpret_cast<char*>(lookback) + (t * (uint32_t)kBins + (uint32_t)own) * 4u); };
	Word count = 0, digit_start;
	{
		typedef std::conditional_t<kOwn == 2, uint32_t, uint16_t> Counts;  // (two counts of 16 bits are added as one number)
		uint32_t prefix = 0;
		if (owns) {
			uint32_t c[kWaves];
#pragma unroll
			for (int w = 0; w < kWaves; w++)
				c[w] = *reinterpret_cast<const Counts*>(&wave_hist[w][own]);
#pragma unroll
			for (int w = 0; w < kWaves; w++) {
				*reinterpret_cast<Counts*>(&wave_hist[w][own]) = (Counts)prefix;
				prefix += c[w];
			}
		}
		count = kOwn == 2 ? (Word)(prefix & 0xFFFFu) | (Word)(prefix >> 16) << (32 * (kOwn - 1)) : (Word)prefix;
		uint32_t total;
		const uint32_t ex = block_exclusive_scan_u32<kWaves>(kOwn == 2 ? (prefix & 0xFFFFu) + (prefix >> 16) : prefix, s_scan, total);
		if (owns) {
			sc.digit_base[own] = (uint16_t)ex;
			if (kOwn == 2)
				sc.digit_base[own + kOwn - 1] = (uint16_t)(ex + (prefix & 0xFFFFu));
		}
		// what fills the tile up is not published
		if ((uint32_t)(own + kOwn - 1) == mask)
			count -= (Word)((uint32_t)kBlock - valid) << (32 * (kOwn - 1));
		else if ((uint32_t)own == mask)
			count -= (Word)((uint32_t)kBlock - valid);
		if (owns)
			__hip_atomic_store(word_of(tile), count | (tile == 0 ? kInclusives : kAggregates), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		// where the digit's run starts in the whole array: the exclusive scan of the digit counts
		uint32_t all;
		Word digit_total = 0;
#pragma unroll
		for (int c = 0; c < kDigitCopies; c++)
			digit_total += totals[c];
		if (kOwn == 2) {
			const uint32_t start = block_exclusive_scan_u32<kWaves>((uint32_t)digit_total + (uint32_t)(digit_total >> (32 * (kOwn - 1))), s_scan, all);
			digit_start = (Word)start | (Word)(start + (uint32_t)digit_total) << (32 * (kOwn - 1));
		} else {
			digit_start = block_exclusive_scan_u32<kWaves>((uint32_t)digit_total, s_scan, all);
		}
	}

	// The tile's pairs in digit order, through LDS.  None of this needs the tiles before this one: by the time
	// the look-back below starts, more of them have finished theirs and it has fewer words to read.
#pragma unroll
	for (int i = 0; i < kItems; i++) {
		const uint32_t d = digit_of(key[i], shift, mask);
		rank[i] += (uint32_t)sc.digit_base[d] + (uint32_t)wave_hist[wave][d];
	}
	__syncthreads();  // the counts have been read
#pragma unroll
	for (int i = 0; i < kItems; i++) {
		s_keys[rank[i]] = key[i];
		s_vals[rank[i]] = val[i];
	}
	__syncthreads();
	// every LDS read of the thread is asked for before anything needs one
	KeyT out_key[kItems];
	uint32_t out_val[kItems];
#pragma unroll
	for (int i = 0; i < kItems; i++) {
		const uint32_t p = (uint32_t)i * kSortThreads + tid;
		const uint32_t q = p < valid ? p : 0u;
		out_key[i] = s_keys[q];
		out_val[i] = s_vals[q];
	}

	// Look back: the pairs of this thread's digit values in all earlier tiles.
	if (owns) {
		Word exclusive = 0;
		if (tile != 0) {
			// Words of the tiles below t are still to be added.  Up to kLookBatch of them are requested
			// together: walked one load at a time, the chain of tiles and not memory sets the pace of a pass.
			uint32_t t = tile;
			bool gave_up = spin_limit < 0, done = false;
			while (!gave_up && !done) {
				Word v[kLookBatch];
#pragma unroll
				for (int q = 0; q < kLookBatch; q++)
					v[q] = (uint32_t)q < t ? __hip_atomic_load(word_of(t - 1u - (uint32_t)q), __ATOMIC_RELAXED,
					                                           __HIP_MEMORY_SCOPE_AGENT)
					                       : kInclusives;  // below the first tile there is nothing
				uint32_t used = 0;
#pragma unroll
				for (int q = 0; q < kLookBatch; q++) {
					// a word counts once every nearer one has been published and none of them closed the sum
					if (!done && used == (uint32_t)q && (v[q] & (kAggregates | kInclusives)) != 0u) {
						exclusive += v[q] & kValues;
						used = (uint32_t)q + 1u;
						done = (v[q] & kInclusives) != 0u;
					}
				}
				t -= used < t ? used : t;
				if (t == 0u)
					done = true;
				if (!done && used < (uint32_t)kLookBatch) {
					// tile t - 1 has not published yet: wait for its word, then look again from there
					const Word* word = word_of(t - 1u);
					Word w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					for (int spins = 0; (w & (kAggregates | kInclusives)) == 0u; spins++) {
						// give up after a bounded wait, or as soon as any other look-back has
						if (spins >= spin_limit ||
						    ((spins & 255) == 255 &&
						     __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
							gave_up = true;
							break;
						}
						__builtin_amdgcn_s_sleep(1);
						w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					}
				}
			}
			if (gave_up)
				atomicOr(status, 1u);
			// On the (never expected) give-up path `exclusive` is too small, which keeps every
			// scatter address inside the array; the status word tells the consumer to discard it.
			__hip_atomic_store(word_of(tile), ((exclusive + count) & kValues) | kInclusives, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		*reinterpret_cast<Word*>(&sc.global_base[own]) = digit_start + exclusive;
	}
	__syncthreads();

	uint32_t out_at[kItems];  // (fewer than 2^30 pairs)
#pragma unroll
	for (int i = 0; i < kItems; i++) {
		const uint32_t p = (uint32_t)i * kSortThreads + tid;
		const uint32_t d = digit_of(out_key[i], shift, mask);
		out_at[i] = p < valid ? sc.global_base[d] + (p - (uint32_t)sc.digit_base[d]) : n;
	}
	if (kKind != kPassPlain && ends_here) {
		// the sort ends here: a value's index and tile count go to arrays of their own (a count stored as all ones did
		// not fit and is looked up; an index that a sort which gave up left behind may be anything and is clamped)
		const uint32_t index_bits = j.index_bits, cap = 0xFFFFFFFFu >> index_bits, index_mask = (1u << index_bits) - 1u;
#pragma unroll
		for (int i = 0; i < kItems; i++) {
			if (out_at[i] < n) {
				const uint32_t index = out_val[i] & index_mask;
				uint32_t c = out_val[i] >> index_bits;
				if (c == cap)
					c = j.count_of[min(index, j.in_size - 1u)];
				j.final_index[out_at[i]] = index;
				j.final_count[out_at[i]] = c;
			}
		}
		return;
	}
#pragma unroll
	for (int i = 0; i < kItems; i++) {
		if (out_at[i] < n) {
			keys_out[out_at[i]] = out_key[i];
			vals_out[out_at[i]] = out_val[i];
		}
	}
}

size_t sort_temp_words(size_t n)
{
	return sort_temp_words_for(n);
}

const uint32_t* sort_status_word(const uint32_t* temp)
{
	return temp + kSortStatus;
}

static size_t sort_tiles(size_t n, int items)
{
	const size_t block = (size_t)kSortThreads * items;
	return (n + block - 1) / block;
}

// (a launch takes its tiles by the room of all its jobs, n among them: never smaller ones than n alone would have)
size_t sort_clear_words(size_t n, int end_bit, int max_bits)
{
	const size_t tiles = sort_tiles(n, sort_items(n, max_bits));
	return kSortHeader + (size_t)sort_passes(end_bit, max_bits) * ((size_t)1 << max_bits) * tiles;
}

// (a view lists between a twentieth and a third of the Gaussians of a large scene)
static int depth_sort_items(size_t n)
{
	const int items = sort_items(n, 9);
	return items == kSortItemsMany ? sort_items(n / 2, 9) : items;
}

size_t depth_sort_clear_words(size_t n)
{
	const size_t tiles = sort_tiles(n, depth_sort_items(n));
	return kSortHeader + (size_t)(kDepthPasses + 1) * 512 * tiles;
}

// One pass over every job of the batch, in tiles by the room for pairs of all its jobs.
template <typename KeyT, int kBits, int kKind, bool kDepth>
static void launch_sort_pass(const Batch<SortJob<KeyT>>& b, size_t most_pairs, size_t pairs, int jobs, int pass, int shift, uint32_t mask,
                             hipStream_t s)
{
	// (64-bit keys, of the stand-alone entry points alone, take the smallest tiles: larger ones fill the LDS)
	const int items = sizeof(KeyT) != 4 ? kSortItemsFew : kDepth ? depth_sort_items(pairs) : sort_items(pairs, kBits);
	const dim3 grid((unsigned)sort_tiles(most_pairs, items), (unsigned)jobs);
	const int spin = g_lookback_spin_limit.load();
	if constexpr (sizeof(KeyT) == 4) {
		if constexpr (kBits >= 9) {
			if (items == kSortItemsMany) {
				hipLaunchKernelGGL((sort_onesweep_kernel<KeyT, kBits, kKind, kSortItemsMany>), grid, dim3(kSortThreads), 0, s, b, pass, shift, mask, spin);
				return;
			}
		}
		if (items == kSortItems) {
			hipLaunchKernelGGL((sort_onesweep_kernel<KeyT, kBits, kKind, kSortItems>), grid, dim3(kSortThreads), 0, s, b, pass, shift, mask, spin);
			return;
		}
	}
	hipLaunchKernelGGL((sort_onesweep_kernel<KeyT, kBits, kKind, kSortItemsFew>), grid, dim3(kSortThreads), 0, s, b, pass, shift, mask, spin);
}

template <typename KeyT, int kBits>
static void sort_pairs(const SortJob<KeyT>* jobs, int count, int end_bit, bool temp_cleared, bool histograms_done, bool mark_stages,
                       hipStream_t s)
{
	const int passes = sort_passes(end_bit, kBits);
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<SortJob<KeyT>> b = {};
		size_t most = 0, pairs = 0;
		int live = 0;
		for (int k = 0; k < nj; k++) {
			const SortJob<KeyT>& j = jobs[at + k];
			if (j.n == 0)
				continue;
			b.job[live++] = j;
			most = j.n > most ? j.n : most;
			pairs += j.n;
			if (!temp_cleared)
				launch_fill_u32(j.temp, 0u, kSortHeader + (size_t)passes * (1u << kBits) * sort_tiles(j.n, kSortItemsFew), s);
		}
		if (live == 0)
			continue;
		if (mark_stages && !histograms_done)
			stage_mark("sort_setup", s);
		// every block ends with an atomic add per digit and pass into its job's counts: a few hundred blocks per
		// job read the keys as fast as thousands would, and queue far fewer adds on the same words
		const uint32_t most_blocks = live >= 8 ? 256u : 2048u / (uint32_t)live;
		const uint32_t hist_blocks = (uint32_t)min(sort_tiles(most, kSortItemsFew), (size_t)most_blocks);
		if (!histograms_done) {
			if constexpr (sizeof(KeyT) == 8)
				hipLaunchKernelGGL(sort_digit_histogram_kernel<KeyT>, dim3(hist_blocks, (unsigned)live), dim3(256), 0, s, b, passes, end_bit);
		}
		for (int p = 0; p < passes; p++) {
			const int shift = sort_digit_shift(end_bit, p, kBits);
			const int bits = sort_digit_bits(end_bit, p, kBits);
			const uint32_t mask = (1u << bits) - 1u;
			if (mark_stages)
				stage_mark("sort_onesweep", s);
			launch_sort_pass<KeyT, kBits, kPassPlain, false>(b, most, pairs, live, p, shift, mask, s);
		}
	}
}

void launch_sort_pairs(uint64_t* keys_in, uint64_t* keys_out, uint32_t* vals_in, uint32_t* vals_out, size_t n,
                       int end_bit, uint32_t* temp, hipStream_t s)
{
	SortJob<uint64_t> job = {};
	job.keys_in = keys_in; job.keys_out = keys_out; job.vals_in = vals_in; job.vals_out = vals_out;
	job.n = n; job.temp = temp;
	sort_pairs<uint64_t, kDigitBitsU64>(&job, 1, end_bit, false, false, true, s);
}

// The digit counts must come from the kernel that wrote the keys (histograms_done): nothing here reads 32-bit keys for them.
void launch_sort_pairs_u32(const SortJob<uint32_t>* jobs, int count, int end_bit, bool temp_cleared, bool histograms_done,
                           const char* stage, hipStream_t s)
{
	switch (sort_max_digit_bits_u32(end_bit)) {
	case 11: sort_pairs<uint32_t, 11>(jobs, count, end_bit, temp_cleared, histograms_done, stage != nullptr, s); break;
	case 10: sort_pairs<uint32_t, 10>(jobs, count, end_bit, temp_cleared, histograms_done, stage != nullptr, s); break;
	case 9: sort_pairs<uint32_t, 9>(jobs, count, end_bit, temp_cleared, histograms_done, stage != nullptr, s); break;
	case 8: sort_pairs<uint32_t, 8>(jobs, count, end_bit, temp_cleared, histograms_done, stage != nullptr, s); break;
	default: sort_pairs<uint32_t, 7>(jobs, count, end_bit, temp_cleared, histograms_done, stage != nullptr, s);
	}
}

// ---- depth order of few Gaussians: one workgroup per job, out of LDS -------------------------------
// The eight kernels of the general path (pairs, four passes, totals, offsets) take 6 to 8 us each over a single tile of pairs, nearly all
// of it launches and dependent reads.  Here the listed Gaussians' keys are read once into LDS, every pass ranks and moves them there,
// and the offsets and the key duplication's table leave at the end.  The same order: stable passes over the same digits, the
// fourth if a key has bits above kDepthKeyBits.  (From the pairs to the offsets, general path and this, us: 4 000 Gaussians 38 and 13.)
template <int kItems>
__global__ __launch_bounds__(1024) void small_depth_order_kernel(Batch<DepthOrderJob> batch)
{
	constexpr int kBlock = 1024 * kItems, kWaves = 16, kBins = 512;
	__shared__ __align__(16) uint32_t s_keys[kBlock], s_vals[kBlock];
	__shared__ __align__(16) uint16_t s_hist[kWaves][kBins];  // per wavefront: counts of the digits, then their prefix over the wavefronts
	__shared__ uint16_t s_digit_base[kBins];
	__shared__ uint32_t s_scan[kWaves];
	__shared__ uint32_t s_above;  // bits above those of the three passes
	__shared__ uint32_t s_tiles[kWaves];
	const DepthOrderJob& j = batch.job[blockIdx.x];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const uint32_t P = (uint32_t)j.P, index_bits = depth_index_bits(P), cap = 0xFFFFFFFFu >> index_bits, index_mask = (1u << index_bits) - 1u;
	uint32_t n;
	{
		// the Gaussians that touch a tile (those with a depth), in index order
		float depth[kItems];
		uint32_t count[kItems], mine = 0, above = 0;
		const uint32_t first = (uint32_t)(tid * kItems);
#pragma unroll
		for (int q = 0; q < kItems; q += 4) {
			float4 d = {0.f, 0.f, 0.f, 0.f};
			uint4 c = {0u, 0u, 0u, 0u};
			if (first + q + 4 <= P) {
				d = *reinterpret_cast<const float4*>(j.depths + first + q);
				c = *reinterpret_cast<const uint4*>(j.tiles_touched + first + q);
			} else {
				float* dv = &d.x;
				uint32_t* cv = &c.x;
#pragma unroll
				for (int k = 0; k < 4; k++)
					if (first + q + k < P) {
						dv[k] = j.depths[first + q + k];
						cv[k] = j.tiles_touched[first + q + k];
					}
			}
			depth[q] = d.x; depth[q + 1] = d.y; depth[q + 2] = d.z; depth[q + 3] = d.w;
			count[q] = c.x; count[q + 1] = c.y; count[q + 2] = c.z; count[q + 3] = c.w;
		}
		if (tid == 0)
			s_above = 0u;
#pragma unroll
		for (int q = 0; q < kItems; q++)
			mine += __float_as_uint(depth[q]) != 0u ? 1u : 0u;
		uint32_t tiles = 0;
#pragma unroll
		for (int q = 0; q < kItems; q++)
			tiles += count[q];
		tiles = wave_inclusive_scan_u32(tiles);
		if (lane == 63)
			s_tiles[wave] = tiles;
		uint32_t at = block_exclusive_scan_u32<kWaves>(mine, s_scan, n);
		if (tid == 0 && j.totals.total_out) {
			uint32_t total = 0;
#pragma unroll
			for (int w = 0; w < kWaves; w++)
				total += s_tiles[w];
			if (j.totals.total_copy)
				__hip_atomic_store(j.totals.total_copy, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);  // (the host waits for this word)
			*j.totals.total_out = total;
			*j.totals.visible_count = n;
		}
#pragma unroll
		for (int q = 0; q < kItems; q++)
			if (__float_as_uint(depth[q]) != 0u) {
				const uint32_t key = __float_as_uint(depth[q]) - kDepthKeyBase;
				s_keys[at] = key;
				s_vals[at] = (first + (uint32_t)q) | (min(count[q], cap) << index_bits);
				above |= key >> kDepthKeyBits;
				at++;
			}
		if (above != 0u)
			atomicOr(&s_above, above);
		// filled up with keys of ones: the last digit values, and after every pair that has them
		for (uint32_t k = n + (uint32_t)tid; k < (uint32_t)kBlock; k += 1024u) {
			s_keys[k] = 0xFFFFFFFFu;
			s_vals[k] = 0u;
		}
		__syncthreads();
	}
	const int passes = s_above != 0u ? kDepthPasses + 1 : kDepthPasses;
	for (int pass = 0; pass < passes; pass++) {
		const int shift = 9 * pass;
		const uint32_t mask = pass < kDepthPasses ? 511u : 31u;
#pragma unroll
		for (int w = 0; w < kWaves * kBins / 2 / 1024; w++)
			reinterpret_cast<uint32_t*>(s_hist)[1024 * w + tid] = 0u;
		__syncthreads();
		uint32_t key[kItems], val[kItems], rank[kItems];
#pragma unroll
		for (int i = 0; i < kItems; i++) {
			const int at = wave * (kItems * 64) + 64 * i + lane;
			key[i] = s_keys[at];
			val[i] = s_vals[at];
		}
#pragma unroll
		for (int i = 0; i < kItems; i++) {  // (as in sort_onesweep_kernel)
			const uint32_t d = (key[i] >> shift) & mask;
			uint32_t same_lo = ~0u, same_hi = ~0u;
#pragma unroll
			for (int b = 0; b < 9; b++) {
				int own = (int)(d << (31 - b)) >> 31;
				asm("" : "+v"(own));
				const uint64_t vote = lanes_where(own != 0);
				same_lo = (uint32_t)__builtin_amdgcn_bitop3_b32((int)same_lo, (int)(uint32_t)vote, own, 0x90);
				same_hi = (uint32_t)__builtin_amdgcn_bitop3_b32((int)same_hi, (int)(uint32_t)(vote >> 32), own, 0x90);
			}
			const uint32_t below = __builtin_amdgcn_mbcnt_hi(same_hi, __builtin_amdgcn_mbcnt_lo(same_lo, 0u));
			const uint32_t prior = s_hist[wave][d];
			if (below == 0u)
				s_hist[wave][d] = (uint16_t)(prior + (uint32_t)__popc(same_lo) + (uint32_t)__popc(same_hi));
			rank[i] = prior + below;
			__builtin_amdgcn_wave_barrier();
		}
		__syncthreads();
		uint32_t count = 0, all;
		if (tid < kBins) {
			uint32_t c[kWaves];
#pragma unroll
			for (int w = 0; w < kWaves; w++)
				c[w] = s_hist[w][tid];
#pragma unroll
			for (int w = 0; w < kWaves; w++) {
				s_hist[w][tid] = (uint16_t)count;
				count += c[w];
			}
		}
		const uint32_t before = block_exclusive_scan_u32<kWaves>(count, s_scan, all);
		if (tid < kBins)
			s_digit_base[tid] = (uint16_t)before;
		__syncthreads();
#pragma unroll
		for (int i = 0; i < kItems; i++) {
			const uint32_t d = (key[i] >> shift) & mask, to = rank[i] + (uint32_t)s_digit_base[d] + (uint32_t)s_hist[wave][d];
			s_keys[to] = key[i];
			s_vals[to] = val[i];
		}
		__syncthreads();
	}
	// the order, the offsets of the instances in it, and where every run of kDupPositions of them starts
	uint32_t count[kItems], sum = 0;
	const uint32_t first = (uint32_t)(tid * kItems);
#pragma unroll
	for (int q = 0; q < kItems; q++) {
		count[q] = 0u;
		if (first + q < n) {
			const uint32_t v = s_vals[first + q], index = v & index_mask;
			count[q] = v >> index_bits;
			if (count[q] == cap)
				count[q] = j.tiles_touched[index];
			j.order[first + q] = index;
		}
		sum += count[q];
	}
	uint32_t total;
	uint32_t run = block_exclusive_scan_u32<kWaves>(sum, s_scan, total);
	const uint32_t table = (uint32_t)dup_first_words((size_t)P);
#pragma unroll
	for (int q = 0; q < kItems; q++)
		if (first + q < n) {
			const uint32_t begin = run;
			run += count[q];
			j.offsets_in_order[first + q] = run;
			for (uint32_t b = (begin + (uint32_t)kDupPositions - 1u) / (uint32_t)kDupPositions;
			     b < table && (uint64_t)b * (uint64_t)kDupPositions < (uint64_t)run; b++)
				j.dup_first[b] = first + (uint32_t)q;
		}
}

// A call's images from the Gaussians, general path and this, us: 4 000 Gaussians at 160x120 111 and 87, 8 000 114 and 99, 8 000 at 800x600
// 147 and 132; with sixteen per thread 12 000 at 320x240 121 and 122, 16 000 122 and 129.

static void launch_small_depth_order(const Batch<DepthOrderJob>& b, int jobs, int most, hipStream_t s)
{
	if (most <= 4096)
		hipLaunchKernelGGL(small_depth_order_kernel<4>, dim3((unsigned)jobs), dim3(1024), 0, s, b);
	else
		hipLaunchKernelGGL(small_depth_order_kernel<8>, dim3((unsigned)jobs), dim3(1024), 0, s, b);
}

void launch_depth_order(const DepthOrderJob* jobs, int count, hipStream_t s)
{
	stage_mark("depth_order", s);
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<DepthOrderJob> b = {};
		Batch<BlockScanJob> scan = {};
		Batch<BlockInclusiveJob> inc = {};
		Batch<SortJob<uint32_t>> sorts = {};
		int max_p = 0;
		size_t pairs = 0;
		for (int k = 0; k < nj; k++) {
			max_p = jobs[at + k].P > max_p ? jobs[at + k].P : max_p;
			pairs += (size_t)jobs[at + k].P;
		}
		const bool few_groups = ((size_t)max_p + kScanGroup - 1) / kScanGroup <= 4096;
		const dim3 grid((unsigned)((max_p + kScanGroup - 1) / kScanGroup), (unsigned)nj);
		// few workgroups per job, each over many groups: every one ends with an atomic add per digit into its job's counts (half and twice
		// as many: 17 and 27 us for 20 at two submodels of 2.8 M, 105 and 94 for 99 at four of 15.7 M)
		const unsigned most = nj >= 8 ? 256u : 2048u / (unsigned)nj;
		const dim3 pairs_grid(grid.x < most ? grid.x : most, (unsigned)nj);
		for (int k = 0; k < nj; k++) {
			DepthOrderJob& j = b.job[k];
			j = jobs[at + k];
			j.digit_copies = digit_copies(pairs_grid.x);
			SortJob<uint32_t>& sj = sorts.job[k];
			sj.keys_in = j.keys_a; sj.keys_out = j.keys_b; sj.vals_in = j.vals_a; sj.vals_out = j.vals_b;
			sj.n = (size_t)j.P; sj.n_device = j.visible_count; sj.temp = j.sort_temp; sj.digit_counts = j.digits; sj.digit_copies = j.digit_copies;
			sj.final_index = j.order; sj.final_count = j.tiles_in_order; sj.count_of = j.tiles_touched;
			sj.index_bits = depth_index_bits((uint32_t)j.P); sj.in_size = (uint32_t)j.P;
			scan.job[k] = BlockScanJob{j.scan_temp, ((size_t)j.P + kScanGroup - 1) / kScanGroup, j.visible_count, (uint32_t)kScanGroup, nullptr, nullptr,
			                           nullptr, nullptr};
			inc.job[k] = BlockInclusiveJob{j.tiles_in_order, j.scan_temp, (size_t)j.P, j.visible_count, j.offsets_in_order, j.dup_first,
			                               (uint32_t)dup_first_words((size_t)j.P), few_groups ? 1u : 0u};
		}
		if (max_p <= kSmallOrder) {
			launch_small_depth_order(b, nj, max_p, s);
			continue;
		}
		hipLaunchKernelGGL(depth_pairs_kernel, pairs_grid, dim3(256), 0, s, b);
		// three passes of nine bits (a -> b -> a -> the order and the tile counts in that order), and the pass on demand
		launch_sort_pass<uint32_t, 9, kPassPlain, true>(sorts, (size_t)max_p, pairs, nj, 0, 0, 511u, s);
		launch_sort_pass<uint32_t, 9, kPassPlain, true>(sorts, (size_t)max_p, pairs, nj, 1, 9, 511u, s);
		launch_sort_pass<uint32_t, 9, kPassEndsUnless, true>(sorts, (size_t)max_p, pairs, nj, 2, 18, 511u, s);
		launch_sort_pass<uint32_t, 9, kPassOnDemand, true>(sorts, (size_t)max_p, pairs, nj, 3, kDepthKeyBits, 31u, s);
		const unsigned resident = 2048u / (unsigned)nj;  // eight workgroups per CU
		hipLaunchKernelGGL(order_totals_kernel, dim3(min(grid.x, resident), (unsigned)nj), dim3(256), 0, s, b);
		if (!few_groups)
			hipLaunchKernelGGL(single_block_exclusive_scan_kernel, dim3(1, (unsigned)nj), dim3(1024), 0, s, scan);
		hipLaunchKernelGGL(block_inclusive_scan_kernel<4>, grid, dim3(256), 0, s, inc);
	}
}

// Sets n words to v, 16 bytes per store where the address allows; a capped grid walks the array.
__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* __restrict__ p, uint32_t v, size_t n)
{
	const size_t tid = (size_t)blockIdx.x * 256 + threadIdx.x, threads = (size_t)gridDim.x * 256;
	// words up to the first 16-byte boundary, whole 16-byte groups, the rest
	const size_t head = min(n, (size_t)((16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15) / 4);
	const size_t groups = (n - head) / 4;
	if (tid < head)
		p[tid] = v;
	uint4* q = reinterpret_cast<uint4*>(p + head);
	const uint4 vv = {v, v, v, v};
	for (size_t g = tid; g < groups; g += threads)
		q[g] = vv;
	const size_t done = head + 4 * groups;
	if (tid < n - done)
		p[done + tid] = v;
}

// A few floats that travel with the launch.
__global__ __launch_bounds__(256) void write_floats_kernel(WriteFloatsArgs a)
{
	for (int k = threadIdx.x; k < a.n; k += 256)
		a.to[k] = a.v[k];
}

void launch_write_floats(const WriteFloatsArgs& a, hipStream_t s)
{
	hipLaunchKernelGGL(write_floats_kernel, dim3(1), dim3(256), 0, s, a);
}

// fill_u32_kernel for several arrays in one launch (the array in blockIdx.y).
__global__ __launch_bounds__(256) void fill_many_kernel(Batch<FillJob> batch, uint32_t v)
{
	uint32_t* __restrict__ p = batch.job[blockIdx.y].p;
	const size_t n = batch.job[blockIdx.y].n;
	const size_t tid = (size_t)blockIdx.x * 256 + threadIdx.x, threads = (size_t)gridDim.x * 256;
	const size_t head = min(n, (size_t)((16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15) / 4);
	const size_t groups = (n - head) / 4;
	if (tid < head)
		p[tid] = v;
	uint4* q = reinterpret_cast<uint4*>(p + head);
	const uint4 vv = {v, v, v, v};
	for (size_t g = tid; g < groups; g += threads)
		q[g] = vv;
	const size_t done = head + 4 * groups;
	if (tid < n - done)
		p[done + tid] = v;
}

void launch_fill_many(const FillJob* jobs, int count, uint32_t v, hipStream_t s)
{
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<FillJob> b = {};
		size_t most = 0;
		for (int k = 0; k < nj; k++) {
			b.job[k] = jobs[at + k];
			most = b.job[k].n > most ? b.job[k].n : most;
		}
		if (most == 0)
			continue;
		const size_t blocks = (most / 4 + 255) / 256 + 1, cap = 4096 / (size_t)nj + 1;
		hipLaunchKernelGGL(fill_many_kernel, dim3((unsigned)(blocks < cap ? blocks : cap), (unsigned)nj), dim3(256), 0, s, b, v);
	}
}

void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s)
{
	if (n == 0)
		return;
	const size_t blocks = (n / 4 + 255) / 256 + 1;
	hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, s, p, v, n);
}

// The status words (may be null) are those of the two sorts: if either reported a failure the
// ranges stay empty, so no later stage walks an unsorted list, and *fault (host memory that the
// device can write, may be null) is set for the host to find.  The keys carry strip bits above the
// tile (key_strips); per workgroup of kFileGroup keys (four neighbouring keys per thread), file_tail
// (may be null) receives how many keys of the tile of its last key have each of the four "filed" bits
// set, which is what the kernel that places the entries in their strips' lists needs from the
// workgroups ahead of its own.
__global__ __launch_bounds__(kFileBlock) void tile_ranges_kernel(Batch<TileRangesJob> batch)
{
	__shared__ uint2 s_tail[4];  // per wave, the four strips' counts packed 16 bits each
	__shared__ uint32_t s_last_tile;
	const TileRangesJob& j = batch.job[blockIdx.y];
	const uint32_t* __restrict__ keys = j.keys;
	size_t n = j.n;
	const uint32_t* __restrict__ n_device = j.n_device;
	uint2* __restrict__ ranges = j.ranges;
	const uint32_t* __restrict__ sort_status = j.sort_status;
	const uint32_t* __restrict__ order_status = j.order_status;
	uint32_t* __restrict__ fault = j.fault;
	uint4* __restrict__ file_tail = j.file_tail;
	size_t first = (size_t)blockIdx.x * kFileGroup;
	if (first >= j.n)
		return;  // the launch is sized for the job with the most keys
	// A workgroup's time is its chain of reads: the keys (there is room for j.n, whatever they hold), the statuses and the count are
	// asked for together, a group's keys while the one before it is worked on, and a thread's previous key comes from its neighbour
	// (71 M keys 100 -> 68 us, 42 M 61 -> 52).
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	uint32_t ahead[4] = {0u, 0u, 0u, 0u}, ahead_prev = 0u;
	auto ask_for = [&](size_t group) {
		const size_t at = group + 4 * (size_t)threadIdx.x;
		if (at + 3 < j.n) {
			const uint4 k4 = *reinterpret_cast<const uint4*>(keys + at);
			ahead[0] = k4.x; ahead[1] = k4.y; ahead[2] = k4.z; ahead[3] = k4.w;
		} else {
#pragma unroll
			for (int q = 0; q < 4; q++)
				if (at + q < j.n)
					ahead[q] = keys[at + q];
		}
		if (lane == 0 && at > 0 && at < j.n)
			ahead_prev = keys[at - 1];
	};
	ask_for(first);
	const uint32_t gave_up = (sort_status ? *sort_status : 0u) | (order_status ? *order_status : 0u);
	if (n_device)
		n = min(n, (size_t)*n_device);  // launched for an upper bound
	// the sort has read its digit counts: zero again for the next to count into them
	if (j.rezero) {
		const size_t threads = min((j.n + kFileGroup - 1) / kFileGroup, (size_t)gridDim.x) * kFileBlock;
		for (size_t w = (size_t)blockIdx.x * kFileBlock + threadIdx.x; w < (size_t)j.rezero_words; w += threads)
			j.rezero[w] = 0u;
	}
	if (gave_up != 0u) {
		if (blockIdx.x == 0 && threadIdx.x == 0 && fault)
			__hip_atomic_store(fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
		return;
	}
	for (const size_t step = (size_t)gridDim.x * kFileGroup; first < n; first += step) {
		const size_t idx0 = first + 4 * (size_t)threadIdx.x;
		const uint32_t key[4] = {ahead[0], ahead[1], ahead[2], ahead[3]};
		const uint32_t lane_before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)key[3], 0x138, 0xF, 0xF, false);  // (wave_shr:1)
		uint32_t prev = key_tile(lane == 0 ? ahead_prev : lane_before);
		if (first + step < n)
			ask_for(first + step);
		const size_t last = min(n, first + kFileGroup) - 1;
#pragma unroll
		for (int q = 0; q < 4; q++) {
			const size_t idx = idx0 + q;
			const uint32_t cur = key_tile(key[q]);
			if (idx < n) {
				if (idx == 0) {
					ranges[cur].x = 0;
				} else if (cur != prev) {
					ranges[prev].y = (uint32_t)idx;
					ranges[cur].x = (uint32_t)idx;
				}
				if (idx == n - 1)
					ranges[cur].y = (uint32_t)n;
				if (idx == last)
					s_last_tile = cur;
			}
			prev = cur;
		}
		if (!file_tail)
			continue;
		__syncthreads();
		const uint32_t last_tile = s_last_tile;
		uint2 own = {0u, 0u};
#pragma unroll
		for (int q = 0; q < 4; q++)
			if (idx0 + q < n && key_tile(key[q]) == last_tile) {  // sorted: these are the workgroup's last keys
				const uint32_t bits = key_strips(key[q]);
				own.x += (bits & 1u) | ((bits & 2u) << 15);
				own.y += ((bits >> 2) & 1u) | ((bits & 8u) << 13);
			}
		const uint2 inc = {wave_inclusive_scan_u32(own.x), wave_inclusive_scan_u32(own.y)};
		if (lane == 63)
			s_tail[wave] = inc;
		__syncthreads();
		if (threadIdx.x == 0) {
			const uint32_t x = s_tail[0].x + s_tail[1].x + s_tail[2].x + s_tail[3].x;
			const uint32_t y = s_tail[0].y + s_tail[1].y + s_tail[2].y + s_tail[3].y;
			file_tail[first / kFileGroup] = uint4{x & 0xFFFFu, x >> 16, y & 0xFFFFu, y >> 16};
		}
	}
}

__global__ void report_sort_status_kernel(const uint32_t* __restrict__ status, uint32_t* __restrict__ fault,
                                          uint32_t* __restrict__ device_fault)
{
	if (threadIdx.x == 0 && *status != 0u) {
		if (fault)
			__hip_atomic_store(fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
		if (device_fault)
			*device_fault = 1u;
	}
}

void launch_report_sort_status(const uint32_t* temp, uint32_t* fault, uint32_t* device_fault, hipStream_t s)
{
	if (fault || device_fault)
		hipLaunchKernelGGL(report_sort_status_kernel, dim3(1), dim3(64), 0, s, temp + kSortStatus, fault, device_fault);
}

void launch_tile_ranges(const TileRangesJob* jobs, int count, hipStream_t s)
{
	stage_mark("tile_ranges", s);
	for (int at = 0; at < count; at += kMaxBatch) {
		const int nj = count - at < kMaxBatch ? count - at : kMaxBatch;
		Batch<TileRangesJob> b = {};
		size_t max_n = 0;
		int live = 0;
		for (int k = 0; k < nj; k++) {
			if (jobs[at + k].n == 0)
				continue;
			b.job[live++] = jobs[at + k];
			max_n = jobs[at + k].n > max_n ? jobs[at + k].n : max_n;
		}
		// Up to 8 192 groups a workgroup each (as fast or faster), beyond that as many workgroups as are resident together, eight per CU.
		const size_t groups = (max_n + kFileGroup - 1) / kFileGroup, most = groups * (size_t)live <= 8192 ? groups : max((size_t)2048 / (size_t)live, (size_t)1);
		if (live)
			hipLaunchKernelGGL(tile_ranges_kernel, dim3((unsigned)min(groups, most), (unsigned)live),
			                   dim3(kFileBlock), 0, s, b);
	}
}

}  // namespace rgs
