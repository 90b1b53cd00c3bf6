// The host path of a training iteration's steps around the rasterizer: activation of stored parameters, boundary
// straddlers, image loss, optimiser.
#include "host.h"

namespace rgs_host {
namespace {

Tensor contiguous_f32(const Tensor& t)
{
	if (!t.defined())
		return t;
	return (t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)).contiguous();
}

std::vector<int64_t> rows_of(int64_t rows, at::IntArrayRef shape)
{
	std::vector<int64_t> s(shape.begin(), shape.end());
	s[0] = rows;
	return s;
}

// A tensor at the start of an allocation with `spare` more rows behind it.
Tensor with_room(at::IntArrayRef shape, int64_t spare, const at::Device& device)
{
	const Tensor room = new_f32(rows_of(shape[0] + spare, shape), device);
	return spare == 0 ? room : carved(room, 0, shape);
}

// ---- activation --------------------------------------------------------------------------------------------------

bool has_shape(const Tensor& t, at::IntArrayRef shape) { return t.sizes() == shape; }

// What the get_* properties of the reference's Gaussian model compute (scene/gaussian_nn_module.py:373-394).
// Outputs SH coefficients, scales, rotations, opacities.
struct Activate : torch::autograd::Function<Activate> {
	static variable_list forward(AutogradContext* ctx, const Tensor& dc_in, const Tensor& rest_in, const Tensor& scaling_in,
	                             const Tensor& rotation_in, const Tensor& opacity_in, int64_t spare)
	{
		for (const Tensor* t : {&dc_in, &rest_in, &scaling_in, &rotation_in, &opacity_in})
			if (!t->is_cuda())
				throw std::runtime_error("activation runs on the GPU only: the parameters must be device tensors");
		const Tensor dc = contiguous_f32(dc_in), rest = contiguous_f32(rest_in), scaling = contiguous_f32(scaling_in),
		             rotation = contiguous_f32(rotation_in), opacity = contiguous_f32(opacity_in);
		const int64_t n = dc.size(0), r = rest.dim() > 1 ? rest.size(1) : 0;
		if (!has_shape(dc, {n, 1, 3}) || !has_shape(rest, {n, r, 3}))
			throw std::runtime_error("features_dc must be (N,1,3) and features_rest (N,R,3)");
		if (!has_shape(scaling, {n, 3}) || !has_shape(rotation, {n, 4}) || !has_shape(opacity, {n, 1}))
			throw std::runtime_error("scaling (N,3), rotation (N,4), opacity (N,1) expected");
		const at::Device device = dc.device();
		const Tensor shs = with_room({n, 1 + r, 3}, spare, device), scales = with_room({n, 3}, spare, device),
		             rotations = with_room({n, 4}, spare, device), opacities = with_room({n, 1}, spare, device);
		c10::DeviceGuard guard(device);
		check(rgs_activate_forward(n, r, ptr(dc), ptr(rest), ptr(scaling), ptr(rotation), ptr(opacity), ptr(shs), ptr(scales),
		                           ptr(rotations), ptr(opacities), current_stream(device)));
		ctx->save_for_backward({rotation, scales, opacities});
		ctx->saved_data["rest"] = r;
		ctx->set_materialize_grads(false);  // an output outside the loss arrives undefined and costs nothing
		return {shs, scales, rotations, opacities};
	}

	static variable_list backward(AutogradContext* ctx, variable_list grads)
	{
		return in_backward([&]() -> variable_list {
			const variable_list saved = ctx->get_saved_variables();
			const Tensor &rotation = saved[0], &scales = saved[1], &opacities = saved[2];
			const int64_t n = rotation.size(0), r = ctx->saved_data["rest"].toInt();
			const at::Device device = rotation.device();
			const Tensor g_shs = contiguous_f32(grads[0]), g_scales = contiguous_f32(grads[1]), g_rotations = contiguous_f32(grads[2]),
			             g_opacities = contiguous_f32(grads[3]);
			auto made = [&](const Tensor& g, at::IntArrayRef shape) { return g.defined() ? new_f32(shape, device) : Tensor(); };
			const Tensor d_dc = made(g_shs, {n, 1, 3}), d_rest = made(g_shs, {n, r, 3}), d_scaling = made(g_scales, {n, 3}),
			             d_rotation = made(g_rotations, {n, 4}), d_opacity = made(g_opacities, {n, 1});
			c10::DeviceGuard guard(device);
			check(rgs_activate_backward(n, r, ptr(rotation), ptr(scales), ptr(opacities), ptr(g_shs), ptr(g_scales), ptr(g_rotations),
			                            ptr(g_opacities), ptr(d_dc), ptr(d_rest), ptr(d_scaling), ptr(d_rotation), ptr(d_opacity),
			                            current_stream(device)));
			return {d_dc, d_rest, d_scaling, d_rotation, d_opacity, Tensor()};
		});
	}
};

py::tuple activate(const Tensor& dc, const Tensor& rest, const Tensor& scaling, const Tensor& rotation, const Tensor& opacity,
                   int64_t spare)
{
	variable_list out;
	{
		py::gil_scoped_release no_gil;
		out = Activate::apply(dc, rest, scaling, rotation, opacity, spare);
	}
	return py::make_tuple(out[0], out[1], out[2], out[3]);
}

// The placeholder through which the reference collects the screen-space gradient norm that densification reads
// (gaussian_renderer/render_half_gs.py:7-19): an (N,1) meta tensor becomes the (N,3) zeros passed as means2D, with `spare` more
// rows of room behind them; the meta tensor's gradient is the length of each row's (x, y) gradient.
struct ScreenPlaceholder : torch::autograd::Function<ScreenPlaceholder> {
	static Tensor forward(AutogradContext*, const Tensor& meta, int64_t spare)
	{
		if (meta.dim() != 2 || meta.size(1) != 1)
			throw std::runtime_error("meta must have shape (N, 1)");
		if (spare == 0)
			return at::zeros({meta.size(0), 3}, meta.options());
		const Tensor room = at::empty({meta.size(0) + spare, 3}, meta.options());
		const Tensor zeros = carved(room, 0, {meta.size(0), 3});
		zeros.zero_();
		return zeros;
	}

	static variable_list backward(AutogradContext*, variable_list grads)
	{
		return {at::norm(grads[0].narrow(1, 0, 2), 2, {-1}, true), Tensor()};
	}
};

Tensor screen_placeholder(const Tensor& meta, int64_t spare)
{
	py::gil_scoped_release no_gil;
	return ScreenPlaceholder::apply(meta, spare);
}

// ---- boundary straddlers -----------------------------------------------------------------------------------------

enum Field { kFieldMeans3D, kFieldMeans2D, kFieldOpacity, kFieldScales, kFieldRotations, kFieldSH, kFields };
const char* const kFieldNames[kFields] = {"means3D", "means2D", "opacity", "scales", "rotations", "shs"};

uint32_t* row_list(const Tensor& t) { return static_cast<uint32_t*>(t.data_ptr()); }

// Selection for every source: (counts[K*K], row lists by source).  `boxes`: K lower corners, then K upper corners, three floats
// each.  `capacity`: longest list there is room for at first, negative for one that depends on the submodel's size; a list
// that needs more is written again.
py::tuple select_straddlers(const std::vector<Tensor>& means3D, const std::vector<Tensor>& scales, const std::vector<float>& boxes,
                            int64_t capacity)
{
	const int K = static_cast<int>(means3D.size());
	if (K < 1 || K > RGS_MAX_SHARE_BOXES || static_cast<int>(scales.size()) != K || static_cast<int>(boxes.size()) != 6 * K)
		throw std::runtime_error("select_straddlers: between 1 and " + std::to_string(RGS_MAX_SHARE_BOXES) + " submodels");
	std::vector<int64_t> counts(K * K);
	variable_list lists(K);
	{
		py::gil_scoped_release no_gil;
		at::NoGradGuard no_grad;
		const at::Device device = means3D[0].device();
		c10::DeviceGuard guard(device);
		const hipStream_t stream = current_stream(device);
		const float *low = boxes.data(), *up = low + 3 * K;
		const at::TensorOptions ints = at::TensorOptions().dtype(at::kInt).device(device);
		AwaitedCounts awaited(device.index(), stream, K * K);
		variable_list scratch;
		std::vector<int64_t> caps(K);
		auto run = [&](int src, uint32_t* counts_at) {
			const int64_t n = means3D[src].size(0);
			lists[src] = at::empty({K, caps[src]}, ints);
			scratch.push_back(new_bytes(std::max<size_t>(1, rgs_straddler_scratch_bytes(n, K)), device));
			check(rgs_straddler_select(n, ptr(means3D[src]), ptr(scales[src]), low + 3 * src, up + 3 * src, K, low, up, src,
			                           counts_at, ptr<uint32_t>(lists[src]), caps[src],
			                           scratch.back().data_ptr(), stream));
		};
		for (int src = 0; src < K; src++) {
			const int64_t n = means3D[src].size(0);
			caps[src] = std::min(n, capacity < 0 ? n / 8 + 4096 : capacity);
			run(src, awaited.on_device() + src * K);
		}
		const uint32_t* arrived = awaited.wait();
		if (!arrived)
			throw std::runtime_error("reading the straddlers' counts failed");
		std::copy(arrived, arrived + K * K, counts.begin());
		for (int src = 0; src < K; src++) {
			const int64_t longest = *std::max_element(counts.begin() + src * K, counts.begin() + (src + 1) * K);
			if (longest > caps[src]) {  // a list was cut short: once more with room for the longest
				caps[src] = longest;
				scratch.push_back(at::empty({K}, ints));  // (the awaited words go to another call when this one returns)
				run(src, ptr<uint32_t>(scratch.back()));
			}
		}
	}
	py::dict rows;
	for (int s = 0; s < K; s++)
		for (int d = 0; d < K; d++)
			if (counts[s * K + d] > 0)
				rows[py::make_tuple(s, d)] = lists[s].select(0, d).narrow(0, 0, counts[s * K + d]);
	return py::make_tuple(counts, rows);
}

// Lent rows of a merge: destination by destination, in merge order.
struct Lent {
	int source;
	Tensor rows;
	int64_t count;
};

struct Merge : torch::CustomClassHolder {
	std::vector<int64_t> own;              // rows of every submodel's own
	std::vector<std::vector<Lent>> lent;   // by destination
	bool reuse_gradients, append;
	std::vector<std::vector<int64_t>> shapes;
	int sh_floats = 0;
	int64_t merged_size(int dst) const
	{
		int64_t n = own[dst];
		for (const Lent& l : lent[dst])
			n += l.count;
		return n;
	}
};

// All destinations at once, so that a lender's gradient is written in one place: its own rows' gradient plus what every
// borrower adds.
struct MergeShared : torch::autograd::Function<MergeShared> {
	static variable_list forward(AutogradContext* ctx, at::TensorList flat, const c10::intrusive_ptr<Merge>* held)
	{
		Merge& m = **held;
		const int K = static_cast<int>(m.own.size());
		const at::Device device = flat[0].device();
		c10::DeviceGuard guard(device);
		const hipStream_t stream = current_stream(device);
		m.sh_floats = flat[kFieldSH].dim() > 1 ? static_cast<int>(c10::multiply_integers(flat[kFieldSH].sizes().slice(1))) : 0;
		for (const Tensor& t : flat)
			m.shapes.push_back(t.sizes().vec());
		variable_list out;
		out.reserve(flat.size());
		std::vector<rgs_shared_rows> segments;
		for (int dst = 0; dst < K; dst++) {
			const int64_t P = m.merged_size(dst), own = m.own[dst];
			std::array<Tensor, kFields> merged;
			segments.clear();
			for (int f = 0; f < kFields; f++) {
				const Tensor& t = flat[kFields * dst + f];
				const std::vector<int64_t> shape = rows_of(P, t.sizes());
				if (m.append) {
					// the lent rows go behind the destination's own rows, which stay where they are
					const size_t end = (t.storage_offset() + c10::multiply_integers(shape)) * t.element_size();
					if (end > t.storage().nbytes())
						throw std::runtime_error("submodel " + std::to_string(dst) + ": no room for " + std::to_string(P - own) +
						                         " lent rows behind its " + kFieldNames[f] +
						                         "; allocate the field with spare rows or merge with append=False");
					merged[f] = carved(t, 0, shape);
				} else {
					merged[f] = new_f32(shape, device);
				}
			}
			if (m.append)
				merged[kFieldMeans2D].narrow(0, own, P - own).zero_();
			else
				merged[kFieldMeans2D].zero_();
			auto add = [&](int source, const Tensor& rows, int64_t count) {
				auto field = [&](int f) { return static_cast<const float*>(flat[kFields * source + f].data_ptr()); };
				segments.push_back({field(kFieldMeans3D), field(kFieldOpacity), field(kFieldScales), field(kFieldRotations), field(kFieldSH),
				                    rows.defined() ? row_list(rows) : nullptr, static_cast<uint32_t>(count)});
			};
			if (!m.append)
				add(dst, Tensor(), own);
			for (const Lent& l : m.lent[dst])
				add(l.source, l.rows, l.count);
			check(rgs_merge_rows(static_cast<int>(segments.size()), segments.data(), m.append ? own : 0, m.sh_floats,
			                     ptr(merged[kFieldMeans3D]), ptr(merged[kFieldOpacity]), ptr(merged[kFieldScales]),
			                     ptr(merged[kFieldRotations]), ptr(merged[kFieldSH]), stream));
			out.insert(out.end(), merged.begin(), merged.end());
		}
		ctx->set_materialize_grads(false);
		ctx->saved_data["merge"] = c10::IValue::make_capsule(*held);
		return out;
	}

	static variable_list backward(AutogradContext* ctx, variable_list grads)
	{
		return in_backward([&]() -> variable_list {
			const auto holder = ctx->saved_data["merge"].toCapsule();
			const Merge& m = static_cast<const Merge&>(*holder);
			const int K = static_cast<int>(m.own.size());
			at::Device device(at::kCPU);
			for (Tensor& g : grads)
				if (g.defined()) {
					g = g.contiguous();
					device = g.device();
				}
			variable_list out(K * kFields + 1);
			if (!device.is_cuda())
				return out;
			c10::DeviceGuard guard(device);
			const hipStream_t stream = current_stream(device);
			// a lender's gradient starts as the gradient of its own rows in its own merged arrays
			for (int i = 0; i < K * kFields; i++) {
				const Tensor& g = grads[i];
				if (!g.defined()) {
					out[i] = new_f32(m.shapes[i], device).zero_();
				} else {
					const Tensor own = carved(g, 0, rows_of(m.own[i / kFields], g.sizes()));
					out[i] = m.reuse_gradients ? own : own.clone();
				}
			}
			std::vector<rgs_shared_grads> segments;
			for (int dst = 0; dst < K; dst++) {
				const Tensor* g = &grads[kFields * dst];
				bool any = false;
				for (int f = 0; f < kFields; f++)
					any = any || g[f].defined();
				if (m.lent[dst].empty() || !any)
					continue;
				segments.clear();
				for (const Lent& l : m.lent[dst]) {
					auto into = [&](int f) { return static_cast<float*>(out[kFields * l.source + f].data_ptr()); };
					segments.push_back({into(kFieldMeans3D), into(kFieldMeans2D), into(kFieldOpacity), into(kFieldScales),
					                    into(kFieldRotations), into(kFieldSH), row_list(l.rows), static_cast<uint32_t>(l.count)});
				}
				check(rgs_merge_rows_backward(static_cast<int>(segments.size()), segments.data(), m.own[dst], m.sh_floats,
				                              ptr(g[kFieldMeans3D]), ptr(g[kFieldMeans2D]), ptr(g[kFieldOpacity]), ptr(g[kFieldScales]),
				                              ptr(g[kFieldRotations]), ptr(g[kFieldSH]), stream));
			}
			return out;
		});
	}
};

// `lent`: for every destination a list of (source, row list, count).
std::vector<Tensor> merge_shared(const std::vector<int64_t>& own, const py::sequence& lent, bool reuse_gradients, bool append,
                                 const std::vector<Tensor>& flat)
{
	auto merge = c10::make_intrusive<Merge>();
	merge->own = own;
	merge->reuse_gradients = reuse_gradients;
	merge->append = append;
	merge->lent.resize(own.size());
	if (own.empty() || lent.size() != own.size() || flat.size() != kFields * own.size())
		throw std::runtime_error("merge_shared: six fields and a list of lent rows per submodel");
	for (size_t d = 0; d < own.size(); d++)
		for (py::handle h : py::reinterpret_borrow<py::sequence>(lent[d])) {
			const py::tuple t = py::reinterpret_borrow<py::tuple>(h);
			merge->lent[d].push_back({py::cast<int>(t[0]), from_python(t[1], "rows"), py::cast<int64_t>(t[2])});
			if (merge->lent[d].back().source < 0 || merge->lent[d].back().source >= static_cast<int>(own.size()))
				throw std::runtime_error("merge_shared: rows of a submodel that is not there");
		}
	py::gil_scoped_release no_gil;
	return MergeShared::apply(at::TensorList(flat), &merge);
}

// ---- the stored models of an iteration ----------------------------------------------------------------------------

// A stored model's tensors in the order of StoredModel.parameters but for the placeholder, which comes last.
enum StoredField { kStoredXyz, kStoredFirst, kStoredRest, kStoredScaling, kStoredRotation, kStoredOpacity, kStoredMeta, kStoredFields };
// What a model becomes for the frame: merged rows (own, then lent ones), its SH rows in parts.
enum ShownField { kShownMeans3D, kShownMeans2D, kShownOpacity, kShownScales, kShownRotations, kShownFirst, kShownRest, kShownLent, kShownFields };

struct Stored : torch::CustomClassHolder {
	int K = 0;
	std::vector<float> boxes;               // lower corners, then upper corners
	std::vector<int64_t> spare;             // rows of room that the models' positions have behind them; used if append
	bool append = false;
	std::vector<int64_t> own, total, counts;  // counts[source * K + destination]
	std::vector<rgs_lend_segment> segments;
	variable_list lists;                    // the row lists that the segments point into
};

// Activation, selection, lending for all models of an iteration at once: what activate, select_straddlers and merge_shared do one
// after another, with one launch per step whatever the number of models (an iteration of two models is 36 kernels instead of 49), and
// without a joined copy of the SH rows, which the rasterizer reads, and whose gradients it writes, as they are stored.
struct ShowStored : torch::autograd::Function<ShowStored> {
	static Tensor with_rows(const Tensor& room, int64_t rows)
	{
		return carved(room, 0, rows_of(rows, room.sizes()));
	}

	static variable_list forward(AutogradContext* ctx, at::TensorList in, const c10::intrusive_ptr<Stored>* held)
	{
		Stored& m = **held;
		const int K = m.K;
		const at::Device device = in[0].device();
		c10::DeviceGuard guard(device);
		const hipStream_t stream = current_stream(device);
		auto given = [&](int k, int f) -> const Tensor& { return in[kStoredFields * k + f]; };
		// activated tensors with room behind them for the lent rows: as much as the positions have, or a guess
		std::vector<std::array<Tensor, 4>> act(K);  // scales, rotations, opacity, means2D
		std::vector<rgs_stored_model> models(K);
		std::vector<int64_t> room(K);
		for (int k = 0; k < K; k++) {
			const int64_t n = given(k, kStoredXyz).size(0);
			m.own.push_back(n);
			room[k] = m.append ? m.spare[k] : n / 8 + 4096;
			act[k] = {new_f32({n + room[k], 3}, device), new_f32({n + room[k], 4}, device), new_f32({n + room[k], 1}, device),
			          new_f32({n + room[k], 3}, device)};
			models[k] = {static_cast<int>(n), static_cast<int>(n + room[k]), ptr(given(k, kStoredScaling)), ptr(given(k, kStoredRotation)),
			             ptr(given(k, kStoredOpacity)), ptr(act[k][0]), ptr(act[k][1]), ptr(act[k][2]), ptr(act[k][3])};
		}
		check(rgs_activate_models(K, models.data(), stream));
		select(m, in, act, device, stream);
		// where lent rows go: destination by destination, lenders in ascending order
		variable_list out;
		out.reserve(K * kShownFields);
		std::vector<rgs_lend_model> lend(K);
		std::vector<rgs_lend_segment> copies;
		for (int d = 0; d < K; d++) {
			int64_t lent = 0;
			for (int s = 0; s < K; s++) {
				const int64_t count = m.counts[s * K + d];
				if (s != d && count > 0) {
					m.segments.push_back({s, d, static_cast<const uint32_t*>(m.lists[s].data_ptr()) + d * m.lists[s].size(1), static_cast<uint32_t>(count),
					                      static_cast<uint32_t>(m.own[d] + lent), static_cast<uint32_t>(lent)});
					lent += count;
				}
			}
			const int64_t n = m.own[d], P = n + lent;
			m.total.push_back(P);
			const Tensor& xyz = given(d, kStoredXyz);
			Tensor means3D;
			if (m.append) {
				const size_t end = (xyz.storage_offset() + 3 * P) * sizeof(float);
				if (lent > room[d] || end > xyz.storage().nbytes())
					throw std::runtime_error("submodel " + std::to_string(d) + ": no room for " + std::to_string(lent) +
					                         " lent rows behind its means3D; allocate the field with spare rows or merge with append=False");
				means3D = carved(xyz, 0, {P, 3});
			} else {
				means3D = new_f32({P, 3}, device);
				copies.push_back({d, d, nullptr, static_cast<uint32_t>(n), 0u, 0u});
				if (lent > room[d])  // more than guessed: once more, with room for them all
					for (Tensor& t : act[d]) {
						const Tensor larger = new_f32(rows_of(P, t.sizes()), device).zero_();
						larger.narrow(0, 0, n).copy_(t.narrow(0, 0, n));
						t = larger;
					}
			}
			const Tensor sh_lent = new_f32({lent, 16, 3}, device);
			const Tensor &first = given(d, kStoredFirst), &rest = given(d, kStoredRest);
			lend[d] = {ptr(xyz), ptr(means3D), ptr(act[d][2]), ptr(act[d][0]), ptr(act[d][1]), ptr(first), ptr(rest), ptr(sh_lent)};
			out.insert(out.end(), {means3D, with_rows(act[d][3], P), with_rows(act[d][2], P), with_rows(act[d][0], P), with_rows(act[d][1], P),
			                       carved(first, 0, first.sizes()), carved(rest, 0, rest.sizes()), sh_lent});
		}
		copies.insert(copies.end(), m.segments.begin(), m.segments.end());
		check(rgs_lend_rows(K, lend.data(), static_cast<int>(copies.size()), copies.data(), stream));
		variable_list saved;
		for (int k = 0; k < K; k++)
			saved.insert(saved.end(), {given(k, kStoredRotation), with_rows(act[k][0], m.own[k]), with_rows(act[k][2], m.own[k])});
		ctx->save_for_backward(std::move(saved));
		ctx->set_materialize_grads(false);
		ctx->saved_data["stored"] = c10::IValue::make_capsule(*held);
		return out;
	}

	// Counts and row lists of all pairs; a list that did not fit is written again with room for it.
	static void select(Stored& m, at::TensorList in, const std::vector<std::array<Tensor, 4>>& act, const at::Device& device, hipStream_t stream)
	{
		const int K = m.K;
		const at::TensorOptions ints = at::TensorOptions().dtype(at::kInt).device(device);
		AwaitedCounts awaited(device.index(), stream, K * K);
		std::vector<rgs_straddler_source> sources(K);
		variable_list scratch;
		m.lists.resize(K);
		auto source = [&](int k, int64_t capacity) {
			m.lists[k] = at::empty({K, capacity}, ints);
			scratch.push_back(new_bytes(std::max<size_t>(1, rgs_straddler_scratch_bytes(m.own[k], K)), device));
			return rgs_straddler_source{static_cast<int>(m.own[k]), ptr(in[kStoredFields * k + kStoredXyz]), ptr(act[k][0]),
			                            awaited.on_device() + k * K, ptr<uint32_t>(m.lists[k]), static_cast<uint32_t>(capacity),
			                            scratch.back().data_ptr()};
		};
		for (int k = 0; k < K; k++)
			sources[k] = source(k, std::min(m.own[k], m.own[k] / 8 + 4096));
		const float *low = m.boxes.data(), *up = low + 3 * K;
		check(rgs_straddler_select_many(K, sources.data(), low, up, stream));
		const uint32_t* arrived = awaited.wait();
		if (!arrived)
			throw std::runtime_error("reading the straddlers' counts failed");
		m.counts.assign(arrived, arrived + K * K);
		for (int k = 0; k < K; k++) {
			const int64_t longest = *std::max_element(m.counts.begin() + k * K, m.counts.begin() + (k + 1) * K);
			if (longest > m.lists[k].size(1)) {
				rgs_straddler_source f = source(k, longest);
				scratch.push_back(at::empty({K}, ints));  // (the awaited words go to another call when this one returns)
				f.counts = ptr<uint32_t>(scratch.back());
				check(rgs_straddler_select(f.n, f.means3D, f.scales, low + 3 * k, up + 3 * k, K, low, up, k, f.counts, f.rows, f.capacity,
				                           f.scratch, stream));
			}
		}
	}

	static variable_list backward(AutogradContext* ctx, variable_list grads)
	{
		return in_backward([&]() -> variable_list {
			const auto holder = ctx->saved_data["stored"].toCapsule();
			const Stored& m = static_cast<const Stored&>(*holder);
			const int K = m.K;
			const variable_list saved = ctx->get_saved_variables();
			const at::Device device = saved[0].device();
			c10::DeviceGuard guard(device);
			const hipStream_t stream = current_stream(device);
			// gradients that did not come are zeros, unless only borrowers would read them
			std::vector<rgs_lend_gradients> all(K);
			for (int k = 0; k < K; k++) {
				const int64_t n = m.own[k], P = m.total[k];
				const std::array<std::vector<int64_t>, kShownFields> shapes = {{{P, 3}, {P, 3}, {P, 1}, {P, 3}, {P, 4}, {n, 1, 3}, {n, 15, 3}, {P - n, 16, 3}}};
				for (int f = 0; f < kShownFields; f++) {
					Tensor& g = grads[kShownFields * k + f];
					if (g.defined())
						g = g.contiguous();
					else if (f != kShownLent)
						g = new_f32(shapes[f], device).zero_();
				}
				auto at = [&](int f) { return ptr(grads[kShownFields * k + f]); };
				all[k] = {at(kShownMeans3D), at(kShownMeans2D), at(kShownOpacity), at(kShownScales), at(kShownRotations), at(kShownFirst), at(kShownRest),
				          at(kShownLent)};
			}
			check(rgs_lend_rows_backward(K, all.data(), static_cast<int>(m.segments.size()), m.segments.data(), stream));
			variable_list out(K * kStoredFields + 1);
			std::vector<rgs_stored_model_grads> models(K);
			for (int k = 0; k < K; k++) {
				const int64_t n = m.own[k];
				const Tensor* g = &grads[kShownFields * k];
				Tensor* d = &out[kStoredFields * k];
				d[kStoredXyz] = carved(g[kShownMeans3D], 0, {n, 3});
				d[kStoredFirst] = g[kShownFirst];
				d[kStoredRest] = g[kShownRest];
				d[kStoredScaling] = new_f32({n, 3}, device);
				d[kStoredRotation] = new_f32({n, 4}, device);
				d[kStoredOpacity] = new_f32({n, 1}, device);
				d[kStoredMeta] = new_f32({n, 1}, device);
				models[k] = {static_cast<int>(n), ptr(saved[3 * k]), ptr(saved[3 * k + 1]), ptr(saved[3 * k + 2]), all[k].scales, all[k].rotations,
				             all[k].opacity, all[k].means2D, ptr(d[kStoredScaling]), ptr(d[kStoredRotation]), ptr(d[kStoredOpacity]),
				             ptr(d[kStoredMeta])};
			}
			check(rgs_activate_models_backward(K, models.data(), stream));
			return out;
		});
	}
};

// Whether show_stored takes these models (kStoredFields tensors each): what one launch can hold, as its kernels read it.
bool stored_together(const variable_list& in)
{
	const size_t K = in.size() / kStoredFields;
	if (K < 1 || K > RGS_MAX_STORED_MODELS)
		return false;
	for (size_t k = 0; k < K; k++) {
		const Tensor* t = &in[kStoredFields * k];
		const int64_t n = t[kStoredXyz].dim() == 2 ? t[kStoredXyz].size(0) : 0;
		if (n < 1 || n >= int64_t(1) << 30)
			return false;
		const std::array<std::vector<int64_t>, kStoredFields> shapes = {{{n, 3}, {n, 1, 3}, {n, 15, 3}, {n, 3}, {n, 4}, {n, 1}, {n, 1}}};
		for (int f = 0; f < kStoredFields; f++)
			if (!t[f].is_cuda() || t[f].device() != in[0].device() || t[f].scalar_type() != at::kFloat || !t[f].is_contiguous() ||
			    t[f].sizes() != at::IntArrayRef(shapes[f]) ||
			    ((f == kStoredScaling || f == kStoredRotation || f == kStoredOpacity) && (reinterpret_cast<uintptr_t>(t[f].data_ptr()) & 15) != 0))
				return false;
	}
	return true;
}

// None where the models cannot be taken together; otherwise (counts[K*K], kShownFields tensors per model).  `boxes` as in select_straddlers.
py::object show_stored(const variable_list& in, const std::vector<float>& boxes, const std::vector<int64_t>& spare, bool append)
{
	if (!stored_together(in))
		return py::none();
	auto stored = c10::make_intrusive<Stored>();
	stored->K = static_cast<int>(in.size() / kStoredFields);
	if (static_cast<int>(boxes.size()) != 6 * stored->K || static_cast<int>(spare.size()) != stored->K)
		throw std::runtime_error("show_stored: a box and a number of spare rows per model");
	stored->boxes = boxes;
	stored->spare = spare;
	stored->append = append;
	variable_list out;
	{
		py::gil_scoped_release no_gil;
		out = ShowStored::apply(at::TensorList(in), &stored);
	}
	return py::make_tuple(stored->counts, out);
}

// Values on the device that the host need not keep: they travel with a launch.
Tensor floats_on_device(const std::vector<float>& values, const Tensor& like)
{
	py::gil_scoped_release no_gil;
	const at::Device device = like.device();
	const Tensor t = new_f32({static_cast<int64_t>(values.size())}, device);
	c10::DeviceGuard guard(device);
	check(rgs_write_floats(static_cast<int>(values.size()), values.data(), ptr(t), current_stream(device)));
	return t;
}

// ---- image loss --------------------------------------------------------------------------------------------------

// (1 - lambda) L1 + lambda (1 - SSIM).  Outputs the loss and (loss, L1, SSIM), of which only the first is differentiable.
struct L1SSIM : torch::autograd::Function<L1SSIM> {
	static variable_list forward(AutogradContext* ctx, const Tensor& image, const Tensor& gt, double lambda_dssim, bool keep)
	{
		const Tensor x = contiguous_f32(image), y = contiguous_f32(gt);
		const int64_t H = x.size(-2), W = x.size(-1), planes = x.numel() / (H * W);  // planes are windowed independently
		const at::Device device = x.device();
		c10::DeviceGuard guard(device);
		const Tensor workspace = new_bytes(rgs_loss_workspace_bytes(planes, H, W), device), out = new_f32({3}, device);
		check(rgs_l1_ssim_forward(planes, H, W, ptr(x), ptr(y), lambda_dssim, ptr(out), ptr<void>(workspace), keep,
		                          current_stream(device)));
		ctx->save_for_backward({x, y, workspace});
		ctx->saved_data["lambda"] = lambda_dssim;
		ctx->saved_data["shape"] = image.sizes().vec();
		ctx->mark_non_differentiable({out});
		ctx->set_materialize_grads(false);
		return {out.select(0, 0), out};
	}

	static variable_list backward(AutogradContext* ctx, variable_list grads)
	{
		return in_backward([&]() -> variable_list {
			const variable_list saved = ctx->get_saved_variables();
			const Tensor &x = saved[0], &y = saved[1], &workspace = saved[2];
			if (!grads[0].defined())
				return {Tensor(), Tensor(), Tensor(), Tensor()};
			const int64_t H = x.size(-2), W = x.size(-1), planes = x.numel() / (H * W);
			const Tensor d_image = new_f32(ctx->saved_data["shape"].toIntVector(), x.device()), g = contiguous_f32(grads[0]);
			c10::DeviceGuard guard(x.device());
			check(rgs_l1_ssim_backward(planes, H, W, ptr(x), ptr(y), ctx->saved_data["lambda"].toDouble(), ptr(g),
			                           ptr<const void>(workspace), ptr(d_image), current_stream(x.device())));
			return {d_image, Tensor(), Tensor(), Tensor()};
		});
	}
};

py::tuple l1_ssim(const Tensor& image, const Tensor& gt, double lambda_dssim)
{
	if (image.sizes() != gt.sizes())
		throw std::runtime_error("image and ground truth differ in shape");
	if (image.dim() != 3 && image.dim() != 4)
		throw std::runtime_error("expected (C,H,W) or (B,C,H,W) images");
	if (image.size(-1) == 0 || image.size(-2) == 0)
		throw std::runtime_error("the loss of an image without pixels is not defined");
	if (!image.is_cuda() || !gt.is_cuda())
		throw std::runtime_error("the loss runs on the GPU only: both images must be device tensors");
	variable_list out;
	{
		py::gil_scoped_release no_gil;
		out = L1SSIM::apply(image, gt, lambda_dssim, at::GradMode::is_enabled() && image.requires_grad());
	}
	return py::make_tuple(out[0], out[1]);
}

// ---- Adam --------------------------------------------------------------------------------------------------------

// The update of every parameter that has a gradient; tensors that share device, betas and eps go into one call.  `groups` and
// `state` are the optimiser's param_groups and state.
void adam_step(const py::list& groups, const py::object& state)
{
	struct Batch {
		at::Device device;
		double beta1, beta2, eps;
		std::vector<rgs_adam_tensor> tensors;
	};
	std::vector<Batch> batches;
	variable_list keep;
	at::NoGradGuard no_grad;
	const py::str key_step("step"), key_m("exp_avg"), key_v("exp_avg_sq");
	for (py::handle group_h : groups) {
		const py::dict group = py::reinterpret_borrow<py::dict>(group_h);
		const double lr = py::cast<double>(py::float_(group["lr"])), eps = py::cast<double>(py::float_(group["eps"]));
		const py::sequence betas = group["betas"];
		const double beta1 = py::cast<double>(py::float_(betas[0])), beta2 = py::cast<double>(py::float_(betas[1]));
		for (py::handle p_h : py::list(group["params"])) {
			const Tensor p = from_python(p_h, "a parameter");
			Tensor grad = p.grad();
			if (!grad.defined())
				continue;
			if (!p.is_cuda())
				throw std::runtime_error("this optimiser updates device tensors only");
			if (grad.is_sparse() || p.scalar_type() != at::kFloat || !p.is_contiguous())
				throw std::runtime_error("parameters must be dense contiguous float32");
			py::dict s = state[p_h];
			if (s.empty()) {
				s[key_step] = 0;
				s[key_m] = at::zeros_like(p, p.suggest_memory_format());
				s[key_v] = at::zeros_like(p, p.suggest_memory_format());
			}
			const int64_t step = py::cast<int64_t>(py::int_(s[key_step])) + 1;
			s[key_step] = step;
			if (!grad.is_contiguous())
				grad = grad.contiguous();
			keep.push_back(grad);
			const Tensor m = from_python(s[key_m], "exp_avg"), v = from_python(s[key_v], "exp_avg_sq");
			Batch* batch = nullptr;
			for (Batch& b : batches)
				if (b.device == p.device() && b.beta1 == beta1 && b.beta2 == beta2 && b.eps == eps)
					batch = &b;
			if (!batch) {
				batches.push_back({p.device(), beta1, beta2, eps, {}});
				batch = &batches.back();
			}
			rgs_adam_tensor t{};
			t.param = static_cast<float*>(p.data_ptr());
			t.grad = static_cast<const float*>(grad.data_ptr());
			t.exp_avg = static_cast<float*>(m.data_ptr());
			t.exp_avg_sq = static_cast<float*>(v.data_ptr());
			t.n = p.numel();
			t.lr = lr;
			t.step = step;
			batch->tensors.push_back(t);
		}
	}
	py::gil_scoped_release no_gil;
	for (const Batch& b : batches) {
		c10::DeviceGuard guard(b.device);
		check(rgs_adam_step(static_cast<int>(b.tensors.size()), b.tensors.data(), b.beta1, b.beta2, b.eps, current_stream(b.device)));
	}
}

}  // namespace

void define_training(py::module_& m)
{
	m.def("activate", &activate);
	m.def("screen_placeholder", &screen_placeholder);
	m.def("select_straddlers", &select_straddlers);
	m.def("merge_shared", &merge_shared);
	m.def("show_stored", &show_stored);
	m.def("floats_on_device", &floats_on_device);
	m.def("l1_ssim", &l1_ssim);
	m.def("adam_step", &adam_step);
}

}  // namespace rgs_host
