// The host path between PyTorch and the C ABI of include/rgs.h, in native code: tensors in, workspaces allocated, library
// called, autograd nodes that do the same for the gradients.  A frame's kernels take some hundreds of microseconds, the
// launches of all of them together about 90; written in Python the steps around them took 800 more per training pass of a
// small frame (argument tables, slices, torch.autograd.Function's own bookkeeping) and the card waited for them.
//
// The library's entry points are taken from the global symbols of the process (the ctypes binding loads it first), so both
// bindings always talk to the same build.  Nothing here holds the interpreter lock while it allocates, launches or waits.
#include "host.h"

namespace rgs_host {
namespace {

// ---- compositor --------------------------------------------------------------------------------------------------

Tensor plane(const Tensor& t, const at::Device& device, int64_t channels, int64_t H, int64_t W)
{
	Tensor p = t.scalar_type() == at::kFloat && t.device() == device ? t : t.to(device, at::kFloat);
	if (p.dim() != 3 || p.size(0) != channels || p.size(1) != H || p.size(2) != W) {
		std::string got;
		for (int64_t s : p.sizes())
			got += (got.empty() ? "" : ", ") + std::to_string(s);
		throw std::runtime_error("partial image plane has shape (" + got + "), expected (" + std::to_string(channels) + ", " +
		                         std::to_string(H) + ", " + std::to_string(W) + ")");
	}
	return p.is_contiguous() ? p : p.contiguous();
}

Tensor background_of(const std::optional<Tensor>& background, const at::Device& device)
{
	if (!background)
		return Tensor();
	Tensor b = background->reshape(-1);
	if (b.numel() != 3)
		throw std::runtime_error("the background needs three values");
	return device_f32(b, device);
}

// The planes of K layers as tables of addresses: colours, depths, alphas.
struct PlaneTables {
	std::array<const float*, RGS_MAX_COMPOSITE> images, depths, alphas;
	void set(int k, const Tensor& image, const Tensor& depth, const Tensor& alpha)
	{
		images[k] = ptr(image);
		depths[k] = ptr(depth);
		alphas[k] = ptr(alpha);
	}
};

// What the layers of a frame bring beside their planes, if they come straight from the rasterizer: their image workspaces, in which it says what
// each strip lists, and the background they all had.
struct LayerStrips {
	variable_list images;  // per layer, undefined ones for layers without
	Tensor background;
};

// Outputs image, depth, alpha.  `planes`: the layers' colours, then their depths, then their alphas.
struct Composite : torch::autograd::Function<Composite> {
	using StripTable = std::array<const uint32_t*, RGS_MAX_COMPOSITE>;
	static StripTable strip_table(const Tensor* images, int K, int64_t H, int64_t W)
	{
		std::array<size_t, RGS_IMG_FIELDS> offset;
		check(rgs_image_layout(W, H, offset.data()));
		StripTable t{};
		for (int k = 0; k < K; k++)
			if (const char* image = ptr<const char>(images[k]))
				t[k] = reinterpret_cast<const uint32_t*>(image + offset[RGS_IMG_STRIP_TOTAL]);
		return t;
	}

	static variable_list forward(AutogradContext* ctx, at::TensorList planes, const std::optional<Tensor>* background,
	                             const LayerStrips* strips)
	{
		const int K = static_cast<int>(planes.size() / 3);
		const at::Device device = planes[0].device();
		if (!planes[0].is_cuda())
			throw std::runtime_error("the compositor needs its inputs on a GPU (device memory)");
		const int64_t H = planes[0].size(-2), W = planes[0].size(-1);
		variable_list saved;
		saved.reserve(4 * K + 2);
		for (int k = 0; k < 3 * K; k++)
			saved.push_back(plane(planes[k], device, k < K ? 3 : 1, H, W));
		const Tensor bg = background_of(*background, device);
		PlaneTables in;
		for (int k = 0; k < K; k++)
			in.set(k, saved[k], saved[K + k], saved[2 * K + k]);
		const Tensor image = new_f32({3, H, W}, device), depth = new_f32({1, H, W}, device), alpha = new_f32({1, H, W}, device);
		c10::DeviceGuard guard(device);
		const bool with_strips = strips->background.defined();
		StripTable counts{};
		if (with_strips)
			counts = strip_table(strips->images.data(), K, H, W);
		check(rgs_composite_layers_forward(K, H, W, in.images.data(), in.depths.data(), in.alphas.data(), ptr(bg),
		                                   with_strips ? counts.data() : nullptr, ptr(strips->background), ptr(image), ptr(depth),
		                                   ptr(alpha), current_stream(device)));
		// an absent depth or alpha gradient comes back undefined and goes down as a null pointer
		ctx->set_materialize_grads(false);
		saved.push_back(bg);
		if (with_strips) {
			saved.push_back(strips->background);
			saved.insert(saved.end(), strips->images.begin(), strips->images.end());
		}
		ctx->save_for_backward(std::move(saved));
		ctx->saved_data["strips"] = with_strips;
		return {image, depth, alpha};
	}

	static variable_list backward(AutogradContext* ctx, variable_list grads)
	{
		return in_backward([&]() -> variable_list {
			const variable_list saved = ctx->get_saved_variables();
			const bool with_strips = ctx->saved_data["strips"].toBool();
			const int K = static_cast<int>(with_strips ? (saved.size() - 2) / 4 : saved.size() / 3);
			const at::Device device = saved[0].device();
			const int64_t H = saved[0].size(1), W = saved[0].size(2);
			auto given = [&](const Tensor& g, int64_t channels) { return g.defined() ? plane(g, device, channels, H, W) : Tensor(); };
			const Tensor g_depth = given(grads[1], 1), g_alpha = given(grads[2], 1);
			Tensor g_image = given(grads[0], 3);
			if (!g_image.defined())
				g_image = new_f32({3, H, W}, device).zero_();
			PlaneTables in;
			std::array<float*, RGS_MAX_COMPOSITE> d_images, d_depths, d_alphas;
			// The background is a constant to the loss: no gradient.  Without a gradient of the composited depth the layers'
			// depths have none either; told so, the rasterizer's backward leaves out the terms it would multiply.
			const bool with_depth = g_depth.defined();
			const int64_t planes = with_depth ? 5 : 4;
			variable_list out(3 * K + 2);
			for (int k = 0; k < K; k++) {
				in.set(k, saved[k], saved[K + k], saved[2 * K + k]);
				// a layer's three gradients in one (5,H,W) block, the layout of RenderResult.zip_grad
				// (parallel_utils/basic_parallel_trainer/task_utils.py:187-195); without the depth's if there is none
				const Tensor block = new_f32({planes, H, W}, device);
				d_images[k] = ptr(block);
				d_depths[k] = d_images[k] + 3 * H * W;
				d_alphas[k] = d_images[k] + (planes - 1) * H * W;
				out[k] = block.narrow(0, 0, 3);
				if (with_depth)
					out[K + k] = block.narrow(0, 3, 1);
				out[2 * K + k] = block.narrow(0, planes - 1, 1);
			}
			c10::DeviceGuard guard(device);
			StripTable counts{};
			if (with_strips)
				counts = strip_table(&saved[3 * K + 2], K, H, W);
			check(rgs_composite_layers_backward(K, H, W, in.images.data(), in.depths.data(), in.alphas.data(), ptr(saved[3 * K]),
			                                    with_strips ? counts.data() : nullptr, with_strips ? ptr(saved[3 * K + 1]) : nullptr,
			                                    ptr(g_image), ptr(g_depth), ptr(g_alpha), d_images.data(),
			                                    with_depth ? d_depths.data() : nullptr, d_alphas.data(), current_stream(device)));
			return out;
		});
	}
};

// `strips`: None, or what rasterize_frame handed out under that name for these layers, in their order here.
py::tuple composite(const std::optional<Tensor>& background, const std::vector<Tensor>& planes, py::handle strips)
{
	if (planes.empty() || planes.size() % 3 != 0 || planes.size() > 3 * RGS_MAX_COMPOSITE)
		throw std::runtime_error("the compositor takes between one layer and " + std::to_string(RGS_MAX_COMPOSITE) + " layers");
	LayerStrips known;
	if (!strips.is_none()) {
		const size_t K = planes.size() / 3;
		const int64_t bytes = static_cast<int64_t>(rgs_image_bytes(planes[0].size(-1), planes[0].size(-2)));
		bool one_background = true;
		for (py::handle h : py::reinterpret_borrow<py::sequence>(strips)) {
			const py::tuple layer = py::reinterpret_borrow<py::tuple>(h);
			const Tensor image = from_python(layer[0], "an image workspace"), bg = tensor_from_python(layer[1], "a background");
			if (present(image) && (image.numel() != bytes || image.scalar_type() != at::kByte || !image.is_contiguous() ||
			                       image.device() != planes[0].device()))
				throw std::runtime_error("the image workspace is not that of such an image");
			if (!known.background.defined())
				known.background = bg;
			one_background = one_background && bg.data_ptr() == known.background.data_ptr();
			known.images.push_back(image);
		}
		if (known.images.size() != K)
			throw std::runtime_error("the strips of every layer are needed");
		if (!one_background || known.background.numel() != 3 || known.background.scalar_type() != at::kFloat ||
		    known.background.device() != planes[0].device() || !known.background.is_contiguous())
			known = LayerStrips();
	}
	variable_list out;
	{
		py::gil_scoped_release no_gil;
		out = Composite::apply(at::TensorList(planes), &background, &known);
	}
	return py::make_tuple(out[0], out[1], out[2]);
}

// ---- rasterizer --------------------------------------------------------------------------------------------------

// A GaussianRasterizationSettings.
struct Settings {
	int64_t H, W;
	double tanfovx, tanfovy;
	Tensor bg;
	double scale_modifier;
	Tensor view, proj, proj_inv, low, up;
	int sh_degree;
	Tensor campos;
	bool prefiltered, debug;
};

bool truth(py::handle h)
{
	const int v = PyObject_IsTrue(h.ptr());
	if (v < 0)
		throw py::error_already_set();
	return v != 0;
}

Settings settings_from_python(py::handle s)
{
	Settings r;
	r.H = py::cast<int64_t>(py::int_(s.attr("image_height")));
	r.W = py::cast<int64_t>(py::int_(s.attr("image_width")));
	r.tanfovx = py::cast<double>(py::float_(s.attr("tanfovx")));
	r.tanfovy = py::cast<double>(py::float_(s.attr("tanfovy")));
	r.bg = tensor_from_python(s.attr("bg"), "bg");
	r.scale_modifier = py::cast<double>(py::float_(s.attr("scale_modifier")));
	r.view = tensor_from_python(s.attr("viewmatrix"), "viewmatrix");
	r.proj = tensor_from_python(s.attr("projmatrix"), "projmatrix");
	r.proj_inv = tensor_from_python(s.attr("projmatrix_inv"), "projmatrix_inv");
	r.low = tensor_from_python(s.attr("range_low"), "range_low");
	r.up = tensor_from_python(s.attr("range_up"), "range_up");
	r.sh_degree = static_cast<int>(py::cast<int64_t>(py::int_(s.attr("sh_degree"))));
	r.campos = tensor_from_python(s.attr("campos"), "campos");
	r.prefiltered = truth(s.attr("prefiltered"));
	r.debug = truth(s.attr("debug"));
	return r;
}

// A layer's inputs in the order of GaussianRasterizer's autograd function.
enum Input { kMeans3D, kMeans2D, kSH, kColors, kOpacities, kScales, kRotations, kCov3D, kInputs };
const char* const kInputNames[kInputs] = {"means3D", "means2D", "sh", "colors_precomp", "opacities", "scales", "rotations",
                                          "cov3Ds_precomp"};

int sh_rows(const Tensor& sh) { return present(sh) ? static_cast<int>(sh.size(1)) : 0; }

void check_means(const Tensor& means3D)
{
	if (!means3D.defined() || means3D.dim() != 2 || means3D.size(1) != 3)
		throw std::runtime_error("means3D must have dimensions (num_points, 3)");
	if (!means3D.is_cuda())
		throw std::runtime_error("the rasterizer needs its inputs on a GPU (device memory)");
}

// What the first half of a forward call leaves behind: the geometry workspace, the radii and the place where the instance
// count lands.  Made by GaussianRasterizer.enqueue_geometry, consumed once by GaussianRasterizer.forward.
struct GeometryStage {
	at::Device device{at::kCPU};
	hipStream_t stream = nullptr;
	int64_t P = 0, H = 0, W = 0;
	Settings s;  // its tensors on the device
	std::array<Tensor, kInputs> in;
	Tensor radii, geom;
	const void* source = nullptr;
	std::atomic<bool> used{false};
	std::optional<int64_t> bound, count;
	bool in_flight = false;
	CountSlot slot;
	std::mutex count_mutex;  // several threads may ask for the count, without the interpreter lock
	py::object settings;     // of a stage that Python holds

	GeometryStage() = default;
	GeometryStage(const GeometryStage&) = delete;
	GeometryStage& operator=(const GeometryStage&) = delete;
	~GeometryStage()
	{
		if (in_flight)
			slot_pool().give_back_in_flight(device.index(), slot);
	}

	// The number of (Gaussian, tile) instances; waits for it if it is still on its way.
	int64_t instances()
	{
		std::lock_guard<std::mutex> lock(count_mutex);
		if (!count) {
			if (!in_flight)
				throw std::runtime_error("this stage has no instance count");
			if (hipEventSynchronize(slot.event) != hipSuccess)
				throw std::runtime_error("waiting for the instance count failed");
			count = slot.words[0];
			in_flight = false;
			slot_pool().give_back(device.index(), slot);
		}
		return *count;
	}
};

// First half of RasterizeGaussiansCUDA_hgs (K/rasterize_points.cu:35-125): argument checks, the geometry workspace,
// per-Gaussian preprocess and the instance count, which with wait = false is still on its way when this returns.
void run_geometry(GeometryStage& g, const Settings& s, const std::array<Tensor, kInputs>& in, bool wait)
{
	check_means(in[kMeans3D]);
	const at::Device device = in[kMeans3D].device();
	g.device = device;
	g.source = in[kMeans3D].data_ptr();
	g.P = in[kMeans3D].size(0);
	g.H = s.H;
	g.W = s.W;
	g.stream = current_stream(device);
	g.s = s;
	for (Tensor* t : {&g.s.bg, &g.s.view, &g.s.proj, &g.s.proj_inv, &g.s.low, &g.s.up, &g.s.campos})
		*t = device_f32(*t, device);
	for (int k = 0; k < kInputs; k++)
		if (k != kMeans2D)
			g.in[k] = device_f32(in[k], device);
	g.radii = at::empty({g.P}, at::TensorOptions().dtype(at::kInt).device(device));
	if (g.P == 0) {
		g.geom = new_bytes(0, device);
		g.count = 0;
		return;
	}
	c10::DeviceGuard guard(device);
	const size_t bytes = rgs_geom_bytes(g.P);
	g.geom = new_bytes(bytes, device);
	const CountSlot slot = slot_pool().take(device.index());
	const auto& t = g.in;
	auto run = [&](auto entry, auto... tail) {
		return entry(g.P, s.sh_degree, sh_rows(t[kSH]), g.W, g.H, ptr(t[kMeans3D]), ptr(t[kSH]), ptr(t[kColors]), ptr(t[kOpacities]),
		             ptr(t[kScales]), s.scale_modifier, ptr(t[kRotations]), ptr(t[kCov3D]), ptr(g.s.view), ptr(g.s.proj),
		             ptr(g.s.campos), s.tanfovx, s.tanfovy, s.prefiltered, ptr<int>(g.radii), ptr<void>(g.geom), bytes, slot.words,
		             tail..., g.stream, s.debug);
	};
	const int rc = wait ? run(rgs_forward_geom) : run(rgs_forward_geom_enqueue, static_cast<void*>(slot.event));
	if (rc != 0 || wait) {
		// on an error the count may have been asked for all the same: the stream is behind it before the words go to another call
		if (rc != 0)
			(void)hipStreamSynchronize(g.stream);
		const uint32_t n = slot.words[0];
		slot_pool().give_back(device.index(), slot);
		check(rc);
		g.count = n;
		return;
	}
	g.slot = slot;
	g.in_flight = true;
}

struct Rendered {
	int64_t instances = 0;
	Tensor package, color, depth, alpha, binning, image;
};

// One (5,H,W) block: colour, depth, accumulated alpha in the order in which the reference packs a partial image for
// transport (RenderResult.zip_content, parallel_utils/basic_parallel_trainer/task_utils.py:156-163).
void make_package(Rendered& r, int64_t H, int64_t W, const at::Device& device)
{
	r.package = new_f32({5, H, W}, device);
	r.color = r.package.narrow(0, 0, 3);
	r.depth = r.package.narrow(0, 3, 1);
	r.alpha = r.package.narrow(0, 4, 1);
}

// Second half: waits for the instance count if it is still on its way, sizes the binning workspace with it, sorts and blends.
Rendered run_raster(GeometryStage& g)
{
	if (g.used.exchange(true))
		throw std::runtime_error("this geometry stage has already been consumed");
	if (current_stream(g.device) != g.stream)
		throw std::runtime_error("the geometry stage was enqueued on another stream than the one current now");
	Rendered r;
	make_package(r, g.H, g.W, g.device);
	if (g.P == 0) {
		r.package.zero_();
		r.binning = new_bytes(0, g.device);
		r.image = new_bytes(0, g.device);
		return r;
	}
	c10::DeviceGuard guard(g.device);
	const size_t image_bytes = rgs_image_bytes(g.W, g.H);
	r.image = new_bytes(image_bytes, g.device);
	// with a bound there is no wait: the kernels read the count on the device; the caller checks it afterwards
	r.instances = g.bound ? *g.bound : g.instances();
	if (r.instances >= int64_t(1) << 30)
		throw LibraryError(std::to_string(r.instances) + " (Gaussian, tile) instances exceed the 2^30 limit of the sort");
	const size_t binning_bytes = r.instances > 0 ? rgs_binning_bytes(r.instances) : 0;
	r.binning = new_bytes(binning_bytes, g.device);
	check((g.bound ? rgs_forward_raster_bounded : rgs_forward_raster)(
	    g.P, r.instances, g.W, g.H, ptr(g.s.bg), g.s.tanfovx, g.s.tanfovy, ptr(g.s.proj_inv), ptr(g.s.low), ptr(g.s.up),
	    ptr(g.in[kColors]), ptr<int>(g.radii), ptr<void>(g.geom), g.geom.numel(), ptr<void>(r.binning), binning_bytes,
	    ptr<void>(r.image), image_bytes, ptr(r.color), ptr(r.depth), ptr(r.alpha), g.stream, g.s.debug));
	return r;
}

// ---- gradient arrays ---------------------------------------------------------------------------------------------

enum Gradient { kGradMeans2D, kGradOpacity, kGradColors, kGradMeans3D, kGradCov3D, kGradSH, kGradScales, kGradRotations, kGradients };
const char* const kGradientNames[kGradients] = {"means2D", "opacity", "colors", "means3D", "cov3D", "sh", "scales", "rotations"};
constexpr int kSumFloats = 12;  // per Gaussian, the sums of the blend's backward

struct GradientArrays {
	std::array<Tensor, kGradients> g;
	Tensor sums;
};

// The gradient arrays of a layer but for those that are left out, each an allocation of its own: a gradient that the caller keeps
// holds no other.
GradientArrays new_gradients(int64_t P, int64_t M, const at::Device& device, const std::array<bool, kGradients>& left_out)
{
	const std::array<std::vector<int64_t>, kGradients> shapes = {{{P, 3}, {P, 1}, {P, 3}, {P, 3}, {P, 6}, {P, M, 3}, {P, 3}, {P, 4}}};
	GradientArrays r;
	for (int k = 0; k < kGradients; k++)
		if (!left_out[k])
			r.g[k] = new_f32(shapes[k], device);
	r.sums = new_f32({P, kSumFloats}, device);
	return r;
}

py::dict gradient_outputs(int64_t P, int64_t M, py::handle device_object, py::handle scratch)
{
	const at::Device device = THPDevice_Check(device_object.ptr()) ? reinterpret_cast<THPDevice*>(device_object.ptr())->device
	                                                               : at::Device(py::cast<std::string>(device_object));
	std::array<bool, kGradients> left_out;
	for (int k = 0; k < kGradients; k++)
		left_out[k] = scratch.contains(kGradientNames[k]);
	const GradientArrays made = new_gradients(P, M, device, left_out);
	py::dict out;
	for (int k = 0; k < kGradients; k++)
		out[kGradientNames[k]] = to_python(made.g[k]);
	out["sums"] = made.sums;
	return out;
}

py::handle rasterizer_module()
{
	// (under the interpreter lock, which the import may hand to another thread: a static initialised by the import would have
	// that thread wait for it while it holds the lock)
	static PyObject* module = nullptr;
	if (!module) {
		PyObject* imported = PyImport_ImportModule("retinags_amd.rasterizer");
		if (!imported)
			throw py::error_already_set();
		module = imported;
	}
	return module;
}

// _gradient_outputs of that module as it was when the module was imported.
PyObject* original_gradient_outputs = nullptr;
void set_original_gradient_outputs(py::object f) { original_gradient_outputs = f.release().ptr(); }

// The gradient arrays of a layer: made here, or by the module's function of that name where another has been put in its place.
GradientArrays make_gradients(int64_t P, int64_t M, const at::Device& device, const std::array<bool, kGradients>& left_out)
{
	{
		py::gil_scoped_acquire gil;
		const py::object f = rasterizer_module().attr("_gradient_outputs");
		if (f.ptr() != original_gradient_outputs) {
			py::list scratch;
			for (int k = 0; k < kGradients; k++)
				if (left_out[k])
					scratch.append(kGradientNames[k]);
			const py::object made = f(P, M, py::reinterpret_steal<py::object>(THPDevice_New(device)), py::arg("scratch") = py::tuple(scratch));
			GradientArrays r;
			for (int k = 0; k < kGradients; k++)
				r.g[k] = from_python(made[kGradientNames[k]], kGradientNames[k]);
			r.sums = tensor_from_python(made["sums"], "sums");
			return r;
		}
	}
	return new_gradients(P, M, device, left_out);
}

// The gradients of a layer without Gaussians.
GradientArrays empty_gradients(int64_t M, const at::Device& device)
{
	GradientArrays r;
	const std::array<std::vector<int64_t>, kGradients> shapes = {{{0, 3}, {0, 1}, {0, 3}, {0, 3}, {0, 6}, {0, M, 3}, {0, 3}, {0, 4}}};
	for (int k = 0; k < kGradients; k++)
		r.g[k] = new_f32(shapes[k], device);
	return r;
}

// Gradients in the order of the inputs; none for inputs that were absent.
void gradients_of_inputs(variable_list& out, size_t at, const GradientArrays& r, bool sh, bool colors, bool scales, bool rotations,
                         bool cov3D)
{
	out[at + kMeans3D] = r.g[kGradMeans3D];
	out[at + kMeans2D] = r.g[kGradMeans2D];
	out[at + kSH] = sh ? r.g[kGradSH] : Tensor();
	out[at + kColors] = colors ? r.g[kGradColors] : Tensor();
	out[at + kOpacities] = r.g[kGradOpacity];
	out[at + kScales] = scales ? r.g[kGradScales] : Tensor();
	out[at + kRotations] = rotations ? r.g[kGradRotations] : Tensor();
	out[at + kCov3D] = cov3D ? r.g[kGradCov3D] : Tensor();
}

// What a layer's backward reads, in the order in which it is saved.
enum Saved { kSavedColors, kSavedMeans3D, kSavedScales, kSavedRotations, kSavedCov3D, kSavedRadii, kSavedSH, kSavedGeom, kSavedBinning,
             kSavedImage, kSavedAlpha, kSavedPerLayer };

// ---- one call ----------------------------------------------------------------------------------------------------

struct Call : torch::CustomClassHolder {
	Settings s;  // as given
	GeometryStage* stage = nullptr;  // during the forward: a stage that is already on its way
	Rendered rendered;
};

// `grads`: of the colour, of nothing, of the depth and of the alpha image; those that are not defined or empty are null pointers.
GradientArrays gradients_of_call(const Settings& s, int64_t instances, const variable_list& saved, const variable_list& grads)
{
	const Tensor& means3D = saved[kSavedMeans3D];
	const at::Device device = means3D.device();
	const int64_t P = means3D.size(0), H = s.H, W = s.W;
	const int M = sh_rows(saved[kSavedSH]);
	GradientArrays out;
	if (P == 0) {
		out = empty_gradients(M, device);
	} else {
		out = make_gradients(P, M, device, {});
		c10::DeviceGuard guard(device);
		const Tensor g_color = grads[0].defined() ? device_f32(grads[0], device) : new_f32({3, H, W}, device).zero_();
		const Tensor g_depth = device_f32(grads[2], device), g_alpha = device_f32(grads[3], device);
		const Tensor bg = device_f32(s.bg, device), view = device_f32(s.view, device), proj = device_f32(s.proj, device),
		             proj_inv = device_f32(s.proj_inv, device), low = device_f32(s.low, device), up = device_f32(s.up, device),
		             campos = device_f32(s.campos, device);
		auto g = [&](int k) { return ptr(out.g[k]); };
		check(rgs_backward(P, s.sh_degree, M, instances, W, H, ptr(bg), ptr(means3D), ptr(saved[kSavedSH]),
		                   ptr(saved[kSavedColors]), ptr(saved[kSavedAlpha]), ptr(saved[kSavedScales]), s.scale_modifier,
		                   ptr(saved[kSavedRotations]), ptr(saved[kSavedCov3D]), ptr(view), ptr(proj), ptr(proj_inv), ptr(low), ptr(up),
		                   ptr(campos), s.tanfovx, s.tanfovy, ptr<int>(saved[kSavedRadii]), ptr<void>(saved[kSavedGeom]),
		                   ptr<void>(saved[kSavedBinning]), ptr<void>(saved[kSavedImage]), ptr(g_color), ptr(g_depth), ptr(g_alpha),
		                   ptr(out.sums), g(kGradMeans2D), g(kGradOpacity), g(kGradColors), g(kGradMeans3D), g(kGradCov3D), g(kGradSH),
		                   g(kGradScales), g(kGradRotations), 0, current_stream(device), s.debug));
	}
	return out;
}

variable_list call_backward(const Call& call, const variable_list& saved, const variable_list& grads)
{
	const GradientArrays out = gradients_of_call(call.s, call.rendered.instances, saved, grads);
	variable_list result(kInputs + 1);
	gradients_of_inputs(result, 0, out, present(saved[kSavedSH]), present(saved[kSavedColors]), present(saved[kSavedScales]),
	                    present(saved[kSavedRotations]), present(saved[kSavedCov3D]));
	return result;
}

// K/diff_gaussian_rasterization_half_gaussian/__init__.py:44-164.  Outputs colour, radii, depth, alpha.
struct RasterizeCall : torch::autograd::Function<RasterizeCall> {
	static variable_list forward(AutogradContext* ctx, at::TensorList in, const c10::intrusive_ptr<Call>* held)
	{
		Call& call = **held;
		GeometryStage own;
		GeometryStage& stage = call.stage ? *call.stage : own;
		if (!call.stage) {
			std::array<Tensor, kInputs> inputs;
			std::copy(in.begin(), in.end(), inputs.begin());
			run_geometry(stage, call.s, inputs, true);
		}
		call.rendered = run_raster(stage);
		Rendered& r = call.rendered;
		ctx->set_materialize_grads(false);  // an output that took no part in the loss comes back undefined
		ctx->save_for_backward({stage.in[kColors], stage.in[kMeans3D], stage.in[kScales], stage.in[kRotations], stage.in[kCov3D],
		                        stage.radii, stage.in[kSH], stage.geom, r.binning, r.image, r.alpha});
		ctx->mark_non_differentiable({stage.radii});
		ctx->saved_data["call"] = c10::IValue::make_capsule(*held);
		const variable_list out = {r.color, stage.radii, r.depth, r.alpha};
		const int64_t instances = r.instances;
		r = Rendered();
		r.instances = instances;
		return out;
	}

	static variable_list backward(AutogradContext* ctx, variable_list grads)
	{
		return in_backward([&]() -> variable_list {
			const auto holder = ctx->saved_data["call"].toCapsule();
			const Call& call = static_cast<const Call&>(*holder);
			const variable_list saved = ctx->get_saved_variables();
			if (!call.s.debug)
				return call_backward(call, saved, grads);
			py::gil_scoped_acquire gil;
			const Settings& s = call.s;
			auto given = [](const Tensor& t) { return t.defined() ? t : at::empty({0}); };
			auto sv = [&](int k) { return to_python(saved[k]); };
			py::tuple args = py::make_tuple(
			    s.bg, sv(kSavedMeans3D), sv(kSavedRadii), sv(kSavedColors), sv(kSavedScales), sv(kSavedRotations), s.scale_modifier,
			    sv(kSavedCov3D), s.view, s.proj, s.proj_inv, s.low, s.up, s.tanfovx, s.tanfovy, given(grads[0]), given(grads[2]),
			    given(grads[3]), sv(kSavedSH), s.sh_degree, s.campos, sv(kSavedGeom), call.rendered.instances, sv(kSavedBinning),
			    sv(kSavedImage), sv(kSavedAlpha), s.debug);
			variable_list result;
			py::cpp_function run([&] {
				py::gil_scoped_release no_gil;
				result = call_backward(call, saved, grads);
			});
			rasterizer_module().attr("_backward_in_debug")(args, run);
			return result;
		});
	}
};

// An absent input comes as an empty tensor; only the placeholder for the screen-space gradient, whose values nobody reads, may be None.
std::array<Tensor, kInputs> inputs_from_python(const py::handle* given)
{
	std::array<Tensor, kInputs> in;
	for (int k = 0; k < kInputs; k++) {
		if (k != kMeans2D)
			in[k] = tensor_from_python(given[k], kInputNames[k]);
		else if (THPVariable_Check(given[k].ptr()))
			in[k] = THPVariable_Unpack(given[k].ptr());
		else
			in[k] = at::empty({0});
	}
	return in;
}

void check_stage(const GeometryStage& g, const Tensor& means3D, py::handle settings)
{
	if (g.source != means3D.data_ptr() || g.P != means3D.size(0) || g.settings.ptr() != settings.ptr() || g.used)
		throw std::runtime_error("the geometry stage was enqueued for other inputs or settings, or already used");
}

py::tuple rasterize(py::handle means3D, py::handle means2D, py::handle sh, py::handle colors, py::handle opacities, py::handle scales,
                    py::handle rotations, py::handle cov3D, py::handle settings, py::handle geometry)
{
	const py::handle given[kInputs] = {means3D, means2D, sh, colors, opacities, scales, rotations, cov3D};
	const std::array<Tensor, kInputs> in = inputs_from_python(given);
	auto call = c10::make_intrusive<Call>();
	call->s = settings_from_python(settings);
	if (!geometry.is_none()) {
		call->stage = &py::cast<GeometryStage&>(geometry);
		check_stage(*call->stage, in[kMeans3D], settings);
	}
	variable_list out;
	{
		py::gil_scoped_release no_gil;
		out = RasterizeCall::apply(at::TensorList(in.data(), in.size()), &call);
		call->stage = nullptr;
	}
	return py::make_tuple(out[0], out[1], out[2], out[3]);
}

std::unique_ptr<GeometryStage> enqueue_geometry(py::handle means3D, py::handle sh, py::handle colors, py::handle opacities,
                                                py::handle scales, py::handle rotations, py::handle cov3D, py::handle settings,
                                                std::optional<int64_t> bound)
{
	const py::none none;
	const py::handle given[kInputs] = {means3D, none, sh, colors, opacities, scales, rotations, cov3D};
	const std::array<Tensor, kInputs> in = inputs_from_python(given);
	const Settings s = settings_from_python(settings);
	auto stage = std::make_unique<GeometryStage>();
	{
		py::gil_scoped_release no_gil;
		at::NoGradGuard no_grad;
		run_geometry(*stage, s, in, false);
	}
	stage->settings = py::reinterpret_borrow<py::object>(settings);
	stage->bound = bound;
	return stage;
}

// RasterizeGaussiansCUDA_hgs (K/rasterize_points.cu:35-125): its arguments in its order, its 8-tuple.
py::tuple rasterize_forward(Tensor bg, py::handle means3D, py::handle colors, py::handle opacities, py::handle scales,
                            py::handle rotations, double scale_modifier, py::handle cov3D, Tensor view, Tensor proj, Tensor proj_inv,
                            Tensor low, Tensor up, double tanfovx, double tanfovy, int64_t H, int64_t W, py::handle sh, int sh_degree,
                            Tensor campos, bool prefiltered, bool debug)
{
	const py::none none;
	const py::handle given[kInputs] = {means3D, none, sh, colors, opacities, scales, rotations, cov3D};
	const std::array<Tensor, kInputs> in = inputs_from_python(given);
	const Settings s = {H,  W,        tanfovx, tanfovy, bg,     scale_modifier, view, proj, proj_inv,
	                    low, up, sh_degree, campos,  prefiltered, debug};
	GeometryStage stage;
	Rendered r;
	{
		py::gil_scoped_release no_gil;
		at::NoGradGuard no_grad;
		run_geometry(stage, s, in, true);
		r = run_raster(stage);
	}
	return py::make_tuple(r.instances, r.color, r.depth, r.alpha, stage.radii, stage.geom, r.binning, r.image);
}

// The same 8-tuple from a stage that is already on its way.
py::tuple rasterize_forward_from_stage(GeometryStage& stage, const Tensor& means3D, py::handle settings)
{
	check_stage(stage, means3D, settings);
	Rendered r;
	{
		py::gil_scoped_release no_gil;
		at::NoGradGuard no_grad;
		r = run_raster(stage);
	}
	return py::make_tuple(r.instances, r.color, r.depth, r.alpha, stage.radii, stage.geom, r.binning, r.image);
}

// RasterizeGaussiansBackwardCUDA_hgs (K/rasterize_points.cu:127-220): its arguments in its order, its 8 tensors.
py::tuple rasterize_backward(Tensor bg, Tensor means3D, Tensor radii, Tensor colors, Tensor scales, Tensor rotations, double scale_modifier,
                             Tensor cov3D, Tensor view, Tensor proj, Tensor proj_inv, Tensor low, Tensor up, double tanfovx, double tanfovy,
                             Tensor grad_color, Tensor grad_depth, Tensor grad_alpha, Tensor sh, int sh_degree, Tensor campos, Tensor geom,
                             int64_t instances, Tensor binning, Tensor image, Tensor alpha, bool debug)
{
	check_means(means3D);
	if (grad_color.dim() != 3 || grad_color.size(0) != 3)
		throw std::runtime_error("grad_color must have dimensions (3, height, width)");
	const at::Device device = means3D.device();
	const Settings s = {grad_color.size(1), grad_color.size(2), tanfovx, tanfovy,   bg,     scale_modifier, view, proj, proj_inv,
	                    low,                up,                 sh_degree, campos, false, debug};
	GradientArrays out;
	{
		py::gil_scoped_release no_gil;
		at::NoGradGuard no_grad;
		auto f = [&](const Tensor& t) { return device_f32(t, device); };
		out = gradients_of_call(s, instances, {f(colors), f(means3D), f(scales), f(rotations), f(cov3D), radii, f(sh), geom, binning, image, f(alpha)},
		                        {grad_color, Tensor(), grad_depth, grad_alpha});
	}
	const auto& g = out.g;
	return py::make_tuple(g[kGradMeans2D], g[kGradColors], g[kGradOpacity], g[kGradMeans3D], g[kGradCov3D], g[kGradSH], g[kGradScales],
	                      g[kGradRotations]);
}

// ---- the layers of a frame together ------------------------------------------------------------------------------

struct FrameLayer {
	Settings s;  // as given
	hipStream_t side = nullptr;
	int64_t P = 0;
	int M = 0;
	Rendered rendered;
	Tensor radii, geom;
	Tensor image, background;  // see Frame::keep_strips
};

struct Frame : torch::CustomClassHolder {
	std::vector<FrameLayer> layers;
	bool keep_workspaces = false;
	bool keep_strips = false;  // the image workspaces, and the backgrounds as the library saw them, for the compositor
	bool split_sh = false;     // SH rows in parts: see rgs_frame_layer::sh_rest
};

// The parts of a layer's SH rows beside the first coefficients.
enum SplitInput { kSplitRest, kSplitLent, kSplitInputs };

// The submodels that a camera sees ("layers"), rasterized together: what the reference does with one call per submodel
// (gather_RenderResult_pool, parallel_utils/basic_parallel_trainer/result_aggregator.py:22-38), as three library calls per
// frame (every layer's geometry stage, then binning and one blend launch for all, and for the backward one blend launch for
// all and every layer's per-Gaussian backward).  `flat`: kInputs tensors per layer, then, with SH rows in parts, kSplitInputs per layer
// (kSH then holds the first coefficients).  Outputs per layer colour, radii, depth, alpha.
struct RasterizeFrame : torch::autograd::Function<RasterizeFrame> {
	static rgs_frame_view view_of(const Settings& s, const std::array<Tensor, 4>& t)
	{
		return {static_cast<int>(s.W), static_cast<int>(s.H), static_cast<float>(s.tanfovx), static_cast<float>(s.tanfovy),
		        ptr(t[0]),             ptr(t[1]),             ptr(t[2]),                     ptr(t[3])};
	}

	static std::array<Tensor, 4> view_tensors(const Settings& s, const at::Device& device)
	{
		return {device_f32(s.view, device), device_f32(s.proj, device), device_f32(s.proj_inv, device), device_f32(s.campos, device)};
	}

	static variable_list forward(AutogradContext* ctx, at::TensorList flat, const c10::intrusive_ptr<Frame>* held)
	{
		Frame& frame = **held;
		const int K = static_cast<int>(frame.layers.size());
		const Settings& s0 = frame.layers[0].s;
		const int64_t H = s0.H, W = s0.W;
		const at::Device device = flat[0].device();
		if (!flat[0].is_cuda())
			throw std::runtime_error("the rasterizer needs its inputs on a GPU (device memory)");
		c10::DeviceGuard guard(device);
		const hipStream_t main = current_stream(device);
		const std::array<Tensor, 4> vt = view_tensors(s0, device);
		const rgs_frame_view view = view_of(s0, vt);
		const size_t image_bytes = rgs_image_bytes(W, H);
		std::vector<rgs_frame_layer> arr;
		std::vector<int> live;
		arr.reserve(K);
		variable_list saved, out, radii, keep, split;
		saved.reserve(K * (kSavedPerLayer + kSplitInputs));
		out.reserve(4 * K);
		for (int k = 0; k < K; k++) {
			FrameLayer& l = frame.layers[k];
			if (l.s.H != H || l.s.W != W)
				throw std::runtime_error("rasterize_frame: the layers of a frame share one image size");
			std::array<Tensor, kInputs> t;
			for (int i = 0; i < kInputs; i++)
				t[i] = i == kMeans2D ? Tensor() : device_f32(flat[kInputs * k + i], device);
			check_means(flat[kInputs * k + kMeans3D]);
			l.P = t[kMeans3D].size(0);
			l.M = sh_rows(t[kSH]);
			std::array<Tensor, kSplitInputs> parts;
			if (frame.split_sh) {
				for (int i = 0; i < kSplitInputs; i++)
					parts[i] = device_f32(flat[kInputs * K + kSplitInputs * k + i], device);
				const int64_t own = t[kSH].dim() == 3 ? t[kSH].size(0) : 0;
				if (own < 1 || t[kSH].sizes() != at::IntArrayRef({own, 1, 3}) || parts[kSplitRest].sizes() != at::IntArrayRef({own, 15, 3}) ||
				    parts[kSplitLent].sizes() != at::IntArrayRef({l.P - own, 16, 3}))
					throw std::runtime_error("rasterize_frame: SH rows in parts are (N,1,3), (N,15,3) and (P-N,16,3) with N >= 1");
				l.M = 16;
				split.insert(split.end(), parts.begin(), parts.end());
			}
			Rendered& r = l.rendered;
			make_package(r, H, W, device);
			l.radii = at::empty({l.P}, at::TensorOptions().dtype(at::kInt).device(device));
			radii.push_back(l.radii);
			if (l.P == 0) {
				r.package.zero_();
				l.geom = new_bytes(0, device);
				r.image = new_bytes(0, device);
				r.binning = new_bytes(0, device);
			} else {
				live.push_back(k);
				arr.emplace_back();
				rgs_frame_layer& L = arr.back();
				const Tensor bg = device_f32(l.s.bg, device), low = device_f32(l.s.low, device), up = device_f32(l.s.up, device);
				keep.insert(keep.end(), {bg, low, up, t[kOpacities]});
				l.background = bg;
				const size_t geom_bytes = rgs_geom_bytes(l.P);
				l.geom = new_bytes(geom_bytes, device);
				r.image = new_bytes(image_bytes, device);
				L.P = l.P;
				L.D = l.s.sh_degree;
				L.M = l.M;
				L.means3D = ptr(t[kMeans3D]);
				L.shs = ptr(t[kSH]);
				if (frame.split_sh) {
					L.sh_rest = ptr(parts[kSplitRest]);
					L.sh_lent = ptr(parts[kSplitLent]);
					L.sh_own = static_cast<int>(t[kSH].size(0));
				}
				L.colors_precomp = ptr(t[kColors]);
				L.opacities = ptr(t[kOpacities]);
				L.scales = ptr(t[kScales]);
				L.rotations = ptr(t[kRotations]);
				L.cov3D_precomp = ptr(t[kCov3D]);
				L.scale_modifier = l.s.scale_modifier;
				L.background = ptr(bg);
				L.range_low = ptr(low);
				L.range_up = ptr(up);
				L.radii = ptr<int>(l.radii);
				L.geom_ws = ptr<void>(l.geom);
				L.image_ws = ptr<void>(r.image);
				L.geom_bytes = geom_bytes;
				L.image_bytes = image_bytes;
				L.out_color = ptr(r.package);
				L.out_depth = L.out_color + 3 * H * W;
				L.out_alpha = L.out_color + 4 * H * W;
			}
			saved.insert(saved.end(), {t[kColors], t[kMeans3D], t[kScales], t[kRotations], t[kCov3D], l.radii, t[kSH], l.geom, r.binning,
			                           r.image, r.alpha});
			out.insert(out.end(), {r.color, l.radii, r.depth, r.alpha});
		}
		const int n = static_cast<int>(live.size());
		if (n != 0) {
			const CountSlot slot = slot_pool().take(device.index());
			const int rc = rgs_frame_forward_geom(n, arr.data(), &view, slot.words, main, s0.debug);
			if (rc != 0)
				(void)hipStreamSynchronize(main);  // as in run_geometry
			std::array<uint32_t, RGS_MAX_FRAME_LAYERS> counts;
			std::copy(slot.words, slot.words + n, counts.begin());
			slot_pool().give_back(device.index(), slot);
			check(rc);
			for (int j = 0; j < n; j++) {
				Rendered& r = frame.layers[live[j]].rendered;
				r.instances = counts[j];
				const size_t bytes = counts[j] > 0 ? rgs_binning_bytes(counts[j]) : 0;
				r.binning = new_bytes(bytes, device);
				saved[live[j] * kSavedPerLayer + kSavedBinning] = r.binning;
				arr[j].R = counts[j];
				arr[j].binning_ws = ptr<void>(r.binning);
				arr[j].binning_bytes = bytes;
			}
			check(rgs_frame_forward_raster(n, arr.data(), &view, main, s0.debug));
		}
		if (frame.keep_strips)
			for (int k : live)
				frame.layers[k].image = frame.layers[k].rendered.image;
		ctx->set_materialize_grads(false);  // an output that took no part in the loss comes back undefined
		saved.insert(saved.end(), split.begin(), split.end());
		ctx->save_for_backward(std::move(saved));
		ctx->mark_non_differentiable(radii);
		ctx->saved_data["frame"] = c10::IValue::make_capsule(*held);
		for (FrameLayer& l : frame.layers) {
			// what the backward needs of these is saved above, where autograd can give it back
			Rendered left;
			left.instances = l.rendered.instances;
			if (frame.keep_workspaces) {
				left.binning = l.rendered.binning;
				left.image = l.rendered.image;
			} else {
				l.geom = Tensor();
			}
			l.radii = Tensor();
			l.rendered = left;
		}
		return out;
	}

	static variable_list backward(AutogradContext* ctx, variable_list grads)
	{
		return in_backward([&]() -> variable_list {
			const auto holder = ctx->saved_data["frame"].toCapsule();
			const Frame& frame = static_cast<const Frame&>(*holder);
			const int K = static_cast<int>(frame.layers.size());
			const variable_list saved = ctx->get_saved_variables();
			const Settings& s0 = frame.layers[0].s;
			const int64_t H = s0.H, W = s0.W;
			const at::Device device = saved[kSavedMeans3D].device();
			c10::DeviceGuard guard(device);
			const hipStream_t main = current_stream(device);
			auto sv = [&](int k, int i) -> const Tensor& { return saved[k * kSavedPerLayer + i]; };
			std::vector<GradientArrays> made(K);
			variable_list split_grads(frame.split_sh ? K * kSplitInputs : 0);
			for (int k = 0; k < K; k++) {
				if (frame.layers[k].P == 0)
					continue;
				// arrays nobody gets to see are not made: the colour gradient when the colours come from SH, the covariance
				// gradient when it comes from scale and rotation
				std::array<bool, kGradients> left_out{};
				left_out[kGradColors] = !present(sv(k, kSavedColors));
				left_out[kGradCov3D] = !present(sv(k, kSavedCov3D));
				left_out[kGradSH] = frame.split_sh;
				made[k] = make_gradients(frame.layers[k].P, frame.layers[k].M, device, left_out);
				if (frame.split_sh) {
					made[k].g[kGradSH] = new_f32(sv(k, kSavedSH).sizes(), device);
					for (int i = 0; i < kSplitInputs; i++)
						split_grads[kSplitInputs * k + i] = new_f32(saved[kSavedPerLayer * K + kSplitInputs * k + i].sizes(), device);
				}
			}
			const std::array<Tensor, 4> vt = view_tensors(s0, device);
			const rgs_frame_view view = view_of(s0, vt);
			std::vector<rgs_frame_layer> arr;
			arr.reserve(K);
			variable_list keep, out(K * kInputs + split_grads.size() + 1);
			std::copy(split_grads.begin(), split_grads.end(), out.begin() + K * kInputs);
			for (int k = 0; k < K; k++) {
				const FrameLayer& l = frame.layers[k];
				if (l.P == 0) {
					made[k] = empty_gradients(l.M, device);
				} else {
					const Tensor &gc = grads[4 * k], &gd = grads[4 * k + 2], &ga = grads[4 * k + 3];
					const Tensor g_color = gc.defined() ? device_f32(gc, device) : new_f32({3, H, W}, device).zero_();
					const Tensor g_depth = device_f32(gd, device), g_alpha = device_f32(ga, device), bg = device_f32(l.s.bg, device),
					             low = device_f32(l.s.low, device), up = device_f32(l.s.up, device);
					keep.insert(keep.end(), {g_color, g_depth, g_alpha, bg, low, up});
					arr.emplace_back();
					rgs_frame_layer& L = arr.back();
					L.P = l.P;
					L.D = l.s.sh_degree;
					L.M = l.M;
					L.R = l.rendered.instances;
					L.means3D = ptr(sv(k, kSavedMeans3D));
					L.shs = ptr(sv(k, kSavedSH));
					if (frame.split_sh) {
						const Tensor* parts = &saved[kSavedPerLayer * K + kSplitInputs * k];
						L.sh_rest = ptr(parts[kSplitRest]);
						L.sh_lent = ptr(parts[kSplitLent]);
						L.sh_own = static_cast<int>(sv(k, kSavedSH).size(0));
						L.dL_dsh_rest = ptr(split_grads[kSplitInputs * k + kSplitRest]);
						L.dL_dsh_lent = ptr(split_grads[kSplitInputs * k + kSplitLent]);
					}
					L.colors_precomp = ptr(sv(k, kSavedColors));
					L.scales = ptr(sv(k, kSavedScales));
					L.rotations = ptr(sv(k, kSavedRotations));
					L.cov3D_precomp = ptr(sv(k, kSavedCov3D));
					L.scale_modifier = l.s.scale_modifier;
					L.background = ptr(bg);
					L.range_low = ptr(low);
					L.range_up = ptr(up);
					L.radii = ptr<int>(sv(k, kSavedRadii));
					L.geom_ws = ptr<void>(sv(k, kSavedGeom));
					L.binning_ws = ptr<void>(sv(k, kSavedBinning));
					L.image_ws = ptr<void>(sv(k, kSavedImage));
					L.out_alpha = ptr(sv(k, kSavedAlpha));
					L.dL_dpix = ptr(g_color);
					L.dL_dpix_depth = ptr(g_depth);
					L.dL_dalphas = ptr(g_alpha);
					const auto& g = made[k].g;
					L.grad_accum = ptr(made[k].sums);
					L.dL_dmean2D = ptr(g[kGradMeans2D]);
					L.dL_dopacity = ptr(g[kGradOpacity]);
					L.dL_dcolor = ptr(g[kGradColors]);
					L.dL_dmean3D = ptr(g[kGradMeans3D]);
					L.dL_dcov3D = ptr(g[kGradCov3D]);
					L.dL_dsh = ptr(g[kGradSH]);
					L.dL_dscale = ptr(g[kGradScales]);
					L.dL_drot = ptr(g[kGradRotations]);
					L.accum_zeroed = 0;  // the library clears the rows of the sums ahead of the blend
					L.stream = l.side != main ? l.side : nullptr;
				}
				gradients_of_inputs(out, k * kInputs, made[k], present(sv(k, kSavedSH)), present(sv(k, kSavedColors)),
				                    present(sv(k, kSavedScales)), present(sv(k, kSavedRotations)), present(sv(k, kSavedCov3D)));
			}
			if (!arr.empty())
				check(rgs_frame_backward(static_cast<int>(arr.size()), arr.data(), &view, main, s0.debug));
			return out;
		});
	}
};

// `inputs`: per layer the kInputs tensors, empty ones for those that are absent.  `streams`: None, or a stream handle per layer.
// `workspaces`: None, or a list that receives (instances, geometry, binning and image workspace) per layer.
// `strips`: None, or a list that receives per layer its image workspace (None for a layer without Gaussians) and its background, which is
// what _host.composite takes under that name.  `split`: None, or per layer the further parts of SH rows whose first coefficients are given
// as the layer's sh: (N,15,3) and, of the Gaussians behind those N, whole rows (P-N,16,3).
py::list rasterize_frame(const py::sequence& settings, const py::sequence& inputs, py::handle streams, py::handle workspaces,
                         py::handle strips, py::handle split)
{
	const size_t K = settings.size();
	if (K == 0 || inputs.size() != kInputs * K)
		throw std::runtime_error("rasterize_frame: one group of eight tensors per layer is needed");
	if (K > RGS_MAX_FRAME_LAYERS)
		throw std::runtime_error("rasterize_frame: at most " + std::to_string(RGS_MAX_FRAME_LAYERS) + " layers");
	auto frame = c10::make_intrusive<Frame>();
	frame->layers.resize(K);
	frame->keep_workspaces = !workspaces.is_none();
	frame->keep_strips = !strips.is_none();
	variable_list flat;
	flat.reserve(K * kInputs);
	for (size_t k = 0; k < K; k++) {
		frame->layers[k].s = settings_from_python(settings[k]);
		if (!streams.is_none())
			frame->layers[k].side = reinterpret_cast<hipStream_t>(py::cast<uintptr_t>(py::reinterpret_borrow<py::sequence>(streams)[k]));
		std::array<py::object, kInputs> held;
		std::array<py::handle, kInputs> given;
		for (int i = 0; i < kInputs; i++)
			given[i] = held[i] = inputs[k * kInputs + i];
		const std::array<Tensor, kInputs> in = inputs_from_python(given.data());
		flat.insert(flat.end(), in.begin(), in.end());
	}
	if (!split.is_none()) {
		frame->split_sh = true;
		for (py::handle h : py::reinterpret_borrow<py::sequence>(split)) {
			const py::tuple parts = py::reinterpret_borrow<py::tuple>(h);
			for (int i = 0; i < kSplitInputs; i++)
				flat.push_back(tensor_from_python(parts[i], "a part of the SH rows"));
		}
		if (flat.size() != (kInputs + kSplitInputs) * K)
			throw std::runtime_error("rasterize_frame: the parts of the SH rows of every layer are needed");
	}
	variable_list out;
	{
		py::gil_scoped_release no_gil;
		out = RasterizeFrame::apply(at::TensorList(flat), &frame);
	}
	if (frame->keep_workspaces)
		for (FrameLayer& l : frame->layers) {
			workspaces.attr("append")(py::make_tuple(l.rendered.instances, l.geom, l.rendered.binning, l.rendered.image));
			l.geom = l.rendered.binning = l.rendered.image = Tensor();
		}
	for (FrameLayer& l : frame->layers) {
		if (frame->keep_strips)
			strips.attr("append")(py::make_tuple(to_python(l.image), l.background.defined() ? l.background : l.s.bg));
		l.image = l.background = Tensor();
	}
	py::list result;
	for (size_t k = 0; k < K; k++)
		result.append(py::make_tuple(out[4 * k], out[4 * k + 1], out[4 * k + 2], out[4 * k + 3]));
	return result;
}

py::dict stage_tensors(const GeometryStage& g)
{
	py::dict d;
	for (int k = 0; k < kInputs; k++)
		if (k != kMeans2D)
			d[kInputNames[k]] = g.in[k];
	d["bg"] = g.s.bg;
	d["viewmatrix"] = g.s.view;
	d["projmatrix"] = g.s.proj;
	d["projmatrix_inv"] = g.s.proj_inv;
	d["range_low"] = g.s.low;
	d["range_up"] = g.s.up;
	d["campos"] = g.s.campos;
	d["tanfovx"] = g.s.tanfovx;
	d["tanfovy"] = g.s.tanfovy;
	d["debug"] = static_cast<int>(g.s.debug);
	return d;
}

}  // namespace
}  // namespace rgs_host

using namespace rgs_host;

PYBIND11_MODULE(_host, m)
{
	library_error_type = py::object(py::module_::import("retinags_amd._capi").attr("RgsError")).release().ptr();
	// For the functions of this module alone: the library's errors by their own type, those of tensor code (out of memory among
	// them, which callers catch to make room and try again) and of Python code that it ran by the types that PyTorch gives them.
	py::register_local_exception_translator([](std::exception_ptr p) {
		try {
			if (p)
				std::rethrow_exception(p);
		} catch (const LibraryError& e) {
			PyErr_SetString(library_error_type, e.what());
		} catch (const c10::Error&) {
			torch::translate_exception_to_python(p);
		} catch (const python_error&) {
			torch::translate_exception_to_python(p);
		}
	});

	m.def("composite", &composite, py::arg("background"), py::arg("planes"), py::arg("strips") = py::none());
	m.def("gradient_outputs", &gradient_outputs);
	m.def("set_original_gradient_outputs", &set_original_gradient_outputs);
	m.def("rasterize", &rasterize);
	m.def("rasterize_forward", &rasterize_forward);
	m.def("rasterize_forward_from_stage", &rasterize_forward_from_stage);
	m.def("rasterize_backward", &rasterize_backward);
	m.def("rasterize_frame", &rasterize_frame, py::arg("settings"), py::arg("inputs"), py::arg("streams"), py::arg("workspaces"),
	      py::arg("strips") = py::none(), py::arg("split") = py::none());
	m.def("enqueue_geometry", &enqueue_geometry);
	define_training(m);

	py::class_<GeometryStage>(m, "GeometryStage",
	                          "What the first half of a forward call leaves behind: the geometry workspace, the radii and the place "
	                          "where the instance count lands.  Made by GaussianRasterizer.enqueue_geometry, consumed once by "
	                          "GaussianRasterizer.forward.")
	    .def_readonly("P", &GeometryStage::P)
	    .def_readonly("H", &GeometryStage::H)
	    .def_readonly("W", &GeometryStage::W)
	    .def_property_readonly("used", [](const GeometryStage& g) { return g.used.load(); })
	    .def_property_readonly("settings", [](const GeometryStage& g) { return g.settings; })
	    .def_readonly("radii", &GeometryStage::radii)
	    .def_readonly("geomBuffer", &GeometryStage::geom)
	    .def_readonly("instance_bound", &GeometryStage::bound)
	    .def_property_readonly("geom_bytes", [](const GeometryStage& g) { return g.geom.numel(); })
	    .def_property_readonly("stream", [](const GeometryStage& g) { return reinterpret_cast<uintptr_t>(g.stream); })
	    .def_property_readonly("device", [](const GeometryStage& g) { return py::reinterpret_steal<py::object>(THPDevice_New(g.device)); })
	    .def_property_readonly("tensors", &stage_tensors)
	    .def("instances", &GeometryStage::instances, py::call_guard<py::gil_scoped_release>(),
	         "The number of (Gaussian, tile) instances of this call; waits for it if it is still on its way.  A stage that was "
	         "given an instance_bound must be asked once its forward has been issued: a count above the bound means the images of "
	         "that forward are wrong.")
	    .def("within_bound", [](GeometryStage& g) { return !g.bound || g.P == 0 || g.instances() <= *g.bound; },
	         py::call_guard<py::gil_scoped_release>());
}
