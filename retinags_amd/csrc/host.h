// What the parts of the host path share: errors, tensors, the landing places of counts.
#pragma once
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/custom_class.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <atomic>
#include <deque>
#include <map>
#include <mutex>
#include <optional>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/rgs.h"
#include "counts.h"

namespace rgs_host {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- errors ------------------------------------------------------------------------------------------------------

struct LibraryError : std::runtime_error {
	using std::runtime_error::runtime_error;
};

inline PyObject* library_error_type = nullptr;  // retinags_amd._capi.RgsError

inline void check(int rc)
{
	if (rc != 0)
		throw LibraryError(rgs_last_error());
}

// What a backward node throws on autograd's own thread keeps its Python type on the way to the caller.
[[noreturn]] inline void throw_to_autograd()
{
	python_error err;
	err.persist();
	throw err;
}

template <class F>
variable_list in_backward(F body)
{
	try {
		return body();
	} catch (const LibraryError& e) {
		py::gil_scoped_acquire gil;
		PyErr_SetString(library_error_type, e.what());
		throw_to_autograd();
	} catch (py::error_already_set& e) {
		py::gil_scoped_acquire gil;
		e.restore();
		throw_to_autograd();
	}
}

// ---- tensors -----------------------------------------------------------------------------------------------------

// Device (or pinned) address; absent and empty tensors are null pointers, the form in which the C ABI takes absent inputs.
template <class T = float>
T* ptr(const Tensor& t)
{
	return t.defined() && t.numel() != 0 ? static_cast<T*>(t.data_ptr()) : nullptr;
}

inline Tensor from_python(py::handle h, const char* name)
{
	if (h.is_none())
		return Tensor();
	if (!THPVariable_Check(h.ptr()))
		throw py::type_error(std::string(name) + " must be a tensor");
	return THPVariable_Unpack(h.ptr());
}

// The same where a tensor has to be given.
inline Tensor tensor_from_python(py::handle h, const char* name)
{
	if (!THPVariable_Check(h.ptr()))
		throw py::type_error(std::string(name) + " must be a tensor");
	return THPVariable_Unpack(h.ptr());
}

inline py::object to_python(const Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

inline bool present(const Tensor& t) { return t.defined() && t.numel() != 0; }

// Contiguous fp32 on `device`; empty and absent tensors as they are.
inline Tensor device_f32(const Tensor& t, const at::Device& device)
{
	if (!present(t))
		return t;
	if (t.scalar_type() == at::kFloat && t.device() == device)
		return t.is_contiguous() ? t : t.contiguous();
	return t.to(device, at::kFloat).contiguous();
}

inline Tensor new_f32(at::IntArrayRef shape, const at::Device& device)
{
	return at::empty(shape, at::TensorOptions().dtype(at::kFloat).device(device));
}

inline Tensor new_bytes(size_t n, const at::Device& device)
{
	return at::empty({static_cast<int64_t>(n)}, at::TensorOptions().dtype(at::kByte).device(device));
}

// A tensor over part of another's allocation that is no view of it: autograd takes such a gradient over as it is, where it
// copies a view.
inline Tensor carved(const Tensor& block, int64_t at_element, at::IntArrayRef shape)
{
	Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(block.storage()), block.key_set(), block.dtype());
	t.unsafeGetTensorImpl()->set_storage_offset(block.storage_offset() + at_element);
	t.unsafeGetTensorImpl()->set_sizes_contiguous(shape);
	return t;
}

inline hipStream_t current_stream(const at::Device& device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

// ---- landing places of counts that the device reports ------------------------------------------------------------

// A few pinned words and an event that says they have arrived.
struct CountSlot {
	uint32_t* words = nullptr;
	uint32_t* on_device = nullptr;  // the same words as kernels write them
	hipEvent_t event = nullptr;
};

constexpr int kSlotWords = RGS_MAX_SHARE_BOXES * RGS_MAX_SHARE_BOXES;
static_assert(kSlotWords >= RGS_MAX_FRAME_LAYERS, "a frame reports one count per layer");

// While a thread captures a graph, queries of events and allocations of pinned memory by any thread would end that capture
// unless they are told not to matter to it.
class OutsideCapture {
public:
	OutsideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode_); }
	~OutsideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode_); }
	OutsideCapture(const OutsideCapture&) = delete;
	OutsideCapture& operator=(const OutsideCapture&) = delete;

private:
	hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
};

// Slots per device, kept for the next call that needs one: at most kKept of them, shared by all threads and streams (a call
// has its slot to itself).  A slot whose count nobody waited for comes back when its event has passed.
class SlotPool {
public:
	CountSlot take(int device)
	{
		std::lock_guard<std::mutex> lock(mutex_);
		PerDevice& d = devices_[device];
		if (d.in_flight.empty() && !d.free.empty()) {
			CountSlot s = d.free.back();
			d.free.pop_back();
			return s;
		}
		OutsideCapture relaxed;
		for (size_t n = d.in_flight.size(); n > 0; n--) {
			CountSlot s = d.in_flight.front();
			d.in_flight.pop_front();
			if (hipEventQuery(s.event) == hipSuccess) {
				keep(d, s);
			} else {
				(void)hipGetLastError();  // not there yet: no error of the caller's
				d.in_flight.push_back(s);
			}
		}
		if (!d.free.empty()) {
			CountSlot s = d.free.back();
			d.free.pop_back();
			return s;
		}
		CountSlot s;
		void* memory = nullptr;
		void* address = nullptr;
		if (hipHostMalloc(&memory, kSlotWords * sizeof(uint32_t), hipHostMallocDefault) != hipSuccess ||
		    hipHostGetDevicePointer(&address, memory, 0) != hipSuccess ||
		    hipEventCreateWithFlags(&s.event, hipEventDisableTiming) != hipSuccess)
			throw std::runtime_error("no pinned memory for an instance count");
		s.words = static_cast<uint32_t*>(memory);
		s.on_device = static_cast<uint32_t*>(address);
		return s;
	}
	void give_back(int device, CountSlot s)
	{
		std::lock_guard<std::mutex> lock(mutex_);
		keep(devices_[device], s);
	}
	void give_back_in_flight(int device, CountSlot s)
	{
		std::lock_guard<std::mutex> lock(mutex_);
		devices_[device].in_flight.push_back(s);
	}

private:
	static constexpr size_t kKept = 64;
	struct PerDevice {
		std::vector<CountSlot> free;
		std::deque<CountSlot> in_flight;
	};
	void keep(PerDevice& d, CountSlot s)
	{
		if (d.free.size() < kKept) {
			d.free.push_back(s);
			return;
		}
		OutsideCapture relaxed;
		(void)hipEventDestroy(s.event);
		(void)hipHostFree(s.words);
	}
	std::mutex mutex_;
	std::map<int, PerDevice> devices_;
};

inline SlotPool& slot_pool()
{
	static SlotPool* pool = new SlotPool;  // stays until the process ends: the runtime may be gone before static objects are
	return *pool;
}

// A slot whose words kernels of `stream` write, for as long as the caller is about to launch them and waits for what they write.
class AwaitedCounts {
public:
	AwaitedCounts(int device, hipStream_t stream, int n) : device_(device), stream_(stream), n_(n), slot_(slot_pool().take(device))
	{
		rgs::expect_counts(slot_.words, n);
	}
	~AwaitedCounts()
	{
		if (!arrived_)
			(void)hipStreamSynchronize(stream_);  // a kernel may yet write them
		slot_pool().give_back(device_, slot_);
	}
	AwaitedCounts(const AwaitedCounts&) = delete;
	AwaitedCounts& operator=(const AwaitedCounts&) = delete;
	uint32_t* on_device() const { return slot_.on_device; }
	// The words, or null if they did not come.
	const uint32_t* wait()
	{
		arrived_ = rgs::wait_for_counts(slot_.words, n_, stream_) == hipSuccess;
		return arrived_ ? slot_.words : nullptr;
	}

private:
	const int device_;
	const hipStream_t stream_;
	const int n_;
	const CountSlot slot_;
	bool arrived_ = false;
};


void define_training(py::module_& m);  // host_training.cpp

}  // namespace rgs_host
