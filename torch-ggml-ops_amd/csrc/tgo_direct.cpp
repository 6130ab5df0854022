// Calls without a gradient, straight from Python: one C function per operator that checks its tensors, allocates and
// launches, instead of the dispatcher, the Python implementation behind it and a ctypes call per step.
//
// What bounds a decode-sized call is the host: 15 us for one projection whose kernel takes 6, 67 us for a
// mixture-of-experts layer whose five kernels take 23.  Here the projection costs two allocations and a launch, the layer two
// allocations and its launches, of which a layer of a few tokens has two (tgo_moe_decode).
//
// A function returns None for every call that is not plainly its own -- a gradient may be wanted, a tensor is not an ordinary
// device tensor, a transform, a mode or a tracer is active, an argument would not pass the operator's checks -- and its
// caller then goes through the registered operator, which handles it or names what is wrong.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdio>
#include <cstring>

#include "../../include/tgo.h"

namespace {

constexpr int64_t SUPER_BLOCK = 256;
constexpr int64_t LIMIT = 0x7fffffff;

// Keys whose presence in the thread's state means that somebody wants to see the operator itself.
bool thread_is_plain() {
    static const c10::DispatchKeySet watched({
        c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
        c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::VmapMode,
        c10::DispatchKey::Functionalize, c10::DispatchKey::PreDispatch, c10::DispatchKey::Tracer, c10::DispatchKey::PythonDispatcher,
        c10::DispatchKey::TESTING_ONLY_GenericMode, c10::DispatchKey::DeferredInit});
    return !c10::impl::tls_local_dispatch_key_set().included_.has_any(watched) && !at::impl::torch_function_mode_enabled();
}

// An ordinary tensor of the current device that no gradient flows through here: contiguous, from the start of its storage.
bool plain(const at::Tensor & t, at::ScalarType dtype, c10::DeviceIndex device) {
    static const c10::DispatchKeySet harmless = c10::autograd_dispatch_keyset_with_ADInplaceOrView |
                                                c10::getAutocastRelatedKeySetFromBackend(c10::BackendComponent::CUDABit);
    return (t.key_set() - harmless) == c10::DispatchKeySet(c10::DispatchKey::CUDA) && t.scalar_type() == dtype &&
           t.device().index() == device && t.is_contiguous() && t.storage_offset() == 0 &&
           !(t.requires_grad() && c10::GradMode::is_enabled()) && !t._fw_grad(0).defined();
}
bool aligned(const at::Tensor & t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// `value` of a Python integer (false: not one, or out of range).
bool integer(PyObject * object, int64_t & value) {
    if (!PyLong_Check(object)) {
        return false;
    }
    value = PyLong_AsLongLong(object);
    if (value == -1 && PyErr_Occurred() != nullptr) {
        PyErr_Clear();
        return false;
    }
    return true;
}

PyObject * declined() { Py_RETURN_NONE; }

// The result of a native call: the output tensor, or the library's message as RuntimeError.
PyObject * finished(int status, const at::Tensor & output) {
    if (status != TGO_OK) {
        PyErr_SetString(PyExc_RuntimeError, tgo_last_error());
        return nullptr;
    }
    return THPVariable_Wrap(output);
}

// mmq(input, packed_weight, quant_type, out_features)
PyObject * direct_mmq(PyObject *, PyObject * const * args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    int64_t quant_type, out_features;
    if (count != 4 || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !integer(args[2], quant_type) ||
        !integer(args[3], out_features) || !thread_is_plain()) {
        return declined();
    }
    const at::Tensor & input = THPVariable_Unpack(args[0]);
    const at::Tensor & weight = THPVariable_Unpack(args[1]);
    if (!input.is_cuda()) {
        return declined();
    }
    const c10::DeviceIndex device = c10::hip::current_device();
    if (!plain(input, at::kBFloat16, device) || !plain(weight, at::kByte, device) || input.dim() < 1) {
        return declined();
    }
    const int64_t in_features = input.size(-1);
    if (in_features <= 0 || in_features % SUPER_BLOCK != 0 || in_features > LIMIT || out_features <= 0 || out_features > LIMIT) {
        return declined();
    }
    const int64_t rows = input.numel() / in_features;
    const int block = quant_type >= 0 && quant_type <= LIMIT ? tgo_block_bytes(static_cast<int>(quant_type)) : 0;
    if (rows <= 0 || rows > LIMIT || block == 0 || weight.numel() != out_features * (in_features / SUPER_BLOCK) * block ||
        !aligned(input) || !aligned(weight)) {
        return declined();
    }
    int status;
    at::Tensor output;
    {
        pybind11::gil_scoped_release release;
        RECORD_FUNCTION("torch_ggml_ops::mmq", c10::ArrayRef<const c10::IValue>());
        c10::SmallVector<int64_t, 5> shape(input.sizes().begin(), input.sizes().end());
        shape.back() = out_features;
        output = at::detail::empty_cuda(shape, at::kBFloat16, input.device(), std::nullopt);
        const int64_t workspace_bytes = (tgo_q8_workspace_bytes(rows, in_features) + 255) / 256 * 256;
        const int64_t scratch_bytes = tgo_forward_scratch_bytes_as(rows, in_features, out_features, static_cast<int>(quant_type), TGO_OPERAND_AUTO);
        const c10::DataPtr workspace = c10::GetAllocator(c10::kCUDA)->allocate(workspace_bytes + scratch_bytes);
        void * const scratch = scratch_bytes > 0 ? static_cast<uint8_t *>(workspace.get()) + workspace_bytes : nullptr;
        status = tgo_mmq_forward_sized(input.data_ptr(), weight.data_ptr(), output.data_ptr(), workspace.get(), scratch, scratch_bytes, rows,
                                       in_features, out_features, static_cast<int>(quant_type),
                                       c10::hip::getCurrentHIPStream(device).stream());
    }
    return finished(status, output);
    END_HANDLE_TH_ERRORS
}

// Pieces of one allocation, 256 bytes apart at least.
struct Pieces {
    int64_t bytes = 0;
    int64_t take(int64_t size) {
        const int64_t at = bytes;
        bytes += (size + 255) / 256 * 256;
        return at;
    }
};

// moe_layer(hidden, slot_experts, slot_weights, gate, up, down, gate_up_type, down_type, intermediate_features)
PyObject * direct_moe_layer(PyObject *, PyObject * const * args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    int64_t gate_up_type, down_type, intermediate;
    if (count != 9 || !integer(args[6], gate_up_type) || !integer(args[7], down_type) || !integer(args[8], intermediate) ||
        !thread_is_plain()) {
        return declined();
    }
    for (int i = 0; i < 6; ++i) {
        if (!THPVariable_CheckExact(args[i])) {
            return declined();
        }
    }
    const at::Tensor & hidden = THPVariable_Unpack(args[0]);
    const at::Tensor & slot_experts = THPVariable_Unpack(args[1]);
    const at::Tensor & slot_weights = THPVariable_Unpack(args[2]);
    const at::Tensor & gate = THPVariable_Unpack(args[3]);
    const at::Tensor & up = THPVariable_Unpack(args[4]);
    const at::Tensor & down = THPVariable_Unpack(args[5]);
    if (!hidden.is_cuda()) {
        return declined();
    }
    const c10::DeviceIndex device = c10::hip::current_device();
    if (!plain(hidden, at::kBFloat16, device) || !plain(slot_experts, at::kLong, device) ||
        !plain(slot_weights, at::kFloat, device) || !plain(gate, at::kByte, device) || !plain(up, at::kByte, device) ||
        !plain(down, at::kByte, device)) {
        return declined();
    }
    if (hidden.dim() != 2 || slot_experts.dim() != 2 || gate.dim() != 3 || down.dim() != 3 || gate.sizes() != up.sizes() ||
        slot_experts.sizes() != slot_weights.sizes() || slot_experts.size(0) != hidden.size(0)) {
        return declined();
    }
    const int64_t tokens = hidden.size(0), features = hidden.size(1), top_k = slot_experts.size(1), experts = gate.size(0);
    const int64_t slots = tokens * top_k;
    const auto known = [](int64_t type) { return type >= 0 && type <= LIMIT ? tgo_block_bytes(static_cast<int>(type)) : 0; };
    const int64_t gate_up_block = known(gate_up_type), down_block = known(down_type);
    if (slots <= 0 || slots > TGO_ROUTE_SLOT_LIMIT || experts <= 0 || experts > TGO_ROUTE_EXPERT_LIMIT || down.size(0) < experts ||
        down.size(0) > LIMIT || features <= 0 || features % SUPER_BLOCK != 0 || features > LIMIT || intermediate <= 0 ||
        intermediate % SUPER_BLOCK != 0 || intermediate > LIMIT || gate_up_block == 0 || down_block == 0 ||
        gate.size(1) != intermediate || gate.size(2) != features / SUPER_BLOCK * gate_up_block || down.size(1) != features ||
        down.size(2) != intermediate / SUPER_BLOCK * down_block || !aligned(hidden) || !aligned(gate) || !aligned(up) ||
        !aligned(down)) {
        return declined();
    }
    int status;
    at::Tensor output;
    {
        pybind11::gil_scoped_release release;
        RECORD_FUNCTION("torch_ggml_ops::moe_layer", c10::ArrayRef<const c10::IValue>());
        output = at::detail::empty_cuda({tokens, features}, at::kBFloat16, hidden.device(), std::nullopt);
        const int64_t decode_bytes = tgo_moe_decode_workspace_bytes(tokens, top_k, experts, features, intermediate, static_cast<int>(gate_up_type),
                                                                    static_cast<int>(down_type));
        if (decode_bytes > 0) {
            const c10::DataPtr memory = c10::GetAllocator(c10::kCUDA)->allocate(decode_bytes);
            status = tgo_moe_decode(hidden.data_ptr(), slot_experts.const_data_ptr<int64_t>(), slot_weights.const_data_ptr<float>(),
                                    gate.data_ptr(), up.data_ptr(), down.data_ptr(), output.data_ptr(), memory.get(), tokens, top_k, experts,
                                    features, intermediate, static_cast<int>(gate_up_type), static_cast<int>(down_type),
                                    c10::hip::getCurrentHIPStream(device).stream());
        } else {
            Pieces pieces;
            const int64_t row_index = pieces.take(slots * 8), slot_rows = pieces.take(slots * 8), indices = pieces.take(experts * 8),
                          offsets = pieces.take(experts * 4), activated = pieces.take(slots * intermediate * 2),
                          rows = pieces.take(slots * std::max(features, intermediate) * 2),   // the gate, then the expert-sorted results
                          route_workspace = pieces.take(tgo_route_workspace_bytes(slots, experts)),
                          workspace = pieces.take(tgo_q8_workspace_bytes(slots, std::max(features, intermediate)) +
                                                  tgo_task_workspace_bytes(slots, experts));
            const c10::DataPtr memory = c10::GetAllocator(c10::kCUDA)->allocate(pieces.bytes);
            uint8_t * const base = static_cast<uint8_t *>(memory.get());
            int64_t * const index = reinterpret_cast<int64_t *>(base + row_index);
            int64_t * const of_slot = reinterpret_cast<int64_t *>(base + slot_rows);
            int64_t * const group_expert = reinterpret_cast<int64_t *>(base + indices);
            int32_t * const group_end = reinterpret_cast<int32_t *>(base + offsets);
            void * const stream = c10::hip::getCurrentHIPStream(device).stream();
            status = tgo_route(slot_experts.const_data_ptr<int64_t>(), tokens, top_k, experts, index, of_slot, group_expert, group_end,
                               base + route_workspace, stream);
            if (status == TGO_OK) {
                status = tgo_grouped_mmq_swiglu(hidden.data_ptr(), index, tokens, gate.data_ptr(), up.data_ptr(), base + rows,
                                                base + activated, group_expert, group_end, base + workspace, slots, features,
                                                intermediate, experts, experts, static_cast<int>(gate_up_type), stream);
            }
            if (status == TGO_OK) {
                status = tgo_grouped_mmq_forward(base + activated, down.data_ptr(), nullptr, base + rows, nullptr, group_expert,
                                                 group_end, base + workspace, slots, intermediate, features, down.size(0), experts,
                                                 static_cast<int>(down_type), stream);
            }
            if (status == TGO_OK) {
                status = tgo_moe_combine(base + rows, of_slot, slot_weights.const_data_ptr<float>(), output.data_ptr(), tokens, top_k,
                                         slots, features, stream);
            }
        }
    }
    return finished(status, output);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"mmq", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(direct_mmq)), METH_FASTCALL, nullptr},
    {"moe_layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(direct_moe_layer)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_definition = {PyModuleDef_HEAD_INIT, "_direct", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

// Whether the running Python and torch are those that this file was compiled against, and the library the one whose header it
// read: it reaches into their structures, so with any other the package does without it.  (Asked through functions that every
// version has.)
bool built_for_this_process() {
    if (tgo_version() != TGO_VERSION) {
        PyErr_Format(PyExc_ImportError, "_direct.so was built for version %d of the library, this is %d", TGO_VERSION, tgo_version());
        return false;
    }
    char python[16];
    snprintf(python, sizeof(python), "%d.%d.", PY_MAJOR_VERSION, PY_MINOR_VERSION);
    if (strncmp(Py_GetVersion(), python, strlen(python)) != 0) {
        PyErr_Format(PyExc_ImportError, "_direct.so was built for Python %s*", python);
        return false;
    }
    PyObject * const torch = PyImport_ImportModule("torch");
    PyObject * const version = torch != nullptr ? PyObject_GetAttrString(torch, "__version__") : nullptr;
    const char * const running = version != nullptr ? PyUnicode_AsUTF8(version) : nullptr;
    const bool same = running != nullptr && strcmp(running, TGO_TORCH_VERSION) == 0;
    if (running != nullptr && !same) {
        PyErr_Format(PyExc_ImportError, "_direct.so was built for torch %s, this is %s", TGO_TORCH_VERSION, running);
    }
    Py_XDECREF(version);
    Py_XDECREF(torch);
    return same;
}

}  // namespace

PyMODINIT_FUNC PyInit__direct() { return built_for_this_process() ? PyModule_Create(&module_definition) : nullptr; }
