// Python front end of the C ABI: the calls that a decode step makes, from torch tensors and
// PackedWeight objects straight to the entry points of libnfn_mi355_tile_ops.so.
//
// What bounds these calls is the host.  A HIP launch costs about 2.8 us here, and the same call
// put together in Python around it (a ctypes structure per weight, pointer arrays, the stream
// object, an output tensor each) took another 7.5 to 13 us: grouped Q/K/V of one token 16.5 us,
// 11.0 us with outputs that the caller keeps, against 6 us that its kernel runs.  Here a
// descriptor is nine stores, the stream one call and an output one allocator call.
//
// Nothing is kept between calls: every descriptor is made from the weight's attributes as they
// are at the call.  The interpreter lock is given up around the entry point, as ctypes does, and
// around nothing else: whatever may raise (a tensor without storage has no data pointer) is
// evaluated before.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cstring>
#include <string>
#include <type_traits>

#include "../../../include/nfn_mi355_tile_ops.h"

namespace {

using Descriptor = NfnNativeTilePackedWeightDescriptorV1;

// A Python error is set; unwinds to the function table's wrapper.
struct Raised {};

// -- the library's entry points, handed over as addresses by bind() ------------------------------

#define NFN_ENTRY_POINTS(X)                                                   \
    X(nfn_native_tile_linear_packed_weight_float32_v1)                        \
    X(nfn_native_tile_k_quant_mmq_multi_linear_float32_v1)                    \
    X(nfn_native_tile_k_quant_mmq_multi_linear_gated_float32_v1)              \
    X(nfn_native_tile_k_quant_mmq_multi_linear_swiglu_float32_v1)             \
    X(nfn_native_tile_k_quant_mmvq_multi_linear_float32_v1)                   \
    X(nfn_native_tile_k_quant_mmvq_multi_linear_gated_float32_v1)             \
    X(nfn_native_tile_k_quant_mmvq_multi_linear_swiglu_float32_v1)            \
    X(nfn_native_tile_k_quant_mmvq_multi_linear_prequantized_float32_v1)      \
    X(nfn_mi355_k_quant_mmq_multi_linear_prequantized_float32_v1)             \
    X(nfn_native_tile_k_quant_mmvq_linear_float32_v1)                         \
    X(nfn_native_tile_glimmer_dual_rms_add_capture_float32_v1)                \
    X(nfn_native_tile_glimmer_dual_rms_add_capture_mmvq_q8_float32_v1)        \
    X(nfn_mi355_dual_rms_add_capture_mmvq_rows_float32_v1)                    \
    X(nfn_mi355_dual_rms_add_capture_mmq_f16_float32_v1)                      \
    X(nfn_mi355_dual_rms_mmvq_multi_linear_float32_v1)                        \
    X(nfn_mi355_k_quant_mmvq_gate_up_swiglu_float32_v1)                       \
    X(nfn_mi355_k_quant_mmq_gate_up_swiglu_float32_v1)                        \
    X(nfn_mi355_lm_head_argmax_workspace_bytes_v1)                            \
    X(nfn_mi355_lm_head_argmax_v1)                                            \
    X(nfn_mi355_k_quant_gemm_workspace_bytes_v1)                              \
    X(nfn_mi355_k_quant_gemm_multi_workspace_bytes_v1)                        \
    X(nfn_mi355_k_quant_gemm_float32_v1)                                      \
    X(nfn_mi355_k_quant_gemm_multi_float32_v1)                                \
    X(nfn_native_tile_glimmer_qk_norm_scale_rope_float32_v1)                  \
    X(nfn_native_tile_glimmer_qk_norm_scale_rope_batch_float32_v1)            \
    X(nfn_native_tile_glimmer_fused_decode_attention_float32_v1)              \
    X(nfn_native_tile_glimmer_fused_decode_attention_device_position_float32_v1) \
    X(nfn_mi355_fused_decode_attention_split_v1)                              \
    X(nfn_mi355_fused_decode_attention_split_device_position_v1)              \
    X(nfn_native_tile_glimmer_gqa_decode_float32_v1)                          \
    X(nfn_mi355_gqa_decode_split_v1)                                          \
    X(nfn_native_tile_dflash_block_attention_float32_v1)                      \
    X(nfn_mi355_dflash_block_attention_split_v1)

struct Library {
#define NFN_MEMBER(name) decltype(&::name) name = nullptr;
    NFN_ENTRY_POINTS(NFN_MEMBER)
#undef NFN_MEMBER
};
Library lib;
PyObject* check_callable = nullptr;  // tile_ops.check(status, operation)
PyObject *name_encoding, *name_output_dim, *name_input_dim, *name_data;

// -- arguments -----------------------------------------------------------------------------------

[[noreturn]] void raise(PyObject* type, const char* text) {
    PyErr_SetString(type, text);
    throw Raised{};
}

const at::Tensor& tensor_of(PyObject* object) {
    if (!THPVariable_Check(object)) raise(PyExc_TypeError, "a torch tensor is expected");
    return THPVariable_Unpack(object);
}

std::int64_t integer_of(PyObject* object) {
    const long long value = PyLong_AsLongLong(object);
    if (value == -1 && PyErr_Occurred()) throw Raised{};
    return value;
}

double number_of(PyObject* object) {
    const double value = PyFloat_AsDouble(object);
    if (value == -1.0 && PyErr_Occurred()) throw Raised{};
    return value;
}

bool truth_of(PyObject* object) {
    const int value = PyObject_IsTrue(object);
    if (value < 0) throw Raised{};
    return value != 0;
}

// null for None
float* floats_or_null(PyObject* object) {
    return object == Py_None ? nullptr : static_cast<float*>(tensor_of(object).data_ptr());
}
float* floats_of(const at::Tensor& tensor) { return static_cast<float*>(tensor.data_ptr()); }

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The attribute of a weight; a new reference is dropped at once, the weight keeps the object.
struct Attribute {
    PyObject* object;
    Attribute(PyObject* owner, PyObject* name) : object(PyObject_GetAttr(owner, name)) {
        if (object == nullptr) throw Raised{};
    }
    ~Attribute() { Py_DECREF(object); }
    Attribute(const Attribute&) = delete;
};

Descriptor descriptor_of(PyObject* weight, void* stream) {
    const Attribute encoding(weight, name_encoding), rows(weight, name_output_dim),
        columns(weight, name_input_dim), data(weight, name_data);
    Descriptor d;
    std::memset(&d, 0, sizeof(d));
    const std::int64_t code = integer_of(encoding.object);
    d.struct_size = sizeof(d);
    d.version = NFN_NATIVE_TILE_PACKED_WEIGHT_V1;
    d.encoding = static_cast<std::uint32_t>(code);
    d.output_dim = integer_of(rows.object);
    d.input_dim = integer_of(columns.object);
    std::int64_t elements = 256, block = 0;
    switch (code) {
        case NFN_NATIVE_TILE_PACKED_WEIGHT_F32: elements = 1, block = 4; break;
        case NFN_NATIVE_TILE_PACKED_WEIGHT_BF16: elements = 1, block = 2; break;
        case NFN_MI355_PACKED_WEIGHT_Q8_0: elements = 32, block = 34; break;
        case NFN_NATIVE_TILE_PACKED_WEIGHT_Q4_K: block = 144; break;
        case NFN_NATIVE_TILE_PACKED_WEIGHT_Q5_K: block = 176; break;
        case NFN_NATIVE_TILE_PACKED_WEIGHT_Q6_K: block = 210; break;
        default:
            PyErr_SetObject(PyExc_KeyError, encoding.object);
            throw Raised{};
    }
    if (d.input_dim % elements != 0) {
        raise(PyExc_ValueError, ("input_dim " + std::to_string(d.input_dim) + " is not a multiple of " +
                                 std::to_string(elements)).c_str());
    }
    d.row_stride_bytes = d.input_dim / elements * block;
    d.data_nbytes = d.output_dim * d.row_stride_bytes;
    d.data = static_cast<const std::uint8_t*>(tensor_of(data.object).data_ptr());
    d.cuda_stream = stream;
    return d;
}

// An optional weight (None: no weight).
struct OptionalWeight {
    Descriptor descriptor;
    const Descriptor* pointer = nullptr;
    OptionalWeight(PyObject* weight, void* stream) {
        if (weight == Py_None) return;
        descriptor = descriptor_of(weight, stream);
        pointer = &descriptor;
    }
};

struct Sequence {
    PyObject* object;
    explicit Sequence(PyObject* source) : object(PySequence_Fast(source, "a sequence is expected")) {
        if (object == nullptr) throw Raised{};
    }
    ~Sequence() { Py_DECREF(object); }
    Sequence(const Sequence&) = delete;
    Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(object); }
    PyObject* operator[](Py_ssize_t index) const { return PySequence_Fast_GET_ITEM(object, index); }
};

at::Tensor new_floats(std::int64_t rows, std::int64_t width, c10::Device device) {
    return at::empty({rows, width}, at::TensorOptions().dtype(at::kFloat).device(device));
}

// An owned reference.
struct Reference {
    PyObject* object = nullptr;
    Reference() = default;
    ~Reference() { Py_XDECREF(object); }
    Reference(const Reference&) = delete;
    PyObject* take() {
        PyObject* taken = object;
        object = nullptr;
        return taken;
    }
};

// The projections of one call: descriptors, output pointers and the Python object to return (the
// caller's `outputs`, or a list of new tensors).
struct Projections {
    c10::SmallVector<Descriptor, 4> descriptors;
    c10::SmallVector<const Descriptor*, 4> pointers;
    c10::SmallVector<float*, 4> outputs;
    Reference result;

    Projections(PyObject* weights, PyObject* given, std::int64_t rows, c10::Device device, void* stream) {
        const Sequence list(weights);
        const Py_ssize_t count = list.size();
        for (Py_ssize_t i = 0; i < count; ++i) descriptors.push_back(descriptor_of(list[i], stream));
        for (const Descriptor& descriptor : descriptors) pointers.push_back(&descriptor);
        if (given != Py_None) {
            const Sequence targets(given);
            if (targets.size() < count) raise(PyExc_ValueError, "an output for every weight is expected");
            for (Py_ssize_t i = 0; i < count; ++i) outputs.push_back(floats_of(tensor_of(targets[i])));
            Py_INCREF(given);
            result.object = given;
            return;
        }
        result.object = PyList_New(count);
        if (result.object == nullptr) throw Raised{};
        for (Py_ssize_t i = 0; i < count; ++i) {
            const at::Tensor out = new_floats(rows, descriptors[i].output_dim, device);
            outputs.push_back(floats_of(out));
            PyList_SET_ITEM(result.object, i, THPVariable_Wrap(out));
        }
    }
    std::int64_t count() const { return static_cast<std::int64_t>(descriptors.size()); }
    PyObject* take() { return result.take(); }
};

// The interpreter lock, given up for a scope; whichever way the scope ends, it is held again.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    Unlocked() = default;
    ~Unlocked() { PyEval_RestoreThread(state); }
    Unlocked(const Unlocked&) = delete;
};

// Runs an entry point without the interpreter lock; a status other than 0 raises what
// tile_ops.check raises.  The arguments are numbers and pointers, evaluated by the caller under
// the lock: nothing that could raise or run Python is left for the region.
template <typename... Parameters, typename... Arguments>
void call(const char* operation, int (*entry)(Parameters...), Arguments... arguments) {
    static_assert(((std::is_arithmetic_v<Arguments> || std::is_pointer_v<Arguments> ||
                    std::is_null_pointer_v<Arguments>) && ...), "plain values only");
    int status;
    {
        const Unlocked unlocked;
        status = entry(arguments...);
    }
    if (status != 0) {
        PyObject* nothing = PyObject_CallFunction(check_callable, "is", status, operation);
        Py_XDECREF(nothing);
        throw Raised{};
    }
}

// an output the caller passed, or a new one
struct Output {
    PyObject* object;
    float* data;
    Output(PyObject* given, std::int64_t rows, std::int64_t width, c10::Device device) {
        if (given != Py_None) {
            data = floats_of(tensor_of(given));
            Py_INCREF(given);
            object = given;
        } else {
            const at::Tensor out = new_floats(rows, width, device);
            data = floats_of(out);
            object = THPVariable_Wrap(out);
        }
    }
    Output(PyObject* given, const at::Tensor& like) {
        if (given != Py_None) {
            data = floats_of(tensor_of(given));
            Py_INCREF(given);
            object = given;
        } else {
            const at::Tensor out = at::empty_like(like);
            data = floats_of(out);
            object = THPVariable_Wrap(out);
        }
    }
    ~Output() { Py_XDECREF(object); }
    Output(const Output&) = delete;
    PyObject* take() {
        PyObject* taken = object;
        object = nullptr;
        return taken;
    }
};

// -- the calls (tile_ops.py and engine_ops.py hold their Python signatures) ------------------------

using Arguments = PyObject* const*;

// weights, x, workspace, second, family, prologue, outputs
PyObject* multi_linear(Arguments a) {
    const at::Tensor& x = tensor_of(a[1]);
    const at::Tensor& workspace = tensor_of(a[2]);
    const std::int64_t rows = x.size(0);
    const char* family = PyUnicode_AsUTF8(a[4]);
    const char* prologue = family == nullptr ? nullptr : PyUnicode_AsUTF8(a[5]);
    if (prologue == nullptr) throw Raised{};
    const bool verifier = std::strcmp(family, "mmvq") == 0;
    const bool plain = std::strcmp(prologue, "plain") == 0, gated = std::strcmp(prologue, "gated") == 0;
    if ((!verifier && std::strcmp(family, "mmq") != 0) ||
        (!plain && !gated && std::strcmp(prologue, "swiglu") != 0)) {
        raise(PyExc_KeyError, "family is 'mmq' or 'mmvq', prologue 'plain', 'gated' or 'swiglu'");
    }
    void* stream = current_stream();
    Projections p(a[0], a[6], rows, x.device(), stream);
    const float* first = floats_of(x);
    const float* second = plain ? nullptr : floats_or_null(a[3]);
    void* scratch = workspace.data_ptr();
    const std::int64_t scratch_bytes = workspace.numel();
    if (plain) {
        const auto entry = verifier ? lib.nfn_native_tile_k_quant_mmvq_multi_linear_float32_v1
                                    : lib.nfn_native_tile_k_quant_mmq_multi_linear_float32_v1;
        call(verifier ? "nfn_native_tile_k_quant_mmvq_multi_linear_float32_v1"
                      : "nfn_native_tile_k_quant_mmq_multi_linear_float32_v1",
             entry, p.pointers.data(), first, p.outputs.data(), p.count(), rows, scratch, scratch_bytes, stream);
    } else {
        const auto entry = gated ? (verifier ? lib.nfn_native_tile_k_quant_mmvq_multi_linear_gated_float32_v1
                                             : lib.nfn_native_tile_k_quant_mmq_multi_linear_gated_float32_v1)
                                 : (verifier ? lib.nfn_native_tile_k_quant_mmvq_multi_linear_swiglu_float32_v1
                                             : lib.nfn_native_tile_k_quant_mmq_multi_linear_swiglu_float32_v1);
        call(gated ? (verifier ? "nfn_native_tile_k_quant_mmvq_multi_linear_gated_float32_v1"
                               : "nfn_native_tile_k_quant_mmq_multi_linear_gated_float32_v1")
                   : (verifier ? "nfn_native_tile_k_quant_mmvq_multi_linear_swiglu_float32_v1"
                               : "nfn_native_tile_k_quant_mmq_multi_linear_swiglu_float32_v1"),
             entry, p.pointers.data(), first, second, p.outputs.data(), p.count(), rows, scratch, scratch_bytes, stream);
    }
    return p.take();
}

// weights, rows, workspace, outputs, verifier family
PyObject* multi_linear_prequantized(Arguments a) {
    const at::Tensor& workspace = tensor_of(a[2]);
    const std::int64_t rows = integer_of(a[1]);
    const bool verifier = truth_of(a[4]);
    void* stream = current_stream();
    Projections p(a[0], a[3], rows, workspace.device(), stream);
    const auto entry = verifier ? lib.nfn_native_tile_k_quant_mmvq_multi_linear_prequantized_float32_v1
                                : lib.nfn_mi355_k_quant_mmq_multi_linear_prequantized_float32_v1;
    void* scratch = workspace.data_ptr();
    const std::int64_t scratch_bytes = workspace.numel();
    call(verifier ? "mmvq_multi_linear_prequantized" : "mmq_multi_linear_prequantized", entry, p.pointers.data(),
         p.outputs.data(), p.count(), rows, scratch, scratch_bytes, stream);
    return p.take();
}

// weight, x, workspace, out
PyObject* mmvq_linear(Arguments a) {
    void* stream = current_stream();
    const Descriptor descriptor = descriptor_of(a[0], stream);
    const at::Tensor& x = tensor_of(a[1]);
    const at::Tensor& workspace = tensor_of(a[2]);
    Output out(a[3], 1, descriptor.output_dim, x.device());
    call("mmvq_linear", lib.nfn_native_tile_k_quant_mmvq_linear_float32_v1, &descriptor, floats_of(x), out.data,
         workspace.data_ptr(), workspace.numel(), stream);
    return out.take();
}

// weight, x, bias
PyObject* linear(Arguments a) {
    void* stream = current_stream();
    const Descriptor descriptor = descriptor_of(a[0], stream);
    const at::Tensor& x = tensor_of(a[1]);
    const std::int64_t rows = x.size(0);
    const float* bias = floats_or_null(a[2]);
    Output out(Py_None, rows, descriptor.output_dim, x.device());
    call("linear_packed_weight", lib.nfn_native_tile_linear_packed_weight_float32_v1, &descriptor, floats_of(x), bias,
         out.data, rows, a[2] != Py_None);
    return out.take();
}

// gate, up, x, out
PyObject* gate_up_swiglu(Arguments a) {
    void* stream = current_stream();
    const Descriptor gate = descriptor_of(a[0], stream), up = descriptor_of(a[1], stream);
    const at::Tensor& x = tensor_of(a[2]);
    Output out(a[3], 1, gate.output_dim, x.device());
    call("gate_up_swiglu", lib.nfn_mi355_k_quant_mmvq_gate_up_swiglu_float32_v1, &gate, &up, floats_of(x), out.data,
         stream);
    return out.take();
}

// gate, up, x or None, rows, workspace, out
PyObject* gate_up_swiglu_rows(Arguments a) {
    void* stream = current_stream();
    const Descriptor gate = descriptor_of(a[0], stream), up = descriptor_of(a[1], stream);
    const float* x = floats_or_null(a[2]);
    const std::int64_t rows = integer_of(a[3]);
    const at::Tensor& workspace = tensor_of(a[4]);
    Output out(a[5], rows, gate.output_dim, workspace.device());
    call("gate_up_swiglu_rows", lib.nfn_mi355_k_quant_mmq_gate_up_swiglu_float32_v1, &gate, &up, x, out.data, rows,
         workspace.data_ptr(), workspace.numel(), stream);
    return out.take();
}

// x, residual, first weight, first centered, second weight, second centered, first eps,
// second eps, handoff workspace or None, verifier family
PyObject* dual_rms_add_capture(Arguments a) {
    void* stream = current_stream();
    const at::Tensor& x = tensor_of(a[0]);
    const at::Tensor& residual = tensor_of(a[1]);
    if (x.dim() != 2) raise(PyExc_ValueError, "x is [rows, width]");
    const std::int64_t rows = x.size(0), width = x.size(1);
    const OptionalWeight first(a[2], stream), second(a[4], stream);
    const bool first_centered = truth_of(a[3]), second_centered = truth_of(a[5]);
    const float first_eps = static_cast<float>(number_of(a[6])), second_eps = static_cast<float>(number_of(a[7]));
    Output hidden(Py_None, x), normalized(Py_None, x), captured(Py_None, x);
    if (a[8] == Py_None) {
        call("dual_rms_add_capture", lib.nfn_native_tile_glimmer_dual_rms_add_capture_float32_v1, floats_of(x),
             first.pointer, floats_of(residual), hidden.data, second.pointer, normalized.data, captured.data, rows,
             width, first_eps, first_centered, second_eps, second_centered, stream);
    } else {
        const at::Tensor& workspace = tensor_of(a[8]);
        const bool verifier = truth_of(a[9]);
        const auto entry = rows == 1 ? lib.nfn_native_tile_glimmer_dual_rms_add_capture_mmvq_q8_float32_v1
            : verifier ? lib.nfn_mi355_dual_rms_add_capture_mmvq_rows_float32_v1
                       : lib.nfn_mi355_dual_rms_add_capture_mmq_f16_float32_v1;
        call(rows == 1 ? "dual_rms_add_capture_mmvq_q8"
             : verifier ? "dual_rms_add_capture_mmvq_rows" : "dual_rms_add_capture_mmq_f16",
             entry, floats_of(x), first.pointer, floats_of(residual), hidden.data, second.pointer, normalized.data,
             captured.data, rows, width, first_eps, first_centered, second_eps, second_centered, workspace.data_ptr(),
             workspace.numel(), stream);
    }
    return Py_BuildValue("(NNN)", hidden.take(), normalized.take(), captured.take());
}

// x, residual, weights, first weight, first centered, second weight, second centered, first eps,
// second eps, outputs
PyObject* dual_rms_multi_linear(Arguments a) {
    void* stream = current_stream();
    const at::Tensor& x = tensor_of(a[0]);
    const at::Tensor& residual = tensor_of(a[1]);
    if (x.dim() != 2) raise(PyExc_ValueError, "x is [rows, width]");
    const std::int64_t width = x.size(1);
    const OptionalWeight first(a[3], stream), second(a[5], stream);
    const bool first_centered = truth_of(a[4]), second_centered = truth_of(a[6]);
    const float first_eps = static_cast<float>(number_of(a[7])), second_eps = static_cast<float>(number_of(a[8]));
    Output hidden(Py_None, x), normalized(Py_None, x), captured(Py_None, x);
    Projections p(a[2], a[9], 1, x.device(), stream);
    call("dual_rms_mmvq_multi_linear", lib.nfn_mi355_dual_rms_mmvq_multi_linear_float32_v1, floats_of(x),
         first.pointer, floats_of(residual), hidden.data, second.pointer, normalized.data, captured.data, width,
         first_eps, first_centered, second_eps, second_centered, p.pointers.data(), p.outputs.data(), p.count(),
         stream);
    return Py_BuildValue("(NNNN)", hidden.take(), normalized.take(), captured.take(), p.take());
}

at::Tensor new_bytes(std::int64_t nbytes, c10::Device device) {
    return at::empty({nbytes}, at::TensorOptions().dtype(at::kByte).device(device));
}

// weight, x, workspace or None, indices or None, maxima or None
PyObject* lm_head_argmax(Arguments a) {
    void* stream = current_stream();
    const Descriptor descriptor = descriptor_of(a[0], stream);
    const at::Tensor& x = tensor_of(a[1]);
    const std::int64_t rows = x.size(0);
    at::Tensor workspace;
    if (a[2] != Py_None) {
        workspace = tensor_of(a[2]);
    } else {
        const std::int64_t nbytes = lib.nfn_mi355_lm_head_argmax_workspace_bytes_v1(rows, descriptor.output_dim);
        if (nbytes <= 0) raise(PyExc_ValueError, "lm_head_argmax supports 1..16 rows");
        workspace = new_bytes(nbytes, x.device());
    }
    const at::Tensor indices = a[3] != Py_None ? tensor_of(a[3])
        : at::empty({rows}, at::TensorOptions().dtype(at::kLong).device(x.device()));
    const at::Tensor maxima = a[4] != Py_None ? tensor_of(a[4])
        : at::empty({rows}, at::TensorOptions().dtype(at::kFloat).device(x.device()));
    call("lm_head_argmax", lib.nfn_mi355_lm_head_argmax_v1, &descriptor, floats_of(x),
         static_cast<std::int64_t*>(indices.data_ptr()), floats_of(maxima), rows, workspace.data_ptr(),
         workspace.numel(), stream);
    return Py_BuildValue("(NN)", THPVariable_Wrap(indices), THPVariable_Wrap(maxima));
}

at::Tensor gemm_workspace(PyObject* given, const Descriptor* descriptors, std::int64_t count, std::int64_t rows,
                          int mode, c10::Device device) {
    if (given != Py_None) return tensor_of(given);
    c10::SmallVector<std::int64_t, 4> widths;
    for (std::int64_t i = 0; i < count; ++i) widths.push_back(descriptors[i].output_dim);
    const std::int64_t nbytes = count == 0 ? 0 : lib.nfn_mi355_k_quant_gemm_multi_workspace_bytes_v1(
        rows, descriptors[0].input_dim, widths.data(), count, mode);
    if (nbytes <= 0) raise(PyExc_ValueError, "unsupported GEMM geometry or mode");
    return new_bytes(nbytes, device);
}

// weight, x, mode, workspace, out
PyObject* gemm(Arguments a) {
    void* stream = current_stream();
    const Descriptor descriptor = descriptor_of(a[0], stream);
    const at::Tensor& x = tensor_of(a[1]);
    const std::int64_t rows = x.size(0);
    const int mode = static_cast<int>(integer_of(a[2]));
    const at::Tensor workspace = gemm_workspace(a[3], &descriptor, 1, rows, mode, x.device());
    Output out(a[4], rows, descriptor.output_dim, x.device());
    call("k_quant_gemm", lib.nfn_mi355_k_quant_gemm_float32_v1, &descriptor, floats_of(x), out.data, rows,
         workspace.data_ptr(), workspace.numel(), mode, stream);
    return out.take();
}

// weights, x, mode, workspace, outputs
PyObject* gemm_multi(Arguments a) {
    void* stream = current_stream();
    const at::Tensor& x = tensor_of(a[1]);
    const std::int64_t rows = x.size(0);
    const int mode = static_cast<int>(integer_of(a[2]));
    Projections p(a[0], a[4], rows, x.device(), stream);
    const at::Tensor workspace = gemm_workspace(a[3], p.descriptors.data(), p.count(), rows, mode, x.device());
    call("k_quant_gemm_multi", lib.nfn_mi355_k_quant_gemm_multi_float32_v1, p.pointers.data(), floats_of(x),
         p.outputs.data(), p.count(), rows, workspace.data_ptr(), workspace.numel(), mode, stream);
    return p.take();
}

// query, key, query weight, key weight, eps, query scale, position, theta, layout, apply rope,
// query centered, key centered
PyObject* qk_norm_scale_rope(Arguments a) {
    void* stream = current_stream();
    const at::Tensor& query = tensor_of(a[0]);
    const at::Tensor& key = tensor_of(a[1]);
    const OptionalWeight query_weight(a[2], stream), key_weight(a[3], stream);
    const float eps = static_cast<float>(number_of(a[4])), scale = static_cast<float>(number_of(a[5]));
    const std::int64_t position = integer_of(a[6]);
    const float theta = static_cast<float>(number_of(a[7]));
    const std::uint32_t layout = static_cast<std::uint32_t>(integer_of(a[8]));
    const bool rope = truth_of(a[9]), query_centered = truth_of(a[10]), key_centered = truth_of(a[11]);
    if (query.dim() == 3) {
        call("qk_norm_scale_rope_batch", lib.nfn_native_tile_glimmer_qk_norm_scale_rope_batch_float32_v1,
             floats_of(query), floats_of(key), query_weight.pointer, key_weight.pointer, query.size(0), query.size(1),
             key.size(1), query.size(2), eps, query_centered, key_centered, scale, position, theta, layout, rope,
             stream);
    } else {
        if (query.dim() != 2) raise(PyExc_ValueError, "query is [heads, head_dim] or [rows, heads, head_dim]");
        call("qk_norm_scale_rope", lib.nfn_native_tile_glimmer_qk_norm_scale_rope_float32_v1, floats_of(query),
             floats_of(key), query_weight.pointer, key_weight.pointer, query.size(0), key.size(0), query.size(1), eps,
             query_centered, key_centered, scale, position, theta, layout, rope, stream);
    }
    Py_RETURN_NONE;
}

void require_matrix(const at::Tensor& tensor, const char* text) {
    if (tensor.dim() != 2) raise(PyExc_ValueError, text);
}

// query, key, value, key cache, value cache, position, first key position, attention scale,
// query weight, key weight, eps, query scale, theta, layout, apply rope, out, device position,
// sliding window, workspace
PyObject* fused_decode_attention(Arguments a) {
    void* stream = current_stream();
    const at::Tensor& query = tensor_of(a[0]);
    const at::Tensor& key = tensor_of(a[1]);
    const at::Tensor& value = tensor_of(a[2]);
    const at::Tensor& key_cache = tensor_of(a[3]);
    const at::Tensor& value_cache = tensor_of(a[4]);
    require_matrix(query, "query is [heads, head_dim]");
    require_matrix(key_cache, "a cache is [capacity, row stride]");
    NfnNativeTileGlimmerFusedDecodeAttentionDescriptorV1 d;
    std::memset(&d, 0, sizeof(d));
    d.struct_size = sizeof(d);
    d.version = 1;
    d.query = floats_of(query);
    d.key = floats_of(key);
    d.current_value = floats_of(value);
    d.key_cache_bf16 = static_cast<decltype(d.key_cache_bf16)>(key_cache.data_ptr());
    d.value_cache_bf16 = static_cast<decltype(d.value_cache_bf16)>(value_cache.data_ptr());
    if (a[8] != Py_None) {
        d.query_norm_weight = descriptor_of(a[8], stream);
        d.has_query_norm_weight = 1;
    }
    if (a[9] != Py_None) {
        d.key_norm_weight = descriptor_of(a[9], stream);
        d.has_key_norm_weight = 1;
    }
    d.query_heads = query.size(0);
    d.head_dim = query.size(1);
    d.kv_heads = key.size(0);
    d.position = integer_of(a[5]);
    d.first_key_position = integer_of(a[6]);
    d.cache_capacity = key_cache.size(0);
    d.cache_row_stride = key_cache.size(1);
    d.attention_scale = static_cast<float>(number_of(a[7]));
    d.norm_eps = static_cast<float>(number_of(a[10]));
    d.query_scale = static_cast<float>(number_of(a[11]));
    d.rope_theta = static_cast<float>(number_of(a[12]));
    d.rope_layout = static_cast<std::uint32_t>(integer_of(a[13]));
    d.apply_rope = truth_of(a[14]) ? 1 : 0;
    d.cuda_stream = stream;
    Output out(a[15], query);
    d.output = out.data;
    const bool device_position = a[16] != Py_None, split = a[18] != Py_None;
    const auto* where = device_position ? static_cast<const std::int64_t*>(tensor_of(a[16]).data_ptr()) : nullptr;
    const std::int64_t window = integer_of(a[17]);
    void* scratch = split ? tensor_of(a[18]).data_ptr() : nullptr;
    const std::int64_t scratch_bytes = split ? tensor_of(a[18]).numel() : 0;
    if (split && device_position) {
        call("fused_decode_attention_split_device_position",
             lib.nfn_mi355_fused_decode_attention_split_device_position_v1, &d, where, window, scratch,
             scratch_bytes);
    } else if (split) {
        call("fused_decode_attention_split", lib.nfn_mi355_fused_decode_attention_split_v1, &d, scratch,
             scratch_bytes);
    } else if (device_position) {
        call("fused_decode_attention_device_position",
             lib.nfn_native_tile_glimmer_fused_decode_attention_device_position_float32_v1, &d, where, window);
    } else {
        call("fused_decode_attention", lib.nfn_native_tile_glimmer_fused_decode_attention_float32_v1, &d);
    }
    return out.take();
}

// query, current key, current value, key cache, value cache, position, first key position, scale,
// out, workspace
PyObject* gqa_decode(Arguments a) {
    const at::Tensor& query = tensor_of(a[0]);
    const at::Tensor& key = tensor_of(a[1]);
    const at::Tensor& key_cache = tensor_of(a[3]);
    require_matrix(query, "query is [heads, head_dim]");
    require_matrix(key_cache, "a cache is [capacity, row stride]");
    NfnNativeTileGlimmerGqaDecodeDescriptorV1 d;
    std::memset(&d, 0, sizeof(d));
    d.struct_size = sizeof(d);
    d.version = 1;
    d.query = floats_of(query);
    d.current_key = floats_of(key);
    d.current_value = floats_of(tensor_of(a[2]));
    d.key_cache_bf16 = static_cast<decltype(d.key_cache_bf16)>(key_cache.data_ptr());
    d.value_cache_bf16 = static_cast<decltype(d.value_cache_bf16)>(tensor_of(a[4]).data_ptr());
    d.query_heads = query.size(0);
    d.head_dim = query.size(1);
    d.kv_heads = key.size(0);
    d.position = integer_of(a[5]);
    d.first_key_position = integer_of(a[6]);
    d.cache_capacity = key_cache.size(0);
    d.cache_row_stride = key_cache.size(1);
    d.scale = static_cast<float>(number_of(a[7]));
    d.cuda_stream = current_stream();
    Output out(a[8], query);
    d.output = out.data;
    if (a[9] != Py_None) {
        const at::Tensor& workspace = tensor_of(a[9]);
        call("gqa_decode_split", lib.nfn_mi355_gqa_decode_split_v1, &d, workspace.data_ptr(), workspace.numel());
    } else {
        call("gqa_decode", lib.nfn_native_tile_glimmer_gqa_decode_float32_v1, &d);
    }
    return out.take();
}

// query, block key, block value, key cache, value cache, context length, sliding window, scale,
// causal, out, workspace
PyObject* block_attention(Arguments a) {
    const at::Tensor& query = tensor_of(a[0]);
    const at::Tensor& key = tensor_of(a[1]);
    const at::Tensor& key_cache = tensor_of(a[3]);
    if (query.dim() != 3 || key.dim() != 3) raise(PyExc_ValueError, "a block is [rows, heads, head_dim]");
    require_matrix(key_cache, "a cache is [capacity, row stride]");
    NfnNativeTileDFlashBlockAttentionDescriptorV1 d;
    std::memset(&d, 0, sizeof(d));
    d.struct_size = sizeof(d);
    d.version = 1;
    d.flags = truth_of(a[8]) ? 1 : 0;
    d.query = floats_of(query);
    d.block_key = floats_of(key);
    d.block_value = floats_of(tensor_of(a[2]));
    d.key_cache_bf16 = static_cast<decltype(d.key_cache_bf16)>(key_cache.data_ptr());
    d.value_cache_bf16 = static_cast<decltype(d.value_cache_bf16)>(tensor_of(a[4]).data_ptr());
    d.query_rows = query.size(0);
    d.query_heads = query.size(1);
    d.head_dim = query.size(2);
    d.block_rows = key.size(0);
    d.kv_heads = key.size(1);
    d.context_length = integer_of(a[5]);
    d.sliding_window = integer_of(a[6]);
    d.cache_capacity = key_cache.size(0);
    d.cache_row_stride = key_cache.size(1);
    d.scale = static_cast<float>(number_of(a[7]));
    d.cuda_stream = current_stream();
    Output out(a[9], query);
    d.output = out.data;
    if (a[10] != Py_None) {
        const at::Tensor& workspace = tensor_of(a[10]);
        call("block_attention_split", lib.nfn_mi355_dflash_block_attention_split_v1, &d, workspace.data_ptr(),
             workspace.numel());
    } else {
        call("block_attention", lib.nfn_native_tile_dflash_block_attention_float32_v1, &d);
    }
    return out.take();
}

// -- module --------------------------------------------------------------------------------------

template <PyObject* (*Function)(Arguments), int Count>
PyObject* guarded(PyObject*, PyObject* const* arguments, Py_ssize_t count) {
    if (count != Count) {
        PyErr_Format(PyExc_TypeError, "%d arguments are expected", Count);
        return nullptr;
    }
    try {
        return Function(arguments);
    } catch (const Raised&) {
        return nullptr;
    } catch (...) {  // as torch's own bindings raise it (no memory: torch.OutOfMemoryError)
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

// bind(addresses: dict of name -> int, check): the library's entry points and tile_ops.check
PyObject* bind(PyObject*, PyObject* arguments) {
    PyObject *addresses, *check;
    if (!PyArg_ParseTuple(arguments, "O!O", &PyDict_Type, &addresses, &check)) return nullptr;
    Library bound;
    const auto address_of = [&](const char* name) -> void* {
        PyObject* value = PyDict_GetItemString(addresses, name);
        if (value == nullptr) {
            PyErr_SetString(PyExc_KeyError, name);
            return nullptr;
        }
        return PyLong_AsVoidPtr(value);
    };
#define NFN_BIND(name)                                                              \
    bound.name = reinterpret_cast<decltype(&::name)>(address_of(#name));            \
    if (bound.name == nullptr) return nullptr;
    NFN_ENTRY_POINTS(NFN_BIND)
#undef NFN_BIND
    lib = bound;
    Py_INCREF(check);
    Py_XDECREF(check_callable);
    check_callable = check;
    Py_RETURN_NONE;
}

PyObject* stream_handle(PyObject*, PyObject*) {
    try {
        return PyLong_FromVoidPtr(current_stream());
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

PyObject* entry_points(PyObject*, PyObject*) {
    PyObject* names = PyList_New(0);
    if (names == nullptr) return nullptr;
    for (const char* name : {
#define NFN_NAME(entry) #entry,
             NFN_ENTRY_POINTS(NFN_NAME)
#undef NFN_NAME
         }) {
        PyObject* text = PyUnicode_FromString(name);
        if (text == nullptr || PyList_Append(names, text) < 0) {
            Py_XDECREF(text);
            Py_DECREF(names);
            return nullptr;
        }
        Py_DECREF(text);
    }
    return names;
}

#define NFN_METHOD(name, count) \
    {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&guarded<name, count>)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"entry_points", entry_points, METH_NOARGS, nullptr},
    {"stream_handle", stream_handle, METH_NOARGS, nullptr},
    NFN_METHOD(multi_linear, 7),
    NFN_METHOD(multi_linear_prequantized, 5),
    NFN_METHOD(mmvq_linear, 4),
    NFN_METHOD(linear, 3),
    NFN_METHOD(gate_up_swiglu, 4),
    NFN_METHOD(gate_up_swiglu_rows, 6),
    NFN_METHOD(dual_rms_add_capture, 10),
    NFN_METHOD(dual_rms_multi_linear, 10),
    NFN_METHOD(lm_head_argmax, 5),
    NFN_METHOD(gemm, 5),
    NFN_METHOD(gemm_multi, 5),
    NFN_METHOD(qk_norm_scale_rope, 12),
    NFN_METHOD(fused_decode_attention, 19),
    NFN_METHOD(gqa_decode, 10),
    NFN_METHOD(block_attention, 11),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef definition = {PyModuleDef_HEAD_INIT, "_front_end", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front_end() {
    name_encoding = PyUnicode_InternFromString("encoding");
    name_output_dim = PyUnicode_InternFromString("output_dim");
    name_input_dim = PyUnicode_InternFromString("input_dim");
    name_data = PyUnicode_InternFromString("data");
    return PyModule_Create(&definition);
}
