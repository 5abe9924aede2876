// abh_bind.cpp -- the host's per-tensor work of one update, natively (Python module _bind).
//
// What a step asks of the host is, for every parameter, to look at its gradient, check it and fill
// the parameter's adambridge_segment.  Through Python that took 2.1 us a tensor, more than the
// kernel for models of many small ones: a step of 74 tensors (6.8M elements, 36 us of kernel) takes
// 198 us of host by the engine's general path and 45 by these loops, which go through the tensors' C++
// objects and the slots' attributes (6 tensors: 44 and 21).  Nothing is kept from one call to the next:
// every address, type and size is read again.
//
// A call takes the ordinary update only (contiguous tensors of plain types on one device, weights
// written in place); describe() says so before it has changed anything, and the engine's general
// path takes the rest.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <new>
#include <vector>

#include "../../include/adambridge_hip.h"

namespace {

PyObject *k_submitted, *k_param, *k_grad, *k_state, *k_bound, *k_plain, *k_in_place, *k_group, *k_step, *k_seg_addr, *k_small;

// A new reference that ends with the scope.
struct Ref {
    PyObject* o;
    explicit Ref(PyObject* p) : o(p) {}
    ~Ref() { Py_XDECREF(o); }
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
    explicit operator bool() const { return o != nullptr; }
};

// 1, 0, or -1 with an exception: the attribute's truth.
int truth(PyObject* o, PyObject* name)
{
    const Ref v(PyObject_GetAttr(o, name));
    return v ? PyObject_IsTrue(v.o) : -1;
}

// 1, 0 or -1: whether the attribute is None.
int is_none(PyObject* o, PyObject* name)
{
    const Ref v(PyObject_GetAttr(o, name));
    return v ? v.o == Py_None : -1;
}

int type_code(at::ScalarType t)
{
    return t == at::kFloat ? ADAMBRIDGE_DT_F32 : t == at::kBFloat16 ? ADAMBRIDGE_DT_BF16 : ADAMBRIDGE_DT_NONE;
}

// A tensor whose memory the kernel can take as it is: not a subclass, strided, contiguous, of the
// kernel's types, on the device.
const at::Tensor* plain_tensor(PyObject* o, int64_t device, int64_t numel)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.device().index() != device) return nullptr;
    if (t.numel() != numel || !t.is_contiguous() || type_code(t.scalar_type()) == ADAMBRIDGE_DT_NONE) return nullptr;
    return &t;
}

// One slot's update, checked and not yet written.
struct Found {
    adambridge_segment* seg;
    PyObject* slot;
    const void* g;
    void* out;
    const adambridge_group* group;
    int64_t step;
    int32_t g_dtype, out_dtype;
};

// describe(slots, grads, array, device, algorithm, delay, group_address) -> bool
//
// Fills the segment of every slot for its next update with its gradient, counts the step, and
// writes the segments' addresses to `array` (a ctypes array of pointers).  False, with nothing
// changed, if any slot needs the general path.  group_address(group) gives the address of a
// parameter group's adambridge_group, refreshed from its dict; it is called once per group.
PyObject* describe_slots(PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 7 || !PyList_CheckExact(args[0]) || !PyList_CheckExact(args[1])) {
        PyErr_SetString(PyExc_TypeError, "describe(slots, grads, array, device, algorithm, delay, group_address)");
        return nullptr;
    }
    PyObject *slots = args[0], *grads = args[1];
    const Py_ssize_t n = PyList_GET_SIZE(slots);
    const long device = PyLong_AsLong(args[3]);
    const long algorithm = PyLong_AsLong(args[4]);
    const int delay = PyObject_IsTrue(args[5]);
    if (PyErr_Occurred() || delay < 0) return nullptr;
    if (PyList_GET_SIZE(grads) != n) Py_RETURN_FALSE;
    std::vector<Found> found((size_t)n);
    std::vector<std::pair<PyObject*, const adambridge_group*>> groups;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* slot = PyList_GET_ITEM(slots, i);
        Found& f = found[(size_t)i];
        f.slot = slot;
        const int submitted = truth(slot, k_submitted), plain = submitted == 0 ? truth(slot, k_plain) : submitted;
        if (submitted < 0 || plain < 0) return nullptr;
        if (submitted || !plain) Py_RETURN_FALSE;
        const Ref state(PyObject_GetAttr(slot, k_state)), bound(PyObject_GetAttr(slot, k_bound));
        const Ref param(PyObject_GetAttr(slot, k_param)), address(PyObject_GetAttr(slot, k_seg_addr));
        const Ref step(PyObject_GetAttr(slot, k_step)), group(PyObject_GetAttr(slot, k_group));
        if (!state || !bound || !param || !address || !step || !group) return nullptr;
        if (state.o == Py_None || state.o != bound.o) Py_RETURN_FALSE;
        f.seg = static_cast<adambridge_segment*>(PyLong_AsVoidPtr(address.o));
        f.step = PyLong_AsLongLong(step.o) + 1;
        if (PyErr_Occurred()) return nullptr;
        const at::Tensor* p = plain_tensor(param.o, device, f.seg->n);
        const at::Tensor* g = plain_tensor(PyList_GET_ITEM(grads, i), device, f.seg->n);
        if (!p || !g) Py_RETURN_FALSE;
        f.g = g->data_ptr();
        f.g_dtype = type_code(g->scalar_type());
        const int in_place = truth(slot, k_in_place);
        if (in_place < 0) return nullptr;
        // a delayed first update owes the parameter nothing (the engine's _describe)
        const bool writes = !in_place && !(delay && f.step == 1);
        f.out = writes ? p->data_ptr() : nullptr;
        f.out_dtype = writes ? type_code(p->scalar_type()) : ADAMBRIDGE_DT_NONE;
        if (writes && !f.out) Py_RETURN_FALSE;   // a parameter of no elements
        f.group = nullptr;
        for (const auto& held : groups)
            if (held.first == group.o) f.group = held.second;
        if (!f.group) {
            const Ref at(PyObject_CallOneArg(args[6], group.o));
            if (!at) return nullptr;
            f.group = static_cast<const adambridge_group*>(PyLong_AsVoidPtr(at.o));
            if (PyErr_Occurred()) return nullptr;
            groups.emplace_back(group.o, f.group);   // the slot keeps the dict alive
        }
    }
    Py_buffer view;
    if (PyObject_GetBuffer(args[2], &view, PyBUF_WRITABLE) < 0) return nullptr;
    if (view.len != (Py_ssize_t)(sizeof(void*) * (size_t)n)) {
        PyBuffer_Release(&view);
        PyErr_SetString(PyExc_ValueError, "describe: the array's length is not the slots'");
        return nullptr;
    }
    adambridge_segment** array = static_cast<adambridge_segment**>(view.buf);
    for (Py_ssize_t i = 0; i < n; ++i) {
        const Found& f = found[(size_t)i];
        const Ref step(PyLong_FromLongLong(f.step));
        if (!step || PyObject_SetAttr(f.slot, k_step, step.o) < 0) {   // out of memory: the counts so far go back
            for (Py_ssize_t k = 0; k < i; ++k) {
                PyErr_Clear();
                const Ref old(PyLong_FromLongLong(found[(size_t)k].step - 1));
                if (old) PyObject_SetAttr(found[(size_t)k].slot, k_step, old.o);
            }
            PyBuffer_Release(&view);
            return PyErr_NoMemory();
        }
        adambridge_segment* s = f.seg;
        s->g = const_cast<void*>(f.g);
        s->g_dtype = f.g_dtype;
        s->out = f.out;
        s->out_dtype = f.out_dtype;
        s->group = const_cast<adambridge_group*>(f.group);
        s->step = f.step;
        s->offset = 0;
        s->algorithm = (int32_t)algorithm;
        s->reserved = delay && f.out ? ADAMBRIDGE_SEG_OUT_PREVIOUS : 0;
        array[i] = s;
    }
    PyBuffer_Release(&view);
    Py_RETURN_TRUE;
}

// C++ exceptions end here.  Torch's come from the checks (a tensor without memory of its own), before
// anything was written: the general path meets the same tensor and raises in Python.
PyObject* describe(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    try {
        return describe_slots(args, nargs);
    } catch (const std::bad_alloc&) {
        return PyErr_NoMemory();
    } catch (const std::exception&) {
        PyErr_Clear();
        Py_RETURN_FALSE;
    }
}

// pending(slots, include_small) -> (slots, grads): those not updated in this step that have a gradient.
PyObject* pending_slots(PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 2 || !PyList_CheckExact(args[0])) {
        PyErr_SetString(PyExc_TypeError, "pending(slots, include_small)");
        return nullptr;
    }
    const int small = PyObject_IsTrue(args[1]);
    const Ref slots(PyList_New(0)), grads(PyList_New(0));
    if (small < 0 || !slots || !grads) return nullptr;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[0]); ++i) {
        PyObject* slot = PyList_GET_ITEM(args[0], i);
        const int submitted = truth(slot, k_submitted);
        if (submitted < 0) return nullptr;
        if (submitted) continue;
        const Ref param(PyObject_GetAttr(slot, k_param));
        if (!param) return nullptr;
        PyObject* found = nullptr;
        if (THPVariable_CheckExact(param.o)) {
            const at::Tensor& g = THPVariable_Unpack(param.o).grad();
            if (!g.defined()) continue;
            found = THPVariable_Wrap(g);
        } else {
            found = PyObject_GetAttr(param.o, k_grad);
        }
        const Ref grad(found);
        if (!grad) return nullptr;
        if (grad.o == Py_None) continue;
        if (!small) {
            const int none = is_none(slot, k_small);
            if (none < 0) return nullptr;
            if (!none) continue;
        }
        if (PyList_Append(slots.o, slot) < 0 || PyList_Append(grads.o, grad.o) < 0) return nullptr;
    }
    return PyTuple_Pack(2, slots.o, grads.o);
}

PyObject* pending(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    try {
        return pending_slots(args, nargs);
    } catch (const std::bad_alloc&) {
        return PyErr_NoMemory();
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// mark(slots, submitted): sets the flag of each.
PyObject* mark(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 2 || !PyList_CheckExact(args[0]) || !PyBool_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "mark(slots, submitted)");
        return nullptr;
    }
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[0]); ++i)
        if (PyObject_SetAttr(PyList_GET_ITEM(args[0], i), k_submitted, args[1]) < 0) return nullptr;
    Py_RETURN_NONE;
}

// record(grads, stream_id, device): each tensor's memory waits for the stream before it is used again.
PyObject* record(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 3 || !PyList_CheckExact(args[0])) {
        PyErr_SetString(PyExc_TypeError, "record(grads, stream_id, device)");
        return nullptr;
    }
    const long long id = PyLong_AsLongLong(args[1]);
    const long device = PyLong_AsLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    try {
        const c10::Stream stream(c10::Stream::UNSAFE, c10::Device(c10::kCUDA, (c10::DeviceIndex)device), id);
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[0]); ++i) {
            PyObject* g = PyList_GET_ITEM(args[0], i);
            if (THPVariable_Check(g)) THPVariable_Unpack(g).record_stream(stream);
        }
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
    Py_RETURN_NONE;
}

#define ABH_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef kMethods[] = {
    {"describe", ABH_FAST(describe), "Fill the segments of an ordinary update; False if it is not one."},
    {"pending", ABH_FAST(pending), "Slots with a gradient and no update yet, and their gradients."},
    {"mark", ABH_FAST(mark), "Set every slot's submitted flag."},
    {"record", ABH_FAST(record), "record_stream for every tensor."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_bind", "Per-tensor host work of an update.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bind()
{
    const struct { PyObject** at; const char* name; } names[] = {
        {&k_submitted, "submitted"}, {&k_param, "param"}, {&k_grad, "grad"}, {&k_state, "state"}, {&k_bound, "bound"},
        {&k_plain, "plain"}, {&k_in_place, "in_place"}, {&k_group, "group"}, {&k_step, "step"}, {&k_seg_addr, "seg_addr"},
        {&k_small, "small"}};
    for (const auto& n : names)
        if (!(*n.at = PyUnicode_InternFromString(n.name))) return nullptr;
    return PyModule_Create(&kModule);
}
