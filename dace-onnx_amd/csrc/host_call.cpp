// The host's part of a model's call: its tensors checked and their addresses collected in one step, then its launches.
//
// A call of a graph of N weights looks every weight up by name, checks that it still is a plain contiguous tensor of its type and shape
// on the GPU, and passes its address on. From Python that is 0.8 us for each tensor and was most of a call's host time (22 of 43 us for
// an encoder layer, 53 of 103 for an image classifier of 15 launches); here it is a few hundredths: 32 and 58 us, a quantised layer of one launch
// 14.3 -> 8.1, a dense classifier of four 25.7 -> 18.3. What is left are the runtime's launches, 3 us each. Nothing is taken over from one call to
// the next: whatever is not a plain tensor of the declared kind (a subclass, a wrapper of a transform, another device, type, shape or
// order) makes `call` return None before anything is launched, and the caller goes the general way, which converts it or refuses it.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <stdint.h>

#include <vector>

namespace {

using ProgramRun = int64_t (*)(const int64_t*, int64_t, int64_t, const int64_t*, int64_t, const int64_t*, void*);

enum Kind { INPUT, OUTPUT, WEIGHT, PACKED };

struct Slot {
    long kind;
    Py_ssize_t index;   // of the input, output or packed copy
    PyObject* name;     // of the weight
    at::ScalarType type;
    std::vector<int64_t> shape;
};

struct Plan {
    PyObject_HEAD
    std::vector<Slot>* slots;   // in the order in which the launches take the addresses
    Py_ssize_t inputs, outputs, weights;   // (a weight that the graph does not know is refused by the general way)
    ProgramRun run;
    int64_t fixed[5];           // program, words, calls, patches, number of patches
    int device;
    uint64_t keys[2];           // dispatch keys of a plain tensor of that device, made outside and inside of inference mode
    PyObject* owner;            // of the program
};

void plan_dealloc(PyObject* self) {
    Plan* plan = reinterpret_cast<Plan*>(self);
    if (plan->slots)
        for (Slot& s : *plan->slots) Py_XDECREF(s.name);
    delete plan->slots;
    Py_XDECREF(plan->owner);
    Py_TYPE(self)->tp_free(self);
}

bool plain(const Plan& plan, const at::Tensor& t, const Slot& s) {
    const uint64_t keys = t.key_set().raw_repr();
    return (keys == plan.keys[0] || keys == plan.keys[1]) && t.scalar_type() == s.type && t.sizes() == at::IntArrayRef(s.shape) &&
           t.device().index() == plan.device && t.is_contiguous();
}

// 1 where copy k (an object with a `record`: name of the weight, the tensor that was packed, its version or None, whether the copy is as good
// as the weight whoever holds that, the copy) stands for the weight now, 0 where not, -1 with an exception set. The record of a copy that
// was never made is None.
int current(PyObject* record, PyObject* weights, PyObject* made, PyObject* handed_out) {
    if (record == Py_None) return 0;
    PyObject *name = PyTuple_GET_ITEM(record, 0), *weight = PyTuple_GET_ITEM(record, 1), *version = PyTuple_GET_ITEM(record, 2);
    PyObject* now = PyDict_GetItemWithError(weights, name);
    if (!now) return PyErr_Occurred() ? -1 : 0;
    if (now != weight) return 0;
    if (version != Py_None) {
        const long long packed_at = PyLong_AsLongLong(version);
        if (packed_at == -1 && PyErr_Occurred()) return -1;
        if ((long long)THPVariable_Unpack(weight)._version() != packed_at) return 0;
    }
    if (PyTuple_GET_ITEM(record, 3) == Py_True) return 1;
    PyObject* own = PyDict_GetItemWithError(made, name);
    if (!own) return PyErr_Occurred() ? -1 : 0;
    if (own != weight) return 0;
    const int known = PySet_Contains(handed_out, name);
    return known < 0 ? -1 : !known;
}

// call(weights, made, handed_out, copies, inputs, stream) -> None, or (status, outputs, tensors in the order of the slots, their addresses)
PyObject* plan_call(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    const Plan& plan = *reinterpret_cast<Plan*>(self);
    if (nargs != 6 || !PyDict_Check(args[0]) || !PyDict_Check(args[1]) || !PyAnySet_Check(args[2]) || !PyList_Check(args[3]) || !PyTuple_Check(args[4]))
        return PyErr_Format(PyExc_TypeError, "call(weights, made, handed_out, copies, inputs, stream)");
    PyObject *weights = args[0], *made = args[1], *handed_out = args[2], *copies = args[3], *inputs = args[4];
    void* stream = PyLong_AsVoidPtr(args[5]);
    if (!stream && PyErr_Occurred()) return nullptr;
    if (PyTuple_GET_SIZE(inputs) != plan.inputs || PyDict_Size(weights) != plan.weights) Py_RETURN_NONE;

    const std::vector<Slot>& slots = *plan.slots;
    const Py_ssize_t count = (Py_ssize_t)slots.size();
    PyObject* bound = PyList_New(count);   // holds what it points to from here on, whatever other threads do to `weights`
    PyObject* addresses = bound ? PyBytes_FromStringAndSize(nullptr, count * (Py_ssize_t)sizeof(int64_t)) : nullptr;
    PyObject* outputs = addresses ? PyList_New(plan.outputs) : nullptr;
    PyObject* result = nullptr;
    bool taken = outputs != nullptr;
    try {
        int64_t* at = taken ? reinterpret_cast<int64_t*>(PyBytes_AS_STRING(addresses)) : nullptr;
        for (Py_ssize_t i = 0; taken && i < count; ++i) {
            const Slot& s = slots[i];
            PyObject* object = nullptr;
            at[i] = 0;
            if (s.kind == OUTPUT) {
                continue;
            } else if (s.kind == INPUT) {
                object = PyTuple_GET_ITEM(inputs, s.index);
            } else if (s.kind == WEIGHT) {
                object = PyDict_GetItemWithError(weights, s.name);
            } else if (s.index < PyList_GET_SIZE(copies)) {
                static PyObject* const attribute = PyUnicode_InternFromString("record");
                PyObject* record = PyObject_GetAttr(PyList_GET_ITEM(copies, s.index), attribute);
                const int use = record ? current(record, weights, made, handed_out) : -1;
                object = use < 0 ? nullptr : use ? PyTuple_GET_ITEM(record, 4) : Py_None;
                Py_XINCREF(object);
                Py_XDECREF(record);
                if (!object) { taken = false; break; }
                PyList_SET_ITEM(bound, i, object);
                if (object == Py_None) continue;
            }
            if (!object || !THPVariable_CheckExact(object) || !plain(plan, THPVariable_Unpack(object), s)) { taken = false; break; }
            if (s.kind != PACKED) {
                Py_INCREF(object);
                PyList_SET_ITEM(bound, i, object);
            }
            at[i] = (int64_t)reinterpret_cast<uintptr_t>(THPVariable_Unpack(object).mutable_data_ptr());
        }
        if (taken) {
            std::vector<at::Tensor> made_here((size_t)plan.outputs);
            int64_t status = 0;
            Py_BEGIN_ALLOW_THREADS
            try {
                for (Py_ssize_t i = 0; taken && i < count; ++i) {
                    const Slot& s = slots[i];
                    if (s.kind != OUTPUT) continue;
                    made_here[s.index] = at::empty(s.shape, at::TensorOptions().dtype(s.type).device(at::kCUDA, (at::DeviceIndex)plan.device));
                    taken = plain(plan, made_here[s.index], s);
                    if (taken) at[i] = (int64_t)reinterpret_cast<uintptr_t>(made_here[s.index].mutable_data_ptr());
                }
                if (taken) status = plan.run(reinterpret_cast<const int64_t*>(plan.fixed[0]), plan.fixed[1], plan.fixed[2], reinterpret_cast<const int64_t*>(plan.fixed[3]), plan.fixed[4], at, stream);
            } catch (...) {   // out of memory, say: the general way runs into it too, and reports it
                taken = false;
            }
            Py_END_ALLOW_THREADS
            for (Py_ssize_t i = 0; taken && i < count; ++i) {
                if (slots[i].kind != OUTPUT) continue;
                PyObject* output = THPVariable_Wrap(made_here[slots[i].index]);
                if (!output) { taken = false; break; }
                Py_INCREF(output);
                PyList_SET_ITEM(bound, i, output);
                PyList_SET_ITEM(outputs, slots[i].index, output);
            }
            if (taken) result = Py_BuildValue("LOOO", (long long)status, outputs, bound, addresses);
        }
    } catch (...) {
        taken = false;
    }
    Py_XDECREF(bound);
    Py_XDECREF(addresses);
    Py_XDECREF(outputs);
    if (result || PyErr_Occurred()) return result;
    Py_RETURN_NONE;
}

PyMethodDef plan_methods[] = {{"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(plan_call)), METH_FASTCALL, "one call of the model"}, {nullptr, nullptr, 0, nullptr}};

PyTypeObject plan_type = {PyVarObject_HEAD_INIT(nullptr, 0) "_host_call.Plan"};

uint64_t keys_of(PyObject* tensor) { return THPVariable_CheckExact(tensor) ? THPVariable_Unpack(tensor).key_set().raw_repr() : 0; }

// plan(run, (program, words, calls, patches, number of patches), owner, slots, inputs, outputs, weights, device, plain, plain in inference mode)
// slots: (kind, index, name, an empty tensor of the type, shape)
PyObject* make_plan(PyObject*, PyObject* args) {
    unsigned long long run;
    long long fixed[5];
    PyObject *owner, *slots, *normal, *inference;
    Py_ssize_t inputs, outputs, weights;
    int device;
    if (!PyArg_ParseTuple(args, "K(LLLLL)OO!nnniOO", &run, &fixed[0], &fixed[1], &fixed[2], &fixed[3], &fixed[4], &owner, &PyList_Type, &slots, &inputs, &outputs,
                          &weights, &device, &normal, &inference))
        return nullptr;
    Plan* plan = PyObject_New(Plan, &plan_type);
    if (!plan) return nullptr;
    plan->slots = new std::vector<Slot>();
    plan->inputs = inputs;
    plan->outputs = outputs;
    plan->weights = weights;
    plan->run = reinterpret_cast<ProgramRun>((uintptr_t)run);
    for (int i = 0; i < 5; ++i) plan->fixed[i] = fixed[i];
    plan->device = device;
    plan->keys[0] = keys_of(normal);
    plan->keys[1] = keys_of(inference);
    Py_INCREF(owner);
    plan->owner = owner;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(slots); ++i) {
        PyObject *name, *type, *shape;
        Slot s;
        if (!PyArg_ParseTuple(PyList_GET_ITEM(slots, i), "lnOOO!", &s.kind, &s.index, &name, &type, &PyTuple_Type, &shape)) break;
        const Py_ssize_t limit = s.kind == INPUT ? inputs : s.kind == OUTPUT ? outputs : PY_SSIZE_T_MAX;
        if (s.kind < INPUT || s.kind > PACKED || s.index < 0 || s.index >= limit || !THPVariable_Check(type)) {
            PyErr_Format(PyExc_ValueError, "slot %zd", i);
            break;
        }
        for (Py_ssize_t d = 0; d < PyTuple_GET_SIZE(shape); ++d) s.shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d)));
        s.type = THPVariable_Unpack(type).scalar_type();
        Py_INCREF(name);
        s.name = name;
        plan->slots->push_back(std::move(s));
    }
    if (PyErr_Occurred()) {
        Py_DECREF(reinterpret_cast<PyObject*>(plan));
        return nullptr;
    }
    return reinterpret_cast<PyObject*>(plan);
}

PyMethodDef methods[] = {{"plan", make_plan, METH_VARARGS, "what the calls of one compiled model have in common"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_call", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host_call() {
    plan_type.tp_basicsize = sizeof(Plan);
    plan_type.tp_dealloc = plan_dealloc;
    plan_type.tp_flags = Py_TPFLAGS_DEFAULT;
    plan_type.tp_methods = plan_methods;
    if (PyType_Ready(&plan_type) < 0) return nullptr;
    PyObject* made = PyModule_Create(&module);
    if (made && PyModule_AddStringConstant(made, "built_against", BUILT_AGAINST) < 0) Py_CLEAR(made);   // torch, whose tensors are read by its inline functions
    return made;
}
