// The host side of a call in native code: what ElasticBuffer.dispatch / combine do between the caller and the C-ABI of this
// library (argument checks, output tensors, stream order, launches, the wait for the row count, the handle), as one CPython
// extension.  A decode step's kernels take about 15 us; the same work in Python took 80 (a dispatch + combine of 31 tokens of
// 256 columns, pass after pass), so the host path was what such a call cost.
//
// Contract with the Python layer (deepep_amd/elastic.py): every entry point here returns None, having done nothing, for
// a call it does not take: one that is invalid (the Python layer then finds out why and raises), or valid but unusual (tensor
// subclasses, inference mode, a handle whose attributes were replaced).  What it takes gives the results, exceptions and
// stream order of the Python layer.
//
// Order of a fresh dispatch, chosen so that the host's own work hides behind the GPU's: checks, three to six allocations,
// launch; then, while the GPU works, the tensor objects and the handle that do not depend on the row count; then the
// wait for the mailbox.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <vector>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/StreamGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/deepep_amd.h"

namespace {

// Bounds of the arguments, given by the Python layer, which has them for its own checks (configure).
int g_max_tokens, g_max_hidden, g_max_topk, g_max_experts, g_low_latency_max_tokens;
constexpr long long kWaitTimeoutUs = 100LL * 1000 * 1000;
constexpr int64_t kSmallBlock = 64 << 10;

// ---- small helpers ---------------------------------------------------------------------------------------------------
struct Ref {  // an owned reference
    PyObject* p = nullptr;
    Ref() = default;
    explicit Ref(PyObject* o) : p(o) {}
    Ref(Ref&& o) noexcept : p(o.p) { o.p = nullptr; }
    Ref& operator=(Ref&& o) noexcept
    {
        std::swap(p, o.p);
        return *this;
    }
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
    ~Ref() { Py_XDECREF(p); }
    PyObject* release()
    {
        PyObject* o = p;
        p = nullptr;
        return o;
    }
    explicit operator bool() const { return p != nullptr; }
};

inline PyObject* new_ref(PyObject* o)
{
    Py_INCREF(o);
    return o;
}

// Attribute and dictionary names, interned once.
#define DPEP_NAMES(X)                                                                                                          \
    X(acquire) X(release) X(current_stream_wait) X(_gpu_index) X(__dict__) X(_plan) X(_marker) X(event) X(_lease) X(num_experts)  \
    X(num_max_tokens_per_rank) X(num_compute_units) X(topk_idx) X(num_recv_tokens) X(num_expanded_tokens)                       \
    X(num_recv_tokens_per_expert_list) X(psum_num_recv_tokens_per_expert) X(num_unaligned_recv_tokens_per_expert)                \
    X(is_low_latency) X(route_to_row) X(weight_return_meta) X(expert_totals) X(expert_offsets) X(source_weights)                 \
    X(send_counts) X(rank) X(world_size) X(num_tokens) X(num_topk) X(hidden) X(metadata_only) X(metadata_version)                \
    X(_buffer_token) X(_row_to_route_full) X(do_expand) X(expert_alignment) X(gate_up) X(logical) X(_versions)
struct Names {
#define X(n) PyObject* n;
    DPEP_NAMES(X)
#undef X
} N;

PyObject* g_empty_tuple;
PyTypeObject* g_handle_type;     // deepep_amd.elastic.EPHandle
PyObject* g_handle_template;     // the __dict__ of a fresh EPHandle
PyTypeObject* g_overlap_type;    // deepep_amd.event.EventOverlap
PyTypeObject* g_event_type;      // deepep_amd.event.EventHandle
PyObject* g_native_error;        // deepep_amd._lib.NativeError

// Status of the C-ABI -> Python exception (as deepep_amd._lib.check).
PyObject* raise_native(int status)
{
    PyErr_SetString(status == DPEP_EINVAL ? PyExc_ValueError : g_native_error, dpep_last_error());
    return nullptr;
}
PyObject* raise_hip(const char* what, hipError_t err)
{
    PyErr_Format(g_native_error, "%s failed: %s", what, hipGetErrorString(err));
    return nullptr;
}

// The value of an exact int in [lower, upper], or `other`.
inline long long exact_int(PyObject* o, long long lower, long long upper, long long other = -1)
{
    if (!PyLong_CheckExact(o)) return other;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow != 0 || v < lower || v > upper ? other : v;
}
inline bool is_bool(PyObject* o) { return o == Py_True || o == Py_False; }

inline bool on_gpu(PyObject* o) { return THPVariable_CheckExact(o) && THPVariable_Unpack(o).is_cuda(); }
// A plain device tensor: exactly torch.Tensor (or Parameter), strided, contiguous, on `device`, without grad.
inline const at::Tensor* plain(PyObject* o, int device)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided || t.requires_grad() || !t.is_contiguous()) return nullptr;
    return &t;
}
inline bool has_shape(const at::Tensor& t, int64_t a, int64_t b) { return t.dim() == 2 && t.size(0) == a && t.size(1) == b; }
inline bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }

at::Tensor allocate(at::IntArrayRef sizes, at::ScalarType type, int device)
{
    return at::Tensor(at::detail::empty_cuda(sizes, type, c10::Device(c10::DeviceType::CUDA, device), std::nullopt));
}
// A contiguous tensor over `storage`, `offset` bytes in.  Not a view: it has a version counter of its own.
at::Tensor over(const c10::Storage& storage, int64_t offset, at::ScalarType type, at::IntArrayRef sizes)
{
    at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(storage), c10::DispatchKeySet(c10::DispatchKey::CUDA),
                                                            c10::scalarTypeToTypeMeta(type));
    t.unsafeGetTensorImpl()->set_storage_offset(offset / static_cast<int64_t>(c10::elementSize(type)));
    t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
    return t;
}
inline PyObject* wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
inline uint32_t version_of(const at::Tensor& t) { return t.unsafeGetTensorImpl()->version_counter().current_version(); }

// ---- stream order and what has to outlive it ------------------------------------------------------------------------------
// The event a buffer orders two streams with: recorded anew each time (a wait that has been queued refers to the recording it
// saw), so one suffices.  It orders streams of one GPU, so it carries no system-scope fence (hipEventDisableSystemFence):
// behind a fenced one a wait of another stream took 8-15 us of host time and 10 us of the GPU's, without the fence 7 and 7.
struct OrderEvent {
    hipEvent_t event;
    // `waits` waits for everything that `on` has been given so far.
    hipError_t order(hipStream_t waits, hipStream_t on)
    {
        hipError_t err = event != nullptr ? hipSuccess : hipEventCreateWithFlags(&event, hipEventDisableTiming | hipEventDisableSystemFence);
        if (err == hipSuccess) err = hipEventRecord(event, on);
        return err == hipSuccess ? hipStreamWaitEvent(waits, event, 0) : err;
    }
    void release()
    {
        if (event != nullptr) (void)hipEventDestroy(event);
        event = nullptr;
    }
};

// A counter that one stream raises and other streams wait for (dpep_stream_raise / hipStreamWaitValue64): the cheaper way to
// order two streams.  A recorded event plus a wait costs 8 us of host time and 7 of the GPU's when the event is still
// pending, this 4.5 and 5 (two streams passing the turn back and forth).  Only one stream at a time may raise a counter,
// or a later value could be seen before an earlier one was written; values only grow, so a counter may go from owner to owner.
// Counters are kept for the life of the process and reused, two for each buffer that lived at the same time as others.
struct Counter {
    uint64_t* word = nullptr;
    uint64_t raised = 0;
    int device = 0;
    bool reached(uint64_t value) const { return __atomic_load_n(word, __ATOMIC_ACQUIRE) >= value; }
};
std::vector<Counter*> g_idle_counters;  // (guarded by the GIL)
Counter* take_counter(int device)
{
    for (size_t i = 0; i < g_idle_counters.size(); ++i) {
        Counter* c = g_idle_counters[i];
        if (c->device != device) continue;
        g_idle_counters.erase(g_idle_counters.begin() + static_cast<long>(i));
        return c;
    }
    int able = 0;
    void* word = nullptr;
    if (hipDeviceGetAttribute(&able, hipDeviceAttributeCanUseStreamWaitValue, device) != hipSuccess || able == 0 ||
        hipExtMallocWithFlags(&word, sizeof(uint64_t), hipMallocSignalMemory) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    Counter* c = new Counter();
    c->word = static_cast<uint64_t*>(word);
    c->device = device;
    __atomic_store_n(c->word, 0, __ATOMIC_RELEASE);
    return c;
}
inline bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}

struct Stream {  // a torch stream: its raw handle and torch's identifier of it
    hipStream_t raw = nullptr;
    int64_t id = 0;
    bool operator==(const Stream& o) const { return raw == o.raw && id == o.id; }
    c10::Stream torch(int device) const { return c10::Stream::unpack3(id, static_cast<c10::DeviceIndex>(device), c10::DeviceType::CUDA); }
};
inline Stream current_stream(int device)
{
    const auto s = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device));
    return Stream{s.stream(), static_cast<int64_t>(s.id())};
}
// A torch stream object of Python -> Stream.
bool stream_from(PyObject* o, Stream* out)
{
    Ref raw(PyObject_GetAttrString(o, "cuda_stream")), id(PyObject_GetAttrString(o, "stream_id"));
    if (!raw || !id) return false;
    out->raw = reinterpret_cast<hipStream_t>(PyLong_AsVoidPtr(raw.p));
    out->id = PyLong_AsLongLong(id.p);
    return !PyErr_Occurred();
}
PyObject* stream_object(const Stream& s, int device)
{
    Ref torch_cuda(PyImport_ImportModule("torch.cuda"));
    if (!torch_cuda) return nullptr;
    Ref type(PyObject_GetAttrString(torch_cuda.p, "Stream"));
    if (!type) return nullptr;
    Ref kwargs(Py_BuildValue("{s:L,s:i,s:i}", "stream_id", static_cast<long long>(s.id), "device_index", device, "device_type",
                             static_cast<int>(c10::DeviceType::CUDA)));
    return kwargs ? PyObject_Call(type.p, g_empty_tuple, kwargs.p) : nullptr;
}

// A value of a stream's counter, reached when the stream has done what it was given before: what deepep_amd.event._Marker is for
// a torch event, with the methods that EventHandle and EventOverlap use.  Who asks the handle for its event gets one of torch's
// (deepep_amd.event.EventHandle.event).
struct Marker {
    PyObject_HEAD
    Counter* counter;
    uint64_t value;
    Stream stream;
    int device;
};
extern PyTypeObject MarkerType;

// Tensors kept alive for work on the communication stream.  `made`: tensors allocated by this very call, on the stream that
// was current (`home`): once home has waited for the work nothing further has to be declared to the allocator, because
// their memory is handed out again in home's order.  The others were declared as used by the communication stream when the
// call was made.
struct Lease {
    PyObject_HEAD
    std::vector<at::Tensor>* tensors;
    size_t made;      // the first `made` tensors
    Stream home, work;
    int device;
    bool joined;      // home has waited for the work
};
extern PyTypeObject LeaseType;

void lease_declare(Lease* l, const Stream& s, size_t from, size_t to)
{
    for (size_t i = from; i < to; ++i) (*l->tensors)[i].record_stream(s.torch(l->device));
}
void Lease_dealloc(PyObject* o)
{
    Lease* l = reinterpret_cast<Lease*>(o);
    if (!l->joined) {
        try {
            lease_declare(l, l->work, 0, l->made);
        } catch (...) {  // (nothing can be reported from here; the tensors are then released in their own stream's order)
        }
    }
    delete l->tensors;
    Py_TYPE(o)->tp_free(o);
}
// The consumer's stream now waits for the work: what the Python _Lease.touch does.
PyObject* Lease_touch(PyObject* o, PyObject*)
{
    HANDLE_TH_ERRORS
    Lease* l = reinterpret_cast<Lease*>(o);
    const Stream consumer = current_stream(l->device);
    if (consumer == l->home) l->joined = true;
    else lease_declare(l, consumer, 0, l->tensors->size());
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}
PyMethodDef lease_methods[] = {{"touch", Lease_touch, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyTypeObject LeaseType = {PyVarObject_HEAD_INIT(nullptr, 0) "deepep_amd._host.Lease", sizeof(Lease)};

// Marks what `stream` has been given so far; `stream` alone raises `counter`.
Marker* marker_new(Counter* counter, const Stream& stream, int device)
{
    if (int rc = dpep_stream_raise(counter->word, ++counter->raised, stream.raw); rc != DPEP_OK) return reinterpret_cast<Marker*>(raise_native(rc));
    Marker* m = reinterpret_cast<Marker*>(MarkerType.tp_alloc(&MarkerType, 0));
    if (m == nullptr) return nullptr;
    m->counter = counter;
    m->value = counter->raised;
    m->stream = stream;
    m->device = device;
    return m;
}
PyObject* marker_wait(Marker* m, hipStream_t s)
{
    if (!m->counter->reached(m->value))
        if (hipError_t err = hipStreamWaitValue64(s, m->counter->word, m->value, hipStreamWaitValueGte, ~0ull); err != hipSuccess)
            return raise_hip("hipStreamWaitValue64", err);
    Py_RETURN_NONE;
}
PyObject* Marker_hold_current_stream(PyObject* o, PyObject*)
{
    HANDLE_TH_ERRORS
    Marker* m = reinterpret_cast<Marker*>(o);
    if (c10::hip::current_device() != m->device) {
        PyErr_SetString(PyExc_RuntimeError, "Cannot wait for an event from another GPU");
        return nullptr;
    }
    return marker_wait(m, current_stream(m->device).raw);  // (None: a lease asks for the current stream itself)
    END_HANDLE_TH_ERRORS
}
PyObject* Marker_wait(PyObject* o, PyObject* stream)
{
    Stream s;
    return stream_from(stream, &s) ? marker_wait(reinterpret_cast<Marker*>(o), s.raw) : nullptr;
}
PyObject* Marker_get_gpu(PyObject* o, void*) { return PyLong_FromLong(reinterpret_cast<Marker*>(o)->device); }
PyObject* Marker_get_stream(PyObject* o, void*)
{
    Marker* m = reinterpret_cast<Marker*>(o);
    return stream_object(m->stream, m->device);
}
PyMethodDef marker_methods[] = {{"hold_current_stream", Marker_hold_current_stream, METH_NOARGS, nullptr},
                                {"wait", Marker_wait, METH_O, nullptr},
                                {nullptr, nullptr, 0, nullptr}};
PyGetSetDef marker_getset[] = {{"gpu", Marker_get_gpu, nullptr, nullptr, nullptr},
                               {"stream", Marker_get_stream, nullptr, nullptr, nullptr},
                               {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject MarkerType = {PyVarObject_HEAD_INIT(nullptr, 0) "deepep_amd._host.Marker", sizeof(Marker)};

// ---- a handle's routing, as the native path keeps it ----------------------------------------------------------------------
// The tensors of a handle under the names the handle has them, with their addresses and versions at dispatch time.  A cached
// dispatch or a combine goes through the native path only while the handle still has these very objects, unmodified.
struct Pinned {
    PyObject* name;    // borrowed from N
    PyObject* object;  // owned
    const void* data;
    uint32_t version;
};
struct Plan {
    PyObject_HEAD
    std::vector<Pinned>* pinned;
    std::vector<Pinned>* same;      // further attributes that must be the objects they were (no version check)
    at::Tensor* routing;            // owner of the routing storage
    at::Tensor* weights;            // low latency: the saved route weights
    const int32_t* route_to_row;
    const int32_t* row_to_route;
    PyObject* owner;                // owned: the buffer's token
    long long rows;                 // rows of the payload outputs (low latency: the capacity)
    int tokens, topk, hidden, experts;
    bool low_latency;
};
extern PyTypeObject PlanType;

void Plan_dealloc(PyObject* o)
{
    Plan* p = reinterpret_cast<Plan*>(o);
    for (auto* list : {p->pinned, p->same}) {
        if (list != nullptr)
            for (Pinned& e : *list) Py_XDECREF(e.object);
        delete list;
    }
    delete p->routing;
    delete p->weights;
    Py_XDECREF(p->owner);
    Py_TYPE(o)->tp_free(o);
}
Plan* plan_new()
{
    Plan* p = reinterpret_cast<Plan*>(PlanType.tp_alloc(&PlanType, 0));
    if (p == nullptr) return nullptr;
    p->pinned = new std::vector<Pinned>();
    p->pinned->reserve(5);
    p->same = new std::vector<Pinned>();
    p->same->reserve(16);
    p->routing = p->weights = nullptr;
    p->owner = nullptr;
    return p;
}
// {name: (address, version)} of the pinned tensors, for the Python layer's own check.
PyObject* Plan_versions(PyObject* o, PyObject*)
{
    Ref d(PyDict_New());
    if (!d) return nullptr;
    for (const Pinned& e : *reinterpret_cast<Plan*>(o)->pinned) {
        Ref v(Py_BuildValue("(NI)", PyLong_FromVoidPtr(const_cast<void*>(e.data)), e.version));
        if (!v || PyDict_SetItem(d.p, e.name, v.p) < 0) return nullptr;
    }
    return d.release();
}
PyMethodDef plan_methods[] = {{"versions", Plan_versions, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0) "deepep_amd._host.Plan", sizeof(Plan)};

// The plan of a handle that is as its dispatch left it, or nullptr.  *dict: the handle's attributes (borrowed).
Plan* intact_plan(PyObject* handle, PyObject* owner, PyObject** dict)
{
    if (Py_TYPE(handle) != g_handle_type) return nullptr;
    PyObject** where = _PyObject_GetDictPtr(handle);
    if (where == nullptr || *where == nullptr) return nullptr;
    *dict = *where;
    PyObject* o = PyDict_GetItemWithError(*dict, N._plan);
    if (o == nullptr || Py_TYPE(o) != &PlanType) return nullptr;
    Plan* p = reinterpret_cast<Plan*>(o);
    if (p->owner != owner) return nullptr;
    for (const Pinned& e : *p->pinned) {
        if (PyDict_GetItemWithError(*dict, e.name) != e.object) return nullptr;
        const at::Tensor& t = THPVariable_Unpack(e.object);
        if (t.data_ptr() != e.data || version_of(t) != e.version) return nullptr;
    }
    for (const Pinned& e : *p->same)
        if (PyDict_GetItemWithError(*dict, e.name) != e.object) return nullptr;
    return p;
}

// ---- the exchange of one buffer -------------------------------------------------------------------------------------------
struct Exchange {
    PyObject_HEAD
    void* workspace;
    PyObject* token;  // the buffer's handle token
    PyObject* lock;   // the buffer's lock (a threading.RLock)
    int device, rank, world;
    int hidden, topk, bound;
    bool fp8, combine_only, low_latency_workspace, failed, closed;
    PyObject* comm_object;  // the communication stream as torch's object; its raw stream is asked for by the first asynchronous
    Stream comm, last;      // call only (torch makes a pooled stream when its handle is first read, 0.25 ms)
    bool has_comm, has_last, has_counters;
    double share;     // rows per route of the most recent fresh dispatch (negative: none yet), see capacity_for
    OrderEvent order;
    // asynchronous calls: the communication stream's counter, and the one that the callers' stream raises (one stream at a
    // time: another takes it over when everything it was told to reach has been reached); nullptr: events instead
    Counter *comm_counter, *caller_counter;
    Stream counted;
};
extern PyTypeObject ExchangeType;

struct Locked {  // the buffer's lock, held
    PyObject* lock;
    bool held;
    explicit Locked(PyObject* l) : lock(l)
    {
        PyObject* r = PyObject_CallMethodNoArgs(l, N.acquire);
        held = r != nullptr;
        Py_XDECREF(r);
    }
    ~Locked()
    {
        if (!held) return;
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        PyObject* r = PyObject_CallMethodNoArgs(lock, N.release);
        if (r == nullptr) PyErr_Clear();
        Py_XDECREF(r);
        PyErr_Restore(type, value, trace);
    }
};

bool wait_for_stream(Exchange* e, hipStream_t waits, hipStream_t on)
{
    const hipError_t err = e->order.order(waits, on);
    return err == hipSuccess ? true : raise_hip("ordering two streams", err) != nullptr;
}

// The communication stream waits for the caller's.
bool join_caller(Exchange* e, const Stream& caller)
{
    Counter* c = e->caller_counter;
    if (c != nullptr && (e->counted == caller || c->reached(c->raised)) && !capturing(caller.raw)) {
        e->counted = caller;
        if (int rc = dpep_stream_raise(c->word, ++c->raised, caller.raw); rc != DPEP_OK) return raise_native(rc) != nullptr;
        const hipError_t err = hipStreamWaitValue64(e->comm.raw, c->word, c->raised, hipStreamWaitValueGte, ~0ull);
        return err == hipSuccess ? true : raise_hip("ordering two streams", err) != nullptr;
    }
    return wait_for_stream(e, e->comm.raw, caller.raw);
}

// Where a call's kernels go (deepep_amd.elastic._Enqueue): the caller's stream, or, asynchronous, the communication stream behind
// it; in either case behind the buffer's previous call.
struct Target {
    Stream caller, stream;
    bool asynchronous;
};
bool choose_target(Exchange* e, bool asynchronous, PyObject* previous_event, Target* t)
{
    if (previous_event != Py_None) {
        Ref done(PyObject_CallMethodNoArgs(previous_event, N.current_stream_wait));
        if (!done) return false;
    }
    t->caller = current_stream(e->device);
    t->asynchronous = asynchronous;
    if (asynchronous && !e->has_comm) {
        if (!stream_from(e->comm_object, &e->comm)) return false;
        e->has_comm = true;
    }
    // By the first asynchronous call outside capture, where nothing may be allocated: under capture events do without them.
    // (A buffer that makes no such call takes none; two cost 2 us, the process's first allocation of the kind 39.)
    if (asynchronous && !e->has_counters && !capturing(t->caller.raw)) {
        e->has_counters = true;
        e->comm_counter = take_counter(e->device);
        e->caller_counter = e->comm_counter != nullptr ? take_counter(e->device) : nullptr;
    }
    t->stream = asynchronous ? e->comm : t->caller;
    if (asynchronous && !(e->comm == t->caller) && !join_caller(e, t->caller)) return false;
    if (e->has_last && !(e->last == t->stream) && !(asynchronous && e->last == t->caller) && !wait_for_stream(e, t->stream.raw, e->last.raw))
        return false;
    e->last = t->stream;
    e->has_last = true;
    return true;
}

// What the call returns as its event.  made: tensors this call allocated; others: tensors its kernels use besides.
PyObject* event_of(Exchange* e, const Target& t, std::initializer_list<const at::Tensor*> made, std::initializer_list<const at::Tensor*> others)
{
    Ref overlap(g_overlap_type->tp_new(g_overlap_type, g_empty_tuple, nullptr));
    if (!overlap || !t.asynchronous) return overlap.release();
    Ref event;
    if (e->comm_counter != nullptr && !capturing(e->comm.raw)) {
        Ref marker(reinterpret_cast<PyObject*>(marker_new(e->comm_counter, e->comm, e->device)));
        if (!marker) return nullptr;
        event = Ref(g_event_type->tp_new(g_event_type, g_empty_tuple, nullptr));
        if (!event || PyObject_SetAttr(event.p, N._marker, marker.p) < 0) return nullptr;
    } else {  // (under capture a value would be frozen into the graph) EventHandle(stream): a torch event
        event = Ref(PyObject_CallOneArg(reinterpret_cast<PyObject*>(g_event_type), e->comm_object));
        if (!event) return nullptr;
    }
    Lease* lease = reinterpret_cast<Lease*>(LeaseType.tp_alloc(&LeaseType, 0));
    if (lease == nullptr) return nullptr;
    Ref owned(reinterpret_cast<PyObject*>(lease));
    lease->tensors = new std::vector<at::Tensor>();
    lease->tensors->reserve(made.size() + others.size());
    lease->home = t.caller;
    lease->work = t.stream;
    lease->device = e->device;
    lease->joined = t.caller == t.stream;
    for (const at::Tensor* x : made)
        if (x != nullptr && x->defined()) lease->tensors->push_back(*x);
    lease->made = lease->tensors->size();
    for (const at::Tensor* x : others)
        if (x != nullptr && x->defined()) lease->tensors->push_back(*x);
    if (!lease->joined) lease_declare(lease, t.stream, lease->made, lease->tensors->size());
    if (PyObject_SetAttr(overlap.p, N.event, event.p) < 0 || PyObject_SetAttr(overlap.p, N._lease, owned.p) < 0) return nullptr;
    return overlap.release();
}

// Answers for the tensors of a call from its first launch until the call has an event (event_of), whatever way the call ends.
// On the communication stream a launch may still be pending when a tensor is let go, and memory that was allocated on the
// caller's stream is handed out again in that stream's order alone: so it is declared to the allocator first, where a launch, a
// wait or an allocation fails behind a launch.  The buffer takes no further calls then either.
struct Pending {
    Exchange* e;
    const Target& t;
    const at::Tensor* used[8];
    int count = 0;
    bool launched = false;
    Pending(Exchange* exchange, const Target& target, std::initializer_list<const at::Tensor*> tensors) : e(exchange), t(target)
    {
        for (const at::Tensor* x : tensors)
            if (x != nullptr) used[count++] = x;
    }
    void declare(const at::Tensor& x) const
    {
        if (x.defined() && crosses()) x.record_stream(t.stream.torch(e->device));
    }
    bool crosses() const { return t.asynchronous && !(t.stream == t.caller); }
    // For an output that the queued launch leaves alone (DPEP_REPORT_ALL_OR_NONE): nothing to declare, its memory can be had again.
    // The new one is allocated on the stream that writes it: the host has waited since without the GIL, and what another thread
    // has queued on the caller's stream meanwhile may still work on memory that is free in that stream's order.  (The
    // communication stream waiting for the caller's once more instead: 5 us more where shares jump from batch to batch.)
    void replace(at::Tensor* x, at::IntArrayRef sizes, at::ScalarType type) const
    {
        *x = at::Tensor();
        if (!crosses()) {
            *x = allocate(sizes, type, e->device);
            return;
        }
        const c10::StreamGuard on_its_stream(t.stream.torch(e->device));
        *x = allocate(sizes, type, e->device);
        x->record_stream(t.caller.torch(e->device));
    }
    ~Pending()
    {
        if (!launched) return;
        e->failed = true;
        for (int i = 0; i < count; ++i) {
            try {
                declare(*used[i]);
            } catch (...) {  // (nothing can be reported from here)
            }
        }
    }
};

// A dispatch's payload, checked as far as it can be without knowing which path it takes.
struct Payload {
    const at::Tensor* x = nullptr;
    const at::Tensor* scales = nullptr;
    bool tuple = false;
    long long tokens = 0, width = 0;
};
bool read_payload(PyObject* o, int device, Payload* p)
{
    PyObject* x = o;
    if (PyTuple_CheckExact(o)) {
        if (PyTuple_GET_SIZE(o) != 2) return false;
        p->tuple = true;
        x = PyTuple_GET_ITEM(o, 0);
        if ((p->scales = plain(PyTuple_GET_ITEM(o, 1), device)) == nullptr) return false;
    }
    p->x = plain(x, device);
    if (p->x == nullptr || p->x->dim() != 2) return false;
    p->tokens = p->x->size(0);
    p->width = p->x->size(1);
    return p->tokens > 0 && p->width > 0 && aligned16(*p->x);
}

inline bool set(PyObject* dict, PyObject* name, PyObject* value) { return PyDict_SetItem(dict, name, value) == 0; }
inline bool set_int(PyObject* dict, PyObject* name, long long v)
{
    Ref o(PyLong_FromLongLong(v));
    return o && set(dict, name, o.p);
}
// Puts a tensor into the handle and pins it.
bool set_pinned(Plan* plan, PyObject* dict, PyObject* name, const at::Tensor& t)
{
    PyObject* o = wrap(t);
    if (o == nullptr) return false;
    plan->pinned->push_back(Pinned{name, o, t.data_ptr(), version_of(t)});
    return set(dict, name, o);
}
// Keeps the handle's present values of `names`: a handle in which one of them was replaced leaves the native path.
bool keep_same(Plan* plan, PyObject* dict, std::initializer_list<PyObject*> names)
{
    for (PyObject* name : names) {
        PyObject* o = PyDict_GetItemWithError(dict, name);
        if (o == nullptr) return false;
        plan->same->push_back(Pinned{name, new_ref(o), nullptr, 0});
    }
    return true;
}

// Rows to allocate for a fresh dispatch's payload before R is known.  Where at least half of the experts are local, or the batch is
// small (one launch, at most 2048 rows), all T*K routes: the surplus is small.  Otherwise an eighth and 256 rows more than the previous batch's share of the routes suggests
// (the first batch: than the expert range does), so that the payload can be queued behind the layout as well, instead of
// after the host has read R, which left the GPU idle for the length of a host round trip.  (Random routes spread around an
// even share of 16 384 rows by 128.)  A batch that jumps out of these bounds, up or down (DPEP_ROWS_KEPT: a received tensor keeps its
// whole storage for as long as it lives), is moved once the host knows R, into outputs of that size: the payload that is
// queued already finds the count on the device and ends without moving anything.  (Cold and hot batches in turn, us a dispatch,
// against moving what fits and then everything: 16 384 tokens of 7168 columns, EP8, 173 -> 136; 4096 of 4096, EP4, 41 -> 37.)
long long capacity_for(const Exchange* e, long long routes, long long local, long long experts)
{
    const double share = e->share >= 0.0 ? e->share : static_cast<double>(local) / static_cast<double>(experts);
    const long long rows = static_cast<long long>(share * static_cast<double>(routes) + 0.5);
    return std::min(DPEP_CAPACITY(rows), routes);
}

struct FreshCall {
    Payload in;
    const at::Tensor* idx;
    const at::Tensor* weights;  // nullptr without
    long long topk, experts, capacity_tokens, capacity_rows;
    bool copy_idx, quantize, low_latency;
};

PyObject* run_fresh(Exchange* e, const FreshCall& c, const Target& t, PyObject* idx_object)
{
    const int device = e->device;
    const long long tokens = c.in.tokens, width = c.in.width, topk = c.topk, routes = tokens * topk;
    const long long local = c.experts / e->world, begin = e->rank * local;
    const bool fp8_out = c.quantize || c.in.x->scalar_type() == at::kFloat8_e4m3fn;
    const at::ScalarType out_type = c.quantize ? at::kFloat8_e4m3fn : c.in.x->scalar_type();
    const long long scale_cols = c.quantize ? width / 128 : c.in.scales != nullptr ? c.in.scales->size(1) : 0;
    const bool all_routes = 2 * local >= c.experts || routes <= 2048;
    const long long capacity = c.low_latency ? c.capacity_rows : all_routes ? routes : capacity_for(e, routes, local, c.experts);

    // One block for all of the routing: [ids 8 B][route_to_row][row_to_route][counts][psum][offsets][num_rows][send_counts], with
    // the row weights behind it where both are small, and one for the payload, which holds the scales too where both are
    // small (an allocation takes 1 us).  Maps and weights start at multiples of 256 bytes, as tensors of their own would; a
    // caller that keeps the received weights for longer than the handle keeps no more than kSmallBlock with them.
    auto aligned = [](int64_t bytes) { return (bytes + 255) / 256 * 256; };
    const int64_t at_forward = c.copy_idx ? aligned(routes * 8) : 0, at_rows = at_forward + aligned(routes * 4);
    const int64_t at_counts = at_rows + aligned(routes * 4);
    const int64_t at_psum = at_counts + local * 4, at_offsets = at_psum + local * 4, at_num = at_offsets + (local + 1) * 4;
    const int64_t at_send = at_num + 4, at_weights = aligned(at_send + (c.low_latency ? c.experts * 4 : 0));
    const bool weights_inside = c.weights != nullptr && at_weights + capacity * 4 <= kSmallBlock;
    at::Tensor routing = allocate({at_weights + (weights_inside ? capacity * 4 : 0)}, at::kByte, device), out, scales, weights;
    const at::ScalarType scale_type = c.quantize || c.in.scales == nullptr ? at::kFloat : c.in.scales->scalar_type();
    const int64_t code_bytes = capacity * width, scale_bytes = capacity * scale_cols * 4;
    if (scale_cols > 0 && code_bytes <= (1 << 20)) {  // (codes of one byte; width is a multiple of 16)
        at::Tensor both = allocate({code_bytes + scale_bytes}, at::kByte, device);
        out = over(both.storage(), 0, out_type, {capacity, width});
        scales = over(both.storage(), code_bytes, scale_type, {capacity, scale_cols});
    } else {
        out = allocate({capacity, width}, out_type, device);
        if (scale_cols > 0) scales = allocate({capacity, scale_cols}, scale_type, device);
    }
    if (c.weights != nullptr)
        weights = weights_inside ? over(routing.storage(), at_weights, at::kFloat, {capacity}) : allocate({capacity}, at::kFloat, device);
    char* base = static_cast<char*>(routing.data_ptr());

    dpep_fresh_dispatch call = {};
    call.topk_idx = static_cast<const int64_t*>(c.idx->data_ptr());
    call.topk_idx_copy = c.copy_idx ? reinterpret_cast<int64_t*>(base) : nullptr;
    call.x = c.in.x->data_ptr();
    call.scales = c.in.scales != nullptr ? static_cast<const float*>(c.in.scales->data_ptr()) : nullptr;
    call.topk_weights = c.weights != nullptr ? static_cast<const float*>(c.weights->data_ptr()) : nullptr;
    call.route_to_row = reinterpret_cast<int32_t*>(base + at_forward);
    call.row_to_route = reinterpret_cast<int32_t*>(base + at_rows);
    call.counts = reinterpret_cast<int32_t*>(base + at_counts);
    call.psum = reinterpret_cast<int32_t*>(base + at_psum);
    call.offsets = reinterpret_cast<int32_t*>(base + at_offsets);
    call.num_rows = reinterpret_cast<int32_t*>(base + at_num);
    call.send_counts = c.low_latency ? reinterpret_cast<int32_t*>(base + at_send) : nullptr;
    call.out = out.data_ptr();
    call.out_scales = scales.defined() ? static_cast<float*>(scales.data_ptr()) : nullptr;
    call.out_weights = weights.defined() ? static_cast<float*>(weights.data_ptr()) : nullptr;
    call.num_tokens = static_cast<int32_t>(tokens);
    call.num_topk = static_cast<int32_t>(topk);
    call.num_experts = static_cast<int32_t>(c.experts);
    call.expert_begin = static_cast<int32_t>(begin);
    call.num_local = static_cast<int32_t>(local);
    call.row_bytes = static_cast<int32_t>(width * c.in.x->element_size());
    call.scale_cols = static_cast<int32_t>(c.quantize ? 0 : scale_cols);
    call.quantize = c.quantize;
    call.capacity_rows = static_cast<int32_t>(capacity);
    call.report_to_host = c.low_latency ? 0 : all_routes ? 1 : DPEP_REPORT_ALL_OR_NONE;
    Pending pending(e, t, {&out, &scales, &weights, &routing, c.in.x, c.in.scales, c.weights, c.idx});
    pending.launched = true;
    if (const int status = dpep_dispatch_fresh(e->workspace, &call, t.stream.raw)) return raise_native(status);

    // ---- while the GPU works: everything that does not depend on R -----------------------------------------------------
    const c10::Storage& storage = routing.storage();
    Ref dict(PyDict_Copy(g_handle_template));
    Ref plan_ref(reinterpret_cast<PyObject*>(plan_new()));
    if (!dict || !plan_ref) return nullptr;
    Plan* plan = reinterpret_cast<Plan*>(plan_ref.p);
    PyObject* d = dict.p;
    plan->routing = new at::Tensor(routing);
    plan->route_to_row = call.route_to_row;
    plan->row_to_route = call.row_to_route;
    plan->owner = new_ref(e->token);
    plan->tokens = call.num_tokens;
    plan->topk = call.num_topk;
    plan->hidden = static_cast<int>(width);
    plan->experts = call.num_experts;
    plan->low_latency = c.low_latency;
    bool ok = set_int(d, N.num_experts, c.experts) && set_int(d, N.num_max_tokens_per_rank, c.capacity_tokens) &&
              set_int(d, N.rank, e->rank) && set_int(d, N.world_size, e->world) && set_int(d, N.num_tokens, tokens) &&
              set_int(d, N.num_topk, topk) && set_int(d, N.hidden, width) && set(d, N.metadata_only, Py_False) &&
              set(d, N._buffer_token, e->token) && set(d, N._plan, plan_ref.p);
    at::Tensor idx = c.copy_idx ? over(storage, 0, at::kLong, {tokens, topk}) : *c.idx;
    at::Tensor forward = over(storage, at_forward, at::kInt, {tokens, topk});
    if (c.copy_idx) {
        ok = ok && set_pinned(plan, d, N.topk_idx, idx);
    } else {
        plan->pinned->push_back(Pinned{N.topk_idx, new_ref(idx_object), idx.data_ptr(), version_of(idx)});
        ok = ok && set(d, N.topk_idx, idx_object);
    }
    ok = ok && set_pinned(plan, d, N.route_to_row, forward);
    at::Tensor send;
    if (c.low_latency) {
        send = over(storage, at_send, at::kInt, {c.experts});
        Ref send_object(wrap(send)), weights_object(wrap(weights)), list(PyList_New(0));
        plan->weights = new at::Tensor(weights);
        plan->rows = capacity;
        ok = ok && send_object && weights_object && list && set(d, N.send_counts, send_object.p) && set(d, N.source_weights, weights_object.p) &&
             set(d, N.num_recv_tokens_per_expert_list, list.p) && set(d, N.is_low_latency, Py_True) && set_int(d, N.num_compute_units, 0) &&
             set_int(d, N.num_recv_tokens, e->world * c.capacity_tokens) && set_int(d, N.num_expanded_tokens, capacity);
    } else {
        at::Tensor counts = over(storage, at_counts, at::kInt, {local}), psum = over(storage, at_psum, at::kInt, {local});
        ok = ok && set_pinned(plan, d, N.expert_totals, counts) && set_pinned(plan, d, N.psum_num_recv_tokens_per_expert, psum) &&
             set(d, N.num_unaligned_recv_tokens_per_expert, PyDict_GetItemWithError(d, N.expert_totals));
        Ref offsets(wrap(over(storage, at_offsets, at::kInt, {local + 1}))), full(wrap(over(storage, at_rows, at::kInt, {routes})));
        ok = ok && offsets && full && set(d, N.expert_offsets, offsets.p) && set(d, N._row_to_route_full, full.p) &&
             set_int(d, N.num_compute_units, fp8_out ? 64 : 32);
    }
    Ref handle(g_handle_type->tp_new(g_handle_type, g_empty_tuple, nullptr));
    if (!ok || !handle) return nullptr;

    long long rows = capacity;
    bool replaced = false;  // the outputs belong to the communication stream
    if (!c.low_latency) {
        // ---- the one host synchronisation -------------------------------------------------------------------------------
        int32_t counts[DPEP_MAX_LOCAL_EXPERTS], reported = 0;
        int status;
        if (dpep_layout_ready(e->workspace)) {
            status = dpep_layout_wait(e->workspace, counts, static_cast<int>(local), &reported, kWaitTimeoutUs);
        } else {
            Py_BEGIN_ALLOW_THREADS;
            status = dpep_layout_wait(e->workspace, counts, static_cast<int>(local), &reported, kWaitTimeoutUs);
            Py_END_ALLOW_THREADS;
        }
        if (status) return raise_native(status);
        rows = reported;
        plan->rows = rows;
        e->share = static_cast<double>(rows) / static_cast<double>(routes);
        if (!all_routes && !DPEP_ROWS_KEPT(rows, capacity)) {  // far from what the share suggested
            pending.replace(&out, {rows, width}, out_type);
            if (scales.defined()) pending.replace(&scales, {rows, scale_cols}, scale_type);
            if (weights.defined()) pending.replace(&weights, {rows}, at::kFloat);
            replaced = pending.crosses();
            float* s_out = scales.defined() ? static_cast<float*>(scales.data_ptr()) : nullptr;
            float* w_out = weights.defined() ? static_cast<float*>(weights.data_ptr()) : nullptr;
            status = c.quantize ? dpep_dispatch_quant_fp8(call.x, call.topk_weights, call.route_to_row, call.row_to_route, call.num_tokens,
                                                          call.num_topk, reported, static_cast<int>(width), out.data_ptr(), s_out, w_out, t.stream.raw)
                                : dpep_dispatch_copy(call.x, call.scales, call.topk_weights, call.route_to_row, call.row_to_route, call.num_tokens,
                                                     call.num_topk, reported, call.row_bytes, call.scale_cols, out.data_ptr(), s_out, w_out, t.stream.raw);
            if (status) return raise_native(status);
        } else if (rows < capacity) {
            out = over(out.storage(), 0, out_type, {rows, width});
            if (scales.defined()) scales = over(scales.storage(), scales.storage_offset() * 4, scale_type, {rows, scale_cols});
            if (weights.defined()) weights = over(weights.storage(), weights.storage_offset() * 4, at::kFloat, {rows});
        }
        Ref list(PyList_New(local));
        if (!list) return nullptr;
        for (long long i = 0; i < local; ++i) {
            PyObject* n = PyLong_FromLong(counts[i]);
            if (n == nullptr) return nullptr;
            PyList_SET_ITEM(list.p, i, n);
        }
        if (!set(d, N.num_recv_tokens_per_expert_list, list.p) || !set_int(d, N.num_expanded_tokens, rows) ||
            !set_pinned(plan, d, N.weight_return_meta, over(storage, at_rows, at::kInt, {rows})))
            return nullptr;
    }
    if (!keep_same(plan, d, {N.num_experts, N.num_expanded_tokens, N.is_low_latency, N.source_weights, N.send_counts, N.rank, N.world_size,
                             N.num_tokens, N.num_topk, N.hidden, N.metadata_only, N.metadata_version, N._buffer_token, N.do_expand,
                             N.expert_alignment}))
        return nullptr;
    if (!c.low_latency && !keep_same(plan, d, {N._row_to_route_full})) return nullptr;
    if (PyObject_SetAttr(handle.p, N.__dict__, d) < 0) return nullptr;

    Ref event(replaced ? event_of(e, t, {&routing}, {&out, &scales, &weights, c.in.x, c.in.scales, c.weights, c.idx})
                       : event_of(e, t, {&out, &scales, &weights, &routing}, {c.in.x, c.in.scales, c.weights, c.idx}));
    pending.launched = !event;
    Ref payload(wrap(out));
    if (!event || !payload) return nullptr;
    if (scales.defined()) {
        Ref second(wrap(scales));
        if (!second) return nullptr;
        payload = Ref(PyTuple_Pack(2, payload.p, second.p));
        if (!payload) return nullptr;
    }
    Ref received(weights.defined() && !c.low_latency ? wrap(weights) : new_ref(Py_None));
    return received ? PyTuple_Pack(5, payload.p, Py_None, received.p, handle.p, event.p) : nullptr;
}

PyObject* run_cached(Exchange* e, const Payload& in, bool quantize, const at::Tensor* weights_in, Plan* plan, PyObject* handle,
                     PyObject* dict, const Target& t)
{
    const int device = e->device;
    const long long rows = plan->rows, width = in.width;
    const bool fp8 = quantize || in.tuple;
    const long long scale_cols = quantize ? width / 128 : in.scales != nullptr ? in.scales->size(1) : 0;
    at::Tensor out = allocate({rows, width}, fp8 ? at::kFloat8_e4m3fn : in.x->scalar_type(), device), scales, weights;
    if (scale_cols > 0) scales = allocate({rows, scale_cols}, at::kFloat, device);
    if (weights_in != nullptr) weights = allocate({rows}, at::kFloat, device);
    const float* w_in = weights_in != nullptr ? static_cast<const float*>(weights_in->data_ptr()) : nullptr;
    float* s_out = scales.defined() ? static_cast<float*>(scales.data_ptr()) : nullptr;
    float* w_out = weights.defined() ? static_cast<float*>(weights.data_ptr()) : nullptr;
    Pending pending(e, t, {&out, &scales, &weights, in.x, in.scales, weights_in, plan->routing});
    pending.launched = true;
    const int status = quantize ? dpep_dispatch_quant_fp8(in.x->data_ptr(), w_in, plan->route_to_row, plan->row_to_route, plan->tokens,
                                                          plan->topk, static_cast<int>(rows), static_cast<int>(width), out.data_ptr(), s_out,
                                                          w_out, t.stream.raw)
                                : dpep_dispatch_copy(in.x->data_ptr(), in.scales != nullptr ? static_cast<const float*>(in.scales->data_ptr()) : nullptr,
                                                     w_in, plan->route_to_row, plan->row_to_route, plan->tokens, plan->topk,
                                                     static_cast<int>(rows), static_cast<int>(width * in.x->element_size()),
                                                     static_cast<int>(scale_cols), out.data_ptr(), s_out, w_out, t.stream.raw);
    if (status) return raise_native(status);
    if (!set_int(dict, N.num_compute_units, fp8 ? 64 : 32)) return nullptr;
    Ref event(event_of(e, t, {&out, &scales, &weights}, {in.x, in.scales, weights_in, plan->routing}));
    pending.launched = !event;
    Ref payload(wrap(out));
    if (!event || !payload) return nullptr;
    if (scales.defined()) {
        Ref second(wrap(scales));
        if (!second) return nullptr;
        payload = Ref(PyTuple_Pack(2, payload.p, second.p));
        if (!payload) return nullptr;
    }
    Ref received(weights.defined() ? wrap(weights) : new_ref(Py_None));
    return received ? PyTuple_Pack(5, payload.p, Py_None, received.p, handle, event.p) : nullptr;
}

inline bool usable(const Exchange* e)
{
    return !e->failed && !e->closed && c10::hip::current_device() == e->device && !c10::InferenceMode::is_enabled();
}
inline bool valid_previous(const Exchange* e, PyObject* event)
{
    if (event == Py_None) return true;
    if (!PyObject_TypeCheck(event, g_event_type)) return false;
    Ref gpu(PyObject_GetAttr(event, N._gpu_index));
    if (!gpu) {
        PyErr_Clear();
        return false;
    }
    return exact_int(gpu.p, 0, 1 << 16) == e->device;
}

// ElasticBuffer.dispatch's arguments in the order of its signature.
PyObject* Exchange_dispatch(PyObject* self, PyObject* const* a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    Exchange* e = reinterpret_cast<Exchange*>(self);
    if (n != 19) {
        PyErr_SetString(PyExc_TypeError, "dispatch takes the 19 arguments of ElasticBuffer.dispatch");
        return nullptr;
    }
    PyObject *x = a[0], *topk_idx = a[1], *topk_weights = a[2], *stats = a[3], *num_experts = a[4], *max_tokens = a[5], *alignment = a[6],
             *num_sms = a[7], *num_qps = a[8], *previous = a[9], *before_epilogue = a[10], *asynchronous = a[11], *alloc_on_comm = a[12],
             *handle = a[13], *handle_copy = a[14], *cpu_sync = a[15], *expand = a[16], *zero_padding = a[17], *col_major = a[18];
    // options
    if (!usable(e) || e->combine_only || stats != Py_None || before_epilogue != Py_None || !is_bool(asynchronous) || alloc_on_comm != Py_False ||
        !is_bool(handle_copy) || zero_padding != Py_False || col_major != Py_False || (expand != Py_None && expand != Py_True) ||
        (cpu_sync != Py_None && !is_bool(cpu_sync)) || (alignment != Py_None && exact_int(alignment, 1, 1) != 1) || !valid_previous(e, previous))
        Py_RETURN_NONE;
    const long long sms = exact_int(num_sms, 0, 64), qps = exact_int(num_qps, 0, 2);
    if (sms < 0 || (qps != 0 && qps != 2)) Py_RETURN_NONE;
    Payload in;
    if (!read_payload(x, e->device, &in)) Py_RETURN_NONE;
    const at::ScalarType type = in.x->scalar_type();
    const at::Tensor* weights = nullptr;
    if (topk_weights != Py_None) {
        weights = plain(topk_weights, e->device);
        if (weights == nullptr || weights->scalar_type() != at::kFloat || weights->dim() != 2) Py_RETURN_NONE;
    }
    const long long per_rank = (in.tokens + e->world - 1) / e->world;
    long long capacity = e->bound != 0 ? e->bound : per_rank;
    if (max_tokens != Py_None && (capacity = exact_int(max_tokens, 0, g_max_tokens)) < 0) Py_RETURN_NONE;
    if (capacity < per_rank || capacity > g_max_tokens || (e->bound != 0 && capacity > e->bound)) Py_RETURN_NONE;
    if (e->hidden != 0 && in.width != e->hidden) Py_RETURN_NONE;

    Plan* plan = nullptr;
    PyObject* dict = nullptr;
    FreshCall c = {};
    c.in = in;
    c.weights = weights;
    c.capacity_tokens = capacity;
    if (handle == Py_None) {
        c.idx = plain(topk_idx, e->device);
        if (c.idx == nullptr || c.idx->scalar_type() != at::kLong || c.idx->dim() != 2 || c.idx->size(0) != in.tokens) Py_RETURN_NONE;
        c.copy_idx = handle_copy == Py_True;
        if (!c.copy_idx && c.idx->is_inference()) Py_RETURN_NONE;
        c.topk = c.idx->size(1);
        c.experts = exact_int(num_experts, e->world, g_max_experts);
        if (c.experts < 0 || c.experts % e->world != 0) Py_RETURN_NONE;
    } else {
        if (topk_idx != Py_None || (plan = intact_plan(handle, e->token, &dict)) == nullptr || plan->low_latency) Py_RETURN_NONE;
        if (num_experts != Py_None && exact_int(num_experts, plan->experts, plan->experts) != plan->experts) Py_RETURN_NONE;
        if (in.tokens != plan->tokens || in.width != plan->hidden) Py_RETURN_NONE;
        c.topk = plan->topk;
        c.experts = plan->experts;
    }
    if (c.topk < 1 || (e->topk != 0 && e->topk != c.topk) || (weights != nullptr && !has_shape(*weights, in.tokens, c.topk))) Py_RETURN_NONE;

    // Path selection as in ElasticBuffer._choose_low_latency: small batches of EP16-EP256 jobs with weights and default options.
    if (handle == Py_None && e->world >= 16 && e->world <= 256 && capacity <= g_low_latency_max_tokens && weights != nullptr && sms == 0 && qps == 0 &&
        previous == Py_None && asynchronous == Py_False && (type == at::kBFloat16 || type == at::kHalf || type == at::kFloat8_e4m3fn) &&
        !(e->fp8 && type != at::kFloat8_e4m3fn) && in.width * in.x->element_size() % 16 == 0 && c.topk <= DPEP_MAX_TOPK &&
        (type == at::kFloat8_e4m3fn
             ? in.scales != nullptr && (in.scales->scalar_type() == at::kFloat || in.scales->scalar_type() == at::kInt) &&
                   has_shape(*in.scales, in.tokens, (in.width + 127) / 128)
             : in.scales == nullptr)) {
        if (!e->low_latency_workspace) Py_RETURN_NONE;
        c.low_latency = true;
        c.capacity_rows = e->world * capacity * std::min<long long>(c.topk, c.experts / e->world);
        if (c.capacity_rows > 0x7fffffffLL) Py_RETURN_NONE;
    } else {
        if (in.tuple ? type != at::kFloat8_e4m3fn || in.scales->scalar_type() != at::kFloat || !has_shape(*in.scales, in.tokens, in.width / 128)
                     : type != at::kBFloat16)
            Py_RETURN_NONE;
        c.quantize = e->fp8 && !in.tuple;
        const bool fp8 = c.quantize || in.tuple;
        if (in.width > g_max_hidden || in.width % (fp8 ? 128 : 16) != 0 || (sms != 0 && sms != (fp8 ? 64 : 32)) || c.topk > g_max_topk ||
            in.tokens > static_cast<long long>(g_max_tokens) * e->world || (handle == Py_None && cpu_sync == Py_False))
            Py_RETURN_NONE;
    }
    Locked held(e->lock);
    if (!held.held) return nullptr;
    if (e->failed) Py_RETURN_NONE;
    Target target;
    PyObject* result = choose_target(e, asynchronous == Py_True, previous, &target)
                           ? plan != nullptr ? run_cached(e, in, c.quantize, weights, plan, handle, dict, target) : run_fresh(e, c, target, topk_idx)
                           : nullptr;
    if (result == nullptr) e->failed = true;
    return result;
    END_HANDLE_TH_ERRORS
}

// ElasticBuffer.combine's arguments in the order of its signature.
PyObject* Exchange_combine(PyObject* self, PyObject* const* a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    Exchange* e = reinterpret_cast<Exchange*>(self);
    if (n != 10) {
        PyErr_SetString(PyExc_TypeError, "combine takes the 10 arguments of ElasticBuffer.combine");
        return nullptr;
    }
    PyObject *x = a[0], *handle = a[1], *topk_weights = a[2], *bias = a[3], *num_sms = a[4], *num_qps = a[5], *previous = a[6],
             *before_epilogue = a[7], *asynchronous = a[8], *alloc_on_comm = a[9];
    if (!usable(e) || bias != Py_None || before_epilogue != Py_None || !is_bool(asynchronous) || alloc_on_comm != Py_False || !valid_previous(e, previous))
        Py_RETURN_NONE;
    const long long sms = exact_int(num_sms, 0, 64), qps = exact_int(num_qps, 0, 2);
    if ((sms != 0 && sms != 64) || (qps != 0 && qps != 2)) Py_RETURN_NONE;
    PyObject* dict = nullptr;
    Plan* plan = intact_plan(handle, e->token, &dict);
    if (plan == nullptr) Py_RETURN_NONE;
    const at::Tensor* rows = plain(x, e->device);
    if (rows == nullptr || !has_shape(*rows, plan->rows, plan->hidden) || (plan->rows > 0 && !aligned16(*rows))) Py_RETURN_NONE;
    const at::ScalarType type = rows->scalar_type();
    if (type != at::kBFloat16 && !(plan->low_latency && type == at::kHalf)) Py_RETURN_NONE;
    const at::Tensor* values = nullptr;
    if (plan->low_latency) {
        if (topk_weights != Py_None || sms != 0 || qps != 0 || previous != Py_None || asynchronous != Py_False) Py_RETURN_NONE;
    } else if (topk_weights != Py_None) {
        values = plain(topk_weights, e->device);
        if (values == nullptr || values->scalar_type() != at::kFloat || values->dim() != 1 || values->size(0) != plan->rows) Py_RETURN_NONE;
    }
    Locked held(e->lock);
    if (!held.held) return nullptr;
    if (e->failed) Py_RETURN_NONE;
    auto run = [&]() -> PyObject* {
        Target t;
        if (!choose_target(e, asynchronous == Py_True, previous, &t)) return nullptr;
        at::Tensor out = allocate({plan->tokens, plan->hidden}, type, e->device), returned;
        if (values != nullptr) returned = allocate({plan->tokens, plan->topk}, at::kFloat, e->device);
        const float* row_weights = plan->low_latency ? static_cast<const float*>(plan->weights->data_ptr()) : nullptr;
        const int expected = plan->low_latency ? static_cast<int>(static_cast<long long>(plan->tokens) * plan->topk / e->world) : static_cast<int>(plan->rows);
        Pending pending(e, t, {&out, &returned, rows, values, plan->routing, plan->weights});
        pending.launched = true;
        if (const int status = dpep_combine_expecting(rows->data_ptr(), type == at::kHalf, row_weights, plan->route_to_row, plan->tokens, plan->topk,
                                                      static_cast<int>(plan->rows), expected, plan->hidden, out.data_ptr(),
                                                      values != nullptr ? static_cast<const float*>(values->data_ptr()) : nullptr,
                                                      returned.defined() ? static_cast<float*>(returned.data_ptr()) : nullptr, t.stream.raw))
            return raise_native(status);
        Ref event(event_of(e, t, {&out, &returned}, {rows, values, plan->routing, plan->weights}));
        pending.launched = !event;
        Ref first(wrap(out)), second(returned.defined() ? wrap(returned) : new_ref(Py_None));
        return event && first && second ? PyTuple_Pack(3, first.p, second.p, event.p) : nullptr;
    };
    PyObject* result = run();
    if (result == nullptr) e->failed = true;
    return result;
    END_HANDLE_TH_ERRORS
}

PyObject* Exchange_new(PyTypeObject* type, PyObject* args, PyObject*)
{
    HANDLE_TH_ERRORS
    PyObject *workspace, *token, *lock, *comm;
    int device, rank, world, hidden, topk, bound, fp8, combine_only, low_latency;
    if (!PyArg_ParseTuple(args, "OOOOiiiiiippp", &workspace, &token, &lock, &comm, &device, &rank, &world, &hidden, &topk, &bound, &fp8,
                          &combine_only, &low_latency))
        return nullptr;
    void* ws = PyLong_AsVoidPtr(workspace);
    if (ws == nullptr && PyErr_Occurred()) return nullptr;
    Exchange* e = reinterpret_cast<Exchange*>(type->tp_alloc(type, 0));
    if (e == nullptr) return nullptr;
    e->workspace = ws;
    e->token = new_ref(token);
    e->lock = new_ref(lock);
    e->device = device;
    e->rank = rank;
    e->world = world;
    e->hidden = hidden;
    e->topk = topk;
    e->bound = bound;
    e->fp8 = fp8;
    e->combine_only = combine_only;
    e->low_latency_workspace = low_latency;
    e->failed = e->closed = e->has_comm = e->has_last = e->has_counters = false;
    e->comm_object = new_ref(comm);
    e->share = -1.0;
    return reinterpret_cast<PyObject*>(e);
    END_HANDLE_TH_ERRORS
}
void Exchange_dealloc(PyObject* o)
{
    Exchange* e = reinterpret_cast<Exchange*>(o);
    e->order.release();
    for (Counter* c : {e->comm_counter, e->caller_counter})
        if (c != nullptr && c->reached(c->raised)) g_idle_counters.push_back(c);  // (one still pending is not used again)
    Py_XDECREF(e->token);
    Py_XDECREF(e->lock);
    Py_XDECREF(e->comm_object);
    Py_TYPE(o)->tp_free(o);
}
PyObject* Exchange_get_failed(PyObject* o, void*) { return PyBool_FromLong(reinterpret_cast<Exchange*>(o)->failed); }
int Exchange_set_failed(PyObject* o, PyObject* v, void*)
{
    const int truth = v == nullptr ? 0 : PyObject_IsTrue(v);
    if (truth < 0) return -1;
    reinterpret_cast<Exchange*>(o)->failed = truth != 0;
    return 0;
}
PyObject* Exchange_get_last(PyObject* o, void*)
{
    Exchange* e = reinterpret_cast<Exchange*>(o);
    if (!e->has_last) Py_RETURN_NONE;
    return stream_object(e->last, e->device);
}
int Exchange_set_last(PyObject* o, PyObject* v, void*)
{
    Exchange* e = reinterpret_cast<Exchange*>(o);
    e->has_last = v != nullptr && v != Py_None;
    return !e->has_last || stream_from(v, &e->last) ? 0 : -1;
}
PyObject* Exchange_close(PyObject* o, PyObject*)
{
    reinterpret_cast<Exchange*>(o)->closed = true;
    Py_RETURN_NONE;
}
PyMethodDef exchange_methods[] = {
    {"dispatch", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(Exchange_dispatch)), METH_FASTCALL, nullptr},
    {"combine", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(Exchange_combine)), METH_FASTCALL, nullptr},
    {"close", Exchange_close, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyGetSetDef exchange_getset[] = {{"failed", Exchange_get_failed, Exchange_set_failed, nullptr, nullptr},
                                 {"last_stream", Exchange_get_last, Exchange_set_last, nullptr, nullptr},
                                 {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject ExchangeType = {PyVarObject_HEAD_INIT(nullptr, 0) "deepep_amd._host.Exchange", sizeof(Exchange)};

// ---- the MegaMoE layer ------------------------------------------------------------------------------------------------------
// One SymmBuffer's forward (deepep_amd.megamoe.api._run), and the FP8 casts.
struct Mega {
    PyObject_HEAD
    PyObject* lock;      // the buffer's lock (a threading.Lock)
    PyObject *logical1, *logical2, *shared1, *shared2;  // (experts, N, K) that l1 / l2 / shared l1 / shared l2 must have
    void* workspace;     // of batches of `batch` rows; nullptr before the first
    int batch;
    int device, experts, first_expert, local, topk, hidden, inter, shared, capacity, padded;
    Stream last;
    bool has_last, closed;
    OrderEvent order;
};
extern PyTypeObject MegaType;
PyTypeObject* g_pair_type;  // deepep_amd.megamoe.api._PreparedPair

// The tensors of an unmodified prepared pair of the right kind and size.
bool read_pair(PyObject* pair, bool gate_up, PyObject* logical, int device, const at::Tensor** w, const at::Tensor** s)
{
    if (Py_TYPE(pair) != g_pair_type || PyTuple_GET_SIZE(pair) != 2) return false;
    *w = plain(PyTuple_GET_ITEM(pair, 0), device);
    *s = plain(PyTuple_GET_ITEM(pair, 1), device);
    if (*w == nullptr || *s == nullptr || (*w)->scalar_type() != at::kByte || (*s)->scalar_type() != at::kByte || !aligned16(**w) || !aligned16(**s) ||
        (*w)->is_inference() || (*s)->is_inference())
        return false;
    Ref kind(PyObject_GetAttr(pair, N.gate_up)), sizes(PyObject_GetAttr(pair, N.logical)), versions(PyObject_GetAttr(pair, N._versions));
    if (!kind || !sizes || !versions || PyObject_RichCompareBool(sizes.p, logical, Py_EQ) != 1 || !PyTuple_CheckExact(versions.p) ||
        PyTuple_GET_SIZE(versions.p) != 2) {
        PyErr_Clear();
        return false;
    }
    return kind.p == (gate_up ? Py_True : Py_False) && exact_int(PyTuple_GET_ITEM(versions.p, 0), 0, 0xffffffffLL) == version_of(**w) &&
           exact_int(PyTuple_GET_ITEM(versions.p, 1), 0, 0xffffffffLL) == version_of(**s);
}

inline bool overlap(const at::Tensor& a, const at::Tensor& b)
{
    const char *x = static_cast<const char*>(a.data_ptr()), *y = static_cast<const char*>(b.data_ptr());
    return x < y + b.nbytes() && y < x + a.nbytes();
}

// forward(x, scales, topk_idx, topk_weights, l1, l2, shared_l1, shared_l2, out, staged) -> (y, counts), or None (see above).
// scales None: x is BF16.  out None: allocated here.  staged: x / scales / topk_idx / topk_weights are the buffer's own input
// tensors, of which the first rows (as many as out has) are meant.
PyObject* Mega_forward(PyObject* self, PyObject* const* a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    Mega* m = reinterpret_cast<Mega*>(self);
    if (n != 10) {
        PyErr_SetString(PyExc_TypeError, "forward takes 10 arguments");
        return nullptr;
    }
    const bool staged = a[9] == Py_True;
    if (m->closed || m->workspace == nullptr || c10::hip::current_device() != m->device || c10::InferenceMode::is_enabled()) Py_RETURN_NONE;
    const at::Tensor *x = plain(a[0], m->device), *scales = a[1] != Py_None ? plain(a[1], m->device) : nullptr, *idx = plain(a[2], m->device),
                     *weights = plain(a[3], m->device), *out = a[8] != Py_None ? plain(a[8], m->device) : nullptr;
    if (x == nullptr || idx == nullptr || weights == nullptr || (a[1] != Py_None && scales == nullptr) || (a[8] != Py_None && out == nullptr) ||
        (staged && out == nullptr) || x->dim() != 2 || idx->dim() != 2 || weights->dim() != 2)
        Py_RETURN_NONE;
    const int64_t rows = staged ? out->dim() == 2 ? out->size(0) : 0 : x->size(0);
    const bool bf16 = scales == nullptr;
    auto fits = [&](const at::Tensor& t, int64_t columns) { return t.size(1) == columns && (staged ? t.size(0) >= rows : t.size(0) == rows); };
    if (rows != m->batch || x->size(1) != m->hidden || !fits(*x, m->hidden) || !fits(*idx, m->topk) || !fits(*weights, m->topk) ||
        idx->scalar_type() != at::kInt || weights->scalar_type() != at::kFloat || x->scalar_type() != (bf16 ? at::kBFloat16 : at::kFloat8_e4m3fn) ||
        !aligned16(*x))
        Py_RETURN_NONE;
    if (!bf16 && (scales->dim() != 2 || !fits(*scales, m->hidden / 32) ||
                  (scales->scalar_type() != at::kByte && scales->scalar_type() != at::kFloat8_e8m0fnu)))
        Py_RETURN_NONE;
    const at::Tensor *w1, *s1, *w2, *s2, *sw1 = nullptr, *ss1 = nullptr, *sw2 = nullptr, *ss2 = nullptr;
    if (!read_pair(a[4], true, m->logical1, m->device, &w1, &s1) || !read_pair(a[5], false, m->logical2, m->device, &w2, &s2)) Py_RETURN_NONE;
    if (m->shared > 0) {
        if (!read_pair(a[6], true, m->shared1, m->device, &sw1, &ss1) || !read_pair(a[7], false, m->shared2, m->device, &sw2, &ss2)) Py_RETURN_NONE;
    } else if (a[6] != Py_None || a[7] != Py_None) {
        Py_RETURN_NONE;
    }
    if (out != nullptr) {
        if (out->scalar_type() != at::kBFloat16 || !has_shape(*out, rows, m->hidden) || !aligned16(*out)) Py_RETURN_NONE;
        for (const at::Tensor* t : {x, scales, idx, weights, w1, s1, w2, s2, sw1, ss1, sw2, ss2})
            if (t != nullptr && overlap(*out, *t)) Py_RETURN_NONE;
    }
    Locked held(m->lock);
    if (!held.held) return nullptr;
    if (m->closed || m->workspace == nullptr || rows != m->batch) Py_RETURN_NONE;
    const Stream stream = current_stream(m->device);
    if (m->has_last && !(m->last == stream))
        if (const hipError_t err = m->order.order(stream.raw, m->last.raw); err != hipSuccess) return raise_hip("ordering two streams", err);
    m->last = stream;
    m->has_last = true;
    at::Tensor y = out != nullptr ? *out : allocate({rows, m->hidden}, at::kBFloat16, m->device);
    at::Tensor counts = allocate({m->local}, at::kInt, m->device), scratch;
    dpep_megamoe_call c = {};
    if (bf16) {
        scratch = allocate({rows * m->padded + rows * (m->padded / 32)}, at::kByte, m->device);
        c.x_bf16 = x->data_ptr();
        c.x_codes_scratch = static_cast<uint8_t*>(scratch.data_ptr());
        c.x_scales_scratch = c.x_codes_scratch + rows * m->padded;
    } else {
        c.x_codes = x->data_ptr();
        c.x_scales = static_cast<const uint8_t*>(scales->data_ptr());
    }
    auto bytes = [](const at::Tensor* t) { return t != nullptr ? static_cast<const uint8_t*>(t->data_ptr()) : nullptr; };
    c.topk_idx = static_cast<const int32_t*>(idx->data_ptr());
    c.topk_weights = static_cast<const float*>(weights->data_ptr());
    c.w1 = bytes(w1);
    c.s1 = bytes(s1);
    c.w2 = bytes(w2);
    c.s2 = bytes(s2);
    c.shared_w1 = bytes(sw1);
    c.shared_s1 = bytes(ss1);
    c.shared_w2 = bytes(sw2);
    c.shared_s2 = bytes(ss2);
    c.y = y.data_ptr();
    c.expert_token_nums = static_cast<int32_t*>(counts.data_ptr());
    c.num_shared = m->shared;
    c.num_tokens = static_cast<int32_t>(rows);
    c.hidden = m->hidden;
    c.intermediate = m->inter;
    c.num_topk = m->topk;
    c.num_experts = m->experts;
    c.expert_begin = m->first_expert;
    c.num_local = m->local;
    if (const int status = dpep_megamoe_run(m->workspace, &c, stream.raw)) return raise_native(status);
    Ref first(out != nullptr ? new_ref(a[8]) : wrap(y)), second(wrap(counts));
    return first && second ? PyTuple_Pack(2, first.p, second.p) : nullptr;
    END_HANDLE_TH_ERRORS
}
PyObject* Mega_new(PyTypeObject* type, PyObject* args, PyObject*)
{
    PyObject* lock;
    int device, experts, first, local, topk, hidden, inter, shared, capacity;
    if (!PyArg_ParseTuple(args, "Oiiiiiiiii", &lock, &device, &experts, &first, &local, &topk, &hidden, &inter, &shared, &capacity)) return nullptr;
    Mega* m = reinterpret_cast<Mega*>(type->tp_alloc(type, 0));
    if (m == nullptr) return nullptr;
    m->lock = new_ref(lock);
    m->device = device;
    m->experts = experts;
    m->first_expert = first;
    m->local = local;
    m->topk = topk;
    m->hidden = hidden;
    m->inter = inter;
    m->shared = shared;
    m->capacity = capacity;
    m->padded = dpep_megamoe_padded_dim(hidden);
    m->logical1 = Py_BuildValue("(iii)", local, 2 * inter, hidden);
    m->logical2 = Py_BuildValue("(iii)", local, hidden, inter);
    m->shared1 = Py_BuildValue("(iii)", shared, 2 * inter, hidden);
    m->shared2 = Py_BuildValue("(iii)", shared, hidden, inter);
    return reinterpret_cast<PyObject*>(m);
}
void Mega_dealloc(PyObject* o)
{
    Mega* m = reinterpret_cast<Mega*>(o);
    m->order.release();
    for (PyObject* p : {m->lock, m->logical1, m->logical2, m->shared1, m->shared2}) Py_XDECREF(p);
    Py_TYPE(o)->tp_free(o);
}
// use(workspace handle, batch): the workspace of the batches to come; use(0, 0): none.
PyObject* Mega_use(PyObject* o, PyObject* args)
{
    Mega* m = reinterpret_cast<Mega*>(o);
    PyObject* workspace;
    int batch;
    if (!PyArg_ParseTuple(args, "Oi", &workspace, &batch)) return nullptr;
    void* ws = PyLong_AsVoidPtr(workspace);
    if (ws == nullptr && PyErr_Occurred()) return nullptr;
    m->workspace = ws;
    m->batch = batch;
    Py_RETURN_NONE;
}
PyObject* Mega_close(PyObject* o, PyObject*)
{
    reinterpret_cast<Mega*>(o)->closed = true;
    Py_RETURN_NONE;
}
PyObject* Mega_get_last(PyObject* o, void*)
{
    Mega* m = reinterpret_cast<Mega*>(o);
    if (!m->has_last) Py_RETURN_NONE;
    return stream_object(m->last, m->device);
}
int Mega_set_last(PyObject* o, PyObject* v, void*)
{
    Mega* m = reinterpret_cast<Mega*>(o);
    m->has_last = v != nullptr && v != Py_None;
    return !m->has_last || stream_from(v, &m->last) ? 0 : -1;
}
PyMethodDef mega_methods[] = {
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(Mega_forward)), METH_FASTCALL, nullptr},
    {"use", Mega_use, METH_VARARGS, nullptr},
    {"close", Mega_close, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyGetSetDef mega_getset[] = {{"last_stream", Mega_get_last, Mega_set_last, nullptr, nullptr}, {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject MegaType = {PyVarObject_HEAD_INIT(nullptr, 0) "deepep_amd._host.Mega", sizeof(Mega)};

// ---- FP8 casts -----------------------------------------------------------------------------------------------------------------
// cast_to_fp8(x) -> (codes, scales): a plain BF16 [T,H] on the current GPU, H a positive multiple of 16; else None.
PyObject* cast_to_fp8(PyObject*, PyObject* o)
{
    HANDLE_TH_ERRORS
    if (!on_gpu(o)) Py_RETURN_NONE;
    const int device = c10::hip::current_device();
    const at::Tensor* x = plain(o, device);
    if (x == nullptr || x->scalar_type() != at::kBFloat16 || x->dim() != 2 || x->size(1) == 0 || x->size(1) % 16 != 0 || x->size(0) > 0x7fffffff ||
        x->size(1) > 0x7fffffff || !aligned16(*x) || c10::InferenceMode::is_enabled())
        Py_RETURN_NONE;
    const int64_t tokens = x->size(0), hidden = x->size(1);
    at::Tensor codes = allocate({tokens, hidden}, at::kFloat8_e4m3fn, device), scales = allocate({tokens, (hidden + 127) / 128}, at::kFloat, device);
    if (const int status = dpep_cast_to_fp8(x->data_ptr(), static_cast<int>(tokens), static_cast<int>(hidden), codes.data_ptr(),
                                            static_cast<float*>(scales.data_ptr()), current_stream(device).raw))
        return raise_native(status);
    Ref first(wrap(codes)), second(wrap(scales));
    return first && second ? PyTuple_Pack(2, first.p, second.p) : nullptr;
    END_HANDLE_TH_ERRORS
}
// cast_back(codes, scales) -> BF16 [T,H]: plain e4m3fn codes and FP32 [T, ceil(H/128)] or packed int32 [T, ceil(H/128)/4] scales.
PyObject* cast_back(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (n != 2) {
        PyErr_SetString(PyExc_TypeError, "cast_back takes 2 arguments");
        return nullptr;
    }
    if (!on_gpu(a[0])) Py_RETURN_NONE;
    const int device = c10::hip::current_device();
    const at::Tensor *codes = plain(a[0], device), *scales = plain(a[1], device);
    if (codes == nullptr || scales == nullptr || codes->scalar_type() != at::kFloat8_e4m3fn || codes->dim() != 2 || codes->numel() == 0 ||
        codes->size(1) % 16 != 0 || codes->size(0) > 0x7fffffff || codes->size(1) > 0x7fffffff || !aligned16(*codes) || c10::InferenceMode::is_enabled())
        Py_RETURN_NONE;
    const int64_t tokens = codes->size(0), hidden = codes->size(1), blocks = (hidden + 127) / 128;
    const bool packed = scales->scalar_type() == at::kInt;
    if (packed ? blocks % 4 != 0 || !has_shape(*scales, tokens, blocks / 4) : scales->scalar_type() != at::kFloat || !has_shape(*scales, tokens, blocks))
        Py_RETURN_NONE;
    at::Tensor out = allocate({tokens, hidden}, at::kBFloat16, device);
    if (const int status = dpep_cast_back(codes->data_ptr(), scales->data_ptr(), packed, static_cast<int>(tokens), static_cast<int>(hidden),
                                          out.data_ptr(), current_stream(device).raw))
        return raise_native(status);
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// configure_mega(_PreparedPair, NativeError)
PyObject* configure_mega(PyObject*, PyObject* args)
{
    PyObject *pair, *error;
    if (!PyArg_ParseTuple(args, "O!O", &PyType_Type, &pair, &error)) return nullptr;
    g_pair_type = reinterpret_cast<PyTypeObject*>(new_ref(pair));
    g_native_error = new_ref(error);
    Py_RETURN_NONE;
}

// configure(EPHandle, template dict, EventOverlap, EventHandle, NativeError, (most tokens, hidden, top-k, experts, low-latency
// tokens)): the Python classes whose objects are made here, and the bounds.
PyObject* configure(PyObject*, PyObject* args)
{
    PyObject *handle, *form, *overlap, *event, *error;
    if (!PyArg_ParseTuple(args, "O!O!O!O!O(iiiii)", &PyType_Type, &handle, &PyDict_Type, &form, &PyType_Type, &overlap, &PyType_Type, &event,
                          &error, &g_max_tokens, &g_max_hidden, &g_max_topk, &g_max_experts, &g_low_latency_max_tokens))
        return nullptr;
    g_handle_type = reinterpret_cast<PyTypeObject*>(new_ref(handle));
    g_handle_template = PyDict_Copy(form);
    g_overlap_type = reinterpret_cast<PyTypeObject*>(new_ref(overlap));
    g_event_type = reinterpret_cast<PyTypeObject*>(new_ref(event));
    g_native_error = new_ref(error);
    if (g_handle_template == nullptr) return nullptr;
    Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {{"configure", configure, METH_VARARGS, nullptr},
                                {"configure_mega", configure_mega, METH_VARARGS, nullptr},
                                {"cast_to_fp8", cast_to_fp8, METH_O, nullptr},
                                {"cast_back", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(cast_back)), METH_FASTCALL, nullptr},
                                {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Native host path of deepep_amd (see csrc/host.cpp).", -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host()
{
#define X(n) \
    if ((N.n = PyUnicode_InternFromString(#n)) == nullptr) return nullptr;
    DPEP_NAMES(X)
#undef X
    if ((g_empty_tuple = PyTuple_New(0)) == nullptr) return nullptr;
    LeaseType.tp_dealloc = Lease_dealloc;
    LeaseType.tp_methods = lease_methods;
    MarkerType.tp_methods = marker_methods;
    MarkerType.tp_getset = marker_getset;
    PlanType.tp_dealloc = Plan_dealloc;
    PlanType.tp_methods = plan_methods;
    ExchangeType.tp_dealloc = Exchange_dealloc;
    ExchangeType.tp_methods = exchange_methods;
    ExchangeType.tp_getset = exchange_getset;
    ExchangeType.tp_new = Exchange_new;
    MegaType.tp_dealloc = Mega_dealloc;
    MegaType.tp_methods = mega_methods;
    MegaType.tp_getset = mega_getset;
    MegaType.tp_new = Mega_new;
    if ((g_native_error = new_ref(PyExc_RuntimeError)) == nullptr) return nullptr;  // (until the Python layer names its own)
    for (PyTypeObject* t : {&LeaseType, &MarkerType, &PlanType, &ExchangeType, &MegaType}) {
        t->tp_flags = Py_TPFLAGS_DEFAULT;
        if (PyType_Ready(t) < 0) return nullptr;
    }
    PyObject* m = PyModule_Create(&module_def);
    if (m == nullptr) return nullptr;
    if (PyModule_AddObject(m, "Exchange", new_ref(reinterpret_cast<PyObject*>(&ExchangeType))) < 0) return nullptr;
    if (PyModule_AddObject(m, "Mega", new_ref(reinterpret_cast<PyObject*>(&MegaType))) < 0) return nullptr;
    return m;
}
