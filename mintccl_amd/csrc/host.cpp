// mintccl_amd._host: the host side of an operator call, native.
//
// A small collective takes the GPU 4 us and used to take the host 30: eight
// rank contexts, eight sets of tensor checks, dictionaries, a descriptor filled
// field by field through ctypes and two foreign calls (allgather of 512 B: 50 us
// per call, 7 of them the kernel).  Here a rank's call is one native call that
// checks the tensor and notes its address, and the call that completes the set
// fills the descriptor and launches.
//
// Board is the part of a communicator (common.VirtualComm) that gathers the
// ranks' arguments.  Where the communicator's rings run inside compute units it
// launches them itself; anything else it hands back to the operator, which goes
// on in Python.  What a launch takes from the communicator's attributes (ring,
// protocol, spin limit, status block, which methods a subclass or the object has
// replaced) is asked for once and again after any of them has been set, or the
// class has been changed (VirtualComm._refresh).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>
#include <strings.h>
#include <vector>

#include "../../include/mintccl.h"

namespace {

// The library's entry points, by address: ctypes has loaded it (_lib.lib), from
// wherever MINTCCL_LIBRARY says.
struct Native {
    int (*launch)(const mint_ring_op*, void*);
    int (*grid)(const mint_ring_op*);
    int (*pack)(const void*, void*, size_t, uint64_t, uint64_t, int, void*);
    int (*unpack)(const void*, void*, size_t, uint64_t, uint64_t, int, void*, void*);
    size_t (*packed_bytes)(size_t, int);
    PyObject* check;             // _lib.check(code, where): raises MintError
    PyObject* empty_bytes;       // _lib.empty_bytes(n, like): torch.empty
} native = {};

PyObject* raise(PyObject* type, const char* text) {
    PyErr_SetString(type, text);
    return nullptr;
}

PyObject* checked(int code, const char* where) {
    if (code == MINT_OK) Py_RETURN_NONE;
    return PyObject_CallFunction(native.check, "is", code, where);
}

// The current device is `device` for as long as this lives (a launch goes to
// the current device's context).  Where there is only one it is that: nothing to
// ask (53 ns, a small collective takes 4 us and the codec's two calls 6).
struct OnDevice {
    int before, device;
    explicit OnDevice(int d) : before(only() ? d : (int)c10::hip::current_device()), device(d) {
        if (before != device) c10::hip::set_device((c10::DeviceIndex)device);
    }
    static bool only() {
        static const bool one = c10::hip::device_count() == 1;
        return one;
    }
    ~OnDevice() {
        if (before != device) c10::hip::set_device((c10::DeviceIndex)before);
    }
    // (stream() goes through a device guard; the default stream, whose id is 0, is null)
    void* stream() const {
        const auto current = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device);
        return current.id() == 0 ? nullptr : (void*)current.stream();
    }
};

// C++ exceptions (torch's, out of memory) become Python's.
template <typename F>
PyObject* guarded(F&& f) {
    try {
        return f();
    } catch (const std::bad_alloc&) {
        return PyErr_NoMemory();
    } catch (const std::exception& e) {
        if (PyErr_Occurred()) return nullptr;
        return raise(PyExc_RuntimeError, e.what());
    }
}

// ---- kinds of collectives ----------------------------------------------------
enum Kind { BROADCAST, REDUCE, ALLGATHER, REDUCESCATTER, ALLREDUCE, ALLTOALL, KINDS };
struct KindInfo {
    const char* name;
    int op;
    bool rows, reducing;         // a buffer of `world` rows; adds elements
    const char* elsewhere;       // the MINTCCL_TOPOLOGY under which another module does it
};
constexpr KindInfo kKinds[KINDS] = {
    {"broadcast", MINT_OP_BROADCAST, false, false, "tree"},
    {"reduce", MINT_OP_REDUCE, false, true, "tree"},
    {"allgather", MINT_OP_ALLGATHER, true, false, "hypercube"},
    {"reducescatter", MINT_OP_REDUCESCATTER, true, true, "hypercube"},
    {"allreduce", MINT_OP_ALLREDUCE, false, true, nullptr},
    {"alltoall", MINT_OP_ALLTOALL, true, false, nullptr},
};
// `variant` of an allgather: 0 spatial, 1 temporal; of an allreduce: 0 split, 1 fused; -1: not said
enum { SPATIAL = 0, TEMPORAL = 1, NO_SCHEDULE = 2, SPLIT = 0, FUSED = 1, UNSAID = -1 };

struct Post {
    uint64_t in, out, count;
    int dtype;
    long root, variant;
    PyObject *keep_in, *keep_out;        // alive until the launch is enqueued
};
struct Gathering {
    uint32_t present;
    bool asked;                  // a rank of this collective has looked at the environment:
    long env_variant;            // what it says (the others go by the same)
    Post post[MINT_MAX_RANKS];
};
struct Transfer {
    bool given;
    int rank;
    long peer;
    uint64_t ptr, count;
    PyObject* keep;
};

struct Board {
    PyObject_HEAD
    PyObject* comm;              // weak reference
    uint64_t id;                 // of this board, in the threads' lists of ranks
    int world, device;
    bool fresh, native_launch;   // `base` is up to date; it is ours to launch
    bool asks_rank, in_turn;     // Get_rank, rank are the communicator's own: called, not passed by
    PyTypeObject* type;          // the communicator's class and its version when last asked
    unsigned version;            // (assigning __class__ is an attribute set: fresh says so)
    bool has_ring;               // (a topology may have routes and no ring)
    bool keeps_routes;           // no topology of the caller's, who may change it in place
    bool launched;
    mint_ring_op base, last;
    int8_t last_route[MINT_MAX_RANKS + 1];
    Gathering gathering[KINDS];
    Transfer send, recv;
    int8_t route[MINT_MAX_RANKS][MINT_MAX_RANKS][MINT_MAX_RANKS + 1];   // ranks of the route, its length last
};

// The rank a thread speaks for, per board: `with comm.rank(r)`.
struct Here {
    uint64_t board;
    int rank;
};
thread_local std::vector<Here> here;
uint64_t next_board = 1;

int current_rank(const Board* b) {
    for (const Here& h : here)
        if (h.board == b->id) return h.rank;
    return -1;
}
int enter_rank(const Board* b, int rank) {
    for (size_t i = 0; i < here.size(); ++i) {
        if (here[i].board != b->id) continue;
        const int before = here[i].rank;
        if (rank >= 0) here[i].rank = rank;
        else here.erase(here.begin() + (long)i);
        return before;
    }
    if (rank >= 0) here.push_back({b->id, rank});
    return -1;
}
bool rank_or_raise(const Board* b, int* rank) {
    *rank = current_rank(b);
    if (*rank >= 0) return true;
    raise(PyExc_RuntimeError, "no current rank: use `with comm.rank(r):`");
    return false;
}

// A strong reference to the communicator, or an exception.
PyObject* comm_of(const Board* b) {
    PyObject* comm = PyWeakref_GetObject(b->comm);
    return comm == Py_None ? raise(PyExc_RuntimeError, "the communicator is gone") : Py_NewRef(comm);
}

void drop(Gathering* g) {
    for (int r = 0; r < MINT_MAX_RANKS; ++r)
        if (g->present >> r & 1u) {
            Py_CLEAR(g->post[r].keep_in);
            Py_CLEAR(g->post[r].keep_out);
        }
    g->present = 0;
}

// A device tensor of this communicator, contiguous; or an exception.
const at::Tensor* tensor_of(const Board* b, PyObject* o) {
    if (!THPVariable_Check(o) || !THPVariable_Unpack(o).is_cuda()) {
        raise(PyExc_TypeError, "buffer must be a device tensor");
        return nullptr;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    if (t.get_device() != b->device) {
        raise(PyExc_ValueError, "buffer lives on another device than the communicator");
        return nullptr;
    }
    if (!t.is_contiguous()) {
        raise(PyExc_ValueError, "buffer must be contiguous");
        return nullptr;
    }
    return &t;
}
int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kHalf: return MINT_F16;
        case at::kBFloat16: return MINT_BF16;
        case at::kFloat: return MINT_F32;
        default: return -1;
    }
}

// Brings `base` up to date with the communicator's attributes and methods.  A class
// has another version, or none, once anything of it or its bases has been changed.
bool ask(Board* b) {
    PyObject* comm = comm_of(b);
    if (!comm) return false;
    PyObject* done = PyObject_CallMethod(comm, "_refresh", nullptr);     // calls configure()
    Py_INCREF(Py_TYPE(comm));
    Py_XSETREF(b->type, Py_TYPE(comm));
    b->version = b->type->tp_version_tag;
    Py_DECREF(comm);
    Py_XDECREF(done);
    return done != nullptr;
}
// (asked for by every rank's call: a few loads)
inline bool refresh(Board* b) {
    return (b->fresh && b->type && (b->type->tp_flags & Py_TPFLAGS_VALID_VERSION_TAG) &&
            b->version == b->type->tp_version_tag) || ask(b);
}

// The rank this call is made for.
bool calling_rank(Board* b, int* rank) {
    if (!refresh(b)) return false;
    if (!b->asks_rank) return rank_or_raise(b, rank);
    PyObject* comm = comm_of(b);
    PyObject* got = comm ? PyObject_CallMethod(comm, "Get_rank", nullptr) : nullptr;
    const long r = got ? PyLong_AsLong(got) : -1;
    Py_XDECREF(got);
    Py_XDECREF(comm);
    if (PyErr_Occurred()) return false;
    if (r < 0 || r >= b->world) {
        PyErr_Format(PyExc_ValueError, "rank %ld outside world of %d", r, b->world);
        return false;
    }
    *rank = (int)r;
    return true;
}

PyObject* launch(Board* b, const mint_ring_op& op) {
    b->last = op;
    b->launched = true;
    int code;
    {
        OnDevice on(b->device);
        void* const stream = on.stream();
        Py_BEGIN_ALLOW_THREADS
        code = native.launch(&op, stream);
        Py_END_ALLOW_THREADS
    }
    return checked(code, "mint_ring_launch");
}

// What all ranks have to say alike; `what` names it in the message.
template <typename Field>
bool alike(const Board* b, const Gathering& g, const char* what, Field field,
           const char* const* names = nullptr) {
    bool same = true;
    for (int r = 1; r < b->world; ++r) same &= field(g.post[r]) == field(g.post[0]);
    if (same) return true;
    PyObject* vals = PySet_New(nullptr);
    for (int r = 0; vals && r < b->world; ++r) {
        const long long v = (long long)field(g.post[r]);
        PyObject* s = names ? PyUnicode_FromString(names[v]) : PyUnicode_FromFormat("%lld", v);
        if (!s || PySet_Add(vals, s) < 0) Py_CLEAR(vals);
        Py_XDECREF(s);
    }
    PyObject* list = vals ? PySequence_List(vals) : nullptr;
    if (list && PyList_Sort(list) == 0)
        PyErr_Format(PyExc_ValueError, "ranks disagree on %s: %R", what, list);
    Py_XDECREF(list);
    Py_XDECREF(vals);
    return false;
}

// All ranks are there, `last` came last: launch, or hand the arguments back as
// (count, dtype, root, variant, {rank: in}, {rank: out}, kept buffers).
PyObject* complete(Board* b, Kind kind, const Gathering& g, int last) {
    const KindInfo& info = kKinds[kind];
    static const char* const kSchedules[] = {"spatial", "temporal"};
    if (!alike(b, g, "the byte count", [](const Post& p) { return p.count; })) return nullptr;
    if (!alike(b, g, "the root", [](const Post& p) { return p.root; })) return nullptr;
    if (info.reducing && !alike(b, g, "the dtype", [](const Post& p) { return p.dtype; })) return nullptr;
    if (kind == ALLGATHER &&
        !alike(b, g, "the schedule", [](const Post& p) { return p.variant; }, kSchedules))
        return nullptr;
    const uint64_t count = g.post[0].count;
    const long root = g.post[0].root;
    if (kind == ALLTOALL)
        for (int i = 0; i < b->world; ++i)
            for (int o = 0; o < b->world; ++o)
                if (g.post[i].in < g.post[o].out + count && g.post[o].out < g.post[i].in + count)
                    return raise(PyExc_ValueError, "alltoall: out overlaps a rank's buff");
    if (!refresh(b)) return nullptr;
    long variant = g.post[last].variant;
    if (kind == ALLREDUCE && variant == UNSAID) {
        const char* e = getenv("MINTCCL_ALLREDUCE");
        if (e && *e) variant = strcasecmp(e, "split") == 0 ? SPLIT : FUSED;
        else if (b->native_launch) variant = FUSED;
    }
    if (b->native_launch && b->has_ring && !(kind == ALLGATHER && variant == TEMPORAL) &&
        !(kind == ALLREDUCE && variant == SPLIT)) {
        mint_ring_op op = b->base;
        op.op = info.op;
        op.dtype = info.reducing ? g.post[0].dtype : MINT_BYTES;
        op.root = (int32_t)root;
        op.count_bytes = info.rows ? count / (uint64_t)b->world : count;
        op.row_stride = info.rows ? op.count_bytes : 0;
        for (int r = 0; r < b->world; ++r) {
            op.input[r] = kind == BROADCAST && r != root ? 0 : g.post[r].in;
            // reduce writes at its root, broadcast everywhere else
            const bool writes = kind == REDUCE ? r == root : !(kind == BROADCAST && r == root);
            op.output[r] = !writes ? 0 : kind == ALLTOALL ? g.post[r].out : g.post[r].in;
        }
        return launch(b, op);
    }
    PyObject *ins = PyDict_New(), *outs = PyDict_New(), *kept = PyList_New(0);
    bool ok = ins && outs && kept;
    for (int r = 0; ok && r < b->world; ++r) {
        const Post& p = g.post[r];
        PyObject *key = PyLong_FromLong(r), *in = PyLong_FromUnsignedLongLong(p.in),
                 *out = PyLong_FromUnsignedLongLong(p.out);
        ok = key && in && out && PyDict_SetItem(ins, key, in) == 0 && PyDict_SetItem(outs, key, out) == 0 &&
             PyList_Append(kept, p.keep_in) == 0 && (!p.keep_out || PyList_Append(kept, p.keep_out) == 0);
        Py_XDECREF(key);
        Py_XDECREF(in);
        Py_XDECREF(out);
    }
    PyObject* result = ok ? Py_BuildValue("KillOOO", (unsigned long long)count, g.post[0].dtype, root,
                                          variant, ins, outs, kept)
                          : nullptr;
    Py_XDECREF(ins);
    Py_XDECREF(outs);
    Py_XDECREF(kept);
    return result;
}

// post(kind, buff[, root[, schedule or fused, or None[, out]]]): None (not all ranks are there yet,
// or launched), the ranks' arguments (complete()), or False: MINTCCL_TOPOLOGY
// has another module do this collective
PyObject* post(Board* b, Kind kind, PyObject* buff, PyObject* root, PyObject* variant, PyObject* out) {
    const KindInfo& info = kKinds[kind];
    return guarded([&]() -> PyObject* {
        Post p{};
        p.variant = UNSAID;
        if (root && (p.root = PyLong_AsLong(root)) == -1 && PyErr_Occurred()) return nullptr;
        if (variant && variant != Py_None) {
            if (kind == ALLGATHER) {
                if (!PyUnicode_Check(variant)) p.variant = NO_SCHEDULE;
                else p.variant = PyUnicode_CompareWithASCIIString(variant, "spatial") == 0    ? SPATIAL
                                 : PyUnicode_CompareWithASCIIString(variant, "temporal") == 0 ? TEMPORAL
                                                                                             : NO_SCHEDULE;
            } else {
                const int fused = PyObject_IsTrue(variant);
                if (fused < 0) return nullptr;
                p.variant = fused ? FUSED : SPLIT;
            }
        }
        Gathering& g = b->gathering[kind];
        bool asked = g.present && g.asked;
        long env_variant = g.env_variant;
        if (info.elsewhere && p.variant == UNSAID) {
            if (!asked) {
                const char* e = getenv("MINTCCL_TOPOLOGY");
                if (e && strcasecmp(e, info.elsewhere) == 0) Py_RETURN_FALSE;
                env_variant = UNSAID;
                if (kind == ALLGATHER) {
                    e = getenv("MINTCCL_ALLGATHER");
                    env_variant = !e || strcasecmp(e, "spatial") == 0 ? SPATIAL : strcasecmp(e, "temporal") == 0 ? TEMPORAL : NO_SCHEDULE;
                }
                asked = true;
            }
            p.variant = env_variant;
        }
        if (kind == ALLGATHER && (p.variant < SPATIAL || p.variant > TEMPORAL))
            return raise(PyExc_ValueError, "allgather schedule is 'spatial' or 'temporal'");
        const at::Tensor* t = tensor_of(b, buff);
        if (!t) return nullptr;
        p.in = (uint64_t)t->data_ptr();
        p.count = (uint64_t)t->numel() * (uint64_t)t->element_size();
        p.dtype = MINT_BYTES;
        if (info.rows &&
            (kind == ALLGATHER ? p.count % (uint64_t)b->world : (uint64_t)t->numel() % (uint64_t)b->world))
            return raise(PyExc_ValueError, "buffer does not split into world_size rows");
        if (info.reducing && (p.dtype = dtype_code(*t)) < 0)
            return raise(PyExc_TypeError, "reductions take float16, bfloat16 or float32 tensors");
        if (out) {
            const at::Tensor* o = tensor_of(b, out);
            if (!o) return nullptr;
            if ((uint64_t)o->numel() * (uint64_t)o->element_size() != p.count)
                return raise(PyExc_ValueError, "buff and out differ in size");
            p.out = (uint64_t)o->data_ptr();
        }
        int rank;
        if (!calling_rank(b, &rank)) return nullptr;
        if (g.present >> rank & 1u) {
            PyErr_Format(PyExc_RuntimeError, "rank %d called %s twice before the others joined", rank, info.name);
            return nullptr;
        }
        p.keep_in = Py_NewRef(buff);
        p.keep_out = Py_XNewRef(out);
        g.post[rank] = p;
        g.present |= 1u << rank;
        g.asked = asked;
        g.env_variant = env_variant;
        if (g.present != (1u << b->world) - 1u) Py_RETURN_NONE;
        // (taken out before anything can call back or raise)
        Gathering all = g;
        g.present = 0;
        PyObject* result = complete(b, kind, all, rank);
        drop(&all);
        return result;
    });
}

PyObject* board_post(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    if (n < 2 || n > 5) return raise(PyExc_TypeError, "post(kind, buff[, root[, variant or None[, out]]])");
    const long k = PyLong_AsLong(args[0]);
    if (k < 0 || k >= KINDS) return PyErr_Occurred() ? nullptr : raise(PyExc_ValueError, "no such collective");
    return post(reinterpret_cast<Board*>(self), (Kind)k, args[1], n > 2 ? args[2] : nullptr,
                n > 3 ? args[3] : nullptr, n > 4 ? args[4] : nullptr);
}

PyObject* transfer(Board* b, Transfer* t, PyObject* const* args, Py_ssize_t n) {
    if (n != 2) return raise(PyExc_TypeError, "takes a buffer and a peer");
    return guarded([&]() -> PyObject* {
        const at::Tensor* x = tensor_of(b, args[0]);
        if (!x) return nullptr;
        const long peer = PyLong_AsLong(args[1]);
        if (peer == -1 && PyErr_Occurred()) return nullptr;
        int rank;
        if (!calling_rank(b, &rank)) return nullptr;
        PyObject* before = t->given ? t->keep : nullptr;
        *t = Transfer{true, rank, peer, (uint64_t)x->data_ptr(),
                      (uint64_t)x->numel() * (uint64_t)x->element_size(), Py_NewRef(args[0])};
        Py_XDECREF(before);
        Py_RETURN_NONE;
    });
}
PyObject* board_send(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    return transfer(reinterpret_cast<Board*>(self), &reinterpret_cast<Board*>(self)->send, args, n);
}
PyObject* board_recv(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    return transfer(reinterpret_cast<Board*>(self), &reinterpret_cast<Board*>(self)->recv, args, n);
}

// Route into op.ring / op.route_len; `given`: the caller's list, or None for the
// topology's (VirtualComm._find_route; where all ranks are alike once per pair).
bool take_route(Board* b, PyObject* given, int src, int dst, int8_t (&route)[MINT_MAX_RANKS + 1]) {
    const bool cache = given == Py_None && b->keeps_routes && src < b->world && dst < b->world;
    if (cache && b->route[src][dst][MINT_MAX_RANKS]) {
        memcpy(route, b->route[src][dst], sizeof(route));
        return true;
    }
    PyObject* list;
    if (given == Py_None) {
        PyObject* comm = comm_of(b);
        PyObject* found = comm ? PyObject_CallMethod(comm, "_find_route", "ii", src, dst) : nullptr;
        Py_XDECREF(comm);
        list = found ? PySequence_Fast(found, "a route is a sequence of ranks") : nullptr;
        Py_XDECREF(found);
    } else {
        list = PySequence_Fast(given, "a route is a sequence of ranks");
    }
    if (!list) return false;
    const Py_ssize_t len = PySequence_Fast_GET_SIZE(list);
    memset(route, 0, sizeof(route));
    bool ok = len > 0;
    for (Py_ssize_t i = 0; ok && i < len; ++i) {
        const long r = PyLong_AsLong(PySequence_Fast_GET_ITEM(list, i));
        if (r == -1 && PyErr_Occurred()) {
            Py_DECREF(list);
            return false;
        }
        ok = !(i == 0 && r != src) && !(i == len - 1 && r != dst);
        // (a route longer than the world, or over ranks that are not there, is
        // refused by the library: what does not fit is written as no rank)
        if (i < MINT_MAX_RANKS) route[i] = r < 0 || r >= MINT_MAX_RANKS ? (int8_t)-1 : (int8_t)r;
    }
    Py_DECREF(list);
    if (!ok) {
        PyErr_Format(PyExc_ValueError, "no route %d -> %d", src, dst);
        return false;
    }
    route[MINT_MAX_RANKS] = (int8_t)(len > MINT_MAX_RANKS ? MINT_MAX_RANKS + 1 : len);
    if (cache) memcpy(b->route[src][dst], route, sizeof(route));
    return true;
}

// sync(route, staged): the first call that finds a matched pair launches it, or
// hands it back as (source, destination, from, to, bytes, route, kept buffers)
PyObject* board_sync(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    Board* b = reinterpret_cast<Board*>(self);
    if (n != 2) return raise(PyExc_TypeError, "sync(route, staged)");
    if (!b->send.given || !b->recv.given) Py_RETURN_NONE;
    return guarded([&]() -> PyObject* {
        const Transfer s = b->send, r = b->recv;
        b->send.given = b->recv.given = false;
        auto go = [&]() -> PyObject* {
            if (s.peer != r.rank || r.peer != s.rank)
                return raise(PyExc_ValueError, "send and recv do not name each other");
            if (s.count != r.count) return raise(PyExc_ValueError, "send and recv sizes differ");
            if (!refresh(b)) return nullptr;
            int8_t route[MINT_MAX_RANKS + 1];
            if (!take_route(b, args[0], s.rank, r.rank, route)) return nullptr;
            const int len = route[MINT_MAX_RANKS];
            memcpy(b->last_route, route, sizeof(route));
            mint_ring_op op = b->base;
            op.op = MINT_OP_SENDRECV;
            op.dtype = MINT_BYTES;
            op.route_len = len;
            for (int i = 0; i < MINT_MAX_RANKS; ++i) op.ring[i] = i < len ? route[i] : 0;
            op.input[s.rank] = s.ptr;
            op.output[r.rank] = r.ptr;
            op.count_bytes = s.count;
            if (b->native_launch && args[1] == Py_False) return launch(b, op);
            PyObject* list = PyList_New(0);
            bool ok = list != nullptr;
            for (int i = 0; ok && i < len && i < MINT_MAX_RANKS; ++i) {
                PyObject* v = PyLong_FromLong(route[i]);
                ok = v && PyList_Append(list, v) == 0;
                Py_XDECREF(v);
            }
            PyObject* result = ok ? Py_BuildValue("iiKKKO(OO)", s.rank, r.rank, (unsigned long long)s.ptr,
                                                  (unsigned long long)r.ptr, (unsigned long long)s.count,
                                                  list, s.keep, r.keep)
                                  : nullptr;
            Py_XDECREF(list);
            return result;
        };
        PyObject* result = go();
        Py_DECREF(s.keep);
        Py_DECREF(r.keep);
        return result;
    });
}

// speak(rank): a context in which the thread speaks for that rank
struct RankContext {
    PyObject_HEAD
    PyObject* comm;              // owns the board
    Board* board;
    int rank, before;
    bool inside;
};
PyTypeObject context_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
void context_dealloc(PyObject* self) {
    Py_DECREF(reinterpret_cast<RankContext*>(self)->comm);
    Py_DECREF(reinterpret_cast<RankContext*>(self)->board);
    Py_TYPE(self)->tp_free(self);
}
PyObject* context_enter(PyObject* self, PyObject*) {
    RankContext* c = reinterpret_cast<RankContext*>(self);
    // (a second way in would forget whose rank the thread had before the first)
    if (c->inside) return raise(PyExc_RuntimeError, "this context of a rank is entered already");
    c->inside = true;
    c->before = enter_rank(c->board, c->rank);
    return Py_NewRef(c->comm);
}
PyObject* context_exit(PyObject* self, PyObject* const*, Py_ssize_t) {
    RankContext* c = reinterpret_cast<RankContext*>(self);
    c->inside = false;
    enter_rank(c->board, c->before);
    Py_RETURN_NONE;
}
// (as a decorator: every call of the function enters a context of its own)
PyObject* context_call(PyObject* self, PyObject* args, PyObject* kwargs) {
    RankContext* c = reinterpret_cast<RankContext*>(self);
    PyObject* fn;
    if (kwargs && PyDict_GET_SIZE(kwargs)) return raise(PyExc_TypeError, "a rank's decorator takes a function");
    if (!PyArg_ParseTuple(args, "O", &fn)) return nullptr;
    return PyObject_CallMethod(c->comm, "_speaking", "iO", c->rank, fn);
}
PyMethodDef context_methods[] = {
    {"__enter__", context_enter, METH_NOARGS, nullptr},
    {"__exit__", (PyCFunction)(void (*)(void))context_exit, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyObject* board_speak(PyObject* self, PyObject* arg) {
    Board* b = reinterpret_cast<Board*>(self);
    const long r = PyLong_AsLong(arg);
    if (r == -1 && PyErr_Occurred()) return nullptr;
    if (r < 0 || r >= b->world) {
        PyErr_Format(PyExc_ValueError, "rank %ld outside world of %d", r, b->world);
        return nullptr;
    }
    RankContext* c = PyObject_New(RankContext, &context_type);
    if (!c) return nullptr;
    c->comm = Py_NewRef(PyWeakref_GetObject(b->comm));
    c->board = reinterpret_cast<Board*>(Py_NewRef(self));
    c->rank = (int)r;
    c->before = -1;
    c->inside = false;
    return reinterpret_cast<PyObject*>(c);
}
PyObject* board_rank(PyObject* self, PyObject*) {
    int rank;
    return rank_or_raise(reinterpret_cast<Board*>(self), &rank) ? PyLong_FromLong(rank) : nullptr;
}
// run(fn): fn(rank) for every rank in turn
PyObject* board_run(PyObject* self, PyObject* fn) {
    Board* b = reinterpret_cast<Board*>(self);
    if (!refresh(b)) return nullptr;
    if (b->in_turn) {
        PyObject* comm = comm_of(b);
        PyObject* done = comm ? PyObject_CallMethod(comm, "_in_turn", "O", fn) : nullptr;
        Py_XDECREF(comm);
        return done;
    }
    const int before = current_rank(b);
    PyObject* result = Py_NewRef(Py_None);
    for (int r = 0; result && r < b->world; ++r) {
        enter_rank(b, r);
        PyObject* arg = PyLong_FromLong(r);
        PyObject* got = arg ? PyObject_CallOneArg(fn, arg) : nullptr;
        Py_XDECREF(arg);
        if (!got) Py_CLEAR(result);
        Py_XDECREF(got);
    }
    enter_rank(b, before);
    return result;
}

PyObject* board_stale(PyObject* self, PyObject*) {
    reinterpret_cast<Board*>(self)->fresh = false;
    Py_RETURN_NONE;
}
// launching(descriptor): what a launch from Python is about to enqueue (last_grid)
PyObject* board_launching(PyObject* self, PyObject* arg) {
    Board* b = reinterpret_cast<Board*>(self);
    Py_buffer view;
    if (PyObject_GetBuffer(arg, &view, PyBUF_SIMPLE) < 0) return nullptr;
    if (view.len == (Py_ssize_t)sizeof(mint_ring_op)) {
        memcpy(&b->last, view.buf, sizeof(mint_ring_op));
        b->launched = true;
    }
    PyBuffer_Release(&view);
    Py_RETURN_NONE;
}
// configure(native_launch, asks_rank, in_turn, keeps_routes, ring, protocol, spin_budget,
// status): what launches take from the communicator; an empty ring where the topology has none
PyObject* board_configure(PyObject* self, PyObject* args) {
    Board* b = reinterpret_cast<Board*>(self);
    int native_launch, asks_rank, in_turn, keeps_routes, protocol;
    unsigned long spin;
    unsigned long long status;
    PyObject* ring;
    if (!PyArg_ParseTuple(args, "ppppOikK", &native_launch, &asks_rank, &in_turn, &keeps_routes, &ring, &protocol,
                          &spin, &status))
        return nullptr;
    mint_ring_op& d = b->base;
    d = mint_ring_op{};
    PyObject* list = PySequence_Fast(ring, "a ring is a sequence of ranks");
    if (!list) return nullptr;
    for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(list) && i <= MINT_MAX_RANKS; ++i)
        d.ring[i] = (int32_t)PyLong_AsLong(PySequence_Fast_GET_ITEM(list, i));
    Py_DECREF(list);
    if (PyErr_Occurred()) return nullptr;
    b->has_ring = PySequence_Size(ring) == b->world + 1;
    d.protocol = protocol;
    d.world = b->world;
    d.placement = MINT_PLACE_CU;
    d.spin_budget = (uint32_t)spin;
    d.status = status;
    memset(b->route, 0, sizeof(b->route));
    b->native_launch = native_launch;
    b->asks_rank = asks_rank;
    b->in_turn = in_turn;
    b->keeps_routes = keeps_routes;
    b->fresh = true;
    Py_RETURN_NONE;
}

PyObject* board_last_grid(PyObject* self, void*) {
    Board* b = reinterpret_cast<Board*>(self);
    return PyLong_FromLong(b->launched ? native.grid(&b->last) : 0);
}
PyObject* board_last_route(PyObject* self, void*) {
    const int8_t* route = reinterpret_cast<Board*>(self)->last_route;
    PyObject* list = PyList_New(0);
    for (int i = 0; list && i < route[MINT_MAX_RANKS] && i < MINT_MAX_RANKS; ++i) {
        PyObject* v = PyLong_FromLong(route[i]);
        if (!v || PyList_Append(list, v) < 0) Py_CLEAR(list);
        Py_XDECREF(v);
    }
    return list;
}

// Board(comm, world, device index)
PyObject* board_new(PyTypeObject* type, PyObject* args, PyObject*) {
    PyObject* comm;
    int world, device;
    if (!PyArg_ParseTuple(args, "Oii", &comm, &world, &device)) return nullptr;
    if (world < 1 || world > MINT_MAX_RANKS) return raise(PyExc_ValueError, "world is 1..8");
    Board* b = reinterpret_cast<Board*>(type->tp_alloc(type, 0));       // (zeroed)
    if (!b) return nullptr;
    b->id = next_board++;
    b->world = world;
    b->device = device;
    b->comm = PyWeakref_NewRef(comm, nullptr);
    if (!b->comm) Py_CLEAR(b);
    return reinterpret_cast<PyObject*>(b);
}
void board_dealloc(PyObject* self) {
    Board* b = reinterpret_cast<Board*>(self);
    for (Gathering& g : b->gathering) drop(&g);
    if (b->send.given) Py_DECREF(b->send.keep);
    if (b->recv.given) Py_DECREF(b->recv.keep);
    Py_XDECREF(b->comm);
    Py_XDECREF(b->type);
    Py_TYPE(self)->tp_free(self);
}

PyMethodDef board_methods[] = {
    {"post", (PyCFunction)(void (*)(void))board_post, METH_FASTCALL, nullptr},
    {"send", (PyCFunction)(void (*)(void))board_send, METH_FASTCALL, nullptr},
    {"recv", (PyCFunction)(void (*)(void))board_recv, METH_FASTCALL, nullptr},
    {"sync", (PyCFunction)(void (*)(void))board_sync, METH_FASTCALL, nullptr},
    {"speak", board_speak, METH_O, nullptr},
    {"rank", board_rank, METH_NOARGS, nullptr},
    {"run", board_run, METH_O, nullptr},
    {"stale", board_stale, METH_NOARGS, nullptr},
    {"launching", board_launching, METH_O, nullptr},
    {"configure", board_configure, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyGetSetDef board_getset[] = {{"last_grid", board_last_grid, nullptr, nullptr, nullptr},
                              {"last_route", board_last_route, nullptr, nullptr, nullptr},
                              {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject board_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- fronts of the operators ---------------------------------------------------
// Front(operator, action, go_on) stands before an operator written in Python: a
// call that names its communicator goes straight to the board; what is left to
// do where the board has not done it all, go_on(comm, posted) does in
// Python, and any other call (the default communicator, arguments that do not
// fit) is the operator's.  A collective of eight ranks is eight such calls: 0.1 us
// each in place of 0.2.  pack and unpack, which take tensors alone, stand behind one
// each likewise (codec_call): a pair for up to 4 MiB 6.42 us, 6.21 with them.
enum Action { SEND = KINDS, RECV, SYNC, PACK, UNPACK, ACTIONS };
constexpr int kParams = 6;
// the parameters in their order; what is not required comes last
struct FrontInfo {
    const char* names[kParams];
    int required;
} kFronts[ACTIONS] = {
    {{"buff", "root", "comm"}, 2},  {{"buff", "root", "comm"}, 2},     {{"buff", "comm", "schedule"}, 1},
    {{"buff", "comm", nullptr}, 1}, {{"buff", "comm", "fused"}, 1},    {{"buff", "out", "comm"}, 2},
    {{"buff", "peer", "comm"}, 2},  {{"buff", "peer", "comm"}, 2},     {{"comm", "route", nullptr}, 0},
    {{"raw", "flag_base", "layout", "flag_stride", "out"}, 1},
    {{"msg", "out", "flag_base", "layout", "flag_stride", "bad_flags"}, 2}};
PyObject* param_names[ACTIONS][kParams];     // interned
PyObject* board_name;

struct Front {
    PyObject_HEAD
    vectorcallfunc call;
    PyObject *op, *go_on, *dict, *weak;
    PyObject* defaults;          // of a codec call: what the operator declares
    int action;
};

// The arguments of a call, each in its parameter's place; false: they do not fit.
bool take(const Front* f, PyObject* const* args, size_t nargsf, PyObject* kwnames, PyObject* (&given)[kParams]) {
    PyObject* const* names = param_names[f->action];
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf), nk = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    bool fits = n <= kParams && (n == 0 || names[n - 1]);
    for (Py_ssize_t i = 0; fits && i < n; ++i) given[i] = args[i];
    for (Py_ssize_t i = 0; fits && i < nk; ++i) {
        int k = 0;
        while (k < kParams && names[k] != PyTuple_GET_ITEM(kwnames, i)) ++k;
        fits = k < kParams && !given[k];
        if (fits) given[k] = args[n + i];
    }
    for (int k = 0; k < kFronts[f->action].required; ++k) fits = fits && given[k];
    return fits;
}

PyObject* front_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
    Front* f = reinterpret_cast<Front*>(self);
    PyObject* given[kParams] = {};
    const bool fits = take(f, args, nargsf, kwnames, given);
    PyObject* comm = nullptr;
    for (int k = 0; fits && k < kParams && kFronts[f->action].names[k]; ++k)
        if (kFronts[f->action].names[k][0] == 'c') comm = given[k];
    PyObject* board = fits && comm && comm != Py_None ? PyObject_GetAttr(comm, board_name) : nullptr;
    if (!board || Py_TYPE(board) != &board_type) {
        Py_XDECREF(board);
        PyErr_Clear();
        return PyObject_Vectorcall(f->op, args, nargsf, kwnames);
    }
    Board* b = reinterpret_cast<Board*>(board);
    PyObject* result;
    switch (f->action) {
        case BROADCAST:
        case REDUCE: result = post(b, (Kind)f->action, given[0], given[1], nullptr, nullptr); break;
        case ALLTOALL: result = post(b, ALLTOALL, given[0], nullptr, nullptr, given[1]); break;
        case SEND: result = transfer(b, &b->send, given, 2); break;
        case RECV: result = transfer(b, &b->recv, given, 2); break;
        case SYNC: {
            PyObject* const pair[2] = {given[1] ? given[1] : Py_None, Py_False};
            result = board_sync(board, pair, 2);
            break;
        }
        default: result = post(b, (Kind)f->action, given[0], nullptr, given[2], nullptr);
    }
    Py_DECREF(board);
    if (!result || result == Py_None) return result;
    PyObject* const rest[2] = {comm, result};
    // (False: MINTCCL_TOPOLOGY has another module do it)
    PyObject* done = result == Py_False ? PyObject_Vectorcall(f->op, args, nargsf, kwnames)
                                        : PyObject_Vectorcall(f->go_on, rest, 2, nullptr);
    Py_DECREF(result);
    return done;
}

// (until the library is bound, the operator binds it)
PyObject* host_pack(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* host_unpack(PyObject*, PyObject* const* args, Py_ssize_t n);
PyObject* codec_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
    Front* f = reinterpret_cast<Front*>(self);
    PyObject* given[kParams] = {};
    if (!native.pack || !take(f, args, nargsf, kwnames, given)) return PyObject_Vectorcall(f->op, args, nargsf, kwnames);
    const int required = kFronts[f->action].required, all = f->action == PACK ? 5 : 6;
    for (int k = required; k < all; ++k)
        if (!given[k]) given[k] = PyTuple_GET_ITEM(f->defaults, k - required);
    return f->action == PACK ? host_pack(nullptr, given, all) : host_unpack(nullptr, given, all);
}

// Front(operator, action, go_on)
PyObject* front_new(PyTypeObject* type, PyObject* args, PyObject*) {
    PyObject *op, *go_on;
    int action;
    if (!PyArg_ParseTuple(args, "OiO", &op, &action, &go_on)) return nullptr;
    if (action < 0 || action >= ACTIONS) return raise(PyExc_ValueError, "no such action");
    Front* f = reinterpret_cast<Front*>(type->tp_alloc(type, 0));
    if (!f) return nullptr;
    f->call = front_call;
    if (action == PACK || action == UNPACK) {
        f->call = codec_call;
        f->defaults = PyObject_GetAttrString(op, "__defaults__");
        if (!f->defaults || !PyTuple_Check(f->defaults) || PyTuple_GET_SIZE(f->defaults) != 4) {
            Py_DECREF(f);
            return raise(PyExc_ValueError, "four parameters of a codec call have defaults");
        }
    }
    f->op = Py_NewRef(op);
    f->go_on = Py_NewRef(go_on);
    f->action = action;
    return reinterpret_cast<PyObject*>(f);
}
void front_dealloc(PyObject* self) {
    Front* f = reinterpret_cast<Front*>(self);
    if (f->weak) PyObject_ClearWeakRefs(self);
    Py_XDECREF(f->op);
    Py_XDECREF(f->go_on);
    Py_XDECREF(f->defaults);
    Py_XDECREF(f->dict);
    Py_TYPE(self)->tp_free(self);
}
// It is handed on like the function it stands for: pickled and copied by its name
// in its module, bound where a class holds it, referred to weakly.
PyObject* front_reduce(PyObject* self, PyObject*) { return PyObject_GetAttrString(self, "__qualname__"); }
PyObject* front_bind(PyObject* self, PyObject* object, PyObject*) {
    return object && object != Py_None ? PyMethod_New(self, object) : Py_NewRef(self);
}
PyMethodDef front_methods[] = {{"__reduce__", front_reduce, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyTypeObject front_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
// (functools.update_wrapper gives it the operator's name, documentation and signature)
PyGetSetDef front_getset[] = {{"__dict__", PyObject_GenericGetDict, PyObject_GenericSetDict, nullptr, nullptr},
                              {nullptr, nullptr, nullptr, nullptr, nullptr}};

// ---- codec ---------------------------------------------------------------------
const at::Tensor* device_tensor(PyObject* o) {
    if (!THPVariable_Check(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() ? &t : nullptr;
}
size_t bytes_of(const at::Tensor& t) { return (size_t)t.numel() * (size_t)t.element_size(); }

// A message of n bytes beside `like`, allocated where whoever looks at allocations
// sees it: dispatch modes and the profiler through the dispatcher (pack and unpack
// of 1 MiB 7.16 us, 6.96 with the allocator's own entry, which they do not see),
// function modes through torch.empty itself.
PyObject* empty_bytes(size_t n, PyObject* like) {
    if (at::impl::torch_function_mode_enabled())
        return PyObject_CallFunction(native.empty_bytes, "nO", (Py_ssize_t)n, like);
    return THPVariable_Wrap(at::empty({(int64_t)n}, THPVariable_Unpack(like).options().dtype(at::kByte)));
}

// pack(raw, flag_base, layout, flag_stride, out or None)
PyObject* host_pack(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 5) return raise(PyExc_TypeError, "pack(raw, flag_base, layout, flag_stride, out)");
    const uint64_t base = PyLong_AsUnsignedLongLongMask(args[1]), stride = PyLong_AsUnsignedLongLongMask(args[3]);
    const int layout = (int)PyLong_AsLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    return guarded([&]() -> PyObject* {
        const at::Tensor* raw = device_tensor(args[0]);
        if (!raw || !raw->is_contiguous())
            return raise(PyExc_ValueError, "pack needs a contiguous device tensor");
        const size_t nbytes = bytes_of(*raw), need = native.packed_bytes(nbytes, layout);
        PyObject* result;
        if (args[4] == Py_None) {
            result = empty_bytes(need, args[0]);
            if (!result) return nullptr;
        } else {
            const at::Tensor* out = device_tensor(args[4]);
            if (!out) return raise(PyExc_ValueError, "pack needs a contiguous device tensor");
            if (bytes_of(*out) < need) return raise(PyExc_ValueError, "output too small");
            result = Py_NewRef(args[4]);
        }
        OnDevice on(raw->get_device());
        void *const from = raw->data_ptr(), *const to = THPVariable_Unpack(result).data_ptr(), *const stream = on.stream();
        int code;
        Py_BEGIN_ALLOW_THREADS
        code = native.pack(from, to, nbytes, base, stride, layout, stream);
        Py_END_ALLOW_THREADS
        if (code != MINT_OK) {
            Py_DECREF(result);
            return checked(code, "mint_ll128_pack");
        }
        return result;
    });
}

// unpack(msg, out, flag_base, layout, flag_stride, bad_flags or None)
PyObject* host_unpack(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 6) return raise(PyExc_TypeError, "unpack(msg, out, flag_base, layout, flag_stride, bad_flags)");
    const uint64_t base = PyLong_AsUnsignedLongLongMask(args[2]), stride = PyLong_AsUnsignedLongLongMask(args[4]);
    const int layout = (int)PyLong_AsLong(args[3]);
    if (PyErr_Occurred()) return nullptr;
    return guarded([&]() -> PyObject* {
        const at::Tensor *msg = device_tensor(args[0]), *out = device_tensor(args[1]);
        if (!msg || !out || !out->is_contiguous())
            return raise(PyExc_ValueError, "unpack needs contiguous device tensors");
        const size_t nbytes = bytes_of(*out);
        if (bytes_of(*msg) < native.packed_bytes(nbytes, layout))
            return raise(PyExc_ValueError, "message too small");
        void* bad = nullptr;
        if (args[5] != Py_None) {
            if (!THPVariable_Check(args[5])) return raise(PyExc_TypeError, "bad_flags is a tensor");
            bad = THPVariable_Unpack(args[5]).data_ptr();
        }
        OnDevice on(out->get_device());
        void *const from = msg->data_ptr(), *const to = out->data_ptr(), *const stream = on.stream();
        int code;
        Py_BEGIN_ALLOW_THREADS
        code = native.unpack(from, to, nbytes, base, stride, layout, bad, stream);
        Py_END_ALLOW_THREADS
        if (code != MINT_OK) return checked(code, "mint_ll128_unpack");
        return Py_NewRef(args[1]);
    });
}

// bind(launch, grid, pack, unpack, packed_bytes, check, empty_bytes): addresses, what raises, what allocates
PyObject* host_bind(PyObject*, PyObject* args) {
    unsigned long long launch, grid, pack, unpack, packed;
    PyObject *check, *empty;
    if (!PyArg_ParseTuple(args, "KKKKKOO", &launch, &grid, &pack, &unpack, &packed, &check, &empty)) return nullptr;
    native.launch = reinterpret_cast<decltype(native.launch)>(launch);
    native.grid = reinterpret_cast<decltype(native.grid)>(grid);
    native.pack = reinterpret_cast<decltype(native.pack)>(pack);
    native.unpack = reinterpret_cast<decltype(native.unpack)>(unpack);
    native.packed_bytes = reinterpret_cast<decltype(native.packed_bytes)>(packed);
    Py_INCREF(check);
    Py_XSETREF(native.check, check);
    Py_INCREF(empty);
    Py_XSETREF(native.empty_bytes, empty);
    Py_RETURN_NONE;
}

PyMethodDef host_methods[] = {
    {"bind", host_bind, METH_VARARGS, nullptr},
    {"pack", (PyCFunction)(void (*)(void))host_pack, METH_FASTCALL, nullptr},
    {"unpack", (PyCFunction)(void (*)(void))host_unpack, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef host_module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, host_methods,
                           nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    board_type.tp_name = "mintccl_amd._host.Board";
    board_type.tp_basicsize = sizeof(Board);
    board_type.tp_flags = Py_TPFLAGS_DEFAULT;
    board_type.tp_new = board_new;
    board_type.tp_dealloc = board_dealloc;
    board_type.tp_methods = board_methods;
    board_type.tp_getset = board_getset;
    context_type.tp_name = "mintccl_amd._host.RankContext";
    context_type.tp_basicsize = sizeof(RankContext);
    context_type.tp_flags = Py_TPFLAGS_DEFAULT;
    context_type.tp_doc = "with comm.rank(r): the thread speaks for rank r inside; @comm.rank(r): in the function";
    context_type.tp_dealloc = context_dealloc;
    context_type.tp_call = context_call;
    context_type.tp_methods = context_methods;
    if (PyType_Ready(&board_type) < 0 || PyType_Ready(&context_type) < 0) return nullptr;
    front_type.tp_name = "mintccl_amd._host.Front";
    front_type.tp_basicsize = sizeof(Front);
    front_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    front_type.tp_new = front_new;
    front_type.tp_dealloc = front_dealloc;
    front_type.tp_call = PyVectorcall_Call;
    front_type.tp_vectorcall_offset = offsetof(Front, call);
    front_type.tp_dictoffset = offsetof(Front, dict);
    front_type.tp_weaklistoffset = offsetof(Front, weak);
    front_type.tp_descr_get = front_bind;
    front_type.tp_methods = front_methods;
    front_type.tp_getset = front_getset;
    if (PyType_Ready(&front_type) < 0) return nullptr;
    for (int k = 0; k < ACTIONS; ++k)
        for (int i = 0; i < kParams; ++i)
            if (kFronts[k].names[i] && !(param_names[k][i] = PyUnicode_InternFromString(kFronts[k].names[i])))
                return nullptr;
    if (!(board_name = PyUnicode_InternFromString("_board"))) return nullptr;
    PyObject* m = PyModule_Create(&host_module);
    if (!m) return nullptr;
    Py_INCREF(&front_type);
    PyModule_AddObject(m, "Front", reinterpret_cast<PyObject*>(&front_type));
    PyModule_AddIntConstant(m, "SEND", SEND);
    PyModule_AddIntConstant(m, "RECV", RECV);
    PyModule_AddIntConstant(m, "SYNC", SYNC);
    PyModule_AddIntConstant(m, "PACK", PACK);
    PyModule_AddIntConstant(m, "UNPACK", UNPACK);
    PyModule_AddIntConstant(m, "ACTIONS", ACTIONS);
    Py_INCREF(&board_type);
    PyModule_AddObject(m, "Board", reinterpret_cast<PyObject*>(&board_type));
    for (int k = 0; k < KINDS; ++k) {
        char name[32];
        size_t i = 0;
        for (; kKinds[k].name[i]; ++i) name[i] = (char)toupper(kKinds[k].name[i]);
        name[i] = 0;
        PyModule_AddIntConstant(m, name, k);
    }
    PyModule_AddIntConstant(m, "DESCRIPTOR_BYTES", sizeof(mint_ring_op));
    return m;
}
