// Native form of the Python binding's calls (tilexr_amd/ep.py has their signatures): arguments straight from the interpreter
// into the C ABI.  Through ctypes a decode-sized dispatch + combine spent more on the conversion of its forty arguments than
// the two launches take.
//
// The module does not link against the library: ep.py hands it the entry points of the one it has loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <initializer_list>
#include <type_traits>

#include "tilexr_ep.h"

namespace {

// What a parameter takes.  Integers are what ctypes takes for the C type: an int, an object with __index__ (numpy integers,
// integer tensors of one element), an instance of that ctypes type, or an object whose _as_parameter_ is one of these.
enum class Kind {
    kPointer,       // None, an address, or an object with data_ptr()
    kInt64,
    kInt32,
    kField,         // a 64-bit integer that becomes a field of an options struct: no _as_parameter_
    kInt32OrNone,
    kEvent,         // an address, or anything false for none
    kStream,        // None, an address, or an object with cuda_stream
    kComm,          // None, an address, or an object whose `handle` is None, an address or has an integer `value`
};

struct Param {
    const char *name;
    Kind kind;
    int64_t preset;             // value of an argument that is left out; required ones come first and have none
};

constexpr int kMaxParams = 40;
constexpr int64_t kNone = INT64_MIN;        // a kInt32OrNone argument that is None

struct Function {
    const char *name;
    const Param *params;
    int required;
    int total;
    PyObject *names[kMaxParams];            // interned
};

PyObject *gDataPtr, *gCudaStream, *gHandle, *gValue, *gAsParameter;
PyObject *gCInt64, *gCInt32;            // ctypes.c_int64, ctypes.c_int32

struct Entries {
    decltype(&TileXRMoeEpDispatchV2) dispatchV2;
    decltype(&TileXRMoeEpDispatchMemoryV2) dispatchMemoryV2;
    decltype(&TileXRMoeEpCombineV2) combineV2;
    decltype(&TileXRMoeEpCombineMemoryV2) combineMemoryV2;
    decltype(&TileXRMoeEpDispatchMemoryEx) dispatchMemoryEx;
    decltype(&TileXRMoeEpCombineMemoryEx) combineMemoryEx;
};
Entries gEntries {};

// Integers are taken modulo 2^64, as ctypes takes them.
bool FromInt(PyObject *o, int64_t *out)
{
    if (!PyLong_Check(o)) {
        PyErr_Format(PyExc_TypeError, "an integer is required, not %.80s", Py_TYPE(o)->tp_name);
        return false;
    }
    *out = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(o));
    return !PyErr_Occurred();
}

// What data_ptr(), cuda_stream or value gave (a new reference): an address, None for a null one.
bool FromResult(PyObject *o, int64_t *out)
{
    *out = 0;
    const bool ok = o != nullptr && (o == Py_None || FromInt(o, out));
    Py_XDECREF(o);
    return ok;
}

bool FromInteger(PyObject *o, Kind kind, int64_t *out)
{
    if (PyLong_Check(o)) {
        return FromInt(o, out);
    }
    if (PyIndex_Check(o)) {
        PyObject *index = PyNumber_Index(o);
        return index != nullptr && FromResult(index, out);
    }
    const int ofType = PyObject_IsInstance(o, kind == Kind::kInt64 || kind == Kind::kField ? gCInt64 : gCInt32);
    if (ofType != 0) {
        return ofType > 0 && FromResult(PyObject_GetAttr(o, gValue), out);
    }
    PyObject *inner = kind == Kind::kField ? nullptr : PyObject_GetAttr(o, gAsParameter);
    if (inner != nullptr) {
        bool ok = false;
        if (Py_EnterRecursiveCall(" while taking _as_parameter_") == 0) {
            ok = FromInteger(inner, kind, out);
            Py_LeaveRecursiveCall();
        }
        Py_DECREF(inner);
        return ok;
    }
    if (PyErr_Occurred() && !PyErr_ExceptionMatches(PyExc_AttributeError)) {
        return false;
    }
    PyErr_Clear();
    return FromInt(o, out);         // says what it is not
}

bool Convert(PyObject *o, Kind kind, int64_t *out)
{
    if (kind == Kind::kInt64 || kind == Kind::kInt32 || kind == Kind::kField || (kind == Kind::kInt32OrNone && o != Py_None)) {
        const bool ok = FromInteger(o, kind, out);
        if (ok && kind != Kind::kInt64 && kind != Kind::kField) {
            *out = static_cast<int32_t>(*out);      // kNone is no value of it
        }
        return ok;
    }
    if (o == Py_None) {
        *out = kind == Kind::kInt32OrNone ? kNone : 0;
        return true;
    }
    if (PyLong_Check(o)) {
        return FromInt(o, out);
    }
    if (kind == Kind::kPointer) {
        return FromResult(PyObject_CallMethodNoArgs(o, gDataPtr), out);
    }
    if (kind == Kind::kStream) {
        return FromResult(PyObject_GetAttr(o, gCudaStream), out);
    }
    if (kind == Kind::kEvent) {
        const int given = PyObject_IsTrue(o);
        *out = 0;
        return given == 0 || (given > 0 && FromInt(o, out));
    }
    PyObject *handle = PyObject_GetAttr(o, gHandle);
    if (handle == nullptr || handle == Py_None || PyLong_Check(handle)) {
        return FromResult(handle, out);
    }
    PyObject *value = PyObject_GetAttr(handle, gValue);
    Py_DECREF(handle);
    return FromResult(value, out);
}

// The arguments of a call in the order of the parameters; false with an exception set.
bool Parse(const Function &f, PyObject *const *args, Py_ssize_t positional, PyObject *keywords, int64_t (&out)[kMaxParams])
{
    if (positional > f.total) {
        PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", f.name, f.total, positional);
        return false;
    }
    uint64_t have = 0;
    for (int i = 0; i < positional; ++i) {
        if (!Convert(args[i], f.params[i].kind, &out[i])) {
            return false;
        }
        have |= uint64_t{1} << i;
    }
    const Py_ssize_t named = keywords == nullptr ? 0 : PyTuple_GET_SIZE(keywords);
    for (Py_ssize_t k = 0; k < named; ++k) {
        PyObject *name = PyTuple_GET_ITEM(keywords, k);
        int at = -1;
        // a keyword written at the call is interned like the names here
        for (int i = 0; i < f.total && at < 0; ++i) {
            at = name == f.names[i] ? i : -1;
        }
        for (int i = 0; i < f.total && at < 0; ++i) {
            at = PyUnicode_Compare(name, f.names[i]) == 0 ? i : -1;
        }
        if (at < 0) {
            PyErr_Format(PyExc_TypeError, "%s() got an unexpected keyword argument '%U'", f.name, name);
            return false;
        }
        if ((have >> at & 1) != 0) {
            PyErr_Format(PyExc_TypeError, "%s() got multiple values for argument '%U'", f.name, name);
            return false;
        }
        if (!Convert(args[positional + k], f.params[at].kind, &out[at])) {
            return false;
        }
        have |= uint64_t{1} << at;
    }
    for (int i = 0; i < f.total; ++i) {
        if ((have >> i & 1) != 0) {
            continue;
        }
        if (i < f.required) {
            PyErr_Format(PyExc_TypeError, "%s() missing required argument: '%s'", f.name, f.params[i].name);
            return false;
        }
        out[i] = f.params[i].preset;
    }
    return true;
}

template <typename T>
T As(int64_t v)
{
    if constexpr (std::is_pointer_v<T>) {
        return reinterpret_cast<T>(static_cast<uintptr_t>(v));
    } else {
        return static_cast<T>(v);
    }
}

// An entry point's parameter, converted to whatever its declaration says.
struct Value {
    int64_t v;
    template <typename T>
    operator T() const
    {
        return As<T>(v);
    }
};

template <typename Entry>
bool Bound(Entry entry)
{
    if (entry == nullptr) {
        PyErr_SetString(PyExc_RuntimeError, "bind() first");
    }
    return entry != nullptr;
}

// The call runs without the interpreter's lock, as a ctypes call does.
template <typename Call>
int Unlocked(Call call)
{
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = call();
    Py_END_ALLOW_THREADS
    return status;
}

using K = Kind;

#define PARSE_OR_RETURN(F, ENTRY)                                                                  \
    int64_t a[kMaxParams];                                                                         \
    const auto entry = gEntries.ENTRY;          /* read with the lock held: bind() writes it so */  \
    if (!Bound(entry) || !Parse(F, args, PyVectorcall_NARGS(nargs), keywords, a)) {                \
        return nullptr;                                                                            \
    }                                                                                              \
    auto p = [&a](int i) { return Value {a[i]}; }

// ---- dispatch_v2 ---------------------------------------------------------------------------------------------------
const Param kDispatchV2[] = {
    {"x", K::kPointer, 0}, {"expert_ids", K::kPointer, 0}, {"comm", K::kComm, 0}, {"bs", K::kInt64, 0}, {"h", K::kInt64, 0},
    {"top_k", K::kInt64, 0}, {"experts", K::kInt64, 0}, {"expand_x", K::kPointer, 0}, {"assist", K::kPointer, 0},
    {"token_nums", K::kPointer, 0}, {"recv_counts", K::kPointer, 0}, {"dtype", K::kInt32, 0}, {"stream", K::kStream, 0},
    {"scales", K::kPointer, 0}, {"active_mask", K::kPointer, 0}, {"expert_scales", K::kPointer, 0},
    {"ep_world_size", K::kInt64, 0}, {"ep_rank_id", K::kInt64, 0}, {"tp_world_size", K::kInt64, 0}, {"tp_rank_id", K::kInt64, 0},
    {"expert_shard_type", K::kInt64, 0}, {"shared_expert_num", K::kInt64, 0}, {"shared_expert_rank_num", K::kInt64, 0},
    {"quant_mode", K::kInt64, 0}, {"global_bs", K::kInt64, 0}, {"token_nums_type", K::kInt64, 1},
    {"dynamic_scales", K::kPointer, 0}, {"tp_recv_counts", K::kPointer, 0}, {"expand_scales", K::kPointer, 0},
    {"workspace", K::kPointer, 0},
};
Function gDispatchV2 {"dispatch_v2", kDispatchV2, 13, sizeof(kDispatchV2) / sizeof(Param), {}};

PyObject *DispatchV2(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *keywords)
{
    PARSE_OR_RETURN(gDispatchV2, dispatchV2);
    return PyLong_FromLong(Unlocked([&] {
        return entry(p(0), p(1), p(13), p(14), p(15), p(2), p(3), p(4), p(5), p(6), p(16), p(17), p(18), p(19),
            p(20), p(21), p(22), p(23), p(24), p(25), p(7), p(26), p(8), p(9), p(10), p(27), p(28), p(29), p(11), p(12));
    }));
}

// ---- dispatch_memory_v2 --------------------------------------------------------------------------------------------
const Param kDispatchMemoryV2[] = {
    {"x", K::kPointer, 0}, {"expert_ids", K::kPointer, 0}, {"comm", K::kComm, 0}, {"bs", K::kInt64, 0}, {"h", K::kInt64, 0},
    {"top_k", K::kInt64, 0}, {"experts", K::kInt64, 0}, {"expand_x", K::kPointer, 0}, {"assist", K::kPointer, 0},
    {"token_nums", K::kPointer, 0}, {"send_counts", K::kPointer, 0}, {"dtype", K::kInt32, 0}, {"stream", K::kStream, 0},
    {"scales", K::kPointer, 0}, {"active_mask", K::kPointer, 0}, {"active_mask_type", K::kInt64, TileXREp::TILEXR_EP_ACTIVE_MASK_NONE},
    {"expert_scales", K::kPointer, 0}, {"ep_world_size", K::kInt64, 0}, {"ep_rank_id", K::kInt64, 0},
    {"tp_world_size", K::kInt64, 1}, {"tp_rank_id", K::kInt64, 0}, {"expert_shard_type", K::kInt64, 0},
    {"shared_expert_num", K::kInt64, 0}, {"shared_expert_rank_num", K::kInt64, 0}, {"quant_mode", K::kInt64, 0},
    {"global_bs", K::kInt64, 0}, {"token_nums_type", K::kInt64, 1}, {"dynamic_scales", K::kPointer, 0},
    {"tp_recv_counts", K::kPointer, 0}, {"expand_scales", K::kPointer, 0},
    {"expand_x_dtype", K::kInt32, TileXR::TILEXR_DATA_TYPE_RESERVED},
};
Function gDispatchMemoryV2 {"dispatch_memory_v2", kDispatchMemoryV2, 13, sizeof(kDispatchMemoryV2) / sizeof(Param), {}};

PyObject *DispatchMemoryV2(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *keywords)
{
    PARSE_OR_RETURN(gDispatchMemoryV2, dispatchMemoryV2);
    return PyLong_FromLong(Unlocked([&] {
        return entry(p(0), p(1), p(13), p(14), p(15), p(16), p(2), p(3), p(4), p(5), p(6), p(17), p(18),
            p(19), p(20), p(21), p(22), p(23), p(24), p(25), p(26), p(7), p(27), p(8), p(9), p(10), p(28), p(29), p(11), p(30),
            p(12));
    }));
}

// ---- combine_v2 ----------------------------------------------------------------------------------------------------
const Param kCombineV2[] = {
    {"expert_out", K::kPointer, 0}, {"assist", K::kPointer, 0}, {"recv_counts", K::kPointer, 0}, {"comm", K::kComm, 0},
    {"bs", K::kInt64, 0}, {"h", K::kInt64, 0}, {"top_k", K::kInt64, 0}, {"experts", K::kInt64, 0}, {"y", K::kPointer, 0},
    {"dtype", K::kInt32, 0}, {"stream", K::kStream, 0}, {"workspace", K::kPointer, 0},
};
Function gCombineV2 {"combine_v2", kCombineV2, 11, sizeof(kCombineV2) / sizeof(Param), {}};

PyObject *CombineV2(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *keywords)
{
    PARSE_OR_RETURN(gCombineV2, combineV2);
    return PyLong_FromLong(Unlocked([&] {
        return entry(p(0), p(1), p(2), p(3), p(4), p(5), p(6), p(7), p(8), p(11), p(9), p(10));
    }));
}

// ---- combine_memory_v2 ---------------------------------------------------------------------------------------------
const Param kCombineMemoryV2[] = {
    {"expert_out", K::kPointer, 0}, {"assist", K::kPointer, 0}, {"send_counts", K::kPointer, 0}, {"comm", K::kComm, 0},
    {"bs", K::kInt64, 0}, {"h", K::kInt64, 0}, {"top_k", K::kInt64, 0}, {"experts", K::kInt64, 0}, {"y", K::kPointer, 0},
    {"dtype", K::kInt32, 0}, {"stream", K::kStream, 0}, {"expert_scales", K::kPointer, 0}, {"active_mask", K::kPointer, 0},
    {"active_mask_type", K::kInt64, TileXREp::TILEXR_EP_ACTIVE_MASK_NONE}, {"shared_expert_x", K::kPointer, 0},
    {"ep_world_size", K::kInt64, 0}, {"ep_rank_id", K::kInt64, 0}, {"tp_world_size", K::kInt64, 1}, {"tp_rank_id", K::kInt64, 0},
    {"expert_shard_type", K::kInt64, 0}, {"shared_expert_num", K::kInt64, 0}, {"shared_expert_rank_num", K::kInt64, 0},
    {"quant_mode", K::kInt64, 0}, {"global_bs", K::kInt64, 0},
};
Function gCombineMemoryV2 {"combine_memory_v2", kCombineMemoryV2, 11, sizeof(kCombineMemoryV2) / sizeof(Param), {}};

PyObject *CombineMemoryV2(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *keywords)
{
    PARSE_OR_RETURN(gCombineMemoryV2, combineMemoryV2);
    return PyLong_FromLong(Unlocked([&] {
        return entry(p(0), p(1), p(2), p(11), p(12), p(13), p(14), p(3), p(4), p(5), p(6), p(7), p(15),
            p(16), p(17), p(18), p(19), p(20), p(21), p(22), p(23), p(8), p(9), p(10));
    }));
}

// ---- dispatch_memory_ex: (status, epoch) ---------------------------------------------------------------------------
const Param kDispatchEx[] = {
    {"x", K::kPointer, 0}, {"expert_ids", K::kPointer, 0}, {"comm", K::kComm, 0}, {"bs", K::kInt64, 0}, {"h", K::kInt64, 0},
    {"top_k", K::kInt64, 0}, {"experts", K::kInt64, 0}, {"expand_x", K::kPointer, 0}, {"assist", K::kPointer, 0},
    {"token_nums", K::kPointer, 0}, {"send_counts", K::kPointer, 0}, {"dtype", K::kInt32, 0}, {"stream", K::kStream, 0},
    {"quant_mode", K::kField, 0}, {"expert_capacity", K::kField, 0}, {"token_nums_type", K::kField, 1},
    {"active_mask", K::kPointer, 0}, {"active_mask_type", K::kField, TileXREp::TILEXR_EP_ACTIVE_MASK_NONE},
    {"dynamic_scales", K::kPointer, 0}, {"expand_x_dtype", K::kInt32OrNone, kNone}, {"row_index_map", K::kPointer, 0},
    {"tile_flags", K::kPointer, 0}, {"tile_rows", K::kField, 0}, {"meta_ready_event", K::kEvent, 0},
};
Function gDispatchEx {"dispatch_memory_ex", kDispatchEx, 13, sizeof(kDispatchEx) / sizeof(Param), {}};

PyObject *DispatchEx(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *keywords)
{
    PARSE_OR_RETURN(gDispatchEx, dispatchMemoryEx);
    int64_t epoch = 0;
    TileXREpDispatchExOptions opt {};
    opt.quantMode = p(13);
    opt.expertCapacity = p(14);
    opt.expertTokenNumsType = p(15);
    opt.xActiveMask = p(16);
    opt.activeMaskType = p(17);
    opt.rowIndexMapOut = p(20);
    opt.tileFlagsOut = p(21);
    opt.tileRows = p(22);
    opt.epochOut = &epoch;
    opt.metaReadyEvent = p(23);
    if (a[19] == kNone) {
        a[19] = a[13] == TileXREp::TILEXR_EP_QUANT_TOKEN_INT8 ? int64_t{TileXR::TILEXR_DATA_TYPE_INT8} :
            a[13] == TileXREp::TILEXR_EP_QUANT_MXFP8 || a[13] == TileXREp::TILEXR_EP_QUANT_FP8_BLOCK128 ? int64_t{TileXR::TILEXR_DATA_TYPE_FP8E4M3} :
            a[11];
    }
    const int status = Unlocked([&] {
        return entry(p(0), p(1), p(2), p(3), p(4), p(5), p(6), &opt, p(7), p(18), p(8), p(9), p(10), p(11),
            p(19), p(12));
    });
    return Py_BuildValue("(iL)", status, static_cast<long long>(epoch));
}

// ---- combine_memory_ex ---------------------------------------------------------------------------------------------
const Param kCombineEx[] = {
    {"expert_out", K::kPointer, 0}, {"assist", K::kPointer, 0}, {"send_counts", K::kPointer, 0}, {"comm", K::kComm, 0},
    {"bs", K::kInt64, 0}, {"h", K::kInt64, 0}, {"top_k", K::kInt64, 0}, {"experts", K::kInt64, 0}, {"y", K::kPointer, 0},
    {"dtype", K::kInt32, 0}, {"stream", K::kStream, 0}, {"comm_quant_mode", K::kField, 0}, {"expert_out_quant_mode", K::kField, 0},
    {"expert_out_scales", K::kPointer, 0}, {"expert_scales", K::kPointer, 0}, {"active_mask", K::kPointer, 0},
    {"active_mask_type", K::kField, TileXREp::TILEXR_EP_ACTIVE_MASK_NONE}, {"shared_expert_x", K::kPointer, 0},
    {"row_index_map", K::kPointer, 0}, {"tile_flags", K::kPointer, 0}, {"tile_rows", K::kField, 0}, {"flag_epoch", K::kField, 0},
    {"wait_timeout_us", K::kField, 0}, {"device_status", K::kPointer, 0},
};
Function gCombineEx {"combine_memory_ex", kCombineEx, 11, sizeof(kCombineEx) / sizeof(Param), {}};

PyObject *CombineEx(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *keywords)
{
    PARSE_OR_RETURN(gCombineEx, combineMemoryEx);
    TileXREpCombineExOptions opt {};
    opt.commQuantMode = p(11);
    opt.expertOutQuantMode = p(12);
    opt.expertOutScales = p(13);
    opt.expertScales = p(14);
    opt.xActiveMask = p(15);
    opt.activeMaskType = p(16);
    opt.sharedExpertX = p(17);
    opt.rowIndexMap = p(18);
    opt.tileFlags = p(19);
    opt.tileRows = p(20);
    opt.flagEpoch = p(21);
    opt.waitTimeoutUs = p(22);
    opt.deviceStatusOut = p(23);
    return PyLong_FromLong(Unlocked([&] {
        return entry(p(0), p(1), p(2), p(3), p(4), p(5), p(6), p(7), &opt, p(8), p(9), p(10));
    }));
}

// bind(addresses): the entry points, as integers, in the order of Entries.
PyObject *Bind(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    int64_t at[6];
    if (nargs != 6) {
        PyErr_SetString(PyExc_TypeError, "bind() takes the addresses of six entry points");
        return nullptr;
    }
    for (int i = 0; i < 6; ++i) {
        if (!FromInt(args[i], &at[i])) {
            return nullptr;
        }
    }
    gEntries = {As<decltype(Entries::dispatchV2)>(at[0]), As<decltype(Entries::dispatchMemoryV2)>(at[1]),
        As<decltype(Entries::combineV2)>(at[2]), As<decltype(Entries::combineMemoryV2)>(at[3]),
        As<decltype(Entries::dispatchMemoryEx)>(at[4]), As<decltype(Entries::combineMemoryEx)>(at[5])};
    Py_RETURN_NONE;
}

template <typename F>
PyCFunction Method(F f)
{
    return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

constexpr int kFast = METH_FASTCALL | METH_KEYWORDS;

PyMethodDef kMethods[] = {
    {"bind", Method(Bind), METH_FASTCALL, nullptr},
    {"dispatch_v2", Method(DispatchV2), kFast,
     "dispatch_v2($module, /, x, expert_ids, comm, bs, h, top_k, experts, expand_x, assist, token_nums, "
     "recv_counts, dtype, stream, scales=None, active_mask=None, expert_scales=None, ep_world_size=0, "
     "ep_rank_id=0, tp_world_size=0, tp_rank_id=0, expert_shard_type=0, shared_expert_num=0, "
     "shared_expert_rank_num=0, quant_mode=0, global_bs=0, token_nums_type=1, dynamic_scales=None, "
     "tp_recv_counts=None, expand_scales=None, workspace=None)\n--\n\nReturns the status code."},
    {"dispatch_memory_v2", Method(DispatchMemoryV2), kFast,
     "dispatch_memory_v2($module, /, x, expert_ids, comm, bs, h, top_k, experts, expand_x, assist, token_nums, "
     "send_counts, dtype, stream, scales=None, active_mask=None, active_mask_type=0, expert_scales=None, "
     "ep_world_size=0, ep_rank_id=0, tp_world_size=1, tp_rank_id=0, expert_shard_type=0, shared_expert_num=0, "
     "shared_expert_rank_num=0, quant_mode=0, global_bs=0, token_nums_type=1, dynamic_scales=None, "
     "tp_recv_counts=None, expand_scales=None, expand_x_dtype=255)\n--\n\nReturns the status code."},
    {"combine_v2", Method(CombineV2), kFast,
     "combine_v2($module, /, expert_out, assist, recv_counts, comm, bs, h, top_k, experts, y, dtype, stream, "
     "workspace=None)\n--\n\nReturns the status code."},
    {"combine_memory_v2", Method(CombineMemoryV2), kFast,
     "combine_memory_v2($module, /, expert_out, assist, send_counts, comm, bs, h, top_k, experts, y, dtype, "
     "stream, expert_scales=None, active_mask=None, active_mask_type=0, shared_expert_x=None, ep_world_size=0, "
     "ep_rank_id=0, tp_world_size=1, tp_rank_id=0, expert_shard_type=0, shared_expert_num=0, "
     "shared_expert_rank_num=0, quant_mode=0, global_bs=0)\n--\n\nReturns the status code."},
    {"dispatch_memory_ex", Method(DispatchEx), kFast,
     "dispatch_memory_ex($module, /, x, expert_ids, comm, bs, h, top_k, experts, expand_x, assist, token_nums, "
     "send_counts, dtype, stream, quant_mode=0, expert_capacity=0, token_nums_type=1, active_mask=None, "
     "active_mask_type=0, dynamic_scales=None, expand_x_dtype=None, row_index_map=None, tile_flags=None, "
     "tile_rows=0, meta_ready_event=None)\n--\n\nReturns (status, epoch)."},
    {"combine_memory_ex", Method(CombineEx), kFast,
     "combine_memory_ex($module, /, expert_out, assist, send_counts, comm, bs, h, top_k, experts, y, dtype, "
     "stream, comm_quant_mode=0, expert_out_quant_mode=0, expert_out_scales=None, expert_scales=None, "
     "active_mask=None, active_mask_type=0, shared_expert_x=None, row_index_map=None, tile_flags=None, "
     "tile_rows=0, flag_epoch=0, wait_timeout_us=0, device_status=None)\n--\n\nReturns the status code."},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__calls()
{
    gDataPtr = PyUnicode_InternFromString("data_ptr");
    gCudaStream = PyUnicode_InternFromString("cuda_stream");
    gHandle = PyUnicode_InternFromString("handle");
    gValue = PyUnicode_InternFromString("value");
    gAsParameter = PyUnicode_InternFromString("_as_parameter_");
    PyObject *ctypes = PyImport_ImportModule("ctypes");
    if (ctypes == nullptr) {
        return nullptr;
    }
    gCInt64 = PyObject_GetAttrString(ctypes, "c_int64");
    gCInt32 = PyObject_GetAttrString(ctypes, "c_int32");
    Py_DECREF(ctypes);
    if (gCInt64 == nullptr || gCInt32 == nullptr) {
        return nullptr;
    }
    for (Function *f : {&gDispatchV2, &gDispatchMemoryV2, &gCombineV2, &gCombineMemoryV2, &gDispatchEx, &gCombineEx}) {
        for (int i = 0; i < f->total; ++i) {
            f->names[i] = PyUnicode_InternFromString(f->params[i].name);
        }
    }
    return PyModule_Create(&kModule);
}
