"""The binding's native calls against the ctypes binding of the same entry points: names, defaults, what is refused, and which
argument of the C ABI each argument becomes (a shared object of the test's own stands in for the library)."""
import ctypes as C
import inspect
import os
import subprocess
import sys
import sysconfig

import pytest

from tilexr_amd import ep

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAMES = list(ep._NATIVE)
PYTHON_FORMS = {n: getattr(ep, n) for n in NAMES}       # replaced once the library is loaded

STAND_IN = r"""
#include <cstdint>
extern "C" {
int64_t seen[64];
int count;
}
#define PUT(v) seen[count++] = (int64_t)(v);
"""


class Tensor:
    def __init__(self, at):
        self.at = at

    def data_ptr(self):
        return self.at


class Stream:
    cuda_stream = 0x5157


class Comm:
    handle = C.c_void_p(0xC033)


@pytest.fixture(scope="module")
def calls(tmp_path_factory):
    """The native module bound to functions that note their arguments, declared as in include/tilexr_ep.h."""
    src = STAND_IN
    header = open(os.path.join(ROOT, "include", "tilexr_ep.h")).read()
    options = {"TileXREpDispatchExOptions": ["quantMode", "expertCapacity", "expertTokenNumsType", "activeMaskType", "xActiveMask",
                                             "rowIndexMapOut", "tileFlagsOut", "tileRows", "metaReadyEvent"],
               "TileXREpCombineExOptions": ["commQuantMode", "expertOutQuantMode", "expertOutScales", "expertScales",
                                            "activeMaskType", "xActiveMask", "sharedExpertX", "rowIndexMap", "tileFlags",
                                            "tileRows", "flagEpoch", "waitTimeoutUs", "deviceStatusOut"]}
    src += '#include "tilexr_ep.h"\nextern "C" {\n'
    for entry in ep._NATIVE.values():
        at = header.index(f"int {entry}(")
        decl = header[at:header.index(";", at)]
        params = [p.split()[-1].lstrip("*") for p in decl[decl.index("(") + 1:decl.rindex(")")].split(",")]
        src += decl.replace(f"int {entry}", f"int stub_{entry}") + " { count = 0;\n"
        for p in params:
            if p == "options":
                kind = "TileXREpDispatchExOptions" if "Dispatch" in entry else "TileXREpCombineExOptions"
                src += "".join(f"PUT(options->{f})" for f in options[kind])
                src += "*options->epochOut = 77;" if "Dispatch" in entry else ""
            else:
                src += f"PUT({p})"
        src += "\nreturn 5; }\n"
    src += "}\n"
    d = tmp_path_factory.mktemp("calls")
    (d / "stub.cpp").write_text(src)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"), str(d / "stub.cpp"), "-o",
                    str(d / "stub.so")], check=True)
    stub = C.CDLL(str(d / "stub.so"))
    from tilexr_amd.lib import _calls
    _calls.bind(*(C.cast(getattr(stub, "stub_" + e), C.c_void_p).value for e in ep._NATIVE.values()))
    yield _calls, stub
    if ep._lib is not None:
        ep._bind(ep._lib)


def _seen(stub):
    n = C.c_int.in_dll(stub, "count").value
    return list((C.c_int64 * 64).in_dll(stub, "seen"))[:n]


# the order of the C ABI, by the binding's names; those of the options in the stand-in's order
ORDER = {
    "dispatch_v2": "x expert_ids scales active_mask expert_scales comm bs h top_k experts ep_world_size ep_rank_id tp_world_size "
                   "tp_rank_id expert_shard_type shared_expert_num shared_expert_rank_num quant_mode global_bs token_nums_type "
                   "expand_x dynamic_scales assist token_nums recv_counts tp_recv_counts expand_scales workspace dtype stream",
    "dispatch_memory_v2": "x expert_ids scales active_mask active_mask_type expert_scales comm bs h top_k experts ep_world_size "
                          "ep_rank_id tp_world_size tp_rank_id expert_shard_type shared_expert_num shared_expert_rank_num "
                          "quant_mode global_bs token_nums_type expand_x dynamic_scales assist token_nums send_counts "
                          "tp_recv_counts expand_scales dtype expand_x_dtype stream",
    "combine_v2": "expert_out assist recv_counts comm bs h top_k experts y workspace dtype stream",
    "combine_memory_v2": "expert_out assist send_counts expert_scales active_mask active_mask_type shared_expert_x comm bs h top_k "
                         "experts ep_world_size ep_rank_id tp_world_size tp_rank_id expert_shard_type shared_expert_num "
                         "shared_expert_rank_num quant_mode global_bs y dtype stream",
    "dispatch_memory_ex": "x expert_ids comm bs h top_k experts quant_mode expert_capacity token_nums_type active_mask_type "
                          "active_mask row_index_map tile_flags tile_rows meta_ready_event expand_x dynamic_scales assist "
                          "token_nums send_counts dtype expand_x_dtype stream",
    "combine_memory_ex": "expert_out assist send_counts comm bs h top_k experts comm_quant_mode expert_out_quant_mode "
                         "expert_out_scales expert_scales active_mask_type active_mask shared_expert_x row_index_map tile_flags "
                         "tile_rows flag_epoch wait_timeout_us device_status y dtype stream",
}


@pytest.mark.parametrize("name", NAMES)
def test_signatures_are_those_of_the_python_forms(name, calls):
    module, _ = calls
    assert str(inspect.signature(getattr(module, name))) == str(inspect.signature(PYTHON_FORMS[name]))


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("by_name", [False, True])
def test_every_argument_reaches_its_place(name, by_name, calls):
    module, stub = calls
    params = list(inspect.signature(PYTHON_FORMS[name]).parameters)
    assert sorted(params) == sorted(ORDER[name].split())
    values = {p: 1000 + i for i, p in enumerate(params)}
    given = {p: (Tensor(v) if i % 2 and p not in ("stream", "comm") else v) for i, (p, v) in enumerate(values.items())}
    ints = {p for p in params if p in ("bs", "h", "top_k", "experts", "dtype", "meta_ready_event", "flag_epoch", "wait_timeout_us")
            or p.endswith(("_num", "_size", "_id", "_type", "_mode", "_bs", "_dtype", "_rows", "_capacity"))}
    for p in ints:
        given[p] = values[p]
    given["stream"], values["stream"] = Stream(), Stream.cuda_stream
    given["comm"], values["comm"] = Comm(), Comm.handle.value
    ret = getattr(module, name)(**given) if by_name else getattr(module, name)(*given.values())
    assert ret == ((5, 77) if name == "dispatch_memory_ex" else 5)
    assert _seen(stub) == [values[p] for p in ORDER[name].split()]


@pytest.mark.parametrize("name", NAMES)
def test_defaults_and_nones(name, calls):
    module, stub = calls
    sig = inspect.signature(PYTHON_FORMS[name]).parameters
    required = [p for p, q in sig.items() if q.default is inspect._empty]
    given = {p: 3 if p in ("bs", "h", "top_k", "experts", "dtype") else None for p in required}
    getattr(module, name)(**given)
    want = {p: (given.get(p, q.default) or 0) for p, q in sig.items()}
    if name == "dispatch_memory_ex":
        want["expand_x_dtype"] = 3
    assert _seen(stub) == [want[p] for p in ORDER[name].split()]


@pytest.mark.parametrize("quant,dtype", [(ep.Q_NONE, ep.DT_BF16), (ep.Q_STATIC_INT8, ep.DT_BF16), (ep.Q_TOKEN_INT8, ep.DT_INT8),
                                         (ep.Q_MXFP8, ep.DT_FP8E4M3), (ep.Q_FP8_BLOCK128, ep.DT_FP8E4M3), (99, ep.DT_BF16)])
def test_payload_type_follows_the_mode(quant, dtype, calls):
    module, stub = calls
    module.dispatch_memory_ex(None, None, None, 1, 2, 3, 4, None, None, None, None, ep.DT_BF16, None, quant_mode=quant)
    assert _seen(stub)[ORDER["dispatch_memory_ex"].split().index("expand_x_dtype")] == dtype


def test_what_is_refused(calls):
    module, _ = calls
    ok = [None, None, None, None, 1, 2, 3, 4, None, 3, None]
    assert module.combine_v2(*ok) == 5
    for args, kwargs, error in ((ok[:-1], {}, TypeError), (ok + [None, None], {}, TypeError), (ok, {"nothing": 1}, TypeError),
                                (ok, {"y": None}, TypeError), (["text"] + ok[1:], {}, AttributeError),
                                (ok[:4] + [1.0] + ok[5:], {}, TypeError), (ok[:4] + [None] + ok[5:], {}, TypeError),
                                (ok[:3] + [object()] + ok[4:], {}, AttributeError), (ok[:-1] + [object()], {}, AttributeError)):
        with pytest.raises(error):
            module.combine_v2(*args, **kwargs)
    closed = Comm()
    closed.handle = None
    assert module.combine_v2(*ok[:3], closed, *ok[4:]) == 5
    # integers are taken as the C types take them
    assert module.combine_v2(*ok[:4], -1, 1 << 64, *ok[6:]) == 5


class Index:
    def __index__(self):
        return 6


class Parameter:
    def __init__(self, inner):
        self._as_parameter_ = inner


def _integers():
    np, torch = pytest.importorskip("numpy"), pytest.importorskip("torch")
    return [True, np.int64(3), np.int32(-4), np.uint64(2 ** 64 - 1), np.array(5), np.array([5]), np.float64(2.0), torch.tensor(7),
            torch.tensor([8]), torch.tensor([1, 2]).max(), torch.tensor(9.0), torch.tensor([1, 2]), Index(), C.c_int64(11), C.c_int32(12),
            C.c_uint64(13), C.c_int16(14), Parameter(15), Parameter(Index()), Parameter(C.c_int64(16)), Parameter(C.c_int32(17)),
            Parameter(Parameter(18)), Parameter("text"), 1.5, "1", b"1", None, 1 << 70, -(1 << 63)]


class Field(C.Structure):
    _fields_ = [("v", C.c_int64)]


def _as_ctypes_takes_it(value, name, param):
    """What the ctypes binding of the entry point makes of an argument; a TypeError where it refuses it."""
    if name.endswith("_ex") and param in ("quant_mode", "expert_capacity", "token_nums_type", "active_mask_type", "tile_rows", "comm_quant_mode",
                                          "expert_out_quant_mode", "flag_epoch", "wait_timeout_us"):
        f = Field()
        f.v = value
        return f.v
    ctype = C.c_int32 if param in ("dtype", "expand_x_dtype") else C.c_int64
    seen = []
    keep = C.CFUNCTYPE(None, ctype)(seen.append)
    raw = C.cast(keep, C.c_void_p).value
    call = C.CFUNCTYPE(None, C.c_int64)(raw) if ctype is C.c_int64 else C.CFUNCTYPE(None, C.c_int32)(raw)
    try:
        call(value)
    except C.ArgumentError as e:
        raise TypeError(str(e))
    return seen[0]


@pytest.mark.parametrize("name", NAMES)
def test_integers_are_those_that_ctypes_takes(name, calls):
    """Every integer argument of every call, given as whatever a program may have a size in: taken, with the value, where ctypes
    takes it, and refused where it is not."""
    module, stub = calls
    sig = inspect.signature(PYTHON_FORMS[name]).parameters
    required = {p: 3 if p in ("bs", "h", "top_k", "experts", "dtype") else None for p, q in sig.items() if q.default is inspect._empty}
    integers = [p for p, q in sig.items() if required.get(p) == 3 or (isinstance(q.default, int) and p != "meta_ready_event")]
    if name.startswith("dispatch_memory"):
        integers = sorted({*integers, "expand_x_dtype"})
    assert len(integers) > 4
    for param in integers:
        for value in _integers():
            if value is None and param == "expand_x_dtype":
                continue            # None stands for the payload type of the mode there
            try:
                want = _as_ctypes_takes_it(value, name, param)
            except TypeError:
                with pytest.raises(TypeError):
                    getattr(module, name)(**{**required, param: value})
                continue
            getattr(module, name)(**{**required, param: value})
            got = _seen(stub)[ORDER[name].split().index(param)]
            # the element types are an enumeration of 32 bits, whose sign is the compiler's choice
            assert (got - want) % (1 << 32 if param in ("dtype", "expand_x_dtype") else 1 << 64) == 0, (param, value)


def test_addresses_that_are_not_plain(calls):
    module, stub = calls
    ok = [None, None, None, None, 1, 2, 3, 4, None, 3, None]

    class Null:
        cuda_stream = None

        def data_ptr(self):
            return None

    raw = Comm()
    raw.handle = 0xC034
    assert module.combine_v2(*ok[:3], raw, *ok[4:]) == 5
    assert _seen(stub)[3] == 0xC034
    assert module.combine_v2(Null(), *ok[1:-1], Null()) == 5
    assert _seen(stub)[0] == 0 and _seen(stub)[-1] == 0
    event = dict(zip("x expert_ids comm bs h top_k experts expand_x assist token_nums send_counts dtype stream".split(),
                     [None, None, None, 1, 2, 3, 4, None, None, None, None, 3, None]))
    at = ORDER["dispatch_memory_ex"].split().index("meta_ready_event")
    for value, want in ((None, 0), (0, 0), (False, 0), ((), 0), (0xE7E, 0xE7E)):
        module.dispatch_memory_ex(**event, meta_ready_event=value)
        assert _seen(stub)[at] == want
    for value in (1.5, "event", object()):
        with pytest.raises(TypeError):
            module.dispatch_memory_ex(**event, meta_ready_event=value)


@pytest.mark.parametrize("name", NAMES)
def test_a_name_taken_before_the_library_was_loaded_binds_nothing_again(name, monkeypatch):
    """`from tilexr_amd.ep import combine_v2` at the top of a program: every call through that name goes straight to the bound
    native module."""
    from tilexr_amd.lib import _calls
    ep._bind(ep.lib())
    binds = []
    monkeypatch.setattr(_calls, "bind", lambda *at: binds.append(at))
    sig = inspect.signature(PYTHON_FORMS[name]).parameters
    given = {p: 3 if p in ("bs", "h", "top_k", "experts", "dtype") else None for p, q in sig.items() if q.default is inspect._empty}
    for _ in range(3):
        ret = PYTHON_FORMS[name](**given)
        assert (ret[0] if name == "dispatch_memory_ex" else ret) == ep.ERR_PARA_CHECK_FAIL
    assert binds == []


def test_a_library_that_cannot_be_bound_is_not_taken_for_loaded(monkeypatch):
    monkeypatch.setattr(ep, "_lib", None)
    monkeypatch.setattr(ep, "_bind", lambda loaded: 1 / 0)
    for _ in range(2):
        with pytest.raises(ZeroDivisionError):
            ep.lib()
    assert ep._lib is None


def _make(*args):
    return subprocess.run(["make", "-C", os.path.join(ROOT, "tilexr_amd", "csrc"), "-n", "-B", *args], capture_output=True, text=True)


def test_the_module_is_for_the_interpreter_that_builds_it(monkeypatch):
    """Its file carries the interpreter's tag (another minor version does not import it), and the build passes the interpreter it
    runs in."""
    from tilexr_amd.lib import _calls
    suffix = sysconfig.get_config_var("EXT_SUFFIX")
    assert os.path.basename(_calls.__file__) == "_calls" + suffix
    built = _make("python", f"PYTHON={sys.executable}")
    assert built.returncode == 0 and f"_calls{suffix}" in built.stdout and "libtilexr-ep" not in built.stdout
    import __graft_entry__ as entry
    ran = []
    monkeypatch.setattr(entry.subprocess, "run", lambda cmd, **kw: ran.append(cmd))
    entry.build()
    assert any(f"PYTHON={sys.executable}" in cmd for cmd in ran)


def test_the_library_builds_without_python_headers():
    for target in ("all", "library"):
        built = _make(target, "PYTHON=/nonexistent/python")
        assert built.returncode == 0, built.stderr
        assert "libtilexr-ep.so" in built.stdout and "py_calls" not in built.stdout
