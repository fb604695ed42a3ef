"""The binding's native calls against the ctypes binding of the same entry points: names, defaults, what is refused, and which
argument of the C ABI each argument becomes (a shared object of the test's own stands in for the library)."""
import ctypes as C
import inspect
import os
import subprocess

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
