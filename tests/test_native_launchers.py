"""The native launchers (host/launch.cpp) on the CPU, over a stand-in for libwdl.so that launches nothing: every entry
point of the C ABI sleeps and returns 0."""

import importlib.machinery
import importlib.util
import shutil
import subprocess
import threading
import time

import pytest
import torch

SLEEP = 0.2
BF = torch.bfloat16


def _stand_in(at, version):
    """A copy of the launchers, whose entry points are its own, and a stand-in of that ABI version."""
    from wdl import _lib

    _lib.host()  # built and loadable
    lines = ["#include <unistd.h>"]
    for name in _lib.SIGNATURES:
        if name == "wdl_last_error":
            lines.append(f'const char* {name}() {{ return ""; }}')
        elif _lib.RESTYPES.get(name) is _lib.c_i64:
            lines.append(f"long {name}() {{ return 64; }}")
        elif name == "wdl_abi_version":
            lines.append(f"int {name}() {{ return {version}; }}")
        else:
            lines.append(f"int {name}() {{ usleep({int(SLEEP * 1e6)}); return 0; }}")
    (at / "stub.c").write_text("\n".join(lines))
    subprocess.run(["gcc", "-w", "-shared", "-fPIC", str(at / "stub.c"), "-o", str(at / "stub.so")], check=True)
    shutil.copy(_lib.HOST_PATH, at / "wdl_host.so")
    loader = importlib.machinery.ExtensionFileLoader("wdl_host", str(at / "wdl_host.so"))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("wdl_host", loader))
    loader.exec_module(module)
    return module, str(at / "stub.so")


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    from wdl import _lib

    module, library = _stand_in(tmp_path_factory.mktemp("stand_in"), _lib.library().wdl_abi_version())
    module.bind(library)
    return module


def test_a_library_of_another_abi_version_is_refused(tmp_path):
    """The launchers pass the arguments of the header they were compiled with: beside a library of another version they
    would pass wrong ones, so binding refuses it and names both."""
    from wdl import _lib

    version = _lib.library().wdl_abi_version()
    assert f"#define WDL_ABI_VERSION {version}\n" in (_lib.LIB_PATH.parents[2] / "include" / "wdl.h").read_text()
    module, library = _stand_in(tmp_path, version + 1)
    with pytest.raises(RuntimeError, match=f"ABI version {version + 1}, .* compiled for {version}"):
        module.bind(library)


def _calls():
    """One valid call of each launcher: name -> arguments."""
    x, f32 = torch.zeros(4, 128, dtype=BF), torch.zeros(256)
    codes, asc, pairs = (torch.zeros(1, 2, 128, 48, dtype=torch.uint8), torch.zeros(2, 128, dtype=BF),
                         torch.zeros(2, 128, dtype=torch.int32))
    lora, vec = torch.zeros(128, 32), torch.zeros(128, dtype=BF)
    ck, cs = torch.zeros(1, 12, 1, 128, dtype=torch.uint8), torch.ones(1, 12, 1, 1)
    table, kv = torch.zeros(2, 16, 64), torch.zeros(1, 4, 1, 128, dtype=BF)
    k8, ks, v8, vs = torch.zeros(1, 64, 128, dtype=torch.int8), f32, torch.zeros(1, 128, 64, dtype=torch.uint8), f32
    stats = torch.zeros(2, 1, 128)
    return dict(
        act_quant=(x, vec, None, 0.0, False, False, None, None, None, None, 1e-6, None, None, 0),
        gemm=(codes, asc, lora, codes, pairs, vec, vec, 4, torch.zeros(4, 128, dtype=BF), 0, None, None, None, 0),
        gelu_quant=(codes, asc, lora, codes, pairs, vec, vec, 4, vec, vec, 0),
        qk_norm_rope=(x, x, vec, vec, table, 1, 2, 2, 0, 1e-6, None, None, 0),
        sage_prep=(ck, cs, ck, cs, x, x, 8, 16, stats, True, 0),
        sage_attn_q16=(x, k8, ks, v8, vs, 64, 0.1, None, 0, None, 0),
        attn_bf16=(x, x, x, 4, 0.1, None, 0),
        kv_append=(kv, kv, ck, cs, ck, cs, 8, 0),
        fp8_quantize=(x, False, 128, 0),
        fp8_gemm=(torch.zeros(128, 128, dtype=torch.uint8), f32, 4, torch.zeros(128, 128, dtype=torch.uint8), f32, None,
                  False, None, 0),
        fp8wo_gemm=(x, torch.zeros(128, 128, dtype=torch.uint8), f32, None, torch.zeros(4, 128, dtype=BF), None, 0),
        rope3d=(kv, table, [1, 2, 2], 0, False, BF, 0),
    )


def test_a_call_of_each_launcher_is_listed(stand_in):
    launchers = {name for name in dir(stand_in) if not name.startswith("_")}
    assert launchers - {"bind", "kv_valid", "attend_valid"} == set(_calls())


@pytest.mark.parametrize("name", sorted(_calls()))
def test_other_threads_run_while_a_launch_waits(stand_in, name):
    """A launch may wait (a full queue, a first module load, an allocator's retry): the interpreter's lock is released
    meanwhile, as a ctypes call releases it, so the program's other Python threads go on."""
    launch = threading.Thread(target=getattr(stand_in, name), args=_calls()[name])
    launch.start()
    ticks = 0
    while launch.is_alive():
        time.sleep(SLEEP / 50)
        ticks += 1
    launch.join()
    assert ticks >= 10, ticks


@pytest.mark.parametrize("name,which,more", [("act_quant", 0, 1), ("act_quant", 0, -1), ("qk_norm_rope", 0, 1),
                                             ("qk_norm_rope", 0, -1), ("kv_append", 0, 1), ("kv_append", 0, -1),
                                             ("kv_append", 1, -1), ("rope3d", 0, 1), ("rope3d", 0, -1),
                                             ("rope3d", 1, -1)])
def test_tensors_of_another_number_of_dimensions_are_refused(stand_in, name, which, more):
    """The operators under the checked functions read sizes and strides by position: a tensor with a dimension too
    many would be read as if its last one were not there."""
    args = list(_calls()[name])
    args[which] = args[which][..., None] if more > 0 else args[which][0]
    with pytest.raises(ValueError, match="dimensions"):
        getattr(stand_in, name)(*args)


def test_the_rotation_needs_a_grid_for_each_sample(stand_in):
    args = list(_calls()["rope3d"])
    args[2] = [1, 2]
    with pytest.raises(ValueError, match="grid"):
        stand_in.rope3d(*args)


@pytest.mark.parametrize("shape,key", [((0, 4, 2, 128), ""), ((1, 0, 2, 128), "0,1,1"), ((0, 0, 2, 128), "1,1,1")])
def test_an_empty_rotation_needs_no_launch(shape, key):
    """The operator gives an empty tensor for an empty one, whatever the grids, also where there is no GPU."""
    import wdl.rope

    y = wdl.rope.rope3d_rotate(torch.empty(shape), torch.zeros(2, 16, 64), key, 0, False, BF)
    assert y.shape == shape and y.dtype == BF
