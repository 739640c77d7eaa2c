"""The extension module in front of the C ABI, without a GPU: built from source with the stream
look-up replaced by a null stream and entry points that only count their calls.

Tensors without storage (sparse ones, batched ones under torch.vmap) have no data pointer; asking
them for one raises, and has to raise with the interpreter lock held, whatever other threads do.
"""
import subprocess
import sys
import sysconfig
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

NULL_STREAM = """#pragma once
namespace c10::hip {
struct NullStream {
    void* stream() const { return nullptr; }
};
inline NullStream getCurrentHIPStream() { return {}; }
}  // namespace c10::hip
"""

PROGRAM = r"""
import ctypes, gc, importlib.machinery, importlib.util, sys, threading
import torch
sys.path.insert(0, sys.argv[1])
from neuralfn_amd import engine_ops, kquant, tile_ops

loader = importlib.machinery.ExtensionFileLoader("_front_end", sys.argv[2])
front = importlib.util.module_from_spec(importlib.util.spec_from_loader("_front_end", loader))
loader.exec_module(front)
calls = []
entry = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: calls.append(1) or 0)
nbytes = ctypes.CFUNCTYPE(ctypes.c_int64)(lambda: 4096)
front.bind({name: ctypes.cast(nbytes if "workspace_bytes" in name else entry, ctypes.c_void_p).value
            for name in front.entry_points()}, tile_ops.check)
tile_ops._front = front

def floats(*shape):
    return torch.zeros(shape)

def weight(data=None):
    data = torch.zeros(288, dtype=torch.uint8) if data is None else data
    return tile_ops.PackedWeight(kquant.Q4_K, 2, 256, data)

x, block, norm = floats(1, 256), floats(3, 256), floats(256)
scratch, cache = torch.zeros(4096, dtype=torch.uint8), torch.zeros((8, 256), dtype=torch.bfloat16)
out, position = floats(1, 2), torch.zeros(1, dtype=torch.int64)
heads, kv, rows, kv_rows = floats(4, 64), floats(2, 64), floats(3, 4, 64), floats(3, 2, 64)
w = weight()

# (name, call, its tensors): every tensor is replaced in turn by one without storage
CALLS = [
    ("linear", lambda d, x, b: tile_ops.linear(weight(d), x, b), [w.data, x, floats(2)]),
    ("mmvq_linear", lambda d, x, s, o: tile_ops.mmvq_linear(weight(d), x, s, out=o), [w.data, x, scratch, out]),
    ("gate_up_swiglu", lambda d, x, o: tile_ops.gate_up_swiglu(weight(d), w, x, out=o), [w.data, x, out]),
    ("gate_up_swiglu_rows", lambda d, x, s, o: tile_ops.gate_up_swiglu_rows(w, weight(d), x, 3, s, out=o),
     [w.data, block, scratch, floats(3, 2)]),
    ("lm_head_argmax", lambda d, x, s, i, m: tile_ops.lm_head_argmax(weight(d), x, s, i, m),
     [w.data, x, scratch, position, floats(1)]),
    ("gemm", lambda d, x, s, o: tile_ops.gemm(weight(d), x, workspace=s, out=o),
     [w.data, block, scratch, floats(3, 2)]),
    ("gemm_multi", lambda d, x, s, o: tile_ops.gemm_multi([w, weight(d)], x, workspace=s, outputs=[floats(3, 2), o]),
     [w.data, block, scratch, floats(3, 2)]),
    ("dual_rms_add_capture", lambda x, r: tile_ops.dual_rms_add_capture(x, r), [x, x.clone()]),
    ("dual_rms_add_capture handoff", lambda x, r, s: tile_ops.dual_rms_add_capture(x, r, handoff_workspace=s),
     [x, x.clone(), scratch]),
    ("dual_rms_multi_linear", lambda x, r, d, o: tile_ops.dual_rms_multi_linear(x, r, [weight(d)], outputs=[o]),
     [x, x.clone(), w.data, out]),
    ("qk_norm_scale_rope", lambda q, k: engine_ops.qk_norm_scale_rope(q, k), [heads, kv]),
    ("qk_norm_scale_rope batch", lambda q, k: engine_ops.qk_norm_scale_rope(q, k), [rows, kv_rows]),
]
for family in ("mmq", "mmvq"):
    for prologue in ("plain", "gated", "swiglu"):
        tensors = [w.data, x, scratch, out] + ([] if prologue == "plain" else [x.clone()])
        CALLS.append((f"multi_linear {family} {prologue}",
                      lambda d, x, s, o, second=None, family=family, prologue=prologue: tile_ops.multi_linear(
                          [w, weight(d)], x, s, second=second, family=family, prologue=prologue, outputs=[out, o]),
                      tensors))
    CALLS.append((f"multi_linear_prequantized {family}",
                  lambda d, s, o, family=family: tile_ops.multi_linear_prequantized([weight(d)], 1, s, [o], family),
                  [w.data, scratch, out]))
for split in (False, True):
    extra = [scratch] if split else []
    CALLS.append((f"gqa_decode split={split}",
                  lambda q, k, v, kc, vc, o, s=None: engine_ops.gqa_decode(q, k, v, kc, vc, 0, 0, 1.0, out=o, workspace=s),
                  [heads, kv, kv.clone(), cache, cache.clone(), heads.clone()] + extra))
    CALLS.append((f"block_attention split={split}",
                  lambda q, k, v, kc, vc, o, s=None: engine_ops.block_attention(q, k, v, kc, vc, 0, 0, 1.0, True, out=o,
                                                                                workspace=s),
                  [rows, kv_rows, kv_rows.clone(), cache, cache.clone(), rows.clone()] + extra))
    for device_position in (False, True):
        CALLS.append((f"fused_decode_attention split={split} device_position={device_position}",
                      lambda q, k, v, kc, vc, o, *rest, split=split, on_device=device_position:
                          engine_ops.fused_decode_attention(q, k, v, kc, vc, 0, 0, 1.0, out=o,
                                                            workspace=rest[0] if split else None,
                                                            device_position=rest[-1] if on_device else None),
                      [heads, kv, kv.clone(), cache, cache.clone(), heads.clone()] + extra +
                      ([position] if device_position else [])))

stop = threading.Event()
def busy():
    while not stop.is_set():
        sum(range(100))
thread = threading.Thread(target=busy, daemon=True)
thread.start()
covered = set()
for name, function, tensors in CALLS:
    print(name, flush=True)
    covered.add(name.split()[0])
    before = len(calls)
    function(*tensors)
    assert len(calls) == before + 1, name
    for index in range(len(tensors)):
        def replaced(other):
            return function(*tensors[:index], other, *tensors[index + 1:])
        for kind, attempt in (("sparse", lambda: replaced(tensors[index].to_sparse())),
                              ("vmap", lambda: torch.vmap(replaced)(tensors[index].unsqueeze(0)))):
            try:
                attempt()
            except RuntimeError as error:
                assert "torage" in str(error), (name, index, kind, str(error))
            else:
                raise AssertionError((name, index, kind, "not refused"))
    assert len(calls) == before + 1, name
stop.set()
thread.join()
functions = {name for name in dir(front) if not name.startswith("_")} - {"bind", "entry_points", "stream_handle"}
assert functions == covered, functions ^ covered
# outputs that were made before an allocation is refused are given back
endless = tile_ops.PackedWeight(kquant.Q4_K, 1 << 50, 256, w.data)
def refused():
    try:
        tile_ops.multi_linear([w, endless], x, scratch)
    except RuntimeError:
        return
    raise AssertionError("an endless output was allocated")
def held():
    return sum(type(item) is torch.Tensor for item in gc.get_objects())
before = held()
for _ in range(20):
    refused()
assert held() == before, held() - before
# the kinds of exception that torch's own methods raise
for function in (lambda: tile_ops.linear(w, torch.tensor(0.0)), lambda: tile_ops.gemm(w, torch.tensor(0.0), workspace=scratch)):
    try:
        function()
    except IndexError:
        pass
    else:
        raise AssertionError("a tensor without rows is not refused")
print("all refused")
"""


@pytest.fixture(scope="module")
def front_end(tmp_path_factory):
    cpp_extension = pytest.importorskip("torch.utils.cpp_extension")
    folder = tmp_path_factory.mktemp("front_end")
    (folder / "c10" / "hip").mkdir(parents=True)
    (folder / "c10" / "hip" / "HIPStream.h").write_text(NULL_STREAM)
    includes = [*cpp_extension.include_paths("cuda"), sysconfig.get_paths()["include"]]
    target = folder / "_front_end.so"
    result = subprocess.run(
        ["g++", "-std=c++17", "-O0", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-I{folder}",
         *(f"-isystem{path}" for path in includes),
         str(ROOT / "neuralfn_amd" / "csrc" / "python" / "front_end.cpp"), "-o", str(target),
         *(f"-L{path}" for path in cpp_extension.library_paths("cuda")), "-lc10", "-ltorch_cpu", "-ltorch_python"],
        capture_output=True, text=True)
    assert result.returncode == 0, result.stderr
    return target


def test_a_tensor_without_storage_is_refused_with_an_exception_by_every_call(front_end):
    """In a process of its own: a raise without the interpreter lock aborts it."""
    result = subprocess.run([sys.executable, "-c", PROGRAM, str(ROOT), str(front_end)], capture_output=True, text=True,
                            timeout=300)
    assert result.returncode == 0, result.stdout[-500:] + result.stderr[-3000:]
    assert result.stdout.strip().endswith("all refused")
