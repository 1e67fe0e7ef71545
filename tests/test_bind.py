"""What the extension behind the device entry points (csrc/bind.cpp) takes and refuses, on the CPU: in a process of its
own the C ABI is replaced by stubs that record that they were called, and torch's stream query by a constant."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PREAMBLE = r"""
import ctypes as C
import torch
torch.cuda.init = lambda: None
torch._C._cuda_getDevice = lambda: 0
torch._C._cuda_getCurrentRawStream = lambda device: 0
from oxillama_amd import _bind, capi, linear, quant

calls = []
STUB = C.CFUNCTYPE(C.c_int)(lambda: calls.append(1) or 0)  # (the arguments stay unread in their registers)
address = {name: C.cast(STUB, C.c_void_p).value for name in capi.SIGNATURES}

def stub(name, *argtypes):
    "this C function records the given leading arguments instead"
    f = C.CFUNCTYPE(C.c_int, *argtypes)(lambda *a: calls.append(a) or 0)
    keep.append(f)
    address[name] = C.cast(f, C.c_void_p).value

keep = []
capi._attached = _bind
T = torch.zeros(64)

def refused(error, f, *a, **kw):
    n = len(calls)
    try:
        f(*a, **kw)
    except error:
        assert len(calls) == n, "the C ABI was called all the same"
        return
    raise AssertionError((f, a, kw))
"""


def run(body):
    p = subprocess.run([sys.executable, "-c", PREAMBLE + body], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-4000:]


def test_required_tensors_are_refused_as_none_or_integers():
    run(r"""
_bind.attach(address)
# R: a tensor the call needs, O: one it can do without, the rest: numbers and None as they are
R, O = "R", "O"
ENTRIES = {
    "rmsnorm_quantize": (R, R, 1e-5, 1, 64, O, O),
    "linear_forward": (8, R, O, O, O, None, R, 1, 32),
    "linear_forward_batch": (8, R, R, O, R, 1, 1, 32, O),
    "gemm_q8": (8, R, R, R, 1, 1, 32, 0, O),
    "matvec_q8_fused": (8, R, R, R, 1, 32, 0),
    "swiglu_quantize": (R, R, O, O),
    "quantize_q8_0": (R, R),
    "ffn_swiglu": (8, R, 8, R, 8, R, R, R, 32, 32, R),
    "topk": (R, 1, R, R, R),
    "lm_head_topk": (8, R, R, R, 1, 32, 1, R, R, R),
    "logits_edit": (R, O, O, O, O, 0, 1.0),
    "sample_candidates": (R, R, 1, 1.0, 0.0, 1.0, R, R, O),
    "moe_forward": (8, R, 1, 8, R, 1, 8, R, 1, 1, R, R, 1, 1, R, 32, 32, R),
}
entries = {n for n in dir(_bind) if not n.startswith("_")} - {"attach", "linear_forward_multi"}
assert entries == set(ENTRIES), entries ^ set(ENTRIES)
for name, form in ENTRIES.items():
    f = getattr(_bind, name)
    full = [T if a in (R, O) else a for a in form]
    n = len(calls)
    assert f(*full) == 0 and f(*[None if a == O else b for a, b in zip(form, full)]) == 0, name
    assert len(calls) == n + 2
    for i, a in enumerate(form):
        if a == R:
            refused(AttributeError, f, *full[:i], None, *full[i + 1:])
        if a in (R, O):
            refused(AttributeError, f, *full[:i], 4096, *full[i + 1:])
            refused(AttributeError, f, *full[:i], 0, *full[i + 1:])
multi = lambda w=T, a=T, b=None, o=T: _bind.linear_forward_multi(8, [T, w], a, b, [T, o], [1, 1], 32)
assert multi() == 0 and multi(b=[None, T]) == 0
for bad in (None, 4096):
    refused(AttributeError, multi, w=bad)
    refused(AttributeError, multi, a=bad)
    refused(AttributeError, multi, o=bad)
refused(AttributeError, multi, b=[4096, None])
# the public entry points on top
refused(AttributeError, quant.quantize_q8_0_dev, None, T)
refused(AttributeError, quant.quantize_q8_0_dev, T, None)
refused(AttributeError, quant.quantize_q8_0_dev, T, T.data_ptr())
refused(AttributeError, linear.swiglu_quantize_dev, None, T)
refused(AttributeError, linear.rmsnorm_quantize_dev, T, None, 1e-5, 1, 64)
refused(AttributeError, linear.linear_forward_dev, 8, T, None, 1, 32, d_acts=T)
""")


def test_linear_forward_multi_with_fewer_biases_than_matrices():
    """A bias list that ends early leaves the matrices past it without one; the row count of a matrix past the end of the
    row counts is 0 and the number of matrices is not cut short (both refused by the C ABI); an output is needed for
    every weight."""
    run(r"""
V, P = C.c_void_p, C.POINTER(C.c_void_p)
seen = []
def record(t, n, w, acts, b, o, rows, cols):
    k = min(n, 64)
    seen.append((n, [b[i] for i in range(k)] if b else None, [rows[i] for i in range(k)]))
    return 0
f = C.CFUNCTYPE(C.c_int, C.c_uint32, C.c_size_t, P, V, P, P, C.POINTER(C.c_size_t), C.c_size_t)(record)
address["oxq_linear_forward_multi_dev"] = C.cast(f, V).value
_bind.attach(address)
multi = linear.linear_forward_multi_dev
b = torch.zeros(8)
multi(8, [T, T, T], T, [T, T, T], [4, 5, 6], 32, [b])
assert seen.pop() == (3, [b.data_ptr(), None, None], [4, 5, 6])
multi(8, [T, T], T, [T, T], [4, 5], 32, [])
assert seen.pop() == (2, [None, None], [4, 5])
multi(8, (T, T), T, (t for t in (T, T)), (4,), 32)
assert seen.pop() == (2, None, [4, 0])
multi(8, [T] * 70, T, [T] * 70, [1] * 70, 32)
assert seen.pop() == (70, None, [1] * 64)
multi(8, [], T, [], [], 32)
assert seen.pop()[0] == 0
for args in (([T, T], T, [T], [1, 1], 32), ([T], T, [T, T], [1], 32), ([T], T, [T], [1, 1], 32), ([T], T, [T], [1], 32, [b, b])):
    refused(ValueError, multi, 8, *args)
assert not seen
""")


def test_types_and_eps_convert_as_int_and_float_do():
    run(r"""
import numpy as np
stub("oxq_linear_forward_dev", C.c_uint32)
stub("oxq_linear_forward_batch_dev", C.c_uint32)
stub("oxq_linear_forward_multi_dev", C.c_uint32)
stub("oxq_ffn_swiglu_dev", C.c_uint32, C.c_void_p, C.c_uint32, C.c_void_p, C.c_uint32)
f = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_void_p, C.c_float)(lambda x, w, e: calls.append(e) or 0)
address["oxq_rmsnorm_quantize_q8_0_dev"] = C.cast(f, C.c_void_p).value
_bind.attach(address)
for t in (12, 12.0, "12", np.float32(12), np.int64(12), torch.tensor(12), quant.GgufTensorType.Q4K):
    linear.linear_forward_dev(t, T, T, 1, 32, d_acts=T)
    linear.linear_forward_batch_dev(t, T, T, T, 1, 1, 32)
    linear.linear_forward_multi_dev(t, [T], T, [T], [1], 32)
    assert [calls.pop() for _ in range(3)] == [(12,)] * 3, t
    linear.ffn_swiglu_dev((t, T), (t, T), (t, T), T, T, 32, 32, T)
    a = calls.pop()
    assert (a[0], a[2], a[4]) == (12, 12, 12)
for e in (0.5, 1, "0.5", np.float32(0.5), torch.tensor(0.5)):
    linear.rmsnorm_quantize_dev(T, T, e, 1, 64, T)
    assert calls.pop() == float(e), e
for bad in (None, "q4", [1]):
    refused((TypeError, ValueError), linear.linear_forward_dev, bad, T, T, 1, 32, d_acts=T)
    refused((TypeError, ValueError), linear.rmsnorm_quantize_dev, T, T, bad, 1, 64, T)
refused(TypeError, linear.linear_forward_dev, 8, T, T, 1.0, 32, d_acts=T)
""")


def test_the_library_loads_without_the_extension():
    """Host-slice calls and the ABI need ctypes alone; the device entry points say what is missing."""
    run(r"""
import sys
capi._attached = None
sys.modules["oxillama_amd._bind"] = None  # importing it raises ImportError
import oxillama_amd
del oxillama_amd._bind
assert capi.load().oxq_block_size(8) == 32
assert quant.KernelDispatcher().get_kernel(8).block_bytes() == 34
refused(RuntimeError, quant.quantize_q8_0_dev, T, T)
refused(RuntimeError, capi.bind)
""")
