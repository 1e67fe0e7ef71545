"""Python mirror of the callers of the kernel trait, over liboxq_hip.so.

  LoraAdapter      crates/oxillama-quant/src/lora.rs:21-124
  QuantLinear      crates/oxillama-arch/src/common/linear.rs:20-132
  swiglu / rmsnorm crates/oxillama-arch/src/common/swiglu.rs:15-21, rms_norm.rs:49-66
  dense FFN        crates/oxillama-arch/src/llama/model.rs:277-310

`QuantLinear.forward` crosses the C ABI with numpy host buffers (everything staged per call);
the `*_dev` functions take torch CUDA tensors and enqueue on torch's current stream.
"""
import ctypes as C

import numpy as np

from . import capi
from .quant import DimensionMismatch, HipKernel, QuantTensor, _check, _ptr, _u8, raw_stream as _stream

_U8, _F32 = np.dtype(np.uint8), np.dtype(np.float32)


def _plain(a, dtype):
    """An array whose memory can be handed over as it is."""
    return type(a) is np.ndarray and a.dtype == dtype and a.ndim == 1 and a.flags.c_contiguous


def _f32(a):
    return a if _plain(a, _F32) else np.ascontiguousarray(a, dtype=np.float32).ravel()


class LoraAdapter:
    """delta = B @ (A @ input) * scale; A is [rank x in_features], B is [out_features x rank]."""

    def __init__(self, a, b, rank, scale, in_features, out_features):
        a = np.ascontiguousarray(a, dtype=np.float32).ravel()
        b = np.ascontiguousarray(b, dtype=np.float32).ravel()
        if a.size != rank * in_features:  # lora.rs:51-57
            raise DimensionMismatch(rank * in_features, a.size)
        if b.size != out_features * rank:  # lora.rs:58-64
            raise DimensionMismatch(out_features * rank, b.size)
        self.a, self.b, self.rank, self.scale = a, b, rank, float(scale)
        self.in_features, self.out_features = in_features, out_features


class QuantLinear:
    """weight: QuantTensor [out_features, in_features]; optional fp32 bias; optional LoRA."""

    def __init__(self, weight: QuantTensor, bias=None):
        self.weight = weight
        self.bias = None if bias is None else np.ascontiguousarray(bias, dtype=np.float32).ravel()
        self.out_features = weight.shape[0] if len(weight.shape) > 0 else 0  # linear.rs:38-48
        self.in_features = weight.shape[1] if len(weight.shape) > 1 else 0
        self.lora = None
        self._shape = self._view = None

    def _weight_args(self):
        """(address, bytes, shape, dimensions, array behind the address) of the weight for the C ABI, from the tensor as it
        is now.  Kept from call to call: the ctypes form of a shape, by its values, and the address of an array that is a
        view (QuantTensor makes one), which stays where it is; an array with memory of its own may move on resize()."""
        w, shape = self.weight.data, tuple(self.weight.shape)
        if not _plain(w, _U8):
            w = _u8(w)
        if self._shape is None or self._shape[0] != shape:
            self._shape = (shape, (C.c_size_t * len(shape))(*shape))
        view = self._view
        if view is None or view[0] is not w:
            view = (w, _ptr(w))
            self._view = None if w.flags.owndata or w is not self.weight.data else view
        return view[1], w.size, self._shape[1], len(shape), w

    def set_lora(self, lora):
        self.lora = lora

    def clear_lora(self):
        self.lora = None

    def forward(self, kernel: HipKernel, input, output):
        """output = weight @ input + bias [+ lora delta] (linear.rs:77-98); output is filled in place."""
        lib = capi.load()
        x = _f32(input)
        bias_p, bias_n = (_ptr(self.bias), self.bias.size) if self.bias is not None else (None, 0)
        if self.lora is not None:
            la, lb = self.lora.a, self.lora.b
            lora_args = (_ptr(la), la.size, _ptr(lb), lb.size, self.lora.rank, self.lora.scale)
        else:
            lora_args = (None, 0, None, 0, 0, 0.0)
        w_p, w_n, shape, n_dims, _array = self._weight_args()
        _check(lib.oxq_linear_forward(kernel.tensor_type, w_p, w_n, shape, n_dims, bias_p, bias_n, *lora_args, _ptr(x), x.size,
                                      _ptr(output), output.size))

    def forward_batch(self, kernel: HipKernel, input, output, batch_size):
        """output[batch x out] = gemm + bias broadcast (linear.rs:105-132; no LoRA in batch mode)."""
        lib = capi.load()
        x = _f32(input)
        bias_p, bias_n = (_ptr(self.bias), self.bias.size) if self.bias is not None else (None, 0)
        w_p, w_n, shape, n_dims, _array = self._weight_args()
        _check(lib.oxq_linear_forward_batch(kernel.tensor_type, w_p, w_n, shape, n_dims, bias_p, bias_n, _ptr(x), x.size,
                                            _ptr(output), output.size, batch_size))


# ---- device route -------------------------------------------------------------------------


class LoraStruct(C.Structure):
    _fields_ = [("d_a", C.c_void_p), ("d_b", C.c_void_p), ("d_r", C.c_void_p), ("rank", C.c_size_t),
                ("scale", C.c_float)]


def lora_struct(d_a, d_b, d_r, rank, scale):
    return LoraStruct(d_a.data_ptr(), d_b.data_ptr(), d_r.data_ptr(), rank, scale)


def lora_apply_dev(lora, d_x, d_out, out_features, in_features):
    _check(capi.load().oxq_lora_apply_dev(C.byref(lora), d_x.data_ptr(), d_out.data_ptr(), out_features, in_features,
                                          _stream()))


def linear_forward_dev(tensor_type, d_weights, d_out, out_features, in_features, d_x=None, d_acts=None, d_bias=None,
                       lora=None):
    _check(capi.bind().linear_forward(tensor_type, d_weights, d_x, d_acts, d_bias, C.addressof(lora) if lora is not None else None,
                                      d_out, out_features, in_features))


def linear_forward_multi_dev(tensor_type, d_weights, d_acts, d_outs, out_features, in_features, d_biases=None):
    _check(capi.bind().linear_forward_multi(tensor_type, d_weights, d_acts, d_biases, d_outs, out_features, in_features))


def linear_forward_batch_dev(tensor_type, d_weights, d_acts, d_out, batch, out_features, in_features, d_bias=None,
                             workspace=None):
    _check(capi.bind().linear_forward_batch(tensor_type, d_weights, d_acts, d_bias, d_out, batch, out_features, in_features, workspace))


def swiglu_quantize_dev(d_gate, d_up, d_h=None, d_out_q8=None):
    _check(capi.bind().swiglu_quantize(d_gate, d_up, d_h, d_out_q8))


def rmsnorm_quantize_dev(d_x, d_weight, eps, rows, n, d_y=None, d_out_q8=None):
    _check(capi.bind().rmsnorm_quantize(d_x, d_weight, eps, rows, n, d_y, d_out_q8))


def gate_up_swiglu_dev(tensor_type, d_gate, d_up, d_acts_q8, d_h, d_out_q8, intermediate, hidden):
    """ffn_gate + ffn_up + SwiGLU + Q8_0 quantizer of h in one launch (d_h optional)."""
    _check(capi.load().oxq_ffn_gate_up_swiglu_q8_dev(int(tensor_type), d_gate.data_ptr(), d_up.data_ptr(),
                                                     d_acts_q8.data_ptr(), d_h.data_ptr() if d_h is not None else None,
                                                     d_out_q8.data_ptr(), intermediate, hidden, _stream()))


def ffn_workspace_bytes(hidden, intermediate):
    return capi.load().oxq_ffn_workspace_bytes(hidden, intermediate)


def ffn_swiglu_dev(gate, up, down, d_acts, d_out, hidden, intermediate, workspace):
    """gate/up/down: (tensor_type, device weights).  d_out = down(silu(gate x) * up x)."""
    _check(capi.bind().ffn_swiglu(gate[0], gate[1], up[0], up[1], down[0], down[1], d_acts, d_out, hidden, intermediate, workspace))


def topk_dev(d_values, k, d_out_values, d_out_indices, workspace):
    """The k largest of a float32 CUDA tensor, largest first, with their indices (uint32 viewed as int32)."""
    _check(capi.bind().topk(d_values, k, d_out_values, d_out_indices, workspace))


def lm_head_topk_workspace_bytes(quant_type, n_rows, n_cols, k):
    return capi.load().oxq_lm_head_topk_workspace_bytes(quant_type, n_rows, n_cols, k)


def lm_head_topk_dev(quant_type, d_weights, d_acts_q8, d_logits, n_rows, n_cols, k, d_out_values, d_out_indices, workspace):
    """The vocabulary projection (logits to d_logits) and the k largest logits with their row indices, in one launch
    where the shape allows it (oxq_lm_head_topk_dev)."""
    _check(capi.bind().lm_head_topk(quant_type, d_weights, d_acts_q8, d_logits, n_rows, n_cols, k, d_out_values, d_out_indices,
                                    workspace))


def logits_edit_dev(d_logits, d_banned=None, d_bias_tokens=None, d_bias_values=None, d_recent=None, window=0,
                    repetition_penalty=1.0):
    """The sampler's edits of the logits before the candidate list (sampling/mod.rs:573-613), in place: banned tokens,
    logit bias, repetition penalty over the last `window` of d_recent.  Token lists: int32 / uint32 CUDA tensors."""
    _check(capi.bind().logits_edit(d_logits, d_banned, d_bias_tokens, d_bias_values, d_recent, window, repetition_penalty))


def sample_candidates_dev(d_values, d_indices, k, temperature, min_p, top_p, d_rng_state, d_token, d_probs=None):
    """The sampler after its candidate list (sampling/mod.rs:487-564): temperature, softmax, min-p, top-p, the draw.
    d_rng_state: one uint64 (the reference's Xorshift64 state), d_token: one uint32, d_probs: optional k floats."""
    _check(capi.bind().sample_candidates(d_values, d_indices, k, temperature, min_p, top_p, d_rng_state, d_token, d_probs))


def topk_workspace_bytes(n, k):
    return capi.load().oxq_topk_workspace_bytes(n, k)
