"""Producers fused into the activation quantizer of a Quartet linear.

In the model the quantized linears sit in (src/models/llama.py of the reference) two of the four linears of a block are
fed by RMSNorm (``c_attn(ln_1(x))``, ``w12(ln_2(x))``, llama.py:170-171) and one by the SwiGLU product
(``c_proj(silu(up) * gate)``, llama.py:113-114).  ``rmsnorm_linear`` and ``swiglu_linear`` compute the same results
without writing the normalised tensor / the product: the quantizer kernel builds each group of 32 values in registers,
the layer consumes the packed operand, and the backward pass recomputes what it needs from the producer's inputs (the
autograd functions are native, csrc/host_ext.cpp).

Both fall back to the unfused composition (same mathematics, more memory traffic) when the layer is not in its
production configuration, uses another Hadamard block than 32, or the tensors are not what the kernels take."""
import torch
import torch.nn.functional as F

from . import _lib, kernels, one_node
from .linear import _GLOBAL_HOOKS, QuantizedLinear, _cached_weight, _dense, _watched
from .one_node import as_one_node

_KERNEL_DTYPES = (torch.float32, torch.bfloat16)


def _fusable_parts(layer, x):
    """(weight, activation, weight and gradient quantizer) of a layer whose input a kernel here may produce, else None."""
    parts = layer._production_parts(x) if isinstance(layer, QuantizedLinear) else None
    if parts is None:
        return None
    weight, a_q = parts[:2]
    return parts if weight.is_cuda and a_q.hadamard_dim == 32 and a_q._dense is None and weight.dtype in _KERNEL_DTYPES else None


@as_one_node
def _rope(qkv, table, n_head):
    return _lib.host().rope_qkv(qkv, table, n_head)


@as_one_node
def _norm_linear(x, add, gain, weight, eps, a_q, w_q, g_q, cache, pass_input):
    key, packed_w = _cached_weight(x, weight, a_q, w_q, g_q, cache)
    y, x_next, packed_w = _lib.host().norm_linear(x, add, gain, weight, eps, a_q.sign_bits, w_q.hadamard_dim, w_q.sign_bits, g_q.hadamard_dim, g_q,
                                                  packed_w, _dense(w_q, weight), pass_input)
    if key is not None:
        cache.put(key, packed_w)
    return (y, x_next) if (pass_input or add is not None) else y


@as_one_node
def _swiglu_linear(h12, weight, a_q, w_q, g_q, cache):
    key, packed_w = _cached_weight(h12, weight, a_q, w_q, g_q, cache)
    y, packed_w = _lib.host().swiglu_linear(h12, weight, a_q.sign_bits, w_q.hadamard_dim, w_q.sign_bits, g_q.hadamard_dim, g_q, packed_w,
                                            _dense(w_q, weight))
    if key is not None:
        cache.put(key, packed_w)
    return y


def rope_qkv(qkv, table, n_head):
    """Split the fused attention projection [B, T, 3C] into q, k, v [B, T, n_head, head_dim] with q and k rotated by the
    (cos, sin) table [T, head_dim/2, 2]."""
    C = qkv.shape[-1] // 3
    hs = C // n_head
    if qkv.is_cuda and qkv.dtype in _KERNEL_DTYPES and hs % 8 == 0 and table.dtype == torch.float32:
        return _rope(qkv, table.contiguous(), n_head)
    from .llama import apply_rotary
    B, T, _ = qkv.shape
    q, k, v = qkv.split(C, dim=2)
    q, k = apply_rotary(q.view(B, T, n_head, hs), k.view(B, T, n_head, hs), table)
    return q, k, v.view(B, T, n_head, hs)


def rmsnorm_linear(norm, layer, x, pass_input=False, add=None):
    """layer(norm(x)) for an RMSNorm module `norm` (attributes ``weight`` and ``eps``) and a QuantizedLinear.  With
    `pass_input` returns (layer(norm(x)), x): use the second value for the residual sum around the norm, so that the sum
    of x's two gradients happens inside the RMSNorm backward kernel.  With `add` returns (layer(norm(x + add)), x + add):
    the residual sum in front of the norm is formed inside the quantizer kernel."""
    parts = _fusable_parts(layer, x)
    fusable = parts is not None and x.is_cuda and x.dtype in _KERNEL_DTYPES
    gain = norm.weight if fusable else None   # in front of any other layer `norm` need not have one
    fusable = fusable and gain.dtype == torch.float32 and x.shape[-1] <= 8192
    if fusable and add is not None and not (x.dtype == torch.float32 and add.dtype in _KERNEL_DTYPES and add.shape == x.shape):
        x, add = x + add, None
        pass_input = True
    if fusable:
        weight, *quantizers = parts
        return _norm_linear(x, add, gain, weight, norm.eps, *quantizers, layer.packed_weight_cache, pass_input)
    if add is not None:
        x = x + add
    y = layer(norm(x))
    return (y, x) if (pass_input or add is not None) else y


def swiglu_linear(layer, h12):
    """layer(silu(up) * gate) with (up, gate) the two halves of h12's last dimension."""
    parts = _fusable_parts(layer, h12)
    if parts is not None and h12.is_cuda and h12.dtype in _KERNEL_DTYPES:
        return _swiglu_linear(h12, *parts, layer.packed_weight_cache)
    up, gate = h12.split(h12.shape[-1] // 2, dim=-1)
    return layer(F.silu(up) * gate)


def _evaluated(norm, layers, x, add):
    """[(weight, its packed form, activation and weight quantizer)] of the layers behind an RMSNorm where nothing asks for a gradient, the
    products are bf16 ones under autocast of more than 64 tokens (up to which the products in question are others), and every weight's packed form is kept
    and up to date; else None."""
    if not (x.is_cuda and x.numel() > 64 * x.shape[-1] and torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16) or one_node.transformed() or torch.compiler.is_compiling():
        return None
    gain = getattr(norm, "weight", None)
    tensors = [x, gain] if add is None else [x, gain, add]
    if not (isinstance(gain, torch.Tensor) and gain.dtype == torch.float32 and x.dtype in _KERNEL_DTYPES and 0 < x.shape[-1] <= 8192 and 0 < x.numel() < 1 << 27):
        return None
    if add is not None and not (x.dtype == torch.float32 and add.dtype in _KERNEL_DTYPES and add.shape == x.shape):
        return None
    if any(t.device != x.device for t in tensors):
        return None
    found = []
    for layer in layers:
        parts = _fusable_parts(layer, x)
        if parts is None or layer.packed_weight_cache is None or parts[0].device != x.device:
            return None
        weight, a_q, w_q, g_q = parts
        if w_q._dense is not None:
            return None
        key, _ = _cached_weight(x, weight, a_q, w_q, g_q, _KEY_ONLY)
        if layer.packed_weight_cache.key != key:
            return None
        found.append((weight, layer.packed_weight_cache, a_q, w_q))
        tensors.append(weight)
    if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
        return None
    return found


class _KeyOnly:
    @staticmethod
    def get(key):
        return None


_KEY_ONLY = _KeyOnly()


def rmsnorm_swiglu_linear(norm, w12, c_proj, x, add=None):
    """(c_proj(silu(up) * gate), x [+ add]) with (up, gate) = w12(norm(x [+ add])): ``rmsnorm_linear`` and ``swiglu_linear``.  In an
    evaluation under bf16 autocast with packed weights kept, w12's product goes on to the SwiGLU and the quantizer in its epilogue and
    its result is never written; the same bits."""
    parts = _evaluated(norm, (w12, c_proj), x, add)
    if parts is not None and w12.out_features == 2 * c_proj.in_features:
        (w, cache, a_q, _), (w2, cache2, a_q2, w_q2) = parts
        out = _lib.host().norm_swiglu_linear(x, add, norm.weight, norm.eps, w, cache.buffer, a_q.sign_bits, w2, cache2.buffer, a_q2.sign_bits, w_q2.hadamard_dim,
                                             w_q2.sign_bits)
        if out is not None:
            cache.hits += 1
            cache2.hits += 1
            return out
    h12, x = rmsnorm_linear(norm, w12, x, pass_input=True, add=add)
    return swiglu_linear(c_proj, h12), x


def rmsnorm_rope_linear(norm, c_attn, x, table, n_head, add=None):
    """(q, k, v, x [+ add]): ``rmsnorm_linear`` and ``rope_qkv``, in an evaluation as ``rmsnorm_swiglu_linear`` with the split and the rotary
    embedding in c_attn's epilogue."""
    parts = _evaluated(norm, (c_attn,), x, add)
    if parts is not None and table.dtype == torch.float32 and c_attn.out_features % (3 * n_head) == 0:
        (w, cache, a_q, _), = parts
        out = _lib.host().norm_rope_linear(x, add, norm.weight, norm.eps, w, cache.buffer, a_q.sign_bits, table, n_head)
        if out is not None:
            cache.hits += 1
            return out
    qkv, x = rmsnorm_linear(norm, c_attn, x, pass_input=True, add=add)
    return (*rope_qkv(qkv, table, n_head), x)


def _plain_rows(norm, layer, x, add):
    """[x, add] as rows, of an RMSNorm module in front of a plain nn.Linear under bf16 autocast that nobody watches, where nothing asks for the norm's
    gradient and a kernel here takes the tensors; else None."""
    if not (type(layer) is torch.nn.Linear and not _watched(layer) and type(x) is torch.Tensor and x.is_cuda and x.dtype == torch.float32 and torch.is_autocast_enabled("cuda")
            and torch.get_autocast_dtype("cuda") == torch.bfloat16 and not (one_node.transformed() or torch.compiler.is_compiling())):
        return None
    from .llama import RMSNorm
    if type(norm) is not RMSNorm or any(_GLOBAL_HOOKS) or _watched(norm):
        return None
    gain, cols = norm.weight, x.shape[-1]
    watched = torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, add, gain))
    if (watched or gain.dtype != torch.float32 or gain.shape != (cols,) or gain.device != x.device or not 0 < cols <= 4096
            or cols % 4 or not 0 < x.numel() < 1 << 31
            or not (add is None or (type(add) is torch.Tensor and add.dtype in _KERNEL_DTYPES and add.shape == x.shape and add.device == x.device))):
        return None
    rows = [t if t is None else t.reshape(-1, cols).contiguous() for t in (x, add)]
    return None if any(t is not None and t.data_ptr() % 16 for t in (*rows, gain)) else rows


def rmsnorm(norm, layer, x, add=None):
    """norm(x [+ add]) in front of `layer`.  Where that is a plain nn.Linear, in an evaluation under bf16 autocast in one pass, rounded to the
    bf16 that autocast hands the layer."""
    rows = _plain_rows(norm, layer, x, add)
    if rows is not None:
        return kernels.rmsnorm(rows[0], norm.weight.contiguous(), norm.eps, rows[1], torch.bfloat16).view(x.shape)
    return norm(x if add is None else x + add)


def _one_pass(T, K, V):
    """Whether logits_and_loss() makes the logits of T tokens x K x V classes and their loss in one pass, which saves the loss's own pass over the logits and
    24 us of a call's host time (44 instead of 68; 36 where the library rounds the weight, too) but rounds the whole weight to bf16 on every call; the library does
    that once per autocast region.  Longer contractions the library multiplies faster by more than the pass costs.

    A weight that takes no longer to round than that (3 * 2^23 elements, 20 us): any number of tokens.  us a pass of an evaluated model of six layers, 32000
    classes, in one pass and apart, batch after batch in one region: 640 wide 64 tokens 657 and 711, 1024 604 and 666, 2048 623 and 677, 4096 791 and 818; 768 wide 64 tokens 640 and
    703, 1024 594 and 654, 4096 873 and 865, 8192 1473 and 1512; but 1536 wide 1024 tokens 782 and 725, 4096 1807 and 1766.  A region for each batch: 768 wide 4096 tokens 879 and 914, 1536
    wide 791 and 786.  (Replayed from a graph, where host time is nothing, 64 tokens of 640 take 300 and 293, 512 475 and 480, 4096 793 and 838.)
    Larger weights, up to 2^26 elements: enough tokens for the pass to cost more than the rounding.  us on the GPU, the library's weight rounded before: 1024 tokens x 384 x
    128000 198 and 190, 2048 320 and 385; 2048 x 640 x 64000 220 and 214, 4096 378 and 406; 4096 x 768 x 64000 438 and 446; past that 4096 x 640 x 128000 904 and 822, 8192 1680 and 1663."""
    return K <= 768 and V * K <= 1 << 26 and (V * K <= 3 << 23 or T >= 6 * K)


def logits_and_loss(norm, layer, x, add, targets, ignore_index=-1):
    """(layer(norm(x [+ add])), its cross-entropy against `targets`): ``rmsnorm``, a plain nn.Linear without bias and ``cross_entropy``, in an evaluation
    under bf16 autocast with the loss's sums of exponentials worked out beside the logits."""
    weight = layer.weight if type(layer) is torch.nn.Linear and layer.bias is None else None
    if (type(weight) is torch.nn.Parameter and type(targets) is torch.Tensor and targets.dtype == torch.int64 and targets.shape == x.shape[:-1] and targets.is_contiguous()
            and weight.dtype == torch.float32 and weight.device == x.device == targets.device and weight.dim() == 2 and weight.shape[1] == x.shape[-1]
            and _one_pass(targets.numel(), weight.shape[1], weight.shape[0]) and weight.is_contiguous() and weight.data_ptr() % 16 == 0 and not (torch.is_grad_enabled() and weight.requires_grad)):
        rows = _plain_rows(norm, layer, x, add)
        if rows is not None:
            out = kernels.logits_loss(rows[0], norm.weight.contiguous(), norm.eps, rows[1], weight.detach(), targets.view(-1), ignore_index)
            if out is not None:
                return out[0].view(*x.shape[:-1], -1), out[1]
    logits = layer(rmsnorm(norm, layer, x, add))
    return logits, cross_entropy(logits.view(-1, logits.size(-1)), targets.view(-1), ignore_index=ignore_index)


def cross_entropy(logits, targets, ignore_index=-1):
    """F.cross_entropy(logits, targets, ignore_index=ignore_index) of logits [rows, classes].  Where nothing asks for a
    gradient and the result is an fp32 one (fp32 logits, or bf16 ones under autocast) the logits are read once by a kernel of
    this package, which keeps log-probabilities in fp32 (the library rounds them to the logits' type).  A target that is
    neither a class nor `ignore_index` is an error of the caller that the device cannot raise: the kernel makes the loss NaN."""
    plain = (type(logits) is torch.Tensor and logits.is_cuda and not (torch.is_grad_enabled() and logits.requires_grad)
             and not (one_node.transformed() or torch.compiler.is_compiling()))
    if (plain and (logits.dtype == torch.float32 or (logits.dtype == torch.bfloat16 and torch.is_autocast_enabled("cuda")))
            and logits.dim() == 2 and logits.shape[1] > 0 and targets.dim() == 1 and targets.dtype == torch.int64
            and targets.device == logits.device and targets.shape[0] == logits.shape[0]):
        return kernels.cross_entropy(logits.contiguous(), targets.contiguous(), ignore_index)
    return F.cross_entropy(logits, targets, ignore_index=ignore_index)
