"""QuantizedLinear (API of the reference's src/models/quantization/__init__.py:11-42) and the fused
packed-MXFP4 autograd Function behind its production configuration.

Production configuration (main_setup.sh:77-93 of the reference): QuestMXFP4Quantizer on weights and
activations, AlbertTsengQuantizer on gradients, scheme "Q(E)Q(Wt)t_Q(Et)Q(Xt)t".  For it the layer
never materialises de-quantized tensors: operands stay packed (E2M1 codes + E8M0 scales + mask
bits, the tensors notebooks/benchmark_mxfp4.ipynb's CudaGemm saves) and the three products run on
the block-scaled FP4 MFMA.  The scheme that quantizes only the error signal ("Q(E)W_Q(Et)X") runs on the same packed
operands where its products are bf16 ones.  Any other mix of quantizers/schemes takes the generic path through the
quantizer modules and library GEMMs, as the reference does."""
import torch
import torch.nn as nn

from . import _lib, one_node
from .backward import BACKWARD_SCHEMES, EW_EtX_Scheme, QEQWtt_QEtQXtt_Scheme, QEW_QEtX_Scheme  # noqa: F401
from .quantizers import QUANTIZER_CLASSES, AlbertTsengQuantizer, NoQuantizer, QuestMXFP4Quantizer  # noqa: F401
from .quantizers.mxfp4 import _autocast_bf16, _fresh_seed


_SEED_BASE = None


def set_device_seed_base(tensor):
    """A one-element int64 tensor on the GPU (or None to switch this off) whose value the gradient quantizers of every
    packed-path layer add to their seeds when their kernels run.  The reference draws a fresh host seed per stochastic
    quantization (mxfp4_triton.py:196-199); a training step replayed from a captured HIP graph would repeat the seeds
    drawn at capture time, so capture the step with a seed base set and let the graph increment the tensor (any
    in-place add recorded in the graph): every replay then rounds with fresh random streams.  The sign flips drawn at
    capture time stay as they are.  Applies to layers on the tiled layout (tokens, in- and out-features multiples of
    128, Hadamard blocks 32, no dense rotation); a stochastic layer outside it raises while a seed base is set, since
    its replays would repeat their random streams."""
    global _SEED_BASE
    if tensor is not None and not (tensor.is_cuda and tensor.dtype == torch.int64 and tensor.numel() >= 1):
        raise ValueError("the seed base must be an int64 tensor on the GPU")
    _SEED_BASE = tensor


def _gradient_draws(g_q, seed_base_ok, T, I, O):
    """What the backward pass of one layer draws on the host, called by it once: fresh column signs, then one seed per
    stochastic quantization in the order e, W^T, e^T, x^T.  Returns (column signs, seeds, stochastic, dense rotation or
    None, device seed base or None)."""
    g_q.re_randomize()
    stochastic, dense = g_q.stochastic, g_q._dense is not None
    seeds = (_fresh_seed(), _fresh_seed(), _fresh_seed(), _fresh_seed()) if stochastic else (0, 0, 0, 0)
    base = _SEED_BASE if stochastic else None
    if base is not None and (dense or not seed_base_ok):
        # the device seed base is read by the pair launches of the tiled layout only: on any other path a captured replay
        # would silently repeat this launch's random streams
        raise _lib.QuartetHipError(
            f"a device seed base is set (set_device_seed_base), but this layer (tokens {T}, in {I}, out {O}"
            f"{', dense gradient rotation' if dense else ''}) does not run on the tiled layout, whose kernels are the "
            "only ones that read it (every extent a multiple of 128 and >= 256, Hadamard blocks 32, no dense rotation); "
            "clear the seed base or change the layer")
    return g_q.sign_bits, seeds, stochastic, g_q._dense, base


def _error_draws(g_q, e):
    """The same for the error-only scheme: no fresh column signs, one seed for e and one for e^T.  Returns (column signs,
    seeds, stochastic)."""
    g_q._note_input(e)
    seeds = (_fresh_seed(), _fresh_seed()) if g_q.stochastic else (0, 0)
    return g_q.sign_bits, seeds, g_q.stochastic


def _cached_weight(x, weight, a_q, w_q, g_q, weight_cache):
    """(cache key, packed Q(W) or None): Q(W) of an unchanged weight (the micro-steps of one accumulation) is quantized
    once and kept by the layer.  The last three entries of the key stand for the code layout, which csrc/host_ext.cpp picks."""
    if weight_cache is None:
        return None, None
    dense = a_q._dense is not None or w_q._dense is not None
    shape, n = weight.shape, x.numel()
    key = (weight.data_ptr(), weight._version, weight.dtype, shape, w_q.hadamard_dim, w_q.sign_bits,
           None if w_q._dense is None else w_q._dense_epoch, dense and n // x.shape[-1] % 128 == 0, n >= 1 << 28 and n >= shape[1] << 23)
    return key, weight_cache.get(key)


def _dense(quantizer, weight):
    """The dense rotation of a forward quantizer (rerotate="O32") on the weight's device, or None."""
    return None if quantizer._dense is None else quantizer.dense_matrix(weight.device)


class QuartetLinearFn:
    """y = Q(x) Q(W)^T with the fully quantized backward of backward.py:57-85, on packed operands.

    forward : F1/F2 quantize (quest RTN + mask) -> F3 FP4 GEMM
    backward: re-randomise signs; B1 Q(e); B2 Q(Q(W)^T); B3 GEMM -> grad wrt Q(x);
              B4 Q(e^T); B5 Q(Q(x)^T); B6 GEMM -> grad wrt Q(W);
              B7/B8 masked inverse rotation (straight-through estimators of F1/F2).
    error_only: the scheme of backward.py:21-45 instead -- no new signs, B1 Q(e), B4 Q(e^T), their products with the packed
    Q(W) and Q(x) as they are, B7/B8.
    The autograd function itself is native (csrc/host_ext.cpp)."""

    @staticmethod
    def apply(x, weight, a_q, w_q, g_q, weight_cache, error_only=False, inside=False):
        if not inside and one_node.transformed():   # here instead of by the decorator: a decoded batch feels 0.1 us
            return one_node.OneNode.apply(QuartetLinearFn.apply, x, weight, a_q, w_q, g_q, weight_cache, error_only, True)
        key, packed_w = _cached_weight(x, weight, a_q, w_q, g_q, weight_cache)
        y, packed_w = _lib.host().linear(x, weight, a_q.hadamard_dim, a_q.sign_bits, w_q.hadamard_dim, w_q.sign_bits, g_q.hadamard_dim, g_q,
                                         packed_w, _dense(a_q, weight), _dense(w_q, weight), error_only)
        if key is not None:
            weight_cache.put(key, packed_w)
        return y


_GLOBAL_HOOKS = (nn.modules.module._global_forward_hooks, nn.modules.module._global_forward_pre_hooks, nn.modules.module._global_backward_hooks,
                 nn.modules.module._global_backward_pre_hooks)


def _watched(module):
    """Whether calling `module` runs more than its class's forward: hooks, or a forward of its own."""
    return bool(module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks
                or "forward" in module.__dict__)


class PackedWeightCache:
    """The packed Q(W) of a layer's current weight, kept across the micro-steps of one gradient accumulation (the
    weight changes only at the optimizer step, src/optim/base.py:188-207 of the reference).  One entry, replaced --
    never overwritten in place, so that a graph built earlier keeps the buffer it saved -- when the weight's storage,
    version counter, rotation or code layout changes.  An update that bypasses the version counter (``weight.data``
    arithmetic) is invisible to the key: whoever steps the optimizer calls ``invalidate_packed_weights`` afterwards,
    as ``quartet_amd.train.train`` does, and the cache is off unless ``enable_packed_weight_cache`` turned it on."""

    def __init__(self):
        self.key, self.buffer, self.hits, self.misses = None, None, 0, 0

    def get(self, key):
        if key == self.key:
            self.hits += 1
            return self.buffer
        self.misses += 1
        return None

    def put(self, key, buffer):
        self.key, self.buffer = key, buffer

    def clear(self):
        self.key, self.buffer = None, None


def enable_packed_weight_cache(model, enabled=True):
    """Give every QuantizedLinear of `model` a PackedWeightCache (or remove it)."""
    for m in model.modules():
        if isinstance(m, QuantizedLinear):
            m.packed_weight_cache = PackedWeightCache() if enabled else None


def invalidate_packed_weights(model):
    """Forget every cached Q(W): call after anything that changes the weights (the optimizer step)."""
    for m in model.modules():
        if isinstance(m, QuantizedLinear) and m.packed_weight_cache is not None:
            m.packed_weight_cache.clear()


class QuantizedLinear(nn.Linear):
    """nn.Linear whose forward is scheme(act_q(x), weight_q(W)); the bias parameter, if requested,
    is never applied -- exactly as in the reference (the scheme calls F.linear(x, w, None)).

    A call's results can depend on how many tokens it has: on the packed path the product of at most 16 tokens, of 17 to 32
    where out_features <= 48 per compute unit (12288) or in_features <= 2048, and of 33 to 64 where out_features <= 32 per
    compute unit (8192), adds its terms in another order than that of more tokens.  FP4 codes times powers of two add up exactly in fp32 in any order as long as the
    group scales of a row span few octaves -- no result differed for normal, heavy-tailed and outlier-ridden activations --
    but with columns whose scales span 2^16 about one bf16 value in 3 * 10^4 rounds differently than the same row's in a
    larger batch, and behind a further quantizer such a difference can become another FP4 code.  Calls of one token count
    are reproducible bit for bit, with and without the packed-weight cache."""

    def __init__(self, in_features, out_features, weight_quantizer=None, activation_quantizer=None,
                 gradient_quantizer=None, backward_scheme=None, **kwargs):
        super().__init__(in_features, out_features, **kwargs)
        if weight_quantizer is None:
            weight_quantizer = NoQuantizer()
        if activation_quantizer is None:
            activation_quantizer = NoQuantizer()
        if gradient_quantizer is None:
            gradient_quantizer = NoQuantizer()
        if backward_scheme is None:
            backward_scheme = EW_EtX_Scheme()
        self.weight_quantizer = weight_quantizer
        self.activation_quantizer = activation_quantizer
        self.backward_scheme = backward_scheme
        self.backward_scheme.g_quantizer = gradient_quantizer
        self.use_packed_path = True
        self.packed_weight_cache = None  # see enable_packed_weight_cache

    def _is_production_config(self, tokens):
        modules = self._modules   # looked up once: nn.Module's attribute protocol costs more than the checks
        a_q, w_q, scheme = modules["activation_quantizer"], modules["weight_quantizer"], modules["backward_scheme"]
        g_q = scheme.g_quantizer
        if not (self.use_packed_path and type(a_q) is QuestMXFP4Quantizer and type(w_q) is QuestMXFP4Quantizer
                and type(g_q) is AlbertTsengQuantizer and type(scheme) is QEQWtt_QEtQXtt_Scheme):
            return False
        # A dense rotation (rerotate="O32") replaces a Hadamard block of 32 only in the kernels.  In the gradient quantizer
        # the packed path serves it when every extent is a multiple of 128; in a forward quantizer (the reference's loop
        # never re-randomises those) the dense quantizer kernel fills the packed operand and the straight-through
        # backward is a small library product.
        if (a_q._dense is not None and a_q.hadamard_dim != 32) or (w_q._dense is not None and w_q.hadamard_dim != 32):
            return False
        if g_q._dense is not None or g_q.rerotate == "O32":
            return g_q.hadamard_dim == 32 and not any(d % 128 for d in (tokens, self.in_features, self.out_features))
        return True

    def _production_parts(self, x):
        """(weight, activation, weight and gradient quantizer) where `_is_production_config` holds for x, else None.  Modules and
        parameters are looked up where they are kept: nn.Module's attribute protocol takes 0.25 us each time, of a decoded
        batch's 9."""
        modules = self._modules
        scheme = modules["backward_scheme"]
        if type(scheme) is not QEQWtt_QEtQXtt_Scheme:
            return None
        a_q, w_q, g_q = modules["activation_quantizer"], modules["weight_quantizer"], scheme._modules.get("g_quantizer")
        if g_q is None:
            g_q = scheme.g_quantizer
        if not (self.use_packed_path and type(a_q) is QuestMXFP4Quantizer and type(w_q) is QuestMXFP4Quantizer
                and type(g_q) is AlbertTsengQuantizer):
            return None
        # without dense rotations the configuration asks nothing of the tokens
        plain = a_q._dense is None and w_q._dense is None and g_q._dense is None and g_q.rerotate != "O32"
        if not plain and not self._is_production_config(x.numel() // max(x.shape[-1], 1)):
            return None
        # a subclass (a parametrization makes one) or the instance itself may have a weight of its own in front of the parameter
        weight = self._parameters.get("weight") if type(self) is QuantizedLinear and "weight" not in self.__dict__ else None
        return self.weight if weight is None else weight, a_q, w_q, g_q

    def _is_error_only_config(self, x):
        """The error-only scheme between the same quantizers, with products in bf16 (bf16 autocast, or bf16 tensors throughout)
        and extents below 2^23 that are multiples of 32 and of the Hadamard blocks."""
        modules = self._modules
        a_q, w_q, scheme = modules["activation_quantizer"], modules["weight_quantizer"], modules["backward_scheme"]
        g_q = scheme.g_quantizer
        if not (self.use_packed_path and type(scheme) is QEW_QEtX_Scheme and type(a_q) is QuestMXFP4Quantizer
                and type(w_q) is QuestMXFP4Quantizer and type(g_q) is AlbertTsengQuantizer):
            return False
        if a_q.is_dense or w_q.is_dense or g_q.is_dense:
            return False
        # this scheme calls its quantizers and itself as modules: where somebody listens, it still does
        if any(_GLOBAL_HOOKS) or _watched(a_q) or _watched(w_q) or _watched(g_q) or _watched(scheme):
            return False
        weight, out = self.weight, (torch.bfloat16, torch.float32)
        if not (x.is_cuda and weight.is_cuda and x.numel() and x.dtype in out and weight.dtype in out
                and (x.dtype == weight.dtype == torch.bfloat16 or _autocast_bf16())):
            return False
        O, I = weight.shape
        T = x.numel() // x.shape[-1]
        return not (x.shape[-1] != I or T % 32 or I % 32 or O % 32 or I % a_q.hadamard_dim or I % w_q.hadamard_dim
                    or T % g_q.hadamard_dim or O % g_q.hadamard_dim or max(T, I, O) >= 1 << 23)

    def forward(self, x):
        parts = self._production_parts(x)
        if parts is not None:
            return QuartetLinearFn.apply(x, *parts, self.packed_weight_cache)
        if self._is_error_only_config(x):
            a_q, w_q, g_q = self.activation_quantizer, self.weight_quantizer, self.backward_scheme.g_quantizer
            a_q._note_input(x)
            w_q._note_input(self.weight)
            return QuartetLinearFn.apply(x, self.weight, a_q, w_q, g_q, self.packed_weight_cache, True)
        xq = self.activation_quantizer(x)
        wq = self.weight_quantizer(self.weight)
        return self.backward_scheme(xq, wq)
