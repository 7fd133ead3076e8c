"""The layers' native calls under callers that record what Python runs: each entry point against its plain call, on kernels
(tests/test_one_node.py holds the mechanism without a GPU)."""
import random

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")]
ENTRIES = ["layer", "error_only", "norm", "norm_add", "swiglu", "rope", "quest", "albert"]


class _Call(torch.nn.Module):
    """A function of one tensor, next to the modules whose parameters it reads (a trace takes them from here)."""

    def __init__(self, function, *modules):
        super().__init__()
        self.function, self.modules_read = function, torch.nn.ModuleList(modules)

    def forward(self, x):
        return self.function(x)


def _entry(name):
    """(call of a tensor, maker of its inputs from a seed)"""
    import quartet_amd as q
    from quartet_amd.fused import rmsnorm_linear, rope_qkv, swiglu_linear
    from quartet_amd.llama import RMSNorm, rotary_table
    dev = torch.device("cuda:0")
    torch.manual_seed(0)
    layer = q.QuantizedLinear(256, 384, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(), activation_quantizer=q.QuestMXFP4Quantizer(),
                              gradient_quantizer=q.AlbertTsengQuantizer(stochastic=True, rerotate="signs"),
                              backward_scheme=q.BACKWARD_SCHEMES["Q(E)W_Q(Et)X" if name == "error_only" else "Q(E)Q(Wt)t_Q(Et)Q(Xt)t"](),
                              device=dev, dtype=torch.bfloat16)

    def inputs(cols, dtype=torch.bfloat16):
        return lambda seed: torch.randn(64, cols, generator=torch.Generator(device=dev).manual_seed(seed), device=dev).to(dtype)
    if name in ("layer", "error_only"):
        return layer, inputs(256)
    if name == "norm":
        norm = RMSNorm(256).to(dev)
        return _Call(lambda x: rmsnorm_linear(norm, layer, x), norm, layer), inputs(256, torch.float32)
    if name == "norm_add":
        norm, add = RMSNorm(256).to(dev), inputs(256)(9)

        def both(x):
            y, s = rmsnorm_linear(norm, layer, x, add=add)
            return torch.cat([y.float().flatten(), s.flatten()])
        return _Call(both, norm, layer), inputs(256, torch.float32)
    if name == "swiglu":
        return _Call(lambda h: swiglu_linear(layer, h), layer), inputs(512)
    if name == "rope":
        table = rotary_table(32, 64).to(dev)
        return _Call(lambda x: torch.cat([t.flatten() for t in rope_qkv(x.view(1, 64, 192), table, 2)])), inputs(192, torch.float32)
    return (q.QuestMXFP4Quantizer() if name == "quest" else q.AlbertTsengQuantizer(stochastic=True)), inputs(256)


def _seeded():
    random.seed(4)
    torch.default_generator.manual_seed(4)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("name", ENTRIES)
def test_traced_calls_run_their_kernels_on_replay(name, grad):
    import quartet_amd as q
    call, make = _entry(name)
    q.enable_packed_weight_cache(call)      # a packed weight from before the trace is in place
    print(f"case trace {name} grad={grad}", flush=True)
    with torch.set_grad_enabled(grad):
        call(make(1))
        traced = torch.jit.trace(call, (make(1).requires_grad_(grad),), check_trace=False)
        for seed in (2, 3):
            results = []
            for f in (traced, call):
                _seeded()
                x = make(seed).requires_grad_(grad)
                y = f(x)
                if grad:
                    y.backward(torch.randn(y.shape, generator=torch.Generator(device=y.device).manual_seed(5), device=y.device).to(y.dtype))
                results.append((y.detach(), x.grad))
            assert torch.equal(results[0][0], results[1][0])
            assert not grad or torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("name", ENTRIES)
def test_tangents_and_transforms_are_refused(name):
    from torch.autograd import forward_ad
    call, make = _entry(name)
    print(f"case transforms {name}", flush=True)
    with torch.no_grad():
        with forward_ad.dual_level():
            with pytest.raises(NotImplementedError):
                call(forward_ad.make_dual(make(1), torch.ones_like(make(1))))
            _seeded()
            plain = call(make(1))
        _seeded()
        assert torch.equal(plain, call(make(1)))
        with pytest.raises(RuntimeError, match="functorch"):
            torch.func.vmap(call)(torch.stack([make(1), make(2)]))


def test_an_evaluated_model_refuses_tangents():
    from torch.autograd import forward_ad

    from quartet_amd.llama import Llama, LlamaConfig
    model = Llama(LlamaConfig(vocab_size=64, n_layer=1, n_head=2, n_embd=64, multiple_of=64, sequence_length=32)).cuda().eval()
    ids = torch.arange(32, device="cuda").view(1, 32)
    with torch.no_grad(), forward_ad.dual_level():
        weight = model.transformer.wte.weight
        with pytest.raises(NotImplementedError):
            torch.func.functional_call(model, {"transformer.wte.weight": forward_ad.make_dual(weight, torch.ones_like(weight))}, (ids,))
