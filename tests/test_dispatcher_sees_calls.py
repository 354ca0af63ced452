"""The native fast paths launch kernels without PyTorch's dispatcher, so they have to stand back wherever somebody looks on
through it: `torch.compile` and export (whose tracer cannot follow a C function), dispatch and function modes, `make_fx`,
`torch.jit.trace` and functional transforms.  Tracing needs no GPU: the operators have fake implementations."""
import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from sglang_amd import _native, fp8_kernel, fp8_utils, sgl_kernel

FP8 = torch.float8_e4m3fn


def _group_quant(x, **options):
    return fp8_kernel.sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True, scale_tma_aligned=True, **options)


def _silu_quant(x):
    return fp8_kernel.per_token_group_quant_8bit(x, 128, FP8, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True,
                                                 fuse_silu_and_mul=True)


def _sgl_kernel_quant(x):
    q, s = torch.empty_like(x, dtype=FP8), torch.empty(x.shape[0], x.shape[1] // 128, device=x.device)
    sgl_kernel.sgl_per_token_group_quant_8bit(x, q, s, 128, 1e-10, -448.0, 448.0)
    return q, s


def _token_linear(x):
    w = torch.zeros(256, x.shape[1], device=x.device, dtype=FP8).t()
    return fp8_utils.apply_fp8_linear(x, w, torch.ones(256, 1, device=x.device), use_per_token_if_dynamic=True)


CALLS = {"group_quant": (_group_quant, "sgl_per_token_group_quant_8bit"), "silu_quant": (_silu_quant, "sgl_per_token_group_quant_8bit_v2"),
         "sgl_kernel_quant": (_sgl_kernel_quant, "sgl_per_token_group_quant_8bit"), "token_linear": (_token_linear, "fp8_scaled_mm")}


@pytest.mark.parametrize("name", CALLS)
def test_compile_sees_the_operators(name):
    """torch.compile(fullgraph=True): one graph that holds the operator.  (Running it needs the GPU.)"""
    fn, op = CALLS[name]
    graphs = []

    def backend(gm, inputs):
        graphs.append(gm)
        return gm.forward

    torch._dynamo.reset()
    with pytest.raises(NotImplementedError, match="sgl_kernel"):  # the operators have no CPU kernel
        torch.compile(fn, fullgraph=True, backend=backend)(torch.ones(8, 512, dtype=torch.bfloat16))
    assert len(graphs) == 1
    assert any(getattr(torch.ops.sgl_kernel, op).default is n.target for n in graphs[0].graph.nodes)


@pytest.mark.parametrize("value,v2", [("1", True), ("true", True), ("0", False)])
def test_v2_by_environment_is_the_same_traced(monkeypatch, value, v2):
    monkeypatch.setenv("SGLANG_PER_TOKEN_GROUP_QUANT_8BIT_V2", value)
    assert sgl_kernel._v2_by_environment() is v2
    torch._dynamo.reset()
    traced = torch.compile(lambda x: x + 1 if sgl_kernel._v2_by_environment() else x, fullgraph=True, backend="eager")
    assert float(traced(torch.zeros(1))) == float(v2)


class _SeesFunctions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _SeesOperators(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(func)
        return func(*args, **(kwargs or {}))


def test_fast_paths_stand_back_where_somebody_looks():
    x = torch.ones(4, 128)
    answers = []
    look = lambda t: (answers.append(_native.plain_dispatch(t)), t * 1)[1]
    plain = [x, x.clone().requires_grad_(True), torch.nn.Parameter(x)]
    for t in plain:
        look(t)
    with torch.inference_mode():
        look(torch.ones(3)), look(x)
    with torch.autocast("cpu", torch.bfloat16):
        look(x)
    assert answers == [True] * 6
    answers.clear()
    with _SeesFunctions():
        look(x)
    with _SeesOperators():
        look(x)
    torch.func.vmap(look)(x)
    torch.func.grad(lambda t: look(t).sum())(x)
    torch.func.jvp(look, (x,), (x,))
    torch.func.functionalize(look)(x)
    torch.jit.trace(look, (x,), check_trace=False)
    make_fx(look)(x)
    look(torch.view_as_complex(torch.ones(2, 2)).conj()), look(torch.ones(2, device="meta"))
    assert len(answers) == 10 and not any(answers[:-1])


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["group_quant", "silu_quant", "sgl_kernel_quant"])
def test_gpu_modes_and_tracers_see_the_kernels(gpu, name):
    """A dispatch mode sees the quantizer's operator, a graph of `make_fx` holds it, with the plain call's result, and computes it
    for other inputs too."""
    fn, op = CALLS[name]
    print(f"case {name}", flush=True)
    op = getattr(torch.ops.sgl_kernel, op)
    data = lambda seed: torch.randn(8, 512, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(gpu)
    same = lambda a, b: all(torch.equal(p.float(), q.float()) for p, q in zip(a, b))
    x, y = data(1), data(2)
    want, other = fn(x), fn(y)
    with _SeesOperators() as mode:
        got = fn(x)
    assert op.default in mode.seen and same(got, want)
    graph = make_fx(fn, tracing_mode="real")(x)
    assert any(n.target is op.default for n in graph.graph.nodes)
    assert same(graph(x), want) and same(graph(y), other)
