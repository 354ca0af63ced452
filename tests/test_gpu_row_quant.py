"""Per-token quantizers at the steps of the launch rule (threads per row, vectors per thread, few and many rows) and the static
per-tensor quantizer at the steps of its: bit-exact against the oracle."""
import pytest
import torch

from sglang_amd.workloads import make_activation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 640, 641, 1025])
@pytest.mark.parametrize("K", [8, 512, 520, 2048, 2056, 4096, 4104, 8192, 8200, 16384, 16392, 24576, 24584])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_per_token(gpu, oracle, M, K, dtype):
    from sglang_amd.fp8_kernel import sglang_per_token_quant_fp8
    from sglang_amd.int8_kernel import per_token_quant_int8

    if M > 1 and K > 8200:
        M -= 600
    print(f"case M={M} K={K} {dtype}", flush=True)
    x = make_activation(M, K, seed=M + K, dtype=dtype)
    x[M // 2] = 0
    for quantize, reference in ((sglang_per_token_quant_fp8, oracle.per_token_quant_fp8), (per_token_quant_int8, oracle.per_token_quant_int8)):
        q, s = quantize(x.to(gpu))
        q_o, s_o = reference(x)
        assert torch.equal(q.cpu().view(torch.uint8), q_o.view(torch.uint8)) and torch.equal(s.cpu().view(-1), s_o.view(-1))


@pytest.mark.parametrize("M,K", [(1, 8), (3, 1000), (41, 7168), (512, 8192), (513, 8192), (700, 8200)])
def test_static_per_tensor(gpu, oracle, M, K):
    from sglang_amd.fp8_kernel import static_quant_fp8

    x = make_activation(M, K, seed=M + K)
    scale = torch.tensor([0.037])
    q, s = static_quant_fp8(x.to(gpu), scale.to(gpu), repeat_scale=True)
    assert torch.equal(q.cpu().view(torch.uint8), oracle.per_tensor_quant_fp8(x, scale)[0].view(torch.uint8))
    assert torch.equal(s.cpu(), scale.repeat(M, 1))
