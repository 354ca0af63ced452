"""The tables of the fused silu quantizer: every finite gate value on each side of the sizes where another table serves them, and
rows whose lanes mix gates inside and outside the magnitudes that a workgroup of the bfloat16 form keeps in LDS."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,T,mixed", [
    (torch.bfloat16, 512, True), (torch.bfloat16, 49152, False), (torch.bfloat16, 49153, True),
    (torch.float16, 12288, False), (torch.float16, 12289, True)])
def test_every_gate_value_of_each_table(gpu, oracle, dtype, T, mixed):
    from sglang_amd.fp8_kernel import sglang_per_token_group_quant_fp8

    H = 128
    gate = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).clone()
    gate[~torch.isfinite(gate.float())] = 0
    if mixed:
        gate = gate[torch.randperm(65536, generator=torch.Generator().manual_seed(T))]
    x = torch.empty(T, 2 * H, dtype=dtype)
    x[:, :H] = gate.repeat(-(-T * H // 65536))[:T * H].view(T, H)
    x[:, H:] = 1.5
    print(f"case {dtype} T={T}", flush=True)
    q, s = sglang_per_token_group_quant_fp8(x.to(gpu), 128, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True,
                                            fuse_silu_and_mul=True, enable_v2=True)
    q_o, s_o = oracle.group_quant(oracle.silu_mul(x), 128, mode="mul", layout="ue8m0")
    assert torch.equal(q.cpu().view(torch.uint8), q_o.view(torch.uint8))
    dense = torch.empty(tuple(s.shape), dtype=torch.int32)
    dense.copy_(s.cpu())
    assert torch.equal(dense.view(torch.uint8).reshape(T, -1)[:, :1], oracle.unpack_ue8m0(s_o, 1))
