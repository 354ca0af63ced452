"""Row bookkeeping of the fused silu quantizer: used rows are dealt out over the launch from prefix sums of the experts' row
counts, unused rows are written as zeros.  Sizes at which that can go wrong: one expert and as many as one scan takes and one
more, no used row at all, row counts outside [0, T], both forms of the kernel (table in LDS or not), a ragged last word."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,T,H,counts", [
    (1, 3, 128, "full"), (1, 1, 384, "none"), (3, 5, 640, "wild"), (257, 2, 128, "random"), (1024, 1, 128, "random"),
    (1025, 2, 128, "random"), (16, 640, 2048, "random"), (2, 4200, 2048, "last")])
def test_zero_rest(gpu, oracle, E, T, H, counts):
    from sglang_amd.fp8_kernel import per_token_group_quant_8bit

    g = torch.Generator().manual_seed(E * 7 + T)
    x = torch.randn(E, T, 2 * H, generator=g).to(torch.bfloat16)
    m = {"full": [T] * E, "none": [0] * E, "wild": [-4, T + 9, 2], "last": [0] * (E - 1) + [T],
         "random": torch.randint(0, T + 1, (E,), generator=g).tolist()}[counts]
    print(f"case E={E} T={T} H={H} {counts}", flush=True)
    q, s = per_token_group_quant_8bit(x.to(gpu), 128, torch.float8_e4m3fn, column_major_scales=True, scale_tma_aligned=True,
                                      scale_ue8m0=True, fuse_silu_and_mul=True, masked_m=torch.tensor(m, dtype=torch.int32, device=gpu))
    used = torch.arange(T)[None, :] < torch.tensor(m).clamp(0, T)[:, None]
    want_q = torch.zeros(E, T, H, dtype=torch.uint8)
    want_s = torch.zeros(E, T, -(-H // 512) * 4, dtype=torch.uint8)
    if bool(used.any()):
        v = oracle.silu_mul(x[used].contiguous())
        q_o, s_o = oracle.group_quant(v, 128, mode="mul", layout="ue8m0")
        want_q[used] = q_o.view(torch.uint8)
        full = torch.zeros(v.shape[0], want_s.shape[2], dtype=torch.uint8)
        full[:, :H // 128] = oracle.unpack_ue8m0(s_o, H // 128)
        want_s[used] = full
    assert torch.equal(q.cpu().view(torch.uint8), want_q)
    words = torch.empty(tuple(s.shape), dtype=torch.int32)
    words.copy_(s.cpu())
    assert torch.equal(words.view(torch.uint8).reshape(want_s.shape), want_s)
