"""The grouped GEMM of a short K that keeps the activations in registers: against the sums themselves on integer data."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,N,K", [((257, 600, 0, 1, 128, 255, 129, 1000, 31, 33), 128, 256), ((900, 90, 33), 8192, 256),
                                       ((256, 300, 97), 2048 + 128, 384), ((700, 130, 64, 1), 1152, 512), ((30000,), 256, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_short_k_with_activations_in_registers_exact(dev, sizes, N, K, dtype):
    """Every K depth, one weight tile and runs of several (a number that the runs do not divide), blocks with one slot, with one wave's
    and with all but one, parts without any, an expert without slots, slots of another rank's expert (stored as zeros), balanced
    blocks and not, routed weights on and off.  The float32 sums are exact, so the result is theirs rounded once."""
    from sglang_amd.fused_moe import moe_align_block_size
    from sglang_amd.sgl_kernel import moe_balance_blocks, moe_block_gemm, moe_sort_scales

    g = torch.Generator().manual_seed(N + K)
    E = len(sizes)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(sizes)] + [torch.full((40,), -1)])
    slots = ids.numel()
    ids = ids[torch.randperm(slots, generator=g)].int()
    assert slots >= 192 * E
    powers = lambda *s: 2.0 ** torch.randint(-2, 2, s, generator=g).float()  # noqa: E731
    x = torch.randint(-1, 2, (slots, K), generator=g).float()
    w = torch.randint(-1, 2, (E, N, K), generator=g).float()
    # one power of two per row and per weight block row: the K blocks of a sum share it, and the sum stays an integer multiple
    xs, ws = powers(slots, 1).expand(slots, K // 128).contiguous(), powers(E, N // 128, 1).expand(E, N // 128, K // 128).contiguous()
    tw = powers(slots, 1)
    sorted_ids, expert_ids, npad = moe_align_block_size(ids.view(-1, 1).to(dev), 256, E)
    A, B, wsd, twd = x.to(dev).to(torch.float8_e4m3fn), w.to(dev).to(torch.float8_e4m3fn), ws.to(dev), tw.to(dev)
    want = torch.zeros((slots, N))
    for e in range(E):
        at = (ids == e).nonzero().flatten()
        want[at] = (x[at] @ w[e].t()) * xs[at, :1] * ws[e, :, 0].repeat_interleave(128)
    for balanced in (False, True):
        if balanced:
            sorted_ids = moe_balance_blocks(sorted_ids, expert_ids, npad, 256, slots, E)
        sc = moe_sort_scales(xs.to(dev), sorted_ids, npad, 1, slots)
        for weigh in (True, False):
            C = torch.full((slots, N), float("nan"), dtype=dtype, device=dev)
            moe_block_gemm(A, B, C, sc, wsd, twd, sorted_ids, expert_ids, npad, weigh, 1, 256, slots, scales_sorted=True, balanced=balanced)
            ref = want * tw if weigh else want
            assert torch.equal(C.float().cpu(), ref.to(dtype).float())
