"""The grouped GEMM of few 16-slot blocks whose workgroups cut K between their waves: exact on integer data."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,top_k,N,K", [((1,), 1, 8, 1024), ((1, 0, 3, 16, 17), 1, 264, 1152), ((5, 1, 1, 1), 4, 512, 7168), ((2, 1, 1), 2, 1032, 4096),
                                             ((40, 1, 16, 15), 1, 2048, 2048), ((1, 1), 1, 4096, 18432)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_blocks_with_k_cut_between_waves_exact(dev, sizes, top_k, N, K, dtype):
    """One, two and four waves along n, a K that the waves do not divide, a last strip of 8 weight rows, blocks of one slot and full
    ones, an expert with several blocks and one without slots, slots of another rank's expert (stored as zeros), routed weights on and off, activation
    scales by row and by column.  Integers below 2^11 times powers of two, exact in float32 in any order of the sums."""
    from sglang_amd.fused_moe import moe_align_block_size
    from sglang_amd.sgl_kernel import moe_block_gemm

    g = torch.Generator().manual_seed(N + K)
    E = len(sizes)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(sizes)])
    ids = torch.cat([ids, torch.full((-ids.numel() % top_k + top_k,), -1)])
    slots = ids.numel()
    ids = ids[torch.randperm(slots, generator=g)].int()
    powers = lambda *s: 2.0 ** torch.randint(-2, 2, s, generator=g).float()  # noqa: E731
    rows, nb, kb = slots // top_k, (N + 127) // 128, K // 128
    x, w = torch.randint(-1, 2, (rows, K), generator=g).float(), torch.randint(-1, 2, (E, N, K), generator=g).float()
    xs, ws, tw = powers(rows, kb), powers(E, nb, kb), powers(slots, 1)
    sorted_ids, expert_ids, npad = moe_align_block_size(ids.view(-1, top_k).to(dev), 16, E)
    A, B, wsd, twd = x.to(dev).to(torch.float8_e4m3fn), w.to(dev).to(torch.float8_e4m3fn), ws.to(dev), tw.to(dev)
    want = torch.zeros((slots, N))
    for e in range(E):
        at = (ids == e).nonzero().flatten()
        scaled = w[e] * ws[e].repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)
        want[at] = (x[at // top_k] * xs[at // top_k].repeat_interleave(128, 1)) @ scaled.t()
    for sc in (xs.to(dev), xs.t().contiguous().to(dev).t()):
        for weigh in (False, True):
            C = torch.full((slots, N), float("nan"), dtype=dtype, device=dev)
            moe_block_gemm(A, B, C, sc, wsd, twd, sorted_ids, expert_ids, npad, weigh, top_k, 16, slots)
            assert torch.equal(C.float().cpu(), (want * tw if weigh else want).to(dtype).float())
