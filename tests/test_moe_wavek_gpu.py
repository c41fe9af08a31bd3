"""The grouped GEMM of few 16-slot blocks whose workgroups cut K between their waves: exact on integer data."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,top_k,N,K", [((1,), 1, 8, 1024), ((1, 0, 3, 16, 17), 1, 264, 1152), ((5, 1, 1, 1), 4, 512, 7168), ((2, 1, 1), 2, 1032, 4096),
                                             ((40, 1, 16, 15), 1, 2048, 2048), ((1, 1), 1, 4096, 18432),
                                             ((1,), 1, 8, 1152), ((1, 0, 3, 16, 17), 8, 264, 1152), ((40, 1, 16, 15), 16, 776, 4096), ((40, 1, 16, 15), 16, 1400, 4224)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_blocks_with_k_cut_between_waves_exact(dev, sizes, top_k, N, K, dtype):
    """One, two and four waves along n, a K that the waves do not divide, a last strip of 8 weight rows, blocks of one slot and full
    ones, an expert with several blocks and one without slots, slots of another rank's expert (stored as zeros), routed weights on and off, activation
    scales by row and by column.  Integers below 2^11 times powers of two, exact in float32 in any order of the sums.  K = 1024, 2048 weight
    rows and the first sizes with top_k = 1 and K = 1152 are past the lines of the rule: the kernel with tiles, the same results."""
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


def _table(blocks, pad, extra, dev):
    """sorted_token_ids, expert_ids and num_tokens_post_padded of (expert, slots) blocks of 16, with `extra` unused blocks behind them."""
    rows = [list(s) + [pad] * (16 - len(s)) for _, s in blocks] + [[pad] * 16] * extra
    return (torch.tensor(rows, dtype=torch.int32, device=dev).flatten(), torch.tensor([e for e, _ in blocks] + [0] * extra, dtype=torch.int32, device=dev),
            torch.tensor([16 * len(blocks)], dtype=torch.int32, device=dev))


# What the caller's table may hold beyond what an aligner over B's experts would write: more blocks than slots, or than those experts fill.
TABLES = {
    # aligned over 64 experts of all ranks, of which this rank has every eighth: one slot each, foreign blocks at -1
    "foreign_experts": (8, [(e // 8 if e % 8 == 3 else -1, [63 - e]) for e in range(64)]),
    # one block per expert whatever the routing (the layout of a captured graph), three of 24 with slots
    "fixed_blocks": (24, [(e, {3: [0, 1, 2], 17: [5], 23: [4, 3]}.get(e, [])) for e in range(24)]),
    # two experts in turn, every block part-filled
    "part_filled": (2, [(b % 2, [2 * b, 2 * b + 1]) for b in range(30)]),
}


@pytest.mark.parametrize("N,K", [(264, 4224), (1024, 1152), (776, 4096), (1032, 4224), (2056, 4224)])
@pytest.mark.parametrize("table", sorted(TABLES))
def test_tables_of_more_blocks_than_the_experts_fill(dev, table, N, K):
    """Every block below num_tokens_post_padded is computed, whatever its number; the rows of foreign blocks are zeros; exact on integers."""
    from sglang_amd.sgl_kernel import moe_block_gemm

    E, blocks = TABLES[table]
    slots = 1 + max(s for _, b in blocks for s in b)
    top_k = (slots + 3) // 4  # few tokens
    rows = (slots + top_k - 1) // top_k
    g = torch.Generator().manual_seed(N + K + E)
    powers = lambda *s: 2.0 ** torch.randint(-2, 2, s, generator=g).float()  # noqa: E731
    x, w = torch.randint(-1, 2, (rows, K), generator=g).float(), torch.randint(-1, 2, (E, N, K), generator=g).float()
    xs, ws = powers(rows, K // 128), powers(E, (N + 127) // 128, K // 128)
    want = torch.zeros((slots, N))
    for e, ids in blocks:
        if e >= 0 and ids:
            scaled = w[e] * ws[e].repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)
            at = torch.tensor(ids) // top_k
            want[ids] = (x[at] * xs[at].repeat_interleave(128, 1)) @ scaled.t()
    A, B = x.to(dev).to(torch.float8_e4m3fn), w.to(dev).to(torch.float8_e4m3fn)
    for extra in (0, 5):
        C = torch.full((slots, N), float("nan"), dtype=torch.bfloat16, device=dev)
        moe_block_gemm(A, B, C, xs.to(dev), ws.to(dev), None, *_table(blocks, slots, extra, dev), False, top_k, 16, slots)
        assert torch.equal(C.float().cpu(), want.to(torch.bfloat16).float())


@pytest.mark.parametrize("T,E,topk,N,K", [(1, 16, 4, 2048, 1024), (3, 8, 2, 1032, 1024), (2, 16, 4, 2048, 896), (1, 4, 1, 512, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_blocks_have_the_bits_of_the_form_with_the_activation_inside(dev, T, E, topk, N, K, dtype):
    """Whatever K fp8k_moe_act_block_gemm takes, the grouped GEMM adds its K blocks in the same order, also where few blocks are hit.  The
    largest terms cancel - the first K block against the last - so that another order shows in the 16-bit result."""
    from sglang_amd._lib import BF16, F16, check, lib, stream_ptr
    from sglang_amd.fp8_kernel import sglang_per_token_group_quant_fp8
    from sglang_amd.fused_moe import moe_align_block_size
    from sglang_amd.sgl_kernel import moe_block_gemm

    g = torch.Generator().manual_seed(K + T)
    x = torch.randn((T * topk, 2, K), generator=g)
    x[:, :, -128:] = x[:, :, :128]
    x = x.to(dtype).to(dev).view(T * topk, 2 * K)
    w = torch.randn((E, N, K), generator=g)
    w[:, :, -128:] = -w[:, :, :128]
    w = w.to(dev).to(torch.float8_e4m3fn)
    ws = torch.rand((E, (N + 127) // 128, K // 128), generator=g) + 0.5
    ws[:, :, -1] = ws[:, :, 0] = 1000.0
    ws = ws.to(dev)
    ids = torch.rand((T, E), generator=g).argsort(dim=1)[:, :topk].int().to(dev)
    sorted_ids, expert_ids, npad = moe_align_block_size(ids, 16, E)
    q, s = sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True, fuse_silu_and_mul=True)
    assert lib.fp8k_moe_act_block_gemm_takes(16, N, K, K) == 1
    want, got = (torch.full((T * topk, N), 7.0, dtype=dtype, device=dev) for _ in range(2))
    moe_block_gemm(q, w, want, s, ws, None, sorted_ids, expert_ids, npad, False, 1, 16, ids.numel())
    check(lib.fp8k_moe_act_block_gemm(x.data_ptr(), w.data_ptr(), ws.data_ptr(), got.data_ptr(), sorted_ids.data_ptr(), expert_ids.data_ptr(),
                                      npad.data_ptr(), None, sorted_ids.numel(), 16, ids.numel(), E, N, K, 2 * K, N * K, K, *ws.stride(), N, 1e-10,
                                      BF16 if dtype == torch.bfloat16 else F16, stream_ptr(dev)))
    torch.cuda.synchronize()
    assert torch.equal(want, got)
