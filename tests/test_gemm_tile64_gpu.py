"""GPU parity of the 64x64 tile kernel (gemm_tile64_kernel), pinned through fp8k_tune_force_gemm_plan: fewer K blocks than waves, remainders
of a round of four waves, rows and columns around the edges of a tile, K cuts, every mode, both scale layouts, biases, strided operand and
output rows in both store forms.
Integer data with power-of-two scales: the sums are exact whatever their order.
"""
import numpy as np
import pytest
import torch

from oracle import fp8_oracle as O
from tests.conftest import fp8_tensor
from tests.test_gemm_gpu import _run_block

pytestmark = pytest.mark.gpu

SHAPES = [(65, 8, 128), (64, 64, 256), (1, 72, 128 * 3), (128, 136, 128 * 4), (127, 200, 128 * 5), (129, 56, 128 * 9), (300, 520, 128 * 19),
          (95, 64, 128 * 33)]


@pytest.fixture
def tile64():
    from sglang_amd._lib import lib

    yield lambda splits: lib.fp8k_tune_force_gemm_plan(8, splits)
    lib.fp8k_tune_force_gemm_plan(-1, 0)


def _integers(M, N, K):
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    xq, wq = (O.f32_to_e4m3fn(rng.integers(-4, 5, (n, K)).astype(np.float32)) for n in (M, N))
    xs = (2.0 ** rng.integers(-3, 4, (M, K // 128))).astype(np.float32)
    ws = (2.0 ** rng.integers(-3, 4, ((N + 127) // 128, K // 128))).astype(np.float32)
    return rng, xq, wq, xs, ws


@pytest.mark.parametrize("splits", [1, 2, 3])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_block_is_exact_on_integers(dev, tile64, M, N, K, splits):
    _, xq, wq, xs, ws = _integers(M, N, K)
    tile64(splits)
    for col_major, dt, name in ((False, torch.bfloat16, "bf16"), (True, torch.float16, "f16")):
        ref = O.w8a8_block_fp8_matmul(xq, wq, xs, ws, out_dtype=name, acc=np.float64)
        np.testing.assert_array_equal(_run_block(xq, xs, wq, ws, dev, col_major_as=col_major, out_dtype=dt), ref)


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_row_scales_and_bias_are_exact_on_integers(dev, tile64, M, N, K, splits):
    from sglang_amd.sgl_kernel import fp8_scaled_mm

    rng, xq, wq, _, _ = _integers(M, N, K)
    sa, sb = ((2.0 ** rng.integers(-3, 3, (n,))).astype(np.float32) for n in (M, N))
    bias = rng.integers(-8, 9, (N,)).astype(np.float32)
    tile64(splits)
    got = fp8_scaled_mm(fp8_tensor(xq, dev), fp8_tensor(wq, dev).t(), torch.from_numpy(sa).to(dev), torch.from_numpy(sb).to(dev),
                        torch.bfloat16, torch.from_numpy(bias).to(dev)).float().cpu().numpy()
    np.testing.assert_array_equal(got, O.fp8_scaled_mm(xq, wq, sa, sb, out_dtype="bf16", bias=bias))


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("M,N,K", [(130, 72, 128 * 4), (129, 264, 128 * 9), (257, 200, 128 * 21)])
def test_hardware_scales_match_float_scales(dev, tile64, M, N, K, splits):
    """Packed UE8M0 activation scales, applied by the matrix core, against the float-scale form of the same kernel."""
    from sglang_amd import fp8_kernel

    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    x = torch.randint(-4, 5, (M, K), device=dev, generator=gen).to(torch.bfloat16)
    w = torch.randint(-4, 5, (N, K), device=dev, generator=gen).float().to(torch.float8_e4m3fn)
    ws = torch.exp2(torch.randint(-3, 4, ((N + 127) // 128, K // 128), device=dev, generator=gen).float())
    tile64(splits)
    outs = []
    for packed in (True, False):
        q, s = fp8_kernel.sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True, scale_tma_aligned=packed, scale_ue8m0=packed)
        if not packed:  # the same powers of two as floats
            amax = x.float().abs().view(M, -1, 128).amax(-1).clamp(min=1e-10)
            s = torch.exp2(torch.ceil(torch.log2(amax / 448.0)))
            q = (x.float().view(M, -1, 128) / s[..., None]).clamp(-448, 448).view(M, K).to(torch.float8_e4m3fn)
        outs.append(fp8_kernel.w8a8_block_fp8_matmul(q, w, s, ws, [128, 128], torch.bfloat16))
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("mode", ["block", "row"])
@pytest.mark.parametrize("dtype,code,name", [(torch.bfloat16, 2, "bf16"), (torch.float16, 1, "f16")])
def test_strided_rows_and_both_store_forms(dev, tile64, splits, mode, dtype, code, name):
    """Operand rows longer than K, output rows longer than N: rows of a multiple of eight elements from a 16-byte aligned start take
    16-byte stores, any other ldc or start the 8-byte ones; what lies between the rows stays as it was.  Exact on integers."""
    from sglang_amd._lib import check, lib, stream_ptr

    M, N, K = 131, 200, 128 * 9
    rng, xq, wq, xs, ws = _integers(M, N, K)
    sa, sb = ((2.0 ** rng.integers(-3, 3, (n,))).astype(np.float32) for n in (M, N))
    A, B = torch.zeros((M, K + 48), dtype=torch.uint8, device=dev), torch.zeros((N, K + 16), dtype=torch.uint8, device=dev)
    A[:, :K], B[:, :K] = torch.from_numpy(xq).to(dev).view(torch.uint8), torch.from_numpy(wq).to(dev).view(torch.uint8)
    if mode == "block":
        want = O.w8a8_block_fp8_matmul(xq, wq, xs, ws, out_dtype=name, acc=np.float64)
    else:
        want = O.fp8_scaled_mm(xq, wq, sa, sb, out_dtype=name)
    xs, ws, sa, sb = (torch.from_numpy(t).to(dev) for t in (xs, ws, sa, sb))
    tile64(splits)
    need = max(lib.fp8k_block_gemm_workspace_bytes(M, N, K), lib.fp8k_scaled_mm_workspace_bytes(M, N, K))
    work = torch.empty(max(need, 1), dtype=torch.uint8, device=dev)
    for ldc, start in ((N, 0), (N + 8, 0), (N + 4, 0), (N, 4), (N + 8, 4)):
        buf = torch.full((M * ldc + 8,), 7.0, dtype=dtype, device=dev)
        C = buf[start:start + M * ldc].view(M, ldc)
        if mode == "block":
            check(lib.fp8k_block_gemm(A.data_ptr(), B.data_ptr(), xs.data_ptr(), ws.data_ptr(), C.data_ptr(), M, N, K, K + 48, K + 16, xs.stride(0),
                                      xs.stride(1), ws.stride(0), ws.stride(1), ldc, code, work.data_ptr(), need, stream_ptr(dev)))
        else:
            check(lib.fp8k_scaled_mm(A.data_ptr(), B.data_ptr(), sa.data_ptr(), sb.data_ptr(), None, C.data_ptr(), M, N, K, K + 48, K + 16, ldc, code, 0,
                                     work.data_ptr(), need, stream_ptr(dev)))
        assert np.array_equal(C[:, :N].float().cpu().numpy(), want), (ldc, start)
        assert (C[:, N:] == 7.0).all() and (buf[:start] == 7.0).all() and (buf[start + M * ldc:] == 7.0).all(), (ldc, start)


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_block_linear_adds_its_bias_to_the_rounded_product(dev, tile64, splits, dtype):
    """Block mode's bias.  Every group's largest value is 448 times a power of two, so the quantisation is exact, and so are the sums."""
    from sglang_amd.fp8_utils import w8a8_block_fp8_linear

    M, N, K = 133, 136, 128 * 9
    rng, _, wq, _, ws = _integers(M, N, K)
    x = rng.integers(-4, 5, (M, K // 128, 128)).astype(np.float32)
    x[:, :, 5] = 448.0 * rng.choice([-1, 1], (M, K // 128))
    scale = (2.0 ** rng.integers(-3, 3, (M, K // 128))).astype(np.float32)
    bias = torch.from_numpy(rng.standard_normal(N).astype(np.float32) * 100).to(dtype)
    product = O.w8a8_block_fp8_matmul(O.f32_to_e4m3fn(x.reshape(M, K)), wq, scale, ws, out_dtype="f32", acc=np.float64)
    want = (torch.from_numpy(product).to(dtype).float() + bias.float()).to(dtype)
    tile64(splits)
    got = w8a8_block_fp8_linear(torch.from_numpy((x * scale[:, :, None]).reshape(M, K)).to(dtype).to(dev), fp8_tensor(wq, dev), [128, 128],
                                torch.from_numpy(ws).to(dev), bias=bias.to(dev))
    assert torch.equal(got.cpu(), want)
