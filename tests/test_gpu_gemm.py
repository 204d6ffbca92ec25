"""GPU parity of the bf16 GEMM x . w^T (the vLLM layer's x_ext = x . w_ext^T).

Reference: the same bf16 operands multiplied in fp32 by torch, rounded once to
bf16.  The kernel accumulates in fp32 in another order, so an element may land
one bf16 step away from the reference's rounding: tolerance 2^-7 relative plus
1e-5 absolute, far inside the 2e-2 bf16 parity bound.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from granite_switch_amd import switched

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _check(got, x, w):
    ref = (x.float() @ w.float().T)
    err = (got.float() - ref).abs()
    bad = err > 2.0 ** -7 * ref.abs() + 1e-5
    assert not bool(bad.any()), f"{int(bad.sum())} elements off, max abs err {float(err.max()):.3e}"


REGISTER, PINGPONG, STREAM = 0, 1, 2


def _form(M, N, K, cus=256, ld=None):
    """(kernel, its tile -- or the ping-pong form's tile rows of 256 and of 128) of a call on ``cus`` compute units."""
    out = (ctypes.c_int32 * 3)()
    assert switched._lib.load().gs_gemm_form(M, N, K, ld or K, ld or K, cus, out) == 0
    return tuple(out)


@pytest.mark.parametrize("M,N,K,seed", [
    (1, 32, 8, 1),              # one row, one partial tile, K below one k-tile
    (7, 300, 72, 2),            # ragged everything, K not a multiple of 64
    (256, 256, 64, 3),          # exactly one tile
    (513, 777, 520, 4),         # partial tiles on both sides
    (300, 7296, 4096, 5),       # decode-sized QKV w_ext (base 6144 + 12 adapters x 3 slices x 32)
    (2048, 4864, 12800, 6),     # down_proj w_ext shape at a prefill chunk
])
def test_gemm_matches_fp32_reference(dev, M, N, K, seed):
    _say(f"gemm M={M} N={N} K={K}")
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device=dev) / K ** 0.5).to(torch.bfloat16)
    got = switched.linear_bf16(x, w)
    torch.cuda.synchronize()
    _check(got, x, w)


@pytest.mark.parametrize("M,N,K,halves", [
    (256, 256, 128, 2),          # the two k-tiles that the direct-to-LDS form's stages hold
    (128, 264, 192, 1),          # a full tile row; an odd number of k-tiles
    (385, 520, 256, 4),          # the last tile row of one row
    (384, 1032, 320, 3),         # full tile rows over four tile columns and a partial one
    (2049, 775, 128, 17),        # columns that end inside an 8-column store
    (300, 301, 256, 3),          # rows of C that are not 16-byte aligned
    (1, 33, 64, 1), (300, 7296, 64, 3), (1025, 257, 64, 9), (128, 264, 64, 1),   # one k-tile
    (777, 7296, 256, 7), (1100, 6001, 192, 9), (129, 300, 128, 2),
])
def test_gemm_pingpong_128_row_tiles(dev, M, N, K, halves):
    assert _form(M, N, K) == (PINGPONG, 0, halves)
    test_gemm_matches_fp32_reference(dev, M, N, K, M + N)


@pytest.mark.parametrize("M,N,K,full,halves", [
    # 256-row tiles alone, the last of 8 rows (its second half past M) and of 200
    (4104, 256, 128, 17, 0), (4104, 250, 64, 17, 0), (4104, 250, 192, 17, 0), (4296, 256, 128, 17, 0),
    (4296, 250, 320, 17, 0), (4360, 512, 64, 18, 0),
    # then 128-row ones that level out the last round: a ragged last row, ragged columns
    (4144, 4864, 128, 13, 7), (2500, 8450, 192, 7, 6), (3333, 6150, 128, 10, 7), (700, 30001, 64, 2, 2),
])
def test_gemm_pingpong_256_row_tiles(dev, M, N, K, full, halves):
    assert _form(M, N, K) == (PINGPONG, full, halves)
    test_gemm_matches_fp32_reference(dev, M, N, K, M + N + K)


@pytest.mark.parametrize("M,N,K,tile", [
    # streaming forms, K from the fewest chunks a wave may have to uneven shares of them; ragged rows and columns
    (1, 33, 1088, (16, 32)), (7, 4480, 4096, (16, 32)), (16, 45, 1024, (16, 32)),
    (32, 7296, 1088, (32, 32)), (27, 9001, 768, (32, 32)),
    (64, 7296, 1024, (64, 32)), (49, 8003, 576, (64, 32)),
    (128, 7296, 576, (64, 64)), (300, 6149, 832, (64, 64)),
    (113, 16000, 512, (128, 64)), (70, 14989, 1344, (128, 64)), (256, 7296, 512, (128, 64)), (255, 7290, 1152, (128, 64)),
])
def test_gemm_streaming_forms(dev, M, N, K, tile):
    assert _form(M, N, K) == (STREAM, *tile)
    test_gemm_matches_fp32_reference(dev, M, N, K, M + N + K)


@pytest.mark.parametrize("M,N,K", [(333, 520, 1024), (200, 9000, 640), (900, 7000, 320)])
def test_gemm_strided_rows_and_output(dev, M, N, K):
    """x and out with row strides (a view into a wider buffer), as the layer's x_ext slices are."""
    g = torch.Generator(device=dev).manual_seed(11)
    xb = torch.randn(M, K + 64, generator=g, device=dev).to(torch.bfloat16)
    x = xb[:, 32:32 + K]
    w = (torch.randn(N, K, generator=g, device=dev) / K ** 0.5).to(torch.bfloat16)
    outb = torch.full((M, N + 40), 7.0, dtype=torch.bfloat16, device=dev)
    out = outb[:, :N]
    switched.linear_bf16(x, w, out)
    torch.cuda.synchronize()
    _check(out, x, w)
    assert bool((outb[:, N:] == 7.0).all()), "columns past N were written"


def test_gemm_empty_and_graph(dev):
    g = torch.Generator(device=dev).manual_seed(12)
    w = torch.randn(64, 128, generator=g, device=dev).to(torch.bfloat16)
    assert switched.linear_bf16(torch.empty(0, 128, dtype=torch.bfloat16, device=dev), w).shape == (0, 64)
    x = torch.randn(300, 128, generator=g, device=dev).to(torch.bfloat16)
    out = torch.empty(300, 64, dtype=torch.bfloat16, device=dev)
    eager = switched.linear_bf16(x, w).clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        switched.linear_bf16(x, w, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def test_vllm_layer_native_and_library_gemm_agree(dev):
    """The vLLM layer's x_ext GEMM through this library's kernel and through torch.mm."""
    from granite_switch_amd import vllm_layers

    K, slices, ranks, T = 1024, (2048, 512, 512), [32, 16, 64], 200
    g = torch.Generator(device=dev).manual_seed(21)
    base = torch.nn.Linear(K, sum(slices), bias=False).to(device=dev, dtype=torch.bfloat16)
    with torch.no_grad():
        base.weight.copy_(torch.randn(sum(slices), K, generator=g, device=dev) / K ** 0.5)
    layer = vllm_layers.SwitchedLoRALinear(base, len(ranks), max(ranks), num_slices=3, output_slices=slices)
    with torch.no_grad():
        for s in range(3):
            for a, r in enumerate(ranks):
                layer.lora_A_slices[s].data[a, 0, :r] = (torch.randn(r, K, generator=g, device=dev) / K ** 0.5).to(torch.bfloat16)
    layer.finalize_weights(ranks)
    x = torch.randn(T, K, generator=g, device=dev).to(torch.bfloat16)
    layer.native_gemm = True
    native = layer._gemm(x)
    layer.native_gemm = False
    library = layer._gemm(x)
    torch.cuda.synchronize()
    assert native.shape == library.shape == (T, layer.w_ext.shape[0])
    _check(native, x, layer.w_ext)
    d = (native.float() - library.float()).abs()
    assert bool((d <= 2.0 ** -7 * library.float().abs() + 1e-5).all())
