"""Which kernels calls run, read from a trace of their launches: the choices whose reasons stand beside the rules of capi.hip."""
import re

import pytest
import torch

import triton_amd
from util import set_knob

pytestmark = pytest.mark.gpu


def launches(call):
    """[(kernel, its numeric template arguments)] of a call's launches."""
    call()   # (the first one sets attributes)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as trace:
        call()
        torch.cuda.synchronize()
    found = []
    for event in trace.events():
        kernel = re.search(r"mi355.*?(?<![a-z_])([a-z][a-z0-9_]*_kernel)", event.name)
        if kernel is None:
            continue
        rest = event.name[kernel.end():]
        numbers = re.findall(r"L[ib](\d+)E", rest) if event.name.startswith("_Z") else re.findall(r"\b(\d+|true|false)\b", rest.rsplit(">(", 1)[0])
        found.append((kernel.group(1), tuple({"true": 1, "false": 0}.get(n) if n in ("true", "false") else int(n) for n in numbers)))
    assert found, [event.name for event in trace.events()]
    return found


def whole(gpu, *shape):
    return torch.randint(-1, 2, shape, device=gpu, generator=torch.Generator(device=gpu).manual_seed(sum(shape)))


def product(gpu, dtype, M, N, K, kmajor, add=False):
    """The launches of a product of whole numbers, which has to be exact."""
    tdt = {"bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn}[dtype]
    a, b = whole(gpu, M, K).to(tdt), (whole(gpu, N, K) if kmajor else whole(gpu, K, N)).to(tdt)
    bt, row, got = b.t() if kmajor else b, whole(gpu, N).to(torch.bfloat16) if add else None, []
    names = launches(lambda: got.append(triton_amd.matmul(a, bt, out_dtype=torch.bfloat16, **({"add": row} if add else {}))))
    want = a.float() @ bt.float()
    want = (want + row.float() if add else want).bfloat16()
    assert all(torch.equal(c, want) for c in got)
    return names


def two_stages(names):
    # (template arguments of the ring kernels: the operands' type, then BM, BN, WN, K-major B, stages, rows on dwords)
    return [numbers[-6:-3] + numbers[-2:-1] for name, numbers in names if name == "gemm_ring_kernel"] == [(128, 128, 2, 2)]


@pytest.mark.parametrize("dtype,M,N,K,kmajor,ring", [
    ("e4m3", 2560, 3712, 64, True, False), ("e4m3", 2432, 3456, 192, True, False), ("e4m3", 4096, 1664, 320, True, False), ("e4m3", 3200, 2176, 128, True, False),
    ("bf16", 2944, 3456, 32, False, False), ("bf16", 1950, 4480, 64, False, False), ("bf16", 2304, 2432, 32, True, False),
    ("e4m3", 2432, 3456, 256, True, True), ("bf16", 2304, 2432, 128, True, True), ("bf16", 1642, 3586, 128, True, True)])
def test_half_filled_steps_of_a_short_k_stay_on_the_kernel_of_64_byte_steps(gpu, dtype, M, N, K, kmajor, ring):
    names = product(gpu, dtype, M, N, K, kmajor)
    assert two_stages(names) if ring else [name for name, _ in names] == ["gemm_kernel"], names


@pytest.mark.parametrize("dtype,M,N,K,ring", [("e4m3", 1344, 6144, 2944, False), ("e4m3", 4782, 1792, 2944, False), ("bf16", 2304, 3648, 384, False), ("bf16", 3085, 2804, 704, False),
                                              ("e4m3", 1536, 4224, 640, True), ("bf16", 3456, 1664, 256, True)])
def test_two_stage_rings_are_taken_where_they_gain(gpu, dtype, M, N, K, ring):
    assert two_stages(product(gpu, dtype, M, N, K, True)) == ring


@pytest.mark.parametrize("M,N,K,kmajor,copied", [
    (2154, 5428, 6548, True, True), (7454, 2496, 4234, True, True), (4390, 1838, 1838, False, True), (7258, 1110, 120, False, False),
    (1024, 1030, 1026, True, False), (771, 2608, 1460, True, False), (1646, 6920, 214, True, False), (4095, 4100, 4100, False, False)])
def test_rows_on_dwords_are_copied_where_that_is_shorter(gpu, M, N, K, kmajor, copied):
    assert any(name == "repack_kernel" for name, _ in product(gpu, "bf16", M, N, K, kmajor)) == copied


@pytest.mark.parametrize("tile", [8, 9, 10, 13])
@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("M,N,K", [(256, 258, 8), (130, 254, 46)])
def test_a_tile_that_is_asked_for_runs_rows_on_dwords_of_any_k(gpu, monkeypatch, tile, kmajor, M, N, K):
    set_knob(monkeypatch, "MI355_GEMM_TILE", tile)
    K -= K % 4   # (46: 44, no whole chunks)
    assert [name for name, _ in product(gpu, "bf16", M, N, K, kmajor, add=True)] == ["gemm_ring_kernel"]


def attention_launches(gpu, dtype, H, N, D, backward):
    g = torch.Generator(device=gpu).manual_seed(N)
    q, k, v = (torch.randn(1, H, N, D, device=gpu, generator=g).half().requires_grad_(backward) for _ in range(3))
    if dtype == "e5m2":
        q, k, v = (t.to(torch.float8_e5m2) for t in (q, k, v))
        v = v.view(torch.uint8).permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2).view(torch.float8_e5m2)
    if not backward:
        return dict(launches(lambda: triton_amd.attention(q, k, v, True, D ** -0.5)))
    o = triton_amd.attention(q, k, v, True, D ** -0.5)
    return dict(launches(lambda: torch.autograd.grad(o, (q, k, v), o.detach(), retain_graph=True)))


# groups in dQ and in dK/dV, the last template argument of either
@pytest.mark.parametrize("H,N,D,groups", [(8, 5248, 64, (2, 2)), (16, 2560, 64, (2, 2)), (16, 4096, 64, (2, 1)), (24, 1536, 64, (2, 1)), (36, 1024, 64, (2, 1)), (24, 4096, 64, (1, 1)),
                                          (6, 5504, 128, (2, 2)), (13, 2560, 128, (2, 2)), (18, 2048, 128, (1, 1)), (12, 3328, 128, (1, 1))])
def test_groups_of_the_backward_beyond_one_round_of_cus(gpu, H, N, D, groups):
    names = attention_launches(gpu, "fp16", H, N, D, True)
    assert (names["attn_bwd_dq_kernel"][-1], names["attn_bwd_dkdv_kernel"][-1]) == groups


@pytest.mark.parametrize("H,N,D", [(216, 896, 128), (60, 1024, 128), (154, 1280, 128), (54, 768, 128)])
def test_short_causal_heads_of_128_columns_run_on_blocks_of_128_rows(gpu, H, N, D):
    name, numbers = list(attention_launches(gpu, "fp16", H, N, D, False).items())[0]
    assert name == "attn_fwd_kernel" and numbers == (D, 1, 4, 0, 1)   # (D, tiles and waves, padded, groups)


@pytest.mark.parametrize("H,N,groups", [(40, 512, 2), (24, 768, 2), (24, 1024, 2), (16, 1536, 2), (16, 1024, 4), (4, 6144, 4)])
def test_groups_of_the_fp8_forward_in_short_heads(gpu, H, N, groups):
    name, numbers = list(attention_launches(gpu, "e5m2", H, N, 64, False).items())[0]
    assert name == "attn_fwd8_kernel" and numbers[-1] == groups
