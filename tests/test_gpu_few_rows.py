"""The few-rows W4A16 kernel at the edges of its tiles: dense rows, grouped rows
by expert, and the expert block's gate_up and down stages."""
import numpy as np
import pytest
import torch

from gpu_util import bf16_normal, int4_words, layer, layer_dev, log, prod_interval, scales
from oracle import qmoe_oracle as O
from parity import assert_bf16_equal, assert_in_interval, assert_rounds_exactly, bits, to_dev


@pytest.mark.gpu
@pytest.mark.parametrize("M", [5, 16, 17, 48, 300])
@pytest.mark.parametrize("K,N,gs", [(64, 32, 32), (2048, 416, 128), (4096, 96, 64), (576, 8224, 96)])
def test_dense(device, M, K, N, gs):
    """Ragged rows and columns, fewer steps than waves, runs that cut scale
    groups, the largest K, both column widths; rows of very different size."""
    from qmoe import weight_quant_batchmatmul
    log(f"few rows dense M={M} K={K} N={N} gs={gs}")
    x = bf16_normal((M, K), M + K)
    x[0] = 0
    x[1] = O.f32_to_bf16_bits(O.bf16_bits_to_f32(x[1]) * np.float32(2.0 ** 90))
    x[2] = O.f32_to_bf16_bits(O.bf16_bits_to_f32(x[2]) * np.float32(2.0 ** -90))
    w, s = int4_words((K, N // 8), K + N), scales((K // gs, N), N + 1)
    y = weight_quant_batchmatmul(to_dev(x, device), to_dev(w, device), to_dev(s, device), antiquant_group_size=gs)
    torch.cuda.synchronize()
    assert_rounds_exactly(y, *O.w4a16_gemm_exact(x, w, s, gs), f"few rows M={M} K={K} N={N}")


@pytest.mark.gpu
@pytest.mark.parametrize("K,N,gs", [(512, 288, 64), (3072, 64, 128), (64, 1056, 32)])
def test_grouped(device, K, N, gs):
    """Tiles of 1 to 12 rows, experts of 12, 13, 24 and 25 rows, empty experts;
    a list short of the rows leaves the rest unwritten; and the tile size's
    rule at its line (five rows per expert)."""
    from qmoe import _lib, grouped_matmul
    counts = [0, 12, 13, 0, 24, 25, 1, 2] + [0] * 16
    E, R = len(counts), int(np.sum(counts)) + 3
    L = _lib.lib()
    assert L.qmoe_gemm_tile_rows_for(5 * E, E, K, N, gs) == 12 and L.qmoe_gemm_tile_rows_for(5 * E + 1, E, K, N, gs) == 32
    assert L.qmoe_gemm_tile_rows_for(20 * E, E, K, N, gs) == 32 and L.qmoe_gemm_tile_rows_for(20 * E + 1, E, K, N, gs) == 128
    log(f"few rows grouped K={K} N={N} gs={gs}")
    ends = np.cumsum(counts).astype(np.int64)
    x, w, s = bf16_normal((R, K), K), int4_words((E, K, N // 8), N), scales((E, K // gs, N), N + 2)
    y = grouped_matmul([to_dev(x, device)], [to_dev(w, device)], antiquant_scale=[to_dev(s, device)],
                       group_list=to_dev(ends, device), split_item=3, group_type=0)[0]
    torch.cuda.synchronize()
    n = int(ends[-1])
    assert_rounds_exactly(y[:n], *O.grouped_gemm_exact(x[:n], w, s, ends), f"few rows grouped K={K} N={N}")


@pytest.mark.gpu
@pytest.mark.parametrize("K,N,gs", [(64, 288, 64), (512, 64, 128), (320, 1056, 32)])
def test_grouped_mid(device, K, N, gs):
    """32-row tiles: experts of 15 to 65 rows, one K chunk, ragged columns."""
    from qmoe import grouped_matmul
    counts = [0, 15, 16, 17, 31, 32, 33, 64, 65] + [0] * 12
    E, R = len(counts), int(np.sum(counts))
    assert 5 * E < R <= 20 * E
    ends = np.cumsum(counts).astype(np.int64)
    x, w, s = bf16_normal((R, K), K), int4_words((E, K, N // 8), N), scales((E, K // gs, N), N + 2)
    y = grouped_matmul([to_dev(x, device)], [to_dev(w, device)], antiquant_scale=[to_dev(s, device)],
                       group_list=to_dev(ends, device), split_item=3, group_type=0)[0]
    torch.cuda.synchronize()
    assert_rounds_exactly(y, *O.grouped_gemm_exact(x, w, s, ends), f"mid rows grouped K={K} N={N}")


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,H,MI,gs,k,zipf", [
    (5, 64, 512, 192, 64, 10, 0.0),     # a partial 128-column act tile
    (32, 64, 320, 256, 32, 10, 1.5),    # 256-column act tiles, experts of more than 12 rows, ragged H
    (8, 32, 4096, 64, 64, 16, 0.0),     # the longest rows, the largest top-k
    (51, 128, 512, 192, 64, 10, 2.0),   # routed in two launches, popular experts of several 12-row tiles
    (70, 64, 512, 192, 64, 10, 0.0),    # 32-row tiles: a partial 128-column act tile
    (120, 64, 320, 64, 32, 10, 1.5),    # and one K chunk in the down projection, experts of more than 32 rows
])
def test_expert_block_stages(device, T, E, H, MI, gs, k, zipf):
    from qmoe import moe_prefill
    from qmoe.workload import zipf_logits
    log(f"few rows block T={T} E={E} H={H} MI={MI}")
    lay = layer(E, H, MI, gs, T + E)
    gu, dn = layer_dev(lay, device)
    x = bf16_normal((T, H), 3)
    lg = zipf_logits(T, E, zipf, 4) if zipf else bf16_normal((T, E), 4)
    out, (idx, w, _, ends, order, inverse), (act, prod) = moe_prefill(
        to_dev(x, device), to_dev(lg, device), gu, dn, k, return_routing=True, return_intermediates=True)
    torch.cuda.synchronize()
    ref = O.moe_prefill(x, lg, lay["gu_w"], lay["gu_s"], lay["dn_w"], lay["dn_s"], k)
    for got, name in ((idx, "idx"), (ends, "ends"), (order, "order"), (inverse, "inverse")):
        assert np.array_equal(got.cpu().numpy(), ref[name]), name
    ab, pb, ob = bits(act), bits(prod), bits(out)
    ge, ga = O.grouped_gemm_exact(x[ref["order"] // k], lay["gu_w"], lay["gu_s"], ref["ends"])
    assert_in_interval(ab, *O.swiglu_interval(ge[:, :MI], ga[:, :MI], ge[:, MI:], ga[:, MI:]), f"T={T} act")
    ye, ya = O.grouped_gemm_exact(ab, lay["dn_w"], lay["dn_s"], ref["ends"])
    lo, hi = prod_interval(ye, ya, ref["w"].reshape(-1)[ref["order"]])
    flo, fhi = np.empty_like(lo), np.empty_like(hi)
    flo[ref["order"]], fhi[ref["order"]] = lo, hi
    assert_in_interval(pb, flo, fhi, f"T={T} prod")
    assert_bf16_equal(ob, O.weighted_reduce(pb, O.f32_to_bf16_bits(np.ones((T, k), np.float32))), f"T={T} sum")


@pytest.mark.gpu
@pytest.mark.parametrize("K,gs", [(64, 32), (256, 64), (1024, 128)])
@pytest.mark.parametrize("over", [0, 1])
def test_dense_rule_sides(device, K, gs, over):
    """Both sides of the dense rule's line: the last row count on the few-rows kernel
    and the next, on the tiled one."""
    from qmoe import _lib, weight_quant_batchmatmul
    N = 4096
    M = next(m for m in range(16, 4096, 16) if not _lib.lib().qmoe_w4a16_gemm_few_rows(m + 1, K, N, gs)) + over
    log(f"dense rule M={M} K={K} gs={gs}")
    x, w, s = bf16_normal((M, K), M + K), int4_words((K, N // 8), K + N), scales((K // gs, N), N + 1)
    y = weight_quant_batchmatmul(to_dev(x, device), to_dev(w, device), to_dev(s, device), antiquant_group_size=gs)
    torch.cuda.synchronize()
    assert_rounds_exactly(y, *O.w4a16_gemm_exact(x, w, s, gs), f"dense rule M={M} K={K}")


def wide_scales(shape, seed, top):
    """Scales of 2^90 to 2^top in some groups among ordinary ones, columns of only
    those, columns without (eight times the largest is still an fp32 value)."""
    r = np.random.default_rng(seed)
    s = O.bf16_bits_to_f32(scales(shape, seed))
    big = np.exp2(r.integers(90, top, size=shape)) * (1 + r.integers(0, 128, size=shape) / 128)
    share = np.broadcast_to(np.array([0.0, 0.1, 0.5, 1.0])[np.arange(shape[-1]) % 4], shape)
    return O.f32_to_bf16_bits(np.where(r.random(shape) < share, big, s).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,gs", [(5, 64, 32, 32), (48, 2048, 416, 128), (300, 576, 8224, 96)])
def test_dense_wide_scales(device, M, K, N, gs):
    """Scales with which a row's sums leave the fp32 range and its results do not."""
    from qmoe import weight_quant_batchmatmul
    log(f"few rows wide scales dense M={M} K={K} N={N} gs={gs}")
    x = bf16_normal((M, K), M + K, 2.0 ** -100)
    x[1] = O.f32_to_bf16_bits(O.bf16_bits_to_f32(x[1]) * np.float32(2.0 ** 60))
    w, s = int4_words((K, N // 8), K + N), wide_scales((K // gs, N), N + 1, 124)
    y = weight_quant_batchmatmul(to_dev(x, device), to_dev(w, device), to_dev(s, device), antiquant_group_size=gs)
    torch.cuda.synchronize()
    assert_rounds_exactly(y, *O.w4a16_gemm_exact(x, w, s, gs), f"few rows wide scales M={M} K={K} N={N}")


@pytest.mark.gpu
@pytest.mark.parametrize("E,H,MI,gs,k", [(64, 512, 192, 64, 10), (64, 320, 256, 32, 10)])
def test_expert_block_wide_scales(device, E, H, MI, gs, k):
    """The same in the block: in the gate and up sums of tiny rows and in the down
    sums (one act tile width each)."""
    from qmoe import moe_prefill
    log(f"few rows wide scales block E={E} H={H} MI={MI}")
    T = 5 * E // k
    lay = layer(E, H, MI, gs, T + E)
    lay["gu_s"] = wide_scales((E, H // gs, 2 * MI), 5, 118)
    lay["dn_s"][:, :, ::3] = 0x7780 | (lay["dn_s"][:, :, ::3] & 0x7f)  # 2^112 to 2^113
    gu, dn = layer_dev(lay, device)
    x, lg = bf16_normal((T, H), 3, 2.0 ** -124), bf16_normal((T, E), 4)
    out, (idx, w, _, ends, order, _), (act, prod) = moe_prefill(
        to_dev(x, device), to_dev(lg, device), gu, dn, k, return_routing=True, return_intermediates=True)
    torch.cuda.synchronize()
    ref = O.moe_prefill(x, lg, lay["gu_w"], lay["gu_s"], lay["dn_w"], lay["dn_s"], k)
    assert np.array_equal(idx.cpu().numpy(), ref["idx"])
    ab, pb = bits(act), bits(prod)
    ge, ga = O.grouped_gemm_exact(x[ref["order"] // k], lay["gu_w"], lay["gu_s"], ref["ends"])
    assert_in_interval(ab, *O.swiglu_interval(ge[:, :MI], ga[:, :MI], ge[:, MI:], ga[:, MI:]), f"T={T} act")
    ye, ya = O.grouped_gemm_exact(ab, lay["dn_w"], lay["dn_s"], ref["ends"])
    lo, hi = prod_interval(ye, ya, ref["w"].reshape(-1)[ref["order"]])
    flo, fhi = np.empty_like(lo), np.empty_like(hi)
    flo[ref["order"]], fhi[ref["order"]] = lo, hi
    assert_in_interval(pb, flo, fhi, f"T={T} prod")
