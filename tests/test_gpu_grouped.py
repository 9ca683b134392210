"""Grouped W4A16 GEMM (npu_grouped_matmul replacement) vs the oracle."""
import numpy as np
import pytest
import torch

from gpu_util import bf16_normal, int4_words, log, scales
from oracle import qmoe_oracle as O
from parity import assert_bf16_close, assert_rounds_exactly, bits, to_dev


@pytest.mark.gpu
@pytest.mark.parametrize("counts,K,N,gs", [
    ([3, 0, 1, 0, 300, 17], 256, 384, 64),     # empty experts, a 3-tile expert, partial tiles
    ([1] * 10, 512, 2048, 128),                 # one row per expert (the diagonal decode shape)
    ([0, 0, 5], 2048, 1024, 128),
    ([128, 129], 768, 3072, 64),
    ([40] * 16, 3072, 1536, 64),
])
def test_grouped_matmul(device, counts, K, N, gs):
    from qmoe import grouped_matmul
    E = len(counts)
    log(f"grouped counts={counts[:8]} K={K} N={N} gs={gs}")
    seed = K + N + E
    ends = np.cumsum(counts).astype(np.int64)
    R = int(ends[-1])
    x = bf16_normal((R, K), seed)
    w = int4_words((E, K, N // 8), seed + 1)
    s = scales((E, K // gs, N), seed + 2)
    y = grouped_matmul([to_dev(x, device)], [to_dev(w, device)], antiquant_scale=[to_dev(s, device)],
                       group_list=to_dev(ends, device), split_item=3, group_type=0, output_dtype=torch.bfloat16)[0]
    torch.cuda.synchronize()
    assert_rounds_exactly(y, *O.grouped_gemm_exact(x, w, s, ends), f"grouped E={E} K={K} N={N}")
    assert_bf16_close(y, O.grouped_gemm(x, w, s, ends), f"grouped E={E} K={K} N={N}")


@pytest.mark.gpu
def test_grouped_matmul_row_permutation_invariance(device):
    """Each output row depends only on its own input row: permuting rows within an
    expert permutes the output rows bit for bit."""
    from qmoe import grouped_matmul
    log("grouped permutation invariance")
    counts = [70, 0, 200]
    E, K, N, gs = 3, 512, 256, 128
    ends = torch.tensor(np.cumsum(counts), dtype=torch.int64, device=device)
    x = to_dev(bf16_normal((270, K), 11), device)
    w = to_dev(int4_words((E, K, N // 8), 12), device)
    s = to_dev(scales((E, K // gs, N), 13), device)
    p = torch.cat([torch.randperm(70, generator=torch.Generator().manual_seed(1)),
                   70 + torch.randperm(200, generator=torch.Generator().manual_seed(2))]).to(device)
    y = grouped_matmul([x], [w], antiquant_scale=[s], group_list=ends, split_item=3, group_type=0)[0]
    yp = grouped_matmul([x[p].contiguous()], [w], antiquant_scale=[s], group_list=ends, split_item=3,
                        group_type=0)[0]
    torch.cuda.synchronize()
    assert torch.equal(yp.view(torch.int16), y[p].view(torch.int16))


@pytest.mark.gpu
def test_grouped_entries_with_128_row_tables(device):
    """The entry points that take no tile size, with tables of 128-row tiles: the
    GEMM against the exact sums, the expert block with the bits that 32-row tiles
    give (a row's sums do not depend on its tile)."""
    from gpu_util import layer, layer_dev
    from qmoe import _lib, moe_prefill
    from qmoe.ops import route_tokens
    L = _lib.lib()
    bm = L.qmoe_gemm_tile_rows()
    counts, K, N, gs = [3, 0, 1, 0, 300, 17], 256, 384, 64
    E, R = len(counts), sum(counts)
    log(f"128-row tables E={E} R={R}")
    ends = np.cumsum(counts).astype(np.int64)
    x, w, s = bf16_normal((R, K), 1), int4_words((E, K, N // 8), 2), scales((E, K // gs, N), 3)
    xd, wd, sd, ed = (to_dev(a, device) for a in (x, w, s, ends))
    st = _lib.stream_of(xd)
    mt = L.qmoe_max_row_tiles(R, E, bm)
    t = torch.empty(3 * mt + 1, dtype=torch.int32, device=device)
    table = [t.data_ptr() + 4 * mt * i for i in range(4)]
    _lib.check(L.qmoe_tiles_from_ends(ed.data_ptr(), E, R, bm, *table, st), "tiles")
    y = torch.empty((R, N), dtype=torch.bfloat16, device=device)
    ws = _lib.workspace(device, L.qmoe_grouped_gemm_workspace(R, K))
    _lib.check(L.qmoe_grouped_gemm(xd.data_ptr(), R, K, N, E, gs, wd.data_ptr(), sd.data_ptr(), *table, mt, y.data_ptr(),
                                   ws.data_ptr(), ws.numel(), st), "grouped_gemm")
    torch.cuda.synchronize()
    assert_rounds_exactly(y, *O.grouped_gemm_exact(x, w, s, ends), "128-row tables")

    T, E, H, MI, gs, k = 90, 64, 512, 192, 64, 8
    gu, dn = layer_dev(layer(E, H, MI, gs, 5), device)
    xd, lg = to_dev(bf16_normal((T, H), 6), device), to_dev(bf16_normal((T, E), 7), device)
    assert L.qmoe_moe_tile_rows(T * k, E, H, MI, gs, gs) == 32
    ref = moe_prefill(xd, lg, gu, dn, k)
    idx, wts, _, _, order, _, t, mt = route_tokens(lg, k, bm)
    out = torch.empty_like(xd)
    ws = _lib.workspace(device, L.qmoe_moe_prefill_workspace(T, k, H, MI))
    _lib.check(L.qmoe_moe_experts_grouped(xd.data_ptr(), T, H, MI, E, k, wts.data_ptr(), order.data_ptr(),
                                          gu.w4.data_ptr(), gu._scales.data_ptr(), gs, dn.w4.data_ptr(),
                                          dn._scales.data_ptr(), gs, *[t.data_ptr() + 4 * mt * i for i in range(4)], mt,
                                          None, out.data_ptr(), ws.data_ptr(), ws.numel(), st), "experts_grouped")
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
