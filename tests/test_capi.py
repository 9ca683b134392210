"""The C-ABI library loads and exports every entry point include/qmoe.h declares (CPU only)."""
import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "qmoe.h"


def declared():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(qmoe_\w+)\s*\(", text)))


def test_header_declares_entry_points():
    names = declared()
    assert "qmoe_w4a16_gemv" in names and "qmoe_grouped_gemm" in names and len(names) >= 20


def test_library_exports_every_declared_symbol():
    from qmoe import _lib
    path = _lib.library_path()
    if not path.exists():
        pytest.fail(f"{path} not built")
    so = ctypes.CDLL(str(path))
    missing = [n for n in declared() if not hasattr(so, n)]
    assert not missing, missing


def test_python_binding_covers_header():
    from qmoe import _lib
    assert sorted(_lib.SIGNATURES) == declared()
    so = _lib.lib()
    for name in _lib.SIGNATURES:
        assert getattr(so, name).restype is not None or name == ""


def test_host_side_shape_queries():
    from qmoe import _lib
    L = _lib.lib()
    assert L.qmoe_gemm_tile_rows() == 128
    assert L.qmoe_max_row_tiles(40960, 512, 128) == 320 + 512
    assert L.qmoe_w4a16_gemm_workspace(1, 2048, 4096) == 0          # partials live in the counters mailbox
    assert L.qmoe_w4a16_gemm_counters(1, 2048, 4096) == 65536 + 2 * 16 * 15 * 4 * 256
    assert L.qmoe_moe_decode_workspace(1, 10, 2048, 512) > 0
    assert L.qmoe_route_group_workspace(40960, 512) == (160 + 1) * 512 * 4  # chunk histograms + expert totals
    # argument validation happens on the host, before any launch
    assert L.qmoe_w4a16_gemv(None, None, None, None, 5, 2048, 4096, 128, None, 0, None, None) == -1
    assert L.qmoe_w4a16_gemv(None, None, None, None, 1, 2048, 4096, 128, None, 0, None, None) == -1  # no counters
    assert L.qmoe_router_topk(None, None, None, 1, 512, 17, None) == -1
    assert L.qmoe_moe_decode(*([None] * 11), 5, 512, 10, 2048, 512, 128, 128, None, 0, None, None) == -1


@pytest.mark.parametrize("R,E,K,N,gs,rows", [
    (1, 512, 2560, 1280, 64, 12), (5 * 64, 64, 4096, 32, 32, 12), (5 * 64 + 1, 64, 4096, 32, 32, 32),
    (20 * 64, 64, 512, 64, 128, 32), (20 * 64 + 1, 64, 512, 64, 128, 128),
    (854, 512, 2560, 1280, 64, 12), (855, 512, 2560, 1280, 64, 32),  # few rows per expert, but 2.8e9 multiply-adds
    (8477, 512, 3072, 1536, 64, 32), (8478, 512, 3072, 1536, 64, 128),  # 4e10
    (10, 512, 4160, 64, 32, 32),      # rows too long for the few-rows kernel's LDS
    (10, 512, 96, 64, 32, 32), (10, 512, 64, 48, 32, 32), (10, 512, 64, 64, 16, 32),  # shapes it does not take
])
def test_tile_rows_rule(R, E, K, N, gs, rows):
    """The row-tile size by rows per expert and work, and the block's as the larger of its
    two GEMMs' (every size here is one the grouped entry points take)."""
    from qmoe import _lib
    L = _lib.lib()
    assert L.qmoe_gemm_tile_rows_for(R, E, K, N, gs) == rows
    for MI in (64, 640, 4096, 4160):
        both = [L.qmoe_gemm_tile_rows_for(R, E, K, 2 * MI, gs), L.qmoe_gemm_tile_rows_for(R, E, MI, K, 64)]
        assert L.qmoe_moe_tile_rows(R, E, K, MI, gs, 64) == max(both)


@pytest.mark.parametrize("K,rounds", [(64, 1), (192, 1), (256, 2), (960, 2), (1024, 3), (1984, 3), (2048, 4), (4096, 4)])
def test_few_rows_rule(K, rounds):
    """The dense W4 GEMM's kernel by rounds of workgroups (16 rows x 128 columns, 256
    at once): more of them only where K is long."""
    from qmoe import _lib
    few = _lib.lib().qmoe_w4a16_gemm_few_rows
    assert few(16 * 8 * rounds, K, 4096, 32) == 1 and few(16 * 8 * rounds + 1, K, 4096, 32) == 0
    assert few(16, K, 128 * 256 * rounds, 32) == 1 and few(16, K, 128 * 256 * rounds + 32, 32) == 0
    assert few(5, K, 48, 32) == 0 and few(5, K + 32, 64, 32) == 0 and few(5, 4160, 64, 64) == 0


def test_stream_handle_without_the_private_name(monkeypatch):
    """A torch without the raw-handle function: the public Stream object's handle."""
    import importlib.util
    from types import SimpleNamespace

    import torch
    from qmoe import _lib
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev: SimpleNamespace(cuda_stream=(dev, 7)))
    spec = importlib.util.spec_from_file_location("qmoe_lib_copy", _lib.__file__)
    copy = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(copy)
    assert copy.stream_of(SimpleNamespace(get_device=lambda: 1, device="cuda:1")) == ("cuda:1", 7)
