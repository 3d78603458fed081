"""The C-ABI library loads and exports every symbol include/af3_mi355x.h declares (CPU)."""
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "af3_mi355x.h"


def declared_symbols():
    text = HEADER.read_text()
    return sorted(set(re.findall(r"^\s*(?:int|size_t|const char\*)\s+(af3_\w+)\s*\(", text, re.M)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert "af3_moe_gemm" in syms and "af3_mxfp4_to_bf16" in syms and len(syms) >= 14


def test_library_exports_every_declared_symbol():
    from agent_factory_3_amd import _capi
    path = _capi.lib_path()
    if not path.exists():
        pytest.skip("library not built (run __graft_entry__.build())")
    out = subprocess.run(["nm", "-D", "--defined-only", str(path)], capture_output=True, text=True, check=True).stdout
    exported = set(re.findall(r"\sT\s(af3_\w+)", out))
    missing = [s for s in declared_symbols() if s not in exported]
    assert not missing, missing
    # the Python binding knows every declared symbol with a signature
    assert sorted(declared_symbols()) == sorted(_capi.exported_symbols())


def test_library_loads_and_reports_abi():
    from agent_factory_3_amd import _capi
    if not _capi.lib_path().exists():
        pytest.skip("library not built")
    lib = _capi.load()
    assert lib.af3_abi_version() == _capi.ABI_VERSION
    # argument errors come back as a Python exception with the library's message, no GPU needed
    with pytest.raises(RuntimeError, match="n_groups"):
        _capi.call("af3_mxfp4_to_bf16", None, None, None, -1, None)
    assert _capi.workspace_bytes(16, 4, 2) > 0


def test_noalloc_routing_rejects_shapes_beyond_its_scratch():
    """af3_routing_replay_noalloc checks the shape against its built-in scratch
    array before touching the device (no GPU needed for the error path)."""
    from agent_factory_3_amd import _capi
    if not _capi.lib_path().exists():
        pytest.skip("library not built")
    lib = _capi.load()
    T, E, K = 1 << 20, 128, 4
    assert _capi.workspace_bytes(T, E, K) > int(lib.af3_routing_scratch_bytes()) == 4 << 20
    with pytest.raises(RuntimeError, match="scratch"):
        _capi.call("af3_routing_replay_noalloc", 1, E, 1, T, E, K, 1, 1, 1, 1, 1, None)


@pytest.mark.parametrize("E", [1, 3, 32, 64, 128, 1024, 1025])
def test_routing_workspace_covers_its_count_rows(E):
    """The reported workspace holds the ids, the weights and every count row the
    launches write, for any number of experts per token, and is never more than
    one row per 256 entries asks for (sizes a caller kept, the built-in array)."""
    from agent_factory_3_amd import _capi
    if not _capi.lib_path().exists():
        pytest.skip("library not built")
    lib = _capi.load()
    up = lambda n: (n + 255) // 256 * 256  # noqa: E731
    for K in range(1, min(E, 16) + 1):
        for T in (0, 1, 63, 64, 65, 255, 257, 300, 512, 4096, 4097, 8191, 65537, 500000):
            rows = int(lib.af3_routing_count_rows(T, E, K))
            head = up(up(4 * T * K) + 2 * T * K)
            assert (T + 255) // 256 <= rows <= (T * K + 255) // 256
            assert _capi.workspace_bytes(T, E, K) >= head + 4 * rows * E
            assert _capi.workspace_bytes(T, E, K) <= head + (T * K + 255) // 256 * E * 4 + 256
            for topk in (0, 1):
                n = int(lib.af3_routing_plan_workspace_bytes(T, E, K, topk))
                one_block = T * K <= 4096 and (not topk or E > 256 or T <= 256)
                assert n == _capi.workspace_bytes(T, E, K) or (n == 0 and one_block)


def test_product_path_has_no_oracle_dependency():
    pkg = ROOT / "agent-factory-3_amd" / "agent_factory_3_amd"
    for f in pkg.glob("*.py"):
        assert "oracle" not in re.findall(r"^\s*(?:from|import)\s+(\w+)", f.read_text(), re.M), f.name


def test_stream_of_refuses_a_host_device():
    # the stream lookup is what stops host tensors from reaching a kernel as pointers
    import pytest
    import torch

    from agent_factory_3_amd import _capi
    with pytest.raises(ValueError, match="cuda device"):
        _capi.stream_of(torch.device("cpu"))
