"""The C-ABI library (CPU checks, no GPU compute): it loads, exports every
function ``include/mlops_mi355x.h`` declares with the binding's signature,
and its argument validation rejects bad shapes with a message before any
kernel is launched."""

import ctypes
import re
from pathlib import Path

import pytest

from mlops_amd import _native

HEADER = Path(__file__).resolve().parents[1] / "include" / "mlops_mi355x.h"


def _declared():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = re.findall(r"\b(mi355x_\w+)\s*\(", text)
    return sorted(set(names))


def test_header_and_binding_agree():
    declared = _declared()
    assert declared == sorted(_native.SIGNATURES), set(declared) ^ set(_native.SIGNATURES)


def test_library_exports_every_declared_symbol():
    lib = _native.library()
    for name in _declared():
        assert hasattr(lib, name), name
    assert lib.mi355x_abi_version() == 1


def test_argument_counts_match_header():
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    for name, (_, argtypes) in _native.SIGNATURES.items():
        match = re.search(rf"\b{name}\s*\(([^)]*)\)", text)
        params = [p for p in match.group(1).split(",") if p.strip() and p.strip() != "void"]
        assert len(params) == len(argtypes), name


@pytest.mark.parametrize("name,args,message", [
    ("mi355x_gemm_fp8_block", (None, None, 10, None, None, 0, 4, 100, 256, None, 0, None, None, None),
     "N must be a multiple of 128"),
    ("mi355x_gemm_fp8_block", (None, None, 10, None, None, 0, 4, 256, 200, None, 0, None, None, None),
     "K must be a multiple of 128"),
    ("mi355x_router_topk", (None, 10, 1000, 2, 0, None, 1, 1, 1.0, None, None, None, None),
     "experts"),
    ("mi355x_permute_plan", (None, 10, 2000, None, None, None, None, None, 0, None), "experts"),
    ("mi355x_quantize_rows_fp8", (None, 4, 100, 100, 0, None, None, None), "multiple of 128"),
])
def test_validation_errors(name, args, message):
    with pytest.raises(_native.NativeError, match=message):
        _native.call(name, *args)


def _gemm_arguments(workspace, size):
    # 4096 rows over 8 experts, N 4096, K 14336: a last round that may be split.
    return _native.GEMM_ARGS.pack(*[0] * 10, workspace, size, 4096, 0, 1, 8, 4096, 14336, *[0] * 5)


def _backward_arguments(workspace, size):
    return _native.MOE_BLOCK_BWD_ARGS.pack(*[0] * 21, workspace, size, 16, 256, 128, 4, 2, 0, 1, 1,
                                           0, 0.0)


@pytest.mark.parametrize("name,args", [
    ("mi355x_moe_route", lambda at, n: (None, 100, 8, 2, 0, None, 1, 1, 1.0, None, 1, None, None,
                                        2, *[None] * 8, at, n, None)),
    ("mi355x_moe_down", lambda at, n: (None, 16, 2, 256, 128, 0.0, 0, None, None, 4, *[None] * 5,
                                       at, n, None)),
    ("mi355x_moe_block_bwd", lambda at, n: (_backward_arguments(at, n), None)),
    ("mi355x_gemm_fp8", lambda at, n: (_gemm_arguments(at, n), None)),
])
def test_workspaces_must_be_aligned(name, args):
    """Every buffer of a sequence lies at 256-byte steps from its workspace and
    takes 16-byte vector accesses."""
    with pytest.raises(_native.NativeError, match="workspace must be 16-byte aligned"):
        _native.call(name, *args(0x10008, 1 << 30))
    with pytest.raises(_native.NativeError, match="workspace too small"):
        _native.call(name, *args(0x10000, 16))


def test_packed_argument_structs_cover_the_c_ones():
    """The entry points copy the whole struct, tail padding included."""
    assert _native.GEMM_ARGS.size == _native.query("mi355x_gemm_args_size")
    assert _native.MOE_BLOCK_BWD_ARGS.size == _native.query("mi355x_moe_block_bwd_args_size")


def test_sizes_are_queries():
    assert _native.query("mi355x_wgrad_padded_rows", 1000, 8) % 128 == 0
    assert _native.query("mi355x_wgrad_padded_rows", 1000, 8) >= 1000 + 8 * 127
    assert _native.query("mi355x_permute_plan_workspace_size", 131072, 128) >= 32 * 128 * 4
