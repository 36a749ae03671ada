"""The C-ABI library: loads, exports every symbol in include/klc_moe.h, checks
arguments on the host.  No call here reaches a kernel launch."""

from __future__ import annotations

import ctypes
import re
import sys
import threading
from pathlib import Path

import numpy as np
import pytest

from klcquant_amd import _native as nat

HEADER = Path(__file__).resolve().parents[1] / "include" / "klc_moe.h"


def header_functions() -> list[str]:
    text = HEADER.read_text()
    return sorted(set(re.findall(r"^\s*(?:const\s+)?[\w\s\*]+?\b(klc_\w+)\s*\(", text, flags=re.M)))


def test_library_loads_and_exports_every_declared_symbol():
    lib = nat.load()
    names = header_functions()
    assert "klc_moe_layer" in names and "klc_mxfp4_dequant" in names
    for name in names:
        assert hasattr(lib, name), name
    assert set(names) == set(nat.SIGNATURES), "ctypes table and header disagree"


def test_abi_version_matches_header():
    m = re.search(r"#define KLC_ABI_VERSION (\d+)", HEADER.read_text())
    assert nat.load().klc_abi_version() == int(m.group(1))


def test_status_codes_match_header():
    text = HEADER.read_text()
    for name, value in [("KLC_ERR_ARGUMENT", nat.KLC_ERR_ARGUMENT), ("KLC_ERR_SHAPE", nat.KLC_ERR_SHAPE),
                        ("KLC_ERR_UNSUPPORTED", nat.KLC_ERR_UNSUPPORTED), ("KLC_ERR_HIP", nat.KLC_ERR_HIP),
                        ("KLC_DTYPE_BF16", nat.DTYPE_BF16), ("KLC_DTYPE_F16", nat.DTYPE_F16),
                        ("KLC_DTYPE_F32", nat.DTYPE_F32), ("KLC_PRECISION_FP32", nat.PRECISION_FP32),
                        ("KLC_PRECISION_BF16", nat.PRECISION_BF16), ("KLC_LAYER_EVENTS", nat.LAYER_EVENTS),
                        ("KLC_DISPATCH_MAX_PAIRS", nat.DISPATCH_MAX_PAIRS),
                        ("KLC_LAYER_MAX_TOKENS", nat.LAYER_MAX_TOKENS)]:
        m = re.search(rf"#define {name} \(?(-?\d+)\)?", text)
        assert m and int(m.group(1)) == value, name


def test_packed_sizes():
    lib = nat.load()
    # 5760 rows x 90 groups: blocks 90 tiles x 90 KiB, scale records of 24 bytes per (row, quarter)
    assert lib.klc_mxfp4_packed_bytes(5760, 90) == 90 * 90 * 1024 + 5760 * 4 * 24
    assert lib.klc_mxfp4_packed_bytes(64, 1) == 1024 + 64 * 4 * 8
    assert lib.klc_mxfp4_packed_bytes(100, 90) == nat.KLC_ERR_SHAPE
    assert "multiple of 64" in nat.last_error()
    assert lib.klc_mxfp4_packed_bytes(0, 90) == nat.KLC_ERR_ARGUMENT


def test_argument_errors_before_any_launch():
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_mxfp4_dequant", None, None, None, 1, 64, 2, nat.DTYPE_BF16, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "null pointer" in ei.value.message
    fake = ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_topk_softmax", fake, fake, fake, fake, 4, 8, 9, None)
    assert ei.value.status == nat.KLC_ERR_SHAPE
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_dispatch", fake, 16, 300, fake, fake, fake, fake, fake, None)
    assert ei.value.status == nat.KLC_ERR_UNSUPPORTED
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_router_logits", fake, fake, fake, fake, None, 2, 100, 8, None)
    assert ei.value.status == nat.KLC_ERR_SHAPE
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_gate_up", fake, fake, fake, 2, 4, 128, fake, fake, fake, 2880, 2880, 7.0, 5, fake,
                 None, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_down", fake, fake, fake, 8, 128, fake, fake, fake, 4096, 2880, 0, fake, None)
    assert ei.value.status == nat.KLC_ERR_UNSUPPORTED
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_synth_fill", fake, 16, 1, 1, 10, 300, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT


def test_route_entry_argument_errors():
    """klc_moe_route: its own outputs may not be NULL, and the one-launch path (which keeps no float32
    SwiGLU outputs) is refused; both before any device work."""
    fake = ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first
    args = [fake] * 7 + [2, 2880, 2880, 128, 4, 7.0, nat.PRECISION_FP32]
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_route", *args, nat.PATH_AUTO, fake, 1 << 30, fake, fake, fake, None, fake, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "null pointer" in ei.value.message
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_route", *args, nat.PATH_FUSED, fake, 1 << 30, fake, fake, fake, fake, fake, None)
    assert ei.value.status == nat.KLC_ERR_UNSUPPORTED and "float32 SwiGLU" in ei.value.message
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_route", *args, nat.PATH_AUTO, fake, 256, fake, fake, fake, fake, fake, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "workspace" in ei.value.message


@pytest.mark.parametrize("n_tok,hidden,inter,n_exp,k,path", [
    (96, 2880, 2880, 128, 4, nat.PATH_GEMM), (95, 2880, 2880, 128, 4, nat.PATH_GEMV),
    (48, 2880, 2880, 64, 4, nat.PATH_GEMM), (47, 2880, 2880, 64, 4, nat.PATH_GEMV),
    (32, 2880, 2880, 32, 4, nat.PATH_GEMM), (31, 2880, 2880, 32, 4, nat.PATH_GEMV),
    # small layers: the GEMV is the faster one at these loads
    (48, 2048, 1024, 64, 4, nat.PATH_GEMV), (65, 2048, 1024, 64, 4, nat.PATH_GEMV),
    (66, 2048, 1024, 64, 4, nat.PATH_GEMM), (32, 2048, 1024, 32, 4, nat.PATH_GEMV),
    (36, 2048, 1024, 32, 4, nat.PATH_GEMM), (96, 2048, 1024, 128, 4, nat.PATH_GEMM),
    (32, 512, 512, 32, 4, nat.PATH_GEMV), (112, 512, 512, 64, 4, nat.PATH_GEMV),
    (33, 256, 128, 32, 4, nat.PATH_GEMV), (100, 256, 128, 128, 4, nat.PATH_GEMV),
    # 8 pairs an expert, whatever the size
    (64, 512, 512, 32, 4, nat.PATH_GEMM), (63, 512, 512, 32, 4, nat.PATH_GEMV),
    (32, 256, 128, 16, 4, nat.PATH_GEMM), (31, 256, 128, 16, 4, nat.PATH_GEMV)])
def test_layer_path_lines(n_tok, hidden, inter, n_exp, k, path):
    """KLC_PATH_AUTO at the lines between the decode GEMVs and the grouped GEMM."""
    assert nat.call("klc_moe_layer_path", n_tok, hidden, inter, n_exp, k, nat.PATH_AUTO, None) == path


def test_attention_step_wait_leaves_the_interpreter_to_other_threads():
    """The wait for a step's record ends by what another Python thread does, with thread switches of the
    interpreter put off past the wait's limit; without the tag it ends at the limit."""
    record = np.zeros(16, dtype=np.int32)
    nat.load()
    started = threading.Event()

    def writer():
        started.wait()
        record[8] = 7

    thread = threading.Thread(target=writer)
    interval = sys.getswitchinterval()
    thread.start()
    try:
        sys.setswitchinterval(60.0)
        started.set()
        assert nat.call("klc_attn_step_wait", record.ctypes.data, 7, 20_000_000) == 1
    finally:
        sys.setswitchinterval(interval)
        thread.join()
    assert nat.call("klc_attn_step_wait", record.ctypes.data, 8, 1000) == 0
    for args in ((None, 7, 0), (record.ctypes.data, 0, 0), (record.ctypes.data, 1 << 32, 0)):
        with pytest.raises(nat.KlcError):
            nat.call("klc_attn_step_wait", *args)


def test_attention_workspace_never_shrinks_with_the_count():
    """A workspace made for a ring's capacity serves every shorter span, across the lines between
    the kernels' block sizes (256, 8,192 and 65,536 keys)."""
    lib = nat.load()
    for nh, nkv, d in ((64, 8, 64), (8, 8, 128), (3, 1, 8)):
        for size in (lambda n: lib.klc_attn_workspace_bytes(nh, d, n),
                     lambda n: lib.klc_attn_step_workspace_bytes(nh, nkv, d, n)):
            sizes = [size(n) for n in (*range(1, 600), *range(8000, 8400), *range(65400, 65800), 1 << 20, 1 << 22)]
            assert all(a > 0 for a in sizes) and sizes == sorted(sizes)


def test_units_size():
    lib = nat.load()
    # 256 pairs over 128 experts: gate_up (256 + 7 * 128) // 8 = 144, down (256 + 3 * 128) // 4 = 160,
    # GEMM (256 + 63 * 128) // 64 = 130
    assert lib.klc_moe_units_size(256, 128) == 4 + 144 + 160 + 130
    assert lib.klc_moe_units_size(4, 128) == 4 + 4 + 4 + 4
    assert lib.klc_moe_units_size(16, 300) == nat.KLC_ERR_UNSUPPORTED


def test_workspace_size_grows_with_tokens():
    lib = nat.load()
    a = lib.klc_moe_workspace_bytes(1, 2880, 2880, 128, 4)
    b = lib.klc_moe_workspace_bytes(64, 2880, 2880, 128, 4)
    assert 0 < a < b and a % 256 == 0 and b % 256 == 0
    assert lib.klc_moe_workspace_bytes(0, 2880, 2880, 128, 4) == nat.KLC_ERR_ARGUMENT


def test_cpu_tensors_are_rejected():
    torch = pytest.importorskip("torch")
    from klcquant_amd import ops

    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="GPU"):
        ops.router_logits(x, torch.zeros((4, 64), dtype=torch.bfloat16), torch.zeros(4, dtype=torch.bfloat16))
    with pytest.raises(ValueError, match="shape mismatch"):
        ops.mxfp4_dequant(torch.zeros((4, 2, 16), dtype=torch.uint8), torch.zeros((4, 3), dtype=torch.uint8))


def test_select_and_experts_argument_errors():
    """klc_moe_select / klc_moe_experts check their arguments before any device work."""
    fake = ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_select", fake, fake, None, 2, 2880, 128, 4, fake, 1 << 30, fake, fake, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "null pointer" in ei.value.message
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_select", fake, fake, fake, 2, 2880, 128, 4, fake, 64, fake, fake, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "workspace" in ei.value.message
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_select", fake, fake, fake, 2, 2880, 8, 9, fake, 1 << 30, fake, fake, None)
    assert ei.value.status == nat.KLC_ERR_SHAPE
    args = [fake] * 7 + [2, 2880, 2880, 128, 4, 7.0, nat.PRECISION_FP32]
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_experts", *args, nat.PATH_FUSED, fake, 1 << 30, fake, None, None, None)
    assert ei.value.status == nat.KLC_ERR_UNSUPPORTED
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_experts", *args, nat.PATH_AUTO, fake, 1 << 30, fake, fake, None, None)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "together" in ei.value.message


def test_route_readback_argument_errors():
    """klc_moe_route_readback: a host record and a nonzero tag are required, before any device work."""
    fake = ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first
    head = [fake] * 7 + [1, 2880, 2880, 128, 4, 7.0, nat.PRECISION_FP32, nat.PATH_AUTO, fake, 1 << 30]
    outs = [fake] * 4
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_route_readback", *head, *outs, None, 1, fake)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "null host record" in ei.value.message
    with pytest.raises(nat.KlcError) as ei:
        nat.call("klc_moe_route_readback", *head, *outs, fake, 0, fake)
    assert ei.value.status == nat.KLC_ERR_ARGUMENT and "tag 0" in ei.value.message
