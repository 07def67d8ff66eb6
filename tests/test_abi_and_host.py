"""No-GPU checks of the product: the C-ABI library loads and exports every symbol the header declares,
rejects bad arguments before touching the device, and the Python operator layer refuses to run
without a HIP device (there is no host fallback)."""
import ctypes
import os
import re
import subprocess
import sys

import pytest
import torch

import _splat_hip as hip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "splat_hip.h")


def header_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(splat_[a-z_0-9]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    syms = header_symbols()
    assert {"splat_acsr_build", "splat_mask_generate", "splat_sddmm", "splat_softmax", "splat_spmm",
            "splat_attention_fwd", "splat_attention_plan_bytes", "splat_attention_plan", "splat_attention_fwd_planned", "splat_attention_fwd_stats", "splat_sddmm_probs",
            "splat_version", "splat_last_error"} <= set(syms)
    handle = ctypes.CDLL(hip.LIB_PATH)
    for s in syms:
        assert hasattr(handle, s), s
    assert sorted(hip.EXPORTS) == syms


def test_the_measurement_library_exports_what_its_header_declares():
    """libsplat_bench.so (bench.py's two ceilings) against include/splat_bench.h and its binding; and the operator header
    declares none of it."""
    import bench_probes as BP
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "splat_bench.h")).read(), flags=re.S)
    syms = sorted(set(re.findall(r"\b(splat_bench_[a-z_0-9]+)\s*\(", text)))
    assert "splat_bench_stream_copy" in syms and "splat_bench_mfma_lds_probe" in syms
    handle = ctypes.CDLL(BP.LIB_PATH)
    for s in syms:
        assert hasattr(handle, s), s
    assert sorted(BP.EXPORTS) == syms
    want = int(re.search(r"#define SPLAT_BENCH_VERSION (\d+)", open(os.path.join(ROOT, "include", "splat_bench.h")).read()).group(1))
    assert BP.lib().splat_bench_version() == want
    assert not [s for s in header_symbols() if "probe" in s or "stream_copy" in s or "bench" in s]
    assert BP.lib().splat_bench_stream_copy(None, None, 16, None) == -1 and b"null" in BP.lib().splat_bench_last_error()


def test_version_matches_header():
    want = int(re.search(r"#define SPLAT_VERSION (\d+)", open(HEADER).read()).group(1))
    assert hip.lib().splat_version() == want


def test_null_and_shape_arguments_are_rejected_without_a_device():
    lib = hip.lib()
    assert lib.splat_softmax(None, None, None, 1, 1, 1, 1, 0, 0, None) == -1
    assert b"null" in lib.splat_last_error()
    seg = (hip.AcsrSeg * 1)()
    assert lib.splat_softmax(8, 8, seg, 0, 1, 1, 1, 0, 0, None) == -2          # n_seg = 0
    assert lib.splat_softmax(8, 8, seg, 1, 1, 1, 0, 0, 0, None) == -2          # T = 0
    assert lib.splat_acsr_build(None, 4, 4, 4, 2, *([None] * 10), None) == -1
    assert lib.splat_acsr_build(8, 4, 4, 2, 2, *([8] * 7), None, None, 8, None) == -2  # ld < cols
    assert lib.splat_mask_generate(8, 4, 4, 4, 99, 1, 1, None) == -5
    assert lib.splat_attention_fwd(8, 0, 0, 64, 8, 0, 0, 1, 64, 8, 0, 0, 64, 8, 0, 0, 64, seg, 1, 1, 1, 16, 48, 1.0, 2,
                                   None) == -5                                   # d = 48 unsupported
    assert b"64 or 128" in lib.splat_last_error()
    assert lib.splat_attention_fwd_planned(8, 0, 0, 64, 8, 0, 0, 1, 64, 8, 0, 0, 64, 8, 0, 0, 64, seg, 1, 1, 1, 16, 48, 1.0, 2,
                                           16, 1 << 20, None) == -5
    assert b"splat_attention_fwd_planned" in lib.splat_last_error()
    assert lib.splat_sddmm(8, 0, 0, 8, 8, 0, 0, 3, 5, 8, seg, 1, 1, 1, 4, 4, 8, 4, 1.0, 0, 0, None) == -4  # no unit stride
    assert lib.splat_spmm(8, 8, 0, 0, 8, 8, seg, 1, 1, 1, 4, 4, 8, 4, 7, 0, None) == -3                    # bad dtype


def test_the_allocation_free_forward_rejects_what_its_built_in_buffer_cannot_hold():
    lib = hip.lib()
    seg = (hip.AcsrSeg * 2)()
    for i in range(2):
        seg[i].sTod_lin = seg[i].sTod_trans = seg[i].nnz = 8
        seg[i].row_stride_hint = 1
    fwd = lambda n_seg, L: lib.splat_attention_fwd_noalloc(8, 0, 0, 64, 8, 0, 0, 1, 64, 8, 0, 0, 64, 8, 0, 0, 64, seg, n_seg, 1, 1, L,
                                                           64, 1.0, 2, None)
    L_big = 1 << 18
    assert lib.splat_attention_plan_bytes(seg, 1, L_big) > hip.STATIC_PLAN_BYTES
    assert fwd(1, L_big) == -2
    msg = lib.splat_last_error()
    assert b"splat_attention_fwd_noalloc" in msg and b"built-in buffer" in msg and str(hip.STATIC_PLAN_BYTES).encode() in msg
    assert fwd(0, 128) == -2 and fwd(1, 0) == -2
    assert lib.splat_attention_fwd_noalloc(8, 0, 0, 64, 8, 0, 0, 1, 64, 8, 0, 0, 64, 8, 0, 0, 64, None, 1, 1, 1, 128, 64, 1.0, 2,
                                           None) == -1
    header = open(HEADER).read()
    assert int(eval(re.search(r"#define SPLAT_STATIC_PLAN_BYTES \((.*?)\)", header).group(1))) == hip.STATIC_PLAN_BYTES


def test_the_fused_backward_checks_its_arguments_on_the_host():
    """splat_attention_bwd refuses what its kernel is not built for before anything is launched."""
    lib = hip.lib()
    seg = (hip.AcsrSeg * 1)()
    seg[0].sTod_lin = seg[0].sTod_trans = seg[0].nnz = 16
    seg[0].row_stride_hint = 1
    L, d = 256, 64
    need = lib.splat_attention_plan_bytes(seg, 1, L)

    def bwd(q=16, lse=16, d=d, dtype=2, scale=1.0, plan_bytes=need, q_sl=d, seg_t=seg, B=1):
        t = [16, 0, 0, d]  # pointer, batch / head / row strides
        return lib.splat_attention_bwd(q, 0, 0, q_sl, *t, *t, *t, *t, lse, 16, 16, 16, 16, seg, 1, 16, plan_bytes,
                                       seg_t, 1, 16, need, B, 1, L, d, scale, dtype, None)
    assert bwd(q=None) == -1 and bwd(lse=None) == -1 and bwd(seg_t=None) == -1
    assert bwd(d=96) == -5 and b"64 or 128" in lib.splat_last_error()
    assert bwd(dtype=0) == -5 and b"16-bit" in lib.splat_last_error()
    assert bwd(scale=0.0) == -5
    assert bwd(q=24) == -4 and bwd(q_sl=d + 4) == -4
    assert bwd(q_sl=32) == -2
    assert bwd(plan_bytes=need - 16) == -2 and b"plan" in lib.splat_last_error()
    assert bwd(B=1 << 29) == -2 and b"too many" in lib.splat_last_error()  # two row blocks a head, two workgroups each: 2^31
    t = [16, 0, 0, d]
    assert lib.splat_attention_bwd_keys(*t, *t, *t, *t, 16, 16, 16, 16, 16, seg, 1, 16, need, 1 << 29, 1, L, 256, d, 1.0, 2, None, None, 0,
                                        None) == -2 and b"too many" in lib.splat_last_error()


def test_the_key_transpose_checks_its_arguments_on_the_host():
    lib = hip.lib()

    def tr(src=16, dst=16, L=100, d=64, sd=100, dtype=2):
        return lib.splat_transpose_keys(src, 0, 0, sd, dst, 1, 1, L, d, dtype, None)
    assert tr(src=None) == -1 and tr(dst=None) == -1
    assert tr(L=0) == -2 and tr(d=0) == -2
    assert tr(sd=99) == -2 and b"stride" in lib.splat_last_error()
    assert tr(dtype=7) == -3
    assert tr(dst=24) == -4 and tr(src=17) == -4


def test_plan_size_is_host_arithmetic():
    lib = hip.lib()
    seg = (hip.AcsrSeg * 2)()
    # per variant and segment: per 128-row block one plan record, four wavefront spans and 128 row windows of 16 bytes
    assert lib.splat_attention_plan_bytes(seg, 1, 16384) == 2 * 128 * (5 + 128) * 16
    assert lib.splat_attention_plan_bytes(seg, 2, 130) == 2 * 2 * 2 * (5 + 128) * 16
    seg[0].row_stride_hint = seg[1].row_stride_hint = 2        # rows 0, 2, 4, .. and 1, 3, 5, .. in separate blocks
    assert lib.splat_attention_plan_bytes(seg, 2, 130) == 2 * 2 * 2 * (5 + 128) * 16
    assert lib.splat_attention_plan_bytes(seg, 2, 300) == 2 * 2 * 4 * (5 + 128) * 16
    assert lib.splat_attention_plan_bytes(seg, 0, 16) == 0 and lib.splat_attention_plan_bytes(None, 1, 16) == 0
    assert lib.splat_attention_plan(seg, 1, 16, None, 0, None) == -1
    seg[0].sTod_lin = seg[0].sTod_trans = seg[0].nnz = 8
    assert lib.splat_attention_plan(seg, 1, 16, 16, 100, None) == -2 and b"bytes" in lib.splat_last_error()
    assert lib.splat_attention_plan(seg, 1, 16, 24, 1 << 20, None) == -4      # misaligned plan


def test_operators_refuse_the_host():
    import acsr_helpers as A
    import r_attention
    with pytest.raises(hip.SplatError):
        A.create_acsr(A.create_blocked_mask(10, 2), 2, "cpu")
    with pytest.raises(hip.SplatError):
        r_attention.RegularAttention(1, 16, 1, 64, A.create_causal_windowed_mask(16, 3), 16, 16, "cpu", torch.float32)
    if not torch.cuda.is_available():
        with pytest.raises(hip.SplatError):
            A.create_acsr(A.create_blocked_mask(10, 2), 2, 0)


def test_product_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "triton-fun_amd")
    for base, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".cpp", ".h")):
                text = open(os.path.join(base, f)).read()
                assert "oracle" not in text, os.path.join(base, f)


def test_spmm_looks_at_nothing_on_the_device_under_stream_capture(monkeypatch):
    """Which kernel a launch of long rows takes hangs on the plan's alignment, which comes with the plan's report: under
    capture it is taken from a plan that is there (SDDMM or the fused forward may have built it), and without one the launch
    counts as one without a table.  Neither builds a plan nor reads one back: both would wait for the stream."""
    import r_spmm
    from acsr_helpers import ACSRSegments
    L, T = 200, 300

    class Table(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            raise AssertionError(f"{func} on the plan table")
    segs = ACSRSegments([(None,) * 5 + (T, None, None)], [None])
    monkeypatch.setattr(hip, "resolve_device", lambda d: torch.device("cuda", 0))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    x, out = torch.empty(1, 1, L, T, dtype=torch.bfloat16), torch.empty(1, 1, L, 64, dtype=torch.bfloat16)
    assert segs.plan_is_aligned(L, 0) is None and not r_spmm._takes_a_plan(x, out, 64, segs)
    for aligned in (True, False, None):  # (None: a table from a file that an earlier version saved)
        segs.splat_plans = {(L, 1, (0,), 0): [torch.zeros(16, dtype=torch.uint8).as_subclass(Table), aligned]}
        assert segs.plan_is_aligned(L, 0) is aligned and r_spmm._takes_a_plan(x, out, 64, segs) == (aligned is False)


def test_the_plans_report_is_checked_before_anything_is_launched():
    lib = hip.lib()
    seg = (hip.AcsrSeg * 1)()
    assert lib.splat_attention_plan_report(seg, 1, 300, 16, 1 << 20, None, 64, None) == -1 and b"report" in lib.splat_last_error()
    assert lib.splat_attention_plan_report(seg, 1, 300, 16, 1 << 20, 24, 64, None) == -4 and b"report" in lib.splat_last_error()
    assert lib.splat_attention_plan_report(seg, 1, 300, 16, 1 << 20, 16, 47, None) == -2 and b"report needs 48" in lib.splat_last_error()
    assert lib.splat_attention_plan_report(None, 1, 300, 16, 1 << 20, 16, 48, None) == -1


def test_metadata_with_native_handles_copies_and_saves(monkeypatch):
    """The handles that a launcher call leaves with ``sTod_translations`` stay with it: a deep copy and a saved file hold the
    tensor and its plain attributes, load without executing anything, and are given handles of their own by the next call."""
    import copy
    import io
    from acsr_helpers import ACSRSegments
    t = torch.arange(4.0)
    t.splat_row_stride = 1
    arrays = [torch.zeros(4), torch.zeros(4), torch.ones(4), t, torch.ones(4)]
    monkeypatch.setattr(hip, "require_device_tensor", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)

    def native(on):
        return ACSRSegments.single(*arrays[:3], on, arrays[4], 1).native(4, torch.device("cuda", 0), False)
    without = native(t)
    t.splat_first_col = torch.zeros(4, dtype=torch.int32)
    handle = native(t)
    assert type(handle).__name__ == "PyCapsule" and native(t) is handle and handle is not without
    file = io.BytesIO()
    torch.save(t, file)
    file.seek(0)
    for other in (copy.deepcopy(t), copy.copy(t), torch.load(file, weights_only=True)):
        assert torch.equal(other, t) and other.splat_row_stride == 1
        own = native(other)
        assert type(own).__name__ == "PyCapsule" and (own is not handle or other.data_ptr() == t.data_ptr())


def test_native_entry_points_raise_what_is_thrown_in_them():
    """No C++ exception leaves an entry point of the native host path: without a device, finding the current one throws, and a call of
    any of them has to be a Python error, not the end of the process (in a process of its own for that)."""
    code = """
import os, sys
sys.path.insert(0, sys.argv[1])
import _splat_hip as hip
for name, n in (("forward", 6), ("attend", 5), ("sddmm", 6), ("softmax", 3), ("spmm", 4), ("operators", 11)):
    try:
        getattr(hip.host(), name)(*[None] * n)
        print(name, "returned")
    except Exception as e:
        print(name, "raised")
"""
    r = subprocess.run([sys.executable, "-c", code, os.path.join(ROOT, "triton-fun_amd", "SPLAT")], capture_output=True, text=True,
                       timeout=300, env={**os.environ, "HIP_VISIBLE_DEVICES": "-1"})
    assert r.returncode == 0 and r.stdout.count("raised") == 6, r.stdout + r.stderr
