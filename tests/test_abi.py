"""The C-ABI library loads without a GPU and exports every entry point the
header declares; the Python binding table matches the header."""
import ctypes as C
import re
from pathlib import Path

from qw3_amd import _native

ROOT = Path(__file__).resolve().parent.parent


def test_header_symbols_exported():
    lib = C.CDLL(str(_native.LIB_DIR / "libds3_hip.so"))
    names = _native.header_functions()
    assert len(names) >= 40
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_binding_table_covers_header():
    assert sorted(_native.SIGNATURES) == _native.header_functions()


def test_every_declaration_cites_the_reference():
    """Each ds3_metal.h replacement sits under a comment citing the reference
    declaration it replaces; the extensions section says it has none."""
    text = (ROOT / "include" / "ds3_hip.h").read_text()
    head, ext = text.split("Device-routed extensions")
    lines = head.splitlines()
    last_cite = -100
    for i, line in enumerate(lines):
        if "reference src/ds3_metal.h" in line:
            last_cite = i
        for name in re.findall(r"\b(ds3_hip_\w+)\s*\(", line):
            assert i - last_cite <= 14, f"{name} has no nearby reference citation"
    assert "no ds3_metal.h counterpart" in ext.splitlines()[0]


def test_generator_exports():
    lib = C.CDLL(str(_native.LIB_DIR / "libds3gen.so"))
    for n in _native.GEN_SIGNATURES:
        assert hasattr(lib, n)


def test_compat_header_maps_every_metal_name():
    """Every replacement of a ds3_metal.h entry point (the header part before
    the extensions section) has its ds3_metal_* alias."""
    compat = (ROOT / "include" / "ds3_metal_compat.h").read_text()
    head = (ROOT / "include" / "ds3_hip.h").read_text().split("Device-routed extensions")[0]
    names = sorted(set(re.findall(r"\b(ds3_hip_\w+)\s*\(", head)))
    assert len(names) >= 30
    for name in names:
        metal = name.replace("ds3_hip_", "ds3_metal_")
        assert f"#define {metal} {name}" in compat, metal


def test_capture_refusals(capfd):
    """While a graph capture is open, every entry point that would allocate,
    copy from or to the host or wait refuses with a diagnostic instead of
    breaking the capture.  The capture is simulated (no device here); the
    refusals come before any device or buffer access, so zeroed stand-in
    handles are enough."""
    lib = C.CDLL(str(_native.LIB_DIR / "libds3_hip.so"))
    _native._bind(lib, _native.SIGNATURES)
    if lib.ds3_hip_debug_simulate_capture(1) != 0:
        import pytest
        pytest.skip("a device context is open in this process")
    fake = C.create_string_buffer(64)            # a zeroed ds3_hip_buffer_t stand-in
    fp = C.cast(fake, C.c_void_p)
    data = C.create_string_buffer(4096)
    idx = (C.c_int32 * 8)(*range(8))
    sc = (C.c_float * 8)(*([0.125] * 8))
    try:
        assert lib.ds3_hip_buffer_alloc(4096) is None
        assert lib.ds3_hip_buffer_from_mmap(C.cast(data, C.c_void_p), 4096) is None
        assert lib.ds3_hip_buffer_write(fp, 0, C.cast(data, C.c_void_p), 0) == -1
        assert lib.ds3_hip_buffer_read(fp, 0, C.cast(data, C.c_void_p), 0) == -1
        assert lib.ds3_hip_moe_ffn_experts(fp, fp, fp, fp, 12, 12, 14, 1152, 1152, 630, None, None, None, 0, 0, 0,
                                           0, 0, 0, fp, None, fp, fp, 2048, 8, 768, 0,
                                           idx, sc) == -1
        assert lib.ds3_hip_router_stats(None, None, 0) == -1
        assert lib.ds3_hip_timer_start() == -1
        assert lib.ds3_hip_graph_launch(fp) == -1
        lib.ds3_hip_synchronize()
        lib.ds3_hip_end_batch()
    finally:
        assert lib.ds3_hip_debug_simulate_capture(0) == 0
    err = capfd.readouterr().err
    for what in ("buffer_alloc", "buffer_from_mmap", "buffer_write", "buffer_read", "moe_ffn_experts",
                 "router_stats", "timer_start", "graph_launch"):
        assert f"{what}" in err and "not allowed during graph capture" in err, what
    assert err.count("not allowed during graph capture") >= 8


def product_plan(t, M, N, K, pad=0, offset=0):
    """(kernel, grid x, grid y, threads, tile, order) that a dense product takes."""
    lib = _native._bind(C.CDLL(str(_native.LIB_DIR / "libds3_hip.so")), _native.SIGNATURES)
    plan = (C.c_int64 * 6)()
    per, nbytes = {12: (256, 144), 14: (256, 210), 8: (32, 34)}[t]
    assert lib.ds3_hip_debug_product_plan(t, M, N, K, K // per * nbytes + pad, offset, plan) == 0, (t, M, N, K)
    return tuple(plan)


def test_product_grids_fit_a_launch():
    """A launch takes fewer than 2^32 threads in x and 2^16 workgroups in y: every
    product whose operands 288 GB can hold has a kernel whose grid fits."""
    for t in (12, 14, 8):
        for K in (256, 512, 1024, 2048, 4096):
            for N in (1, 2048, (1 << 27) - 16, 1 << 27, (1 << 27) + 1, 1 << 28, 1 << 29, 1 << 30):
                for M in (1, 2, 40, 1000):
                    if N * K // 256 * {12: 144, 14: 210, 8: 272}[t] + 4 * M * N > 288e9:
                        continue
                    kernel, gx, gy, threads, _, _ = product_plan(t, M, N, K, pad=8)
                    assert gx * threads < 1 << 32 and gy < 1 << 16, (t, M, N, K, kernel, gx, gy, threads)


def test_product_kernel_choice():
    """The fp32 product kernel at sizes on both sides of each line of the
    dispatch: where the matrix-core kernel (2) measured slower than the general
    one (0), the call keeps the general one."""
    q4, q6, q8 = 12, 14, 8
    want = {
        (q6, 1, 8192, 512): 0, (q6, 1, 12288, 512): 2, (q4, 1, 8192, 512): 0, (q4, 1, 12288, 512): 2,
        (q8, 1, 2048, 512): 2, (q8, 1, 2047, 512): 0, (q4, 1, 2048, 1024): 2, (q6, 1, 2048, 1024): 0,
        (q6, 1, 2560, 1024): 2, (q6, 1, 4096, 1536): 2, (q6, 1, 8192, 1536): 0, (q6, 1, 100000, 1536): 0,
        (q4, 1, 100000, 1536): 2, (q6, 1, 2048, 8192): 0, (q6, 1, 4096, 8192): 2, (q8, 1, 32000, 768): 0,
        (q4, 2, 768, 256): 0, (q4, 2, 12288, 256): 2, (q6, 2, 12288, 256): 0, (q6, 2, 24000, 256): 2,
        (q8, 2, 64, 256): 2, (q6, 2, 32000, 1280): 0, (q6, 2, 8192, 1280): 2, (q4, 2, 32000, 1280): 2,
        (q6, 2, 2048, 768): 2, (q4, 3, 64, 256): 2, (q6, 3, 32000, 1280): 2, (q8, 8, 300, 288): 0,
        (q4, 63, 768, 2048): 2, (q4, 64, 768, 2048): 3, (q4, 64, 768, 768): 2, (q6, 64, 700, 2048): 2,
    }
    got = {k: product_plan(*k, pad=2)[0] for k in want}
    assert got == want
    # dense rows of 2048 and 4096 from a 16-byte boundary run on the one-token kernel
    assert [product_plan(q6, 1, 2048, 2048)[0], product_plan(q6, 1, 2048, 2048, offset=8)[0],
            product_plan(q4, 1, 17, 4096)[0], product_plan(q4, 1, 17, 4096, pad=16)[0]] == [1, 0, 1, 0]
    # the fp16 product's tile order: the larger operand's tiles vary slowest (A 2 bytes a
    # weight, W 0.5625 in Q4_K and 1.0625 in Q8_0)
    assert [product_plan(t, M, N, 512)[5] for t, M, N in ((q4, 4096, 4096), (q4, 4096, 5120), (q4, 512, 16384),
                                                         (q8, 1000, 8192), (q8, 3000, 4096), (q4, 512, 4096))] == \
        [1, 1, 0, 0, 1, 0]
