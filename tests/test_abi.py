"""The C-ABI library loads without a GPU and exports every declared entry point."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def _declared_functions() -> list[str]:
    text = (ROOT / "include" / "ftx.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ftx_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_core_entry_points():
    names = _declared_functions()
    for required in ("ftx_arena_alloc", "ftx_copy_h2d", "ftx_scatter", "ftx_event_record", "ftx_last_error"):
        assert required in names


def test_library_exports_every_declared_symbol():
    from flextensor_amd import _native

    lib = _native.load()
    missing = [n for n in _declared_functions() if not hasattr(lib, n)]
    assert missing == []
    assert _native.version() == 1


def test_binding_covers_every_declared_symbol():
    from flextensor_amd import _native

    assert sorted(_native.exported_symbols()) == _declared_functions()


def test_error_path_without_device_call():
    from flextensor_amd import _native

    lib = _native.load()
    rc = lib.ftx_set_copy_policy(0, 0, 99, 0)
    assert rc == _native.FTX_ERR_INVALID
    assert b"n_copy_streams" in lib.ftx_last_error()


def test_missing_library_fails_loudly():
    """With no built library the product refuses to run: the first native call raises
    FtxLibraryMissing (an ImportError); nothing falls back to a host path or to the oracle."""
    import subprocess
    import sys

    code = (
        "from pathlib import Path\n"
        "import flextensor_amd._native as nat\n"
        "nat.LIB_PATH = Path('/nonexistent/libftx_hip.so')\n"
        "for attempt in (lambda: nat.load(), lambda: nat.checksum64(0, 0, 0),\n"
        "                lambda: nat.call('ftx_scatter', None, None, 0, None)):\n"
        "    try:\n"
        "        attempt()\n"
        "    except nat.FtxLibraryMissing as e:\n"
        "        assert isinstance(e, ImportError) and 'libftx_hip.so is missing' in str(e)\n"
        "    else:\n"
        "        raise SystemExit('a native call ran without the library')\n"
        "import sys\n"
        "assert not any(m == 'oracle' or m.startswith('oracle.') for m in sys.modules), 'oracle imported'\n"
        "print('refused')\n"
    )
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                         cwd=str(Path(__file__).resolve().parents[1]))
    assert out.returncode == 0 and out.stdout.strip().endswith("refused"), out.stdout + out.stderr


def test_arena_register_is_refused_in_c_without_the_runtime():
    """In-place page-locking is refused by the C entry point itself, for any input, before any runtime call
    (host_pinning.py:206-265 is the reference's pin_in_place it stands in for): a C caller that binds
    ``pin_in_place`` to it gets FTX_ERR_UNSUPPORTED on a box with no GPU at all."""
    import ctypes

    from flextensor_amd import _native

    lib = _native.load()
    buf = ctypes.create_string_buffer(1 << 16)
    for ptr, n in ((ctypes.addressof(buf), 1 << 16), (None, 0), (ctypes.addressof(buf), 1)):
        assert lib.ftx_arena_register(ptr, n, 0) == _native.FTX_ERR_UNSUPPORTED
        assert b"refused in this build" in lib.ftx_last_error()
    assert lib.ftx_arena_unregister(ctypes.addressof(buf)) == _native.FTX_ERR_INVALID
    with pytest.raises(_native.FtxError, match="refused in this build") as info:
        _native.arena_register(ctypes.addressof(buf), 1 << 16)
    assert info.value.code == _native.FTX_ERR_UNSUPPORTED


def test_a_per_call_copy_policy_is_checked_before_any_device_call():
    """``ftx_copy_h2d_policy`` validates the caller's policy first: out-of-range values are refused with no
    device present, and the library default is not changed by a per-call policy."""
    import ctypes

    from flextensor_amd import _native

    lib = _native.load()
    before = _native.get_copy_policy()
    for bad in (_native.copy_policy(0, 0, 0, 0), _native.copy_policy(0, 0, 9, 0), _native.copy_policy(0, 0, 1, -1),
                _native.copy_policy(0, 0, 1, (1 << 20) + 1)):
        assert lib.ftx_copy_h2d_policy(None, None, 0, _native.COPY_SDMA, ctypes.byref(bad), None) == \
            _native.FTX_ERR_INVALID
    with pytest.raises(_native.FtxError, match="n_copy_streams"):
        _native.copy_h2d(0, 0, 0, _native.COPY_AUTO, 0, _native.copy_policy(0, 0, 0, 0))
    # a valid policy and nothing to copy: done without touching a device
    _native.copy_h2d(0, 0, 0, _native.COPY_AUTO, 0, _native.copy_policy(1 << 30, 1, 8, 8))
    assert _native.get_copy_policy() == before
    p = _native.copy_policy(5, 2**64, 2, 3)  # above the 64-bit range reads as "never split"
    assert p.astuple() == (5, 2**64 - 1, 2, 3) and p == _native.copy_policy(5, 2**64 - 1, 2, 3)


def _run_python(code: str) -> "subprocess.CompletedProcess":
    import subprocess
    import sys

    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                          cwd=str(ROOT))


def test_shutdown_is_idempotent_and_refuses_later_work():
    """``ftx_shutdown`` (core/transfer.py:133-142: synchronize, then refuse further work) releases the
    library's own resources once; a second call is a no-op; afterwards calls that would start work or
    allocate fail with FTX_ERR_UNSUPPORTED and a message, and calls that release handles still succeed.
    Run in a child process: a shut-down library stays shut down for the rest of its process."""
    code = (
        "import ctypes\n"
        "import flextensor_amd._native as nat\n"
        "lib = nat.load()\n"
        "src, dst = ctypes.create_string_buffer(8 << 20), ctypes.create_string_buffer(8 << 20)\n"
        "nat.host_memcpy(ctypes.addressof(dst), ctypes.addressof(src), 8 << 20)  # starts the host thread pool\n"
        "assert lib.ftx_shutdown() == 0 and lib.ftx_shutdown() == 0\n"
        "nat.shutdown()\n"
        "refused = {\n"
        "  'host_memcpy': lib.ftx_host_memcpy(ctypes.addressof(dst), ctypes.addressof(src), 64),\n"
        "  'copy_h2d': lib.ftx_copy_h2d(None, None, 0, 0, None),\n"
        "  'arena_alloc': lib.ftx_arena_alloc(4096, 0, ctypes.byref(ctypes.c_void_p())),\n"
        "  'event_create': lib.ftx_event_create(0, ctypes.byref(ctypes.c_void_p())),\n"
        "  'scatter': lib.ftx_scatter(None, None, 0, None),\n"
        "  'fp8_linear': lib.ftx_fp8_linear(None, None, None, None, 0, 0, 0, None, 0, None),\n"
        "}\n"
        "assert all(rc == nat.FTX_ERR_UNSUPPORTED for rc in refused.values()), refused\n"
        "assert b'shut down' in lib.ftx_last_error()\n"
        "released = [lib.ftx_event_destroy(None), lib.ftx_stream_destroy(None), lib.ftx_arena_free(None),\n"
        "            lib.ftx_device_free(None), lib.ftx_scatter_plan_destroy(None)]\n"
        "assert released == [0] * 5, released\n"
        "print('shut down')\n"
    )
    out = _run_python(code)
    assert out.returncode == 0 and out.stdout.strip() == "shut down", out.stdout + out.stderr


def test_exit_releases_the_library_quietly():
    """At interpreter exit the binding calls ``ftx_shutdown`` ahead of torch's exit handlers: a process whose
    host thread pool is running exits with status 0 and nothing on stderr. Exit handlers run last-registered
    first, so a probe registered before the binding is imported runs after its shutdown (and is refused),
    and one registered after it runs before (and still works)."""
    code = (
        "import atexit, ctypes\n"
        "held = {}\n"
        "def probe(when):\n"
        "    rc = held['lib'].ftx_host_memcpy(ctypes.addressof(held['dst']), ctypes.addressof(held['src']), 64)\n"
        "    print(when, 'refused' if rc == 4 else 'live', flush=True)\n"
        "atexit.register(probe, 'after')\n"
        "import flextensor_amd._native as nat\n"
        "held['lib'] = nat.load()\n"
        "held['src'], held['dst'] = ctypes.create_string_buffer(32 << 20), ctypes.create_string_buffer(32 << 20)\n"
        "nat.host_memcpy(ctypes.addressof(held['dst']), ctypes.addressof(held['src']), 32 << 20)\n"
        "atexit.register(probe, 'before')\n"
    )
    out = _run_python(code)
    assert out.returncode == 0 and out.stderr == "", out.stderr
    assert out.stdout.split() == ["before", "live", "after", "refused"], out.stdout


def test_event_flags_are_checked_before_the_runtime():
    """``ftx_event_create`` takes FTX_EVENT_TIMING and FTX_EVENT_DEVICE_ONLY; any other bit is refused on the
    host, with no device involved."""
    import ctypes

    from flextensor_amd import _native

    lib = _native.load()
    ev = ctypes.c_void_p()
    for bad in (4, 8, 0x20000000, 0x80000003):
        assert lib.ftx_event_create(bad, ctypes.byref(ev)) == _native.FTX_ERR_INVALID
        assert b"unknown event flags" in lib.ftx_last_error()
    assert (_native.EVENT_TIMING, _native.EVENT_DEVICE_ONLY) == (1, 2)


def test_layer_entry_points_refuse_bad_shapes_before_any_device_call():
    """Head dimensions, head groups, empty keys, alignment of sizes and strides beyond any memory are refused on
    the host, with no device present."""
    import ctypes

    from flextensor_amd import _native as nat

    lib = nat.load()
    b = ctypes.c_size_t(0)
    for shape, code in (((1, 1, 8, 4, 4, 96), nat.FTX_ERR_UNSUPPORTED), ((1, 1, 8, 4, 3, 64), nat.FTX_ERR_INVALID),
                        ((1, 1, 0, 4, 4, 64), nat.FTX_ERR_INVALID), ((-1, 1, 8, 4, 4, 64), nat.FTX_ERR_INVALID)):
        assert lib.ftx_attention_workspace(*shape, ctypes.byref(b)) == code
    assert lib.ftx_attention_workspace(0, 1, 8, 4, 4, 64, ctypes.byref(b)) == nat.FTX_OK and b.value == 0
    big = (ctypes.c_int64 * 12)(*[1 << 62] * 12)
    assert lib.ftx_attention(None, None, None, None, 2, 2, 8, 4, 4, 64, big, 0, 0, 1.0, None, 0, None) == \
        nat.FTX_ERR_INVALID
    assert lib.ftx_attention(None, None, None, None, 2, 2, 8, 4, 4, 64, big, 0, 0, 0.0, None, 0, None) == \
        nat.FTX_ERR_INVALID
    assert lib.ftx_rope_cache(None, None, None, None, None, None, None, None, 1, 1, 4, 4, 24, 0, big, None) == \
        nat.FTX_ERR_UNSUPPORTED
    assert lib.ftx_rope_cache(None, None, None, None, None, None, None, None, 2, 2, 4, 4, 64, 1 << 29, big, None) == \
        nat.FTX_ERR_INVALID
    assert lib.ftx_norm(None, None, None, None, 4, 12, nat.NORM_RMS, None, None, None, None, 1, -1, -1, -1, 1e-5,
                        None) == nat.FTX_ERR_UNSUPPORTED
    assert lib.ftx_silu_mul(None, None, None, 12, None) == nat.FTX_ERR_UNSUPPORTED
    n = (ctypes.c_int64 * 1)(64)
    ptr = (ctypes.c_void_p * 1)(None)
    assert lib.ftx_bf16_linear(None, 1, ptr, ptr, n, 17, 64, 0, None, None) == nat.FTX_ERR_UNSUPPORTED
    assert lib.ftx_bf16_linear(None, 1, ptr, ptr, n, 4, 12, 0, None, None) == nat.FTX_ERR_INVALID


def test_layer_size_limits_hold_where_the_product_of_sizes_wraps():
    """Sizes within each limit whose product is 2^64 are refused as the smaller ones beyond the limit are."""
    import ctypes

    from flextensor_amd import _native as nat

    lib = nat.load()
    b = ctypes.c_size_t(0)
    for t in (1 << 10, 1 << 24):
        assert lib.ftx_attention_workspace(1 << 24, t, 8, 65536, 65536, 64, ctypes.byref(b)) == nat.FTX_ERR_INVALID
        assert b"too large" in lib.ftx_last_error()
    for t in (1 << 12, 1 << 24):  # batch * t * (heads + 2 kv_heads) * d is a multiple of 2^64 for the second
        assert lib.ftx_rope_cache(None, None, None, None, None, None, None, None, 1 << 24, t, 32768, 16384, 1 << 12, 0,
                                  None, None) == nat.FTX_ERR_INVALID
        assert b"too large" in lib.ftx_last_error()


def test_launches_beyond_the_threads_of_a_grid_are_refused_or_planned_otherwise():
    """A launch holds fewer than 2^32 threads: the layer entry points refuse more before any operand is looked at,
    and an fp8 linear of that many channels keeps the split-K kernel (whose workspace shows it)."""
    import ctypes

    from flextensor_amd import _native as nat

    lib = nat.load()
    b = ctypes.c_size_t(0)
    assert lib.ftx_attention_workspace(1 << 24, 1, 8, 64, 64, 64, ctypes.byref(b)) == nat.FTX_ERR_UNSUPPORTED
    assert lib.ftx_attention_workspace(1 << 19, 1, 8, 64, 64, 64, ctypes.byref(b)) == nat.FTX_OK
    for rows, dim in ((1 << 26, 2048), (1 << 24, 8192), (1 << 22, 32768)):
        assert lib.ftx_norm(None, None, None, None, rows, dim, nat.NORM_RMS, None, None, None, None, 1, -1, -1, -1,
                            1e-5, None) == nat.FTX_ERR_UNSUPPORTED
    assert lib.ftx_silu_mul(None, None, None, 1 << 35, None) == nat.FTX_ERR_UNSUPPORTED
    ptr = (ctypes.c_void_p * 1)(None)
    n = (ctypes.c_int64 * 1)(1 << 27)
    assert lib.ftx_bf16_linear(None, 1, ptr, ptr, n, 4, 64, 0, None, None) == nat.FTX_ERR_UNSUPPORTED
    for channels, split in ((1 << 26, False), (1 << 28, True)):
        n[0] = channels
        assert lib.ftx_fp8_linear_scratch(4, n, 1, 8192, 0, ctypes.byref(b)) == nat.FTX_OK and (b.value > 0) == split


def test_static_scratch_refusal_names_the_workspace_it_is_measured_by():
    import ctypes

    from flextensor_amd import _native as nat

    lib = nat.load()
    b, touched = ctypes.c_size_t(0), ctypes.c_size_t(0)
    m, n, k = 64, 28672, 8192
    assert lib.ftx_fp8_linear_workspace(m, n, k, ctypes.byref(b)) == nat.FTX_OK
    assert lib.ftx_fp8_linear_scratch(m, (ctypes.c_int64 * 1)(n), 1, k, 0, ctypes.byref(touched)) == nat.FTX_OK
    assert touched.value < 64 << 20 < b.value
    assert lib.ftx_fp8_linear_static(None, None, None, None, m, n, k, None) == nat.FTX_ERR_UNSUPPORTED
    assert f"ftx_fp8_linear_workspace, {b.value} bytes" in lib.ftx_last_error().decode()


@pytest.mark.parametrize("m,n,k,one_launch", [
    (1, 65536, 2048, True), (1, 65552, 2048, False), (3, 39935, 2048, True), (3, 39936, 2048, False),
    (8, 8192, 512, True), (8, 8193, 512, False), (1, 28671, 1024, True), (1, 28672, 1024, False),
    (8, 131072, 5120, True), (4, 65536, 4096, False), (4, 1024, 11008, True), (4, 512, 11008, False),
    (1, 2048, 16384, True), (1, 1024, 16384, False), (4, 4096, 28672, True), (5, 4096, 28672, False),
    (9, 8192, 4096, True), (9, 8193, 4096, False), (16, 12288, 2048, True), (16, 32768, 1024, False),
    (16, 4096, 11008, True), (16, 1024, 11008, False), (17, 64, 64, False)])
def test_few_row_fp8_calls_take_the_kernel_measured_faster(m, n, k, one_launch):
    """Under an epilogue every call but a one-launch one goes through partial sums, which shows the choice."""
    import ctypes

    from flextensor_amd import _native as nat

    b = ctypes.c_size_t(0)
    nat.call("ftx_fp8_linear_scratch", m, (ctypes.c_int64 * 1)(n), 1, k, nat.FP8_EPILOGUE_RESIDUAL, ctypes.byref(b))
    assert (b.value == 0) == one_launch
