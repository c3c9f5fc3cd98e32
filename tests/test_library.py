"""CPU: the C-ABI library loads, exports every declared symbol, and validates arguments.

No call here reaches a kernel launch: every invocation fails argument
validation on the host (or is a pure size query), so no GPU is touched.
"""
import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "dflash_hip.h"


def _declared_functions():
    text = HEADER.read_text()
    return sorted(set(re.findall(r"\b(dflash_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_binding_table(pkg):
    assert _declared_functions() == sorted(pkg._lib.SIGNATURES)


def test_library_loads_and_exports_every_symbol(pkg):
    lib = pkg._lib.load()
    for name in _declared_functions():
        assert hasattr(lib, name), name
    header_abi = int(re.search(r"#define DFLASH_ABI_VERSION (\d+)", HEADER.read_text()).group(1))
    assert lib.dflash_abi_version() == pkg._lib.ABI_VERSION == header_abi


def test_integration_binding_asserts_the_current_abi():
    """The reference-side ctypes stub in INTEGRATION.md checks the ABI the header declares."""
    header_abi = int(re.search(r"#define DFLASH_ABI_VERSION (\d+)", HEADER.read_text()).group(1))
    stub = re.findall(r"dflash_abi_version\(\) == (\d+)", (ROOT / "INTEGRATION.md").read_text())
    assert stub and all(int(v) == header_abi for v in stub), stub


def test_library_has_no_unresolved_internal_symbols(pkg):
    nm = shutil.which("nm")
    if nm is None:
        pytest.skip("nm not available")
    out = subprocess.run([nm, "-D", "--undefined-only", str(pkg._lib.LIBRARY_PATH)], capture_output=True, text=True,
                         check=True).stdout
    assert "dflash" not in out, out


@pytest.mark.parametrize("compiler,lang", [("gcc", "c"), ("g++", "c++")])
def test_header_compiles_standalone(compiler, lang, tmp_path):
    exe = shutil.which(compiler)
    if exe is None:
        pytest.skip(f"{compiler} not available")
    src = tmp_path / ("probe.c" if lang == "c" else "probe.cc")
    src.write_text('#include "dflash_hip.h"\nint main(void) { dflash_w4 w; (void)w; return DFLASH_ABI_VERSION; }\n')
    subprocess.run([exe, "-x", lang, "-Wall", "-Wextra", "-Werror", "-I", str(HEADER.parent), "-fsyntax-only",
                    str(src)], check=True)


host_only = pytest.mark.skipif(
    __import__("torch").cuda.is_available(),
    reason="passes fake device pointers that must fail host validation; run only where no GPU is visible")


def _desc(pkg, experts=1, rows=512, cols=2048, group=128, dtype=0, packed=16, scales=16, layout=0):
    return pkg._lib.W4Desc(packed=packed, scales=scales, experts=experts, rows=rows, cols=cols, group_size=group,
                           scale_dtype=dtype, layout=layout)


def _status(pkg, name, *args):
    lib = pkg._lib.load()
    return getattr(lib, name)(*args), lib.dflash_last_error().decode()


@host_only
def test_qlinear_f32_validation(pkg):
    ws = ctypes.c_void_p(4096)
    st, msg = _status(pkg, "dflash_qlinear_w4a16_f32", ctypes.c_void_p(16), 16, None, ctypes.c_void_p(16), ws,
                      1 << 20, None)
    assert st == 1 and "NULL" in msg
    d = _desc(pkg, rows=48)
    st, msg = _status(pkg, "dflash_qlinear_w4a16_f32", ctypes.c_void_p(16), 16, ctypes.byref(d),
                      ctypes.c_void_p(16), ws, 1 << 20, None)
    assert st == 2 and "N % 32" in msg
    d = _desc(pkg)
    st, msg = _status(pkg, "dflash_qlinear_w4a16_f32", ctypes.c_void_p(16), 16, ctypes.byref(d),
                      ctypes.c_void_p(16), ws, 16, None)
    assert st == 3 and "workspace" in msg


@host_only
def test_qlinear_validation(pkg):
    ws = ctypes.c_void_p(4096)
    st, msg = _status(pkg, "dflash_qlinear_w4a16", ctypes.c_void_p(16), 16, None, ctypes.c_void_p(16), ws, 1 << 20, None)
    assert st == 1 and "NULL" in msg
    d = _desc(pkg, group=64)
    st, msg = _status(pkg, "dflash_qlinear_w4a16", ctypes.c_void_p(16), 16, ctypes.byref(d), ctypes.c_void_p(16), ws,
                      1 << 20, None)
    assert st == 2 and "group_size" in msg
    d = _desc(pkg, rows=48)
    st, msg = _status(pkg, "dflash_qlinear_w4a16", ctypes.c_void_p(16), 16, ctypes.byref(d), ctypes.c_void_p(16), ws,
                      1 << 20, None)
    assert st == 2 and "N % 32" in msg
    d = _desc(pkg, packed=17)
    st, msg = _status(pkg, "dflash_qlinear_w4a16", ctypes.c_void_p(16), 16, ctypes.byref(d), ctypes.c_void_p(16), ws,
                      1 << 20, None)
    assert st == 1 and "aligned" in msg
    d = _desc(pkg)
    st, msg = _status(pkg, "dflash_qlinear_w4a16", ctypes.c_void_p(16), 16, ctypes.byref(d), ctypes.c_void_p(16), ws,
                      16, None)
    assert st == 3 and "workspace" in msg
    st, _ = _status(pkg, "dflash_qlinear_w4a16", None, 0, ctypes.byref(d), None, None, 0, None)
    assert st == 0  # m == 0 is a no-op


@host_only
def test_to_tiled_validation(pkg):
    out = ctypes.c_void_p(1 << 20)
    st, msg = _status(pkg, "dflash_w4_to_tiled", None, out, out, None)
    assert st == 1 and "NULL" in msg
    d = _desc(pkg, rows=40)
    st, msg = _status(pkg, "dflash_w4_to_tiled", ctypes.byref(d), out, out, None)
    assert st == 2 and "rows % 16" in msg
    d = _desc(pkg, layout=1)
    st, msg = _status(pkg, "dflash_w4_to_tiled", ctypes.byref(d), out, out, None)
    assert st == 1 and "PORTABLE" in msg
    d = _desc(pkg, layout=5)
    st, msg = _status(pkg, "dflash_w4_to_tiled", ctypes.byref(d), out, out, None)
    assert st == 1 and "layout" in msg
    d = _desc(pkg)
    st, msg = _status(pkg, "dflash_w4_to_tiled", ctypes.byref(d), ctypes.c_void_p(16), out, None)
    assert st == 1 and "alias" in msg
    st, msg = _status(pkg, "dflash_w4_to_tiled", ctypes.byref(d), ctypes.c_void_p((1 << 20) + 8), out, None)
    assert st == 1 and "aligned" in msg


def test_from_int8_validation(pkg):
    """The int8-carried repack validates shapes, layout, dtypes and pointers before any launch."""
    v = ctypes.c_void_p(1 << 20)
    bad = ctypes.c_void_p(1 << 21)

    def call(experts=1, rows=512, cols=2048, group=256, dtype=1, layout=1, values=v, invalid=bad):
        return _status(pkg, "dflash_w4_from_int8", values, v, dtype, experts, rows, cols, group, layout, v, v,
                       invalid, None)

    st, msg = call(group=64)
    assert st == 2 and "group_size" in msg
    st, msg = call(cols=2048 + 16)
    assert st == 2 and "multiple of 32" in msg
    st, msg = call(rows=40)
    assert st == 1 and "rows % 16" in msg
    st, msg = call(layout=7)
    assert st == 1 and "layout" in msg
    st, msg = call(dtype=9)
    assert st == 1 and "scales_dtype" in msg
    st, msg = call(values=None)
    assert st == 1 and "NULL" in msg
    st, msg = call(values=ctypes.c_void_p((1 << 20) + 8))
    assert st == 1 and "alignment" in msg
    st, msg = call(experts=0)
    assert st == 1 and "positive" in msg


@host_only
def test_tiled_weights_refused_where_no_kernel_reads_them(pkg):
    """qlinear with group 256 and m > 32 has no tiled-reading kernel: status 2 before any launch."""
    ws = ctypes.c_void_p(4096)
    d = _desc(pkg, rows=64, cols=1024, group=256, layout=1)
    st, msg = _status(pkg, "dflash_qlinear_w4a16", ctypes.c_void_p(16), 33, ctypes.byref(d), ctypes.c_void_p(16), ws,
                      1 << 20, None)
    assert st == 2 and "tiled" in msg


@host_only
def test_route_validation(pkg):
    p = ctypes.c_void_p(16)
    st, msg = _status(pkg, "dflash_moe_route", p, 16, 2048, 8, p, p, p, p, p, p, 1 << 20, None)
    assert st == 2 and "experts" in msg
    st, msg = _status(pkg, "dflash_moe_route", p, 16, 256, 0, p, p, p, p, p, p, 1 << 20, None)
    assert st == 1 and "top_k" in msg
    st, msg = _status(pkg, "dflash_moe_route", p, 16, 256, 8, p, p, p, p, None, p, 1 << 20, None)
    assert st == 1 and "expert_offsets" in msg
    st, msg = _status(pkg, "dflash_moe_route", p, 16, 256, 8, p, p, p, p, p, p, 8, None)
    assert st == 3


@host_only
def test_moe_validation(pkg):
    p = ctypes.c_void_p(16)
    gu = _desc(pkg, experts=256, rows=1024, cols=2048)
    dn = _desc(pkg, experts=256, rows=2048, cols=512)
    bad_dn = _desc(pkg, experts=256, rows=2048, cols=1024)
    lib = pkg._lib.load()
    args = lambda g, d, k=8, h=2048: (p, 16, h, None, p, k, ctypes.byref(g), ctypes.byref(d), None, None, None,  # noqa: E731
                                      p, None, p, p, p, p, p, p, 1 << 30, None)
    assert lib.dflash_moe_w4a16(*args(gu, bad_dn)) == 1
    assert "down" in lib.dflash_last_error().decode()
    assert lib.dflash_moe_w4a16(*args(gu, dn, k=300)) == 1
    assert lib.dflash_moe_w4a16(*args(gu, dn, h=1000)) == 2
    shared_only_gate = (p, 16, 2048, None, p, 8, ctypes.byref(gu), ctypes.byref(dn), None, None, p,
                        p, None, p, p, p, p, p, p, 1 << 30, None)
    assert lib.dflash_moe_w4a16(*shared_only_gate) == 1
    assert "shared" in lib.dflash_last_error().decode()
    small_ws = (p, 16, 2048, None, p, 8, ctypes.byref(gu), ctypes.byref(dn), None, None, None,
                p, None, p, p, p, p, p, p, 64, None)
    assert lib.dflash_moe_w4a16(*small_ws) == 3


def test_workspace_queries(pkg):
    lib = pkg._lib.load()
    a = lib.dflash_moe_workspace_bytes(16, 2048, 512, 256, 8, 128, 1)
    b = lib.dflash_moe_workspace_bytes(2048, 2048, 512, 256, 8, 128, 1)
    assert 0 < a < b
    assert lib.dflash_moe_workspace_bytes(-1, 2048, 512, 256, 8, 128, 1) == 0
    assert lib.dflash_qlinear_workspace_bytes(16, 2048, 128) >= 16 * 2048 * 2
    assert lib.dflash_moe_route_workspace_bytes(16, 256, 8) > 0


def test_python_wrappers_refuse_cpu_tensors(pkg):
    """No CPU fallback: the HIP entry points reject host tensors before any launch."""
    import torch
    w = pkg.synthetic.int4_weight(torch.Generator().manual_seed(0), (64, 512))
    x = torch.zeros((4, 512), dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="ROCm device"):
        pkg.ops.qlinear(x, w)
    with pytest.raises(ValueError, match="ROCm device"):
        pkg.ops.route(torch.zeros((4, 16)), 2)


def test_measure_stage_validation(pkg):
    lib = pkg._lib.load()
    assert lib.dflash_set_measure_stage(7) == 1
    assert "stage" in lib.dflash_last_error().decode()
    assert lib.dflash_set_measure_stage(0) == 0


def test_tile_pieces_switch_validation(pkg):
    lib = pkg._lib.load()
    for bad in (-1, 3, 5, 8):
        assert lib.dflash_set_tile_pieces(bad) == 1
        assert "pieces" in lib.dflash_last_error().decode()
    for good in (1, 2, 4, 0):
        assert lib.dflash_set_tile_pieces(good) == 0


def test_split_down_switch_validation(pkg):
    lib = pkg._lib.load()
    assert lib.dflash_set_split_down(2) == 1
    assert "enable" in lib.dflash_last_error().decode()
    assert lib.dflash_set_split_down(1) == 0
    assert lib.dflash_set_split_down(0) == 0  # back to the default
    # the query needs no device for shapes it refuses on their arguments
    assert lib.dflash_moe_split_down(0, 2048, 512, 256, 8, 128, 1, 0, 1) == 0
    assert lib.dflash_moe_split_down(16, 1000, 512, 256, 8, 128, 1, 0, 1) == 0
    assert lib.dflash_moe_split_down(16, 2048, 512, 256, 8, 64, 1, 0, 1) == 0


def test_moe_experts_refuses_malformed_routing(pkg):
    """A caller-given routing is checked for dtype, shape, device and contiguity before its
    pointers reach the kernels (they index the work table and the weights with it)."""
    import torch
    t, e, k = 4, 16, 2
    cpu = torch.device("cpu")

    def routing(**over):
        parts = dict(ids=torch.zeros((t, k), dtype=torch.int32), weights=torch.zeros((t, k)),
                     perm=torch.arange(t * k, dtype=torch.int32), inv=torch.arange(t * k, dtype=torch.int32),
                     offsets=torch.zeros(e + 1, dtype=torch.int32))
        parts.update(over)
        return pkg.ops.Routing(**parts)

    assert pkg.ops._check_routing(routing(), t, e, cpu) == k
    bad = {
        "perm": torch.arange(t * k, dtype=torch.int64),                 # int64 permutation
        "offsets": torch.zeros(e, dtype=torch.int32),                   # one offset short
        "weights": torch.zeros((t, k), dtype=torch.bfloat16),           # not fp32
        "inv": torch.arange(2 * t * k, dtype=torch.int32)[::2],         # strided view
        "ids": torch.zeros((t + 1, k), dtype=torch.int32),              # wrong token count
    }
    for name, value in bad.items():
        with pytest.raises(ValueError, match=f"routing.{name}|routing top_k|ids"):
            pkg.ops._check_routing(routing(**{name: value}), t, e, cpu)
    with pytest.raises(ValueError, match="on meta"):
        pkg.ops._check_routing(routing(), t, e, torch.device("meta"))
    with pytest.raises(ValueError, match="top_k"):
        pkg.ops._check_routing(routing(ids=torch.zeros((t, e + 1), dtype=torch.int32)), t, e, cpu)
    with pytest.raises(ValueError, match="Routing"):
        pkg.ops._check_routing(tuple(routing()), t, e, cpu)


@host_only
def test_route_caps_tokens_times_top_k(pkg):
    """T * k above 2^28 is refused before any launch (32-bit routing offsets)."""
    p = ctypes.c_void_p(16)
    st, msg = _status(pkg, "dflash_moe_route", p, 1 << 23, 1024, 64, p, p, p, p, p, p, 1 << 40, None)
    assert st == 2 and "2^28" in msg


@host_only
def test_noalloc_refuses_oversized_layers_before_any_launch(pkg):
    """dflash_moe_w4a16_noalloc: a layer whose scratch exceeds the static array is refused on
    the host (status 2) before the array's address is even looked up."""
    p = ctypes.c_void_p(16)
    gu = _desc(pkg, experts=256, rows=1024, cols=2048)
    dn = _desc(pkg, experts=256, rows=2048, cols=512)
    lib = pkg._lib.load()
    assert lib.dflash_moe_workspace_bytes(2048, 2048, 512, 256, 8, 128, 0) > 8 << 20
    st = lib.dflash_moe_w4a16_noalloc(p, 2048, 2048, None, p, 8, ctypes.byref(gu), ctypes.byref(dn), None, None,
                                      None, p, None, p, p, p, p, p, None)
    assert st == 2 and "scratch" in lib.dflash_last_error().decode()
    # T=16 fits the static scratch: the call passes the size check and fails only for want of a
    # device (the workspace query also counts the split-K down's partial rows, which the static
    # scratch does not hold: that entry point runs the separate down launch)
    gu16 = _desc(pkg, experts=256, rows=1024, cols=2048)
    st = lib.dflash_moe_w4a16_noalloc(p, 16, 2048, None, p, 8, ctypes.byref(gu16), ctypes.byref(dn), None, None,
                                      None, p, None, p, p, p, p, p, None)
    assert st != 0 and "above the static" not in lib.dflash_last_error().decode(), lib.dflash_last_error().decode()


def test_library_serves_without_the_host_module(pkg, monkeypatch, tmp_path):
    """No dflash_host.so, a broken one, or one for another torch: one warning, then ops.py's Python form."""
    import torch
    lib = pkg._lib
    broken = tmp_path / "dflash_host.so"
    broken.write_bytes(b"not a library")
    for path, version in ((tmp_path / "missing.so", torch.__version__), (broken, torch.__version__), (lib.HOST_PATH, "0.0")):
        with monkeypatch.context() as m:
            m.setattr(lib, "_HOST", None)
            m.setattr(lib, "HOST_PATH", path)
            m.setattr(torch, "__version__", version)
            with pytest.warns(RuntimeWarning, match="not used"):
                assert lib.host() is None
            assert lib.host() is None
    assert lib.host() is not None


def test_build_goes_on_without_a_host_compiler(monkeypatch, tmp_path, capsys):
    """No g++, or a compile that fails (torch's headers missing): the kernels' library is built all the same."""
    import importlib.util
    spec = importlib.util.spec_from_file_location("_build_under_test", ROOT / "qwen3.5-35b-dflash_amd" / "build.py")
    builder = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(builder)
    monkeypatch.setenv("PATH", str(tmp_path))
    job = builder._start_host(tmp_path / "host.so")
    assert job is None and not builder._finish_host(job)
    assert not builder._finish_host(builder._start(["/bin/sh", "-c", "exit 1"]))
    assert builder._finish_host(builder._start(["/bin/sh", "-c", "exit 0"]))
    assert capsys.readouterr().err.count("is not built") == 2


def _attention_args(pkg, tokens=1, position=0, capacity=64, heads=4, kv=2, d=128, hidden=512, layout=0, **over):
    p = 1 << 20
    desc = pkg._lib.AttentionDesc(
        in_proj=_desc(pkg, rows=2 * (heads + kv) * d, cols=hidden, layout=layout), out_proj=_desc(pkg, rows=hidden, cols=heads * d, layout=layout),
        input_norm=p, post_norm=p, q_norm=p, k_norm=p, inv_freq=p, hidden_size=hidden, heads=heads, kv_heads=kv, head_dim=d,
        rotary_dim=d // 4, eps=1e-6)
    for name, value in over.items():
        setattr(desc, name, value)
    v = ctypes.c_void_p(p)
    return ctypes.byref(desc), v, tokens, position, v, v, capacity, v, v, v, 1 << 40, None


@host_only
@pytest.mark.parametrize("tokens,position,capacity", [
    (1, (1 << 63) - 1, 64), (16, (1 << 63) - 16, 64), (2, 63, 64), (1, -1, 64), (65, 0, 64), (1, 0, 1 << 25), (1, 0, -(1 << 63))])
def test_attention_block_outside_the_cache(pkg, tokens, position, capacity):
    """Refused on the host, also where position + tokens leaves 64 bits."""
    st, msg = _status(pkg, "dflash_attention_mixer", *_attention_args(pkg, tokens, position, capacity))
    assert st == 1 and "capacity" in msg


@host_only
def test_attention_token_counts_past_64_bits(pkg):
    """tokens * heads = 2^64 wraps to 0."""
    st, msg = _status(pkg, "dflash_attention_mixer", *_attention_args(pkg, 1 << 62, 0, 64))
    assert st == 2 and "2^22" in msg
    assert pkg._lib.load().dflash_attention_workspace_bytes(1 << 62, 512, 4, 2, 128) == 0


@host_only
def test_mixers_refuse_a_projection_without_a_kernel(pkg):
    """Tiled K = 4096 above 32 rows, and N that is no multiple of 32: status 2 from the host, before the norm, the cache
    rows or anything else is launched (which would report the missing device)."""
    st, msg = _status(pkg, "dflash_attention_mixer", *_attention_args(pkg, 33, 0, 64, heads=16, d=256, layout=1))
    assert st == 2 and "tiled" in msg
    st, msg = _status(pkg, "dflash_attention_mixer", *_attention_args(pkg, 1, 0, 64, heads=6, kv=3, d=128))
    assert st == 2 and "K % 512" in msg
    v = ctypes.c_void_p(1 << 20)
    for tokens, hk, hv, layout, why in ((33, 16, 32, 1, "tiled"), (1, 4, 4, 0, "N % 32"), (1, 4, 16, 0, None)):
        desc = pkg._lib.GdnDesc(
            in_proj=_desc(pkg, rows=256 * hk + 258 * hv, cols=512, layout=layout), out_proj=_desc(pkg, rows=512, cols=128 * hv, layout=layout),
            input_norm=v, post_norm=v, norm=v, a_log=v, dt_bias=v, conv=v, hidden_size=512, key_heads=hk, value_heads=hv, eps=1e-6)
        st, msg = _status(pkg, "dflash_gdn_mixer", ctypes.byref(desc), v, tokens, v, v, v, v, v, v, v, v, v, v, v, v, 16, None)
        assert (st, why in msg) == (2, True) if why else (st, "workspace" in msg) == (3, True)


@host_only
@pytest.mark.parametrize("residual,out", [(None, 16), (16, None), (24, 16), (16, 24)])
def test_moe_residual_validation(pkg, residual, out):
    """NULL or misaligned residual and sum are refused on the host."""
    p = ctypes.c_void_p(16)
    gu, dn = _desc(pkg, experts=256, rows=1024, cols=2048), _desc(pkg, experts=256, rows=2048, cols=512)
    st, msg = _status(pkg, "dflash_moe_w4a16_residual", p, 16, 2048, p, 8, ctypes.byref(gu), ctypes.byref(dn), None, None, None,
                      ctypes.c_void_p(residual), ctypes.c_void_p(out), p, p, p, p, p, p, p, 1 << 30, None)
    assert st == 1 and "residual" in msg
