"""CPU checks of the C-ABI library: it loads, exports every declared entry
point, and its host-only parts (blob format, synthetic inputs, the routing
expf, descriptor layout, error reporting) behave -- no device calls."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

import llmpager_amd as lp
import _oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "llmpager_hip.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lp_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = declared_functions()
    assert len(names) > 40
    lib = C.CDLL(lp.LIBPATH)
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_code_objects_hold_every_kernel_the_runtime_loads():
    src = open(os.path.join(ROOT, "llmpager_amd", "csrc", "lp_runtime.cpp")).read()
    specs = re.findall(r'\{"(lp_[a-z_]+\.hsaco)", "(lp_[a-z0-9_]+)"\}', src)
    assert len(specs) >= 10
    for module, kernel in specs:
        data = open(os.path.join(lp.LIBDIR, module), "rb").read()
        # an ELF code object, or hipcc's offload bundle wrapping one
        assert data[:4] == b"\x7fELF" or data.startswith(b"__CLANG_OFFLOAD_BUNDLE__")
        assert b"gfx950" in data
        assert kernel.encode() in data, (module, kernel)


def test_version_and_init_error_without_device():
    assert b"gfx950" in lp.lib().lp_version()
    ctx = C.c_void_p()
    rc = lp.lib().lp_init(0, None, C.byref(ctx))
    if rc == 0:  # a device is present: nothing to check here
        lp.lib().lp_destroy(ctx)
        pytest.skip("a GPU is present")
    assert rc != 0 and not ctx
    assert lp.lib().lp_last_error()


def test_blob_format_matches_converter():
    # convert/src/lib.rs:448-471 (H128/I64 at group 64) and decode.rs:161-185
    H, I, g = 128, 64, 64
    assert lp.blob_bytes(H, I, g) == 32 + 2 * O.q4_bytes(I, H, g) + O.q4_bytes(H, I, g)
    go, uo, do = lp.blob_offsets(H, I, g)
    assert (go, uo, do) == (32, 32 + O.q4_bytes(I, H, g), 32 + 2 * O.q4_bytes(I, H, g))
    b = lp.synth_blob(H, I, g, 1, 2, 3)
    hdr = b[:32].view(np.uint32)
    assert list(hdr) == [64, 128, 64, 128, 128, 64, 64, 0]  # lib.rs:276-281
    # config-1 shape (Qwen3-30B-A3B, H 2048, I 768, group 32): 2,654,240 B per blob
    assert lp.blob_bytes(2048, 768, 32) == 2654240
    assert lp.blob_offsets(2048, 768, 32) == (32, 884768, 1769504)


def test_synth_deterministic_and_thread_independent():
    H, I, g = 256, 128, 32
    span = 65536
    a = lp.synth_blobs(6, span, H, I, g, 0, 3, threads=1)
    b = lp.synth_blobs(6, span, H, I, g, 0, 3, threads=4)
    assert np.array_equal(a, b)
    one = lp.synth_blob(H, I, g, 0, 3, 4)
    assert np.array_equal(a[4 * span: 4 * span + one.size], one)
    assert not np.array_equal(lp.synth_blob(H, I, g, 0, 3, 5), one)
    assert np.array_equal(lp.synth_bf16(100, 0.02, 0, 7), lp.synth_bf16(100, 0.02, 0, 7))


def test_synth_distributions():
    # nibbles uniform 0..15; f16 scales |N(0, 0.02)|/8;
    # router bf16 N(0, 0.02); activations bf16 N(0, 1)
    H, I, g = 2048, 768, 32
    b = lp.synth_blob(H, I, g, 0, 0, 0)
    go, uo, do = lp.blob_offsets(H, I, g)
    ns = I * (H // g)
    sc = b[go: go + 2 * ns].view(np.float16).astype(np.float64)
    assert sc.min() >= 0
    assert abs(sc.mean() - 0.02 * np.sqrt(2 / np.pi) / 8) < 0.02 * 0.02
    nib = b[go + 2 * ns: uo]
    counts = np.bincount(np.concatenate([nib & 15, nib >> 4]), minlength=16)
    assert counts.min() > 0.98 * counts.mean() and counts.max() < 1.02 * counts.mean()
    w = lp.synth_bf16(1 << 16, 0.02, 0, 1)
    wf = (w.astype(np.uint32) << 16).view(np.float32)
    assert abs(wf.std() - 0.02) < 0.001 and abs(wf.mean()) < 0.001
    x = lp.synth_f32_bf16(1 << 16, 1.0, 0, 1)
    assert np.array_equal(x.view(np.uint32) & 0xFFFF, np.zeros_like(x.view(np.uint32)))
    assert abs(x.std() - 1) < 0.02


def test_route_expf_matches_glibc_strided():
    # Every 97th float bit pattern (44 million inputs) against libm expf.
    n = (1 << 32) // 97
    for start in range(0, n, 1 << 22):
        cnt = min(1 << 22, n - start)
        mine = lp.route_expf_sweep(start * 97, 97, cnt)
        ref = O.expf_sweep(start * 97, 97, cnt)
        same = (mine.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(mine) & np.isnan(ref))
        assert same.all(), hex(start * 97 + 97 * int(np.argmin(same)))


@pytest.mark.slow
def test_route_expf_matches_glibc_exhaustive():
    chunk = 1 << 24
    for first in range(0, 1 << 32, chunk):
        mine = lp.route_expf_sweep(first, 1, chunk)
        ref = O.expf_sweep(first, 1, chunk)
        same = (mine.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(mine) & np.isnan(ref))
        assert same.all(), hex(first + int(np.argmin(same)))


def test_layer_desc_layout_matches_header(tmp_path):
    fields = [f[0] for f in lp.LayerDesc._fields_]
    src = tmp_path / "off.c"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "llmpager_hip.h"\nint main(){'
                   + "".join(f'printf("%zu\\n", offsetof(lp_moe_layer_desc, {f}));' for f in fields)
                   + 'printf("%zu\\n", sizeof(lp_moe_layer_desc));'
                   + "".join(f'printf("%zu\\n", offsetof(lp_moe_ws_layout, {f[0]}));'
                             for f in lp.WsLayout._fields_)
                   + "return 0;}\n")
    exe = tmp_path / "off"
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    out = [int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True).stdout.split()]
    want = [getattr(lp.LayerDesc, f).offset for f in fields] + [C.sizeof(lp.LayerDesc)]
    want += [getattr(lp.WsLayout, f[0]).offset for f in lp.WsLayout._fields_]
    assert out == want


def test_ws_layout_alignment_and_size():
    d = lp.LayerDesc(hidden=2048, inter=768, experts=128, top_k=8, group=32)
    for T in (1, 8, 32, 2048):
        lay = lp.ws_layout(d, T)
        offs = [getattr(lay, f[0]) for f in lp.WsLayout._fields_[:-1]]
        assert all(o % 256 == 0 for o in offs)
        assert offs == sorted(offs)
        assert lay.total >= lay.y + T * 8 * 2048 * 4
        # the digit images of x fill their part; the bf16 images only exist
        # for the prefill GEMM (T = 2048 here)
        assert lay.sh_et - lay.xd >= T * lp.dimage_bytes(2048) > lay.sh_et - lay.xd - 256
        assert (lay.xd - lay.xf > 0) == (T == 2048)


def test_ws_layout_has_room_for_every_tile_list():
    """Batches whose experts average 16 picks go through the prefill GEMM
    whatever their size (8 experts top 2 at 64 tokens): its tile list, up to
    pairs / 128 + min(E, pairs) entries, has a part of its own."""
    for E, k in [(1, 1), (8, 2), (8, 8), (16, 4), (16, 10), (32, 8), (20, 6), (128, 8)]:
        for T in range(1, 301):
            pairs = T * k
            if pairs < 16 * min(E, pairs):
                continue
            lay = lp.ws_layout(lp.LayerDesc(hidden=256, inter=128, experts=E, top_k=k, group=32), T)
            offs = [getattr(lay, f[0]) for f in lp.WsLayout._fields_ if f[0] != "tiles"]
            assert lay.tiles not in (lay.actimg, lay.xexp), (E, k, T)
            room = min(o for o in offs if o > lay.tiles) - lay.tiles
            assert room >= 4 * (pairs // 128 + min(E, pairs)), (E, k, T)


def _align256(n):
    return (n + 255) // 256 * 256


def _decode_or_gemm_bytes(H, I, E, k, T, sI):
    """A workspace's bytes, as the sum of its parts: the routing tables, then
    the grouped kernels' buffers (act, y, the digit images of x) or the prefill
    GEMM's, and the shared MLP's."""
    ngp = lambda n: 4 * ((n // 32 + 3) // 4)
    pairs, gemm = T * k, T * k >= 16 * min(E, T * k)
    parts = [T * E * 4, pairs * 4, pairs * 4, T * 4, (E + 1) * 4, pairs * 4, pairs * 4, E * 4, 64, E * 32,
             pairs * (ngp(I) // 4 if gemm else I) * 4, pairs * H * 4, T * 64 * ngp(H) if gemm else 0, T * 76 * ngp(H),
             ((T + 3) // 4 if T <= 64 else 1) * 32 if sI else 0, T * 4 if sI else 0, T * sI * 4, T * H * 4 if sI else 0,
             (pairs // 128 + min(E, pairs) + 1) * 4 if gemm else 0, pairs * 64 * ngp(I) if gemm else 0, T * 4,
             (2 * ((T + 255) // 256) + 1) * E * 4 if T > 64 else 0]
    return sum(map(_align256, parts))


def test_ws_layout_between_decode_and_prefill_asks_for_no_more():
    """The kernels of batches above 64 tokens keep their images, exponents and
    tile list in parts that the decode kernels or the GEMM need anyway: a
    workspace holds the same bytes whichever of them run (so one made for a
    chunk of 279 to 304 tokens takes its 255-token tail), and what is in use at
    the same time does not overlap."""
    checked = 0
    for H, I, E, k, sI in [(2048, 768, 128, 8, 0), (4096, 1536, 128, 8, 0), (2048, 1408, 64, 6, 2816), (160, 96, 16, 2, 0),
                           (128, 128, 12, 1, 0), (64, 64, 300, 4, 64), (288, 544, 24, 3, 96), (256, 128, 64, 2, 352),
                           (160, 256, 64, 1, 128), (64, 2048, 1024, 16, 0), (256, 256, 64, 2, 352)]:
        go, uo, do = lp.blob_offsets(H, I, 32)
        d = lp.LayerDesc(hidden=H, inter=I, experts=E, top_k=k, group=32, gate_off=go, up_off=uo, down_off=do)
        if sI:
            d.shared_blob, d.shared_inter, d.shared_group = 1 << 32, sI, 32
            d.sh_gate_off, d.sh_up_off, d.sh_down_off = lp.blob_offsets(H, sI, 32)
        for T in list(range(1, 330)) + [511, 1100, 2048]:
            lay = lp.ws_layout(d, T)
            assert lay.total == _decode_or_gemm_bytes(H, I, E, k, T, sI), (H, I, E, k, T)
            pairs, img = T * k, 64 * 4 * ((H // 32 + 3) // 4)
            if lay.xf != lay.y or lay.act < lay.y:
                continue
            checked += 1  # routed experts by blocks of 32 tokens
            use = {"tiles": (lay.tiles, 4 * (pairs // 32 + min(E, pairs) + 1)), "exponents": (lay.act, pairs * I // 16),
                   "act": (lay.actimg, pairs * I * 4)}
            for name, (at, n) in use.items():
                for other, (at2, n2) in list(use.items()) + [("y", (lay.y, pairs * H * 4)), ("x", (lay.xf, 2 * T * img)),
                                                             ("shared", (lay.sh_et, lay.total - lay.sh_et))]:
                    assert name == other or at + n <= at2 or at2 + n2 <= at, (name, other, H, I, E, k, T)
    chunk = lp.LayerDesc(hidden=2048, inter=768, experts=128, top_k=8, group=32)
    assert checked > 500
    assert lp.ws_layout(chunk, 279).total >= lp.ws_layout(chunk, 255).total


@pytest.mark.parametrize("H,I,E,k,T,group", [
    (2048, 768, 64, 4, 96, 32),     # both projections balanced below: 6 pairs per expert
    (2048, 768, 128, 8, 81, 32),    # more token groups than CUs
    (2048, 1408, 64, 2, 65, 32),    # down one-shot: decode batches end at 64 tokens
    (4096, 1536, 64, 8, 65, 32)])
def test_mid_batches_begin_at(H, I, E, k, T, group):
    """Which kernels a batch between decode and prefill takes, as its layout
    shows it (x's images in y, the act exponents behind it)."""
    d = lp.LayerDesc(hidden=H, inter=I, experts=E, top_k=k, group=group)
    assert [(lay.xf == lay.y and lay.act > lay.y) for lay in (lp.ws_layout(d, T - 1), lp.ws_layout(d, T))] == [False, True]


def test_workspace_check_rejects_undersized_workspaces():
    """lp_moe_workspace_check, the pre-launch check of every MoE entry point
    that takes a workspace: null, misaligned and short workspaces are refused
    (a short one would be written past its end by the kernels), for one layer
    and for a stack sized by its largest layer."""
    d = lp.LayerDesc(hidden=2048, inter=768, experts=128, top_k=8, group=32, router_w=1 << 20,
                     slot_table=2 << 20, arena_base=1 << 30, slot_span=2658304,
                     gate_off=32, up_off=884768, down_off=1769504)
    for T in (1, 8, 32, 2048):
        need = lp.ws_layout(d, T).total
        ws = 1 << 32
        assert lp.workspace_check([d], T, ws, need) == 0
        assert lp.workspace_check([d], T, ws, need + 4096) == 0
        assert lp.workspace_check([d], T, ws, need - 1) == -1
        assert "needs %d" % need in lp.lib().lp_last_error().decode()
        assert lp.workspace_check([d], T, ws, 0) == -1
        assert lp.workspace_check([d], T, 0, need) == -1
        assert lp.workspace_check([d], T, ws + 16, need) == -2
    # a stack: the largest layer decides; the failing layer is named
    big = lp.LayerDesc(**{f: getattr(d, f) for f, _ in lp.LayerDesc._fields_})
    big.inter = 1536
    big.up_off, big.down_off = lp.blob_offsets(2048, 1536, 32)[1:]
    T = 32
    need = max(lp.ws_layout(x, T).total for x in (d, big))
    assert need > lp.ws_layout(d, T).total
    assert lp.workspace_check([d, big], T, 1 << 32, need) == 0
    assert lp.workspace_check([d, big], T, 1 << 32, lp.ws_layout(d, T).total) == -1
    assert lp.lib().lp_last_error().decode().startswith("layer 1:")
    # a bad descriptor is refused before the size is looked at
    bad = lp.LayerDesc(**{f: getattr(d, f) for f, _ in lp.LayerDesc._fields_})
    bad.top_k = 0
    assert lp.workspace_check([d, bad], T, 1 << 32, 1 << 40) == -2
    # the Python wrappers take the size from an allocation, or refuse
    with pytest.raises(TypeError):
        lp._ws_bytes(1 << 32, None)
    assert lp._ws_bytes(lp.DevPtr(1 << 32, 4096), None) == 4096


def _c_decl_args(text):
    """{name: argument count} of the header's function declarations."""
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    out = {}
    for m in re.finditer(r"\b(lp_[a-z0-9_]+)\s*\(([^;{]*?)\)\s*;", text, flags=re.S):
        args = m.group(2).strip()
        out[m.group(1)] = 0 if args in ("", "void") else args.count(",") + 1
    return out


def _rs_decl_args(text):
    out = {}
    for m in re.finditer(r"pub fn (lp_[a-z0-9_]+)\((.*?)\)\s*(->[^;]*)?;", text, flags=re.S):
        args = [a for a in m.group(2).split(",") if a.strip()]
        out[m.group(1)] = len(args)
    return out


def _c_struct_fields(text, name):
    body = re.search(r"typedef struct %s \{(.*?)\} %s;" % (name, name), text, flags=re.S).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    fields = []
    for decl in body.split(";"):
        decl = decl.strip()
        if not decl:
            continue
        names = decl.split(None, 1)[1] if not decl.startswith("const ") else decl.split(None, 2)[2]
        fields += [re.sub(r"[\s*]|\[.*\]", "", n) for n in names.split(",")]
    return fields


def test_rust_bindings_follow_the_header():
    """rust/llmpager-hip/src/ffi.rs declares only functions the header
    declares, and its repr(C) structs list the header's fields in order."""
    rs = open(os.path.join(ROOT, "rust", "llmpager-hip", "src", "ffi.rs")).read()
    hdr = open(HEADER).read()
    fns = set(re.findall(r"pub fn (lp_[a-z0-9_]+)\(", rs))
    assert len(fns) > 80
    assert not fns - set(declared_functions())
    # and each with the header's number of arguments
    c_args, rs_args = _c_decl_args(hdr), _rs_decl_args(rs)
    assert set(rs_args) == fns
    assert {n: rs_args[n] for n in fns} == {n: c_args[n] for n in fns}
    for st in ("lp_moe_layer_desc", "lp_moe_ws_layout", "lp_pager_config", "lp_pager_metrics", "lp_expert_handle"):
        body = re.search(r"pub struct %s \{(.*?)\n\}" % st, rs, flags=re.S).group(1)
        rs_fields = re.findall(r"pub ([a-z0-9_]+):", body)
        assert rs_fields == _c_struct_fields(hdr, st), st
