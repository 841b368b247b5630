"""The C-ABI library on the CPU: it loads, exports every function include/nt/nt.h declares,
its struct layouts match the ctypes mirror, and its host-only helpers and argument checks
work (no kernel is launched: every call here fails validation before touching HIP)."""
import ctypes as C
import os
import re
import subprocess
import tempfile

import numpy as np
import pytest

import neural_textures_amd as nt
from neural_textures_amd import abi, params as P

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "nt", "nt.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(nt_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(nt.LIBRARY_PATH):
        pytest.fail("libnt_hip.so is not built (run __graft_entry__.build())")
    return nt.load()


def test_exports_every_declared_function(lib):
    names = declared_functions()
    assert len(names) >= 17
    out = subprocess.run(["nm", "-D", "--defined-only", nt.LIBRARY_PATH], capture_output=True,
                         text=True, check=True).stdout
    exported = set(re.findall(r" T (nt_\w+)", out))
    assert set(names) <= exported, set(names) - exported
    assert set(names) == set(abi.SIGNATURES), "abi.py and nt.h disagree"


def test_struct_layout_matches_c():
    structs = {"nt_adam": abi.nt_adam, "nt_grid": abi.nt_grid, "nt_latents": abi.nt_latents,
               "nt_mlp": abi.nt_mlp, "nt_texture": abi.nt_texture, "nt_params": abi.nt_params,
               "nt_codec_grid": abi.nt_codec_grid, "nt_decode_params": abi.nt_decode_params,
               "nt_model_info": abi.nt_model_info, "nt_model_data": abi.nt_model_data}
    lines = ['#include <stdio.h>', '#include <stddef.h>', f'#include "{HEADER}"', "int main(void){"]
    for name, cls in structs.items():
        lines.append(f'printf("{name} %zu\\n", sizeof({name}));')
        for fname, _ in cls._fields_:
            lines.append(f'printf("{name}.{fname} %zu\\n", offsetof({name}, {fname}));')
    lines.append("return 0;}")
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "l.c"), os.path.join(d, "l")
        open(src, "w").write("\n".join(lines))
        subprocess.run(["gcc", "-o", exe, src], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    got = dict(line.rsplit(" ", 1) for line in out.strip().splitlines())
    for name, cls in structs.items():
        assert int(got[name]) == C.sizeof(cls), name
        for fname, _ in cls._fields_:
            assert int(got[f"{name}.{fname}"]) == getattr(cls, fname).offset, f"{name}.{fname}"


def test_layout_helpers(lib):
    offs = (C.c_int64 * 16)()
    for w, h, m in [(512, 512, 8), (1024, 256, 11), (3, 5, 3), (1, 1, 1)]:
        total = lib.nt_mip_chain_layout(w, h, m, offs)
        want, wt = P.mip_chain_layout(w, h, m)
        assert total == wt and list(offs)[:m] == want
        total = lib.nt_block_chain_layout(w, h, m, offs)
        want, wt = P.block_chain_layout(w, h, m)
        assert total == wt and list(offs)[:m] == want
        for c in (4, 8, 16):
            total = lib.nt_codec_mip_chain_layout(w, h, m, c, offs)
            want, wt = P.codec_chain_layout(w, h, m, c)
            assert total == wt and list(offs)[:m] == want
    assert lib.nt_mip_chain_layout(0, 4, 1, offs) == -1
    assert lib.nt_codec_block_bytes(16) == 192 and lib.nt_codec_block_bytes(3) == 0
    assert lib.nt_abi_version() == abi.NT_ABI_VERSION
    assert lib.nt_status_string(abi.NT_ERR_WORKSPACE) == b"workspace too small"


def _state():
    from helpers import make_state
    return make_state("c2", image=64, region=(32, 16))


def test_argument_errors_enqueue_nothing(lib):
    st = _state()
    p = st.params()
    assert lib.nt_train_step(None, 0, None) == abi.NT_ERR_NULL_POINTER
    assert lib.nt_train_step(C.byref(p), 7, None) == abi.NT_ERR_INVALID_ARGUMENT
    bad = st.params()
    bad.mlp.sizes[1] = 48
    assert lib.nt_train_step(C.byref(bad), 0, None) == abi.NT_ERR_UNSUPPORTED
    assert b"no kernel is built" in lib.nt_last_error()
    bad = st.params()
    bad.latents.channels = 8
    assert lib.nt_train_step(C.byref(bad), 0, None) == abi.NT_ERR_UNSUPPORTED
    bad = st.params()
    bad.latents.grids[0].values = None
    assert lib.nt_train_step(C.byref(bad), 0, None) == abi.NT_ERR_NULL_POINTER
    bad = st.params()
    bad.num_samples = 0
    assert lib.nt_train_step(C.byref(bad), 0, None) == abi.NT_ERR_INVALID_ARGUMENT
    need = lib.nt_train_workspace_bytes(C.byref(p), 0)
    assert need > 0
    assert lib.nt_train_step(C.byref(p), 0, None) == abi.NT_ERR_WORKSPACE
    ws = np.zeros(need // 4 + 8, np.float32)
    small = st.params()
    small.workspace, small.workspace_bytes = C.c_void_p(ws.ctypes.data), need - 4
    assert lib.nt_train_step(C.byref(small), 0, None) == abi.NT_ERR_WORKSPACE
    misaligned = st.params()
    misaligned.latents.grids[0].values = C.cast(st.grids[0].values.ctypes.data + 4, abi.f32p)
    assert lib.nt_train_step(C.byref(misaligned), 0, None) == abi.NT_ERR_MISALIGNED
    assert lib.nt_optimize_latents(C.byref(p), 9, None) == abi.NT_ERR_INVALID_ARGUMENT
    bad = st.params()
    bad.mlp.weight_moment1[0] = None
    assert lib.nt_optimize_network(C.byref(bad), None) == abi.NT_ERR_NULL_POINTER
    assert lib.nt_inference(C.byref(p), None) == abi.NT_ERR_NULL_POINTER  # no output buffers
    assert lib.nt_codec_encode(None, 4, 4, 16, None, None) == abi.NT_ERR_NULL_POINTER
    buf = np.zeros(64, np.float32)
    assert lib.nt_codec_encode(buf.ctypes.data, 4, 4, 3, buf.ctypes.data, None) == abi.NT_ERR_INVALID_ARGUMENT
    assert lib.nt_mlp_forward(None, None, None, 1, None) == abi.NT_ERR_NULL_POINTER
    assert lib.nt_bc6_init(None, None) == abi.NT_ERR_NULL_POINTER
    lat = st.params().latents  # no block_params
    assert lib.nt_bc6_init(C.byref(lat), None) == abi.NT_ERR_NULL_POINTER
    lat.channels = 5
    assert lib.nt_bc6_init(C.byref(lat), None) == abi.NT_ERR_UNSUPPORTED
    lat = st.params().latents
    lat.grids[0].width = 6
    assert lib.nt_bc6_init(C.byref(lat), None) == abi.NT_ERR_INVALID_ARGUMENT
    with pytest.raises(nt.NtError) as e:
        nt.check(lib.nt_decode(None, None))
    assert e.value.status == abi.NT_ERR_NULL_POINTER


@pytest.mark.parametrize("margins", [None, "0"])
@pytest.mark.parametrize("shape,ng", [("c2", 2), ("c4", 1)])
def test_config_shapes_plan_the_16_channel_kernel(lib, shape, ng, margins):
    """The BASELINE config 2 / 4 shapes (grid-to-image ratios, textures, MLP) must be planned
    on the 16-channel train kernel: its LDS layout has to fit. That plan's workspace is
    exactly one gradient partial row per 64 x 8*groups tile (no prepared weight image), which
    tells it apart from the generic kernel's."""
    from helpers import make_state
    assert lib.nt_set_test_hooks(0, 1 if margins else 0) == 0
    try:
        st = make_state(shape, image=256, region=(64, 64))
        p = st.params()
        sizes = list(st.net.sizes)
        pads = [abi.pad16(s) for s in sizes]
        P_total = sum(pads[l + 1] * pads[l] + pads[l + 1] for l in range(len(sizes) - 1))
        tiles = (64 // 64) * (64 // (8 * ng))
        assert lib.nt_train_workspace_bytes(C.byref(p), 0) == tiles * P_total * 4
    finally:
        assert lib.nt_set_test_hooks(0, 0) == 0


def _need(lib, st, ktype=0):
    need = lib.nt_train_workspace_bytes(C.byref(st.params()), ktype)
    assert need > 0, lib.nt_last_error()
    return need


def _region(st, w, h, update=abi.NT_LATENT_DENSE):
    st.region_width, st.num_samples, st.latent_update = w, w * h, update
    return st


@pytest.mark.parametrize("shape", ["c2", "c4", "ref16", "ref16f"])
@pytest.mark.parametrize("update,blocks", [(abi.NT_LATENT_DENSE, False), (abi.NT_LATENT_TOUCHED, False),
                                           (abi.NT_LATENT_DENSE, True)])
def test_workspace_grows_with_the_region(lib, shape, update, blocks):
    """A workspace sized for a region holds every smaller one's step: the bytes never fall as a
    region grows in width or height, whatever tiles each size takes."""
    from helpers import make_state
    st = make_state(shape, image=256, blocks=blocks)
    ktype = abi.NT_BLOCK_FEATURES if blocks else abi.NT_UNCONSTRAINED
    sizes = [1, 15, 16, 17, 33, 64, 65, 100, 160, 161, 208, 255, 256, 331, 400, 509, 512, 700, 1024]
    need = np.array([[_need(lib, _region(st, w, h, update), ktype) for h in sizes] for w in sizes])
    assert np.all(np.diff(need, axis=0) >= 0) and np.all(np.diff(need, axis=1) >= 0)


@pytest.mark.parametrize("shape", ["c2", "c4"])
def test_workspace_grows_with_random_samples(lib, shape):
    """The same for random texels: over sample counts (groups, tile widths, sort) at each image
    size, and over image sizes from the sort's least count up."""
    from helpers import make_state
    st = make_state(shape, image=256)
    st.sample_mode = abi.NT_SAMPLES_RANDOM
    counts = [1, 127, 128, 129, 4096, 16384, 32767, 32768, 32769, 65535, 65536, 65537, 100000, 262143, 262144, 262145,
              266241, 1 << 20, (1 << 20) + 1, 3 << 20]
    need = []
    for image in (64, 512, 1448, 2048, 4096, 8192, 16384, 20000):
        st.image_width = st.image_height = image
        for t in st.textures:
            t.width = t.height = image
        need.append([_need(lib, _region(st, n, 1)) for n in counts])
    need = np.array(need)
    assert np.all(np.diff(need, axis=1) >= 0)
    assert np.all(np.diff(need[:, counts.index(65536):], axis=0) >= 0)


@pytest.mark.parametrize("shape,ng,w,h,mode,blocks", [
    ("c2", 2, 509, 331, abi.NT_SAMPLES_REGION, False), ("c4", 1, 300, 217, abi.NT_SAMPLES_REGION, False),
    ("ref16", 2, 509, 331, abi.NT_SAMPLES_REGION, False), ("c4", 1, 256, 256, abi.NT_SAMPLES_REGION, True),
    ("c2", 2, 16384, 1, abi.NT_SAMPLES_RANDOM, False), ("c4", 2, 100000, 1, abi.NT_SAMPLES_RANDOM, False),
])
def test_workspace_of_wide_tiles_is_enough(lib, shape, ng, w, h, mode, blocks):
    """A step is not refused for want of the speed-only scratch (rows of narrow tiles, the sort
    of fewer than 262,144 samples): a row per workgroup of four-chunk tiles is enough, 16 bytes
    less is not. The argument after the workspace in nt_train_iteration's checks is invalid, so
    nothing is launched."""
    from helpers import make_state
    st = _region(make_state(shape, image=256, blocks=blocks), w, h)
    st.sample_mode = mode
    ktype = abi.NT_BLOCK_FEATURES if blocks else abi.NT_UNCONSTRAINED
    pads = [abi.pad16(s) for s in st.net.sizes]
    row = 4 * sum(pads[l + 1] * pads[l] + pads[l + 1] for l in range(len(pads) - 1))
    tiles = -(-w // (512 * ng)) if mode == abi.NT_SAMPLES_RANDOM else -(-w // 64) * -(-h // (8 * ng))
    least = min(tiles, 256) * row
    if blocks:
        least = -(-least // 256) * 256 + sum(2 * -(-g.width * g.height * g.channels * 4 // 256) * 256 for g in st.grids)
    assert _need(lib, st, ktype) > least
    p = st.params()
    p.mlp.weight_moment1[0] = None
    ws = np.zeros(least + 16, np.uint8)
    p.workspace = C.c_void_p((ws.ctypes.data + 15) // 16 * 16)
    for size, want in ((least, abi.NT_ERR_NULL_POINTER), (least - 16, abi.NT_ERR_WORKSPACE)):
        p.workspace_bytes = size
        assert lib.nt_train_iteration(C.byref(p), ktype, None) == want, lib.nt_last_error()


def test_static_step_takes_the_smaller_plan(lib):
    """nt_train_step_static is not refused either where only the wide tiles' rows fit its scratch
    (block phase, four grids whose expanded chains leave 12 MB of the 32 MiB: 256 narrow tiles
    need 14.9 MB of rows, 128 wide ones half). Without a device the launch is what fails."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("would launch over host buffers")
    from helpers import make_state
    st = _region(make_state("c4", image=256, blocks=True), 256, 256)
    for g, (w, h) in zip(st.grids, [(400, 384), (64, 200), (32, 32), (16, 16)]):
        g.width, g.height, g.num_mips = w, h, 1
    p = st.params()
    p.workspace = None
    need = _need(lib, st, abi.NT_BLOCK_FEATURES)
    assert need > lib.nt_train_static_scratch_bytes()
    assert lib.nt_train_step_static(C.byref(p), abi.NT_BLOCK_FEATURES, None) == abi.NT_ERR_HIP, lib.nt_last_error()


def test_random_sample_order_refusals(lib):
    """nt_random_sample_order refuses, before touching a device, parameters that train in
    slot order (random texels below the sort's sample count without the hook, region
    samples) and a null order buffer."""
    from helpers import make_state
    st = make_state("c2", image=256, region=(64, 64))
    st.sample_mode = abi.NT_SAMPLES_RANDOM
    p = st.params()
    order = np.zeros(64 * 64, np.uint32)
    assert lib.nt_random_sample_order(C.byref(p), C.c_void_p(order.ctypes.data), None) == abi.NT_ERR_UNSUPPORTED
    assert b"slot order" in lib.nt_last_error()
    region = make_state("c2", image=256, region=(64, 64)).params()
    assert lib.nt_set_test_hooks(0, abi.NT_HOOK_SORT_RANDOM) == 0
    try:
        assert lib.nt_random_sample_order(C.byref(region), C.c_void_p(order.ctypes.data), None) == abi.NT_ERR_UNSUPPORTED
        assert lib.nt_random_sample_order(C.byref(p), None, None) == abi.NT_ERR_NULL_POINTER
        assert lib.nt_random_sample_order(C.byref(p), C.c_void_p(order.ctypes.data), None) == abi.NT_ERR_WORKSPACE
    finally:
        assert lib.nt_set_test_hooks(0, 0) == 0
