"""Host-side logic that needs no GPU: operator schema and fake kernels, input
validation, stride handling, the tile cache and the tune CLI."""

import json
from pathlib import Path

import pytest
import torch

import trifast
import trifast_amd
from trifast_amd import _lib, tune, tuner
from trifast_amd import torch as tt


def meta_inputs(b=1, h=2, n=8, d=16, dtype=torch.bfloat16):
    q = torch.empty(b, h, n, n, d, device="meta", dtype=dtype)
    bias = torch.empty(b, h, n, n, device="meta", dtype=dtype)
    mask = torch.empty(b, n, n, device="meta", dtype=torch.bool)
    return q, q, q, bias, mask


def test_public_surface_matches_reference_names():
    # reference src/trifast/__init__.py:1-3, src/trifast/torch.py:17,68,185,210,220
    assert trifast.triangle_attention is trifast_amd.triangle_attention
    import trifast.torch as rt

    for name in ("triangle_attention", "_triangle_attention", "triangle_attention_bwd", "backwards", "setup_context"):
        assert hasattr(rt, name)
    assert hasattr(torch.ops.trifast, "triangle_attention")
    assert hasattr(torch.ops.trifast, "triangle_attention_backward")
    from trifast.utils import clone_and_clear_grad, disable_tf32, enable_tf32, gen_tensors  # noqa: F401


def test_fake_kernels_give_reference_shapes():
    q, k, v, b, m = meta_inputs()
    o, lse = torch.ops.trifast.triangle_attention(q, k, v, b, m)
    assert o.shape == q.shape and o.dtype == q.dtype
    assert lse.shape == (1, 2, 8, 8) and lse.dtype == torch.float32
    outs = torch.ops.trifast.triangle_attention_backward(o, q, k, v, b, o, lse, m)
    assert [t.shape for t in outs] == [q.shape, q.shape, q.shape, b.shape, m.shape]
    assert outs[4].dtype == torch.bool


def test_cpu_tensors_are_rejected_not_computed():
    g = torch.Generator().manual_seed(0)
    q = torch.randn(1, 1, 4, 4, 16, generator=g)
    b = torch.randn(1, 1, 4, 4, generator=g)
    m = torch.zeros(1, 4, 4, dtype=torch.bool)
    with pytest.raises(RuntimeError, match="GPU only"):
        trifast_amd.triangle_attention(q, q, q, b, m)


@pytest.mark.parametrize(
    "mutate, err",
    [
        (lambda a: a.__setitem__(0, a[0][..., :3, :, :]), ValueError),      # not square
        (lambda a: a.__setitem__(3, a[3][..., :3]), ValueError),            # bias shape
        (lambda a: a.__setitem__(4, a[4].to(torch.uint8)), TypeError),      # mask dtype
        (lambda a: a.__setitem__(1, a[1].to(torch.float16)), TypeError),    # mixed dtypes
        (lambda a: a.__setitem__(0, a[0][0]), ValueError),                  # rank
    ],
)
def test_input_validation(mutate, err):
    q = torch.zeros(1, 2, 4, 4, 16, dtype=torch.bfloat16)
    args = [q, q.clone(), q.clone(), torch.zeros(1, 2, 4, 4, dtype=torch.bfloat16), torch.zeros(1, 4, 4, dtype=torch.bool)]
    mutate(args)
    with pytest.raises(err):
        tt._check_inputs(*args)


def test_vector_ready_keeps_transposed_views_and_copies_the_rest():
    x = torch.zeros(1, 2, 8, 8, 16, dtype=torch.bfloat16)
    assert tt._vector_ready(x) is x
    xt = x.transpose(2, 3)
    assert tt._vector_ready(xt) is xt                       # i<->j view: read in place
    assert tt._vector_ready(x[..., ::2]).is_contiguous()    # d stride 2: copied
    ones = torch.ones((), dtype=torch.bfloat16).expand(1, 2, 8, 8, 16)
    assert tt._vector_ready(ones).is_contiguous()           # stride-0 upstream gradient
    assert tt._strides(torch.zeros(1, 2, 8, 8, 16))[0] == 0  # size-1 dims report stride 0


def test_key_and_closest_n():
    assert tuner.closest_n(1) == 1 and tuner.closest_n(17) == 32 and tuner.closest_n(1024) == 1024 and tuner.closest_n(1025) == 2048
    assert tuner.make_key(191, 4, 32, torch.bfloat16) == "4_32_256_torch.bfloat16"


def test_tile_cache_roundtrip_and_corruption(tmp_path, monkeypatch, capsys):
    monkeypatch.setenv("TRIFAST_CONFIG_DIR", str(tmp_path))
    monkeypatch.setattr(tuner, "_device_tag", lambda device=None: "Test-GPU_9-5")
    tuner.reset()
    c = tuner.TileCache(_lib.KERNEL_FWD)
    assert c.cache_file == tmp_path / "_fwd_Test-GPU_9-5.json"
    c.cache["4_32_1024_torch.bfloat16"] = 1
    c.write()
    raw = json.loads(c.cache_file.read_text())
    assert raw["4_32_1024_torch.bfloat16"]["tile"] == 1
    assert raw["4_32_1024_torch.bfloat16"]["kwargs"] == {k: v for k, v in _lib.tile_info(0, 1).items() if k != "num_waves"}
    assert tuner.TileCache(_lib.KERNEL_FWD).cache == {"4_32_1024_torch.bfloat16": 1}
    # an entry from another tile table is dropped, a corrupt file is reported and ignored
    raw["4_32_1024_torch.bfloat16"]["kwargs"]["BLOCK_J"] = 12345
    c.cache_file.write_text(json.dumps(raw))
    assert tuner.TileCache(_lib.KERNEL_FWD).cache == {}
    c.cache_file.write_text("{not json")
    assert tuner.TileCache(_lib.KERNEL_FWD).cache == {}
    assert "Could not load autotune cache" in capsys.readouterr().out
    tuner.reset()


def test_pick_without_autotune_uses_library_heuristic(monkeypatch):
    monkeypatch.setenv("TRIFAST_AUTOTUNE", "0")
    monkeypatch.delenv("TRIFAST_FORCE_TUNE", raising=False)
    called = []
    t = tuner.pick(_lib.KERNEL_FWD, 1024, 4, 32, torch.bfloat16, called.append)
    assert t == _lib.load().trifast_default_tile(0, 1024, 4, 32, _lib.BF16) and called == []


def test_pick_times_every_supported_tile_on_a_miss(tmp_path, monkeypatch):
    monkeypatch.setenv("TRIFAST_CONFIG_DIR", str(tmp_path))
    monkeypatch.setenv("TRIFAST_AUTOTUNE", "1")
    monkeypatch.delenv("TRIFAST_FORCE_TUNE", raising=False)
    monkeypatch.setattr(tuner, "_device_tag", lambda device=None: "Test-GPU_9-5")
    fake_ms = {0: 3.0, 1: 1.0, 2: 5.0, 3: 2.0}
    monkeypatch.setattr(tuner, "_time_launch", lambda launch, tile, **kw: fake_ms.get(tile, 9.0))
    tuner.reset()
    assert tuner.pick(_lib.KERNEL_FWD, 300, 4, 32, torch.bfloat16, lambda t: None) == 1
    assert json.loads((tmp_path / "_fwd_Test-GPU_9-5.json").read_text())["4_32_512_torch.bfloat16"]["tile"] == 1
    # a hit does not time again
    monkeypatch.setattr(tuner, "_time_launch", lambda *a, **k: pytest.fail("re-tuned on a cache hit"))
    assert tuner.pick(_lib.KERNEL_FWD, 400, 4, 32, torch.bfloat16, lambda t: None) == 1
    # TRIFAST_FORCE_TUNE re-tunes even on a hit
    monkeypatch.setenv("TRIFAST_FORCE_TUNE", "yes")
    monkeypatch.setattr(tuner, "_time_launch", lambda launch, tile, **kw: float(tile != 3))
    assert tuner.pick(_lib.KERNEL_FWD, 400, 4, 32, torch.bfloat16, lambda t: None) == 3
    tuner.reset()


def test_pick_prefers_the_default_tile_on_a_near_tie(tmp_path, monkeypatch):
    monkeypatch.setenv("TRIFAST_CONFIG_DIR", str(tmp_path))
    monkeypatch.setenv("TRIFAST_AUTOTUNE", "1")
    monkeypatch.delenv("TRIFAST_FORCE_TUNE", raising=False)
    monkeypatch.setattr(tuner, "_device_tag", lambda device=None: "Test-GPU_9-5")
    default = _lib.load().trifast_default_tile(_lib.KERNEL_BWD_KV, 1024, 4, 32, _lib.BF16)
    other = next(t for t in tuner.supported_tiles(_lib.KERNEL_BWD_KV, 1024, 4, 32, torch.bfloat16) if t != default)
    # 1 % faster is within the scatter of the timings: the default stays
    monkeypatch.setattr(tuner, "_time_launch", lambda launch, tile, **kw: 0.99 if tile == other else (1.0 if tile == default else 5.0))
    tuner.reset()
    assert tuner.pick(_lib.KERNEL_BWD_KV, 1024, 4, 32, torch.bfloat16, lambda t: None) == default
    # 10 % faster replaces it
    monkeypatch.setenv("TRIFAST_FORCE_TUNE", "1")
    monkeypatch.setattr(tuner, "_time_launch", lambda launch, tile, **kw: 0.9 if tile == other else (1.0 if tile == default else 5.0))
    assert tuner.pick(_lib.KERNEL_BWD_KV, 1024, 4, 32, torch.bfloat16, lambda t: None) == other
    tuner.reset()


def test_pick_charges_a_tile_what_it_leaves_to_other_kernels(tmp_path, monkeypatch):
    """dk/dv tiles that do not also produce dq are charged the dq kernel's time: the
    row-resident tile wins although its own launch is the longest."""
    monkeypatch.setenv("TRIFAST_CONFIG_DIR", str(tmp_path))
    monkeypatch.setenv("TRIFAST_AUTOTUNE", "1")
    monkeypatch.delenv("TRIFAST_FORCE_TUNE", raising=False)
    monkeypatch.setattr(tuner, "_device_tag", lambda device=None: "Test-GPU_9-5")
    lib = _lib.load()
    tiles = tuner.supported_tiles(_lib.KERNEL_BWD_KV, 1024, 4, 32, torch.bfloat16)
    fused = [t for t in tiles if lib.trifast_bwd_kv_tile_writes_dq(t)]
    assert len(fused) == 1 and len(tiles) > 1  # 1024 keys: only the largest row-resident tile fits
    monkeypatch.setattr(tuner, "_time_launch", lambda launch, tile, **kw: 2.1 if tile in fused else 1.6)
    tuner.reset()
    assert tuner.pick(_lib.KERNEL_BWD_KV, 1024, 4, 32, torch.bfloat16, lambda t: None) not in fused
    monkeypatch.setenv("TRIFAST_FORCE_TUNE", "1")
    extra = lambda t: 0.0 if lib.trifast_bwd_kv_tile_writes_dq(t) else 1.4
    assert tuner.pick(_lib.KERNEL_BWD_KV, 1024, 4, 32, torch.bfloat16, lambda t: None, extra_cost=extra) == fused[0]
    tuner.reset()


def test_pick_times_what_can_win(tmp_path, monkeypatch):
    """On a miss every tile is timed once, and a second time unless it is far behind; of the row-resident
    tiles only the one that fits the length, which is what a later hit takes too."""
    monkeypatch.setenv("TRIFAST_CONFIG_DIR", str(tmp_path))
    monkeypatch.setenv("TRIFAST_AUTOTUNE", "1")
    monkeypatch.delenv("TRIFAST_FORCE_TUNE", raising=False)
    monkeypatch.setattr(tuner, "_device_tag", lambda device=None: "Test-GPU_9-5")
    lib = _lib.load()
    for n in (31, 256, 300, 700, 1024):
        timed = []
        fits = lib.trifast_default_tile(_lib.KERNEL_BWD_KV, n, 4, 32, _lib.BF16)
        slow = {0: 9.0, fits: 2.0}  # (the first time of the tile that fits is a cold one)
        monkeypatch.setattr(tuner, "_time_launch", lambda launch, t, **kw: timed.append(t) or (1.0 if timed.count(t) > 1 and t == fits else slow.get(t, 1.6)))
        tuner.reset()
        assert tuner.pick(_lib.KERNEL_BWD_KV, n, 4, 32, torch.bfloat16, lambda t: None) == fits
        rows = [t for t in timed if lib.trifast_bwd_kv_tile_writes_dq(t)]
        streaming = [t for t in tuner.supported_tiles(_lib.KERNEL_BWD_KV, n, 4, 32, torch.bfloat16) if not lib.trifast_bwd_kv_tile_writes_dq(t)]
        assert rows == [fits, fits] and timed.count(0) == 1
        assert [timed.count(t) for t in streaming[1:]] == [2] * len(streaming[1:])
        for f in tmp_path.glob("*.json"):
            f.unlink()
    tuner.reset()


def test_row_resident_tiles_in_the_library_tables():
    """The row-resident kernel appears as the last eight tiles of the dk/dv family: seven for rows
    of up to 256, 384, ..., 1024 keys, for 16-bit inputs, and one that runs longer rows (up to
    8192 keys at head dim 32) in passes of 1024 keys; they are the default where they are fastest."""
    lib = _lib.load()
    nt = lib.trifast_num_tiles(_lib.KERNEL_BWD_KV)
    fused = [t for t in range(nt) if lib.trifast_bwd_kv_tile_writes_dq(t)]
    assert fused == list(range(nt - 8, nt))
    assert not lib.trifast_bwd_kv_tile_writes_dq(-1) and not lib.trifast_bwd_kv_tile_writes_dq(nt)
    passes = fused[7]
    sup = lambda n, d, code: bool(lib.trifast_supports(_lib.KERNEL_BWD_KV, passes, n, 4, d, code))
    assert sup(1025, 32, _lib.BF16) and sup(8192, 32, _lib.F16) and sup(2047, 32, _lib.BF16)
    assert not sup(1024, 32, _lib.BF16) and not sup(8193, 32, _lib.BF16)
    assert not sup(2048, 64, _lib.BF16) and not sup(2048, 16, _lib.BF16) and not sup(2048, 32, _lib.F32)
    # its low parts of dq live in the workspace tail, which is at least one more 16-bit tensor
    ws = lambda n, d: lib.trifast_bwd_workspace_bytes(1, 4, n, d, _lib.BF16)
    assert ws(2048, 32) - ws(2048, 64) >= 4 * 2048 * 2048 * 32 * 2 - 4 * 4 * 2048 * 2048 * 4
    for t, keys in zip(fused[:7], (256, 384, 512, 640, 768, 896, 1024)):
        assert _lib.tile_info(_lib.KERNEL_BWD_KV, t)["BLOCK_K"] == keys
        assert lib.trifast_supports(_lib.KERNEL_BWD_KV, t, keys, 4, 32, _lib.BF16)
        assert lib.trifast_supports(_lib.KERNEL_BWD_KV, t, keys - 37, 2, 32, _lib.F16)
        assert not lib.trifast_supports(_lib.KERNEL_BWD_KV, t, keys + 1, 4, 32, _lib.BF16)
        assert not lib.trifast_supports(_lib.KERNEL_BWD_KV, t, keys, 4, 32, _lib.F32)
        assert not lib.trifast_supports(_lib.KERNEL_BWD_KV, t, keys, 4, 128, _lib.BF16)
    default = lambda n, d, code: lib.trifast_default_tile(_lib.KERNEL_BWD_KV, n, 4, d, code)
    assert default(1024, 32, _lib.BF16) == fused[6] and default(300, 32, _lib.F16) == fused[1] and default(385, 32, _lib.F16) == fused[2]
    assert default(640, 32, _lib.BF16) == fused[3] and default(641, 32, _lib.BF16) == fused[4] and default(896, 32, _lib.BF16) == fused[5]
    assert default(129, 32, _lib.BF16) == fused[0] and default(1025, 32, _lib.BF16) == passes and default(8193, 32, _lib.BF16) not in fused
    # (from the smallest rows on: one launch instead of two; head dim 16 like 32, head dim 64 up to 384 keys)
    assert default(128, 32, _lib.BF16) == fused[0] and default(16, 32, _lib.F16) == fused[0]
    assert default(700, 16, _lib.BF16) == fused[4] and default(1025, 16, _lib.BF16) not in fused
    assert default(300, 64, _lib.F16) == fused[1] and default(385, 64, _lib.F16) not in fused and default(512, 64, _lib.BF16) not in fused
    assert default(512, 32, _lib.F32) not in fused and default(64, 128, _lib.BF16) not in fused


def test_default_forward_tiles_of_128_byte_rows():
    """The scheduled loop (tile 6) from more than 256 keys on, its general twin below."""
    pick = lambda n, code, d=64: _lib.load().trifast_default_tile(_lib.KERNEL_FWD, n, 8, d, code)
    for code in (_lib.BF16, _lib.F16):
        assert [pick(n, code) for n in (65, 192, 256, 257, 300, 384, 768)] == [4, 4, 4, 6, 6, 6, 6]
    assert pick(300, _lib.F32, 32) == 4  # (fp32 has no scheduled loop)


def test_tune_cli_flags_and_sweep():
    p = tune.build_parser()
    a = p.parse_args([])
    assert (a.min_n, a.max_n, a.h, a.d, a.dtype) == (16, 1024, [4], [32], [torch.bfloat16])
    a = p.parse_args(["--min-n", "64", "--max-n", "300", "--dtype", "float16,float32", "--h", "1,4", "--d", "16,64"])
    assert a.h == [1, 4] and a.d == [16, 64] and set(a.dtype) == {torch.float16, torch.float32}
    assert tune.sweep_ns(a.min_n, a.max_n) == [64, 128, 256]
    assert len(tune.valid_dtypes("all")) == 3
    with pytest.raises(SystemExit):
        p.parse_args(["--dtype", "int8"])


def test_equiv_module_matches_the_oracle():
    """``trifast.equiv`` (the reference's public pure-PyTorch functions) gives the
    oracle's numbers, fully masked rows included."""
    from trifast.equiv import attention_reference, triangle_attention_simple
    from oracle import triangle_oracle as orc

    g = torch.Generator().manual_seed(3)
    q, k, v, b, m = orc.gen_tensors(9, 8, 2, True, "cpu", torch.float32, 2, 1.0, generator=g)
    m[:, 4, :] = True
    q, k, v, b = (t.detach() for t in (q, k, v, b))
    torch.testing.assert_close(attention_reference(q, k, v, b, m), orc.attention_reference(q, k, v, b, m), rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(triangle_attention_simple(q, k, v, b, m), orc.triangle_attention_simple(q, k, v, b, m), rtol=1e-6, atol=1e-6)


def test_wide_j_strides_are_copied_and_their_gradients_allocated_contiguous():
    # the kernels address the rows of a tile through 32-bit offsets: a stride between
    # consecutive j of 2^24 bytes or more is not run in place (the library would refuse it)
    t = torch.empty_strided((1, 1, 2, 2, 8), (0, 0, 64, 1 << 24, 1), dtype=torch.bfloat16, device="meta")
    assert tt._vector_ready(t).is_contiguous()
    assert tt._grad_like(t).is_contiguous()
    ok = torch.empty_strided((1, 1, 2, 2, 8), (0, 0, 8, 16, 1), dtype=torch.bfloat16, device="meta")  # transposed view
    assert tt._vector_ready(ok) is ok


def test_equiv_simple_takes_any_number_of_batch_dims():
    from trifast_amd import equiv

    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(2, 3, 2, 5, 5, 4, generator=g) for _ in range(3))
    b = torch.randn(2, 3, 2, 5, 5, generator=g)
    m = torch.rand(2, 3, 5, 5, generator=g) < 0.3
    whole = equiv.triangle_attention_simple(q, k, v, b, m)
    parts = torch.stack([equiv.attention_reference(q[x], k[x], v[x], b[x], m[x]) for x in range(2)])
    assert torch.allclose(whole, parts, atol=1e-6)
    assert torch.allclose(equiv.triangle_attention_simple(q[0, 0], k[0, 0], v[0, 0], b[0, 0], m[0, 0]), whole[0, 0], atol=1e-6)


def test_tensors_with_a_tangent_do_not_take_the_native_path():
    """The native path launches the kernels without the dispatcher: a forward-mode tangent would be
    dropped there, so such tensors are declined."""
    import torch.autograd.forward_ad as fwad

    native = tt._native()
    x = torch.randn(3)
    assert native.plain_eager([x, x.clone().requires_grad_(True)])
    for lazy in (torch._neg_view(x), torch._efficientzerotensor(3), torch.randn(3, dtype=torch.cfloat).conj()):
        assert not native.plain_eager([lazy])  # (nor do tensors whose memory does not hold their numbers)
    with fwad.dual_level():
        assert native.plain_eager([x])
        assert not native.plain_eager([x, fwad.make_dual(x, torch.ones_like(x))])


def test_nothing_takes_the_native_path_while_torch_jit_traces():
    """A tracer under the native path records the allocation of the output and no launch."""
    seen = []

    def fn(x):
        seen.append(tt._native().plain_eager([x]))
        return x + 1

    torch.jit.trace(fn, (torch.randn(3),), check_trace=False)
    assert seen == [False] and tt._native().plain_eager([torch.randn(3)])


def test_bench_prices_fp32_by_the_products_it_runs_as():
    import re

    import bench

    src = (Path(tt.__file__).parent / "csrc" / "tri_common.hpp").read_text()
    body = re.search(r"mfma\(const frag& a, const frag& b, f32x16 c\) \{(.*?)\n  \}", src, re.S).group(1)
    assert bench.PEAK_F32_TFLOPS == bench.PEAK_BF16_TFLOPS / body.count("mfma(a.")


@pytest.mark.parametrize("source,flags", [
    ("tri_bwd_b.hip", ("-DTRI_DB_TIMING",)),
    ("tri_bwd_b.hip", ("-DTRI_DB_TIMING", "-DTRI_DB_TIMING_LOADS=2")),
    ("tri_bwd_row_bf16.hip", ("-DTRI_ROW_TIMING",)),
], ids=["db", "db_loads", "row"])
def test_probe_builds_of_the_kernels_compile(source, flags):
    """The builds that time the kernels from inside (benchmark/microbench) keep up with the kernels."""
    import subprocess

    from trifast_amd import build

    cmd = [build._hipcc(), *build.HIPCC_FLAGS, *flags, "-DTRI_DEV_ONLY_BF16_D32", "--cuda-device-only", "-fsyntax-only", "-I", str(build.CSRC), str(build.CSRC / source)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]


@pytest.fixture(scope="module", params=["__bf16", "_Float16"])
def wide_row_kernels(request, tmp_path_factory):
    """Assembly of the row-resident backward at head dim 64: key tiles per wave -> (lines of the kernel)."""
    import re
    import subprocess

    from trifast_amd import build

    if build._compiler_flags():
        pytest.skip("not the compiler that the kernels are laid out for")
    tiles = (2, 3)
    tmp = tmp_path_factory.mktemp("row")
    source, asm = tmp / "row.hip", tmp / "row.s"
    source.write_text('#include "tri_bwd_row.hpp"\nnamespace tri {\n' + "".join(
        f"template __global__ void tri_bwd_row_kernel<{request.param}, 64, {kt}, false>(const BwdArgs);\n" for kt in tiles) + "}\n")
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", "-I", str(build.CSRC), "-o", str(asm), str(source)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    kernels = re.findall(r"^_Z\w*tri_bwd_row_kernel\w*Li64ELi(\d)E\w*:(.*?)^\.Lfunc_end", asm.read_text(), re.S | re.M)
    assert sorted(int(kt) for kt, _ in kernels) == list(tiles)
    return {int(kt): body.splitlines() for kt, body in kernels}


def test_row_resident_loop_keeps_nothing_in_scratch(wide_row_kernels):
    """One branch, the loop's own, and no scratch access in the loop over the query tiles: a reload waits for every load in
    flight, those of the ring among them."""
    import re

    for kt, lines in wide_row_kernels.items():
        label = {m.group(1): at for at, line in enumerate(lines) if (m := re.match(r"(\.LBB\w+):", line))}
        loops = [lines[label[m.group(1)]:at + 1] for at, line in enumerate(lines)
                 if (m := re.match(r"\s+s_c?branch\w*\s+(\.LBB\w+)", line)) and label[m.group(1)] <= at]
        # the two versions of the loop (with and without masked keys) are the ones that request stages of the ring and take exponentials
        loops = [x for x in loops if "Inner Loop" in x[0] and any("global_load_lds" in y for y in x) and sum("v_exp_f32" in y for y in x) == 16 * kt]
        assert len(loops) == 2, kt
        for loop in loops:
            assert [y for y in loop if "scratch_" in y] == [], kt
            assert sum(bool(re.match(r"\s+s_c?branch", y)) for y in loop) == 1, kt


def test_fully_masked_rows_leave_nothing_in_scratch(wide_row_kernels):
    """The sums of a fully masked row (two 64 x 64 products and three vectors) take no address per element: that filled
    the registers of the whole kernel, and every address came back from scratch with a wait of its own."""
    for kt, lines in wide_row_kernels.items():
        assert [line for line in lines if "scratch_" in line] == [], kt


def test_fully_masked_rows_of_the_forward_load_together(tmp_path):
    """The pass over V of a workgroup of fully masked rows has eight loads in flight, those of all its rows and the last ones of
    each too, and no wait for the stage that was requested before it was known that nobody needs it."""
    import re
    import subprocess

    from trifast_amd import build

    if build._compiler_flags():
        pytest.skip("not the compiler that the kernels are laid out for")
    tiles = ((32, 1), (32, 2), (32, 4), (128, 1))
    source, asm = tmp_path / "fwd.hip", tmp_path / "fwd.s"
    source.write_text('#include "tri_fwd.hpp"\nnamespace tri {\n' + "".join(
        f"template __global__ void tri_fwd_kernel<__bf16, {d}, 4, {r}, 32>(const FwdArgs);\n" for d, r in tiles) + "}\n")
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", "-I", str(build.CSRC), "-o", str(asm), str(source)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    kernels = re.findall(r"^_Z\w*tri_fwd_kernel\w*:(.*?)^\.Lfunc_end", asm.read_text(), re.S | re.M)
    assert len(kernels) == len(tiles)
    for tile, body in zip(tiles, kernels):
        lines = body.splitlines()
        label = {m.group(1): at for at, line in enumerate(lines) if (m := re.match(r"(\.LBB\w+):", line))}
        loops = [lines[label[m.group(1)]:at + 1] for at, line in enumerate(lines)
                 if (m := re.match(r"\s+s_c?branch\w*\s+(\.LBB\w+)", line)) and label[m.group(1)] <= at]
        # (the only loop without products that loads 16 bytes a lane into registers)
        passes = [x for x in loops if not any("v_mfma" in y or "s_barrier" in y for y in x) and any("global_load_dwordx4" in y for y in x)]
        assert [sum("global_load_dwordx4" in y for y in x) for x in passes] == [8], tile


def test_row_timeline_probe_spills_no_scalars(tmp_path):
    """The build that times the row-resident backward runs the loop of the regular one where every key is attended: its readings stay
    in scalar registers (spilled ones made the steps 50 clocks longer than they are)."""
    import re
    import subprocess

    from trifast_amd import build

    if build._compiler_flags():
        pytest.skip("not the compiler that the kernels are laid out for")
    source, asm = tmp_path / "row.hip", tmp_path / "row.s"
    source.write_text('#include "tri_bwd_row.hpp"\nnamespace tri {\ntemplate __global__ void tri_bwd_row_kernel<__bf16, 32, 8, false>(const BwdArgs);\n}\n')
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, "-DTRI_ROW_TIMING", "--cuda-device-only", "-S", "-I", str(build.CSRC), "-o", str(asm), str(source)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    lines = asm.read_text().splitlines()
    label = {m.group(1): at for at, line in enumerate(lines) if (m := re.match(r"(\.LBB\w+):", line))}
    loops = [lines[label[m.group(1)]:at + 1] for at, line in enumerate(lines)
             if (m := re.match(r"\s+s_c?branch\w*\s+(\.LBB\w+)", line)) and label[m.group(1)] <= at]
    # (16 exponentials of every key tile, and the clock once per step; the loops over fully masked rows have neither)
    loops = [x for x in loops if "Inner Loop" in x[0] and sum("v_exp_f32" in y for y in x) == 128 and any("s_memtime" in y for y in x)]
    assert len(loops) == 2
    assert min(sum(bool(re.match(r"\s+v_(read|write)lane", y)) for y in x) for x in loops) == 0


# (key tiles, head dim, rows per XCD): the form of the row-resident backward that was measured to be at least 4 % faster there than the other
ROW_FORMS = {
    "kOneWave": [(5, 32, 65), (5, 16, 140), (5, 32, 260), (6, 32, 66), (6, 16, 110), (6, 32, 215), (6, 16, 384), (7, 32, 100), (7, 16, 250), (7, 32, 252),
                 (8, 32, 115), (8, 16, 128), (3, 32, 70), (4, 16, 84), (4, 32, 140)],
    "kTwoWaves": [(4, 32, 64), (9, 16, 65), (10, 32, 75), (11, 32, 42), (11, 16, 126), (12, 32, 144), (13, 16, 150), (16, 32, 64)],
    "kFourWaves": [(3, 32, 9), (5, 16, 54), (6, 32, 43), (6, 32, 129), (6, 16, 144), (7, 32, 140), (7, 16, 175), (7, 32, 280), (7, 16, 400), (7, 32, 450), (8, 32, 64), (8, 16, 145),
                   (8, 32, 160), (8, 16, 192), (8, 32, 261), (8, 16, 288), (8, 32, 384), (8, 16, 416), (8, 32, 768), (11, 32, 83)],
}


def test_waves_of_a_row_where_one_form_is_faster(tmp_path):
    import subprocess

    from trifast_amd import build

    checks = "".join(f"static_assert(tri::bwd_row_form({w}, {d}, {r}) == tri::RowForm::{form}, \"{w} key tiles, head dim {d}, {r} rows\");\n"
                     for form, launches in ROW_FORMS.items() for w, d, r in launches)
    source = tmp_path / "rule.cpp"
    source.write_text('#include "tri_bwd_row_rule.hpp"\n' + checks)
    res = subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", str(build.CSRC), str(source)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
