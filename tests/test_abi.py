"""CPU-side checks of the C ABI library: it loads, exports what the headers under include/ declare,
its host-only functions (schedules) match the reference's golden vectors, and it refuses to
compute without a GPU instead of falling back to anything."""
import ctypes
import os
import re

import numpy as np
import pytest

import fluxhip
from model_spec import KLEIN_4B, TINY, tensor_shapes, make_weights, write_safetensors, bf16_to_f32, f32_to_bf16, normal_f32

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    L = fluxhip.lib()
    import glob
    headers = sorted(glob.glob(os.path.join(ROOT, "include", "*.h")))
    assert [os.path.basename(h) for h in headers] == ["flux_hip.h", "flux_hip_debug.h"]
    funcs = set()
    for h in headers:
        hdr = re.sub(r"/\*.*?\*/", "", open(h).read(), flags=re.S)
        funcs |= set(re.findall(r"\b((?:flux|qwen3)_[a-z0-9_]+)\s*\(", hdr))
    assert len(funcs) > 100
    for name in sorted(funcs):
        assert hasattr(L, name), name
    for var in ("flux_timing_transformer_total", "flux_timing_transformer_double", "flux_timing_transformer_single",
                "flux_timing_transformer_final"):
        ctypes.c_double.in_dll(L, var)
    for var in ("flux_substep_callback", "flux_step_callback"):
        ctypes.c_void_p.in_dll(L, var)
    ctypes.c_int.in_dll(L, "flux_verbose")


def test_schedules_match_reference_golden(golden_dir):
    g = np.load(os.path.join(golden_dir, "ops.npz"))
    for n in (1, 4, 7):
        np.testing.assert_allclose(fluxhip.schedule("linear", n), g[f"sched_linear_{n}"], atol=1e-7)
    np.testing.assert_allclose(fluxhip.schedule("power", 5, 2.0), g["sched_power_5_2"], atol=1e-7)
    for n, sl in ((4, 256), (4, 1024), (4, 4096), (50, 1024), (4, 5000), (1, 16), (28, 4300)):
        np.testing.assert_allclose(fluxhip.schedule("official", n, sl), g[f"sched_official_{n}_{sl}"], atol=6e-7)   # a few fp32 ulp: expf/powf vs the -ffast-math build
    for n, sh in ((4, 0.0), (7, 1.5), (1, -2.0)):
        np.testing.assert_allclose(fluxhip.schedule("sigmoid", n, sh), g[f"sched_sigmoid_{n}_{sh}"], atol=6e-7)
    for n, hh, ww in ((4, 256, 256), (6, 512, 512), (5, 1024, 1024), (3, 2048, 256), (4, 768, 1024)):
        np.testing.assert_allclose(fluxhip.schedule("resolution", n, hh, ww), g[f"sched_resolution_{n}_{hh}_{ww}"], atol=6e-7)


def test_patch_convolution_keeps_skipped_positions_outside():
    """The 3x3 convolution that holds a tile's neighbourhood in LDS gives positions beyond the image an offset of 0xF0000000
    and adds up to seven image rows of fp32 results to it: the sum must not come round to the buffer's start. Images too wide for that are
    refused (the other tiles take them); everything the VAE has is taken."""
    f = fluxhip.lib()._Z11conv3_takesiiii
    f.argtypes, f.restype = [ctypes.c_int] * 4, ctypes.c_bool
    taken = 0
    for cout in (128, 256, 512, 4096):
        for W in [1, 1792] + [int(1000 * 1.05 ** i) for i in range(140)]:
            for H in (1, 16, 500):
                if f(H, W, 128, cout):
                    taken += 1
                    last = 0xF0000000 + 7 * (W + 2) * cout * 4 + 128 + 64 + 16      # (bytes of the last access behind its lane's row)
                    assert last <= 1 << 32, (H, W, cout)
    assert taken > 100
    assert not f(16, 20001, 128, 512) and f(16, 18000, 128, 512)
    for H, W, cin, cout in ((1, 1, 128, 128), (1792, 1792, 256, 128), (1792, 1792, 128, 128), (896, 896, 512, 256), (448, 448, 512, 512), (16, 1792, 256, 256)):
        assert f(H, W, cin, cout), (H, W, cin, cout)


def test_exponential_scores_tell_switched_off_from_failed():
    """With the ring kernel switched off the VAE's attention without scores is not to be had: that is no error, nothing is
    launched, and its caller goes on with the scores in memory. What the product itself refuses is an error with its own text."""
    L = fluxhip.lib()
    vp, ci, cf = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    L.flux_hip_linear_exp.argtypes = [vp] * 3 + [ci] * 5 + [vp, cf, ci, vp, vp]
    L.flux_hip_vae_attention.argtypes = [vp] * 7 + [ci] * 3 + [cf, vp]
    buf = np.zeros(4096, np.uint8)
    p = (buf.ctypes.data + 15) & ~15
    done, pieces = ci(7), ci(7)

    def exp(P=p, M=256, N=256, K=512):
        L.flux_hip_vae_attention(p, p, p, p, p, p, p, 0, 0, 0, 1.0, ctypes.byref(ci(0)))       # an error of another function
        assert b"flux_hip_vae_attention" in L.flux_hip_last_error()
        return L.flux_hip_linear_exp(p, p, P, M, N, K, 512, 512, p, 1.0, 256, p, ctypes.byref(pieces))

    for bad in (dict(P=p + 8), dict(P=None), dict(M=0), dict(N=384), dict(K=192)):
        assert exp(**bad) == 0 and b"flux_hip_linear_exp" in L.flux_hip_last_error(), bad
    L.flux_hip_linear_ring(0)
    try:
        assert exp() == 0 and b"switched off" in L.flux_hip_last_error()
        assert L.flux_hip_vae_attention(p, p, p, p, p, p, p, 256, 256, 256, 1.0, ctypes.byref(done)) == 1 and done.value == 0
    finally:
        L.flux_hip_linear_ring(1)


@pytest.mark.parametrize("name", ["flux_hip_linear_slices", "flux_hip_linear_f32_slices"])
def test_projections_that_leave_slices_check_their_arguments(name):
    """Widths and K that no tile takes, missing and unaligned operands are refused on the host, by name."""
    f, vp, ci = getattr(fluxhip.lib(), name), ctypes.c_void_p, ctypes.c_int
    f.argtypes = [vp] * 3 + [ci] * 3 + [vp] * 2
    buf = np.zeros(64, np.uint8)
    p, ws, n = (buf.ctypes.data + 15) & ~15, vp(0), ci(7)
    for A, W, C, N, K in ((p, p, p, 192, 512), (p, p, p, 0, 512), (p, p, p, 256, 96), (p, p, p, 256, 0), (None, p, p, 256, 512), (p, None, p, 256, 512),
                          (p, p, None, 256, 512), (p + 8, p, p, 256, 512), (p, p + 2, p, 256, 512), (p, p, p + 4, 256, 512)):
        assert f(A, W, C, 256, N, K, ctypes.byref(ws), ctypes.byref(n)) == 0
        assert name.encode() in fluxhip.lib().flux_hip_last_error() and n.value == 0
    assert f(None, None, None, 0, 256, 512, ctypes.byref(ws), ctypes.byref(n)) == 1      # no rows: nothing to do


def test_attention_reference_samples_every_column():
    """The 256 keys that give the VAE attention's reference are spread over the image: over its columns - all of them, or as many as there
    are keys - and over at least two fifths of its rows; for every image from 2560 positions on that a picture or a latent can have. (The position
    count alone decides, so the step has no factor in common with it.)"""
    f = fluxhip.lib().flux_hip_vae_attention_sample_step
    f.argtypes = [ctypes.c_int]
    for h in range(2, 225, 2):
        for w in range(2, 225, 2):
            keys = h * w
            if keys < 2560:
                continue
            step = f(keys)
            assert 1 <= step <= keys // 256, (h, w)
            sample = np.arange(256) * step
            assert len(np.unique(sample % w)) >= min(w, 256), (h, w, step)
            assert sample[-1] >= 0.4 * keys, (h, w, step)
    assert f(256) == 1 and f(511) == 1


@pytest.mark.parametrize("hp,wp,cin", [(10, 12, 256), (130, 130, 256), (130, 130, 512)])
def test_norm_with_shortcut_refuses_sums_without_rows(hp, wp, cin):
    """flux_hip_group_norm_stats refuses sums of no rows, and so does the norm that takes the block's shortcut along, in its two launches and in its one: a
    mean of nothing would go through as 0."""
    L = fluxhip.lib()
    f = L.flux_hip_vae_group_norm_skip
    vp, ci = ctypes.c_void_p, ctypes.c_int
    f.argtypes = [vp] * 7 + [ci, ci, ci, ctypes.c_float, vp, ci, vp, vp, ci]
    p = 1 << 20                                                  # never read: the call ends at its checks
    for rows in (0, -1):
        assert f(p, p, p, p, p, p, p, hp, wp, cin, 1e-6, p, rows, p, p, 128) == 0
        assert b"flux_hip_vae_group_norm_skip: conv_stats_rows" in L.flux_hip_last_error()


def test_bench_names_the_kernels_that_tiles_launch():
    """bench.py's names of the tiles, which are looked up in kernel traces, have the template arguments of the launches."""
    source, bench = (open(os.path.join(ROOT, *p)).read() for p in (("flux2.c_amd", "csrc", "gemm.hip"), ("bench.py",)))
    body = source[source.index("static int launch_epi("):]
    body = body[:body.index("\n}\n")]
    launched = {}
    for i, kind, args in re.findall(r"case (\d+):.*?return launch_(cfg|few|4d|4w|4x)<([^>]*)>", body):
        launched.setdefault(int(i), {})[kind] = [a for a in args.replace(" ", "").split(",") if a != "EPI"]
    kinds = {"gemm_kernel": "cfg", "gemm_few_kernel": "few", "gemm4d_kernel": "4d", "gemm4w_kernel": "4w", "gemm4x_kernel": "4x"}
    named = {int(i): (kinds[kernel], args.split(",")) for i, kernel, args in re.findall(r'(\d+): f"(gemm\w*_kernel)<([^>]*)>', bench)}
    assert len(named) >= 13 and len(launched) >= 20 and sum(kind == "few" for kind, _ in named.values()) == 5
    for tile, (kind, args) in named.items():
        if tile in launched:                                     # (0 is the default)
            want = launched[tile][kind]
            got = [a for a in args if a != "{epi_name}"]
            assert got == (want[:2] if len(got) == 2 and kind != "cfg" else want), (tile, args, want)      # (a ring's depths are left out)


def test_touching_a_result_buffer_leaves_its_contents():
    """The result's pages are touched while the device computes it; when the call fails afterwards the caller's buffer
    holds what it held before. Sizes around a page, at offsets of every kind."""
    f = fluxhip.lib().flux_hip_prefault
    f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_size_t], None
    want = np.random.default_rng(3).integers(0, 256, 1 << 17).astype(np.uint8)
    want[::3] = 0
    got = want.copy()
    for offset in (0, 1, 4095, 4097):
        for size in (0, 1, 2, 4095, 4096, 4097, 8192, 70001):
            f(got[offset:].ctypes.data, size)
    np.testing.assert_array_equal(got, want)


def test_host_generator_matches_reference_golden(golden_dir):
    g = np.load(os.path.join(golden_dir, "ops.npz"))
    np.testing.assert_allclose(fluxhip.randn(64, seed=42), g["randn_42"], atol=1e-6)
    a = fluxhip.randn(8)                              # continues the stream
    assert not np.array_equal(a, g["randn_42"][:8])
    np.testing.assert_allclose(fluxhip.randn(64, seed=42), g["randn_42"], atol=1e-6)


def test_init_noise_matches_reference_golden(golden_dir):
    g = np.load(os.path.join(golden_dir, "ops.npz"))
    np.testing.assert_allclose(fluxhip.init_noise(128, 4, 4, 42), g["noise_42_4x4"], atol=1e-6)
    np.testing.assert_allclose(fluxhip.init_noise(128, 3, 5, 123), g["noise_123_3x5"], atol=1e-6)
    a = fluxhip.init_noise(128, 4, 4, 42)
    b = fluxhip.init_noise(128, 4, 4, -1)          # unseeded: continues the stream
    assert not np.array_equal(a, b)


def test_no_cpu_fallback():
    """Without a GPU nothing computes: init fails with a message and model creation raises."""
    L = fluxhip.lib()
    if L.flux_hip_init():
        pytest.skip("a GPU is present")
    assert b"HIP device" in L.flux_hip_last_error() or L.flux_hip_last_error()
    assert not L.flux_hip_available()
    assert not L.flux_hip_malloc(16)
    with pytest.raises(fluxhip.FluxHipError):
        fluxhip.Transformer(TINY)


def test_model_spec_and_synthetic_tensors(tmp_path):
    shapes = tensor_shapes(KLEIN_4B)
    assert len(shapes) == 169                                  # what the reference loader asks for
    assert sum(int(np.prod(s)) for s in shapes.values()) == 3_875_544_576
    W = make_weights(TINY, 42, 0.02, "sharp")
    W2 = make_weights(TINY, 42, 0.02, "sharp", only=["proj_out.weight"])
    assert np.array_equal(W["proj_out.weight"], W2["proj_out.weight"])      # streams are per tensor
    w = bf16_to_f32(W["context_embedder.weight"])
    assert abs(w.std() - 0.02) < 5e-4 and abs(w.mean()) < 5e-4
    assert np.all(bf16_to_f32(W["transformer_blocks.0.attn.norm_q.weight"]) == 1.0)
    x = normal_f32((1000,), 1, 1)
    assert np.array_equal(f32_to_bf16(bf16_to_f32(f32_to_bf16(x))), f32_to_bf16(x))
    # round to nearest even on the bf16 boundary
    edge = np.array([1.0 + 2.0 ** -8, 1.0 + 3 * 2.0 ** -8], np.float32)
    assert list(f32_to_bf16(edge)) == [0x3F80, 0x3F82]
    p = tmp_path / "t.safetensors"
    write_safetensors(str(p), W)
    raw = open(p, "rb").read()
    hlen = int.from_bytes(raw[:8], "little")
    import json
    meta = json.loads(raw[8:8 + hlen])
    assert meta["proj_out.weight"]["dtype"] == "BF16" and meta["proj_out.weight"]["shape"] == [128, 256]
    assert len(raw) == 8 + hlen + sum(a.size * 2 for a in W.values())


@pytest.mark.skipif(not os.path.isfile("/root/reference/flux_transformer.c"), reason="needs the reference checkout")
def test_reference_cli_links_against_the_library():
    """Drop-in check: the reference's own main.c / flux.c / text encoder / VAE link, unmodified,
    against libflux_hip.so once flux_transformer.c and flux_sample.c are left out."""
    import subprocess
    r = subprocess.run(["make", "-C", os.path.join(ROOT, "oracle"), "dropin"], capture_output=True, text=True)
    assert r.returncode == 0 and "linked _ref/flux_dropin" in r.stdout, r.stdout + r.stderr
    exe = os.path.join(ROOT, "oracle", "_ref", "flux_dropin")
    syms = subprocess.run(["nm", "-D", "--undefined-only", exe], capture_output=True, text=True).stdout
    for name in ("flux_sample_euler", "flux_sample_euler_cfg_with_multi_refs", "flux_transformer_forward",
                 "flux_transformer_load_safetensors_mmap", "flux_transformer_free", "flux_official_schedule",
                 "flux_init_noise"):
        assert re.search(rf"\bU {name}\b", syms), name          # imported from the shared library
    h = subprocess.run([exe, "--help"], capture_output=True, text=True)
    assert "Usage" in (h.stdout + h.stderr) or "usage" in (h.stdout + h.stderr)
    # the library level (flux.h) as a shared library over the backend, used by tests/test_hip_pipeline.py
    r = subprocess.run(["make", "-C", os.path.join(ROOT, "oracle"), "pipeline"], capture_output=True, text=True)
    assert r.returncode == 0 and "linked _ref/libfluxpipe.so" in r.stdout, r.stdout + r.stderr
    syms = subprocess.run(["nm", "-D", os.path.join(ROOT, "oracle", "_ref", "libfluxpipe.so")], capture_output=True, text=True).stdout
    for name in ("flux_sample_euler", "flux_transformer_forward", "flux_transformer_load_safetensors"):
        assert re.search(rf"\bU {name}\b", syms), name
    for name in ("flux_load_dir", "flux_generate_with_embeddings", "flux_denoise_step"):
        assert re.search(rf"\bT {name}\b", syms), name
    # the same with the VAE decoder taken from the backend: flux.c's three decoder-side calls are imports,
    # the reference's CPU decoder and encoder are still there under the renamed/original names
    r = subprocess.run(["make", "-C", os.path.join(ROOT, "oracle"), "pipeline_gpuvae"], capture_output=True, text=True)
    assert r.returncode == 0 and "linked _ref/libfluxpipe_gpuvae.so" in r.stdout, r.stdout + r.stderr
    syms = subprocess.run(["nm", "-D", os.path.join(ROOT, "oracle", "_ref", "libfluxpipe_gpuvae.so")], capture_output=True, text=True).stdout
    for name in ("flux_vae_decode", "flux_vae_load_safetensors", "flux_vae_free", "flux_sample_euler"):
        assert re.search(rf"\bU {name}\b", syms), name
    for name in ("flux_vae_decode_cpu", "flux_vae_encode", "flux_generate_with_embeddings"):
        assert re.search(rf"\bT {name}\b", syms), name
    # all stages from the backend: the VAE encoder is an import too, flux_qwen3.c is left out, the tokenizer stays
    r = subprocess.run(["make", "-C", os.path.join(ROOT, "oracle"), "pipeline_gpuall"], capture_output=True, text=True)
    assert r.returncode == 0 and "linked _ref/libfluxpipe_gpuall.so" in r.stdout, r.stdout + r.stderr
    syms = subprocess.run(["nm", "-D", os.path.join(ROOT, "oracle", "_ref", "libfluxpipe_gpuall.so")], capture_output=True, text=True).stdout
    for name in ("qwen3_encoder_load", "qwen3_encode_text", "qwen3_encoder_free", "flux_vae_decode", "flux_vae_encode", "flux_sample_euler"):
        assert re.search(rf"\bU {name}\b", syms), name
    for name in ("qwen3_tokenizer_load", "qwen3_tokenize_chat", "flux_generate", "flux_img2img", "flux_image_to_tensor"):
        assert re.search(rf"\bT {name}\b", syms), name
