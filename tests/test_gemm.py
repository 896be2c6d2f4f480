"""The projections of a decoder layer (include/crane_gemm.h): candle Linear
y = x W^T + b -- Crane's merged qkv_proj, whose rows feed the fused append
(qwen3/modeling.rs:382-387; with the Qwen2.5 bias, qwen25/qwen2.rs:136-138),
o_proj (:466, :502), the MLP projections and the lm_head; on hipBLASLt, or on
the per-wave ring, streaming and LDS-tile kernels for bf16 products of few rows.

The oracle's linear is pinned to numpy float64 matmul (a transposed weight
fails); the GPU is held to the oracle within the rounding bound of its two
differences (f32 accumulation in another order, and one rounding of product
+ bias where candle rounds twice) and the mean-relative bar, with weights
scaled like trained ones (std 1/sqrt(K)) so outputs are O(1)."""
import ctypes
import math
import os

import numpy as np
import pytest

import cases
from tolerance import assert_close, assert_ulp_close, bf16_ulp


def assert_linear_close(got, x, w, bias, dtype, orc, what):
    """Two references.  Against the oracle with the GPU's rounding (product +
    bias rounded once) every element lies within the f32 accumulation bound,
    K * 2^-24 * sum|x||w| (any summation order) plus one ulp, and at least 99%
    of them are bit-identical.  Against candle's (product rounded, then the
    sum) the two roundings differ by at most half an ulp at |p| plus an ulp at
    |y|: elements within 1.5 ulp of max(|y|, |p|, |b|) plus the accumulation
    bound, and the mean-relative bar.  f32: the f32 bar."""
    ref = orc.linear(x, w, bias, dtype)
    if dtype == "f32":
        return assert_close(got, ref, dtype, what)
    K = x.shape[-1]
    acc = (K * 2.0 ** -24) * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T)
    fused = orc.linear(x, w, bias, dtype, fused=True)
    d = np.abs(got.astype(np.float64) - fused)
    assert np.all(d <= acc + bf16_ulp(fused)), f"{what}: beyond the accumulation bound"
    exact = float(np.mean(got == fused))
    assert exact >= 0.99, f"{what}: only {exact:.4f} bit-identical to the fused-rounding oracle"
    b = np.zeros(ref.shape[-1], np.float32) if bias is None else bias
    scale = np.maximum(np.maximum(np.abs(ref), np.abs(ref - b)), np.abs(b))
    d2 = np.abs(got.astype(np.float64) - ref)
    assert np.all(d2 <= 1.5 * bf16_ulp(scale) + acc), f"{what}: beyond the candle rounding bound"
    from tolerance import errors, BF16_MEAN_REL
    assert errors(got, ref)[1] <= BF16_MEAN_REL, what


def _case(seed, M, N, K, dtype, bias=True):
    r = cases.rng(seed)
    x = cases.cast(cases.normal(r, (M, K)), dtype)
    w = cases.cast(cases.normal(r, (N, K), 1.0 / math.sqrt(K)), dtype)
    b = cases.cast(cases.normal(r, (N,), 0.5), dtype) if bias else None
    return x, w, b


# ------------------------------------------------------------------ CPU

def test_linear_oracle_vs_numpy_float64(orc):
    x, w, b = _case(1, 37, 96, 640, "bf16")
    exact = x.astype(np.float64) @ w.astype(np.float64).T
    y32 = orc.linear(x, w, None, "f32")
    assert np.max(np.abs(y32 - exact) / np.maximum(np.abs(exact), 1e-6)) < 1.5e-7
    yb = orc.linear(x, w, None, "bf16")
    assert np.all(np.abs(yb - exact) <= 0.5 * bf16_ulp(exact) * (1 + 1e-9))   # one rounding
    ybb = orc.linear(x, w, b, "bf16")
    np.testing.assert_array_equal(ybb, cases.bf16(yb + b[None, :]))          # then the bias in T
    wrong = orc.linear(x, np.ascontiguousarray(w[:, ::-1]), None, "f32")      # a planted mistake
    assert np.max(np.abs(wrong - exact)) > 0.5
    fb = orc.linear(x, w, b, "bf16", fused=True)                               # epilogue rounding
    assert np.all(np.abs(fb - (exact + b)) <= 0.5 * bf16_ulp(exact + b) * (1 + 1e-9))


def test_gemm_null_context():
    from crane_amd import _lib
    assert _lib.lib().crane_gemm_linear(None, 16, 16, None, 16, 4, 4, 4, 1, None) == _lib.E_INVALID


def test_gated_shape_query():
    """Which shapes the one-launch gate_up + SiLU*mul takes (host logic, no
    GPU): bf16, at most 32 token rows, K <= 8192, inter > 4096 with inter a
    multiple of 48 (K of 512) or of 32 (K of 1024)."""
    from crane_amd import _lib
    q = _lib.lib().crane_gemm_silu_mul_supported
    BF16, F32 = 1, 0
    assert q(32, 12288, 4096, BF16) == 1      # Qwen3-8B decode gate_up
    assert q(1, 12288, 512, BF16) == 1
    assert q(3, 4160, 1024, BF16) == 1        # 32-feature pairs
    assert q(3, 4160, 512, BF16) == 0         # ... which need K % 1024
    assert q(33, 12288, 4096, BF16) == 0      # more token rows than the kernel takes
    assert q(0, 12288, 4096, BF16) == 0
    assert q(32, 4096, 4096, BF16) == 0       # narrow: the two-call path
    assert q(32, 12288, 4096, F32) == 0
    assert q(32, 12296, 4096, BF16) == 0      # inter a multiple of neither 48 nor 32
    assert q(32, 12288, 12288, BF16) == 0     # K past the ring kernel's limit
    assert _lib.lib().crane_gemm_linear_silu_mul(None, 16, 16, 16, 4, 12288, 4096, BF16, None) == _lib.E_INVALID


# ------------------------------------------------------------------ GPU

def _t(x, dtype, dev):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(x))
    return (t.to(torch.bfloat16) if dtype == "bf16" else t).to(dev)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("M,N,K,bias", [
    (64, 4608, 3584, True),    # Qwen2.5-7B qkv_proj (28 q + 2 x 4 kv heads), with bias
    (32, 6144, 4096, False),   # Qwen3-8B qkv_proj at the c3 decode batch
    (300, 3584, 3584, False),  # Qwen2.5-7B o_proj
    (5, 136, 72, True),        # odd small shape
])
def test_linear_parity(gpu, orc, dtype, M, N, K, bias):
    from crane_amd import ops
    print(f"linear {dtype} M={M} N={N} K={K} bias={bias}", flush=True)
    x, w, b = _case(500 + N, M, N, K, dtype, bias)
    got = ops.linear(_t(x, dtype, gpu), _t(w, dtype, gpu), _t(b, dtype, gpu) if bias else None)
    assert_linear_close(got.float().cpu().numpy(), x, w, b, dtype, orc, f"linear {M}x{N}x{K}")
    # twice: the cached plan gives the same bits
    got2 = ops.linear(_t(x, dtype, gpu), _t(w, dtype, gpu), _t(b, dtype, gpu) if bias else None)
    assert bool((got == got2).all())


@pytest.mark.gpu
@pytest.mark.parametrize("workspace", [0, 1 << 20])
def test_library_product_keeps_to_its_workspace(gpu, workspace):
    """Qwen2.5-7B gate_up over 1000 token rows: hipBLASLt's first choice needs
    64 MiB of workspace, whatever limit it was given.  The context takes an
    algorithm its own workspace holds (the default's 64 MiB, and 1 MiB).
    Every value lies within an ulp and the f32 accumulation bound of the f32
    product."""
    import ctypes
    import torch
    from crane_amd import _lib
    M, N, K = 1000, 37888, 3584
    print(f"linear with a workspace of {workspace} bytes, M={M} N={N} K={K}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(17)
    x = torch.randn((M, K), generator=gen, device=gpu, dtype=torch.bfloat16)
    w = torch.randn((N, K), generator=gen, device=gpu, dtype=torch.bfloat16) * K ** -0.5
    y = torch.empty((M, N), dtype=torch.bfloat16, device=gpu)
    lib = _lib.lib()
    h = ctypes.c_void_p()
    _lib.check(lib.crane_gemm_create(workspace, ctypes.byref(h)), "create")
    try:
        _lib.check(lib.crane_gemm_linear(h, x.data_ptr(), w.data_ptr(), None, y.data_ptr(), M, N, K, _lib.BF16,
                                         torch.cuda.current_stream(gpu).cuda_stream), "linear")
        torch.cuda.synchronize()
    finally:
        lib.crane_gemm_destroy(h)
    for n0 in range(0, N, 9472):
        ref = x.float() @ w[n0:n0 + 9472].float().T
        bound = x.float().abs() @ w[n0:n0 + 9472].float().abs().T * (2 * K * 2.0 ** -24) + ref.abs() * 2.0 ** -8 + 1e-30
        assert bool(((y[:, n0:n0 + 9472].float() - ref).abs() <= bound).all())


def _rule(name, nargs):
    """One of gemm.hip's dispatch rules (host logic), by its C++ name."""
    from crane_amd import _lib
    fn = getattr(_lib.lib(), f"_ZN5crane{len(name)}{name}E" + "l" * nargs)
    fn.argtypes, fn.restype = [ctypes.c_int64] * nargs, ctypes.c_bool
    return fn


def test_stream_rule():
    """Wide products of few rows over a short K take the streaming kernel, at the
    lines both of whose sides were measured."""
    takes = _rule("stream_takes", 3)
    for M, N, K in [(1, 151936, 896), (16, 32000, 1024), (4, 57344, 256), (32, 16384, 640), (17, 16448, 384),
                    (1, 16384, 128)]:
        assert takes(M, N, K), (M, N, K)
    for M, N, K in [(1, 151936, 1152), (17, 151936, 768), (33, 32000, 256), (1, 16320, 256), (1, 32008, 256),
                    (1, 32000, 192), (0, 32000, 256)]:
        assert not takes(M, N, K), (M, N, K)


def test_ring_rule():
    """Wide products the ring kernel takes too go to the LDS-tile kernel only past
    16 rows or a K of 4096."""
    yields = _rule("ring_yields", 3)
    for M, N, K in [(17, 151936, 2048), (32, 40960, 1024), (1, 151936, 5120), (16, 32784, 8192)]:
        assert yields(M, N, K), (M, N, K)
    for M, N, K in [(1, 151936, 1024), (16, 151936, 2048), (8, 40960, 4096), (32, 32768, 8192)]:
        assert not yields(M, N, K), (M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,bias", [
    (32, 16384, 1152, False),  # the decode batch of config 3; 9 stages of 128
    (17, 16448, 384, True),    # a partial second token group; 3 stages; 257 workgroups
    (8, 16384, 640, True),     # 5 stages: the unrolled-by-three loop's remainder of 2
    (1, 16384, 256, True),     # one token row; 2 stages
    (3, 20480, 128, False),    # one stage
    (16, 16448, 896, True),    # 7 stages: the loop's remainder of 1; a full token group
    (32, 16384, 640, False),   # two full token groups, the longest K for them
])
def test_linear_streaming_parity(gpu, orc, M, N, K, bias):
    """Wide bf16 products with few token rows run the streaming kernel over a
    short K (the first of them the LDS-tile kernel) when K is not a whole number
    of the per-wave ring kernel's pipelines; same bar as the library path."""
    from crane_amd import ops
    print(f"linear (streaming) M={M} N={N} K={K} bias={bias}", flush=True)
    x, w, b = _case(900 + M + K, M, N, K, "bf16", bias)
    got = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert_linear_close(got.float().cpu().numpy(), x, w, b, "bf16", orc, f"streaming linear {M}x{N}x{K}")
    got2 = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert bool((got == got2).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,bias", [
    (32, 4096, 4096, False),   # o_proj at the c3 decode batch: 16 features x 4 waves, 2 stages ahead
    (5, 4096, 2048, True),     # one token group; each wave's 4 stages fill the ring once (no loop trip)
    (3, 2048, 6144, True),     # 128 workgroups; 12 stages a wave
    (32, 6144, 4096, True),    # qkv_proj at c3: 32 features x 2 waves, rotated k walk (16 stages)
    (17, 8192, 1024, False),   # a partial second token group; 4 stages a wave, rotation over 4
    (32, 24576, 1024, True),   # gate_up's N: 96 features x 2 waves (256 workgroups), rotated k walk
    (32, 24576, 1536, False),  # ... K a multiple of 512, not of 1024: still 96 features (6 stages a wave)
    (32, 16384, 2048, True),   # 64 features x 4 waves (256 workgroups)
    (9, 9072, 1024, False),    # N a multiple of 48, not of 64: 48 features
    (1, 12288, 2048, False),   # one token row, wide (48 features: 256 workgroups)
    (32, 4096, 12288, False),  # down_proj's shape: K past the ring kernel's limit, the LDS-tile kernel in splits
])
def test_linear_ring_parity(gpu, orc, M, N, K, bias):
    """bf16 products with M <= 32 token rows, N a multiple of the workgroup's
    16/32 or 48/64/96 features (N <= 4096 / <= 8192 / wider) and K <= 8192 a
    whole number of the per-wave rings (K % 2048 == 0 for the narrowest, 1024
    or 512 for the others) run the per-wave ring kernel: the decode step's qkv_proj,
    o_proj and gate_up (a longer K takes the LDS tiles).  Same bar as the library path, and a second
    call repeats the bits (the waves' partial products are added in a fixed
    order)."""
    from crane_amd import ops
    print(f"linear (ring) M={M} N={N} K={K} bias={bias}", flush=True)
    x, w, b = _case(1300 + M + N // 64 + K, M, N, K, "bf16", bias)
    got = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert_linear_close(got.float().cpu().numpy(), x, w, b, "bf16", orc, f"ring linear {M}x{N}x{K}")
    got2 = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert bool((got == got2).all())


class TileCfg(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("ft", "mt", "splits")]


class TileArgs(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "w", "bias", "y", "parts")] + \
               [(n, ctypes.c_int) for n in ("M", "N", "K")]


def launch_tile(out, cfg, args, stream=None):
    """One form (cfg) of the LDS-tile kernel with output "rows", "gated" or
    "parts" (tile_gemm.h); False where it has no kernel."""
    from crane_amd import _lib
    name = f"launch_tile_{out}"
    fn = getattr(_lib.lib(), f"_ZN5crane{len(name)}{name}ERKNS_7TileCfgERKNS_8TileArgsEP12ihipStream_t")
    fn.argtypes, fn.restype = [ctypes.c_void_p] * 3, ctypes.c_bool
    c, a = TileCfg(*cfg), TileArgs(*args)
    return fn(ctypes.addressof(c), ctypes.addressof(a), stream)


def _tile_rule(name, M, N, K, gated, ws_bytes):
    from crane_amd import _lib
    fn = getattr(_lib.lib(), f"_ZN5crane{len(name)}{name}Elllbm")
    fn.argtypes, fn.restype = [ctypes.c_int64] * 3 + [ctypes.c_bool, ctypes.c_size_t], TileCfg
    c = fn(M, N, K, gated, ws_bytes)
    return c.ft, c.mt, c.splits


def test_tile_launch_refuses_a_form_without_a_kernel():
    """A form that has no kernel for the row count (4 token tiles that do not
    cover the rows, 4 feature by 4 token tiles) launches nothing and says so:
    every product's caller returns an error instead of an unwritten output."""
    for out in ("rows", "gated", "parts"):
        for ft, mt in ((1, 4), (2, 4), (3, 4), (4, 4)):
            assert not launch_tile(out, (ft, mt, 1), (16, 16, None, 16, 16, 129, 512, 512)), (out, ft, mt)


def tile_form(M, N, K, gated=False, ws_bytes=64 << 20):
    """The LDS-tile kernel's form of a product of M rows and N weight rows:
    (features / 32 per workgroup (/ 16 gated), token rows / 32, splits of K)."""
    return _tile_rule("tile_cfg", M, N, K, gated, ws_bytes)


@pytest.mark.parametrize("M,N,K,form", [
    (200, 4608, 3584, (2, 3, 1)),   # 17.9 us; (4, 1, 1), 252 workgroups of which 35 on each of four XCDs, 33.8
    (257, 3584, 3584, (2, 3, 1)),   # 21.3; (4, 1, 1) 33.3
    (320, 4096, 14336, (4, 3, 2)),  # 62.1; (2, 3, 1), 256 workgroups in 8 rounds of feature tiles, 107.9
    (129, 2560, 9728, (3, 3, 4)),   # 23.2; (4, 2, 4) 38.6
    (320, 1536, 8960, (3, 3, 4)),   # 22.5; (1, 2, 1) 40.3
    (77, 4096, 12288, (2, 3, 4)),   # 27.1, the fastest by either count
    (300, 4608, 3584, (3, 2, 1)),   # 22.6, likewise
    (200, 3584, 18944, (4, 2, 2)),  # 63.4; (3, 3, 2) 72.8
    (208, 3776, 23808, (4, 2, 2)),  # 82.8; (3, 3, 2) 101.3
    (77, 1024, 3072, (1, 1, 1)),    # a split saves 2 us on the GPU and costs a launch
])
def test_tile_form_counts_workgroups_by_xcd(M, N, K, form):
    """Token blocks and splits of a feature tile share an XCD: the choice is a form
    at or near the measured fastest (us in the list) also where an even spread over
    the chip is uneven over the XCDs (host logic)."""
    assert tile_form(M, N, K) == form


def tile_taken(M, N, K, gated=False, ws_bytes=64 << 20):
    """Whether a product of M rows goes to the LDS-tile kernel."""
    return _tile_rule("tile_route", M, N, K, gated, ws_bytes)[0] != 0


def test_tile_route_follows_the_measured_sides():
    """Products measured slower on the LDS-tile kernel than on the library (us,
    tile and library) stay with the library, faster ones on the kernel (host
    logic)."""
    from crane_amd import _lib
    slower = [
        (128, 57344, 3584), (128, 28672, 18944),    # 119, 84; 302, 222: wide past 96 rows
        (77, 57344, 1024), (37, 49752, 896),        # 33.8, 27.2; 23.7, 20.1: wide over a short K
        (321, 2048, 1024),                          # past the rows compared
    ]
    faster = [
        (300, 4608, 3584), (200, 6144, 4096),       # 23.3, 23.9; 22.4, 26.3
        (77, 24576, 4096), (77, 4096, 12288),       # 37.2, 50.0; 27.4, 42.6
        (224, 8192, 28672), (11, 96, 18496),        # 204, 259; 35.6, 58.2
        (128, 4096, 4096), (128, 24576, 4096),      # 16.5, 24.1; 44, 52
        (32, 3584, 18944), (32, 151936, 4096),      # 27.6, 105; 200, 222
        (1, 1024, 1024), (250, 1000, 768),          # small ones
    ]
    for shape in slower:
        assert not tile_taken(*shape), shape
    for shape in faster:
        assert tile_taken(*shape), shape
    q, s = _lib.lib().crane_gemm_tile_silu_mul_preferred, _lib.lib().crane_gemm_tile_silu_mul_supported
    for M, inter, K in [(1, 768, 8192), (8, 1536, 4096), (121, 56, 11264)]:   # 17.9, 10.4; 11.4, 8.9; 25.2, 17.3
        assert s(M, inter, K, 1) and not q(M, inter, K, 1), (M, inter, K)
    assert s(128, 16384, 5120, 1) and not q(128, 16384, 5120, 1)              # 97.6, 75.7
    for M, inter, K in [(77, 12288, 4096), (77, 3072, 1024), (20, 18944, 3584), (1, 768, 1024)]:  # 39.0, 52.7; ...
        assert q(M, inter, K, 1), (M, inter, K)
    assert not s(321, 1024, 1024, 1) and not q(321, 1024, 1024, 1) and not q(8, 1024, 1024, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,bias", [
    (33, 4096, 64, True),      # one stage; a second token tile of one row
    (40, 1000, 448, True),     # N a multiple of 8 only: a last tile of 8 features; 7 stages, ring of 6
    (64, 200, 4096, False),    # few features: 8 splits of K, two whole token tiles
    (77, 2056, 1024, True),    # 13 rows of the last of three token tiles, each a block of its own
    (97, 512, 2048, False),    # four blocks of one token tile, the last of one row
    (129, 4096, 640, True),    # two blocks of 3 token tiles, the second of 33 rows
    (224, 1024, 3072, False),  # the last row count at any K
    (320, 2048, 1024, True),   # the last row count of the kernel
    (321, 2048, 1024, True),   # ... and the library's first
    (1, 32776, 192, True),     # one row, N past the ring kernel's: 3 stages, a last tile of 8 features
    (20, 1024, 3072, False),   # a decode batch over a small weight, split
    (32, 512, 8256, True),     # K past the ring kernel's limit, 129 stages: no even split
])
def test_linear_tile_parity(gpu, orc, M, N, K, bias):
    """bf16 products on the LDS-tile kernel, at the edges of its tiles, rings,
    splits and row limits; same bar as the library path, and a second call
    repeats the bits (fixed summation order)."""
    from crane_amd import ops
    print(f"linear (tile) M={M} N={N} K={K} bias={bias}", flush=True)
    x, w, b = _case(2100 + M + N + K, M, N, K, "bf16", bias)
    got = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert_linear_close(got.float().cpu().numpy(), x, w, b, "bf16", orc, f"tile linear {M}x{N}x{K}")
    got2 = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert bool((got == got2).all())


TILE_FORMS = [(ft, mt) for ft in range(1, 5) for mt in range(1, 5 if ft < 4 else 4)]


def _tile_shapes(ft, mt):
    """(M, features, stages) of a form: 9 feature tiles, the last of 8 features,
    over rows in one block and (up to 3 token tiles) two, each ending in a partial
    tile; 2 D - 1 stages of a ring of D, a turn and the longest remainder."""
    d = min(6, 40 // (ft + mt))
    for M in [32 * mt - 3] + ([32 * mt + 9] if mt < 4 else []):
        yield M, lambda per: 8 * per * ft + 8, 2 * d - 1


@pytest.mark.gpu
@pytest.mark.parametrize("ft,mt", TILE_FORMS)
def test_tile_forms(gpu, orc, ft, mt):
    """Every form of the LDS-tile kernel, launched directly: the output rows with
    bias, and 2 splits' f32 partial products summed in split order."""
    import torch
    from crane_amd import ops
    for M, features, stages in _tile_shapes(ft, mt):
        N, K = features(32), 64 * stages
        print(f"tile form {ft} x {mt}: M={M} N={N} K={K}", flush=True)
        x, w, b = _case(2700 + 10 * ft + mt + M, M, N, 2 * K, "bf16", True)
        h, wh = np.ascontiguousarray(x[:, :K]), np.ascontiguousarray(w[:, :K])
        xd, wd, bd = _t(h, "bf16", gpu), _t(wh, "bf16", gpu), _t(b, "bf16", gpu)
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=gpu)
        assert launch_tile("rows", (ft, mt, 1), (xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), y.data_ptr(), None, M, N,
                                                 K), ops._stream(gpu))
        assert_linear_close(y.float().cpu().numpy(), h, wh, b, "bf16", orc, f"tile rows {ft}x{mt} {M}x{N}x{K}")
        xd, wd = _t(x, "bf16", gpu), _t(w, "bf16", gpu)
        parts = torch.full((2, M, N), float("nan"), device=gpu)
        assert launch_tile("parts", (ft, mt, 2), (xd.data_ptr(), wd.data_ptr(), None, None, parts.data_ptr(), M, N,
                                                  2 * K), ops._stream(gpu))
        got = cases.bf16((parts[0] + parts[1]).cpu().numpy())
        assert_linear_close(got, x, w, None, "bf16", orc, f"tile parts {ft}x{mt} {M}x{N}x{2 * K}")


@pytest.mark.gpu
@pytest.mark.parametrize("ft,mt", TILE_FORMS + [(5, 1), (5, 2), (5, 3)])
def test_tile_gated_forms(gpu, orc, ft, mt):
    """Every gated form of the LDS-tile kernel, launched directly, against the
    oracle chain within the bound of its roundings."""
    import torch
    from crane_amd import ops
    for M, features, stages in _tile_shapes(ft, mt):
        inter, K = features(16), 64 * stages
        print(f"gated tile form {ft} x {mt}: M={M} inter={inter} K={K}", flush=True)
        x, w, _ = _case(2900 + 10 * ft + mt + M, M, 2 * inter, K, "bf16", False)
        xd, wd = _t(x, "bf16", gpu), _t(w, "bf16", gpu)
        y = torch.full((M, inter), float("nan"), dtype=torch.bfloat16, device=gpu)
        assert launch_tile("gated", (ft, mt, 1), (xd.data_ptr(), wd.data_ptr(), None, y.data_ptr(), None, M, 2 * inter,
                                                  K), ops._stream(gpu))
        ref, bound = _silu_mul_bound(x, w, orc)
        got = y.float().cpu().numpy()
        assert np.all(np.abs(got.astype(np.float64) - ref) <= bound)
        assert float(np.mean(got == ref)) >= 0.98


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits,bias", [
    (33, 200, 5760, 2, True), (12, 400, 3840, 4, True), (37, 136, 3584, 8, True), (290, 72, 4864, 4, False),
])
def test_linear_tile_splits(gpu, orc, M, N, K, splits, bias):
    """Products whose K the LDS-tile kernel splits: the sums through the context's
    workspace, with and without the bias; in a context too small for them the
    product runs unsplit."""
    import torch
    from crane_amd import _lib, ops
    assert tile_taken(M, N, K) and tile_form(M, N, K)[2] == splits and tile_form(M, N, K, ws_bytes=4096)[2] == 1
    print(f"linear (tile, {splits} splits) M={M} N={N} K={K} bias={bias}", flush=True)
    x, w, b = _case(3000 + M + N + K, M, N, K, "bf16", bias)
    xd, wd, bd = _t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None
    got = ops.linear(xd, wd, bd)
    assert_linear_close(got.float().cpu().numpy(), x, w, b, "bf16", orc, f"tile splits {M}x{N}x{K}")
    assert torch.equal(got, ops.linear(xd, wd, bd))
    h = ctypes.c_void_p()
    assert _lib.lib().crane_gemm_create(4096, ctypes.byref(h)) == 0
    try:
        y = torch.empty_like(got)
        assert _lib.lib().crane_gemm_linear(h, xd.data_ptr(), wd.data_ptr(), bd.data_ptr() if bias else None,
                                            y.data_ptr(), M, N, K, _lib.BF16, ops._stream(gpu)) == 0
        assert_linear_close(y.float().cpu().numpy(), x, w, b, "bf16", orc, f"tile unsplit {M}x{N}x{K}")
    finally:
        _lib.lib().crane_gemm_destroy(h)


def test_split_shape_query():
    """Which shapes the split-K partial products take (host logic, no GPU):
    bf16, at most 32 token rows, N a multiple of 32 or 48, K a multiple of the
    splits with a share of at most 32768 that is a multiple of 512 (of 256
    from 3072 up: one wave a workgroup), 2 to 16 splits."""
    from crane_amd import _lib
    q = _lib.lib().crane_gemm_split_supported
    BF16, F32 = 1, 0
    assert q(32, 4096, 4096, 4, BF16) == 1    # Qwen3-8B decode o_proj
    assert q(32, 4096, 12288, 4, BF16) == 1   # ... and down_proj
    assert q(1, 64, 2048, 2, BF16) == 1
    assert q(32, 6144, 4096, 2, BF16) == 1    # ... and qkv_proj
    assert q(32, 4096, 4096, 3, BF16) == 0    # K not a multiple of the splits
    assert q(32, 4096, 2048, 4, BF16) == 1    # 512 per split: one ring turn of 2 waves
    assert q(32, 4096, 1024, 4, BF16) == 0    # 256 per split: less than a ring turn
    assert q(32, 4096, 3840, 2, BF16) == 0    # 1920 per split (2 waves): not a multiple of 512
    assert q(32, 4096, 6656, 2, BF16) == 1    # 3328 per split (1 wave): a multiple of 256
    assert q(33, 4096, 4096, 4, BF16) == 0    # more token rows than the kernel takes
    assert q(32, 4100, 4096, 4, BF16) == 0    # N not a multiple of 32 or 48
    assert q(32, 4112, 4096, 4, BF16) == 0    # ... nor of 48
    assert q(32, 144, 4096, 4, BF16) == 1     # 3 tiles of 48 features
    assert q(32, 4096, 4096, 1, BF16) == 0    # no split
    assert q(32, 4096, 4096, 4, F32) == 0
    assert q(32, 4096, 65536, 2, BF16) == 1   # 32768 per split: the limit
    assert q(32, 4096, 131072, 2, BF16) == 0  # ... past it
    assert _lib.lib().crane_gemm_linear_split(None, 16, 16, 16, 4, 4096, 4096, 4, BF16, None) == _lib.E_INVALID


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits", [
    (32, 4096, 4096, 4),    # o_proj at the c3 decode batch: 64 workgroups of 64 features x 4 splits, 2 waves
    (32, 4096, 12288, 4),   # down_proj at c3: 1 wave, 24 stages through a ring of 3
    (32, 6144, 4096, 2),    # qkv_proj at c3: 128 workgroups of 48 features x 2 splits
    (5, 1024, 2048, 2),     # one token group, 32 features a workgroup; one ring turn a wave
    (17, 256, 8192, 8),     # a partial second token group, 8 splits
    (1, 640, 3072, 3),      # one token row, 3 splits
    (9, 512, 6144, 2),      # one token group, 1 wave, ring of 3
    (20, 320, 9216, 3),     # a partial second token group, 10 feature tiles, 1 wave, ring of 3
    (11, 336, 3072, 2),     # 48 features, 2 waves, ring of 3
    (24, 48, 8192, 2),      # one 48-feature tile, 1 wave, ring of 2
])
def test_linear_split_parity(gpu, orc, M, N, K, splits):
    """The f32 partial products of crane_gemm_linear_split, summed in split
    order and rounded once, are the product at the library path's bar; a
    second call repeats the bits."""
    import torch
    from crane_amd import _lib, ops
    print(f"linear split M={M} N={N} K={K} splits={splits}", flush=True)
    x, w, _ = _case(1700 + M + N // 64 + K, M, N, K, "bf16", False)
    xd, wd = _t(x, "bf16", gpu), _t(w, "bf16", gpu)
    outs = []
    for _ in range(2):
        parts = torch.empty((splits, M, N), dtype=torch.float32, device=gpu)
        assert _lib.lib().crane_gemm_linear_split(ops._gemm(gpu)._h, xd.data_ptr(), wd.data_ptr(), parts.data_ptr(),
                                                  M, N, K, splits, _lib.BF16, ops._stream(gpu)) == 0
        outs.append(parts.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    acc = np.zeros((M, N), np.float32)
    for p in outs[0]:
        acc = (acc + p).astype(np.float32)
    assert_linear_close(cases.bf16(acc), x, w, None, "bf16", orc, f"split linear {M}x{N}x{K}/{splits}")


def _silu_mul_bound(x, w, orc):
    """The oracle chain of the gated product and a per-element bound for the
    GPU: each projection lies within the f32 accumulation bound plus one ulp
    of its rounding; out = silu(g) u moves by at most |u| |silu'(g)| <= 1.1 |u|
    per unit of g and |silu(g)| per unit of u, plus two ulps (its own rounding
    and the f32 exp)."""
    K = x.shape[-1]
    gu = orc.linear(x, w, None, "bf16", fused=True)
    acc = (K * 2.0 ** -24) * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T)
    dgu = acc + bf16_ulp(gu)
    inter = w.shape[0] // 2
    g, u = gu[:, :inter].astype(np.float64), gu[:, inter:].astype(np.float64)
    silu = g / (1.0 + np.exp(-g))
    ref = orc.silu_mul(gu, False, "bf16")
    bound = 1.1 * np.abs(u) * dgu[:, :inter] + np.abs(silu) * dgu[:, inter:] + 2 * bf16_ulp(ref)
    return ref, bound


@pytest.mark.gpu
@pytest.mark.parametrize("M,inter,K", [
    (1, 40, 64),        # one stage; a last tile of 8 outputs
    (32, 3072, 1024),   # narrow: past the ring kernel's gated shapes
    (33, 18944, 256),   # 80 outputs a workgroup in one round
    (77, 6144, 512),    # three token tiles
    (97, 1032, 448),    # two blocks of 2 token tiles; 8 outputs in the last tile
    (300, 2048, 576),   # four blocks of 3 token tiles
])
def test_linear_silu_mul_tile_parity(gpu, orc, M, inter, K):
    """crane_gemm_tile_silu_mul against the oracle chain within the bound of
    its roundings, bit-repeatable."""
    from crane_amd import _lib, ops
    assert _lib.lib().crane_gemm_silu_mul_supported(M, inter, K, _lib.BF16) == 0
    assert _lib.lib().crane_gemm_tile_silu_mul_supported(M, inter, K, _lib.BF16) == 1
    print(f"silu_mul (tile) M={M} inter={inter} K={K}", flush=True)
    x, w, _ = _case(2500 + M + inter + K, M, 2 * inter, K, "bf16", False)
    ref, bound = _silu_mul_bound(x, w, orc)
    xd, wd = _t(x, "bf16", gpu), _t(w, "bf16", gpu)
    got = ops.linear_silu_mul(xd, wd)
    assert np.all(np.abs(got.float().cpu().numpy().astype(np.float64) - ref) <= bound)
    assert bool((got == ops.linear_silu_mul(xd, wd)).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,inter,K", [
    (32, 12288, 4096),  # Qwen3-8B decode: 48 gate + 48 up features a workgroup, 256 workgroups
    (17, 9216, 1024),   # partial second token group
    (1, 12288, 512),    # one token row; each wave's two stages fill the ring once
    (3, 4160, 1024),    # inter a multiple of 32, not 48: 32 + 32 features, one token group
    (24, 4160, 2048),   # the same with two token groups
])
def test_linear_silu_mul_parity(gpu, orc, M, inter, K):
    """crane_gemm_linear_silu_mul (one launch) against the oracle chain
    linear -> silu_mul (candle's Mlp at qwen3/modeling.rs:573-585 with Crane's
    fused_silu_mul): every element within the propagated accumulation bound,
    at least 98% bit-identical, the mean-relative bar, and a second call
    repeats the bits.  The two-call GPU path (ops.linear + ops.silu_mul) lies
    within the same bound."""
    from crane_amd import _lib, ops
    from tolerance import errors, BF16_MEAN_REL
    assert _lib.lib().crane_gemm_silu_mul_supported(M, inter, K, 1) == 1
    print(f"linear_silu_mul M={M} inter={inter} K={K}", flush=True)
    x, w, _ = _case(1700 + M + inter // 64 + K, M, 2 * inter, K, "bf16", False)
    ref, bound = _silu_mul_bound(x, w, orc)
    xt, wt = _t(x, "bf16", gpu), _t(w, "bf16", gpu)
    got = ops.linear_silu_mul(xt, wt)
    g = got.float().cpu().numpy()
    assert g.shape == (M, inter)
    d = np.abs(g.astype(np.float64) - ref)
    assert np.all(d <= bound), f"gated {M}x{inter}x{K}: beyond the bound by {float((d - bound).max())}"
    exact = float(np.mean(g == ref))
    assert exact >= 0.98, f"gated {M}x{inter}x{K}: only {exact:.4f} bit-identical"
    assert errors(g, ref)[1] <= BF16_MEAN_REL
    assert bool((ops.linear_silu_mul(xt, wt) == got).all())
    two = ops.silu_mul(ops.linear(xt, wt)).float().cpu().numpy()
    assert np.all(np.abs(two.astype(np.float64) - ref) <= bound)


N_RANDOM = int(os.environ.get("CRANE_RANDOM_GEMM", 12))
SEED = int(os.environ.get("CRANE_RANDOM_SEED", 0))


def linear_draw(seed: int, i: int):
    """Draw i of the randomised decode-projection sweep: (M, N, K, bias) with
    1-32 token rows, cycling over the shapes each path takes -- the ring
    kernel's three configurations (N <= 4096, <= 8192, wider), wide N with K not
    a multiple of 1024 (the streaming and LDS-tile kernels) and anything else
    (the latter or hipBLASLt) -- and M N K at most 1.5e9 so the oracle finishes in seconds."""
    r = cases.rng(seed + 9100 + i)
    M = int(r.integers(1, 33))
    kind = i % 5
    if kind == 0:
        N, K = 16 * int(r.integers(1, 257)), 2048 * int(r.integers(1, 5))
    elif kind == 1:
        N, K = 32 * int(r.integers(129, 257)), 1024 * int(r.integers(1, 9))
    elif kind == 2:
        N, K = 64 * int(r.integers(129, 1025)), 1024 * int(r.integers(1, 5))
    elif kind == 3:
        N, K = 64 * int(r.integers(256, 513)), 128 * int(r.choice([1, 3, 5, 7, 9, 11, 13]))
    else:
        N, K = int(r.integers(1, 3000)), int(r.integers(1, 1500))
    while M * N * K > 1.5e9 and K > 1024:
        K -= 1024
    return M, N, K, bool(r.random() < 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(N_RANDOM))
def test_random_decode_linear(gpu, orc, i):
    """Random decode-shaped bf16 products against the oracle (same bar as the
    fixed shapes), each repeated for identical bits."""
    from crane_amd import ops
    M, N, K, bias = linear_draw(SEED, i)
    print(f"random linear {i} (seed {SEED}): M={M} N={N} K={K} bias={bias}", flush=True)
    x, w, b = _case(SEED + 9200 + i, M, N, K, "bf16", bias)
    got = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert_linear_close(got.float().cpu().numpy(), x, w, b, "bf16", orc, f"random linear {M}x{N}x{K}")
    got2 = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None)
    assert bool((got == got2).all())


def tile_draw(seed: int, i: int, gated: bool):
    """Draw i of the LDS-tile kernel's random sweep: (M, N, K) it takes, 1 to 320
    rows in its four row ranges, N (gated: inter) a multiple of 8 and K of 64, M N
    K at most 8e8."""
    r = cases.rng(seed + (9300 if gated else 9400) + i)
    lo, hi = ((1, 32), (33, 96), (97, 128), (129, 320))[i % 4]
    while True:
        M = int(r.integers(lo, hi + 1))
        N, K = 8 * int(2 ** r.uniform(0, 9.5)), 64 * int(2 ** r.uniform(0, 6.5))
        rows = 2 * N if gated else N
        if M * rows * K <= 8e8 and tile_taken(M, rows, K, gated, 0 if gated else 64 << 20):
            return M, N, K


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(N_RANDOM))
def test_random_tile_linear(gpu, orc, i):
    """Random shapes of the LDS-tile kernel through the projections' entry points,
    plain and gated, at the bars of the fixed shapes."""
    from crane_amd import _lib, ops
    M, N, K = tile_draw(SEED, i, False)
    print(f"random tile linear {i} (seed {SEED}): M={M} N={N} K={K} {tile_form(M, N, K)}", flush=True)
    x, w, b = _case(SEED + 9350 + i, M, N, K, "bf16", i % 2 == 0)
    got = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), None if b is None else _t(b, "bf16", gpu))
    assert_linear_close(got.float().cpu().numpy(), x, w, b, "bf16", orc, f"random tile linear {M}x{N}x{K}")
    M, inter, K = tile_draw(SEED, i, True)
    print(f"  gated: M={M} inter={inter} K={K} {tile_form(M, 2 * inter, K, True)}", flush=True)
    assert _lib.lib().crane_gemm_tile_silu_mul_preferred(M, inter, K, 1) == 1
    x, w, _ = _case(SEED + 9450 + i, M, 2 * inter, K, "bf16", False)
    ref, bound = _silu_mul_bound(x, w, orc)
    got = ops.linear_silu_mul(_t(x, "bf16", gpu), _t(w, "bf16", gpu)).float().cpu().numpy()
    assert np.all(np.abs(got.astype(np.float64) - ref) <= bound), f"random gated tile {M}x{inter}x{K}"


def split_draw(seed: int, i: int):
    """Draw i of the randomised split-K sweep: (M, N, K, splits) that
    crane_gemm_split_supported takes, cycling over the feature widths (N a
    multiple of 64, of 48, of 32) and the two wave counts (a share of K below
    3072, a multiple of 512, takes 2 waves; from 3072, a multiple of 256, 1),
    with M N K at most 1.5e9."""
    r = cases.rng(seed + 9700 + i)
    M = int(r.integers(1, 33))
    splits = int(r.choice([2, 3, 4, 6, 8]))
    base = (64, 48, 32)[i % 3]
    N = base * int(r.integers(1, 129))
    share = 512 * int(r.integers(1, 6)) if (i // 3) % 2 == 0 else 256 * int(r.integers(12, 33))
    while M * N * splits * share > 1.5e9 and N > base:
        N -= base
    return M, N, splits * share, splits


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(N_RANDOM))
def test_random_linear_split(gpu, orc, i):
    """Random shapes of the split-K partial products, summed in split order
    and rounded once, against the oracle at the bar of
    test_linear_split_parity; a second call repeats the bits."""
    import torch
    from crane_amd import _lib, ops
    M, N, K, splits = split_draw(SEED, i)
    print(f"random linear split {i} (seed {SEED}): M={M} N={N} K={K} splits={splits}", flush=True)
    assert _lib.lib().crane_gemm_split_supported(M, N, K, splits, _lib.BF16) == 1
    x, w, _ = _case(SEED + 9800 + i, M, N, K, "bf16", False)
    xd, wd = _t(x, "bf16", gpu), _t(w, "bf16", gpu)
    outs = []
    for _ in range(2):
        parts = torch.empty((splits, M, N), dtype=torch.float32, device=gpu)
        assert _lib.lib().crane_gemm_linear_split(ops._gemm(gpu)._h, xd.data_ptr(), wd.data_ptr(), parts.data_ptr(),
                                                  M, N, K, splits, _lib.BF16, ops._stream(gpu)) == 0
        outs.append(parts.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    acc = np.zeros((M, N), np.float32)
    for p in outs[0]:
        acc = (acc + p).astype(np.float32)
    assert_linear_close(cases.bf16(acc), x, w, None, "bf16", orc, f"random split linear {M}x{N}x{K}/{splits}")


def silu_mul_draw(seed: int, i: int):
    """Draw i of the randomised one-launch gate_up + SiLU*mul sweep: (M, inter,
    K) that crane_gemm_silu_mul_supported takes -- inter a multiple of 48
    with K of 512, or of 32 with K of 1024 -- with M * 2 inter * K <= 1.5e9."""
    r = cases.rng(seed + 9500 + i)
    M = int(r.integers(1, 33))
    if i % 2 == 0:
        inter, K = 48 * int(r.integers(86, 300)), 512 * int(r.integers(1, 9))
    else:
        inter, K = 32 * int(r.integers(129, 400)), 1024 * int(r.integers(1, 5))
    while M * 2 * inter * K > 1.5e9 and K > 1024:
        K -= 1024
    return M, inter, K


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(N_RANDOM // 2))
def test_random_linear_silu_mul(gpu, orc, i):
    """Random shapes of the one-launch gated product against the oracle chain,
    the bar of test_linear_silu_mul_parity."""
    from crane_amd import _lib, ops
    M, inter, K = silu_mul_draw(SEED, i)
    print(f"random linear_silu_mul {i} (seed {SEED}): M={M} inter={inter} K={K}", flush=True)
    assert _lib.lib().crane_gemm_silu_mul_supported(M, inter, K, 1) == 1
    x, w, _ = _case(SEED + 9600 + i, M, 2 * inter, K, "bf16", False)
    ref, bound = _silu_mul_bound(x, w, orc)
    got = ops.linear_silu_mul(_t(x, "bf16", gpu), _t(w, "bf16", gpu)).float().cpu().numpy()
    d = np.abs(got.astype(np.float64) - ref)
    assert np.all(d <= bound), f"random gated {M}x{inter}x{K}: beyond the bound"
    assert float(np.mean(got == ref)) >= 0.98


@pytest.mark.gpu
def test_qkv_proj_feeds_the_append(gpu, orc):
    """Hidden states -> qkv_proj (bias) -> fused QK-norm/RoPE append, against
    the oracle's Linear followed by its append."""
    import torch
    from crane_amd import ops
    B, S, H, Hq, Hkv, D = 2, 33, 512, 8, 2, 128
    W = (Hq + 2 * Hkv) * D
    x, w, b = _case(600, B * S, W, H, "bf16")
    qkv = ops.linear(_t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu)).reshape(B, S, W)
    assert_linear_close(qkv.float().cpu().numpy().reshape(B * S, W), x, w, b, "bf16", orc, "qkv_proj")
    cos, sin = orc.rope_tables(D, 1e6, 64)
    cos, sin = orc.round_bf16(cos), orc.round_bf16(sin)
    kc = torch.zeros((B, Hkv, 64, D), dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros_like(kc)
    zero = torch.zeros(B, dtype=torch.int32, device=gpu)
    q = ops.qk_norm_rope_append(qkv, _t(cos, "bf16", gpu), _t(sin, "bf16", gpu), zero, kc, vc, zero, S, Hq, Hkv,
                                order="rope_only")
    kref = np.zeros((B, Hkv, 64, D), np.float32)
    vref = np.zeros_like(kref)
    # the append is applied to the GPU's own qkv rows: this checks the hand-off
    # (layout and row stride), the append's parity is tested on its own
    qkv_np = qkv.float().cpu().numpy()
    q_ref = orc.qk_norm_rope_append(qkv_np, Hq, Hkv, cos, sin, np.zeros(B, np.int32), kref, vref,
                                    np.zeros(B, np.int32), order=orc.ROPE_ONLY, dtype="bf16")
    assert_ulp_close(q.float().cpu().numpy(), q_ref, "bf16", "q after the append", min_exact=0.999)
    assert_ulp_close(kc.float().cpu().numpy(), kref, "bf16", "k cache after the append", min_exact=0.999)
    np.testing.assert_array_equal(vc.float().cpu().numpy(), vref)


@pytest.mark.gpu
def test_linear_on_two_streams_and_threads(gpu, orc):
    """Each stream gets its own context (its own workspace), so projections on
    two streams may overlap; host threads calling into one context at once,
    while new shapes are being planned, are serialised.  Every result is
    bit-identical to the same product on the default stream."""
    import threading
    import torch
    from crane_amd import ops
    shapes = [(64 + 7 * i, 256 + 32 * i, 512) for i in range(6)]
    xs, ws, refs = [], [], []
    for i, (M, N, K) in enumerate(shapes):
        x, w, _ = _case(700 + i, M, N, K, "bf16", False)
        xs.append(_t(x, "bf16", gpu))
        ws.append(_t(w, "bf16", gpu))
    torch.cuda.synchronize()
    refs = [ops.linear(x, w) for x, w in zip(xs, ws)]
    torch.cuda.synchronize()
    print("linear: two streams", flush=True)
    s1, s2 = torch.cuda.Stream(device=gpu), torch.cuda.Stream(device=gpu)
    outs = {}
    for s in (s1, s2):
        s.wait_stream(torch.cuda.current_stream(gpu))
    with torch.cuda.stream(s1):
        outs[1] = [ops.linear(x, w) for x, w in zip(xs, ws)]
    with torch.cuda.stream(s2):
        outs[2] = [ops.linear(x, w) for x, w in reversed(list(zip(xs, ws)))][::-1]
    torch.cuda.synchronize()
    assert ops._gemm(gpu) is not None and len({k for k in ops._GEMMS if k[0] == gpu}) >= 3
    for k in (1, 2):
        for got, ref in zip(outs[k], refs):
            assert torch.equal(got, ref), "a side stream's product differs"
    for st in (s1, s2):  # retire the side streams' contexts
        ops.release_stream(gpu, st)
        assert (gpu, st.cuda_stream) not in ops._GEMMS
    assert torch.equal(ops.linear(xs[0], ws[0]), refs[0])  # the default stream's context is untouched
    print("linear: four host threads on one stream", flush=True)
    results, errors = {}, []

    def worker(j):
        try:
            new = [(40 + 3 * j + i, 192 + 64 * j, 256) for i in range(3)]  # shapes no one planned yet
            got = []
            for (M, N, K) in new:
                x, w, _ = _case(800 + 10 * j + M, M, N, K, "bf16", False)
                xt, wt = _t(x, "bf16", gpu), _t(w, "bf16", gpu)
                got.append((ops.linear(xt, wt), xt, wt))
            results[j] = got
        except Exception as e:  # reported below, in the test's thread
            errors.append(repr(e))

    threads = [threading.Thread(target=worker, args=(j,)) for j in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for j, got in results.items():
        for y, xt, wt in got:
            assert torch.equal(y, ops.linear(xt, wt)), f"thread {j}: product differs on a second call"
