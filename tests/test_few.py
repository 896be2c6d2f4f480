"""The projections of a decode step of one sequence
(include/crane_few.h): the add + norm, the product and SiLU * up in one launch
against the launches they stand for, and a model step that takes them against
the same step without."""
import numpy as np
import pytest

import cases
from test_gemm import _case, _silu_mul_bound, _t, assert_linear_close
from tolerance import bf16_ulp


def test_few_shape_query():
    """Which shapes the one-row calls take (host logic, no GPU)."""
    from crane_amd import _lib
    q = _lib.lib().crane_few_supported
    BF16, F32 = 1, 0
    assert q(1, 4096, 1024, 1, 0, BF16) == 1      # Qwen3-0.6B qkv_proj
    assert q(1, 24576, 4096, 1, 1, BF16) == 1     # Qwen3-8B gate_up
    assert q(1, 4096, 12288, 0, 0, BF16) == 1     # ... and down_proj
    assert q(1, 4096, 4608, 1, 0, BF16) == 0      # the norm's registers
    assert q(2, 4096, 1024, 0, 0, BF16) == 0
    assert q(0, 4096, 1024, 0, 0, BF16) == 0
    assert q(1, 4096, 1000, 0, 0, BF16) == 0      # K not a multiple of 512
    assert q(1, 4096, 33280, 0, 0, BF16) == 0
    assert q(1, 4097, 1024, 1, 1, BF16) == 0      # gated: N = 2 inter
    assert q(1, 4096, 1024, 1, 0, F32) == 0
    L = _lib.lib()
    assert L.crane_few_linear(16, 16, None, 16, 2, 64, 512, BF16, None) == _lib.E_INVALID
    assert L.crane_few_linear(16, 24, None, 16, 1, 64, 512, BF16, None) == _lib.E_ALIGN
    assert L.crane_few_linear(16, 16, None, 16, 0, 64, 512, BF16, None) == _lib.OK
    assert L.crane_few_norm_linear(16, 32, 16, None, 1e-6, 16, None, 48, 1, 64, 512, 0, BF16, None) == _lib.E_INVALID
    assert L.crane_few_norm_linear(16, 32, 16, 32, 1e-6, 16, None, 48, 1, 64, 512, 0, BF16, None) == _lib.E_INVALID
    assert L.crane_few_norm_linear(16, 32, 16, 64, 1e-6, 16, 48, 48, 1, 64, 512, 1, BF16, None) == _lib.E_INVALID


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,bias", [
    (1, 1, 512, True),        # one output: three waves have none
    (1, 2049, 1024, False),   # two turns, the second of few waves
    (1, 1000, 1536, True),
    (1, 6150, 3584, True),    # four turns of 7 slices
    (1, 515, 4096, False),    # the widest in registers
    (1, 260, 4608, True),     # the long kernel: 9 slices, a ring of 8
    (1, 2100, 18944, False),  # ... 37 slices over two turns
    (1, 70, 32768, True),     # the longest K: its row fills 64 KiB of LDS
])
def test_few_linear(gpu, orc, M, N, K, bias):
    from crane_amd import ops
    print(f"few_linear M={M} N={N} K={K}", flush=True)
    x, w, b = _case(3100 + N + K, M, N, K, "bf16", bias)
    args = _t(x, "bf16", gpu), _t(w, "bf16", gpu), _t(b, "bf16", gpu) if bias else None
    got = ops.few_linear(*args)
    assert_linear_close(got.float().cpu().numpy(), x, w, b, "bf16", orc, f"few linear {M}x{N}x{K}")
    assert bool((got == ops.few_linear(*args)).all())


@pytest.mark.gpu
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 2, 512), (1, 4100, 1024), (1, 3000, 2048), (1, 516, 3584), (1, 4104, 4096)])
def test_norm_linear(gpu, orc, M, N, K, add, gated):
    """The residual bits of add_rms_norm, and the product of the normed row at the
    bars of the product alone.  The kernel sums the squares in its own order, so
    the row's rms may round to a neighbour of the exact one's bf16 value: the row is
    rebuilt for it and both neighbours, and y has to be the product of one of the
    three rows."""
    import torch
    from crane_amd import ops
    print(f"norm_linear M={M} N={N} K={K} add={add} gated={gated}", flush=True)
    r = cases.rng(3300 + N + K)
    x, h = (_t(cases.cast(cases.normal(r, (M, K)), "bf16"), "bf16", gpu) for _ in range(2))
    nw = _t(cases.cast(1 + 0.1 * cases.normal(r, (K,)), "bf16"), "bf16", gpu)
    _, w, b = _case(3400 + N + K, M, N, K, "bf16", True)
    wd, bd = _t(w, "bf16", gpu), None if gated else _t(b, "bf16", gpu)
    want_res = x.clone()
    if add:
        ops.add_rms_norm(want_res, h, nw, 1e-6)
    x0 = x.clone()
    y, res = ops.norm_linear(x, h if add else None, nw, 1e-6, wd, bd, gated)
    assert torch.equal(x, x0) and torch.equal(res, want_res)
    v, weight = res.float().cpu().numpy(), nw.float().cpu().numpy()
    got = y.float().cpu().numpy()
    m = cases.bf16(np.sqrt(np.mean(v.astype(np.float64) ** 2) + 1e-6))[0]
    ulp = bf16_ulp(m)
    fits = []
    for rms in (m, cases.bf16(m - ulp)[0], cases.bf16(m + ulp)[0]):
        n = cases.bf16(cases.bf16(v / np.float32(rms)) * weight)
        try:
            if gated:
                ref, bound = _silu_mul_bound(n, w, orc)
                assert np.all(np.abs(got.astype(np.float64) - ref) <= bound)
                assert N < 100 or float(np.mean(got == ref)) >= 0.98
            else:
                assert_linear_close(got, n, w, b, "bf16", orc, f"norm_linear {N}x{K}")
            fits.append(float(rms))
        except AssertionError as e:
            print(f"  rms {float(rms)}: {str(e)[:80]}", flush=True)
    assert fits, (N, K, add, gated)


@pytest.mark.gpu
@pytest.mark.parametrize("std", [2.0 ** -70, 2.0 ** 70, float("inf"), float("nan")])
def test_norm_linear_outside_the_fast_divide(gpu, std):
    """Rows whose rms leaves the range of the fast division, or is not finite: with
    every |x| the same power of two the rms is exact, and the row is bit for bit that
    of rms_norm and few_linear."""
    import torch
    from crane_amd import ops
    K, N = 1024, 130
    r = cases.rng(77)
    x = _t(np.sign(cases.normal(r, (1, K))).astype(np.float32), "bf16", gpu)
    if np.isfinite(std):
        x = x * std
    else:
        x[0, 5] = std
    nw = _t(cases.cast(1 + 0.1 * cases.normal(r, (K,)), "bf16"), "bf16", gpu)
    w = _t(cases.cast(cases.normal(r, (N, K), K ** -0.5), "bf16"), "bf16", gpu)
    y, res = ops.norm_linear(x, None, nw, 0.0, w)
    want = ops.few_linear(ops.rms_norm(x, nw, 0.0), w)
    assert res is x
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(y.nan_to_num(), want.nan_to_num())
    assert bool(torch.isnan(y).all()) == (not np.isfinite(std))


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,n,max_kv,N", [
    (4, 1, 257, 257, 1),          # two chunks, the second of one key; one output
    (16, 8, 1000, 1064, 1024),    # 4 chunks in 5 slots
    (16, 16, 2048, 2048, 1021),   # 8 full chunks; the last workgroup's waves partly without outputs
    (12, 4, 1793, 2048, 1000),    # the last chunk of one key; fewer pieces than threads
    (4, 4, 200, 2000, 61),        # one chunk: the row is the chunk kernel's
    (8, 2, 0, 300, 96),           # an empty sequence
])
def test_attention_decode_linear(gpu, Hq, Hkv, n, max_kv, N):
    """One sequence's decode attention with the merge inside o_proj against
    the merge kernel and few_linear, over a workspace of NaN.  The merge's f32
    sums associate differently, so a few of the row's elements may round to the
    neighbouring bf16 value (2^-16 of them per f32 ulp; eight are allowed), and
    y, rounded once, by one ulp more."""
    import torch
    from crane_amd import ops
    print(f"attention_decode_linear Hq={Hq} Hkv={Hkv} n={n} max_kv={max_kv} N={N}", flush=True)
    assert ops._lib.lib().crane_few_attn_linear_supported(max_kv, Hq, N, ops._lib.BF16)
    gen = torch.Generator(device=gpu).manual_seed(41 + n)
    rnd = lambda *s: torch.randn(s, generator=gen, device=gpu).to(torch.bfloat16)
    q, k, v = rnd(1, Hq, 128), rnd(1, Hkv, max_kv + 8, 128), rnd(1, Hkv, max_kv + 8, 128)
    w = rnd(N, Hq * 128)
    length = torch.tensor([n], dtype=torch.int32, device=gpu)
    row = ops.attention_decode(q, k, v, length, max_kv).view(1, -1)
    want = ops.few_linear(row, w).float()
    ws = torch.full((ops.decode_workspace_bytes(1, Hq, Hkv, max_kv) // 4 + 1,), float("nan"), device=gpu)
    got = ops.attention_decode_linear(q, k, v, length, max_kv, w, workspace=ws).float()
    # the merged row itself, read by weight rows of one 1: every element within
    # one bf16 ulp of the merge kernel's, and at most eight of them off
    pick = torch.arange(N, device=gpu) * (Hq * 128 // N if N < Hq * 128 else 1) % (Hq * 128)
    one = torch.zeros((N, Hq * 128), dtype=torch.bfloat16, device=gpu)
    one[torch.arange(N, device=gpu), pick] = 1
    merged = ops.attention_decode_linear(q, k, v, length, max_kv, one, workspace=ws).float()[0]
    exact = row.float()[0][pick]
    assert bool(((merged - exact).abs() <= 2.0 ** -7 * exact.abs()).all())
    assert int((merged != exact).sum()) <= 8
    bound = 2.0 ** -7 * want.abs() + 8 * 2.0 ** -7 * (row.float().abs() * w.float().abs()).amax(1)
    assert bool(((got - want).abs() <= bound).all())


def test_attention_decode_linear_query():
    """The sizes the merging o_proj takes, and what it refuses (host logic)."""
    from crane_amd import _lib
    L = _lib.lib()
    q = L.crane_few_attn_linear_supported
    assert q(257, 16, 1024, 1) and q(2048, 4, 1, 1)
    assert not q(256, 16, 1024, 1) and not q(2049, 16, 1024, 1) and not q(1000, 16, 1025, 1) and not q(1000, 20, 1024, 1)
    assert not q(1000, 6, 1024, 1) and not q(1000, 16, 1024, 0) and not q(1000, 16, 0, 1)
    call = lambda cap=1000, max_kv=1000, Hq=16, Hkv=8, D=128, ws=1 << 30, w=16, N=64, dt=1: L.crane_few_attn_linear(
        16, 16, 16, cap, 16, max_kv, Hq, Hkv, D, 0.1, 0, 16, ws, 16, w, 16, N, dt, None)
    assert call(cap=999) == _lib.E_CAPACITY and call(Hkv=3) == _lib.E_GQA and call(D=64) == _lib.E_HEAD_DIM
    assert call(ws=64) == _lib.E_WORKSPACE and call(w=24) == _lib.E_ALIGN and call(dt=0) == _lib.E_INVALID
    assert call(max_kv=200) == _lib.E_INVALID


def _twins(gpu, family, batch, capacity):
    """Three models of one small stack over one set of weights, the second without
    the few-row projections."""
    import torch
    from crane_amd.decoder import LayerWeights
    from crane_amd.model import DecoderModel, ModelConfig
    hidden, Hq, Hkv, inter, L, D = 1024, 8, 2, 1536, 2, 128
    gen = torch.Generator(device=gpu).manual_seed(5)
    rnd = lambda *s, std=1.0: (torch.randn(s, generator=gen, device=gpu) * std).to(torch.bfloat16)
    cla = 2 if family == "hunyuan" else 1
    layers = []
    for i in range(L):
        rows = Hq * D if cla > 1 and i % cla else (Hq + 2 * Hkv) * D
        norms = family != "qwen2"
        layers.append(LayerWeights(1 + rnd(hidden, std=0.1), rnd(rows, hidden, std=hidden ** -0.5),
                                   rnd(hidden, Hq * D, std=(Hq * D) ** -0.5), 1 + rnd(hidden, std=0.1),
                                   rnd(2 * inter, hidden, std=hidden ** -0.5), rnd(hidden, inter, std=inter ** -0.5),
                                   rnd(rows, std=0.1) if family == "qwen2" else None,
                                   1 + rnd(D, std=0.1) if norms else None, 1 + rnd(D, std=0.1) if norms else None))
    cfg = ModelConfig(hidden, Hq, Hkv, inter, L, family, max_position=capacity, cla_share_factor=cla)
    head = rnd(512, hidden, std=hidden ** -0.5)
    models = [DecoderModel(cfg, layers, 1 + rnd(hidden, std=0.1) * 0, head, batch, capacity) for _ in range(3)]
    assert all(m.few for m in models)
    models[1].few = False
    return models, rnd, hidden, L


@pytest.mark.gpu
@pytest.mark.parametrize("family,batch", [("qwen3", 1), ("qwen2", 1), ("hunyuan", 1)])
def test_model_step_takes_them(gpu, family, batch):
    """Two decode steps of a stack that takes the few-row projections against
    the same steps of a twin without them: same cache rows written up to the
    projections' rounding, logits within two bf16 roundings per layer."""
    import torch
    from crane_amd.model import DecodeGraph
    models, rnd, hidden, L = _twins(gpu, family, batch, 600)
    graph = DecodeGraph(models[2])
    for step in range(2):
        x = rnd(batch, 1, hidden)
        pos = torch.full((batch,), step, dtype=torch.int32, device=gpu)
        a, b = (m.step_batch_decode(x, pos) for m in models[:2])
        graph.x.copy_(x)
        graph.positions.copy_(pos)
        assert torch.equal(graph.replay(), a), "replay differs from the eager step"
        rel = float((a.float() - b.float()).norm() / b.float().norm())
        print(f"  {family} step {step}: rel {rel:.2e}", flush=True)
        assert rel <= 2 * L * 2.0 ** -8
    trace = []
    models[0].forward(x, pos, trace)
    assert len(trace) == L and trace[0][0].shape == trace[0][1].shape == (batch, hidden)


@pytest.mark.gpu
@pytest.mark.parametrize("capacity", [600, 2100])
@pytest.mark.parametrize("length", [255, 511])
def test_model_steps_grow_past_a_chunk(gpu, length, capacity):
    """Steps of one sequence whose cache grows from one 256-key chunk to two and from
    two to three under replays of one captured graph: o_proj merges the chunks'
    partials (capacity 600) or takes the merge kernel's row (past 2048)."""
    import torch
    from crane_amd import ops
    from crane_amd.model import DecodeGraph
    models, rnd, hidden, L = _twins(gpu, "qwen3", 1, capacity)
    merges = ops._lib.lib().crane_few_attn_linear_supported(capacity, 8, hidden, ops._lib.BF16)
    assert bool(merges) == (capacity <= 2048)
    caches = [rnd(1, 2, length, 128) for _ in range(2 * L)]
    for m in models:
        for i in range(L):
            m.k[i][:, :, :length], m.v[i][:, :, :length] = caches[2 * i], caches[2 * i + 1]
        m.lengths.fill_(length)
        m.host_lengths[:] = length
    graph = DecodeGraph(models[2])
    for step in range(3):
        x = rnd(1, 1, hidden)
        pos = torch.full((1,), length + step, dtype=torch.int32, device=gpu)
        a, b = (m.step_batch_decode(x, pos) for m in models[:2])
        graph.x.copy_(x)
        graph.positions.copy_(pos)
        assert torch.equal(graph.replay(), a), "replay differs from the eager step"
        rel = float((a.float() - b.float()).norm() / b.float().norm())
        print(f"  capacity {capacity}, {length + step + 1} keys: rel {rel:.2e}", flush=True)
        assert rel <= 2 * L * 2.0 ** -8
    for i in range(L):
        assert torch.equal(models[0].k[i], models[2].k[i]) and torch.equal(models[0].v[i], models[2].v[i])
