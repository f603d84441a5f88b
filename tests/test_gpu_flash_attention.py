"""GPU parity of the gfx950 flash-attention entry (kg_gfx950_flash_attention_entry).

Cases follow the reference's runtime test (test/cuda/test_cuda_sm89_kernel_demos_runtime.py:
571-597: default_rng(2026052901) inputs of shape (1,2,4,3), tiles 2/2), the flash-attention
demos' random shapes (kernel/flash_attention/*.py: S in {257,321,389}, D in {48,64,80}) and
BASELINE configs C4 (bf16 B=4,H=32,S=2048,D=128, non-causal) and C5 (bf16 B=1,H=32,
S=16384, D=128 and 64, causal), all against the oracle's restatement of the demo loop nest
(plus the scale/causal extension), at full size through sampled heads and query blocks.
"""

from __future__ import annotations

import random
from pathlib import Path

import numpy as np
import pytest

from kernelcode_generate_amd import native
from tests.golden.make_golden import attention_closed_form
from tests.gpu_util import (assert_f32_close, assert_h16_close, assert_within, attention_f32_tolerance, round_to,
                            to_numpy)

pytestmark = pytest.mark.gpu
GOLDEN = Path(__file__).resolve().parent / "golden"


def run(device, dtype, q, k, v, br=64, bc=64, scale=None, causal=False):
    import torch

    qt, kt, vt = (torch.as_tensor(a).to(device) for a in (q, k, v))
    out = torch.full(tuple(qt.shape), float("nan"), dtype=dtype, device=device)
    print(f"[fa] shape={tuple(qt.shape)} {dtype} scale={scale} causal={causal}", flush=True)
    if scale is None and not causal:
        native.call_entry("kg_gfx950_flash_attention_entry", (out, qt, kt, vt, br, bc))
    else:
        native.flash_attention(out, qt, kt, vt, br, bc, 1.0 if scale is None else scale, causal)
    return out


def test_runtime_vector(device):
    import torch

    v = dict(np.load(GOLDEN / "cuda_runtime_vectors.npz"))
    out = run(device, torch.float32, v["fa_q"], v["fa_k"], v["fa_v"], 2, 2)
    # the reference's own bar for this vector (test/cuda/test_cuda_sm89_kernel_demos_runtime.py:595)
    assert_f32_close(to_numpy(out), v["fa_expected"], rtol=1e-4, atol=1e-4, what="runtime vector")
    # the 4-slot form (static demo) gives the same result
    import torch as _t

    qt, kt, vt = (_t.as_tensor(a).to(device) for a in (v["fa_q"], v["fa_k"], v["fa_v"]))
    o4 = _t.empty_like(qt)
    native.call_entry("kg_gfx950_flash_attention_entry", (o4, qt, kt, vt))
    assert_f32_close(to_numpy(o4), v["fa_expected"], rtol=1e-4, atol=1e-4, what="4-slot form")


@pytest.mark.parametrize("seed", [2026052721, 5, 6])
def test_demo_random_profiles_f32(device, oracle_mod, seed):
    """Shapes drawn like kernel/flash_attention/inputs_static_tile_static.py:213-226."""

    import torch

    r = random.Random(seed)
    b, h = r.choice((1, 2)), r.choice((4, 8))
    s, d = r.choice((257, 321, 389)), r.choice((48, 64, 80))
    br, bc = random.Random(seed + 1).choice(((48, 64), (64, 80), (80, 96)))
    rng = np.random.default_rng(seed)
    q, k, v = (rng.standard_normal((b, h, s, d), dtype=np.float32) for _ in range(3))
    ref = oracle_mod.flash_attention_demo(q, k, v, br, bc)
    tol = attention_f32_tolerance(q, k, v)
    assert_within(to_numpy(run(device, torch.float32, q, k, v, br, bc)), ref, tol, what=str(seed))


@pytest.mark.parametrize("scale,causal", [(0.125, False), (0.3, True), (None, True)])
def test_extensions_f32(device, oracle_mod, scale, causal):
    import torch

    rng = np.random.default_rng(17)
    q, k, v = (rng.standard_normal((1, 3, 200, 40), dtype=np.float32) for _ in range(3))
    ref = oracle_mod.flash_attention_demo(q, k, v, 48, 80, scale=scale, causal=causal)
    out = run(device, torch.float32, q, k, v, 48, 80, scale, causal)
    assert_within(to_numpy(out), ref, attention_f32_tolerance(q, k, v, scale, causal), what=f"scale={scale} causal={causal}")


@pytest.mark.parametrize(
    "shape,s_kv,causal",
    [
        ((1, 2, 256, 128), 256, False),
        ((1, 2, 700, 128), 700, True),  # ragged causal over several 128-query blocks
        ((2, 1, 130, 64), 300, False),  # one partial query block, ragged key tail, S_q != S_kv
        ((1, 1, 1000, 64), 1000, True),
        ((1, 2, 1, 128), 1, False),  # one query, one key
        ((1, 1, 33, 64), 1000, False),
        ((1, 40, 256, 128), 256, False),  # more than 512 blocks of 16 queries from here on
        ((2, 20, 230, 128), 230, True),  # partial query block and key tail, causal
        ((8, 16, 65, 64), 300, False),
        ((1, 33, 250, 64), 250, True),
    ],
)
def test_f32_matrix_cores(device, oracle_mod, shape, s_kv, causal):
    """fp32 Q/K/V with D in {64, 128} take an fp32 MFMA kernel: the tiled one (32x32x2 MFMAs of 64
    cycles), or up to 512 blocks of 16 queries the split-key one (16x16x4, 32 cycles), as the
    cost record tells. The oracle's demo loop nest is the reference where S_q == S_kv, the float64
    closed form of the demo's check (kernel/flash_attention/inputs_static_tile_static.py:57-87)
    otherwise."""

    import torch

    b, h, sq, d = shape
    scale = 1.0 / np.sqrt(d)
    specs = [native.TensorSpec(x, "float32") for x in (shape, shape, (b, h, s_kv, d), (b, h, s_kv, d))]
    model = native.cost("flash_attention", [*specs, 64, 64, scale, int(causal)])
    cycles = 32 if sq <= 16 or b * h * -(-sq // 16) <= 512 else 64
    assert model["MFMA"] > 0 and model["MFMA_CYCLES"] == cycles * model["MFMA"]
    rng = np.random.default_rng(sq * 3 + s_kv + d)
    q = rng.standard_normal(shape, dtype=np.float32)
    k, v = (rng.standard_normal((b, h, s_kv, d), dtype=np.float32) for _ in range(2))
    if sq == s_kv:
        ref = oracle_mod.flash_attention_demo(q, k, v, 64, 64, scale=scale, causal=causal)
    else:
        ref = attention_closed_form(q, k, v, scale).astype(np.float32)
    out = run(device, torch.float32, q, k, v, 64, 64, scale, causal)
    assert_within(to_numpy(out), ref, attention_f32_tolerance(q, k, v, scale, causal),
                  what=f"{shape} s_kv={s_kv} causal={causal}")


def test_f32_c4_shape_sampled_heads(device):
    """BASELINE C4's shape (B=4, H=32, S=2048, D=128) in fp32: two heads against the float64
    closed form of the demo's check."""

    import torch

    shape = (4, 32, 2048, 128)
    gen = torch.Generator(device=device).manual_seed(4)
    q, k, v = (torch.randn(shape, generator=gen, device=device) for _ in range(3))
    out = torch.full(shape, float("nan"), device=device)
    print("[fa] f32 C4 shape", flush=True)
    native.flash_attention(out, q, k, v, 64, 64, 1.0 / np.sqrt(128), False)
    for bi, hi in ((0, 0), (3, 31)):
        qh, kh, vh = (to_numpy(t[bi, hi]) for t in (q, k, v))
        ref = attention_closed_form(qh, kh, vh, 1.0 / np.sqrt(128))
        assert_within(to_numpy(out[bi, hi]), ref, attention_f32_tolerance(qh, kh, vh, 1.0 / np.sqrt(128)),
                      what=f"head {bi},{hi}")


@pytest.mark.parametrize("dtype_name", ["bfloat16", "float16"])
@pytest.mark.parametrize(
    "shape,causal",
    [
        ((1, 2, 256, 128), False),
        ((1, 2, 512, 128), True),
        ((2, 1, 384, 64), False),
        ((1, 2, 512, 64), True),
        ((1, 1, 300, 128), False),  # ragged S
        ((1, 1, 200, 64), True),  # ragged S, causal
        ((1, 2, 257, 48), False),  # demo-like D
        ((1, 2, 700, 128), True),  # ragged causal over several 256-query blocks
        ((2, 3, 130, 128), False),  # one partial query block, ragged key tail
        ((1, 1, 64, 128), True),  # a single key tile
        ((1, 2, 1, 128), False),  # one query, one key
        ((1, 1, 1000, 64), True),  # D=64 ragged causal over several 128-query blocks
    ],
)
def test_16bit(device, oracle_mod, dtype_name, shape, causal):
    import torch

    dt = getattr(torch, dtype_name)
    rng = np.random.default_rng(shape[2] + shape[3])
    (qt, q), (kt, k), (vt, v) = (round_to(rng.standard_normal(shape, dtype=np.float32), dt) for _ in range(3))
    scale = 1.0 / np.sqrt(shape[3])
    ref = oracle_mod.flash_attention_demo(q, k, v, 64, 64, scale=scale, causal=causal)
    out = run(device, dt, qt, kt, vt, 64, 64, scale, causal)
    assert_h16_close(to_numpy(out), ref, what=f"{dtype_name} {shape} causal={causal}")


@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16"])
@pytest.mark.parametrize("shape,causal,scale", [((1, 2, 300, 64), True, 2.0), ((1, 1, 256, 128), False, 0.9),
                                                ((2, 1, 130, 128), True, 0.05)])
def test_16bit_scales(device, oracle_mod, dtype_name, shape, causal, scale):
    """Scales away from 1/sqrt(D) (the kernel scales each fp32 score before its exp2; Q is used
    as stored: multiplying it by the scale in its own 16-bit format would add a rounding of the
    size of the format's unit roundoff to every score, twice the error of the exact scale for
    bf16 on this test's inputs)."""
    import torch

    dt = getattr(torch, dtype_name)
    rng = np.random.default_rng(shape[2] * 7 + shape[3])
    (qt, q), (kt, k), (vt, v) = (round_to(rng.standard_normal(shape, dtype=np.float32), dt) for _ in range(3))
    ref = oracle_mod.flash_attention_demo(q, k, v, 64, 64, scale=scale, causal=causal)
    out = run(device, dt, qt, kt, vt, 64, 64, scale, causal)
    assert_h16_close(to_numpy(out), ref, what=f"{dtype_name} {shape} causal={causal} scale={scale}")


def _sampled_check(oracle_mod, got, q, k, v, heads, blocks, scale, causal, name):
    for (b, h) in heads:
        for m0, m1 in blocks:
            ref = oracle_mod.flash_attention_demo(
                q[b : b + 1, h : h + 1], k[b : b + 1, h : h + 1], v[b : b + 1, h : h + 1], 64, 64,
                scale=scale, causal=causal, threads=1, m_range=(m0, m1),
            )
            assert_h16_close(got[b, h, m0:m1], ref[0, 0, m0:m1], what=f"{name} b={b} h={h} rows {m0}:{m1}")


def test_c4_full_size(device, oracle_mod):
    import torch

    shape = (4, 32, 2048, 128)
    rng = np.random.default_rng(20261205)
    (qt, q), (kt, k), (vt, v) = (round_to(rng.standard_normal(shape, dtype=np.float32), torch.bfloat16) for _ in range(3))
    scale = 1.0 / np.sqrt(128.0)
    got = to_numpy(run(device, torch.bfloat16, qt, kt, vt, 128, 64, scale, False))
    assert np.isfinite(got).all()
    _sampled_check(oracle_mod, got, q, k, v, [(0, 0), (3, 31)], [(0, 64), (1984, 2048)], scale, False, "C4")
    # every output row is a convex combination of V rows: it lies inside V's per-column range
    vmin = v.min(axis=2, keepdims=True)
    vmax = v.max(axis=2, keepdims=True)
    slack = 1e-2 * (vmax - vmin)
    assert ((got >= vmin - slack) & (got <= vmax + slack)).all()


@pytest.mark.parametrize(
    "shape,causal",
    [((2, 64, 1000, 128), False), ((1, 128, 700, 128), True), ((1, 8, 2048, 128), False)],
    ids=["8wave_ragged", "8wave_ragged_causal", "4wave_small_grid"],
)
def test_workgroup_shapes_d128(device, oracle_mod, shape, causal):
    """D=128 takes 8-wave workgroups (256 queries) when they give every CU one and 4-wave
    workgroups (128 queries) otherwise: the first two shapes are 512 and 384 ragged 8-wave
    workgroups, the third 128 4-wave ones. Sampled heads and row blocks against the oracle."""

    import torch

    b, h, s, d = shape
    rng = np.random.default_rng(s + h)
    (qt, q), (kt, k), (vt, v) = (round_to(rng.standard_normal(shape, dtype=np.float32), torch.bfloat16) for _ in range(3))
    scale = 1.0 / np.sqrt(128.0)
    got = to_numpy(run(device, torch.bfloat16, qt, kt, vt, 128, 64, scale, causal))
    assert np.isfinite(got).all()
    heads = [(0, 0), (b - 1, h - 1)]
    blocks = [(0, 64), (s - 64 - s % 7, s - s % 7), (s - 40, s)]
    _sampled_check(oracle_mod, got, q, k, v, heads, blocks, scale, causal, f"{shape}")


@pytest.mark.parametrize("d,seed", [(128, 20261206), (64, 20261207)])
def test_c5_full_size_causal(device, oracle_mod, d, seed):
    import torch

    shape = (1, 32, 16384, d)
    rng = np.random.default_rng(seed)
    (qt, q), (kt, k), (vt, v) = (round_to(rng.standard_normal(shape, dtype=np.float32), torch.bfloat16) for _ in range(3))
    scale = 1.0 / np.sqrt(float(d))
    got = to_numpy(run(device, torch.bfloat16, qt, kt, vt, 128, 64, scale, True))
    assert np.isfinite(got).all()
    _sampled_check(oracle_mod, got, q, k, v, [(0, 0), (0, 21)], [(0, 64), (8192, 8256), (16320, 16384)], scale, True,
                   f"C5 D={d}")
    # causal row 0 attends only to key 0: out[:, :, 0] == V[:, :, 0] (bf16-rounded)
    np.testing.assert_allclose(got[0, :, 0, :], v[0, :, 0, :], rtol=1e-2, atol=1e-2)


PERSISTENT = [
    ((1, 65, 2048, 128), 2048, "bfloat16"),  # 520 items on 256 workgroups: 8 of them take a third
    ((2, 64, 2048, 128), 2048, "float16"),   # 1024 items, 4 per workgroup
    ((1, 64, 2048, 128), 256, "bfloat16"),   # 4 key tiles per item, the fewest: Q staged in tiles 0-1
    ((1, 64, 2048, 128), 384, "float16"),    # 6 key tiles per item
    ((1, 64, 2048, 128), 128, "bfloat16"),   # 2 key tiles: too few, one workgroup per item
    ((1, 130, 1024, 64), 1024, "bfloat16"),  # D=64: 1040 items on 512 four-wave workgroups
]


@pytest.mark.parametrize("shape,s_kv,dtype", PERSISTENT)
def test_persistent_form_matches_one_item_per_workgroup(device, oracle_mod, shape, s_kv, dtype):
    """Non-causal whole-tile attention with an even key-tile count of at least 4 and at least
    two items (query blocks) per workgroup slot runs persistent workgroups: each walks the
    items gridDim.x apart as one sequence of key tiles (the next item's Q staged in LDS during
    tiles nt-4 and nt-3, its K tiles 0-1 and V tile 0 copied and its first S tile computed in
    this item's last two tiles). A three-deep ring (memory_stage=3) launches one workgroup per
    item instead.
    Both do the same arithmetic per item, so the bits must agree; sampled rows of two heads
    also against the oracle (S_kv = S_q: the demo's loop nest) or the float64 formula."""

    import torch

    tdt = getattr(torch, dtype)
    b, h, s, d = shape
    rng = np.random.default_rng(s + h + s_kv)
    q, qn = round_to(rng.standard_normal(shape, dtype=np.float32), tdt)
    (k, kn), (v, vn) = (round_to(rng.standard_normal((b, h, s_kv, d), dtype=np.float32), tdt) for _ in range(2))
    q, k, v = (t.to(device) for t in (q, k, v))
    scale = 1.0 / np.sqrt(d)
    outs = []
    for stages in (2, 3):
        out = torch.full(shape, float("nan"), dtype=tdt, device=device)
        print(f"[fa] persistent check {shape} s_kv={s_kv} {dtype} memory_stage={stages}", flush=True)
        native.flash_attention(out, q, k, v, 64, 64, scale, False, memory_stage=stages)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    got = to_numpy(outs[0])
    assert np.isfinite(got).all()
    heads, blocks = [(0, 0), (b - 1, h - 1)], [(0, 64), (s - 64, s)]
    if s_kv == s:
        _sampled_check(oracle_mod, got, qn, kn, vn, heads, blocks, scale, False, f"{shape}")
        return
    for bb, hh in heads:
        for m0, m1 in blocks:
            logits = qn[bb, hh, m0:m1].astype(np.float64) @ kn[bb, hh].astype(np.float64).T * scale
            w = np.exp(logits - logits.max(axis=1, keepdims=True))
            ref = (w / w.sum(axis=1, keepdims=True)) @ vn[bb, hh].astype(np.float64)
            assert_h16_close(got[bb, hh, m0:m1], ref, what=f"{shape} s_kv={s_kv} b={bb} h={hh} rows {m0}:{m1}")


def test_rejects_bad_args(device):
    import torch

    q = torch.zeros(1, 1, 8, 4, device=device)
    o = torch.zeros(1, 1, 8, 4, device=device)
    with pytest.raises(native.NativeLibraryError):
        native.flash_attention(o, q, q, q, 0, 4)
    with pytest.raises(native.NativeLibraryError):
        native.call_entry("kg_gfx950_flash_attention_entry", (o, q, q, q, 4, 4, 1.0, 2))


DECODE = [
    # (b, h, s_q, s_kv, d): one step of keys, a step's edges, ranges that end mid-step, splits
    (1, 2, 1, 1, 128), (2, 1, 3, 31, 64), (1, 3, 16, 33, 128), (1, 2, 7, 64, 64), (2, 3, 1, 257, 128),
    (1, 5, 2, 4097, 128), (3, 2, 16, 2049, 64), (4, 32, 1, 1000, 128),
    (1, 3, 17, 1030, 128), (1, 2, 300, 1025, 64),  # blocks of 16 queries, the last one partial
]


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("b,h,s_q,s_kv,d", DECODE)
def test_few_queries(device, b, h, s_q, s_kv, d, dtype):
    """Few queries take the kernel that splits the keys over workgroups (the entry's cost record
    shows the route). Reference: the softmax formula in float64 on the rounded inputs; bar:
    gpu_util.attention_h16_tolerance. The first 40 keys of a head with more are then made to
    score -inf for every query (whole steps without a finite score): they must weigh nothing."""

    import torch

    from tests.gpu_util import attention_h16_tolerance

    tdt = getattr(torch, dtype)
    rng = np.random.default_rng(s_q + s_kv + d)
    q, qn = round_to(rng.standard_normal((b, h, s_q, d), dtype=np.float32), tdt)
    (k, kn), (v, vn) = (round_to(rng.standard_normal((b, h, s_kv, d), dtype=np.float32), tdt) for _ in range(2))
    scale = 1.0 / np.sqrt(d)
    steps, chunks = (-(-s_kv // 32), 1) if d == 128 else (-(-s_kv // 64), 2)
    specs = [native.TensorSpec(x, dtype) for x in (q.shape, q.shape, k.shape, k.shape)]
    assert native.cost("flash_attention", [*specs, 64, 64, scale, 0])["MFMA"] == \
        b * h * -(-s_q // 16) * steps * chunks * (d // 8 + 1)

    def check(qn, kn, what):
        out = torch.full(q.shape, float("nan"), dtype=tdt, device=device)
        print(f"[fa] few queries {what} {(b, h, s_q, s_kv, d)} {dtype}", flush=True)
        native.flash_attention(out, torch.from_numpy(qn).to(tdt).to(device), torch.from_numpy(kn).to(tdt).to(device),
                               v.to(device), 64, 64, scale, False)
        live = np.isfinite(kn).all(axis=(0, 1, 3))
        s = qn.astype(np.float64) @ kn[:, :, live].astype(np.float64).swapaxes(-1, -2) * scale
        w = np.exp(s - s.max(-1, keepdims=True))
        ref = (w / w.sum(-1, keepdims=True)) @ vn[:, :, live].astype(np.float64)
        tol = attention_h16_tolerance(qn, kn[:, :, live], vn[:, :, live], scale, False, dtype)
        assert_within(to_numpy(out), ref, tol, what=what)

    check(qn, kn, "normal")
    if s_kv > 60:
        dead = kn.copy()
        dead[:, :, :40] = -np.inf
        check(np.abs(qn) + np.float32(0.125), dead, "dead keys")


def test_few_queries_under_capture(device):
    """A graph's call with split keys has a workspace of the graph's own; every replay gives the
    softmax formula's result."""

    import torch

    q = torch.randn(1, 2, 1, 128, device=device).bfloat16()
    k, v = (torch.randn(1, 2, 3000, 128, device=device).bfloat16() for _ in range(2))
    out = torch.empty_like(q)
    stream = torch.cuda.Stream(device=device)
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    try:
        with torch.cuda.graph(graph, stream=stream):
            native.set_launch_mode(False, stream.cuda_stream)
            native.flash_attention(out, q, k, v, 64, 64, 0.088, False)
    finally:
        native.set_launch_mode(True, None)
    qd, kd, vd = (t.double()[0] for t in (q, k, v))
    ref = torch.stack([torch.softmax(0.088 * (qd[i] @ kd[i].t().contiguous()), -1) @ vd[i] for i in range(2)])
    eager = torch.empty_like(out)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        native.flash_attention(eager, q, k, v, 64, 64, 0.088, False)
        torch.cuda.synchronize()
        for got in (out, eager):
            assert_h16_close(to_numpy(got[0]), ref.cpu().numpy(), what="replay")


ANY_DIM = [
    # (b, h, s_q, s_kv, d, causal): dims with and without whole 16-column blocks, blocks of 16 queries
    # with a partial last one, split keys (few heads), one step, more steps than waves
    (1, 2, 70, 70, 24, True), (2, 1, 33, 130, 40, False), (1, 3, 257, 257, 48, True), (1, 1, 16, 1000, 72, False),
    (1, 2, 300, 300, 80, True), (2, 2, 100, 65, 96, False), (1, 1, 1, 33, 120, False), (1, 1, 700, 700, 104, True),
]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("b,h,s_q,s_kv,d,causal", ANY_DIM + [(1, 5, 77, 77, 64, True), (1, 2, 16, 500, 128, False)])
def test_any_head_dim(device, b, h, s_q, s_kv, d, causal, dtype):
    """Head dims without a tiled kernel (and small fp32 calls with D = 64 and 128) take the
    split-key kernels. Reference: the softmax formula in float64; bars: gpu_util's, plus for
    fp32 the float64 reference's distance to the bar's own. The inputs sit in buffers whose other
    elements are NaN, so a read outside a row's columns shows."""

    import torch

    from tests.gpu_util import attention_h16_tolerance

    tdt = getattr(torch, dtype)
    rng = np.random.default_rng(s_q + s_kv + d)
    arrays, tensors = [], []
    for s in (s_q, s_kv, s_kv):
        t, a = round_to(rng.standard_normal((b, h, s, d), dtype=np.float32), tdt)
        guard = torch.full((t.numel() + 512,), float("nan"), dtype=tdt, device=device)
        guard[256 : 256 + t.numel()] = t.flatten().to(device)
        arrays.append(a)
        tensors.append(guard[256 : 256 + t.numel()].view(b, h, s, d))
    scale = 1.0 / np.sqrt(d)
    guard = torch.full((b * h * s_q * d + 512,), float("nan"), dtype=tdt, device=device)
    out = guard[256:-256].view(b, h, s_q, d)
    print(f"[fa] any dim {(b, h, s_q, s_kv, d)} causal={causal} {dtype}", flush=True)
    native.flash_attention(out, *tensors, 64, 64, scale, causal)
    qn, kn, vn = (a.astype(np.float64) for a in arrays)
    s = qn @ kn.swapaxes(-1, -2) * scale
    if causal:
        s = np.where(np.tril(np.ones((s_q, s_kv), bool)), s, -np.inf)
    w = np.exp(s - s.max(-1, keepdims=True))
    ref = (w / w.sum(-1, keepdims=True)) @ vn
    tol = attention_f32_tolerance(*arrays, scale, causal) if dtype == "float32" else \
        attention_h16_tolerance(*arrays, scale, causal, dtype)
    assert_within(to_numpy(out), ref, tol, what=f"{(b, h, s_q, s_kv, d)} {causal} {dtype}")
    assert torch.isnan(guard[:256]).all() and torch.isnan(guard[-256:]).all(), "store outside the output"


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("b,h,s_q,s_kv,d,causal", ANY_DIM)
def test_any_head_dim_keeps_probabilities_in_fp32(device, b, h, s_q, s_kv, d, causal, dtype):
    """16-bit calls of other head dims round to 16 bits once, in the output: scores, probabilities
    and both sums are fp32. Reference: the softmax formula in float64 on the rounded inputs. Bar:
    the output's own rounding (u = 2^-8 for bf16's 8 significand bits, 2^-11 for f16's 11; 2^-25
    below f16's normal range) of a value that the fp32 arithmetic has moved by at most
    attention_f32_tolerance's first-order terms (without its flat 1e-5 + 1e-4 |o|, which is
    no rounding bound). Probabilities in 16 bits miss it where an output cancels: they move O_i by about
    u sqrt(sum_j w_j^2 (V_j - O_i)^2), which does not shrink with |O_i|."""

    import torch

    tdt = getattr(torch, dtype)
    rng = np.random.default_rng(3 * s_q + s_kv + d)
    (q, qn), (k, kn), (v, vn) = (round_to(rng.standard_normal((b, h, s, d), dtype=np.float32), tdt)
                                 for s in (s_q, s_kv, s_kv))
    scale = 1.0 / np.sqrt(d)
    out = torch.full(q.shape, float("nan"), dtype=tdt, device=device)
    print(f"[fa] fp32 probabilities {(b, h, s_q, s_kv, d)} causal={causal} {dtype}", flush=True)
    native.flash_attention(out, q.to(device), k.to(device), v.to(device), 64, 64, scale, causal)
    s = qn.astype(np.float64) @ kn.astype(np.float64).swapaxes(-1, -2) * scale
    if causal:
        s = np.where(np.tril(np.ones((s_q, s_kv), bool)), s, -np.inf)
    w = np.exp(s - s.max(-1, keepdims=True))
    ref = (w / w.sum(-1, keepdims=True)) @ vn.astype(np.float64)
    moved = attention_f32_tolerance(qn, kn, vn, scale, causal) - 1e-5 - 1e-4 * np.abs(ref)
    u = {"bfloat16": 2.0**-8, "float16": 2.0**-11}[dtype]
    assert_within(to_numpy(out), ref, u * (np.abs(ref) + moved) + 2.0**-25 + moved, what=f"{(b, h, s_q, s_kv, d)} {dtype}")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("b,h,s,d", [(1, 2, 70, 24), (1, 1, 45, 72), (2, 1, 300, 80), (1, 1, 16, 96), (1, 1, 700, 120)])
def test_causal_masked_values_are_not_read(device, b, h, s, d, dtype):
    """Head dims of the split-key kernels, causal: an infinity or NaN in V's row j belongs to queries
    j and later only; earlier queries of the same block keep the bits they have without it. Rows at a
    block's start, middle and end, one step and several, the last key among them."""

    import torch

    tdt = getattr(torch, dtype)
    gen = torch.Generator(device=device).manual_seed(s + d)
    q, k, v = (torch.randn(b, h, s, d, generator=gen, device=device).to(tdt) for _ in range(3))
    scale = 1.0 / d**0.5

    def run(values):
        out = torch.full(q.shape, float("nan"), dtype=tdt, device=device)
        native.flash_attention(out, q, k, values, 64, 64, scale, True)
        return out

    clean = run(v)
    assert torch.isfinite(clean).all()
    for j in sorted({0, 5, 15, s // 2, s // 16 * 16 - 1, s // 16 * 16, s - 1} & set(range(s))):
        for value in (float("inf"), float("-inf"), float("nan")):
            print(f"[fa] masked value {value} at key {j} {(b, h, s, d)} {dtype}", flush=True)
            bad = v.clone()
            bad[:, :, j, 3] = value
            bad[:, :, j, d - 1] = value
            got = run(bad)
            cols = [3, d - 1]
            rest = [c for c in range(d) if c not in cols]
            assert torch.equal(got[:, :, :j], clean[:, :, :j]), f"queries before key {j}"
            assert torch.equal(got[..., rest], clean[..., rest]), f"other columns, key {j}"
            seen = got[:, :, j:, cols]
            # (a weight above fp32's smallest normal: exp(-87); the scores here span far less)
            assert (torch.isnan(seen) if value != value else seen == value).all(), f"queries from key {j} on"


@pytest.mark.parametrize("s,d", [(77, 64), (200, 128)])
def test_causal_masked_values_are_not_read_small_fp32(device, s, d):
    """The same for the small fp32 calls with D = 64 and 128 that the split-key kernel takes."""

    test_causal_masked_values_are_not_read(device, 1, 2, s, d, "float32")
