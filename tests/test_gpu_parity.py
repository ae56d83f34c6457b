"""GPU parity: the HIP path (through the C ABI) against the CPU oracle on the
same seeded inputs.

Bar: top-k expert ids, per-expert offsets and row lists bit-exact (ties to the
lowest expert id); layer outputs within max-abs 2e-3 x output RMS.  Below the
f16 threshold the kernels accumulate quantized block dots exactly (f64) and use the
same deterministic exp, so outputs are in practice bit-identical; that is
asserted separately as a fraction so a rare router rounding flip does not hide
behind it.  From MoELayer.f16_min_tokens on (22 rows per expert in Q4_0 and 28 in Q8_0
with prefill copies, 36 and 56 without; 128 tokens at least) or when forced, the grouped
GEMMs run f16 MFMAs: the block dots are exact, their scaled sum is accumulated in f32, and every h
value whose Q8_0 rounding that error could change is recomputed exactly, so the
h quants match the oracle's; outputs differ by f32 rounding of the sums (about
1e-6 x RMS), held to MFMA_TOL, a hundred times tighter than the bar.
"""
import numpy as np
import pytest
import torch

from oracle import pyoracle as po
from qwenium_amd import TYPE_Q4_0, TYPE_Q8_0, synthetic
from qwenium_amd.synthetic import LayerSpec

pytestmark = pytest.mark.gpu

TOL = 2e-3
# bound on the f16-MFMA prefill path's error (max |y - y_ref| / rms of y_ref;
# measured <= 1.6e-6 at 35B-A3B prefill shapes); one h quant off by one would
# exceed it
MFMA_TOL = 2e-5


def host_layer(spec: LayerSpec, tensors: dict) -> po.Layer:
    host = {}
    for k, v in tensors.items():
        a = v.data.cpu().numpy()
        if k == "router":
            a = a.reshape(spec.n_experts, spec.n_embd)
        host[k] = a
    return po.Layer(spec.n_embd, spec.n_experts, spec.top_k, spec.ffn_dim, spec.shared, spec.wtype, host)


def run_pair(spec: LayerSpec, T: int, seed: int, batch: int = 0, x=None, copies: bool = True):
    tensors = synthetic.make_layer_tensors(spec, seed)
    layer = synthetic.make_layer(spec, seed, tensors=tensors, prefill_copies=copies)
    if x is None:
        x = synthetic.make_x(spec, T, seed, batch)
    y, dbg = layer.forward(x, debug=True)
    torch.cuda.synchronize()
    ref = host_layer(spec, tensors)
    y_ref, d_ref = ref.forward(x.cpu().numpy(), debug=True)
    got = {k: v.cpu().numpy() for k, v in dbg.items()}
    return y.cpu().numpy(), got, y_ref, d_ref, layer, tensors, ref


def ref_h_q8(d_ref, spec: LayerSpec):
    """The oracle's Q8_0 of h, as the down projection reads it: quants [R, F] and
    block scales [R, F/32] (R = assignment rows, then the shared expert's rows)."""
    h = d_ref["h"]
    if spec.shared:
        h = np.concatenate([h, d_ref["sh_h"]], axis=0)
    R, F = h.shape
    blocks = po.quantize_act(h).reshape(R, F // 32, 34)
    d = blocks[:, :, :2].copy().view(np.float16)[..., 0].astype(np.float32)
    q = blocks[:, :, 2:].copy().view(np.int8).reshape(R, F)
    return q, d


def assert_h_exact(got, d_ref, spec: LayerSpec):
    """h's Q8_0 (every quant and block scale) equals the oracle's, bit for bit."""
    q, d = ref_h_q8(d_ref, spec)
    bad = np.argwhere(got["h_qs"] != q)
    assert bad.size == 0, f"{len(bad)} h quants differ, first at (row, col) {tuple(bad[0])}: " \
                          f"{int(got['h_qs'][tuple(bad[0])])} vs {int(q[tuple(bad[0])])}"
    np.testing.assert_array_equal(got["h_d"].view(np.int32), d.view(np.int32), err_msg="h block scales")


def assert_parity(y, got, y_ref, d_ref, spec: LayerSpec, min_identical=0.999, mfma=False):
    np.testing.assert_array_equal(got["topk_idx"], d_ref["topk_idx"])
    np.testing.assert_array_equal(got["offsets"], d_ref["offsets"])
    np.testing.assert_array_equal(got["rows"], d_ref["rows"])
    # logits: correctly rounded f32 of an exact dot on both sides
    ulp = np.abs(got["logits"].view(np.int32).astype(np.int64) - d_ref["logits"].view(np.int32).astype(np.int64))
    assert ulp.max() <= 1, f"router logits differ by {ulp.max()} ulp"
    np.testing.assert_allclose(got["topk_w"], d_ref["topk_w"], rtol=1e-6, atol=0)
    if spec.shared:
        np.testing.assert_allclose(got["sh_gate"], d_ref["sh_gate"], rtol=1e-6, atol=0)
    if "h_qs" in got and "h" in d_ref:
        assert_h_exact(got, d_ref, spec)
        assert got["h_fixed"][0] >= 0 and (mfma or got["h_fixed"][0] == 0)
    rms = float(np.sqrt(np.mean(y_ref.astype(np.float64) ** 2)))
    err = float(np.max(np.abs(y - y_ref)))
    assert err <= TOL * rms, f"max |y - y_ref| = {err:.3e} > {TOL} * rms ({rms:.3e})"
    identical = float(np.mean(y.view(np.int32) == y_ref.view(np.int32)))
    if mfma:
        assert err <= MFMA_TOL * rms, f"f16-MFMA path: max |y - y_ref| = {err / rms:.2e} x rms > {MFMA_TOL}"
    else:
        assert identical >= min_identical, f"only {identical:.5f} of outputs bit-identical"
    return err, rms, identical


@pytest.mark.parametrize("wtype", [TYPE_Q4_0, TYPE_Q8_0])
def test_synth_generator_matches_cpu(gpu, wtype):
    """Device generator == CPU recipe, byte for byte (f32 and quantized)."""
    x = synthetic.synth_f32(100_003, 11, 5, 0.0, 1.0).cpu().numpy()
    np.testing.assert_array_equal(x.view(np.uint32), po.gen_normal_f32(11, 5, 100_003).view(np.uint32))
    q = synthetic.synth_quant(wtype, 37, 256, 3, 9, 0.02).cpu().numpy()
    ref = po.quantize(wtype, po.gen_normal_f32(3, 9, 37 * 256, 0.0, 0.02))
    np.testing.assert_array_equal(q, ref)


def test_config1_q8_0(gpu):
    """hidden 1024, 16 experts, top-2, ffn 512, no shared, Q8_0, 32 tokens, seed 0."""
    spec = synthetic.CONFIG1
    y, got, y_ref, d_ref, *_ = run_pair(spec, 32, seed=0)
    assert_parity(y, got, y_ref, d_ref, spec)


def test_decode_35b_q4_0_t10(gpu):
    """35B-A3B shape at decode: hidden 2048, 256 experts, top-8 + shared, Q4_0, 10 tokens."""
    spec = synthetic.QWEN35B
    y, got, y_ref, d_ref, *_ = run_pair(spec, 10, seed=1)
    assert_parity(y, got, y_ref, d_ref, spec)
    distinct = len(np.unique(got["topk_idx"]))
    assert 40 <= distinct <= 80


@pytest.mark.parametrize("spec,T", [(synthetic.QWEN35B, 1), (synthetic.QWEN35B, 3), (synthetic.QWEN35B, 16),
                                    (synthetic.QWEN35B_Q8, 5)])
def test_decode_35b_token_counts(gpu, spec, T):
    """35B shape (shared expert of ffn 512) at decode sizes: the shared expert's down projection
    runs in the gate/up launch (odd and even tokens on separate waves) and enters the down+combine
    kernel as its last step; routing and outputs match the oracle as on every other path."""
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=200 + T)
    assert_parity(y, got, y_ref, d_ref, spec)


@pytest.mark.parametrize("wtype,copies,T,f16_from", [
    (TYPE_Q4_0, True, 160, 704), (TYPE_Q4_0, True, 176, 704), (TYPE_Q4_0, True, 703, 704), (TYPE_Q4_0, True, 704, 704),
    (TYPE_Q4_0, False, 1151, 1152), (TYPE_Q4_0, False, 1152, 1152),
    (TYPE_Q8_0, True, 895, 896), (TYPE_Q8_0, True, 896, 896),
    (TYPE_Q8_0, False, 1791, 1792), (TYPE_Q8_0, False, 1792, 1792)])
def test_35b_around_mfma_threshold(gpu, wtype, copies, T, f16_from):
    """The 35B shape switches to the f16-MFMA GEMMs where an expert averages 22 rows (Q4_0 with
    prefill copies), 36 (without), 28 or 56 (Q8_0): one token below, the exact int8 GEMMs give
    the oracle's bits; at the switch the f16 GEMMs list h blocks for their fixup, h quants are
    exact and outputs within MFMA_TOL; routing bit-exact on all."""
    spec = synthetic.QWEN35B if wtype == TYPE_Q4_0 else synthetic.QWEN35B_Q8
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=500 + T, copies=copies)
    assert layer.f16_min_tokens == f16_from
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T >= f16_from, min_identical=1.0)
    assert (got["h_fixed"][0] > 0) == (T >= f16_from)


@pytest.mark.parametrize("spec,T", [(LayerSpec(4096, 64, 4, 256, True, TYPE_Q8_0), 7),
                                    (LayerSpec(3072, 96, 6, 512, True, TYPE_Q4_0), 12),
                                    (LayerSpec(1280, 40, 4, 512, False, TYPE_Q4_0), 9)])
def test_decode_hidden_sizes(gpu, spec, T):
    """Decode routing at hidden 4096 / 3072 / 1280: four, three and two 256-column slabs per
    router wave (the last two waves of 3072 and the last of 1280 with one slab fewer)."""
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=300 + T)
    assert_parity(y, got, y_ref, d_ref, spec)


@pytest.mark.parametrize("spec,T", [(LayerSpec(4096, 64, 4, 256, True, TYPE_Q8_0), 20),
                                    (LayerSpec(3072, 96, 6, 512, True, TYPE_Q4_0), 40),
                                    (LayerSpec(1280, 40, 4, 512, False, TYPE_Q4_0), 50)])
def test_grouped_router_hidden_sizes(gpu, spec, T):
    """17 tokens to the batched router's threshold at hidden 4096 / 3072 / 1280: four, three and two
    256-column slabs per router wave, x's Q8_0 rows written by the router's blocks."""
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=310 + T)
    assert_parity(y, got, y_ref, d_ref, spec)


@pytest.mark.parametrize("spec,T", [(LayerSpec(96, 8, 2, 32, True, TYPE_Q4_0), 1),
                                    (LayerSpec(96, 8, 2, 32, True, TYPE_Q4_0), 10),
                                    (LayerSpec(320, 16, 4, 96, True, TYPE_Q8_0), 17),
                                    (LayerSpec(160, 12, 3, 224, False, TYPE_Q4_0), 300),
                                    (LayerSpec(160, 12, 3, 224, False, TYPE_Q4_0), 1100),
                                    (LayerSpec(1056, 32, 4, 96, True, TYPE_Q4_0), 10),
                                    (LayerSpec(1056, 32, 4, 96, True, TYPE_Q4_0), 150)])
def test_padded_widths(gpu, spec, T):
    """n_embd and ffn_dim that Q4_0/Q8_0 rows allow (multiples of 32) but the kernels'
    grid does not (multiples of 256 and 64): the layer runs on zero-padded weight copies
    and zero-padded rows, and routing and outputs match the oracle at the caller's widths
    as on every other path (decode, the int8 GEMMs (17 and 150 tokens), the f16 GEMMs below the
    batched router (300 tokens) and with it (1100))."""
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=400 + T)
    assert layer.n_embd == spec.n_embd and y.shape == (T, spec.n_embd)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T >= layer.f16_min_tokens)


@pytest.mark.parametrize("spec,T", [(LayerSpec(256, 256, 16, 64, True, TYPE_Q4_0), 300),
                                    (LayerSpec(256, 256, 17, 64, True, TYPE_Q4_0), 300),
                                    (LayerSpec(256, 64, 24, 128, False, TYPE_Q8_0), 1100)])
def test_expert_lists_wide_top_k(gpu, spec, T):
    """The per-expert lists built from the top-k blocks' token masks (top-k blocks x experts
    above 4096) at top_k 16, 17 and 24: each listed token's slot comes from the four-bit
    fields that the top-k writes up to top_k 16 and from a search of the token's selection
    above it; f64-MFMA router and int8 GEMMs (300 tokens), batched router and f16 GEMMs (1100)."""
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=450 + spec.top_k)
    assert (T >= layer.f16_min_tokens) == (T == 1100)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T == 1100)


@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 33, 64])
def test_token_counts_small_layer(gpu, T):
    """Edge token counts: single token, block boundaries of the top-k sort (16 per block)."""
    spec = LayerSpec(256, 32, 4, 128, True, TYPE_Q4_0)
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=100 + T)
    assert_parity(y, got, y_ref, d_ref, spec)


def test_zero_tokens_is_noop(gpu):
    spec = LayerSpec(256, 32, 4, 128, True, TYPE_Q4_0)
    layer = synthetic.make_layer(spec, 3)
    x = torch.empty((0, spec.n_embd), dtype=torch.float32, device="cuda")
    y = layer.forward(x)
    assert y.shape == (0, spec.n_embd)


def test_router_ties_lowest_index(gpu):
    """Duplicate router rows give exactly equal logits: the lower expert id wins."""
    spec = LayerSpec(256, 16, 4, 128, False, TYPE_Q8_0)
    tensors = synthetic.make_layer_tensors(spec, 21)
    r = tensors["router"].data.view(spec.n_experts, spec.n_embd)
    for a, b in ((3, 9), (4, 12), (0, 15), (7, 8)):
        r[b].copy_(r[a])
    layer = synthetic.make_layer(spec, 21, tensors=tensors)
    x = synthetic.make_x(spec, 64, 21)
    y, dbg = layer.forward(x, debug=True)
    torch.cuda.synchronize()
    ref = host_layer(spec, tensors)
    y_ref, d_ref = ref.forward(x.cpu().numpy(), debug=True)
    got = {k: v.cpu().numpy() for k, v in dbg.items()}
    assert_parity(y.cpu().numpy(), got, y_ref, d_ref, spec)
    idx = got["topk_idx"]
    for a, b in ((3, 9), (4, 12), (0, 15), (7, 8)):
        both = (idx == a).any(1) & (idx == b).any(1)
        pa = np.argmax(idx == a, axis=1)
        pb = np.argmax(idx == b, axis=1)
        assert np.all(pa[both] < pb[both]), "tied experts must be ordered lowest id first"


def test_residual_add(gpu):
    spec = LayerSpec(256, 32, 4, 128, True, TYPE_Q4_0)
    tensors = synthetic.make_layer_tensors(spec, 5)
    layer = synthetic.make_layer(spec, 5, tensors=tensors)
    x = synthetic.make_x(spec, 9, 5)
    res = synthetic.make_x(spec, 9, 5, batch=1)
    y0 = layer.forward(x)
    y1 = layer.forward(x, residual=res)
    torch.cuda.synchronize()
    expect = (y0.cpu().numpy() + res.cpu().numpy()).astype(np.float32)
    np.testing.assert_array_equal(y1.cpu().numpy(), expect)


def test_deterministic_repeat(gpu):
    spec = synthetic.QWEN35B
    tensors = synthetic.make_layer_tensors(spec, 2)
    layer = synthetic.make_layer(spec, 2, tensors=tensors)
    x = synthetic.make_x(spec, 37, 2)
    a = layer.forward(x).cpu().numpy()
    b = layer.forward(x).cpu().numpy()
    np.testing.assert_array_equal(a.view(np.int32), b.view(np.int32))


def test_rms_norm_matches_oracle(gpu):
    from qwenium_amd import rms_norm
    x = synthetic.synth_f32(7 * 2048, 4, 77).view(7, 2048)
    w = synthetic.synth_f32(2048, 4, 78, 1.0, 0.02)
    y = rms_norm(x, w, 1e-6).cpu().numpy()
    ref = po.rms_norm(x.cpu().numpy(), w.cpu().numpy(), 1e-6)
    np.testing.assert_allclose(y, ref, rtol=2e-7, atol=0)


@pytest.mark.parametrize("H", [2048, 1000, 4096])
def test_rms_partials_matches_oracle(gpu, H):
    """The RMSNorm partial sums (32 columns per entry) equal the oracle's bits."""
    from qwenium_amd import rms_partials
    x = synthetic.synth_f32(7 * H, 4, 91).view(7, H)
    got = rms_partials(x).cpu().numpy()
    np.testing.assert_array_equal(got, po.rms_partials(x.cpu().numpy()))


def test_config1_matches_committed_golden(gpu):
    """GPU path vs tests/golden/config1_seed0.npz (written by the CPU oracle)."""
    import os
    ref = np.load(os.path.join(os.path.dirname(__file__), "golden", "config1_seed0.npz"), allow_pickle=False)
    spec = synthetic.CONFIG1
    layer = synthetic.make_layer(spec, 0)
    x = synthetic.make_x(spec, 32, 0)
    y, dbg = layer.forward(x, debug=True)
    got = {k: v.cpu().numpy() for k, v in dbg.items()}
    d_ref = {k: ref[k] for k in ("topk_idx", "offsets", "rows", "logits", "topk_w")}
    assert_parity(y.cpu().numpy(), got, ref["y"], d_ref, spec, min_identical=1.0)


def test_constant_weights_closed_form(gpu):
    """All experts identical (the constant fills of tests/unit/test_moe.cpp:93-101):
    routing cannot matter and y has a closed form in the quantized constants."""
    import math
    H, E, K, F, T = 256, 8, 2, 64, 3
    wt = TYPE_Q8_0
    dev = "cuda"
    from qwenium_amd.moe import GGMLTensor, Hparams, MoELayer

    def qconst(v, n):
        return torch.from_numpy(po.quantize(wt, np.full(n, v, np.float32))).to(dev)

    t = {
        "router": GGMLTensor(torch.full((E * H,), 0.1, device=dev), 0, (H, E)),
        "gate": GGMLTensor(qconst(0.05, E * F * H), wt, (H, F, E)),
        "up": GGMLTensor(qconst(0.05, E * F * H), wt, (H, F, E)),
        "down": GGMLTensor(qconst(0.05, E * H * F), wt, (F, H, E)),
        "sh_gate": GGMLTensor(qconst(0.02, F * H), wt, (H, F)),
        "sh_up": GGMLTensor(qconst(0.02, F * H), wt, (H, F)),
        "sh_down": GGMLTensor(qconst(0.02, H * F), wt, (F, H)),
        "sh_norm": GGMLTensor(torch.full((H,), 0.5, device=dev), 0, (H,)),
    }
    layer = MoELayer(t["router"], t["gate"], t["up"], t["down"], t["sh_gate"], t["sh_up"], t["sh_down"],
                     t["sh_norm"], Hparams(E, K, F, True))
    y, dbg = layer.forward(torch.full((T, H), 0.5, device=dev), debug=True)
    idx = dbg["topk_idx"].cpu().numpy()
    assert idx.tolist() == [[0, 1]] * T  # all logits tie: lowest ids win

    def q8(v):
        return float(po.dequantize(po.TYPE_Q8_0, po.quantize(po.TYPE_Q8_0, np.full(32, v, np.float32)), 32)[0])

    xq = q8(0.5)
    g = H * q8(0.05) * xq
    routed = F * q8(0.05) * q8(g / (1 + math.exp(-g)) * g)
    gs = H * q8(0.02) * xq
    ys = F * q8(0.02) * q8(gs / (1 + math.exp(-gs)) * gs)
    expect = routed + ys / (1 + math.exp(-(H * 0.5 * 0.5)))
    np.testing.assert_allclose(y.cpu().numpy(), expect, rtol=2e-6)


def test_graph_replay_matches_eager(gpu):
    """The forward captured in a HIP graph: every replay (with eager work and
    synchronizations between replays) equals the eager result bit for bit."""
    from qwenium_amd import Workspace
    spec = synthetic.QWEN35B
    layers = [synthetic.make_layer(spec, 40 + i) for i in range(2)]
    xs = [synthetic.make_x(spec, 10, 40, batch=b) for b in range(2)]
    ws = Workspace(layers[0], 10)
    eager = [layers[i].forward(xs[i], workspace=ws).clone() for i in range(2)]
    outs = [torch.empty_like(xs[0]) for _ in range(2)]
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    with torch.cuda.graph(g, stream=s):
        for i in range(2):
            layers[i].forward(xs[i], out=outs[i], workspace=ws)
    for rep in range(4):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for i in range(2):
            np.testing.assert_array_equal(outs[i].cpu().numpy().view(np.int32), eager[i].cpu().numpy().view(np.int32))
        layers[1].forward(xs[0], workspace=ws)  # eager work between replays
        torch.cuda.synchronize()


@pytest.mark.parametrize("spec,T", [(synthetic.QWEN35B, 40), (synthetic.QWEN35B, 512), (synthetic.QWEN35B, 720),
                                    (LayerSpec(4096, 16, 2, 128, True, TYPE_Q8_0), 17)])
def test_graph_replay_prefill_matches_eager(gpu, spec, T):
    """Forwards past decode captured in a HIP graph: every replay equals the eager result bit
    for bit.  40 and 512 tokens: f64-MFMA router, int8 GEMMs (the merged top-k, whose last
    workgroup builds the lists, and the list launch); 720: batched router, f16-MFMA GEMMs,
    fixups; the small layer: the router's row pairs, gate/up workgroups split in four parts
    (above 64 KiB of LDS)."""
    from qwenium_amd import Workspace
    layers = [synthetic.make_layer(spec, 70 + i) for i in range(2)]
    assert (T >= layers[0].f16_min_tokens) == (T == 720)
    xs = [synthetic.make_x(spec, T, 70, batch=b) for b in range(2)]
    ws = Workspace(layers[0], T)
    eager = [layers[i].forward(xs[i], workspace=ws).clone() for i in range(2)]
    outs = [torch.empty_like(xs[0]) for _ in range(2)]
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    with torch.cuda.graph(g, stream=s):
        for i in range(2):
            layers[i].forward(xs[i], out=outs[i], workspace=ws)
    for rep in range(3):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for i in range(2):
            np.testing.assert_array_equal(outs[i].cpu().numpy().view(np.int32), eager[i].cpu().numpy().view(np.int32))
        layers[1].forward(xs[0], workspace=ws)  # eager work between replays
        torch.cuda.synchronize()


# ---- f16-MFMA grouped GEMM path (prefill) -------------------------------------------------
@pytest.mark.parametrize("wtype", [TYPE_Q4_0, TYPE_Q8_0])
@pytest.mark.parametrize("T", [1, 17, 64, 65, 130])
def test_mfma_path_small_layer(gpu, monkeypatch, wtype, T):
    """Forced MFMA path (QMOE_MFMA_MIN_TOKENS=1) on small shapes: tile edges at 64 rows."""
    monkeypatch.setenv("QMOE_MFMA_MIN_TOKENS", "1")
    spec = LayerSpec(256, 16, 4, 128, True, wtype)
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=200 + T)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=True)


def test_mfma_config1_forced(gpu, monkeypatch):
    monkeypatch.setenv("QMOE_MFMA_MIN_TOKENS", "1")
    spec = synthetic.CONFIG1
    y, got, y_ref, d_ref, *_ = run_pair(spec, 32, seed=0)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=True)


def test_mfma_35b_q4_0_t256(gpu, monkeypatch):
    monkeypatch.setenv("QMOE_MFMA_MIN_TOKENS", "256")
    spec = synthetic.QWEN35B
    y, got, y_ref, d_ref, *_ = run_pair(spec, 256, seed=9)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=True)


def check_router_bound(got, exact_logits):
    """The batched router's approximate logits lie within their stated bound of
    the exact logits; returns the largest |error| / bound."""
    approx, bound = got["router_approx"], got["router_bound"]
    assert np.isfinite(approx).all() and np.isfinite(bound).all(), "batched router did not run"
    err = np.abs(approx.astype(np.float64) - exact_logits.astype(np.float64))
    ratio = err / bound.astype(np.float64)
    assert ratio.max() <= 1.0, f"approximate logit outside its bound (max |err|/bound {ratio.max():.3f})"
    return float(ratio.max())


@pytest.mark.parametrize("T", [17, 33, 100, 300])
def test_batched_router_forced_small_layer(gpu, monkeypatch, T):
    """bf16-MFMA router + exact refinement forced at small T: tile edges in tokens and
    experts (E=16 < one 64-expert tile)."""
    monkeypatch.setenv("QMOE_BIG_ROUTER_MIN_TOKENS", "1")
    spec = LayerSpec(256, 16, 4, 128, True, TYPE_Q4_0)
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=300 + T)
    assert_parity(y, got, y_ref, d_ref, spec, min_identical=1.0, mfma=T >= layer.f16_min_tokens)
    check_router_bound(got, d_ref["logits"])


@pytest.mark.parametrize("T", [200, 223, 224, 300, 600, 719, 720])
def test_router_threshold_35b(gpu, T):
    """At the 35B-A3B shape the f64-MFMA router runs up to 719 tokens and the batched router
    from 720, with debug buffers as without them: both give the oracle's routing, and only
    the batched one writes approximate logits and bounds."""
    spec = synthetic.QWEN35B
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=31)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T >= layer.f16_min_tokens)
    if T >= 720:
        assert check_router_bound(got, d_ref["logits"]) < 0.5
    else:
        assert not np.isfinite(got["router_approx"]).any(), "the batched router ran below its threshold"


@pytest.mark.parametrize("hidden,experts,T,batched", [(1024, 1024, 623, False), (1024, 1024, 624, True),
                                                      (4096, 1024, 399, False), (4096, 1024, 400, True)])
def test_router_threshold_large(gpu, hidden, experts, T, batched):
    """Routers of more than 655360 weights: the batched one runs from 720 tokens times the cube
    root of 655360 / weights, in steps of 16; the oracle's routing on both sides."""
    spec = LayerSpec(hidden, experts, 2, 64, False, TYPE_Q4_0)
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=33)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T >= layer.f16_min_tokens)
    if batched:
        check_router_bound(got, d_ref["logits"])
    else:
        assert not np.isfinite(got["router_approx"]).any()


@pytest.mark.parametrize("dup", ["pairs", "all"])
def test_batched_router_ties(gpu, monkeypatch, dup):
    """Exactly tied logits through the refinement: duplicated router rows ("pairs"), or
    every row equal ("all": every expert is a candidate and the lowest ids win)."""
    monkeypatch.setenv("QMOE_BIG_ROUTER_MIN_TOKENS", "1")
    spec = LayerSpec(256, 128, 8, 128, False, TYPE_Q8_0)
    tensors = synthetic.make_layer_tensors(spec, 41)
    r = tensors["router"].data.view(spec.n_experts, spec.n_embd)
    if dup == "pairs":
        for a, b in ((3, 90), (4, 12), (0, 127), (64, 65), (63, 64)):
            r[b].copy_(r[a])
    else:
        r.copy_(r[0:1].expand_as(r))
    layer = synthetic.make_layer(spec, 41, tensors=tensors)
    x = synthetic.make_x(spec, 40, 41)
    y, dbg = layer.forward(x, debug=True)
    torch.cuda.synchronize()
    ref = host_layer(spec, tensors)
    y_ref, d_ref = ref.forward(x.cpu().numpy(), debug=True)
    got = {k: v.cpu().numpy() for k, v in dbg.items()}
    assert_parity(y.cpu().numpy(), got, y_ref, d_ref, spec, min_identical=1.0)
    check_router_bound(got, d_ref["logits"])
    if dup == "all":
        assert (got["topk_idx"] == np.arange(spec.top_k)[None, :]).all()


def assert_rows_close(got, d_ref, spec: LayerSpec, T: int):
    """The unweighted expert rows (moe_exp_down, moe_shared_out) against the
    oracle's: within MFMA_TOL x their rms plus a few f32 ulps of the value
    itself (2^-20 |ref|: the f32 accumulation of large rows, e.g. under outlier
    activations, rounds at the scale of the row's own values)."""
    rows = got["exp_down"]
    ref = d_ref["y"] if not spec.shared else np.concatenate([d_ref["y"], d_ref["sh_out"]], axis=0)
    assert rows.shape == ref.shape and np.isfinite(rows).all()
    rms = float(np.sqrt(np.mean(ref.astype(np.float64) ** 2)))
    err = np.abs(rows.astype(np.float64) - ref)
    lim = MFMA_TOL * rms + 2.0 ** -20 * np.abs(ref.astype(np.float64))
    worst = np.unravel_index(np.argmax(err - lim), err.shape)
    assert (err <= lim).all(), f"expert rows: |err| {err[worst]:.3e} at {worst} (ref {ref[worst]:.4g}, rms {rms:.3g})"


def run_prefill(spec: LayerSpec, T: int, seed: int):
    """Forward on the GPU and the oracle over every token, with the per-row
    intermediates of both."""
    tensors = synthetic.make_layer_tensors(spec, seed)
    layer = synthetic.make_layer(spec, seed, tensors=tensors)
    x = synthetic.make_x(spec, T, seed)
    y, dbg = layer.forward(x, debug="rows")
    torch.cuda.synchronize()
    got = {k: v.cpu().numpy() for k, v in dbg.items()}
    ref = host_layer(spec, tensors)
    y_ref, d_ref = ref.forward(x.cpu().numpy(), debug=True)
    return y.cpu().numpy(), got, y_ref, d_ref


def test_prefill_35b_q4_0_t4096(gpu):
    """The 4096-token prefill workload against the oracle on every token: routing,
    h's Q8_0 (every quant and scale, through the exact fixup of the blocks the f32
    sums leave open, which must have run), the unweighted expert rows and the
    layer output."""
    spec = synthetic.QWEN35B
    T = 4096
    y, got, y_ref, d_ref = run_prefill(spec, T, 3)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=True)
    assert check_router_bound(got, d_ref["logits"]) < 0.5
    assert got["h_fixed"][0] > 0, "the exact fixup listed no h block"
    assert_rows_close(got, d_ref, spec, T)
    counts = np.diff(d_ref["offsets"])
    assert counts.sum() == T * spec.top_k and counts.max() < 4 * T * spec.top_k / spec.n_experts


def test_skewed_q8_0_t2048(gpu):
    """Zipf-skewed routing (2048 tokens, Q8_0): hot experts with hundreds of rows, ~46
    empty experts; every token against the oracle (routing, h's Q8_0, expert rows,
    outputs)."""
    spec = synthetic.QWEN35B_SKEW
    T = 2048
    y, got, y_ref, d_ref = run_prefill(spec, T, 5)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=True)
    assert_rows_close(got, d_ref, spec, T)
    counts = np.diff(d_ref["offsets"])
    hot = spec.skew.hot_experts(spec.n_experts)
    share = counts[hot].sum() / counts.sum()
    assert 0.4 <= share <= 0.6, f"hot-8 share {share:.3f}"
    assert (counts == 0).sum() >= 40 and counts.max() > 16 * 64


def heavy_tail_x(spec: LayerSpec, T: int, seed: int, cols: int = 6, scale: float = 50.0):
    """x ~ N(0,1) with a few columns about `scale` times larger on every token: the
    outlier columns of real residual streams."""
    x = synthetic.make_x(spec, T, seed)
    c = np.random.default_rng(seed).choice(spec.n_embd, cols, replace=False)
    x[:, torch.as_tensor(c, device=x.device)] *= scale
    return x


@pytest.mark.parametrize("wtype", [TYPE_Q4_0, TYPE_Q8_0])
def test_mfma_heavy_tails(gpu, wtype):
    """The f16-MFMA path where its f32 error estimate is stressed: 6 activation columns
    50x the others (partial sums far larger than the results they cancel to) and
    outlier weight rows (a few gate/up rows of each expert scaled 30x before
    quantization).  h's Q8_0 must still equal the oracle's exactly (the fixup
    catches every value the estimate leaves open) and outputs stay within MFMA_TOL."""
    spec = LayerSpec(2048, 32, 8, 512, True, wtype)
    T, seed = 512, 61
    tensors = synthetic.make_layer_tensors(spec, seed)
    rng = np.random.default_rng(seed)
    for name, n_rows in (("gate", spec.n_experts * spec.ffn_dim), ("up", spec.n_experts * spec.ffn_dim),
                         ("sh_gate", spec.ffn_dim)):
        rows = rng.choice(n_rows, max(4, n_rows // 64), replace=False)
        t = tensors[name]
        rb = po.row_bytes(wtype, spec.n_embd)
        raw = t.data.view(torch.uint8).view(n_rows, rb)
        # the f32 values of the chosen rows, scaled 30x and requantized
        vals = po.dequantize(wtype, raw[torch.as_tensor(rows, device=raw.device)].cpu().numpy().reshape(-1),
                             len(rows) * spec.n_embd)
        raw[torch.as_tensor(rows, device=raw.device)] = torch.as_tensor(
            po.quantize(wtype, vals * 30.0).reshape(len(rows), rb), device=raw.device)
    layer = synthetic.make_layer(spec, seed, tensors=tensors)
    x = heavy_tail_x(spec, T, seed)
    y, dbg = layer.forward(x, debug="rows")
    torch.cuda.synchronize()
    got = {k: v.cpu().numpy() for k, v in dbg.items()}
    ref = host_layer(spec, tensors)
    y_ref, d_ref = ref.forward(x.cpu().numpy(), debug=True)
    assert_parity(y.cpu().numpy(), got, y_ref, d_ref, spec, mfma=True)
    assert_rows_close(got, d_ref, spec, T)
    assert got["h_fixed"][0] > 0


@pytest.mark.parametrize("T", [1, 10, 64, 8192])
def test_stack_40_layers(gpu, T):
    """Config 5: 40 consecutive blocks x <- x + MoE_l(RMSNorm(x) * w_l) (qwen36.cpp:297-304 at
    prefill, :427-432 at decode) through the fused-norm call, at decode batches 1, 10 and 64
    and at 8192-token prefill, each block's RMSNorm partial sums carried to the next.  Layers 0
    and 39 are checked against the oracle on their actual inputs (and against the unfused
    rms_norm + forward and the call without partial sums), on every token: routing and h's
    Q8_0 bit-exact, outputs within tolerance."""
    from qwenium_amd import Workspace, rms_norm, ssq_parts

    spec = synthetic.QWEN35B
    L, seed = 40, 11
    ws = None
    x = synthetic.make_x(spec, T, seed)
    h = torch.empty_like(x)
    ssq = [None, torch.empty((T, ssq_parts(spec.n_embd)), dtype=torch.float64, device=x.device),
           torch.empty((T, ssq_parts(spec.n_embd)), dtype=torch.float64, device=x.device)]
    x_ssq = None
    keep = {}
    for l in range(L):
        t = synthetic.make_layer_tensors(spec, seed, layer=l)
        layer = synthetic.make_layer(spec, seed, layer=l, tensors=t)
        if ws is None:
            ws = Workspace(layer, T)
        wn = synthetic.make_norm_weight(spec, seed, l)
        y_ssq = ssq[1 + (l & 1)]
        if l in (0, L - 1):
            rms_norm(x, wn, synthetic.NORM_EPS, out=h)
            y, dbg = layer.forward(h, workspace=ws, residual=x, debug=True)
            y_fused = layer.forward_norm(x, wn, synthetic.NORM_EPS, workspace=ws)
            y_chain = layer.forward_norm(x, wn, synthetic.NORM_EPS, workspace=ws, x_ssq=x_ssq, y_ssq=y_ssq)
            torch.cuda.synchronize()
            assert torch.equal(y, y_fused), f"layer {l}: fused RMSNorm path"
            assert torch.equal(y, y_chain), f"layer {l}: with carried partial sums"
            keep[l] = (x.cpu().numpy(), wn.cpu().numpy(), t, y.cpu().numpy(),
                       {k: dbg[k].cpu().numpy() for k in ("topk_idx", "offsets", "rows", "h_qs", "h_d", "h_fixed")})
        else:
            y = layer.forward_norm(x, wn, synthetic.NORM_EPS, workspace=ws, x_ssq=x_ssq, y_ssq=y_ssq)
        x, x_ssq = y, y_ssq
        del t, layer
    torch.cuda.synchronize()
    assert np.isfinite(x.cpu().numpy()).all()
    assert ws.check() == 0
    for l, (xin, wn, t, yg, got) in keep.items():
        hh = po.rms_norm(xin, wn, synthetic.NORM_EPS)
        ref = host_layer(spec, t)
        # routing of every token
        idx, _ = po.topk_softmax(po.router_logits(ref.t["router"], hh), spec.top_k)
        off, rows, _ = po.sort_assignments(idx, spec.n_experts)
        np.testing.assert_array_equal(got["topk_idx"], idx, err_msg=f"layer {l}")
        np.testing.assert_array_equal(got["offsets"], off, err_msg=f"layer {l}")
        np.testing.assert_array_equal(got["rows"], rows, err_msg=f"layer {l}")
        yr, d_ref = ref.forward(hh, debug=True)
        yr = yr + xin
        ys = yg
        assert_h_exact(got, d_ref, spec)
        assert (got["h_fixed"][0] > 0) == (T >= 128), f"layer {l}: h blocks fixed {got['h_fixed'][0]}"
        rms = float(np.sqrt(np.mean(yr.astype(np.float64) ** 2)))
        assert np.max(np.abs(ys - yr)) <= TOL * rms, f"layer {l}"
        if T >= 128:  # the f16-MFMA prefill path
            assert np.max(np.abs(ys - yr)) <= MFMA_TOL * rms, f"layer {l}"
        else:
            assert np.mean(ys.view(np.int32) == yr.view(np.int32)) >= 0.999, f"layer {l}"


@pytest.mark.parametrize("n_experts,T", [(256, 10), (1024, 16), (16, 3)])
def test_fused_decode_routing_repeated(gpu, n_experts, T):
    """The decode routing (the router launch, then the routing-table launch) over
    several forwards on one workspace: every forward's routing matches the oracle,
    and Workspace.check() reports no fault."""
    from qwenium_amd import Workspace

    spec = LayerSpec(256, n_experts, 8 if n_experts >= 8 else 2, 64, True, TYPE_Q4_0)
    tensors = synthetic.make_layer_tensors(spec, 17)
    layer = synthetic.make_layer(spec, 17, tensors=tensors)
    ref = host_layer(spec, tensors)
    ws = Workspace(layer, 16)
    for batch in range(5):
        x = synthetic.make_x(spec, T, 17, batch=batch)
        y, dbg = layer.forward(x, workspace=ws, debug=True)
        torch.cuda.synchronize()
        y_ref, d_ref = ref.forward(x.cpu().numpy(), debug=True)
        got = {k: v.cpu().numpy() for k, v in dbg.items()}
        assert_parity(y.cpu().numpy(), got, y_ref, d_ref, spec, min_identical=1.0)
    assert ws.check() == 0


def _random_cases(n=32, seed=2024):
    """Seeded layer shapes and token counts across every path (decode, grouped
    router + int8 GEMMs, f16 GEMMs, batched router), padded widths and both
    weight types; fixed at import, so the parametrization is stable."""
    rng = np.random.default_rng(seed)
    cases = []
    for i in range(n):
        H = int(rng.choice([256, 512, 1024, 1056, 2048]))
        E = int(rng.choice([8, 16, 64, 128, 256]))
        K = int(min(E, rng.choice([1, 2, 4, 6, 8])))
        F = int(rng.choice([64, 96, 128, 256, 512]))
        shared = bool(rng.integers(2))
        wtype = TYPE_Q4_0 if rng.integers(2) else TYPE_Q8_0
        T = int(rng.choice([1, 5, 16, 17, 40, 130, 200, 300, 600]))
        cases.append(pytest.param(LayerSpec(H, E, K, F, shared, wtype), T, id=f"H{H}-E{E}-k{K}-F{F}-s{int(shared)}-"
                                  f"{'q4' if wtype == TYPE_Q4_0 else 'q8'}-T{T}"))
    return cases


@pytest.mark.parametrize("spec,T", _random_cases())
def test_random_shapes(gpu, spec, T):
    """Seeded random shapes against the oracle: routing bit-exact; outputs bit-identical
    below the f16 threshold, within MFMA_TOL with exact h quants from it on."""
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=700 + T)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T >= layer.f16_min_tokens, min_identical=1.0)


def _random_prefill_cases(n=48, seed=12):
    """Seeded prefill-size shapes for the per-expert lists, the top-k block sizes and the
    split router tiles: 129 to 2048 tokens, up to 1024 experts, top_k up to 20, hidden up
    to 4096 (sizes bounded so the oracle stays quick)."""
    rng = np.random.default_rng(seed)
    cases = []
    while len(cases) < n:
        H = int(rng.choice([256, 512, 1056, 2048, 2816, 4096]))
        E = int(rng.choice([8, 16, 64, 128, 256, 512, 1024]))
        K = int(min(E, rng.choice([1, 2, 4, 8, 8, 16, 17, 20])))
        F = int(rng.choice([64, 128, 512]))
        T = int(rng.choice([129, 160, 224, 300, 545, 777, 1024, 1500, 2048]))
        shared = bool(rng.integers(2))
        wtype = TYPE_Q4_0 if rng.integers(2) else TYPE_Q8_0
        if T * K * F * H > 6e9 or T * E * H > 8e9:
            continue
        cases.append(pytest.param(LayerSpec(H, E, K, F, shared, wtype), T, id=f"H{H}-E{E}-k{K}-F{F}-s{int(shared)}-"
                                  f"{'q4' if wtype == TYPE_Q4_0 else 'q8'}-T{T}"))
    return cases


@pytest.mark.parametrize("spec,T", _random_prefill_cases())
def test_random_prefill_shapes(gpu, spec, T):
    """Seeded prefill-size shapes against the oracle: routing and lists bit-exact, h quants
    exact and outputs within MFMA_TOL on the f16 path (bit-identical below it)."""
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=800 + T)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T >= layer.f16_min_tokens, min_identical=1.0)


def _chain_cases(n=12, seed=77):
    rng = np.random.default_rng(seed)
    cases = []
    for _ in range(n):
        H = int(rng.choice([256, 512, 1056, 2048, 4096]))
        E = int(rng.choice([8, 16, 64, 256]))
        K = int(min(E, rng.choice([2, 4, 8])))
        F = int(rng.choice([64, 96, 256, 512]))
        T = int(rng.choice([1, 7, 16, 17, 64, 200, 600, 1100]))
        cases.append(pytest.param(LayerSpec(H, E, K, F, bool(rng.integers(2)), TYPE_Q4_0), T,
                                  id=f"H{H}-E{E}-k{K}-F{F}-T{T}"))
    return cases


@pytest.mark.parametrize("spec,T", _chain_cases())
def test_forward_norm_chain_random(gpu, spec, T):
    """Seeded random shapes, two chained blocks: with the RMSNorm partial sums carried
    (normalized on the fly at decode and in the batched router, into the workspace
    otherwise) every block equals rms_norm + forward bit for bit, and y's partial
    sums equal the oracle's."""
    from qwenium_amd import Workspace, rms_norm, ssq_parts

    x = synthetic.make_x(spec, T, 80 + T, batch=1)
    x_ssq = None
    ws = None
    for l in range(2):
        layer = synthetic.make_layer(spec, 80 + T, layer=l)
        if ws is None:
            ws = Workspace(layer, T)
        wn = synthetic.make_norm_weight(spec, 80 + T, l)
        y_ssq = torch.empty((T, ssq_parts(spec.n_embd)), dtype=torch.float64, device=x.device)
        y = layer.forward_norm(x, wn, synthetic.NORM_EPS, workspace=ws, x_ssq=x_ssq, y_ssq=y_ssq)
        y_ref = layer.forward(rms_norm(x, wn, synthetic.NORM_EPS), residual=x, workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(y, y_ref), f"block {l}"
        np.testing.assert_array_equal(y_ssq.cpu().numpy(), po.rms_partials(y.cpu().numpy()), err_msg=f"block {l}")
        x, x_ssq = y, y_ssq
    assert ws.check() == 0


@pytest.mark.parametrize("T", [300, 720, 800])
def test_1024_experts_prefill(gpu, monkeypatch, T):
    """1024 experts (the most a layer takes): the f64-MFMA router with the int8 GEMMs (300
    tokens), the f16-MFMA GEMMs (held at 704 tokens here, below the shape's own 2816) with
    the f64-MFMA router (720) and with the batched router (800 tokens; its threshold held at
    784, so that both routers meet the f16 GEMMs), sixteen 64-expert router tiles and the
    per-expert lists."""
    monkeypatch.setenv("QMOE_BIG_ROUTER_MIN_TOKENS", "784")
    monkeypatch.setenv("QMOE_MFMA_MIN_TOKENS", "704")
    spec = LayerSpec(256, 1024, 8, 64, True, TYPE_Q4_0)
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=600 + T)
    assert_parity(y, got, y_ref, d_ref, spec, mfma=T >= 704, min_identical=1.0)
    if T >= 784:
        check_router_bound(got, d_ref["logits"])
    else:
        assert not np.isfinite(got["router_approx"]).any()


@pytest.mark.parametrize("which,T", [("35b", 1), ("35b", 10), ("35b", 16), ("35b", 17), ("35b", 300),
                                     ("35b", 1024), ("config1", 5), ("config1", 300), ("h4096", 10), ("h4096", 300),
                                     ("h4096", 1100), ("pad", 10), ("pad", 300)])
def test_forward_norm_chain(gpu, which, T):
    """Three blocks with the RMSNorm partial sums carried from each to the next
    (x_ssq in, y_ssq out; the first block without x_ssq): every block's y has the
    bits of forward_norm without them, and y_ssq equals the oracle's partial sums
    of y (written by the down+combine epilogue at decode sizes, by one more
    launch otherwise)."""
    from qwenium_amd import Workspace, ssq_parts

    spec = {"35b": synthetic.QWEN35B, "config1": synthetic.CONFIG1,
            "h4096": synthetic.LayerSpec(4096, 16, 2, 64, True, synthetic.TYPE_Q4_0),
            "pad": synthetic.LayerSpec(96, 8, 2, 32, True, synthetic.TYPE_Q4_0)}[which]
    seed = 23
    x = synthetic.make_x(spec, T, seed, batch=T)
    x_ssq = None
    ws = None
    for l in range(3):
        layer = synthetic.make_layer(spec, seed, layer=l)
        if ws is None:
            ws = Workspace(layer, T)
        wn = synthetic.make_norm_weight(spec, seed, l)
        y_ssq = torch.empty((T, ssq_parts(spec.n_embd)), dtype=torch.float64, device=x.device)
        y = layer.forward_norm(x, wn, synthetic.NORM_EPS, workspace=ws, x_ssq=x_ssq, y_ssq=y_ssq)
        y_ref = layer.forward_norm(x, wn, synthetic.NORM_EPS, workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(y, y_ref), f"block {l}"
        np.testing.assert_array_equal(y_ssq.cpu().numpy(), po.rms_partials(y.cpu().numpy()), err_msg=f"block {l}")
        x, x_ssq = y, y_ssq
    assert ws.check() == 0


@pytest.mark.parametrize("which,T", [("35b", 1), ("35b", 10), ("35b", 16), ("35b", 17), ("35b", 64), ("35b", 100),
                                     ("35b", 300), ("35b", 1024), ("config1", 5), ("config1", 32), ("config1", 300),
                                     ("h4096", 10), ("h4096", 300), ("pad", 10), ("pad", 130), ("pad", 300)])
def test_forward_norm_matches_unfused(gpu, which, T):
    """y = x + MoE(RMSNorm(x) * w) in one call (the decode routing normalizes while it
    stages x, the batched router's preparation and refinement normalize from its
    threshold on (720 tokens), other sizes normalize into the workspace) gives the bits of rms_norm
    followed by forward(residual=x)."""
    from qwenium_amd import Workspace, rms_norm

    spec = {"35b": synthetic.QWEN35B, "config1": synthetic.CONFIG1,
            "h4096": synthetic.LayerSpec(4096, 16, 2, 64, True, synthetic.TYPE_Q4_0),
            "pad": synthetic.LayerSpec(96, 8, 2, 32, True, synthetic.TYPE_Q4_0)}[which]
    seed = 21
    layer = synthetic.make_layer(spec, seed)
    ws = Workspace(layer, T)
    x = synthetic.make_x(spec, T, seed, batch=T)
    wn = synthetic.make_norm_weight(spec, seed, 0)
    y_fused = layer.forward_norm(x, wn, synthetic.NORM_EPS, workspace=ws)
    y_ref = layer.forward(rms_norm(x, wn, synthetic.NORM_EPS), residual=x, workspace=ws)
    torch.cuda.synchronize()
    assert ws.check() == 0
    assert torch.equal(y_fused, y_ref)


def test_decode_forwards_queued_back_to_back(gpu):
    """Decode forwards queued on one workspace with nothing between them (no
    synchronisation, no check): the routing launches carry no state from one forward
    to the next, so every forward's routing and output match the oracle, and
    Workspace.check() reports no fault."""
    from qwenium_amd import Workspace

    spec = synthetic.QWEN35B
    T, seed = 10, 5
    tensors = synthetic.make_layer_tensors(spec, seed)
    layer = synthetic.make_layer(spec, seed, tensors=tensors)
    ref = host_layer(spec, tensors)
    ws = Workspace(layer, 16)
    xs = [synthetic.make_x(spec, T, seed, batch=b) for b in range(4)]
    outs = [layer.forward(x, workspace=ws, debug=True) for x in xs]
    torch.cuda.synchronize()
    for x, (y, dbg) in zip(xs, outs):
        y_ref, d_ref = ref.forward(x.cpu().numpy(), debug=True)
        assert_parity(y.cpu().numpy(), {k: v.cpu().numpy() for k, v in dbg.items()}, y_ref, d_ref, spec,
                      min_identical=1.0)
    assert ws.check() == 0


def test_python_checks_on_device_operands(gpu):
    """out, residual and the norm weights are checked before any launch (a short or
    strided out would make the kernels write past it)."""
    from qwenium_amd import Workspace

    spec = synthetic.CONFIG1
    layer = synthetic.make_layer(spec, 3)
    x = synthetic.make_x(spec, 4, 3)
    H = spec.n_embd
    for bad in (torch.empty(3, H, device=gpu), torch.empty(H, 4, device=gpu).t(),
                torch.empty(4, H, dtype=torch.float16, device=gpu), torch.empty(4, H)):
        with pytest.raises(ValueError, match="out expected"):
            layer.forward(x, out=bad)
    with pytest.raises(ValueError, match="residual expected"):
        layer.forward(x, residual=torch.empty(4, H - 32, device=gpu))
    with pytest.raises(ValueError, match="norm_weight expected"):
        layer.forward_norm(x, torch.ones(H - 1, device=gpu), 1e-6)
    with pytest.raises(ValueError, match="distinct"):
        layer.forward(x, out=x)
    # a strided residual is copied on the launch stream; an explicit stream works end to end
    ws = Workspace(layer, 4)
    s = torch.cuda.Stream()
    res = torch.randn(H, 4, device=gpu).t()
    want = layer.forward(x, residual=res.contiguous(), workspace=ws)
    torch.cuda.synchronize()
    got = layer.forward(x, residual=res, workspace=ws, stream=s)
    s.synchronize()
    assert torch.equal(got, want)


# ---- int8-MFMA expert GEMMs (17 tokens to the f16 path) ------------------------------------
@pytest.mark.parametrize("wtype", [TYPE_Q4_0, TYPE_Q8_0])
@pytest.mark.parametrize("hidden,ffn", [(256, 64), (512, 192), (768, 704), (1280, 576)])
@pytest.mark.parametrize("experts,top_k,T", [
    # all rows on one expert: 32-row tiles whose last group of four rows is full or holds one row
    (1, 1, 17), (1, 1, 20), (1, 1, 21), (1, 1, 24), (1, 1, 25), (1, 1, 28), (1, 1, 29), (1, 1, 31), (1, 1, 32),
    (1, 1, 33), (1, 1, 129),
    (16, 2, 17), (16, 2, 40), (16, 2, 112), (16, 2, 113),  # 1 to ~20 rows, both tile heights (from 14 rows)
    (64, 4, 40), (64, 4, 300),                             # grids past the CUs at ffn 576 and 704
    (96, 6, 128), (96, 6, 129),                            # at ffn 704 32-row tiles from 8 rows in Q4_0
])
def test_i8_experts_tile_edges(gpu, monkeypatch, wtype, hidden, ffn, experts, top_k, T):
    """Tiles of 16 and 32 rows at both ends of every group of four, reduction lengths that end
    in a partial chunk (Q4_0 chunks of 8 block pairs, Q8_0 of 4: 1 to 20 pairs here), ffn widths
    of odd column groups, and gate/up workgroups that are whole or split in two or four parts
    (of equal and unequal numbers of chunks): routing bit-exact, h quants and outputs
    bit-identical to the oracle's (the sums are exact in f64 on both sides)."""
    monkeypatch.setenv("QMOE_MFMA_MIN_TOKENS", "100000")
    spec = LayerSpec(hidden, experts, top_k, ffn, True, wtype)
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=300 + T + hidden)
    assert_parity(y, got, y_ref, d_ref, spec, min_identical=1.0)


class Strided(synthetic.GGMLTensor):
    """Rows of a wider 2-d byte tensor."""

    def desc(self):
        d = super().desc()
        d.nb[1] = self.data.shape[1]
        d.nb[2] = d.nb[1] * self.ne[1]
        return d


def test_row_strides_beyond_32_bits(gpu):
    """Gate rows 300 MB apart: 15 rows reach past 2^32 bytes.  Decode, the int8 GEMMs and the
    f16 GEMMs give the packed layer's bits."""
    spec = LayerSpec(256, 1, 1, 64, False, TYPE_Q4_0)
    tensors = synthetic.make_layer_tensors(spec, 12)
    rows = tensors["gate"].data.view(64, -1)
    buf = torch.empty((64, 300_000_000), dtype=torch.uint8, device=rows.device)
    buf[:, :rows.shape[1]] = rows
    wide = dict(tensors, gate=Strided(buf, tensors["gate"].type, tensors["gate"].ne))
    packed, strided = (synthetic.make_layer(spec, 12, tensors=t, prefill_copies=False) for t in (tensors, wide))
    for T in (1, 17, 200):
        x = synthetic.make_x(spec, T, 12)
        assert torch.equal(packed.forward(x), strided.forward(x)), f"{T} tokens"
    del wide, strided, buf
    torch.cuda.empty_cache()


def test_i8_experts_gate_up_strides(gpu):
    """Gate and up rows of different strides (views into wider rows): the int8 GEMM's two
    column bases; equal to the packed layer's results bit for bit."""
    spec = LayerSpec(512, 8, 2, 128, False, TYPE_Q4_0)
    tensors = synthetic.make_layer_tensors(spec, 11)
    x = synthetic.make_x(spec, 50, 11)
    y = synthetic.make_layer(spec, 11, tensors=tensors).forward(x)
    wide = dict(tensors)
    for name, pad in (("gate", 36), ("up", 92)):
        t = tensors[name]
        rows = t.data.view(8 * 128, -1)
        buf = torch.full((rows.shape[0], rows.shape[1] + pad), 0x7f, dtype=torch.uint8, device=rows.device)
        buf[:, :rows.shape[1]] = rows
        wide[name] = Strided(buf, t.type, t.ne)
    y2 = synthetic.make_layer(spec, 11, tensors=wide, prefill_copies=False).forward(x)
    torch.cuda.synchronize()
    assert torch.equal(y, y2)


@pytest.mark.parametrize("H", [4, 32, 100, 256, 260, 2048, 2816, 4092, 4096])
def test_norm_rows_aligned_equals_general(gpu, H):
    """The one-pass RMSNorm and Gemma 4 input kernel of 16-byte aligned rows against the general
    one (the same rows at an odd float offset): equal bits, at one thread, whole and partial
    waves, and the widest row."""
    from qwenium_amd import gemma4_moe_inputs, rms_norm

    T = 3
    x, w, w2 = (torch.randn(n, dtype=torch.float32, device="cuda") for n in (T * H, H, H))

    def odd(v):
        return torch.cat([v.new_zeros(1), v])[1:]

    assert odd(x).data_ptr() % 16 == 4
    y = rms_norm(x.view(T, H), w, 1e-6)
    assert torch.equal(y, rms_norm(odd(x).view(T, H), odd(w), 1e-6))
    assert torch.equal(rms_norm(x.view(T, H), None, 1e-6), rms_norm(odd(x).view(T, H), None, 1e-6))
    a = gemma4_moe_inputs(x.view(T, H), w, w2, 1e-6)
    b = gemma4_moe_inputs(odd(x).view(T, H), odd(w), odd(w2), 1e-6)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and torch.equal(a[0], y)


@pytest.mark.parametrize("hidden,experts,T", [(256, 1, 17), (256, 15, 31), (512, 16, 32), (2304, 17, 33), (4096, 40, 47),
                                              (1024, 300, 65)])
def test_group_router_tile_edges(gpu, hidden, experts, T):
    """The f64-MFMA router (17 tokens to the batched router): tiles of 16 tokens x 16 router rows
    with every kind of remainder (the shared gate as a row of its own past 16 or 32), one to
    sixteen 16-column steps per wave, 9 among them (a second batch of loads with one step):
    logits within one ulp of the oracle's correctly rounded ones, routing and outputs equal."""
    spec = LayerSpec(hidden, experts, min(2, experts), 64, True, TYPE_Q8_0)
    y, got, y_ref, d_ref, *_ = run_pair(spec, T, seed=500 + T)
    assert_parity(y, got, y_ref, d_ref, spec, min_identical=1.0)


@pytest.mark.parametrize("hidden,experts,T", [(1024, 7, 17), (1024, 8, 64), (2048, 31, 33), (2816, 6, 200), (3840, 30, 255),
                                              (4096, 64, 112), (4096, 64, 113)])
def test_row_pair_router_groups(gpu, hidden, experts, T):
    """17 tokens and more where the router's blocks of two rows over groups of 16 tokens fit the
    CUs once: one to four slabs per wave (fewer in the last waves), an odd last row, whole and
    partial groups, the fewest blocks per group (four: each quantizes up to four tokens), and the
    most blocks before the f64-MFMA tiles take over (33 x 7 against 33 x 8): logits within one
    ulp of the oracle's, routing and outputs equal."""
    spec = LayerSpec(hidden, experts, min(2, experts), 64, True, TYPE_Q8_0)
    y, got, y_ref, d_ref, layer, *_ = run_pair(spec, T, seed=600 + T)
    assert_parity(y, got, y_ref, d_ref, spec, min_identical=1.0, mfma=T >= layer.f16_min_tokens)
