"""GPU parity for the MoE FFN: batch-1 decode (config 1), the device grouped
schedule (bit-exact), the grouped prefill (config 2) and small edge cases."""

import os

import numpy as np
import pytest
import torch

import oracle
from tests.helpers import assert_parity, f16_to_f32, moe_to_oracle

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


@pytest.fixture(scope="module")
def layer_full(pkg, dev):
    """Config 1/2 layer: H=2048, 256 routed experts, I=512, shared I=512, group 128."""
    layer = pkg.synth.moe_layer(hidden=2048, inter=512, experts=256, seed=1, device=dev)
    return layer, moe_to_oracle(layer)


@pytest.fixture(scope="module")
def layer_small(pkg, dev):
    layer = pkg.synth.moe_layer(hidden=512, inter=128, experts=16, seed=21, device=dev)
    return layer, moe_to_oracle(layer)


def _decode(pkg, dev, layer, mw, seed, residual=True, k=8):
    H, E = layer.hidden, layer.experts
    x = pkg.synth.activations(1, H, seed, dev)[0]
    logits = pkg.synth.router_logits(1, E, seed + 1, dev)
    ids, w = pkg.select_router_topk(logits, k)
    res = pkg.synth.activations(1, H, seed + 2, dev)[0] if residual else None
    out = pkg.run_moe_ffn_layer(layer, x, ids[0].contiguous(), w[0].contiguous(), residual=res)
    torch.cuda.synchronize()
    ref = oracle.moe_ffn_tokens(mw, f16_to_f32(x)[None], ids.cpu().numpy(), w.cpu().numpy(),
                                residual=None if res is None else f16_to_f32(res)[None],
                                threads=1)
    return f16_to_f32(out), ref[0]


def test_config1_decode(pkg, dev, layer_full):
    layer, mw = layer_full
    for seed in (0, 10, 20):
        got, ref = _decode(pkg, dev, layer, mw, seed)
        assert_parity(got, ref, what=f"config1 seed={seed}")


def test_decode_without_residual(pkg, dev, layer_full):
    layer, mw = layer_full
    got, ref = _decode(pkg, dev, layer, mw, 5, residual=False)
    assert_parity(got, ref, what="no residual")


@pytest.mark.parametrize("k", [1, 4, 8, 16])
def test_decode_small_topk(pkg, dev, layer_small, k):
    layer, mw = layer_small
    got, ref = _decode(pkg, dev, layer, mw, 30 + k, k=k)
    assert_parity(got, ref, what=f"small k={k}")


@pytest.mark.parametrize("k", [23, 24, 40])
def test_decode_wide_topk(pkg, dev, k):
    """k + 1 > 24 slots: the down phase takes its slots in several batches."""
    layer = pkg.synth.moe_layer(hidden=512, inter=128, experts=40, seed=23, device=dev)
    g = np.random.default_rng(50 + k)
    ids = g.permutation(40)[:k].astype(np.int32)[None]  # router top-k stops at 16
    w = g.random(k).astype(np.float32)
    w = (w / w.sum())[None]
    x = pkg.synth.activations(1, 512, 51 + k, dev)[0]
    res = pkg.synth.activations(1, 512, 52 + k, dev)[0]
    out = pkg.run_moe_ffn_layer(layer, x, torch.from_numpy(ids[0]).to(dev),
                                torch.from_numpy(w[0]).to(dev), residual=res)
    torch.cuda.synchronize()
    ref = oracle.moe_ffn_tokens(moe_to_oracle(layer), f16_to_f32(x)[None], ids, w,
                                residual=f16_to_f32(res)[None], threads=1)
    assert_parity(f16_to_f32(out), ref[0], what=f"wide k={k}")


def test_decode_flags_bad_expert_id(pkg, dev, layer_small):
    layer, _ = layer_small
    ws = pkg.Workspace(dev)
    x = pkg.synth.activations(1, layer.hidden, 1, dev)[0]
    ids = torch.tensor([0, 1, 2, 3, 4, 5, 6, 99], dtype=torch.int32, device=dev)
    w = torch.full((8,), 0.125, device=dev)
    out = pkg.run_moe_ffn_layer(layer, x, ids, w, ws=ws)
    torch.cuda.synchronize()
    assert ws.error_bits() & pkg._lib.AIMA_DEVERR_EXPERT_RANGE
    assert torch.isfinite(out.float()).all()
    assert ws.error_bits() == 0  # reading clears the word


# ---------------------------------------------------------------------------
# grouped schedule
# ---------------------------------------------------------------------------

# (1024, 1024, 16): the largest expert count and k, 16 chunks of 1024
# assignments; (2049, 256, 8): a partial last chunk of 8 assignments.
@pytest.mark.parametrize("T,E,k,zipf", [(2048, 256, 8, 1.1), (1, 256, 8, None),
                                        (37, 16, 8, None), (1000, 64, 6, None),
                                        (16384, 256, 8, None), (2049, 256, 8, 1.1),
                                        (1024, 1024, 16, 1.1), (1025, 1024, 16, None),
                                        (3, 1024, 16, None)])
def test_schedule_bit_exact(pkg, dev, T, E, k, zipf):
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(T, E, seed=T, device=dev,
                                                            zipf_s=zipf), k)
    s = pkg.build_grouped_schedule(ids, w, E)
    torch.cuda.synchronize()
    r = oracle.build_grouped_schedule(ids.cpu().numpy(), E, w.cpu().numpy())
    for name in ("offsets", "token_map", "inverse_map", "compact_weights"):
        assert np.array_equal(s[name].cpu().numpy(), r[name]), name


def test_schedule_flags_errors(pkg, dev):
    ws = pkg.Workspace(dev)
    ids = torch.tensor([[0, 1, 2, 3], [4, 5, 6, 4]], dtype=torch.int32, device=dev)
    w = torch.ones((2, 4), device=dev)
    pkg.build_grouped_schedule(ids, w, 8, ws=ws)
    assert ws.error_bits() == pkg._lib.AIMA_DEVERR_EXPERT_DUPLICATE
    ids = torch.tensor([[0, 1, 2, 8]], dtype=torch.int32, device=dev)
    pkg.build_grouped_schedule(ids, torch.ones((1, 4), device=dev), 8, ws=ws)
    assert ws.error_bits() & pkg._lib.AIMA_DEVERR_EXPERT_RANGE


@pytest.mark.parametrize("T", [200, 3000])
def test_schedule_flags_duplicate_across_chunks(pkg, dev, T):
    """At k = 6, token 170 holds assignments 1020..1025, across the boundary of
    the 1024-assignment blocks of the schedule.  A duplicate between its rank
    0 and rank 5 (in different blocks) is flagged, with 2 blocks (T = 200) and
    18 (T = 3000); a clean routing flags nothing and ranks as the oracle."""
    ws = pkg.Workspace(dev)
    g = torch.Generator(device="cpu")
    g.manual_seed(T)
    ids = torch.stack([torch.randperm(64, generator=g)[:6] for _ in range(T)]).to(torch.int32)
    ids = ids.to(dev)
    w = torch.ones((T, 6), device=dev)
    s = pkg.build_grouped_schedule(ids, w, 64, ws=ws)
    torch.cuda.synchronize()
    assert ws.error_bits() == 0
    r = oracle.build_grouped_schedule(ids.cpu().numpy(), 64, w.cpu().numpy())
    assert np.array_equal(s["token_map"].cpu().numpy(), r["token_map"])
    bad = ids.clone()
    bad[170, 5] = bad[170, 0]
    pkg.build_grouped_schedule(bad, w, 64, ws=ws)
    assert ws.error_bits() == pkg._lib.AIMA_DEVERR_EXPERT_DUPLICATE


# ---------------------------------------------------------------------------
# grouped prefill
# ---------------------------------------------------------------------------

def _prefill(pkg, dev, layer, mw, T, seed, zipf=None, residual=False, k=8, tokens=None):
    H, E = layer.hidden, layer.experts
    x = pkg.synth.activations(T, H, seed, dev)
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(T, E, seed + 1, dev, zipf_s=zipf), k)
    res = pkg.synth.activations(T, H, seed + 2, dev) if residual else None
    out = pkg.grouped_moe_prefill(layer, x, ids, w, residual=res)
    torch.cuda.synchronize()
    sel = np.arange(T) if tokens is None else np.asarray(tokens)
    ref = oracle.moe_ffn_tokens(mw, f16_to_f32(x)[sel], ids.cpu().numpy()[sel],
                                w.cpu().numpy()[sel],
                                residual=None if res is None else f16_to_f32(res)[sel],
                                threads=THREADS)
    return f16_to_f32(out)[sel], ref


def test_config2_prefill(pkg, dev, layer_full):
    """T=2048, Zipf(1.1)-skewed routing, every token against the oracle."""
    layer, mw = layer_full
    got, ref = _prefill(pkg, dev, layer, mw, 2048, seed=2, zipf=1.1)
    assert_parity(got, ref, what="config2")


def test_prefill_uniform_routing_residual(pkg, dev, layer_full):
    layer, mw = layer_full
    got, ref = _prefill(pkg, dev, layer, mw, 512, seed=40, residual=True)
    assert_parity(got, ref, what="uniform+residual")


@pytest.mark.parametrize("T", [1, 2, 37, 129, 300])
def test_prefill_ragged(pkg, dev, layer_small, T):
    layer, mw = layer_small
    got, ref = _prefill(pkg, dev, layer, mw, T, seed=T, residual=(T % 2 == 1))
    assert_parity(got, ref, what=f"ragged T={T}")


def test_prefill_all_tokens_same_experts(pkg, dev, layer_small):
    """Every token routes to experts 0..7: a few maximal groups, most empty."""
    layer, mw = layer_small
    T = 333
    x = pkg.synth.activations(T, layer.hidden, 9, dev)
    ids = torch.arange(8, dtype=torch.int32, device=dev).repeat(T, 1).contiguous()
    w = torch.full((T, 8), 0.125, device=dev)
    out = pkg.grouped_moe_prefill(layer, x, ids, w)
    torch.cuda.synchronize()
    ref = oracle.moe_ffn_tokens(mw, f16_to_f32(x), ids.cpu().numpy(), w.cpu().numpy(),
                                threads=THREADS)
    assert_parity(f16_to_f32(out), ref, what="same experts")


def test_prefill_matches_decode(pkg, dev, layer_small):
    """One token through the grouped path equals the decode path's result."""
    layer, _ = layer_small
    x = pkg.synth.activations(1, layer.hidden, 77, dev)
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(1, 16, 78, dev), 8)
    a = pkg.grouped_moe_prefill(layer, x, ids, w)[0]
    b = pkg.run_moe_ffn_layer(layer, x[0], ids[0].contiguous(), w[0].contiguous())
    torch.cuda.synchronize()
    assert_parity(f16_to_f32(a), f16_to_f32(b), tol=2e-3, what="prefill vs decode")


def test_prefill_runtime_contract(pkg, dev, layer_small):
    layer, mw = layer_small
    rt = pkg.GroupedU4PrefillRuntime(dev)
    h = rt.LoadLayer(layer)
    T = 200
    x = pkg.synth.activations(T, layer.hidden, 5, dev)
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(T, 16, 6, dev), 8)
    run = rt.RunLayer(h, pkg.GroupedU4PrefillInput(x, ids, w, warmup=1, repeat=3,
                                                   capture_intermediates=True,
                                                   include_shared=True))
    assert len(run.timing.samples_us) == 3 and run.timing.minimum_us > 0
    assert run.active_experts > 0 and run.max_group_size > 0
    ref = oracle.moe_ffn_tokens(mw, f16_to_f32(x), ids.cpu().numpy(), w.cpu().numpy(),
                                threads=THREADS)
    assert_parity(f16_to_f32(run.output), ref, what="runtime")
    st = rt.stats()
    assert st["run_count"] == 1 and st["layer_count"] == 1
    with pytest.raises(KeyError):
        rt.RunLayer(99, pkg.GroupedU4PrefillInput(x, ids, w, include_shared=True))


def test_decode_phases_compose(pkg, dev, layer_full):
    """gate_up then down == the one-call decode (same kernels, same order)."""
    layer, _ = layer_full
    x = pkg.synth.activations(1, 2048, 91, dev)[0]
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(1, 256, 92, dev), 8)
    ids, w = ids[0].contiguous(), w[0].contiguous()
    res = pkg.synth.activations(1, 2048, 93, dev)[0]
    act, sigma = pkg.moe_decode_gate_up(layer, x, ids)
    a = pkg.moe_decode_down(layer, act, sigma, ids, w, residual=res)
    b = pkg.run_moe_ffn_layer(layer, x, ids, w, residual=res)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    # the activations themselves against the oracle's SwiGLU (f32 -> f16 rounding)
    mw = moe_to_oracle(layer)
    d = oracle.moe_ffn_token_detail(mw, f16_to_f32(x), None, ids.cpu().numpy(),
                                    w.cpu().numpy())
    ref_act = np.concatenate([d["selected_swiglu"], d["shared_swiglu"]]).reshape(9, 512)
    assert_parity(f16_to_f32(act), ref_act, what="decode SwiGLU activations")
    assert abs(float(sigma.item()) - float(d["shared_gate"][1])) < 1e-5


def test_prefill_largest_batch(pkg, dev, layer_full):
    """T = 233016, the largest batch whose row offsets stay below 2^31 bytes
    (tokens * (k + 1) * inter < 2^30 f16 elements at k = 8, inter = 512):
    every token finite, sampled tokens against the oracle."""
    layer, mw = layer_full
    T = 233016
    x = pkg.synth.activations(T, 2048, 77, dev)
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(T, 256, 78, dev), 8)
    out = pkg.grouped_moe_prefill(layer, x, ids, w)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    sel = torch.tensor([0, 1, 116508, T - 2, T - 1], device=dev)
    got = f16_to_f32(out[sel])
    ref = oracle.moe_ffn_tokens(mw, f16_to_f32(x[sel]), ids[sel].cpu().numpy(),
                                w[sel].cpu().numpy(), threads=THREADS)
    assert_parity(got, ref, what="largest batch")
    del out, x


def _off_alignment(layer):
    """Moves scales and zero points one element off their vector alignment."""
    def off(t):
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        flat[1:] = t.reshape(-1)
        return flat[1:].reshape(t.shape)

    for w in (layer.gate_up, layer.down, layer.shared_gate_up, layer.shared_down):
        w.scale, w.zp = off(w.scale), off(w.zp)


@pytest.mark.parametrize("H,I", [(512, 512), (512, 128), (768, 384)])
@pytest.mark.parametrize("experts", [96, 16])
@pytest.mark.parametrize("shift", [0, 1])
def test_prefill_thin_tiles(pkg, dev, H, I, experts, shift):
    """Tiles at the edges of the thin-tile path (1, 15, 16, 17, 31, 32 rows),
    one row above it (33) and a full tile with a one-row remainder, in 16-row
    tiles (96 experts: at most 10 rows per expert) and 256-row ones (16).  K of
    1, 3, 4 and 6 quantization groups, and scales and zero points off their
    vector alignment (shift), cover both ways of loading them.  f16 operands
    and intermediates: 2e-3, as the other prefill tests."""
    layer = pkg.synth.moe_layer(hidden=H, inter=I, experts=experts, seed=300 + H + I, device=dev)
    mw = moe_to_oracle(layer)
    if shift:
        _off_alignment(layer)
    counts = [1, 15, 16, 17, 31, 32, 33] if experts == 96 else [1, 15, 16, 17, 31, 32, 33, 257]
    ids = np.repeat(np.arange(len(counts)) * (experts // len(counts)), counts).astype(np.int32)
    ids = np.random.default_rng(H + I).permutation(ids)[:, None].copy()
    T = len(ids)
    assert (T <= 10 * experts) == (experts == 96)
    x = pkg.synth.activations(T, H, 301, dev)
    w = torch.ones((T, 1), device=dev)
    out = pkg.grouped_moe_prefill(layer, x, torch.from_numpy(ids).to(dev), w)
    torch.cuda.synchronize()
    ref = oracle.moe_ffn_tokens(mw, f16_to_f32(x), ids, w.cpu().numpy(), threads=THREADS)
    assert_parity(f16_to_f32(out), ref, what=f"thin tiles H={H} I={I} E={experts}")


@pytest.mark.parametrize("H,I", [(1024, 256), (2048, 768)])
def test_prefill_thin_tiles_unbiased(pkg, dev, H, I):
    """A thin tile's result is off by roundings, not to one side: an offset
    common to all outputs passes through the next layers' weights (whose mean
    is not zero) enlarged.  The outputs' errors are roundings of the f16
    intermediates, below 2^-11 of the output's size and independent, so their
    mean over n outputs lies within 6 * 2^-11 / sqrt(n) of zero (1.7e-5 and
    1.2e-5 of the outputs' size)."""
    layer = pkg.synth.moe_layer(hidden=H, inter=I, experts=60, seed=320 + H, device=dev)
    T, k = 30, 2
    x = pkg.synth.activations(T, H, 321, dev).float()
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(T, 60, 322, dev), k)
    out = pkg.grouped_moe_prefill_routed(layer, x, ids, w, expert_used_count=k)
    torch.cuda.synchronize()
    ref = oracle.moe_routed_tokens(moe_to_oracle(layer), x.cpu().numpy(), ids.cpu().numpy(),
                                   w.cpu().numpy(), threads=THREADS).astype(np.float64)
    off = (out.cpu().numpy() - ref).mean() / np.sqrt((ref ** 2).mean())
    assert abs(off) <= 6 * 2.0 ** -11 / np.sqrt(ref.size)


@pytest.mark.parametrize("H,reps,more", [(2048, 4, 700), (2304, 4, 100), (768, 6, 1300)])
@pytest.mark.parametrize("capture,shift", [(False, 0), (False, 1), (True, 0)])
def test_prefill_resident_down_rows(pkg, dev, H, reps, more, capture, shift):
    """The down GEMM that keeps a tile's token rows in LDS (inter 512, over 32
    assignments per expert, at least 384 blocks at hidden 1536 and more):
    remainders around each 32-row block of both 128-row halves, thin halves, and
    a column count that leaves waves of a block without a chunk (2304); the same
    at hidden 768, where the rows are not kept.  Scales and zero points off
    their vector alignment (shift) take the instance that loads them value by
    value.  With the f32 copies requested, the f16 contributions are those values
    rounded.  Tolerance as the other prefill tests."""
    I = 512
    counts = [1, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 256, 289] * reps + [more]
    layer = pkg.synth.moe_layer(hidden=H, inter=I, experts=len(counts), seed=400 + H, device=dev)
    mw = moe_to_oracle(layer)
    ids = np.repeat(np.arange(len(counts)), counts).astype(np.int32)
    ids = np.random.default_rng(H + I).permutation(ids)[:, None].copy()
    T = len(ids)
    assert T > 32 * len(counts) and -(-2 * T // 128) * -(-H // 512) >= 320
    assert pkg.prefill_tiling(layer, T, 1)[2] == (128 if H >= 1536 else 256)
    if shift:
        _off_alignment(layer)
    x = pkg.synth.activations(T, H, 401, dev)
    w = torch.rand((T, 1), device=dev) + 0.5
    d_ids = torch.from_numpy(ids).to(dev)
    if capture:
        ws, cap = pkg.Workspace(dev), {}
        out = pkg.grouped_moe_prefill_routed(layer, x, d_ids, w, expert_used_count=1, ws=ws,
                                             capture_f32=cap)
        ref = oracle.moe_routed_tokens(mw, f16_to_f32(x), ids, w.cpu().numpy(), threads=THREADS)
        got = out.cpu().numpy()
        rows = pkg.prefill_workspace_views(layer, T, 1, ws, with_shared=False)
        assert torch.equal(rows["contributions"], cap["contributions_f32"].half())
        assert torch.equal(rows["swiglu"], cap["swiglu_f32"].half())
    else:
        out = pkg.grouped_moe_prefill(layer, x, d_ids, w)
        ref = oracle.moe_ffn_tokens(mw, f16_to_f32(x), ids, w.cpu().numpy(), threads=THREADS)
        got = f16_to_f32(out)
    torch.cuda.synchronize()
    assert_parity(got, ref, what=f"resident down rows H={H} I={I}")


@pytest.mark.parametrize("H,I", [(512, 256), (768, 384)])
def test_prefill_capture_tall_tiles(pkg, dev, H, I):
    """The f32 copies of tiles over 32 rows (every height in 32-row blocks, full
    tiles, remainders) where the down GEMM does not keep its token rows: near
    the oracle's, and the f16 rows are those values rounded, bit for bit."""
    counts = [33, 64, 65, 97, 130, 161, 200, 256, 290]
    layer = pkg.synth.moe_layer(hidden=H, inter=I, experts=len(counts), seed=450 + H, device=dev)
    mw = moe_to_oracle(layer)
    ids = np.repeat(np.arange(len(counts)), counts).astype(np.int32)
    ids = np.random.default_rng(H).permutation(ids)[:, None].copy()
    T = len(ids)
    assert pkg.prefill_tiling(layer, T, 1, with_shared=False)[::2] == (256, 256)
    x = pkg.synth.activations(T, H, 451, dev)
    w = torch.rand((T, 1), device=dev) + 0.5
    ws, cap = pkg.Workspace(dev), {}
    pkg.grouped_moe_prefill_routed(layer, x, torch.from_numpy(ids).to(dev), w,
                                   expert_used_count=1, ws=ws, capture_f32=cap)
    rows = pkg.prefill_workspace_views(layer, T, 1, ws, with_shared=False)
    assert torch.equal(rows["swiglu"], cap["swiglu_f32"].half())
    assert torch.equal(rows["contributions"], cap["contributions_f32"].half())
    token = rows["token_map"].long().cpu()
    ref = oracle.moe_routed_tokens(mw, f16_to_f32(x), ids, w.cpu().numpy(), threads=THREADS)
    assert_parity(cap["contributions_f32"].cpu().numpy(), ref[token.numpy()], what="contributions")
    for row in range(0, T, 97):
        t = int(token[row])
        d = oracle.moe_ffn_token_detail(mw, f16_to_f32(x[t]), None, ids[t], w[t].cpu().numpy())
        assert_parity(cap["swiglu_f32"][row].cpu().numpy(), d["selected_swiglu"].reshape(-1),
                      what=f"swiglu row {row}")


@pytest.mark.parametrize("T,E,k", [(128, 256, 8), (1025, 8, 1), (147, 1024, 7), (32768, 256, 8),
                                   (32770, 130, 8)])
def test_schedule_launch_forms(pkg, dev, T, E, k):
    """A schedule of one block of assignments (1024, one launch), just past
    it, and around the most blocks whose row bases every block sums itself
    (256; beyond, the scan is a launch of its own).  Integers: exact."""
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(T, E, seed=T + E, device=dev), k)
    s = pkg.build_grouped_schedule(ids, w, E)
    torch.cuda.synchronize()
    r = oracle.build_grouped_schedule(ids.cpu().numpy(), E, w.cpu().numpy())
    for name in ("offsets", "token_map", "inverse_map", "compact_weights"):
        assert np.array_equal(s[name].cpu().numpy(), r[name]), name


@pytest.mark.parametrize("E,k", [(5, 5), (64, 16), (65, 3), (256, 8), (256, 16), (1000, 16)])
def test_router_selection_ties(pkg, dev, E, k):
    """Equal probabilities across lanes, within a lane (ids 64 apart) and
    everywhere, and fewer finite logits than picks: ids exact, lowest first."""
    g = np.random.default_rng(E + k)
    rows = [np.zeros(E), np.round(g.normal(size=E)), g.normal(size=E),
            np.tile(g.normal(size=64), -(-E // 64))[:E], np.full(E, -np.inf)]
    rows[4][g.permutation(E)[:max(1, k // 2)]] = 1.0
    logits = np.stack(rows).astype(np.float32)
    ids, w = pkg.select_router_topk(torch.from_numpy(logits).to(dev), k)
    torch.cuda.synchronize()
    ref_ids, ref_w = oracle.router_topk_tokens(logits, k)
    assert np.array_equal(ids.cpu().numpy(), ref_ids)
    assert_parity(w.cpu().numpy(), ref_w, tol=1e-6, what="router weights")


@pytest.mark.parametrize("T,H", [(1, 512), (128, 768), (129, 512), (700, 256)])
def test_prefill_f32_input_conversion(pkg, dev, T, H):
    """An f32 input is rounded to f16 by spare blocks of the schedule's first
    launch (one-launch schedules up to 1024 assignments, and above; partial
    last blocks): the bits of the f16 input's run."""
    layer = pkg.synth.moe_layer(hidden=H, inter=128, experts=16, seed=700 + H, device=dev)
    g = torch.Generator(device=dev)
    g.manual_seed(T)
    x = torch.randn((T, H), generator=g, device=dev)
    ids, w = pkg.select_router_topk(pkg.synth.router_logits(T, 16, T, dev), 8)
    a = pkg.grouped_moe_prefill_routed(layer, x, ids, w)
    b = pkg.grouped_moe_prefill_routed(layer, x.half(), ids, w)
    assert torch.equal(a, b)


def _dequant_f64(w):
    q = w.qweight.cpu().numpy().reshape(w.rows, w.k // 2)
    s = w.scale.cpu().view(torch.uint16).numpy().reshape(w.rows, -1)
    z = w.zp.cpu().numpy().reshape(-1)
    return torch.from_numpy(oracle.u4_dequant(q, s, z, w.rows, w.k, w.group)).double()


def _expert_f64(layer, x):
    """SwiGLU and down rows of a one-expert layer in float64, the SwiGLU rows
    rounded to f16 in between."""
    gu = _dequant_f64(layer.gate_up) @ x.double().cpu().T
    g, u = gu[:layer.inter], gu[layer.inter:]
    act = (g * torch.sigmoid(g) * u).T
    return act, act.half().double() @ _dequant_f64(layer.down).T


def _same_class(got, ref):
    """The same elements are +inf, -inf and NaN."""
    return all(torch.equal(f(got.double().cpu()), f(ref))
               for f in (torch.isposinf, torch.isneginf, torch.isnan))


@pytest.mark.parametrize("rows", [5, 12, 20, 40])
@pytest.mark.parametrize("inter", [128, 512])
def test_prefill_infinities(pkg, dev, rows, inter):
    """An infinite activation and a SwiGLU value past f16's range reach the
    result as +-inf or NaN just where (q - z) * s * x gives them, in every
    tile height: 16-row tiles (5), thin tiles of one and two 16-row blocks (12,
    20) and a taller one (40)."""
    layer = pkg.synth.moe_layer(hidden=512, inter=inter, experts=1, seed=60 + rows, device=dev)
    ids = torch.zeros((rows, 1), dtype=torch.int32, device=dev)
    w = torch.ones((rows, 1), device=dev)
    x = pkg.synth.activations(rows, 512, 61, dev)
    x[0, 77] = float("inf")
    x[rows - 1, 300] = -float("inf")
    x[2, 5], x[2, 6] = float("inf"), -float("inf")
    cap = {}
    pkg.grouped_moe_prefill_routed(layer, x, ids, w, expert_used_count=1, capture_f32=cap)
    act, _ = _expert_f64(layer, x)
    assert torch.isinf(act).any() and torch.isfinite(act[1]).all()
    assert _same_class(cap["swiglu_f32"], act)
    # one intermediate column of a few rows past 65504 (x = +-400 against a
    # gate and an up row of ones), positive down weights but for one column
    for t, code in ((layer.gate_up, 0x11), (layer.down, None)):
        t.zp.zero_()
        if code is not None:
            v = t.qweight.view(2 * inter, 256)
            v[7], v[inter + 7] = code, code
            t.scale.view(2 * inter, -1)[7] = 1.0
            t.scale.view(2 * inter, -1)[inter + 7] = 1.0
    d = layer.down.qweight.view(512, inter // 2)
    d[:, 3] = (d[:, 3] & 0x0F) | 0x10   # column 7: code 1, +inf, ...
    d[9, 3] = d[9, 3] & 0x0F            # ... and 0, NaN, in row 9
    x = pkg.synth.activations(rows, 512, 62, dev) * 0.01
    x[1] = 400.0 / 512
    x[rows - 1] = 400.0 / 512
    out = pkg.grouped_moe_prefill_routed(layer, x, ids, w, expert_used_count=1)
    act, ref = _expert_f64(layer, x)
    assert torch.isposinf(act.half()[1, 7]) and torch.isfinite(act.half()[0]).all()
    assert torch.isposinf(ref[1, 0]) and torch.isnan(ref[1, 9])
    assert _same_class(out, ref)
    fin = torch.isfinite(ref)
    assert_parity(out.cpu()[fin].numpy(), ref[fin].numpy(), what=f"finite rows of {rows}")


@pytest.mark.parametrize("rows", [12, 20, 40])
@pytest.mark.parametrize("factor", [2.0 ** 4, 2.0 ** 8, 2.0 ** 12])
def test_prefill_outlier_channels(pkg, dev, rows, factor):
    """A few channels 2^4 to 2^12 times the rest cost no precision: an output
    passes through at most four independent f16 roundings (the operands of the
    two GEMMs, the SwiGLU value, the contribution), each at most 2^-11, so the
    outputs are off by at most sqrt(4) * 2^-11 of their root mean square."""
    H, I = 1024, 256
    layer = pkg.synth.moe_layer(hidden=H, inter=I, experts=1, seed=80 + rows, device=dev)
    x = pkg.synth.activations(rows, H, 81, dev).float()
    ch = torch.arange(3, H, 341, device=dev)
    x[:, ch] *= factor
    x = (x / (1.0 + factor * len(ch) / H ** 0.5)).half()
    ids = torch.zeros((rows, 1), dtype=torch.int32, device=dev)
    w = torch.ones((rows, 1), device=dev)
    out = pkg.grouped_moe_prefill_routed(layer, x, ids, w, expert_used_count=1)
    gu = _dequant_f64(layer.gate_up) @ x.double().cpu().T
    g, u = gu[:I], gu[I:]
    ref = (g * torch.sigmoid(g) * u).T @ _dequant_f64(layer.down).T
    err = (out.double().cpu() - ref).square().mean().sqrt() / ref.square().mean().sqrt()
    assert err <= 2.0 ** -10
