"""GPU parity of the grouped path (more than 8 rows): router GEMM, device
token-by-expert sort, MFMA grouped gate/up/down and the combines, against the
oracle.

The router logits of the grouped path come from an MFMA GEMM with fp32
accumulation, the oracle's from float64; a logit that sits on a bf16 rounding
boundary can round the other way, which can swap two experts whose gates tie
within one bf16 step.  Index sets are therefore required to match exactly
except on tokens whose oracle gates at ranks k-1 and k are within one bf16
step (a near tie, counted and bounded), and outputs are compared on the tokens
whose index sets match.

The matrix-form kernels round every dequantised weight to bf16 before the
MFMA, as the reference's gather_qmm matrix kernels stage weights in the
activation type; they are compared elementwise with the oracle's matrix form
(moe_oracle.qmm_project) and, at the layer tolerance (max-abs-rel 2e-2), with
the vector-form oracle that keeps the weights unrounded.
"""
import numpy as np
import pytest
import torch

from gpu_util import bf16_device, host, packs, to_device, ulp_diff_bf16
from oracle import moe_oracle as mo
from veymoe import _lib, assemble, synth
from veymoe.device import ptr, stream_handle
from veymoe.grouped import COMBINE_FUSED, COMBINE_GENERIC, COMBINE_NONE, grouped_experts
from veymoe.layer import HipSwitchGLU
from veymoe.layout import RecordLayout, pack_record
from veymoe.pool import ExpertPool

pytestmark = pytest.mark.gpu


def _near_tie(gates_row, k):
    order = np.sort(mo.f32_to_bf16_bits(np.asarray(gates_row, np.float32)).astype(np.int64))[::-1]
    return order[k - 1] - order[k] <= 1


def _check_selection(inds, ref, k, max_near_ties, label=""):
    """Rows whose index sets differ must be near ties; returns the matching
    rows.  The number of differing rows seen is printed (pytest -s / -v
    output) next to the bound, so a run shows what it found."""
    same = np.array([set(a) == set(b) for a, b in zip(inds.tolist(), ref["inds"].tolist())])
    for t in np.nonzero(~same)[0]:
        assert _near_tie(ref["gates"][t], k), (t, inds[t], ref["inds"][t])
    print(f"[selection] {label} rows {len(same)}: index sets differing from the oracle "
          f"{int((~same).sum())} (near ties; bound {max_near_ties})", flush=True)
    assert (~same).sum() <= max_near_ties, int((~same).sum())
    return same


def _layer_ref(spec, seed, x_np, rows, qmm=True):
    layer_np = synth.numpy_layer(spec, seed)
    return mo.moe_layer(x_np[rows], layer_np, "bf16", path="prefill", qmm=qmm)


def _close_qmm(actual, expected, message):
    """Against the matrix-form oracle the remaining differences are bf16
    rounding-boundary flips of intermediate values (fp32 against float64
    accumulation): each at most one bf16 step at the scale of the output,
    and rare."""
    actual = np.asarray(actual, np.float64)
    expected = np.asarray(expected, np.float64)
    scale = float(np.abs(expected).max())
    np.testing.assert_allclose(actual, expected, rtol=2e-2, atol=2.0 ** -7 * scale, err_msg=message)
    assert mo.max_abs_rel(actual, expected) <= 2.0 ** -7, (message, mo.max_abs_rel(actual, expected))
    far = ulp_diff_bf16(actual, expected) > 1
    assert far.mean() < 2e-3, (message, far.mean())


def _assert_layer(actual, spec, seed, x_np, rows, same, ref, message):
    """Elementwise against the matrix-form oracle, max-abs-rel 2e-2 against
    the vector-form oracle."""
    _close_qmm(actual[same], ref["output"][same], message)
    vec = _layer_ref(spec, seed, x_np, rows, qmm=False)
    assert mo.max_abs_rel(actual[same], vec["output"][same]) <= 2e-2, message


@pytest.mark.parametrize("tokens", [9, 40, 130])
def test_grouped_layer_small(device, tokens):
    spec = synth.CONFIGS["decode_small"]
    seed = 300 + tokens
    layer = assemble.build_layer(spec, seed, device, dense=True)
    x_np = mo.bf16_bits_to_f32(synth.tokens(spec, seed, tokens))
    y = layer(bf16_device(x_np, device))
    torch.cuda.synchronize()
    rows = np.arange(tokens)
    ref = _layer_ref(spec, seed, x_np, rows)
    same = _check_selection(layer.last_inds.cpu().numpy(), ref, spec.top_k, max(1, tokens // 20), f"T={tokens}")
    _assert_layer(host(y), spec, seed, x_np, rows, same, ref, f"grouped layer T={tokens}")


@pytest.mark.parametrize("tokens", [130, 300])
def test_grouped_layer_narrow_hidden_with_shared_expert(device, tokens):
    """Hidden 256 with a shared expert: at 130 rows one more group of the
    sorted GEMMs, at 300 rows on the side stream, whose rows and sigmoid gates
    the combine reads back.
    At this width a token's 32 combine threads share a wave with another
    token's, so the combine takes its per-lane loads (wider layers read a
    token's indices, scores and gate through scalar loads)."""
    spec = synth.LayerSpec("narrow_shared", 256, 128, 64, 4, 128, 1)
    seed = 320 + tokens
    layer = assemble.build_layer(spec, seed, device, dense=True)
    x_np = mo.bf16_bits_to_f32(synth.tokens(spec, seed, tokens))
    y = layer(bf16_device(x_np, device))
    torch.cuda.synchronize()
    rows = np.arange(tokens)
    ref = _layer_ref(spec, seed, x_np, rows)
    same = _check_selection(layer.last_inds.cpu().numpy(), ref, spec.top_k, max(1, tokens // 20), f"T={tokens}")
    _assert_layer(host(y), spec, seed, x_np, rows, same, ref, f"narrow grouped layer T={tokens}")


def test_grouped_layer_tile_heights_agree(device):
    """768, 1024 and 4096 tokens over 64 experts top-4: 48, 64 and 256 rows
    per expert on average.  A call whose experts average more rows than one
    tile of the usual height holds takes 96-row tiles: neither GEMM at 768
    tokens, the down GEMM at 1024 (above its 48), both at 4096 (several row
    tiles per group).  Each call is checked against the oracle on a sample,
    and a row's result does not depend on its tile, so the first 768 rows of
    every call are equal bit for bit."""
    spec = synth.CONFIGS["decode_small"]
    seed = 311
    layer = assemble.build_layer(spec, seed, device, dense=True)
    x_all = mo.bf16_bits_to_f32(synth.tokens(spec, seed, 4096))
    first = None
    for tokens in (768, 1024, 4096):
        x_np = x_all[:tokens]
        y = layer(bf16_device(x_np, device))
        torch.cuda.synchronize()
        sample = np.random.default_rng(tokens).choice(tokens, 48, replace=False)
        ref = _layer_ref(spec, seed, x_np, sample)
        inds = layer.last_inds.cpu().numpy()[sample]
        same = _check_selection(inds, ref, spec.top_k, 3, f"T={tokens} over 64 experts")
        _assert_layer(host(y)[sample], spec, seed, x_np, sample, same, ref, f"grouped layer T={tokens} (sample)")
        if first is None:
            first = y[:768].clone()
        else:
            assert torch.equal(first.view(torch.int16), y[:768].view(torch.int16)), tokens


@pytest.mark.parametrize("hidden,experts,tokens,zipf", [(4096, 128, 300, None), (4096, 128, 8256, None),
                                                         (1024, 512, 4096, None), (2048, 512, 1000, 1.1),
                                                         (1024, 96, 300, None)],
                         ids=["k4096-8stage", "k4096-4stage", "k1024-4stage", "k2048-bias", "chunked-e96"])
def test_router_gemm_instances(device, hidden, experts, tokens, zipf):
    """The router GEMM of calls above 64 rows at the K and ring depths the
    prefill shapes do not reach (K = 4096 with eight and four stages, K = 1024
    with four), with a router bias (the log-Zipf popularity of the
    synthetic layers), and at 96 experts, which the ring does not take (the
    chunked GEMM computes those logits): the experts chosen per row equal the decode router's,
    which sums every logit in another order, except on near ties (bounded,
    and checked against the oracle's gates); at 300 rows the whole layer is
    compared with the oracle."""
    from veymoe.router import router_topk

    spec = synth.LayerSpec(f"router_k{hidden}", hidden, 256, experts, 6, 0, tokens, zipf_s=zipf)
    seed = 340 + hidden // 1024 + experts
    layer = assemble.build_layer(spec, seed, device, dense=True)
    x_np = mo.bf16_bits_to_f32(synth.tokens(spec, seed, tokens))
    x = bf16_device(x_np, device)
    y = layer(x)
    grouped = layer.last_inds.sort(dim=1).values
    bias = layer.gate.bias.float() if layer.gate.bias is not None else None
    decode, _ = router_topk(x, layer.gate.weight, spec.top_k, logit_bias=bias)
    decode = decode.sort(dim=1).values
    torch.cuda.synchronize()
    differ = np.nonzero(~(grouped == decode).all(dim=1).cpu().numpy())[0]
    print(f"[selection] router GEMM K={hidden} E={experts} T={tokens}: {len(differ)} rows differ from the "
          f"decode router", flush=True)
    if len(differ):
        layer_np = synth.numpy_layer(spec, seed)
        _, _, gates = mo.route(x_np[differ], layer_np["router"], spec.top_k, "bf16", layer_np.get("router_bias"))
        for i in range(len(differ)):
            assert _near_tie(gates[i], spec.top_k), int(differ[i])
    assert len(differ) <= max(1, tokens // 1000)
    if tokens <= 512:
        rows = np.arange(tokens)
        ref = _layer_ref(spec, seed, x_np, rows)
        same = _check_selection(layer.last_inds.cpu().numpy(), ref, spec.top_k, max(1, tokens // 20),
                                f"K={hidden} T={tokens}")
        _assert_layer(host(y), spec, seed, x_np, rows, same, ref, f"layer K={hidden} T={tokens}")


def test_grouped_batched_config_pool(device):
    """The full-size layer with Zipf(1.1) routing at 32 tokens, experts in a
    pool behind a permuted slot table, shared expert included."""
    spec = synth.CONFIGS["batched"]
    seed = 320
    pool = ExpertPool(spec.layout, spec.experts + 8, layers=1, experts=spec.experts, device=device)
    layer = assemble.build_layer(spec, seed, device, pool=pool)
    x_np = mo.bf16_bits_to_f32(synth.tokens(spec, seed, 32))
    y = layer(bf16_device(x_np, device))
    torch.cuda.synchronize()
    rows = np.arange(32)
    ref = _layer_ref(spec, seed, x_np, rows)
    same = _check_selection(layer.last_inds.cpu().numpy(), ref, spec.top_k, 2, "batched T=32")
    _assert_layer(host(y), spec, seed, x_np, rows, same, ref, "batched layer")
    distinct = len(np.unique(ref["inds"]))
    assert 40 <= distinct <= 320, distinct


def test_grouped_prefill_matches_decode_rows(device):
    """At the full prefill shape (2048 tokens, 512 experts top-10 + shared):
    256 rows spread over the call against the oracle, and the first 8 rows
    against the decode kernels run on those 8 rows alone.

    The grouped router is an MFMA GEMM and the decode router a v_dot2
    reduction: both accumulate in fp32, in different orders, so a logit on a
    bf16 rounding boundary can round differently and swap two experts whose
    gates tie within one bf16 step.  The number of such rows is printed."""
    spec = synth.CONFIGS["prefill"]
    seed = 330
    pool = ExpertPool(spec.layout, spec.experts, layers=1, experts=spec.experts, device=device)
    layer = assemble.build_layer(spec, seed, device, pool=pool)
    x_np = mo.bf16_bits_to_f32(synth.tokens(spec, seed, 2048))
    x = bf16_device(x_np, device)
    y = layer(x)
    inds_all = layer.last_inds.clone()
    y8 = layer(x[:8].contiguous())
    torch.cuda.synchronize()
    agree = (inds_all[:8].sort(dim=1).values == layer.last_inds.sort(dim=1).values).all(dim=1).cpu().numpy()
    print(f"[selection] prefill rows 0..7: grouped and decode routers agree on {int(agree.sum())} of 8", flush=True)
    assert int(agree.sum()) >= 7
    # matrix form + generic combine against vector form + fused combine: the layer tolerance
    assert mo.max_abs_rel(host(y)[:8][agree], host(y8)[agree]) <= 2e-2
    sample = np.linspace(0, 2047, 256).astype(np.int64)
    ref = _layer_ref(spec, seed, x_np, sample)
    same = _check_selection(inds_all.cpu().numpy()[sample], ref, spec.top_k, 3, "prefill T=2048 (256 rows)")
    _assert_layer(host(y)[sample], spec, seed, x_np, sample, same, ref, "prefill sample vs oracle")


def test_grouped_router_against_the_decode_router_over_8192_rows(device):
    """The rate at which the grouped (MFMA) router and the decode (v_dot2)
    router pick different expert sets for the same token, over 8192 tokens
    at the full prefill shape: the layer in 2048-row calls (MFMA router)
    against vm_router_topk, which sums every logit in the decode order at
    any row count.  Calls of up to 64 rows route with the decode router, so
    only calls above that can differ; the differing rows must be near ties
    and their count is printed."""
    from veymoe.router import router_topk

    spec = synth.CONFIGS["prefill"]
    seed = 331
    pool = ExpertPool(spec.layout, spec.experts, layers=1, experts=spec.experts, device=device)
    layer = assemble.build_layer(spec, seed, device, pool=pool)
    rows = 8192
    x_np = mo.bf16_bits_to_f32(synth.tokens(spec, seed, rows))
    x = bf16_device(x_np, device)
    grouped = []
    for c in range(0, rows, 2048):
        layer(x[c:c + 2048].contiguous())
        grouped.append(layer.last_inds.clone())
    grouped = torch.cat(grouped).sort(dim=1).values
    bias = layer.gate.bias.float() if layer.gate.bias is not None else None
    decode, _ = router_topk(x, layer.gate.weight, spec.top_k, logit_bias=bias)
    decode = decode.sort(dim=1).values
    torch.cuda.synchronize()
    differ = np.nonzero(~(grouped == decode).all(dim=1).cpu().numpy())[0]
    print(f"[selection] grouped vs decode router over {rows} rows: {len(differ)} rows differ "
          f"({len(differ) / rows:.2e})", flush=True)
    if len(differ):
        layer_np = synth.numpy_layer(spec, seed)
        _, _, gates = mo.route(x_np[differ], layer_np["router"], spec.top_k, "bf16", layer_np["router_bias"])
        for i in range(len(differ)):
            assert _near_tie(gates[i], spec.top_k), int(differ[i])
    assert len(differ) <= rows // 1000


def _switch(np_packs, hidden, inter, experts, device):
    return HipSwitchGLU(hidden, inter, experts, projections=to_device(np_packs, device))


@pytest.mark.parametrize("mode", [COMBINE_NONE, COMBINE_GENERIC, COMBINE_FUSED])
@pytest.mark.parametrize("tokens,crowd,hidden,inter", [(150, 100, 256, 128), (60, 40, 256, 256), (24, 17, 4096, 512)],
                         ids=["64-row-tiles", "16-row-tiles", "16-row-tiles-k4096"])
def test_grouped_experts_modes(device, mode, tokens, crowd, hidden, inter):
    """150 tokens run the 64-row tile GEMM; calls of up to 64 rows whose
    hidden and intermediate sizes have an instance run the 16-row tile
    kernels (K = 256 both ways; K = 4096 for gate/up with 512 for down, the
    largest instance).  One expert takes `crowd` rows, so it spans two
    (three, two) tiles."""
    experts, k = 12, 3
    np_packs = packs(41, hidden, inter, experts)
    rng = np.random.default_rng(42)
    inds = np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32)
    inds[:crowd, 0] = 5                     # expert 5: several row tiles
    scores = mo.bf16r(rng.uniform(0.05, 0.6, (tokens, k)).astype(np.float32))
    x_np = mo.bf16r(rng.normal(size=(tokens, hidden)).astype(np.float32))
    shared_y = mo.bf16r(rng.normal(0, 0.1, (tokens, hidden)).astype(np.float32))
    switch = _switch(np_packs, hidden, inter, experts, device)
    out = grouped_experts(switch, bf16_device(x_np, device), torch.tensor(inds, device=device),
                          bf16_device(scores, device), bf16_device(shared_y, device), mode)
    torch.cuda.synchronize()
    _, _, _, d_out, _ = mo.execute(x_np, inds, np_packs, "bf16", qmm=True)
    if mode == COMBINE_NONE:
        _close_qmm(host(out), d_out, "per-slot rows")
    elif mode == COMBINE_GENERIC:
        _close_qmm(host(out), mo.generic_combine(d_out, scores, "bf16", shared_y), "generic combine")
    else:
        _close_qmm(host(out), mo.fused_combine(d_out, scores, "bf16", shared_y=shared_y), "fused combine")


def test_grouped_invalid_expert_id_contributes_nothing(device):
    hidden, inter, experts, tokens, k = 128, 64, 6, 12, 2
    np_packs = packs(51, hidden, inter, experts)
    rng = np.random.default_rng(52)
    inds = np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32)
    inds[3, 1] = 99                          # outside 0..experts-1
    x_np = mo.bf16r(rng.normal(size=(tokens, hidden)).astype(np.float32))
    switch = _switch(np_packs, hidden, inter, experts, device)
    out = grouped_experts(switch, bf16_device(x_np, device), torch.tensor(inds, device=device))
    torch.cuda.synchronize()
    assert float(out[3, 1].abs().max()) == 0.0
    ok = np.ones(tokens * k, bool)
    ok[3 * k + 1] = False
    inds_ok = inds.copy()
    inds_ok[3, 1] = 0
    _, _, _, d_out, _ = mo.execute(x_np, inds_ok, np_packs, "bf16", qmm=True)
    _close_qmm(host(out).reshape(-1, hidden)[ok], d_out.reshape(-1, hidden)[ok], "valid rows")


def test_grouped_pool_matches_dense_bitwise(device):
    """The same experts through a pool + permuted slot table give the same bits."""
    hidden, inter, experts, tokens, k = 256, 128, 16, 70, 4
    np_packs = packs(61, hidden, inter, experts)
    rng = np.random.default_rng(62)
    inds = torch.tensor(np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32),
                        device=device)
    x = bf16_device(rng.normal(size=(tokens, hidden)).astype(np.float32), device)
    dense = _switch(np_packs, hidden, inter, experts, device)
    layout = RecordLayout(hidden, inter)
    pool = ExpertPool(layout, experts + 5, layers=1, experts=experts, device=device)
    slots = rng.permutation(experts + 5)[:experts]
    for e in range(experts):
        parts = {(name, part): np_packs[name][i][e] for name in np_packs
                 for i, part in enumerate(("weight", "scales", "biases"))}
        pool.record(int(slots[e])).copy_(torch.from_numpy(pack_record(parts, layout)))
    pool.place_all(0, slots)
    pooled = HipSwitchGLU(hidden, inter, experts, pool=pool, layer_id=0)
    a = grouped_experts(dense, x, inds)
    b = grouped_experts(pooled, x, inds)
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_pooled_switch_above_the_decode_bound_takes_one_lru_pass(device):
    """A pool-backed HipSwitchGLU called with more than 8 rows assigns and
    fills once per call: pool and switch hit/miss counts, slot table and free
    list follow the reference's LRU (expert_pool.py:123-159) fed the same
    routed ids, and the per-slot outputs equal the dense expert block's."""
    from oracle import pool_oracle
    from veymoe.pool import HostRecordStore

    spec = synth.LayerSpec("sw_pool", 256, 128, 96, 4, 0, 12)
    seed = 404
    store = HostRecordStore(spec.layout, spec.experts)
    for e in range(spec.experts):
        store.put(0, e, synth.expert_record(spec, seed, 0, e))
    pool = ExpertPool(spec.layout, 48, layers=1, experts=spec.experts, device=device)
    pooled = HipSwitchGLU(spec.hidden, spec.inter, spec.experts, pool=pool, layer_id=0, host_store=store)
    layer_np = synth.numpy_layer(spec, seed, materialise=True)
    dense = HipSwitchGLU(spec.hidden, spec.inter, spec.experts, layer_id=0,
                         projections={n: assemble.projection(*layer_np[n], device)
                                      for n in ("gate_proj", "up_proj", "down_proj")})
    ref = pool_oracle.LruSlots(48)
    rng = np.random.default_rng(5)
    for step in range(6):
        rows = 9 + 3 * step
        # each call routes within a window of 40 experts (fits the pool), moving by 17 per call
        window = (17 * step + np.arange(40)) % spec.experts
        inds = np.stack([rng.choice(window, spec.top_k, replace=False) for _ in range(rows)]).astype(np.int32)
        x = assemble.tokens_tensor(spec, seed, device, rows, stream=50 + step)
        got = pooled(x[None], torch.tensor(inds[None], device=device))
        want = dense(x[None], torch.tensor(inds[None], device=device))
        torch.cuda.synchronize()
        assert got.shape == (1, rows, spec.top_k, spec.hidden)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), step
        routed = inds.reshape(-1).tolist()
        _, misses = ref.assign(0, routed)
        hits = len(routed) - len(misses)
        assert (pool.hits, pool.misses) == (ref.hits, ref.misses), step
        assert pooled.misses == ref.misses, step
        assert list(pool._slot_of.items()) == list(ref.slot_of.items()), step
        assert pool._free == ref.free, step
        assert hits >= 0
    assert ref.misses > 48                      # evictions happened


@pytest.mark.parametrize("tokens", [12, 150, 330], ids=["16-row-class", "48-row-tiles", "96-row-tiles"])
@pytest.mark.parametrize("inter", [384, 640, 896, 320], ids=["8+4", "8+8+4", "3x8+4", "8+2-clamped"])
def test_down_gemm_half_chunk_tail(device, tokens, inter):
    """Intermediate sizes of half a K chunk over (12, 20 and 28 groups) run
    the down GEMM's staged half-tail instances, 10 groups the clamped tail.
    One expert takes two thirds of the rows (several tiles, a ragged last
    one); 330 tokens over 12 experts take the tall tiles.  Weight scales of
    the last row end the bank, so a load past a row would be past its end."""
    hidden, experts, k = 256, 12, 3
    np_packs = packs(71, hidden, inter, experts)
    rng = np.random.default_rng(72 + inter)
    inds = np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32)
    inds[:2 * tokens // 3, 0] = experts - 1
    x_np = mo.bf16r(rng.normal(size=(tokens, hidden)).astype(np.float32))
    switch = _switch(np_packs, hidden, inter, experts, device)
    out = grouped_experts(switch, bf16_device(x_np, device), torch.tensor(inds, device=device))
    torch.cuda.synchronize()
    _, _, _, d_out, _ = mo.execute(x_np, inds, np_packs, "bf16", qmm=True)
    _close_qmm(host(out), d_out, f"inter {inter}, {tokens} rows")


@pytest.mark.parametrize("inter", [256, 640])
@pytest.mark.parametrize("hidden", [96, 1088])
def test_down_gemm_of_whole_rows_gives_the_chunked_bits(device, hidden, inter):
    """At these widths calls of up to 48 rows per expert keep a tile's whole rows in LDS (k_down_rows), calls above
    take the chunked GEMM's 96-row tiles: the same tokens give the same bits in both, and match the oracle.  Two
    thirds of the rows go to the last expert (several tiles, a ragged last one, the bank's end); output widths that
    end inside a block and inside its second pass."""
    experts, k = 24, 3
    np_packs = packs(73, hidden, inter, experts)
    rng = np.random.default_rng(74 + inter + hidden)
    tokens, more = 150, 500
    inds = np.stack([rng.choice(experts - 1, k, replace=False) for _ in range(more)]).astype(np.int32)
    inds[:2 * tokens // 3, 0] = experts - 1
    valid = inds[:tokens].copy()
    inds[5, 2] = 99                          # names no expert: a row of zeros
    x_np = mo.bf16r(rng.normal(size=(more, hidden)).astype(np.float32))
    switch = _switch(np_packs, hidden, inter, experts, device)
    x, i = bf16_device(x_np, device), torch.tensor(inds, device=device)
    out = grouped_experts(switch, x[:tokens].contiguous(), i[:tokens].contiguous())
    tall = grouped_experts(switch, x, i)
    torch.cuda.synchronize()
    _, _, _, d_out, _ = mo.execute(x_np[:tokens], valid, np_packs, "bf16", qmm=True)
    d_out[5, 2] = 0.0
    assert float(out[5, 2].abs().max()) == 0.0
    _close_qmm(host(out), d_out, f"hidden {hidden}, inter {inter}")
    assert torch.equal(out.view(torch.int16), tall[:tokens].view(torch.int16))


def test_slot_rows_of_a_sort_over_many_blocks(device):
    """One output row per token and slot, stored by the down GEMM itself: 1400 tokens top-3 over 96 experts (more
    pairs than one sort block takes) give the bits of two calls of 700."""
    hidden, inter, experts, tokens, k = 128, 256, 96, 1400, 3
    np_packs = packs(75, hidden, inter, experts)
    rng = np.random.default_rng(76)
    inds = torch.tensor(np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32))
    inds[900, 1] = -1
    inds = inds.to(device)
    x = bf16_device(mo.bf16r(rng.normal(size=(tokens, hidden)).astype(np.float32)), device)
    switch = _switch(np_packs, hidden, inter, experts, device)
    whole = grouped_experts(switch, x, inds)
    halves = torch.cat([grouped_experts(switch, x[:700].contiguous(), inds[:700].contiguous()),
                        grouped_experts(switch, x[700:].contiguous(), inds[700:].contiguous())])
    torch.cuda.synchronize()
    assert float(whole[900, 1].abs().max()) == 0.0
    assert torch.equal(whole.view(torch.int16), halves.view(torch.int16))


@pytest.mark.parametrize("inter", [256, 640])
@pytest.mark.parametrize("hidden,tokens", [(96, 70), (1088, 150), (128, 1400)])
@pytest.mark.parametrize("share", [0.35, 1.0], ids=["third", "all"])
def test_slot_rows_of_ids_without_an_expert(device, monkeypatch, inter, hidden, tokens, share):
    """Slot rows of pairs padded with ids that name no expert (-1 and one past the last) are zeros in an output that
    held NaN before, and the other rows are the bits of the call without padding: output rows shorter and longer than
    a wave's store, a grid with fewer waves than pairs (1400 tokens), one sort block and several."""
    experts, k = 96, 3
    rng = np.random.default_rng(81 + inter + hidden)
    switch = _switch(packs(80, hidden, inter, experts), hidden, inter, experts, device)
    inds = np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32)
    dead = rng.random(inds.shape) < share
    padded = np.where(dead, np.where(rng.random(inds.shape) < 0.5, -1, experts), inds).astype(np.int32)
    x = bf16_device(mo.bf16r(rng.normal(size=(tokens, hidden)).astype(np.float32)), device)
    whole = grouped_experts(switch, x, torch.tensor(inds, device=device))
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: empty(*a, **kw).fill_(0xff if kw["dtype"] == torch.uint8
                                                                               else float("nan")))
    out = grouped_experts(switch, x, torch.tensor(padded, device=device))
    monkeypatch.undo()
    torch.cuda.synchronize()
    mask = torch.tensor(dead, device=device).unsqueeze(-1)
    assert torch.equal(out.view(torch.int16), torch.where(mask, 0, whole.view(torch.int16)))


@pytest.mark.parametrize("hidden,inter,experts,tokens,k", [(1024, 256, 64, 700, 4), (2560, 640, 32, 120, 10)])
def test_padded_ids_do_not_slow_an_experts_call(device, hidden, inter, experts, tokens, k):
    """A call all of whose ids name no expert writes its zeros and computes nothing, so it takes no longer than the
    call with every id valid (half as long where this was written; zeros stored row by row from the sort's own
    threads took 4 to 25 times as long)."""
    rng = np.random.default_rng(83)
    switch = _switch(packs(82, hidden, inter, experts), hidden, inter, experts, device)
    inds = torch.tensor(np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32),
                        device=device)
    x = bf16_device(rng.normal(size=(tokens, hidden)).astype(np.float32), device)

    def median(ids):
        times = []
        for _ in range(25):
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(4):
                grouped_experts(switch, x, ids)
            stop.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(stop))
        return sorted(times)[len(times) // 2]

    none = torch.full_like(inds, -1)
    valid, padded = median(inds), median(none)
    print(f"[time] four calls: valid ids {valid * 1e3:.0f} us, no id valid {padded * 1e3:.0f} us", flush=True)
    assert padded <= 1.25 * valid


@pytest.mark.parametrize("hidden,inter", [(384, 512), (384, 256), (256, 384), (256, 640)])
def test_small_calls_of_one_supported_size_give_the_larger_calls_bits(device, hidden, inter):
    """The 16-row tile kernels, whose K order is their own, run only where both sizes have an instance: with one of
    them alone, the rows of a 40-token call have the bits of the same rows in a call of 130."""
    experts, k = 24, 3
    rng = np.random.default_rng(85 + hidden + inter)
    switch = _switch(packs(84, hidden, inter, experts), hidden, inter, experts, device)
    inds = torch.tensor(np.stack([rng.choice(experts, k, replace=False) for _ in range(130)]).astype(np.int32),
                        device=device)
    x = bf16_device(mo.bf16r(rng.normal(size=(130, hidden)).astype(np.float32)), device)
    small = grouped_experts(switch, x[:40].contiguous(), inds[:40].contiguous())
    large = grouped_experts(switch, x, inds)
    torch.cuda.synchronize()
    assert torch.equal(small.view(torch.int16), large[:40].view(torch.int16))


@pytest.mark.parametrize("inter", [256, 384, 640, 896])
@pytest.mark.parametrize("hidden", [1088, 2080])
def test_down_gemm_of_whole_rows_at_half_chunks_over(device, hidden, inter):
    """Every instance of k_down_rows whose K has half a chunk over, with two column blocks per wave (hidden 1088) and
    four (2080), both ending inside a block, and K of one chunk, which is the chunked GEMM's at hidden 2080: the bits
    of the chunked GEMM's 96-row tiles, which a call of 500 tokens takes, and the oracle's values.  Calls of 20 and
    150 tokens; two thirds of their rows go to the last expert."""
    experts, k, more = 24, 3, 500
    np_packs = packs(86, hidden, inter, experts)
    rng = np.random.default_rng(87 + inter + hidden)
    inds = np.stack([rng.choice(experts - 1, k, replace=False) for _ in range(more)]).astype(np.int32)
    inds[:100, 0] = experts - 1
    x_np = mo.bf16r(rng.normal(size=(more, hidden)).astype(np.float32))
    switch = _switch(np_packs, hidden, inter, experts, device)
    x, i = bf16_device(x_np, device), torch.tensor(inds, device=device)
    tall = grouped_experts(switch, x, i)
    for tokens in (20, 150):
        out = grouped_experts(switch, x[:tokens].contiguous(), i[:tokens].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), tall[:tokens].view(torch.int16)), tokens
    _, _, _, d_out, _ = mo.execute(x_np[:20], inds[:20], np_packs, "bf16", qmm=True)
    _close_qmm(host(tall[:20]), d_out, f"hidden {hidden}, inter {inter}")


@pytest.mark.parametrize("hidden", [96, 1088])
def test_down_gemm_of_half_chunks_gives_one_result_by_every_way(device, hidden):
    """Inter 1152, whose half chunk over is too wide for k_down_rows: calls of few blocks let the lanes fetch their
    own weights, larger ones stage them, calls above 48 rows per expert take 96-row tiles.  One row, the same bits."""
    experts, k, inter, more = 96, 3, 1152, 1700
    np_packs = packs(88, hidden, inter, experts)
    rng = np.random.default_rng(89 + hidden)
    inds = np.stack([rng.choice(experts, k, replace=False) for _ in range(more)]).astype(np.int32)
    x_np = mo.bf16r(rng.normal(size=(more, hidden)).astype(np.float32))
    switch = _switch(np_packs, hidden, inter, experts, device)
    x, i = bf16_device(x_np, device), torch.tensor(inds, device=device)
    tall = grouped_experts(switch, x, i)
    for tokens in (20, 150, 1500):
        out = grouped_experts(switch, x[:tokens].contiguous(), i[:tokens].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), tall[:tokens].view(torch.int16)), tokens
    _, _, _, d_out, _ = mo.execute(x_np[:20], inds[:20], np_packs, "bf16", qmm=True)
    _close_qmm(host(tall[:20]), d_out, f"hidden {hidden}")


@pytest.mark.parametrize("hidden,inter,tokens", [(256, 640, 12), (256, 640, 150), (256, 256, 150), (256, 1152, 150),
                                                 (256, 640, 300), (2048, 640, 300), (2048, 640, 400)])
def test_grouped_layer_with_a_shared_expert_over_half_chunks(device, hidden, inter, tokens):
    """The shared expert's rows as one more group of the whole-row and the chunked down GEMM (up to 256 rows), and on
    the side stream in tiles of the usual height (300 rows: few blocks) and in tall ones (400 rows at hidden 2048)."""
    spec = synth.LayerSpec("half_shared", hidden, inter, 24, 4, inter, 1)
    seed = 340 + inter + tokens
    layer = assemble.build_layer(spec, seed, device, dense=True)
    x_np = mo.bf16_bits_to_f32(synth.tokens(spec, seed, tokens))
    y = layer(bf16_device(x_np, device))
    torch.cuda.synchronize()
    rows = np.unique(np.linspace(0, tokens - 1, 40).astype(int))
    ref = _layer_ref(spec, seed, x_np, rows)
    same = _check_selection(layer.last_inds.cpu().numpy()[rows], ref, spec.top_k, 3, f"T={tokens}")
    _assert_layer(host(y)[rows], spec, seed, x_np, rows, same, ref, f"{hidden}/{inter} T={tokens}")


@pytest.mark.parametrize("inter", [256, 640])
@pytest.mark.parametrize("tokens", [30, 150])
def test_down_gemm_of_whole_rows_over_pool_records(device, inter, tokens):
    """k_down_rows over records behind a slot table, one record a load past whose end would leave the pool: the dense
    bits; experts without a record set the status bit and leave rows of zeros, in the slot rows and in the combine."""
    hidden, experts, k = 1088, 24, 3
    np_packs = packs(90, hidden, inter, experts)
    rng = np.random.default_rng(91 + inter)
    inds_np = np.stack([rng.choice(experts, k, replace=False) for _ in range(tokens)]).astype(np.int32)
    inds = torch.tensor(inds_np, device=device)
    x = bf16_device(mo.bf16r(rng.normal(size=(tokens, hidden)).astype(np.float32)), device)
    scores = torch.rand((tokens, k), device=device).to(torch.bfloat16)
    dense = _switch(np_packs, hidden, inter, experts, device)
    layout = RecordLayout(hidden, inter)
    pool = ExpertPool(layout, experts, layers=1, experts=experts, device=device)
    slots = rng.permutation(experts)
    for e in range(experts):
        parts = {(name, part): np_packs[name][i][e] for name in np_packs
                 for i, part in enumerate(("weight", "scales", "biases"))}
        pool.record(int(slots[e])).copy_(torch.from_numpy(pack_record(parts, layout)))
    pool.place_all(0, slots)
    pooled = HipSwitchGLU(hidden, inter, experts, pool=pool, layer_id=0)
    rows = grouped_experts(dense, x, inds)
    assert torch.equal(grouped_experts(pooled, x, inds), rows)

    hole = int(inds_np[0, 0])
    table = pool.table(0).clone()
    table[hole] = -1
    lib = _lib.lib()
    for mode in (COMBINE_NONE, COMBINE_FUSED):
        want = torch.where((inds == hole).unsqueeze(-1), torch.zeros_like(rows), rows)
        if mode == COMBINE_FUSED:   # an expert of all-zero rows adds nothing to a token's sum
            kept = torch.where(inds == hole, torch.full_like(inds, -1), inds)
            want = grouped_experts(dense, x, kept, scores, None, mode)
        out = torch.full_like(want, float("nan"))
        status = torch.zeros(1, dtype=torch.int32, device=device)
        ws = torch.empty(int(lib.vm_moe_grouped_workspace(tokens, k, hidden, inter, experts, 0)), dtype=torch.uint8,
                         device=device)
        a = _lib.VmGroupedArgs()
        a.x, a.inds, a.output, a.status = ptr(x), ptr(inds), ptr(out), ptr(status)
        a.scores = ptr(scores)
        a.pool, a.slot_table = pool.view(), ptr(table)
        a.workspace, a.workspace_bytes = ptr(ws), ws.numel()
        a.tokens, a.top_k, a.hidden_size, a.inter_size, a.expert_count = tokens, k, hidden, inter, experts
        a.group_size, a.act_dtype, a.combine_mode = 32, 0, mode
        _lib.check(lib.vm_moe_grouped(a, stream_handle()))
        torch.cuda.synchronize()
        assert int(status.item()) & 1
        assert torch.equal(out, want), mode
