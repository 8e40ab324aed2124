"""GPU parity of the decoder glue around the MoE call (veymoe.glue).

* vm_hyper_mix (qwen4_verifier.py:20-33) against oracle.glue_oracle.hyper_mix
  on the shapes of the reference's own glue test (hc 4, hidden 256, low rank
  32; test_compile_glue.py:17-29) and at hidden 2048: the normalised streams
  within one bf16 step (the mean of squares is summed in another order), the
  branch input and the injection weights within the layer tolerance; with
  selector projections (each output reads one input, so every dot product is
  exact) nearly all values bit for bit.
* The injection in the experts' epilogue (compile_glue.py:32-35): for decode
  and grouped calls, bit for bit the oracle's ``inject`` of the layer's own
  output, also in place.
* ``mlp_branch``: hyper-connection, MoE layer and injection against the oracle
  chain.
"""
import numpy as np
import pytest
import torch

from gpu_util import assert_close, host
from oracle import glue_oracle as go
from oracle import moe_oracle as mo
from veymoe import assemble, synth
from veymoe.glue import HyperConnection, mlp_branch

pytestmark = pytest.mark.gpu

SEED = 123


def _hyper_np(rng, hc, H, r):
    n = hc * H
    norm_w = mo.bf16r(rng.normal(1.0, 0.3, n).astype(np.float32))
    down = synth.q4_projection(rng, r, n)
    up = synth.q4_projection(rng, n, r)
    inj = synth.q4_projection(rng, hc, n)
    return norm_w, down, up, inj


def _hyper_dev(parts, hc, device, dtype=torch.bfloat16, **kw):
    norm_w, down, up, inj = parts
    return HyperConnection(torch.from_numpy(norm_w).to(device).to(dtype),
                           *(assemble.projection(*p, device) for p in (down, up, inj)), hc, **kw)


def _streams(rng, T, n, device, dtype=torch.bfloat16):
    x = mo.bf16r(rng.normal(0, 1.5, (T, n)).astype(np.float32))
    return x, torch.from_numpy(x).to(device).to(dtype)


def _ulps(a, b):
    ia = mo.f32_to_bf16_bits(np.asarray(a, np.float32)).astype(np.int32)
    ib = mo.f32_to_bf16_bits(np.asarray(b, np.float32)).astype(np.int32)
    return np.abs(ia - ib)


@pytest.mark.parametrize("hc,H,r,T,group", [(4, 256, 32, 1, 0), (4, 256, 32, 5, 256), (4, 2048, 32, 3, 0),
                                             (2, 512, 64, 37, 0)])
def test_hyper_mix_matches_the_oracle(device, hc, H, r, T, group):
    rng = np.random.default_rng(SEED + H + T)
    parts = _hyper_np(rng, hc, H, r)
    x, xd = _streams(rng, T, hc * H, device)
    hyper = _hyper_dev(parts, hc, device, norm_group=group)
    mixed, same, weights = hyper(xd)
    torch.cuda.synchronize()
    assert same is xd
    want_m, want_w, want_n = go.hyper_mix(x, parts[0], parts[1], parts[2], parts[3], hc, 1e-6, group_size=group)
    normed = hyper._ws[(T, 0, xd.device)][: T * hc * H * 2].view(torch.bfloat16).view(T, hc * H)
    u = _ulps(host(normed), want_n)
    assert u.max() <= 1 and (u == 0).mean() >= 0.99, (u.max(), (u == 0).mean())
    assert_close(host(weights), want_w, f"weights T={T}")
    assert_close(host(mixed), want_m, f"mixed T={T}")


@pytest.mark.parametrize("hc,H,r,T,group,one_centered", [
    (4, 2560, 32, 67, 0, True), (4, 256, 32, 641, 256, False), (2, 512, 64, 655, 0, True), (5, 512, 32, 257, 512, True),
    (4, 2048, 96, 80, 0, True), (1, 4096, 32, 160, 64, True)])
def test_hyper_mix_tiles_match_the_oracle_and_the_per_token_kernels(device, hc, H, r, T, group, one_centered):
    """Calls of 655,360 stream values and more: 16-token tiles with a ragged last one, more than 48 projection
    rows, several norm groups, every stream-count instance.  The per-token kernels serve the same call from a
    workspace without the tiles' scratch: the normalised streams are the same bits."""
    rng = np.random.default_rng(SEED + H + T)
    parts = _hyper_np(rng, hc, H, r)
    x, xd = _streams(rng, T, hc * H, device)
    hyper = _hyper_dev(parts, hc, device, norm_group=group, one_centered=one_centered)
    mixed, _, weights = hyper(xd)
    n = hc * H
    normed_bytes = (2 * T * n + 255) // 256 * 256
    base = normed_bytes + (2 * T * r + 255) // 256 * 256
    ws = hyper._ws[(T, 0, xd.device)]
    assert ws.numel() > base
    ws[base:] = 0xcd
    mixed, _, weights = hyper(xd)
    torch.cuda.synchronize()
    assert bool((ws[base:] != 0xcd).any()), "the tile kernels wrote nothing"
    normed = ws[: 2 * T * n].clone()
    low = ws[normed_bytes: normed_bytes + 2 * T * r].clone().view(torch.bfloat16)
    hyper._ws[(T, 0, xd.device)] = torch.zeros(base, dtype=torch.uint8, device=device)
    mixed1, _, weights1 = hyper(xd)
    torch.cuda.synchronize()
    one = hyper._ws[(T, 0, xd.device)]
    assert torch.equal(one[: 2 * T * n], normed)
    low1 = one[normed_bytes: normed_bytes + 2 * T * r].view(torch.bfloat16)
    for got, per_token, what in ((low, low1, "d"), (weights, weights1, "weights"), (mixed, mixed1, "mixed")):
        assert_close(host(got).reshape(T, -1), host(per_token).reshape(T, -1), f"{what}: tiles and per token")
    want_m, want_w, _ = go.hyper_mix(x, *parts, hc, 1e-6, group_size=group, one_centered=one_centered)
    assert_close(host(weights), want_w, f"weights T={T}")
    assert_close(host(mixed), want_m, f"mixed T={T}")


def _tiles_and_per_token(hyper, xd, r):
    """(mixed, weights) of a call on 16-token tiles, whose scratch behind the workspace's base it must have written,
    and of the same call from a workspace without that scratch, which runs the per-token kernels."""
    T, n = xd.shape
    hyper(xd)
    key = (T, 0, xd.device)
    base = (2 * T * n + 255) // 256 * 256 + (2 * T * r + 255) // 256 * 256
    ws = hyper._ws[key]
    ws[base:] = 0xcd
    mixed, _, weights = hyper(xd)
    torch.cuda.synchronize()
    assert bool((ws[base:] != 0xcd).any()), "the tile kernels wrote nothing"
    hyper._ws[key] = torch.zeros(base, dtype=torch.uint8, device=xd.device)
    mixed1, _, weights1 = hyper(xd)
    torch.cuda.synchronize()
    hyper._ws[key] = ws
    return (mixed.clone(), weights.clone()), (mixed1, weights1)


def _power_of_two_inject(exps, hc, n, device):
    """Injection projection of ones: row j scales the 128 columns of block b by 2 ** exps[b * hc + j]."""
    scales = np.ldexp(np.float32(1), np.asarray(exps).reshape(n // 128, hc)).astype(np.float32)
    scales = np.repeat(scales.T, 4, axis=1)                                  # four groups of 32 per block
    words = np.full((hc, n // 8), 0x11111111, np.uint32)
    return assemble.projection(words, mo.f32_to_bf16_bits(scales), np.zeros((hc, n // 32), np.uint16), device)


@pytest.mark.parametrize("hc,exps", [(8, range(-130, 126)), (1, [*range(-133, -128), 126, 127] + [127] * 25)],
                         ids=["-133..122", "ends"])
def test_hyper_weights_pin_the_sigmoid_over_the_bf16_values(device, hc, exps):
    """The injection weights are 2 * sigmoid(a): with one value of every token's row set, a runs over the bf16 values
    of both signs, all 128 significands of each power of two from the smallest subnormal to the largest finite one, and
    over infinity and NaN; bit for bit the oracle's op-by-op sigmoid, from the tile and from the per-token kernels."""
    n, r = 4096, 32
    H = n // hc
    col = np.arange(n)
    gain = ((128 + col % 128) / 128.0 / 64.0).astype(np.float32)             # normalised, 64 * gain: 1 .. 255/128
    zero = lambda rows, width: assemble.projection(np.zeros((rows, width // 8), np.uint32),
                                                   np.zeros((rows, width // 32), np.uint16),
                                                   np.zeros((rows, width // 32), np.uint16), device)
    hyper = HyperConnection(torch.from_numpy(gain).to(device).to(torch.bfloat16), zero(r, n), zero(n, r),
                            _power_of_two_inject(exps, hc, n, device), hc, eps=1e-30)
    x = torch.zeros((2 * n + 1, n), dtype=torch.bfloat16, device=device)
    x[torch.arange(n), torch.arange(n)] = 1.0
    x[n + torch.arange(n), torch.arange(n)] = -1.0
    x[2 * n, 0] = float("nan")
    (_, tiles), (_, per_token) = _tiles_and_per_token(hyper, x, r)
    power = np.asarray(exps).reshape(n // 128, hc)[col // 128]               # [n, hc]
    with np.errstate(over="ignore", under="ignore"):
        a = np.ldexp((128 + col % 128)[:, None] / 128.0, power).astype(np.float32)
        a = mo.bf16r(mo.bf16r(a) / np.float32(hc))
    a = np.concatenate([a, -a])
    with np.errstate(over="ignore"):
        want = mo.f32_to_bf16_bits(mo.bf16r(np.float32(2) * mo.sigmoid(a, "bf16")))
    for got, what in ((tiles, "tiles"), (per_token, "per token")):
        bits = got.view(torch.int16).cpu().numpy().view(np.uint16)
        np.testing.assert_array_equal(bits[:-1], want, err_msg=what)
        assert bool(torch.isnan(got[-1].float()).all()), what


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_hyper_mix_tiles_keep_a_bad_token_to_itself(device, bad):
    """One stream value that is not finite: its token's outputs are what the per-token kernels make of it (NaN), every
    other token's, in the same tile too, the bits of the call without it."""
    hc, H, r, T = 4, 2560, 32, 67
    rng = np.random.default_rng(SEED + 11)
    hyper = _hyper_dev(_hyper_np(rng, hc, H, r), hc, device)
    _, xd = _streams(rng, T, hc * H, device)
    (clean_m, clean_w), _ = _tiles_and_per_token(hyper, xd, r)
    xd[35, 4321] = bad
    (mixed, weights), (mixed1, weights1) = _tiles_and_per_token(hyper, xd, r)
    rest = [t for t in range(T) if t != 35]
    assert torch.equal(mixed[rest].view(torch.int16), clean_m[rest].view(torch.int16))
    assert torch.equal(weights[rest].view(torch.int16), clean_w[rest].view(torch.int16))
    for got, one in ((mixed[35], mixed1[35]), (weights[35], weights1[35])):
        assert bool(torch.isnan(got.float()).any())
        assert torch.equal(torch.isnan(got.float()), torch.isnan(one.float()))


def test_hyper_mix_float32(device):
    hc, H, r, T = 4, 256, 32, 2
    rng = np.random.default_rng(SEED)
    parts = _hyper_np(rng, hc, H, r)
    x, xd = _streams(rng, T, hc * H, device, torch.float32)
    mixed, _, weights = _hyper_dev(parts, hc, device, torch.float32)(xd)
    torch.cuda.synchronize()
    want_m, want_w, _ = go.hyper_mix(x, parts[0], *parts[1:], hc, 1e-6, mode="f32")
    np.testing.assert_allclose(host(mixed), want_m, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(host(weights), want_w, rtol=1e-4, atol=1e-5)


def _selector(rows, cols, pick):
    q = np.zeros((rows, cols), np.uint32)
    q[np.arange(rows), pick] = 1
    words = np.zeros((rows, cols // 8), np.uint32)
    for k in range(8):
        words |= q[:, k::8] << np.uint32(4 * k)
    one = mo.f32_to_bf16_bits(np.ones((rows, cols // 32), np.float32))
    zero = mo.f32_to_bf16_bits(np.zeros((rows, cols // 32), np.float32))
    return words, one, zero


def test_hyper_mix_with_selector_projections_is_nearly_exact(device):
    hc, H, r, T = 4, 256, 32, 3
    n = hc * H
    rng = np.random.default_rng(SEED + 1)
    norm_w = mo.bf16r(rng.normal(1.0, 0.3, n).astype(np.float32))
    parts = (norm_w, _selector(r, n, (7 * np.arange(r) + 3) % n), _selector(n, r, (5 * np.arange(n) + 1) % r),
             _selector(hc, n, np.array([1, 300, 600, 1000])))
    x, xd = _streams(rng, T, n, device)
    mixed, _, weights = _hyper_dev(parts, hc, device)(xd)
    torch.cuda.synchronize()
    want_m, want_w, _ = go.hyper_mix(x, *parts, hc, 1e-6)
    for got, want in ((host(mixed), want_m), (host(weights), want_w)):
        u = _ulps(got, want)
        assert u.max() <= 1 and (u == 0).mean() >= 0.98, (u.max(), (u == 0).mean())


SMALL = synth.LayerSpec("glue_small", 256, 128, 64, 4, 128, 1)


@pytest.mark.parametrize("T", [1, 3, 8, 40])
@pytest.mark.parametrize("in_place", [False, True])
def test_injection_in_the_experts_epilogue_is_exact(device, T, in_place):
    hc = 4
    layer = assemble.build_layer(SMALL, SEED, device, dense=True)
    rng = np.random.default_rng(SEED + T)
    x = assemble.tokens_tensor(SMALL, SEED, device, T, stream=9)
    streams = torch.from_numpy(mo.bf16r(rng.normal(0, 1, (T, hc * SMALL.hidden)).astype(np.float32))).to(device)
    streams = streams.to(torch.bfloat16)
    weights = torch.from_numpy(mo.bf16r(rng.uniform(0, 2, (T, hc)).astype(np.float32))).to(device).to(torch.bfloat16)
    before = host(streams)
    target = streams if in_place else torch.empty_like(streams)
    y = layer.forward(x, inject=(streams, weights, target))
    torch.cuda.synchronize()
    want = go.inject(before, host(y), host(weights))
    np.testing.assert_array_equal(host(target), want)
    # the plain call afterwards leaves no injection behind
    y2 = layer.forward(x)
    torch.cuda.synchronize()
    assert torch.equal(y2.view(torch.int16), y.view(torch.int16))
    np.testing.assert_array_equal(host(target), want)


@pytest.mark.parametrize("hidden,inter", [(256, 640), (1280, 320), (256, 1280)])
@pytest.mark.parametrize("T,dtype", [(1, torch.bfloat16), (5, torch.bfloat16), (3, torch.float32)])
def test_injection_over_folded_down_rows_is_exact(device, hidden, inter, T, dtype):
    """The injecting down instances of rows a quarter over a power of two (10, 20 and 40 groups): the plain call's
    output, and its injection, in bf16 to the bit."""
    hc = 3
    spec = synth.LayerSpec("glue_folded", hidden, inter, 16, 4, inter, 1)
    layer = assemble.build_layer(spec, SEED, device, dense=True)
    rng = np.random.default_rng(SEED + inter + T)
    x = assemble.tokens_tensor(spec, SEED, device, T, stream=9).to(dtype)
    streams = torch.from_numpy(mo.bf16r(rng.normal(0, 1, (T, hc * hidden)).astype(np.float32))).to(device).to(dtype)
    weights = torch.from_numpy(mo.bf16r(rng.uniform(0, 2, (T, hc)).astype(np.float32))).to(device).to(dtype)
    plain = layer.forward(x).clone()
    target = torch.empty_like(streams)
    y = layer.forward(x, inject=(streams, weights, target))
    torch.cuda.synchronize()
    assert torch.equal(y, plain)
    if dtype == torch.bfloat16:
        np.testing.assert_array_equal(host(target), go.inject(host(streams), host(y), host(weights)))
    else:
        # the product may be fused into the sum: its own rounding is then missing, half a step of the product, which
        # can move the sum's rounding by one more half step
        product = y.unsqueeze(1) * weights.unsqueeze(2)
        want = streams.view(T, hc, hidden) + product
        bound = 2.0 ** -24 * product.abs() + 2.0 ** -23 * want.abs()
        assert bool(((target.view(T, hc, hidden) - want).abs() <= bound).all())


def test_mlp_branch_matches_the_oracle_chain(device):
    hc, T = 4, 2
    spec = SMALL
    H = spec.hidden
    rng = np.random.default_rng(SEED + 7)
    parts = _hyper_np(rng, hc, H, 32)
    hyper = _hyper_dev(parts, hc, device)
    layer = assemble.build_layer(spec, SEED, device, dense=True)
    x, xd = _streams(rng, T, hc * H, device)
    out = mlp_branch(hyper, layer, xd)
    torch.cuda.synchronize()
    mixed, weights, _ = go.hyper_mix(x, *parts, hc, 1e-6)
    y = mo.moe_layer(mixed, synth.numpy_layer(spec, SEED, 0, materialise=True), "bf16")["output"]
    want = go.inject(x, y, weights)
    assert_close(host(out), want, "mlp branch")
    # in place on the streams
    again = xd.clone()
    mlp_branch(hyper, layer, again, out=again)
    torch.cuda.synchronize()
    assert torch.equal(again.view(torch.int16), out.view(torch.int16))
