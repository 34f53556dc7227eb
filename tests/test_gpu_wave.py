"""GPU tests of the wave kernels (csrc/flare_wave.h): the chunked forward on fp32 matrix
products, for fp32 inputs and for the banks without an instance of the 16-bit kernels.

The oracle is the fp64 tokenwise recurrence.  Bars: fp32 and every state |a - b| <= 1e-5 +
1e-4 |b| (sums of at most N = 150 fp32 terms of size O(1): N 2^-24 = 9e-6), 16-bit outputs
one rounding on top (2^-8 bf16, 2^-11 fp16, of |b|)."""
import numpy as np
import pytest
import torch

import flare_oracle as O
from _util import seeded, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROUND = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _close(a, b, dtype, what):
    a, b = to_np(a).astype(np.float64), np.asarray(b, dtype=np.float64)
    bound = 1e-5 + (1e-4 + ROUND[dtype]) * np.abs(b)
    worst = float((np.abs(a - b) - bound).max())
    assert np.isfinite(a).all() and worst <= 0, f"{what}: past the bar by {worst:.3e}"


def _prefill(q, k, v, **kw):
    from causal_flare import flare_autoregressive_prefill_triton
    put = lambda t: {n: x.to(DEV) for n, x in t.items()} if isinstance(t, dict) else t.to(DEV)
    kw = {n: put(t) for n, t in kw.items() if t is not None}
    return flare_autoregressive_prefill_triton(q.to(DEV), k.to(DEV), v.to(DEV), **kw)


# one per head dim and latent-tile count; latents and lengths off every tile edge
SHAPES = [(5, 16, 3), (16, 16, 16), (33, 32, 17), (64, 32, 150), (80, 32, 33), (256, 32, 40), (40, 48, 65),
          (64, 64, 1), (96, 64, 95), (192, 96, 50), (256, 128, 47)]


@pytest.mark.parametrize("M,D,N", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", ["plain", "state_mask", "separate"])
def test_wave_prefill(M, D, N, dtype, form):
    print("CASE wave_prefill", M, D, N, dtype, form, flush=True)
    if (M, D) == (256, 128) and dtype is not torch.float32:
        pytest.skip("this bank has a 16-bit kernel")
    B, H = 2, 2
    q, k, v = seeded(31 * M + D, B, N, H, M, D, D, dtype, q_std=D ** -0.5)
    g = torch.Generator().manual_seed(M + D)
    state = mask = qd = kd = None
    if form == "state_mask":
        state = {"m": torch.randn(B, H, M, generator=g), "d": 1.0 + torch.rand(B, H, M, generator=g),
                 "u": torch.randn(B, H, M, D, generator=g)}
        mask = (torch.rand(B, N, generator=g) < 0.7).to(torch.int32)
        mask[0, : min(N, 18)] = 0          # a whole tile of masked tokens, and a masked start
    if form == "separate":
        qd = torch.randn(B, N, H, D, generator=g).to(dtype)
        kd = (torch.randn(H, M, D, generator=g) * D ** -0.5).to(dtype)
    y, st = _prefill(q, k, v, state=state, attention_mask=mask, Q_dec=qd, K_dec=kd)
    ref, rst = O.brute_ar_state(q, k, v, state=state, scale=1.0, attention_mask=mask, Q_dec=qd, K_dec=kd)
    _close(y, ref, dtype, "y")
    for n in ("m", "d", "u"):
        _close(st[n], rst[n], torch.float32, n)


@pytest.mark.parametrize("M,D,dtype", [(64, 32, torch.bfloat16), (96, 64, torch.float16), (128, 64, torch.float32),
                                       (40, 16, torch.float32)])
def test_wave_score_jumps_and_infinite_values(M, D, dtype):
    """Scores that rise by 90 to 400 nats inside a tile (at the start of the sequence, mid-tile
    and on a tile's last token) and, apart from them, an infinite value row: the tokens before
    each keep their exact outputs, as the tokenwise recurrence gives them."""
    print("CASE wave_jumps", M, D, dtype, flush=True)
    B, N, H = 1, 70, 2
    q, k, v = seeded(77 + M, B, N, H, M, D, D, dtype, q_std=D ** -0.5)
    kj = k.clone()
    for t, nats, lat in ((3, 90.0, 1), (21, 200.0, 7), (47, 400.0, 12)):
        for h in range(H):
            row = q[h, lat].float()
            kj[0, t, h] = (row * (nats / row.square().sum())).to(dtype)
    y, st = _prefill(q, kj, v)
    ref, rst = O.brute_ar_state(q, kj, v, scale=1.0)
    # a score of 400 nats carries |s| 2^-24 = 2.4e-5 of its fp32 sum into e^s
    a, b = to_np(y).astype(np.float64), np.asarray(ref)
    assert np.isfinite(a).all()
    assert (np.abs(a - b) - (1e-4 + (2e-4 + ROUND[dtype]) * np.abs(b))).max() <= 0
    vi = v.clone()
    vi[0, 37, 0, 5] = float("inf")
    y, _ = _prefill(q, k, vi)
    clean, _ = _prefill(q, k, v)
    assert torch.equal(y[0, :32], clean[0, :32]) and torch.equal(y[0, :, 1], clean[0, :, 1])
    _close(y[0, 32:37, 0], to_np(clean[0, 32:37, 0]), dtype, "tokens of the tile before the infinite one")
    assert not torch.isfinite(y[0, 37:, 0, 5]).any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wave_unaligned_inputs(dtype):
    """Inputs that start off a 16-byte boundary run on the tokenwise kernels, with the same
    results."""
    print("CASE wave_unaligned", dtype, flush=True)
    B, N, H, M, D = 1, 40, 2, 64, 32
    q, k, v = seeded(5, B, N, H, M, D, D, dtype, q_std=D ** -0.5)
    y0, _ = _prefill(q, k, v)

    def shifted(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
        buf[1:] = t.reshape(-1).to(DEV)
        return buf[1:].view(t.shape)

    from causal_flare import flare_autoregressive_prefill_triton
    for which in range(3):
        args = [t.to(DEV) for t in (q, k, v)]
        args[which] = shifted((q, k, v)[which])
        assert args[which].data_ptr() % 16 != 0
        y, _ = flare_autoregressive_prefill_triton(*args)
        _close(y, to_np(y0), dtype, f"input {which} unaligned")


def _grads(q, k, v, g, qd=None, kd=None, chunk=None):
    from causal_flare import flare_autoregressive_triton
    leaves = {n: t.to(DEV).requires_grad_(True) for n, t in (("q", q), ("k", k), ("v", v), ("qd", qd), ("kd", kd))
              if t is not None}
    y = flare_autoregressive_triton(leaves["q"], leaves["k"], leaves["v"], Q_dec=leaves.get("qd"), K_dec=leaves.get("kd"))
    y.backward(g.to(DEV))
    return {n: t.grad for n, t in leaves.items()}


# the backward's bars (test_gpu_backward.py): fp32 1e-4 of the largest entry, 16-bit the rounding
# of the results and of the saved output in g.y (2e-2 bf16, an eighth of it fp16).  With one token
# gz - g.y cancels to a true gradient of 0 and leaves 2^-24 |g| |v| (16 at D = 16: 1e-6) against
# the floor of 1e-2: 1e-4 more in fp32.
GRAD_BAR = {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 2.5e-3}


def _check_grads(got, refs, dtype, what, one_token=False):
    bar = GRAD_BAR[dtype] + (1e-4 if one_token and dtype is torch.float32 else 0.0)
    for (n, x), r in zip(got.items(), refs):
        a, r = to_np(x).astype(np.float64), np.asarray(r)
        assert np.isfinite(a).all(), f"{what} d{n}: not finite"
        err = np.abs(a - r).max() / max(np.abs(r).max(), 1e-2)
        assert err <= bar, f"{what} d{n}: {err:.3e}"


@pytest.mark.parametrize("M,D,N", [(16, 16, 1), (48, 32, 70), (64, 32, 150), (16, 48, 33), (64, 64, 200), (96, 96, 47),
                                   (128, 64, 135), (192, 128, 129), (256, 128, 80)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sep", ["", "q", "k", "qk"])
def test_wave_backward(M, D, N, dtype, sep):
    """Off every tile edge: latents that fill no wave, partial token tiles, several chunks
    (64 tokens each at these sizes), each decoder-sharing mode."""
    print("CASE wave_backward", M, D, N, dtype, sep, flush=True)
    B, H = 2, 2
    q, k, v = seeded(7 * M + D, B, N, H, M, D, D, dtype)
    gen = torch.Generator().manual_seed(M)
    g = torch.randn(B, N, H, D, generator=gen).to(dtype)
    qd = torch.randn(B, N, H, D, generator=gen).to(dtype) if "q" in sep else None
    kd = torch.randn(H, M, D, generator=gen).to(dtype) if "k" in sep else None
    got = _grads(q, k, v, g, qd, kd)
    refs = O.ar_grads(q, k, v, g, Q_dec=qd, K_dec=kd)
    refs = list(refs[:3]) + [r for r, t in zip(refs[3:], (qd, kd)) if t is not None]
    _check_grads(got, refs, dtype, f"M={M} D={D} N={N} sep={sep}", one_token=N == 1)


# dV is a sum without cancellation of fp32 factors, so a share of about 2 |error| / ulp of its
# entries does not come out as the rounded exact value.  fp32 sums here end within some 2^-22 of the
# value: 0.1% of fp16's ulp of 2^-10, an eighth of that in bf16; factors of 16 to 17 bits 0.8 to
# 1.5%.  The 16-bit kernels' own banks, whose states were two bf16 parts before the walks, had 0.75%
# (0.5% in 33 tokens, where the sums inside a tile, then in fp32, count for more).
@pytest.mark.parametrize("M,D,dtype,share", [(64, 32, torch.float16, 4e-3), (48, 48, torch.float16, 4e-3),
                                             (96, 64, torch.float16, 4e-3), (208, 96, torch.float16, 4e-3),
                                             (192, 128, torch.float16, 4e-3), (64, 32, torch.bfloat16, 1e-3),
                                             (128, 64, torch.float16, 6.5e-3), (256, 128, torch.float16, 6.5e-3)])
@pytest.mark.parametrize("block,N,H", [(0, 512, 2), (64, 512, 2), (0, 40, 16)])
def test_wave_backward_keeps_fp32_factors(M, D, dtype, share, block, N, H):
    """What the walks hold in fp32 enters their products whole: dV is the rounded exact value up to
    fp32 sums (one wave to a full workgroup, one X tile in LDS and two, both layers)."""
    from causal_flare import flare_semi_autoregressive_trition
    print("CASE wave_fp32_factors", M, D, dtype, block, N, flush=True)
    B = 1
    q, k, v = seeded(3 * M + D, B, N, H, M, D, D, dtype)
    g = torch.randn(B, N, H, D, generator=torch.Generator().manual_seed(M)).to(dtype)
    if block:
        leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
        y, _ = flare_semi_autoregressive_trition(*leaves, block_size=block, chunk_size=16)
        y.backward(g.to(DEV))
        dv, ref = leaves[2].grad, O.semi_grads(q, k, v, g, block)[2]
    else:
        dv, ref = _grads(q, k, v, g)["v"], O.ar_grads(q, k, v, g)[2]
    wrong = float((dv.cpu() != torch.from_numpy(np.asarray(ref)).to(dtype)).double().mean())
    assert wrong <= min(share, 5.5e-3 if N < 64 else share), f"{wrong:.4f} of dV is not the rounded value"


@pytest.mark.parametrize("M,D,dtype", [(64, 32, torch.float32), (128, 64, torch.float32), (128, 64, torch.bfloat16)])
def test_wave_backward_jumps_and_infinite_gradient(M, D, dtype):
    """Scores that rise by 90 to 400 nats inside a tile, at the start, mid-tile and on a chunk's
    last token: those tiles are walked token by token.  An infinite dY entry reaches dV of its
    own and earlier tokens only."""
    print("CASE wave_backward_jumps", M, D, dtype, flush=True)
    B, N, H = 1, 150, 2
    q, k, v = seeded(13 + M, B, N, H, M, D, D, dtype, q_std=D ** -0.5)
    k = k * 0.5
    for t, nats, lat in ((3, 90.0, 1), (63, 200.0, 7), (105, 400.0, 12)):
        for h in range(H):
            row = q[h, lat].float()
            k[0, t, h] = (row * (nats * D ** 0.5 / row.square().sum())).to(dtype)
    gen = torch.Generator().manual_seed(M)
    g = torch.randn(B, N, H, D, generator=gen).to(dtype)
    got = _grads(q, k, v, g)
    refs = O.ar_grads(q, k, v, g)
    if dtype is torch.float32:
        # (16-bit: da cancels where the softmax peaks, from the rounded output; dV has no such term)
        _check_grads(got, refs[:3], dtype, "jumps")
    _check_grads({"v": got["v"]}, refs[2:3], dtype, "jumps")
    q, k, v = seeded(14 + M, B, N, H, M, D, D, dtype)
    gi = g.clone()
    gi[0, 37, 0, 5] = float("inf")
    clean, inf = _grads(q, k, v, g)["v"], _grads(q, k, v, gi)["v"]
    assert torch.isfinite(inf[0, 38:]).all()
    _check_grads({"v": inf[0, 38:]}, [to_np(clean[0, 38:])], dtype, "past the infinite entry")
    assert not torch.isfinite(inf[0, :38, 0, 5]).any()


@pytest.mark.parametrize("M,D,N,block", [(16, 16, 48, 16), (48, 32, 96, 32), (64, 32, 240, 48), (16, 48, 64, 64),
                                         (96, 64, 192, 96), (128, 64, 256, 64), (192, 96, 128, 32), (256, 128, 96, 48)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sep", ["", "q", "k", "qk"])
def test_wave_semi_backward(M, D, N, block, dtype, sep):
    """The block-causal walks: one block, several blocks a chunk, several chunks, blocks that are
    no power of two, latents that fill no wave, each decoder-sharing mode."""
    print("CASE wave_semi_backward", M, D, N, block, dtype, sep, flush=True)
    from causal_flare import flare_semi_autoregressive_trition
    B, H = 2, 2
    q, k, v = seeded(5 * M + D, B, N, H, M, D, D, dtype)
    gen = torch.Generator().manual_seed(M)
    g = torch.randn(B, N, H, D, generator=gen).to(dtype)
    qd = torch.randn(B, N, H, D, generator=gen).to(dtype) if "q" in sep else None
    kd = torch.randn(H, M, D, generator=gen).to(dtype) if "k" in sep else None
    leaves = {n: t.to(DEV).requires_grad_(True) for n, t in (("q", q), ("k", k), ("v", v), ("qd", qd), ("kd", kd))
              if t is not None}
    y, _ = flare_semi_autoregressive_trition(leaves["q"], leaves["k"], leaves["v"], block_size=block, chunk_size=16,
                                             Q_dec=leaves.get("qd"), K_dec=leaves.get("kd"))
    y.backward(g.to(DEV))
    refs = O.semi_grads(q, k, v, g, block, Q_dec=qd, K_dec=kd)
    refs = list(refs[:3]) + [r for r, t in zip(refs[3:], (qd, kd)) if t is not None]
    _check_grads({n: t.grad for n, t in leaves.items()}, refs, dtype, f"M={M} D={D} N={N} block={block} sep={sep}")


@pytest.mark.parametrize("M,D,dtype", [(64, 32, torch.float32), (96, 64, torch.float16), (128, 64, torch.bfloat16),
                                       (256, 128, torch.bfloat16), (256, 64, torch.float16), (40, 80, torch.float32)])
@pytest.mark.parametrize("sep", [False, True])
def test_all_kept_mask_is_no_mask(M, D, dtype, sep):
    """A mask that keeps every token is not looked for on the host at these sizes: its launches
    have to give what the unmasked ones do, also where a value row is infinite."""
    from causal_flare import flare_autoregressive_prefill_triton
    print("CASE all_kept", M, D, dtype, sep, flush=True)
    B, N, H = 2, 209, 2
    q, k, v = seeded(31 + M, B, N, H, M, D, D, dtype, q_std=D ** -0.5)
    dec = {}
    if sep:
        qd, kd, _ = seeded(32 + M, B, N, H, M, D, D, dtype, q_std=D ** -0.5)
        dec = dict(Q_dec=kd.to(DEV), K_dec=qd.to(DEV))
    v[1, 150, 0, 3] = float("inf")
    args = [t.to(DEV) for t in (q, k, v)]
    y, st = flare_autoregressive_prefill_triton(*args, **dec)
    for mask in (torch.ones(B, N, dtype=torch.bool), torch.full((B, N), 2, dtype=torch.int64, device=DEV)):
        ym, sm = flare_autoregressive_prefill_triton(*args, **dec, attention_mask=mask)
        a, b = to_np(ym).astype(np.float64), to_np(y).astype(np.float64)
        same = np.isfinite(b)
        assert np.array_equal(np.isfinite(a), same)
        _close(torch.from_numpy(a[same]), b[same], dtype, "y")
        for n in ("m", "d"):
            _close(sm[n], to_np(st[n]), torch.float32, n)


@pytest.mark.parametrize("M,D,N,block", [(1, 16, 16, 16), (40, 32, 96, 32), (96, 48, 144, 48), (192, 64, 64, 64),
                                         (100, 96, 160, 32), (256, 96, 96, 96), (17, 128, 128, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sep", [False, True])
def test_wave_semi_forward(M, D, N, block, dtype, sep):
    """The block-causal readout: one and several blocks, one and two token tiles a wave, a last
    workgroup with idle waves, latents that fill no tile, both decoder modes; then inputs off a
    16-byte boundary, which run on the kernel without matrix products."""
    from causal_flare import flare_semi_autoregressive_trition
    print("CASE wave_semi_forward", M, D, N, block, dtype, sep, flush=True)
    B, H = 2, 3
    q, k, v = seeded(7 * M + D, B, N, H, M, D, D, dtype, q_std=D ** -0.5)
    gen = torch.Generator().manual_seed(M)
    qd = torch.randn(B, N, H, D, generator=gen).to(dtype) if sep else None
    kd = (torch.randn(H, M, D, generator=gen) * D ** -0.5).to(dtype) if sep else None
    ref = np.asarray(O.brute_semi_ar(q, k, v, block, scale=1.0, Q_dec=qd, K_dec=kd))
    put = lambda t: None if t is None else t.to(DEV)

    def shifted(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
        buf[1:] = t.reshape(-1).to(DEV)
        return buf[1:].view(t.shape)

    for args in ((put(q), put(k)), (put(q), shifted(k))):
        y, _ = flare_semi_autoregressive_trition(*args, put(v), block_size=block, chunk_size=16, scale=1.0,
                                                 Q_dec=put(qd), K_dec=put(kd))
        _close(y, ref, dtype, f"y M={M} D={D} N={N} block={block} sep={sep}")


def test_wave_backward_most_heads():
    """The most (sequence, head) pairs a grid holds, of a 256 x 128 bank: more than 2^31 sums of
    the scan over chunks.  The last sequences' gradients are those of the same sequences alone."""
    from causal_flare import flare_autoregressive_triton
    print("CASE wave_backward_most_heads", flush=True)
    B, N, H, M, D = 8131, 1, 8, 256, 128             # 65,048 pairs
    assert B * H * M * (D + 1) > 2 ** 31 and B * H < 65536
    gen = torch.Generator(device=DEV).manual_seed(3)
    rnd = lambda *s: torch.randn(s, generator=gen, device=DEV, dtype=torch.bfloat16)
    q, k, v, g = rnd(H, M, D), rnd(B, N, H, D), rnd(B, N, H, D), rnd(B, N, H, D)

    def grads(rows):
        kk, vv = k[rows].clone().requires_grad_(True), v[rows].clone().requires_grad_(True)
        return torch.autograd.grad(flare_autoregressive_triton(q, kk, vv), (kk, vv), g[rows])

    for whole, alone in zip(grads(slice(None)), grads(slice(B - 3, B))):
        assert torch.equal(whole[-3:], alone)
    torch.cuda.empty_cache()                         # (some 40 GB of workspace)


@pytest.mark.parametrize("B,N,H,M,D,block", [(3, 1920, 16, 96, 32, 128), (1, 960, 8, 64, 32, 64), (2, 6336, 4, 64, 128, 64),
                                             (1, 16, 1, 16, 16, 16)])
@pytest.mark.parametrize("layer", ["token", "block"])
def test_backward_of_own_decoder_weights_walks(B, N, H, M, D, block, layer):
    """Decoder weights of their own, chunks of one block: the sizes asked for hold the walks'
    arrays, and the walks are what runs."""
    from torch.profiler import ProfilerActivity, profile
    from causal_flare import flare_autoregressive_triton, flare_semi_autoregressive_trition
    print("CASE backward_route", B, N, H, M, D, block, layer, flush=True)
    gen = torch.Generator(device=DEV).manual_seed(M)
    rnd = lambda *s: torch.randn(s, generator=gen, device=DEV, dtype=torch.bfloat16).requires_grad_(True)
    q, k, v, qd, kd = rnd(H, M, D), rnd(B, N, H, D), rnd(B, N, H, D), rnd(B, N, H, D), rnd(H, M, D)
    if layer == "token":
        y = flare_autoregressive_triton(q, k, v, Q_dec=qd, K_dec=kd)
    else:
        y, _ = flare_semi_autoregressive_trition(q, k, v, block_size=block, chunk_size=16, Q_dec=qd, K_dec=kd)
    g = torch.ones_like(y)
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        torch.autograd.grad(y, (q, k, v, qd, kd), g)
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    walk = "wave_ds_kernel" if layer == "token" else "wave_semi_ds_kernel"
    assert walk in names and "wave_rows_kernel" in names and "wave_cols_kernel" in names, names


@pytest.mark.parametrize("M,D,dtype", [(64, 32, torch.bfloat16), (48, 48, torch.float16), (128, 64, torch.bfloat16),
                                       (80, 128, torch.float16), (256, 128, torch.bfloat16), (48, 32, torch.float32),
                                       (64, 96, torch.float32)])
@pytest.mark.parametrize("block", [0, 48])
def test_wave_backward_infinite_gradients(M, D, dtype, block):
    """Infinite dY entries make dV of their column infinite, with their sign, in their own and all
    earlier tokens (of the block-causal layer: blocks); both signs give NaN.  Other columns are as
    without them."""
    from causal_flare import flare_semi_autoregressive_trition
    print("CASE wave_infinite_gradients", M, D, dtype, block, flush=True)
    B, N, H = 1, 240, 2
    q, k, v = seeded(9 * M + D, B, N, H, M, D, D, dtype)
    g = torch.randn(B, N, H, D, generator=torch.Generator().manual_seed(M)).to(dtype)

    def dv(g):
        leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
        if block:
            y, _ = flare_semi_autoregressive_trition(*leaves, block_size=block, chunk_size=16)
        else:
            from causal_flare import flare_autoregressive_triton
            y = flare_autoregressive_triton(*leaves)
        y.backward(g.to(DEV))
        return leaves[2].grad.float().cpu()

    inf = float("inf")
    entries = [(37, 0, 5, inf), (150, 0, 5, inf), (201, 0, D - 1, -inf), (3, 0, D - 1, inf), (239, 1, 0, -inf)]
    gi = g.clone()
    want = dv(g)
    wild = torch.zeros(N, H, D, dtype=torch.bool)
    for t, h, d, x in entries:
        gi[0, t, h, d] = x
        last = (t // block + 1) * block if block else t + 1
        new = torch.where(wild[:last, h, d], want[0, :last, h, d] + x, torch.full((last,), x))     # (inf - inf: NaN)
        want[0, :last, h, d] = new
        wild[:last, h, d] = True
    got = dv(gi)
    odd = wild[None]
    assert torch.equal(torch.nan_to_num(got[odd], nan=7.0), torch.nan_to_num(want[odd], nan=7.0))
    _check_grads({"v": got[~odd]}, [want[~odd].double().numpy()], dtype, "other columns")


@pytest.mark.parametrize("M,D", [(40, 32), (17, 64), (64, 48)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wave_semi_forward_infinite_value(M, D, dtype):
    """An infinite value is infinite in y of its column from its block on, also for a bank that ends
    inside a tile of latents; everything else is as without it."""
    from causal_flare import flare_semi_autoregressive_trition
    print("CASE wave_semi_infinite_value", M, D, dtype, flush=True)
    B, N, H, block = 1, 192, 2, 48
    q, k, v = (t.to(DEV) for t in seeded(11 * M + D, B, N, H, M, D, D, dtype, q_std=D ** -0.5))
    vi = v.clone()
    vi[0, 100, 1, 7] = float("-inf")
    y, yi = (flare_semi_autoregressive_trition(q, k, x, block_size=block, chunk_size=16, scale=1.0)[0] for x in (v, vi))
    assert torch.isneginf(yi[0, 96:, 1, 7]).all()
    yi[0, 96:, 1, 7] = y[0, 96:, 1, 7]
    assert torch.equal(yi, y)
