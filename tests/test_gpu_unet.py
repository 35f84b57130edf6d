"""The U-Net's matrix-core kernels against torch's CPU library, on the GPU.

Inputs and weights are rounded to bfloat16 first, so both sides see the same
values: bfloat16 products are exact in float32, and the kernels accumulate in
float32, so before the output's own rounding the two agree to float32 sums.
- forward (bias and ReLU fused): within bfloat16's rounding of the output;
- the input gradient: within bfloat16's rounding of the output;
- the weight gradient (float32 out): within 1e-4 relative L2;
- AdamW against torch.optim.AdamW over several steps: 1e-6 relative;
- the whole network against the oracle network (`oracle/unet.py`, float32
  throughout): the output within 3 % relative L2, every parameter gradient
  within 10 % relative L2 at a cosine above 0.99, the drift of bfloat16
  activations and gradients through fourteen layers.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from cuwave_amd import unet  # noqa: E402
from oracle import unet as O  # noqa: E402


def _bf(t: torch.Tensor) -> torch.Tensor:
    return t.to(torch.bfloat16).float()


def _rel(a: torch.Tensor, b: torch.Tensor) -> float:
    a, b = a.detach().float().cpu(), b.detach().float().cpu()
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("cin, cout, relu", [(16, 32, True), (32, 32, True), (64, 128, False),
                                             (128, 64, True), (128, 128, True)])
def test_a_convolution_and_its_gradients_match_the_library(cin, cout, relu):
    print(f"case conv3x3 {cin}->{cout} relu={relu}", flush=True)
    g = torch.Generator().manual_seed(cin * 1000 + cout)
    n, h, w = 2, 37, 41  # an odd size: tiles that run past the last pixel
    x = _bf(torch.randn(n, h, w, cin, generator=g))
    conv = unet.Conv3x3(cin, cout, relu)
    with torch.no_grad():
        conv.weight.copy_(_bf(conv.weight))
    xg = x.cuda().to(torch.bfloat16).requires_grad_(cin in (32, 64, 128))
    convg = conv.cuda()
    y = convg(xg)
    ref_x = x.clone().requires_grad_(True)
    ref_w = conv.weight.detach().cpu().clone().requires_grad_(True)
    ref_b = conv.bias.detach().cpu().clone().requires_grad_(True)
    ref = O.conv3x3(ref_x, ref_w, ref_b, relu)
    # within bfloat16's rounding of the output (relative 2^-8 per element)
    err = (y.detach().float().cpu() - ref.detach()).abs()
    assert float((err - ref.detach().abs() * 2.0**-8).max()) <= 1e-5
    dy = _bf(torch.randn(n, h, w, cout, generator=g))
    y.backward(dy.cuda().to(torch.bfloat16))
    ref.backward(dy)
    # the kernels take the gradient before the activation in bfloat16: the same
    # rounded values on the reference side give the weight gradient in float32
    mask = (y.float().cpu() > 0) if relu else torch.ones_like(dy, dtype=torch.bool)
    dpre = torch.where(mask, dy, torch.zeros_like(dy))
    dw_ref = torch.einsum("nhwo,nhwk->ok", dpre.double(),
                          torch.nn.functional.unfold(x.permute(0, 3, 1, 2).double(), 3, padding=1)
                          .reshape(n, cin, 9, h, w).permute(0, 3, 4, 2, 1).reshape(n, h, w, 9 * cin))
    assert _rel(convg.weight.grad, dw_ref.float()) < 1e-4
    assert _rel(convg.bias.grad, dpre.sum((0, 1, 2))) < 1e-5
    if xg.requires_grad:
        assert _rel(xg.grad, ref_x.grad) < 1e-2


def test_adamw_makes_torch_s_update():
    torch.manual_seed(0)
    p = torch.randn(1000)
    grads = [torch.randn(1000) for _ in range(5)]
    ours = p.clone().cuda()
    theirs = p.clone().requires_grad_(True)
    opt = unet.AdamW([ours.requires_grad_(True)], lr=1e-2, weight_decay=0.05)
    ref = torch.optim.AdamW([theirs], lr=1e-2, weight_decay=0.05)
    for g in grads:
        ours.grad = g.cuda()
        opt.step()
        theirs.grad = g.clone()
        ref.step()
    assert _rel(ours, theirs) < 1e-6


def test_the_network_matches_the_oracle_forward_and_backward():
    print("case unet 2x28x36", flush=True)
    torch.manual_seed(1)
    net = unet.UNet().cuda()
    with torch.no_grad():
        for p in net.parameters():
            p.copy_(_bf(p))
    x = torch.randn(2, 28, 36, 2)
    y = net(x.cuda())
    params = {k: v.detach().cpu().clone().requires_grad_(True) for k, v in net.named_parameters()}
    ref = O.unet(params, x, net.cin_k)
    assert y.shape == (2, 28, 36, 1)
    assert _rel(y, ref) < 3e-2
    target = torch.randn_like(ref)
    torch.mean((y - target.cuda()) ** 2).backward()
    torch.mean((ref - target) ** 2).backward()
    # each layer rounds its activations and the gradient it passes back to
    # bfloat16; the deepest parameters see that fourteen times over
    for name, p in net.named_parameters():
        a, b = p.grad.detach().float().cpu().ravel(), params[name].grad.ravel()
        rel, cos = _rel(a, b), float(a @ b / (a.norm() * b.norm()))
        print(f"{name}: rel {rel:.3e} cos {cos:.6f}", flush=True)
        assert rel < 1e-1 and cos > 0.99, name
    count = sum(p.numel() for p in net.parameters())
    assert 440_000 < count < 500_000


def test_training_fits_a_target_on_the_gpu():
    torch.manual_seed(0)
    x = torch.randn(4, 16, 16, 2).cuda()
    y = 0.5 * x[..., :1] - 0.25 * x[..., 1:]
    net = unet.UNet(base=32).cuda()
    opt = unet.AdamW(net.parameters(), lr=3e-3, weight_decay=1e-4)
    losses = []
    for _ in range(60):
        opt.zero_grad()
        loss = torch.mean((net(x) - y) ** 2)
        loss.backward()
        opt.step()
        losses.append(loss.item())
    assert np.isfinite(losses).all()
    assert losses[-1] < 0.3 * losses[0]


@pytest.mark.parametrize("n, h, w, cin, cout", [
    (1, 1, 1, 32, 32),      # smaller than any tile
    (3, 8, 32, 32, 64),     # whole tiles of pixels
    (2, 7, 31, 64, 32),     # one short of a tile
    (1, 9, 65, 16, 128),    # one past a tile, half a channel chunk
    (2, 17, 33, 48, 64),    # a channel count of the 16-channel chunks only
    (1, 40, 130, 96, 128),  # several tiles and chunks each way
    (700, 3, 5, 32, 64),    # small images: the flat kernels', runs of pixels across them
    (400, 4, 6, 128, 128),
    (1, 1200, 2, 64, 32),
])
def test_a_convolution_at_its_tiles_edges(n, h, w, cin, cout):
    print(f"case conv3x3 {n}x{h}x{w} {cin}->{cout}", flush=True)
    g = torch.Generator().manual_seed(h * 100 + w)
    x = _bf(torch.randn(n, h, w, cin, generator=g))
    conv = unet.Conv3x3(cin, cout, True)
    with torch.no_grad():
        conv.weight.copy_(_bf(conv.weight))
    ref_x = x.clone().double().requires_grad_(True)
    ref_w = conv.weight.detach().clone().double().requires_grad_(True)
    ref_b = conv.bias.detach().clone().double().requires_grad_(True)
    ref = O.conv3x3(ref_x, ref_w, ref_b, True)
    conv = conv.cuda()
    xg = x.cuda().to(torch.bfloat16).requires_grad_(cin in (32, 64, 128))
    y = conv(xg)
    # half an ulp of bfloat16 (2^-9) and the float32 sums of 9 cin terms
    err = (y.detach().double().cpu() - ref.detach()).abs()
    assert float((err - ref.detach().abs() * 2.0**-8).max()) <= 1e-5
    dy = _bf(torch.randn(n, h, w, cout, generator=g))
    # outputs whose sign the rounding could turn carry no gradient
    dy = torch.where(ref.detach().abs() < 1e-4, torch.zeros_like(dy), dy)
    y.backward(dy.cuda().to(torch.bfloat16))
    ref.backward(dy.double())
    assert _rel(conv.weight.grad, ref_w.grad) < 1e-4
    assert _rel(conv.bias.grad, ref_b.grad) < 1e-5
    if xg.requires_grad:  # bfloat16 outputs: 2^-9 relative each
        assert _rel(xg.grad, ref_x.grad) < 4e-3


@pytest.mark.parametrize("shape, outputs", [((1, 1, 1), 1), ((1, 7, 9), 2), ((2, 8, 8), 3),
                                            ((3, 61, 67), 4), ((4, 260, 300), 1)])
def test_the_output_layer_and_its_gradients(shape, outputs):
    print(f"case head {shape} outputs={outputs}", flush=True)
    g = torch.Generator().manual_seed(outputs)
    x = _bf(torch.randn(*shape, 32, generator=g))
    w, b = torch.randn(32, outputs, generator=g), torch.randn(outputs, generator=g)
    dy = torch.randn(*shape, outputs, generator=g)
    ref = [t.double().requires_grad_(True) for t in (x, w, b)]
    out = ref[0] @ ref[1] + ref[2]
    out.backward(dy.double())
    ours = [t.cuda().requires_grad_(True) for t in (x.bfloat16(), w, b)]
    y = unet._Head.apply(*ours)
    y.backward(dy.cuda())
    # float32 sums of 32 terms, then of the pixels in slices; dx rounded to bfloat16
    assert _rel(y, out) < 1e-6
    assert _rel(ours[1].grad, ref[1].grad) < 1e-5
    assert _rel(ours[2].grad, ref[2].grad) < 1e-5
    assert _rel(ours[0].grad, ref[0].grad) < 4e-3


def _summed(x, w, taps_first):
    """The convolution with one product a 16-channel group (the others are zero), each
    added in float32: tap by tap, or group by group."""
    n, h, wd, cin = x.shape
    cout = w.shape[0]
    wide = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    wk = w.reshape(cout, 9, cin)
    acc = torch.zeros(n, h, wd, cout)
    pairs = [(t, c) for t in range(9) for c in range(0, cin, 16)]
    for t, c in pairs if taps_first else sorted(pairs, key=lambda p: p[1]):
        at = wide[:, t // 3:t // 3 + h, t % 3:t % 3 + wd, c:c + 16]
        term = at[..., None, :] * wk[:, t, c:c + 16]  # exact: eight bits by eight
        acc = acc + term.sum(-1)                      # one of the sixteen is not zero
    return acc


@pytest.mark.parametrize("cin, cout, n, h, w", [
    *((*c, 2, 11, 45) for c in ((16, 32), (32, 32), (48, 64), (64, 64), (64, 128), (128, 64),
                                (128, 128))),
    # the flat kernel's: many small images, and more than 128 channels
    (32, 128, 1100, 2, 3), (64, 64, 600, 3, 5), (128, 32, 300, 5, 6), (160, 32, 2, 11, 45),
])
def test_a_convolution_adds_its_terms_tap_by_tap(cin, cout, n, h, w):
    print(f"case order {n}x{h}x{w} {cin}->{cout}", flush=True)
    g = torch.Generator().manual_seed(cin + cout)

    def halves(*shape):  # products in quarters: a sum's rounding needs two bits below it
        return torch.randint(-8, 9, shape, generator=g) * 0.5

    keep = torch.zeros(cin, dtype=torch.bool)
    keep[[c + (c // 16) % 16 for c in range(0, cin, 16)]] = True
    x = halves(n, h, w, cin) * keep
    weight = halves(cout, 9, cin) * keep
    # a large term at the first tap and its negative at the last: every sum between is
    # rounded to whole numbers, so the order of the others is in the result
    x[..., 0] = 4096.0
    weight[..., 0] = 0.0
    weight[:, 0, 0], weight[:, 8, 0] = 2048.0, -2048.0
    weight = weight.reshape(cout, 9 * cin)
    ref, other = (_summed(x, weight, first) for first in (True, False))
    if cin > 16 and h > 8:  # in a small image most nodes miss one of the two
        assert float((ref.bfloat16() != other.bfloat16()).float().mean()) > 0.1
    conv = unet.Conv3x3(cin, cout, False).cuda()
    with torch.no_grad():
        conv.weight.copy_(weight)
        conv.bias.zero_()
        y = conv(x.cuda().bfloat16())
    # the same additions in the same order: the same bits
    torch.testing.assert_close(y.cpu(), ref.bfloat16(), rtol=0, atol=0)


@pytest.mark.parametrize("w", [57, 64, 70, 95])  # the last column at places of a run, a strip
@pytest.mark.parametrize("cin, cout", [(32, 32), (64, 128)])
def test_an_infinity_in_the_last_column_stays_in_its_taps(w, cin, cout):
    print(f"case infinity {w} {cin}->{cout}", flush=True)
    g = torch.Generator().manual_seed(w)
    x = _bf(torch.randn(2, 40, w, cin, generator=g))
    dy = _bf(torch.randn(2, 40, w, cout, generator=g))
    conv = unet.Conv3x3(cin, cout, False)
    ref_w = conv.weight.detach().clone().double().requires_grad_(True)
    O.conv3x3(x.double(), ref_w, torch.zeros(cout).double(), False).backward(dy.double())
    x[1, 17, w - 1, 5] = float("inf")
    conv = conv.cuda()
    conv(x.cuda().bfloat16()).backward(dy.cuda().bfloat16())
    ours = conv.weight.grad.cpu().reshape(cout, 3, 3, cin)
    met = torch.zeros(3, 3, cin, dtype=torch.bool)
    met[:, 1:, 5] = True  # no pixel lies right of it: the taps from the left never read it
    assert bool(torch.isfinite(ours[:, ~met]).all())
    assert not bool(torch.isfinite(ours[:, met]).any())
    # the others are the sums without it (float32 sums of 2 x 40 x w products)
    theirs = ref_w.grad.reshape(cout, 3, 3, cin)
    assert _rel(ours[:, ~met], theirs[:, ~met]) < 1e-4


def test_the_output_layer_is_differentiated_again_as_the_product_is():
    print("case head, second derivatives and a tangent", flush=True)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 5, 7, 32, generator=g).bfloat16().cuda()
    w, t = torch.randn(2, 32, 3, generator=g).cuda()
    b = torch.randn(3, generator=g).cuda()

    def seconds(layer):
        p = [v.clone().requires_grad_(True) for v in (x, w, b)]
        (gw,) = torch.autograd.grad((layer(*p) ** 2).sum(), p[1], create_graph=True)
        return torch.autograd.grad((gw**2).sum(), p)

    ours = seconds(unet._Head.apply)
    for a, r in zip(ours, seconds(lambda x, w, b: x.float() @ w + b)):
        assert a.dtype == r.dtype
        # float32 products; the one at x rounded to bfloat16
        assert _rel(a, r) < (4e-3 if a.dtype == torch.bfloat16 else 1e-5)
    fwd = torch.autograd.forward_ad
    with fwd.dual_level():
        y = unet._Head.apply(x, fwd.make_dual(w, t), b)
        assert _rel(fwd.unpack_dual(y).tangent, x.float() @ t) < 1e-5


@pytest.mark.parametrize("how", ["plain", "autocast", "wide bias", "one bias for all", "vector"])
def test_the_output_layer_s_kernels_step_aside_for_other_products(how):
    print(f"case head {how}", flush=True)
    torch.manual_seed(5)
    net = unet.UNet(cout=2).cuda()
    if how == "wide bias":
        net.out_b = torch.nn.Parameter(net.out_b.detach().double())
    if how == "one bias for all":
        net.out_b = torch.nn.Parameter(net.out_b.detach()[:1])
    if how == "vector":
        net.out_w = torch.nn.Parameter(net.out_w.detach()[:, 0])
        net.out_b = torch.nn.Parameter(net.out_b.detach()[0])
    seen = []
    net.dec1.register_forward_hook(lambda module, args, out: seen.append(out))
    with torch.no_grad(), torch.autocast("cuda", torch.bfloat16, enabled=how == "autocast"):
        out = net(torch.randn(1, 8, 12, 2, device="cuda"))
        ref = seen[0].float() @ net.out_w + net.out_b
    assert out.dtype == ref.dtype
    if how == "plain":  # float32 sums of 32 terms
        assert _rel(out, ref) < 1e-6
    else:
        torch.testing.assert_close(out, ref, rtol=0, atol=0)


def test_a_gradient_that_starts_inside_another_tensor():
    print("case misaligned gradients", flush=True)
    g = torch.Generator().manual_seed(9)
    conv = unet.Conv3x3(32, 32).cuda()
    x = torch.randn(1, 9, 11, 32, generator=g).bfloat16().cuda()
    flat = torch.randn(x.numel() + 1, generator=g).bfloat16().cuda()
    w, b = torch.randn(32, 1, generator=g).cuda(), torch.zeros(1, device="cuda")
    results = []
    for dy in (flat[1:].clone(), flat[1:]):  # the second two bytes past an aligned address
        p = x.clone().requires_grad_(True)
        results.append(torch.autograd.grad(conv(p), [p, conv.weight, conv.bias],
                                           dy.view(x.shape)))
    results.append([unet._Head.apply(flat[1:].view(x.shape), w, b)])
    results.append([unet._Head.apply(flat[1:].clone().view(x.shape), w, b)])
    for a, c in (*zip(*results[:2]), *zip(*results[2:])):
        torch.testing.assert_close(a, c, rtol=0, atol=0)


@pytest.mark.parametrize("most", [1, 3, 40])
@pytest.mark.parametrize("n, h, w", [(2, 40, 70), (700, 3, 5)])  # the strips', the flat kernel's
def test_a_weight_gradient_keeps_to_the_slices_it_is_given(n, h, w, most, monkeypatch):
    print(f"case slices {n}x{h}x{w} most {most}", flush=True)
    g = torch.Generator().manual_seed(most)
    x = _bf(torch.randn(n, h, w, 32, generator=g))
    dy = _bf(torch.randn(n, h, w, 64, generator=g))
    conv = unet.Conv3x3(32, 64, False)
    ref_w = conv.weight.detach().clone().double().requires_grad_(True)
    O.conv3x3(x.double(), ref_w, torch.zeros(64).double(), False).backward(dy.double())
    monkeypatch.setattr(unet, "_splits", lambda *a: most)
    conv = conv.cuda()
    conv(x.cuda().bfloat16()).backward(dy.cuda().bfloat16())
    assert _rel(conv.weight.grad, ref_w.grad) < 1e-4
