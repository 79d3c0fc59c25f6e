"""The layer input of a hyper-connection block formed from the streams in one call (torch.ops.ks_mi355x.mhc_input)
against the same mathematics in 64 bits."""
import pytest
import torch

from kernelswift_amd import _lib
from kernelswift_amd.mhc import HyperConnection

pytestmark = pytest.mark.gpu


def _block(device, C, seed):
    g = torch.Generator().manual_seed(seed)
    hc = HyperConnection(C).requires_grad_(False)
    hc.phi.copy_(torch.randn(4 * C, 24, generator=g) * (4 * C) ** -0.5)
    hc.alpha.copy_(torch.rand(3, generator=g) + 0.5)
    hc.base.copy_(torch.randn(24, generator=g))
    return hc.to(device)


def _exact(hc, x):
    xf = x.flatten(1).double().cpu()
    phi, al, base = hc.phi.double().cpu(), hc.alpha.double().cpu(), hc.base.double().cpu()
    rn = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + hc.norm_eps)
    al24 = torch.cat([al[:1].expand(4), al[1:2].expand(4), al[2:].expand(16)])
    lg = al24 * ((xf @ phi) * rn) + base
    mag = al24.abs() * ((xf.abs() @ phi.abs()) * rn) + base.abs()
    h = (torch.sigmoid(lg[:, :4])[:, :, None] * x.double().cpu()).sum(1)
    return lg, mag, h


# token tiles of 16, 32 and 64 with remainders; one 32-wide step, ranges that end inside a wave, an odd step count
@pytest.mark.parametrize("N,C", [(1, 8), (15, 16), (16, 264), (17, 1032), (33, 520), (64, 4096), (65, 72), (200, 2056),
                                 (1000, 1024)])
def test_mhc_input_matches_64_bits(device, N, C):
    hc = _block(device, C, N + C)
    x = (torch.randn(N, 4, C, generator=torch.Generator().manual_seed(N)) * 3).bfloat16().to(device)
    print(f"[case] mhc_input N={N} C={C}", flush=True)
    h, post, res = _lib.torch_ops().mhc_input(x, hc.phi, hc.alpha, hc.base, hc.norm_eps)
    lg, mag, want = _exact(hc, x)
    got = torch.cat([post.cpu(), res.flatten(1).cpu()], 1).double()
    # fp32 sums: a wave's chain rounds 4 times per 32 products (at most 64 steps of the plans here), 9 grid units per
    # 8 products for the truncations, then at most 4 + 64 partials: below 2^-17 of the sum of magnitudes
    assert ((got - lg[:, 4:]).abs() <= 2.0 ** -17 * mag[:, 4:]).all()
    # h: four products with gates within 2^-17 mag of theirs, one bf16 rounding (8 significant bits: half an ulp is up to
    # 2^-8 of the value)
    hm = x.double().cpu().abs().sum(1)
    tol = 2.0 ** -8 * want.abs() + hm * (2.0 ** -17 * mag[:, :4].amax(1, keepdim=True) + 2.0 ** -21)
    assert ((h.double().cpu() - want).abs() <= tol * 1.01).all()


def test_mhc_input_special_values(device):
    C = 64
    hc = _block(device, C, 1)
    x = torch.randn(20, 4, C, generator=torch.Generator().manual_seed(2)).bfloat16()
    x[3] = 0.0
    x[5, 1, 7] = float("inf")
    x[6, 2, 9] = float("nan")
    x = x.to(device)
    ops = _lib.torch_ops()
    h, post, res = ops.mhc_input(x, hc.phi, hc.alpha, hc.base, hc.norm_eps)
    pre_t, post_t, res_t = hc.logits(x)
    assert torch.equal(torch.isnan(post), torch.isnan(post_t)) and torch.equal(torch.isnan(res), torch.isnan(res_t))
    assert torch.equal(post[3].cpu(), hc.base[4:8].cpu())
    hc.phi[10, 3] = float("inf")  # an infinite weight reaches its own column only
    hc.phi[11, 20] = 3.4e38       # rounds past the bf16 range
    h, post, res = ops.mhc_input(x[:3], hc.phi, hc.alpha, hc.base, hc.norm_eps)
    pre_t, post_t, res_t = hc.logits(x[:3])
    assert torch.isfinite(post).all()
    torch.testing.assert_close(res, res_t, rtol=1e-5, atol=1e-4)


# products of the plain streams past the fp32 range where those of the normalised streams are not: streams past the square
# root of the range (their RMS is infinite, so they normalise to zero), large weights, some tokens only
def test_mhc_input_large_values(device):
    C = 264
    hc = _block(device, C, 5)
    g = torch.Generator().manual_seed(8)
    x = torch.randn(40, 4, C, generator=g)
    x[3] *= 2.0 ** 125
    x[17] = 2.0 ** 127
    x[30] *= 2.0 ** 50
    x[33] *= 2.0 ** 66
    x = x.bfloat16().to(device)
    for scale in (1.0, 64.0, 2.0 ** 90):
        hc.phi.copy_((torch.randn(4 * C, 24, generator=g) * ((4 * C) ** -0.5 * scale)).to(device))
        hc.alpha.fill_(1.0 / scale)
        print(f"[case] mhc_input large values scale={scale}", flush=True)
        h, post, res = _lib.torch_ops().mhc_input(x, hc.phi, hc.alpha, hc.base, hc.norm_eps)
        pre_t, post_t, res_t = hc.logits(x)
        assert torch.isfinite(post_t).all() and torch.isfinite(res_t).all()
        torch.testing.assert_close(post, post_t, rtol=1e-5, atol=1e-4)
        torch.testing.assert_close(res, res_t, rtol=1e-5, atol=1e-4)
        assert torch.equal(post[17], hc.base[4:8])


def test_block_with_and_without_gradients(device):
    # with gradients the logits stay torch operations, and phi receives its gradient
    hc = _block(device, 512, 3)
    x = torch.randn(40, 4, 512).bfloat16().to(device)
    h0, post0, res0 = hc.pre(x)
    hc.requires_grad_(True)
    assert not hc._fused(x)
    h1, post1, res1 = hc.pre(x)
    res1.sum().backward()
    assert hc.phi.grad is not None and post1.requires_grad
    torch.testing.assert_close(post0, post1.detach(), rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(res0, res1.detach(), rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(h0.float(), h1.detach().float(), rtol=2 ** -7, atol=1e-4)
    with torch.no_grad():
        assert hc._fused(x)
        assert not hc._fused(x.transpose(1, 2).contiguous().transpose(1, 2)) and not hc._fused(x[:0])
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not hc._fused(x)


def test_own_logits_are_used(device):
    class Shifted(HyperConnection):
        def logits(self, x):
            pre, post, res = super().logits(x)
            return pre + 1.0, post + 2.0, res + 3.0

    x = torch.randn(20, 4, 128, generator=torch.Generator().manual_seed(1)).bfloat16().to(device)
    plain = _block(device, 128, 6)
    own = Shifted(128).to(device).requires_grad_(False)
    own.load_state_dict(plain.state_dict())
    patched = _block(device, 128, 6)
    patched.logits = lambda x: Shifted.logits(own, x)
    with torch.no_grad():
        _, post, res = plain.pre(x)
        want = _lib.torch_ops().mhc_pre(x, own.logits(x)[0])
        for hc in (own, patched):
            h, p, r = hc.pre(x)
            assert torch.equal(h, want)
            torch.testing.assert_close(p, post + 2.0, rtol=1e-5, atol=1e-5)
            torch.testing.assert_close(r, res + 3.0, rtol=1e-5, atol=1e-5)


def test_dispatch_modes_see_the_logits(device):
    from torch.utils._python_dispatch import TorchDispatchMode
    seen = []

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    hc = _block(device, 64, 7)
    x = torch.randn(4, 4, 64).bfloat16().to(device)
    want = hc.pre(x)
    with torch.no_grad(), Seen():
        got = hc.pre(x)
    assert any("mm" in f for f in seen) and not any("mhc_input" in f for f in seen)
    torch.testing.assert_close(got[1], want[1], rtol=1e-5, atol=1e-5)


def test_mhc_input_errors(device):
    hc = _block(device, 64, 4)
    x = torch.zeros(2, 4, 64, dtype=torch.bfloat16, device=device)
    ops = _lib.torch_ops()
    for bad in [dict(phi=hc.phi[:, :23].contiguous()), dict(phi=hc.phi.double()), dict(alpha=hc.alpha[:2]),
                dict(base=hc.base[:8]), dict(x=x.float()), dict(x=x[:, :3])]:
        a = dict(x=x, phi=hc.phi, alpha=hc.alpha, base=hc.base, norm_eps=1e-6, **{}) | bad
        with pytest.raises(RuntimeError):
            ops.mhc_input(a["x"], a["phi"], a["alpha"], a["base"], a["norm_eps"])
