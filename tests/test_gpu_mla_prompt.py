"""Matrix-core attention over a prompt's rows (more than 16 rows in a call:
positions split by how many rows there are, or not at all) against float64
and against the same rows in calls of up to 16.

Bound: products keep hi*hi + hi*lo + lo*hi of bf16 hi/lo parts, 2^-16 of each
product, so a score of standard deviation 1.7 (values up to 8) moves by about
1e-4 and the context by that share of its largest value.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def f64(qabs, qr, lat, kr, base, scale):
    s = (torch.einsum("rhl,tl->rht", qabs.double(), lat.double()) +
         torch.einsum("rhp,tp->rht", qr.double(), kr.double())) * scale
    R, T = qabs.shape[0], lat.shape[0]
    t = torch.arange(T, device=s.device)
    n = base + 1 + torch.arange(R, device=s.device)
    s.masked_fill_(t[None, None] >= n[:, None, None], float("-inf"))
    return torch.einsum("rht,tl->rhl", torch.softmax(s, -1), lat.double())


# one slice a row, several (an uneven split's last one is short or empty), a
# tail tile of one position, contexts that end inside the first slice, fewer
# heads, few column groups either side of the longest context they split
@pytest.mark.parametrize("R,H,T", [(17, 128, 17), (17, 128, 129), (17, 128, 700), (33, 32, 33), (40, 64, 2049),
                                   (100, 128, 100), (257, 128, 257), (260, 128, 900), (37, 96, 1500),
                                   (24, 32, 16384), (24, 32, 16385), (25, 32, 16385)])
def test_prompt_rows(ctx, R, H, T):
    import undertow_amd as U
    g = torch.Generator(device="cuda").manual_seed(R * T)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)
    qabs, qr, lat, kr = rnd(R, H, 512), rnd(R, H, 64), rnd(T, 512), rnd(T, 64)
    base, scale = T - R, float(1 / np.sqrt(192.0))
    kc = U.mla_cache_split(ctx, lat, kr)
    got = U.mla_attend_split(ctx, qabs, qr, kc, base, scale)
    want = f64(qabs, qr, lat, kr, base, scale)
    tol = 1e-4 * max(1.0, float(want.abs().max()))
    assert float((got - want).abs().max()) <= tol
    assert torch.equal(U.mla_attend(ctx, qabs, qr, lat, kr, base, scale), got)
    few = torch.cat([U.mla_attend_split(ctx, qabs[r:r + 16].contiguous(), qr[r:r + 16].contiguous(),
                                        kc, base + r, scale) for r in range(0, R, 16)])
    assert float((got - few).abs().max()) <= tol
    # no further from float64 than the short calls
    assert float((got - want).norm()) <= 1.05 * float((few - want).norm())


@pytest.mark.parametrize("R,H,T", [(16, 128, 16), (16, 128, 129), (16, 128, 513), (20, 128, 100),
                                   (17, 128, 128), (128, 32, 128), (4, 128, 33), (24, 32, 16400)])
def test_rows_merge_equals_single_rows(ctx, R, H, T):
    """Calls that keep the slices of the context length merge them with the
    same sums whatever kernel merges: rows equal their own one-row calls."""
    import undertow_amd as U
    g = torch.Generator(device="cuda").manual_seed(R + T)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)
    qabs, qr, lat, kr = rnd(R, H, 512), rnd(R, H, 64), rnd(T, 512), rnd(T, 64)
    kc, scale = U.mla_cache_split(ctx, lat, kr), float(1 / np.sqrt(192.0))
    got = U.mla_attend_split(ctx, qabs, qr, kc, T - R, scale)
    one = torch.cat([U.mla_attend_split(ctx, qabs[r:r + 1].contiguous(), qr[r:r + 1].contiguous(),
                                        kc, T - R + r, scale) for r in range(R)])
    assert torch.equal(got, one)


@pytest.mark.parametrize("R,T", [(20, 100), (40, 700), (257, 257)])
def test_output_aligned_to_one_float(ctx, R, T):
    import undertow_amd as U
    g = torch.Generator(device="cuda").manual_seed(R)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)
    qabs, qr, lat, kr = rnd(R, 128, 512), rnd(R, 128, 64), rnd(T, 512), rnd(T, 64)
    kc, scale = U.mla_cache_split(ctx, lat, kr), float(1 / np.sqrt(192.0))
    out = torch.empty(R * 128 * 512 + 1, device="cuda")[1:].view(R, 128, 512)
    U.mla_attend_split(ctx, qabs, qr, kc, T - R, scale, out=out)
    assert torch.equal(out, U.mla_attend_split(ctx, qabs, qr, kc, T - R, scale))
