"""vc_ibp_conv_split (the interval forward of a conv as products of bf16 parts)
against 64-bit sums, at the edges of its pixel tiles, chunks and column tiles."""
import pytest
import torch
import torch.nn.functional as F

from vibecheck_amd import _lib
from vibecheck_amd._lib import call, ptr, stream

# B, C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, boxes at a time
CASES = [
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0, 1),
    (5, 8, 9, 7, 13, 3, 3, 1, 1, 1, 1, 2),      # 63 pixels: quads across images
    (3, 32, 16, 16, 64, 4, 4, 2, 2, 1, 1, 3),
    (7, 17, 10, 13, 65, 5, 3, 2, 3, 2, 0, 7),   # two column tiles a wave
    (2, 40, 6, 6, 130, 3, 2, 1, 2, 0, 1, 1),
]


# row blocks of 64 pixels, from 384 of them up: one and two column tiles a wave,
# a last block of 36 pixels, a second slice of boxes with blocks of 32
CASES_TALL = [
    (100, 5, 17, 17, 33, 3, 3, 1, 1, 1, 1, 100),
    (100, 5, 17, 17, 65, 3, 3, 1, 1, 1, 1, 90),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES + CASES_TALL, ids=lambda c: '-'.join(map(str, c)))
def test_ibp_conv_split_against_fp64(gpu, case):
    B, C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, chunk = case
    Ho, Wo = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1
    g = torch.Generator(device=gpu).manual_seed(C_in * 31 + H)
    K = torch.randn(C_out, C_in, kh, kw, generator=g, device=gpu)
    b = torch.randn(C_out, generator=g, device=gpu)
    l = torch.randn(B, C_in, H, W, generator=g, device=gpu)
    h = l + torch.rand(B, C_in, H, W, generator=g, device=gpu)
    n = C_in * kh * kw
    size = _lib.load().vc_fc_split_pack_bytes
    parts = [torch.empty(size(n, C_out), dtype=torch.uint8, device=gpu) for _ in range(2)]
    Ka = K.abs()
    for k, p in zip((K, Ka), parts):
        call('vc_fc_split_pack', ptr(k), n, C_out, 1, ptr(p), stream())
    work = torch.empty(2 * chunk * size(n, Ho * Wo), dtype=torch.uint8, device=gpu)
    lo, hi = (torch.empty(B, C_out, Ho, Wo, device=gpu) for _ in range(2))
    call('vc_ibp_conv_split', ptr(l), ptr(h), B, C_in, H, W, ptr(parts[0]), ptr(parts[1]),
         ptr(b), C_out, kh, kw, sh, sw, ph, pw, Ho, Wo, ptr(lo), ptr(hi), ptr(work),
         work.numel(), stream())
    mid, rad = (l.double() + h.double()) / 2, (h.double() - l.double()) / 2
    c = F.conv2d(mid, K.double(), b.double(), (sh, sw), (ph, pw))
    r = F.conv2d(rad, K.double().abs(), None, (sh, sw), (ph, pw))
    for got, want in ((lo, c - r), (hi, c + r)):
        # the centres' and radii's own rounding and the sums': 2^-24 each of |c| + |r|
        assert float((got.double() - want).norm() / (c.abs() + r).norm()) < 2e-7
