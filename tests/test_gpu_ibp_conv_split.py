"""vc_ibp_conv_split (the interval forward of a conv as products of bf16 parts)
against 64-bit sums, at the edges of its pixel tiles, chunks and column tiles."""
import ctypes

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


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(map(str, c)))
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


# row blocks of 64 pixels, from 384 of them up: one and two column tiles a wave,
# a last block of 36 pixels, a second slice of boxes with blocks of 32
CASES_TALL = [
    (100, 5, 17, 17, 33, 3, 3, 1, 1, 1, 1, 100),
    (100, 5, 17, 17, 65, 3, 3, 1, 1, 1, 1, 90),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES_TALL, ids=lambda c: '-'.join(map(str, c)))
def test_ibp_conv_split_tall_blocks(gpu, case):
    test_ibp_conv_split_against_fp64(gpu, case)


@pytest.mark.gpu
def test_ibp_conv_split_infinities(gpu):
    """Bounds that are infinite, NaN or round to infinity in bf16: what the
    gathering product gives, in the pixels that read them only."""
    B, C_in, H, W, C_out, k = 3, 9, 8, 7, 20, 3
    g = torch.Generator(device=gpu).manual_seed(2)
    K = torch.randn(C_out, C_in, k, k, generator=g, device=gpu)
    b = torch.randn(C_out, generator=g, device=gpu)
    l = torch.randn(B, C_in, H, W, generator=g, device=gpu)
    h = l + torch.rand(B, C_in, H, W, generator=g, device=gpu)
    h[0, 2, 0, 0] = float('inf')
    l[0, 5, 7, 6] = float('-inf')
    l[1, 0, 3, 3] = h[1, 0, 3, 3] = float('nan')
    l[2, 8, 1, 1], h[2, 8, 1, 1] = 3.39e38, 3.395e38  # the sum of both is infinite
    n = C_in * k * k
    size = _lib.load().vc_fc_split_pack_bytes
    parts = [torch.empty(size(n, C_out), dtype=torch.uint8, device=gpu) for _ in range(2)]
    call('vc_fc_split_pack_abs', ptr(K), n, C_out, 1, ptr(parts[0]), ptr(parts[1]), stream())
    work = torch.empty(2 * B * size(n, H * W), dtype=torch.uint8, device=gpu)
    got, want = ([torch.empty(B, C_out, H, W, device=gpu) for _ in range(2)] for _ in range(2))
    geom = (C_out, k, k, 1, 1, 1, 1, H, W)
    call('vc_ibp_conv_split', ptr(l), ptr(h), B, C_in, H, W, ptr(parts[0]), ptr(parts[1]), ptr(b),
         *geom, ptr(got[0]), ptr(got[1]), ptr(work), work.numel(), stream())
    call('vc_ibp_conv', ptr(l), ptr(h), B, C_in, H, W, ptr(K), ptr(b), *geom, ptr(want[0]),
         ptr(want[1]), stream())
    for x, y in zip(got, want):
        assert torch.equal(x.isnan(), y.isnan())
        assert torch.equal(x[y.isinf()], y[y.isinf()])
        ok = y.isfinite()
        assert 0 < int(ok.sum()) < y.numel()
        # both within 2e-7 of the sums' terms
        assert float((x - y)[ok].norm() / y[ok].norm()) < 4e-7


@pytest.mark.gpu
def test_pack_abs_is_two_packs(gpu):
    g = torch.Generator(device=gpu).manual_seed(3)
    W = torch.randn(37, 75, generator=g, device=gpu)
    out = [torch.empty(_lib.load().vc_fc_split_pack_bytes(75, 37), dtype=torch.uint8, device=gpu)
           for _ in range(4)]
    call('vc_fc_split_pack_abs', ptr(W), 75, 37, 1, ptr(out[0]), ptr(out[1]), stream())
    Wa = W.abs()
    for w, o in ((W, out[2]), (Wa, out[3])):
        call('vc_fc_split_pack', ptr(w), 75, 37, 1, ptr(o), stream())
    assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3])


@pytest.mark.gpu
@pytest.mark.parametrize('trans', [0, 1])
def test_pack_many_is_each_pack(gpu, trans):
    """Nineteen matrices, more than a launch takes, of one to eight workgroups."""
    g = torch.Generator(device=gpu).manual_seed(4)
    size = _lib.load().vc_fc_split_pack_bytes
    KN = [(1 + 37 * i, 1 + 11 * (18 - i)) for i in range(19)]
    W = [torch.randn(*((N, K) if trans else (K, N)), generator=g, device=gpu) for K, N in KN]
    many = [torch.empty(size(K, N), dtype=torch.uint8, device=gpu) for K, N in KN]
    arrays = [_lib.host_array(ctypes.c_void_p, [ptr(w) for w in W]),
              _lib.host_array(ctypes.c_int32, [K for K, _ in KN]),
              _lib.host_array(ctypes.c_int32, [N for _, N in KN]),
              _lib.host_array(ctypes.c_int32, [trans] * 19),
              _lib.host_array(ctypes.c_void_p, [ptr(m) for m in many])]
    call('vc_fc_split_pack_many', *(p for _, p in arrays), 19, stream())
    for (K, N), w, m in zip(KN, W, many):
        one = torch.empty_like(m)
        call('vc_fc_split_pack', ptr(w), K, N, trans, ptr(one), stream())
        assert torch.equal(m, one)
        # the parts' sum is the value (bf16 in operand order)
        p = one.view(torch.bfloat16).view((N + 15) // 16, -1, 3, 4, 16, 8).double().sum(2)
        B = p.permute(1, 2, 4, 0, 3).reshape(64 * -(-K // 64), -1)
        assert torch.equal(B[:K, :N], (w.T if trans else w).double())
        assert not B[K:].any() and not B[:, N:].any()
