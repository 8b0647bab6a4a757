"""vc_backward_conv_split (the conv backward on the bf16 matrix cores, relu
relaxation fused) against 64-bit sums, at the edges of its image groups, bands,
channel chunks, output tiles and parity classes."""
import ctypes

import pytest
import torch

from vibecheck_amd import _lib
from vibecheck_amd._lib import call, ptr, stream

# B, R, shared, relu, beta, C_out, C_in, H, W, kh, kw, sh, sw, ph, pw
CASES = [
    (1, 1, 0, 0, 0, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0),
    (3, 5, 1, 1, 0, 64, 32, 32, 32, 4, 4, 2, 2, 1, 1),
    (3, 5, 0, 1, 1, 64, 64, 16, 16, 4, 4, 2, 2, 1, 1),
    (2, 3, 1, 1, 0, 32, 3, 32, 32, 3, 3, 1, 1, 1, 1),       # bands of one image
    (2, 4100, 0, 1, 1, 33, 17, 7, 9, 3, 5, 2, 3, 1, 2),     # groups of images, 6 classes
    (2, 2057, 1, 1, 0, 40, 31, 10, 10, 4, 4, 2, 2, 0, 0),
    (5, 7, 0, 1, 1, 13, 8, 14, 13, 3, 3, 1, 1, 0, 0),
    (1, 9, 0, 0, 0, 100, 70, 13, 17, 3, 2, 3, 1, 1, 0),     # two output blocks, short taps
    (4, 16, 1, 1, 1, 70, 40, 23, 11, 5, 5, 1, 1, 2, 2),     # 75 steps: rounding carried
    (2, 6, 0, 1, 0, 8, 16, 19, 40, 5, 3, 3, 3, 0, 1),       # 9 classes: three passes
]


def _setup(gpu, B, R, shared, relu, beta, C_out, C_in, H, W, kh, kw, sh, sw, ph, pw):
    Ho, Wo = (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1
    g = torch.Generator(device=gpu).manual_seed(C_out * 31 + H)
    M, n = B * R, C_out * Ho * Wo
    t = {'x': torch.randn(R if shared else M, n, generator=g, device=gpu),
         'K': torch.randn(C_out, C_in, kh, kw, generator=g, device=gpu),
         'b': torch.randn(C_out, generator=g, device=gpu),
         'acc': torch.randn(M, generator=g, device=gpu)}
    lo = torch.randn(B, n, generator=g, device=gpu) - 0.5
    hi = lo + 2 * torch.rand(B, n, generator=g, device=gpu)
    if relu:
        for k in ('ls', 'us', 'ut'):
            t[k] = torch.empty(B, n, device=gpu)
        call('vc_relax_slopes', ptr(lo), ptr(hi), None, B * n, ptr(t['ls']), ptr(t['us']),
             ptr(t['ut']), stream())
    if beta:
        t['beta'] = torch.randn(B, n, generator=g, device=gpu)
    return t, Ho, Wo


def _run(gpu, t, Ho, Wo, B, R, shared, relu, beta, C_out, C_in, H, W, kh, kw, sh, sw, ph, pw):
    lib = _lib.load()
    assert lib.vc_backward_conv_split_ok(C_out, Ho, Wo, C_in, H, W, kh, kw, sh, sw, ph, pw)
    parts = torch.empty(lib.vc_conv_split_pack_bytes(C_out, C_in, kh, kw, sh, sw),
                        dtype=torch.uint8, device=gpu)
    call('vc_conv_split_pack', ptr(t['K']), C_out, C_in, kh, kw, sh, sw, ptr(parts), stream())
    out = torch.empty(B * R, C_in, H, W, device=gpu)
    acc = t['acc'].clone()
    call('vc_backward_conv_split', ptr(t['x']), B * R, R, shared, ptr(t.get('ls')),
         ptr(t.get('us')), ptr(t.get('ut')), ptr(t.get('beta')), ptr(t['K']), ptr(parts),
         ptr(t['b']), C_out, Ho, Wo, C_in, H, W, kh, kw, sh, sw, ph, pw, ptr(out), ptr(acc),
         stream())
    return out, acc


def _exact(t, rows, B, R, shared, relu, beta, C_out, C_in, H, W, kh, kw, sh, sw, ph, pw):
    d = rows // R
    e = t['x'][rows % R if shared else rows].double()
    acc = t['acc'][rows].double()
    if relu:
        acc = acc + (e.clamp(max=0) * t['ut'][d].double()).sum(1)
        e = e.clamp(min=0) * t['ls'][d].double() + e.clamp(max=0) * t['us'][d].double()
    if beta:
        e = e + t['beta'][d].double()
    e = e.reshape(rows.numel(), C_out, -1)
    acc = acc + (e.sum(2) * t['b'].double()).sum(1)
    cols = t['K'].double().reshape(C_out, -1).T @ e
    return torch.nn.functional.fold(cols, (H, W), (kh, kw), padding=(ph, pw), stride=(sh, sw)), acc


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES)
def test_conv_split_against_fp64(gpu, case):
    t, Ho, Wo = _setup(gpu, *case)
    out, acc = _run(gpu, t, Ho, Wo, *case)
    rows = torch.unique(torch.linspace(0, case[0] * case[1] - 1, 48, device=gpu).long())
    ref, racc = _exact(t, rows, *case)
    # per step of 32 products one fp32 sum of parts and one running sum, at
    # most 9 steps or carried: 2-norm below sqrt(2 * 9) half-ulps of 2^-24
    assert (out[rows].double() - ref).norm() <= 1.3e-7 * ref.norm()
    assert (acc[rows].double() - racc).norm() <= 1.3e-7 * racc.norm()


@pytest.mark.gpu
def test_conv_split_infinities(gpu):
    """Values that are infinite, NaN or round to infinity in bf16 give what the
    plain sum gives, in their own outputs only."""
    case = (2, 3, 0, 1, 0, 34, 20, 9, 8, 3, 3, 2, 1, 1, 1)
    t, Ho, Wo = _setup(gpu, *case)
    x = t['x'].view(6, 34, Ho, Wo)
    x[0, 3, 1, 2] = float('inf')
    x[1, 33, 0, 0] = float('-inf')
    x[2, 0, 2, 5] = float('nan')
    for c, (y, z) in enumerate([(0, 0), (0, 4), (3, 0), (3, 4)]):  # no output meets two
        x[3, 7 + c, y, z] = x[4, 17 + c, y, z] = 3.4e38
    t['K'].mul_(0.25)  # 3.4e38 stays finite through one tap
    out, _ = _run(gpu, t, Ho, Wo, *case)
    ref, _ = _exact(t, torch.arange(6, device=gpu), *case)
    ref = ref.float().double()
    got = out.double()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isinf(got), torch.isinf(ref))
    inf = torch.isinf(ref)
    assert torch.equal(got[inf], ref[inf])
    ok = torch.isfinite(ref)
    # entries that 3.4e38 enters are sums rounded at its size
    big = ref.abs() > 1e30
    assert (got - ref)[ok & ~big].norm() <= 1.3e-7 * ref[ok & ~big].norm()
    assert ((got - ref).abs() <= 1e-6 * ref.abs())[ok & big].all()
    assert (~ok).sum() > 0 and big.sum() > 0


@pytest.mark.gpu
@pytest.mark.parametrize('which', ['vc_conv_split_pack', 'vc_conv_t_pack'])
def test_conv_pack_many_is_each_pack(gpu, which):
    """Eighteen kernels, more than a launch takes, of one to a few workgroups."""
    lib, taps = _lib.load(), which == 'vc_conv_t_pack'
    g = torch.Generator(device=gpu).manual_seed(6)
    geom = [(1 + 5 * i, 1 + 7 * (17 - i), 1 + i % 5, 1 + (i + 2) % 4, 1 + i % 3, 1 + (i + 1) % 2,
             i % 3, i % 2) for i in range(18)]
    K = [torch.randn(*q[:4], generator=g, device=gpu) for q in geom]

    def out(q):
        if taps:
            return torch.full((lib.vc_conv_t_pack_floats(*q[:6]),), float('nan'), device=gpu)
        return torch.full((lib.vc_conv_split_pack_bytes(*q[:6]),), 255, dtype=torch.uint8,
                          device=gpu)
    many, n = [out(q) for q in geom], 8 if taps else 6
    arrays = [_lib.host_array(ctypes.c_void_p, [ptr(k) for k in K]),
              _lib.host_array(ctypes.c_int32, [v for q in geom for v in q[:n]]),
              _lib.host_array(ctypes.c_void_p, [ptr(m) for m in many])]
    call(which + '_many', *(p for _, p in arrays), 18, stream())
    for q, k, m in zip(geom, K, many):
        co, ci, kh, kw, sh, sw, ph, pw = q
        one = out(q)
        call(which, ptr(k), *q[:n], ptr(one), stream())
        assert torch.equal(m, one)
        if not taps:
            # the parts' sum, by class, chunk of 32 channels, tap, 16-channel tile
            Ty, Tx, nch = -(-kh // sh), -(-kw // sw), -(-co // 32)
            v = one.view(torch.bfloat16).view(sh, sw, nch, Ty, Tx, -1, 3, 4, 16, 8).double().sum(6)
            # co = 32 chunk + 8 g + j, ci = 16 tile + r, ky = class + sh tap
            v = v.permute(2, 6, 8, 5, 7, 3, 0, 4, 1).reshape(nch * 32, -1, Ty * sh, Tx * sw)
            want = torch.zeros_like(v)
            want[:co, :ci, :kh, :kw] = k
            assert torch.equal(v, want)
