"""vc_ibp_fc_sliced against vc_ibp_fc, bit for bit but for ties of the 64-bit
sums' order, at slices that end on, before and after a row's last K-tile."""
import pytest
import torch

from vibecheck_amd import _lib
from vibecheck_amd._lib import call, ptr, stream


@pytest.mark.gpu
@pytest.mark.parametrize('B,n_in,n_out', [(1, 512, 10), (5, 4096, 2), (33, 1601, 65),
                                          (512, 4096, 512), (3, 700, 130)])
def test_ibp_fc_slices(gpu, B, n_in, n_out):
    g = torch.Generator(device=gpu).manual_seed(n_in)
    W = torch.randn(n_out, n_in, generator=g, device=gpu)
    b = torch.randn(n_out, generator=g, device=gpu)
    l = torch.randn(B, n_in, generator=g, device=gpu)
    h = l + torch.rand(B, n_in, generator=g, device=gpu)
    want = [torch.empty(B, n_out, device=gpu) for _ in range(2)]
    call('vc_ibp_fc', ptr(l), ptr(h), B, n_in, ptr(W), ptr(b), n_out, ptr(want[0]),
         ptr(want[1]), stream())
    rule = _lib.load().vc_ibp_fc_slices(B, n_in, n_out)
    for slices in {rule, 2, 3, n_in // 64}:
        work = torch.empty(slices * B * n_out * 2, dtype=torch.float64, device=gpu)
        got = [torch.empty(B, n_out, device=gpu) for _ in range(2)]
        call('vc_ibp_fc_sliced', ptr(l), ptr(h), B, n_in, ptr(W), ptr(b), n_out, ptr(got[0]),
             ptr(got[1]), slices, ptr(work), stream())
        for x, y in zip(got, want):
            # sums in another order differ by 2^-52: a rounding to fp32 that they
            # straddle, one value in 1e6, is one step of its terms' size
            assert int((x != y).sum()) <= 1 + B * n_out // 100000
            assert float((x - y).abs().max()) <= 2 ** -22 * float(y.abs().max())


@pytest.mark.gpu
def test_ibp_fc_slices_infinities(gpu):
    """Infinities and NaN in a slice reach the outputs of their own rows, as in
    one sum."""
    B, n_in, n_out = 6, 700, 12
    g = torch.Generator(device=gpu).manual_seed(1)
    W = torch.randn(n_out, n_in, generator=g, device=gpu)
    l = torch.randn(B, n_in, generator=g, device=gpu)
    h = l + torch.rand(B, n_in, generator=g, device=gpu)
    h[0, 3], l[1, 699], l[2, 350], h[3, 223] = (float(v) for v in ('inf', '-inf', 'nan', '3.4e38'))
    want, got = ([torch.empty(B, n_out, device=gpu) for _ in range(2)] for _ in range(2))
    call('vc_ibp_fc', ptr(l), ptr(h), B, n_in, ptr(W), None, n_out, ptr(want[0]), ptr(want[1]),
         stream())
    work = torch.empty(4 * B * n_out * 2, dtype=torch.float64, device=gpu)
    call('vc_ibp_fc_sliced', ptr(l), ptr(h), B, n_in, ptr(W), None, n_out, ptr(got[0]),
         ptr(got[1]), 4, ptr(work), stream())
    for x, y in zip(got, want):
        assert torch.equal(x.isnan(), y.isnan())
        ok = ~y.isnan()
        assert torch.equal(x[ok].isinf(), y[ok].isinf()) and y[4:].isfinite().all()
        assert float((x - y)[4:].abs().max()) <= 2 ** -22 * float(y[4:].abs().max())
