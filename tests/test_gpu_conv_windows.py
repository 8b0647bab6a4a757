"""CROWN bounds of conv neurons carried as windows of their images
(vc_patch_seed, vc_patch_relax, vc_patch_concretize, vc_patch_dense) against the whole-image oracle in 64 bits."""
import copy

import pytest
import torch

from oracle import ref_bound as rb
from vibecheck_amd import verify_zono_bnb as vz
from vibecheck_amd import workloads as wk

NETS = [
    # windows to the input; a ragged image
    ([(8, 3, 1, 1), (13, 4, 2, 1), (17, 3, 1, 1)], [21, 4], (3, 17, 19)),
    # the third layer's window outgrows half of the image on its way down
    ([(6, 5, 2, 2), (33, 5, 2, 2), (9, 3, 1, 0)], [5], (1, 24, 23)),
    # kernels over half of their image: whole rows from the start
    ([(5, 3, 1, 1), (7, 5, 1, 2)], [4, 3], (2, 6, 6)),
    # stride 3, no padding
    ([(12, 3, 3, 0), (20, 2, 1, 0)], [6, 3], (3, 29, 31)),
]


def _check(gg64, gg, B, n_in, gpu, chunk):
    xl, xh = wk.linf_boxes(B, n_in, 0.03, seed=5)
    ref = rb.ibp_forward_batched(xl.double(), xh.double(), gg64)
    want = rb.crown_intermediate_batched(gg64, xl.double(), xh.double(), sb=ref)
    got = vz._crown_intermediate_batched(
        gg, xl.to(gpu), xh.to(gpu), gpu, torch.float32, chunk=chunk,
        sb={L: (lo.float().to(gpu), hi.float().to(gpu)) for L, (lo, hi) in ref.items()})
    tightened = 0
    for L, (lo, hi) in want.items():
        tightened += int((lo > ref[L][0] + 1e-4).sum())
        for g, r in zip(got[L], (lo, hi)):
            # fp32 sums through at most five layers
            assert (g.cpu().double() - r).norm() <= 2e-6 * r.norm(), L
    return tightened


def _with_bias(gg, seed):
    g = torch.Generator().manual_seed(seed)
    for op in gg['ops']:
        if 'bias' in op:
            op['bias'] = 0.2 * torch.randn(op['bias'].shape, generator=g, dtype=torch.float64)


@pytest.mark.gpu
@pytest.mark.parametrize('net', range(len(NETS)))
@pytest.mark.parametrize('B,chunk', [(1, 2048), (5, 37)])
def test_windows_against_fp64(gpu, net, B, chunk):
    convs, fcs, shape = NETS[net]
    gg64 = wk.cnn_gg(convs, fcs, shape, seed=net, dtype=torch.float64)
    _with_bias(gg64, net)
    gg = copy.deepcopy(gg64)
    # the third net's conv windows are refused: 5 x 5 of 6 x 6
    assert _check(gg64, gg, B, shape[0] * shape[1] * shape[2], gpu, chunk) > 0


@pytest.mark.gpu
def test_windows_through_residual_merge(gpu):
    """relu(conv1(x) + x): the window rows of the next conv meet a merge."""
    gg64 = wk.cnn_gg([(6, 3, 1, 1), (6, 3, 1, 1), (5, 3, 2, 1)], [7, 3], (2, 15, 14), seed=9,
                     dtype=torch.float64)
    _with_bias(gg64, 3)
    ops = gg64['ops']
    at = next(i for i, op in enumerate(ops) if op['name'] == 'conv1')
    ops.insert(at + 1, {'name': 'merge', 'type': 'add', 'inputs': ['conv1', 'relu0'],
                        'is_merge': True, 'bias': None})
    ops[at + 2]['inputs'] = ['merge']
    gg64['fork_points'] = {'relu0'}
    assert _check(gg64, copy.deepcopy(gg64), 4, 2 * 15 * 14, gpu, 2048) > 0


@pytest.mark.gpu
@pytest.mark.parametrize('what', ['beta', 'alpha', 'plain'])
def test_windows_as_whole_images(gpu, what):
    """Window rows meet a relu with a beta, whose values outside the window
    count, or an alpha: as the same rows seeded as whole images."""
    gg = wk.cnn_gg([(9, 3, 1, 1), (13, 3, 1, 1)], [4], (3, 11, 12), seed=2, device=gpu)
    B, k = 3, 20
    xl, xh = (t.to(gpu) for t in wk.linf_boxes(B, 3 * 11 * 12, 0.03, seed=5))
    sb = vz._ibp_forward_graph_batched(xl, xh, gg, gpu, torch.float32)
    p = vz._op_params(gg['ops'][2], gpu)
    C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
    g = torch.Generator().manual_seed(1)
    idx = torch.randperm(p['n_out'], generator=g)[:k].to(gpu, torch.int32)
    rows = vz._Rows(torch.empty(2 * k, C_in * kh * kw, device=gpu), True)
    origin = torch.empty(2 * k, 2, dtype=torch.int32, device=gpu)
    acc0 = torch.empty(2 * k, device=gpu)
    vz.call('vc_patch_seed', vz.ptr(p['K']), vz.ptr(p['b']), vz.ptr(idx), k, C_out, Ho, Wo, C_in,
            kh, kw, sh, sw, ph, pw, vz.ptr(rows.ew), vz.ptr(origin), vz.ptr(acc0), vz.stream())
    rows.window = vz._Window(origin, kh, kw, C_in, H, W)
    n = p['n_in']
    beta = {0: 0.1 * torch.randn(B, n, generator=g).to(gpu)} if what == 'beta' else None
    alpha = {0: torch.rand(B, n, generator=g).to(gpu)} if what == 'alpha' else None
    got = vz._backward(sb, xl, xh, gg, 'relu0', rows, True, acc0, alpha, beta, split=False)[0]
    seed = torch.zeros(2 * k, p['n_out'], device=gpu)
    seed[torch.arange(k), idx.long()] = 1.0
    seed[torch.arange(k) + k, idx.long()] = -1.0
    want = vz._backward(sb, xl, xh, gg, 'conv1', seed, True, torch.zeros(2 * k, device=gpu),
                        alpha, beta, split=False)[0]
    # fp32 sums of the same values in another order
    assert (got.double() - want.double()).norm() <= 2e-6 * want.double().norm()


@pytest.mark.gpu
def test_window_steps_infinities(gpu):
    """vc_patch_relax and vc_patch_concretize on windows partly outside their
    images, with infinities and NaN inside: the values of the plain formula;
    what lies outside the image or the window enters nothing."""
    B, R, C, H, W, wh, ww = 3, 5, 2, 9, 8, 4, 3
    g = torch.Generator().manual_seed(0)
    rows = torch.randn(B * R, C, wh, ww, generator=g)
    rows[1, 0, 2, 1], rows[7, 1, 3, 2], rows[12, 0, 0, 0] = float('inf'), float('-inf'), float('nan')
    origin = torch.tensor([[-2, -1], [7, 6], [0, 0], [3, 2], [5, 5]], dtype=torch.int32)
    ls, us, ut = (torch.rand(B, C, H, W, generator=g) for _ in range(3))
    us[0, 0, 4, 3] = float('inf')
    ut[1, 1, 1, 1] = float('inf')
    acc = torch.randn(B * R, generator=g)
    xl = torch.randn(B, C, H, W, generator=g)
    xh = xl + torch.rand(B, C, H, W, generator=g)
    xh[2, 1, 6, 6] = float('inf')
    want, wacc, wlb = torch.zeros(B * R, C, wh, ww, dtype=torch.float64), [], []
    for m in range(B * R):
        b, (oy, ox) = m // R, origin[m % R].tolist()
        a, lb = acc[m].double(), acc[m].double()
        for c in range(C):
            for dy in range(wh):
                for dx in range(ww):
                    y, x = oy + dy, ox + dx
                    if 0 <= y < H and 0 <= x < W:
                        e = rows[m, c, dy, dx].double()
                        en, ep = e.clamp(max=0), e.clamp(min=0)
                        a = a + en * ut[b, c, y, x].double()
                        want[m, c, dy, dx] = ep * ls[b, c, y, x].double() + en * us[b, c, y, x].double()
                        lb = lb + e * (xh if e < 0 else xl)[b, c, y, x].double()
        wacc.append(a)
        wlb.append(lb)
    d = [t.to(gpu) for t in (rows, origin, ls, us, ut, acc, xl, xh)]
    out, a2, lb2 = torch.empty_like(d[0]), d[5].clone(), torch.empty_like(d[5])
    p, st = vz.ptr, vz.stream()
    vz.call('vc_patch_relax', p(d[0]), B * R, R, 0, p(d[2]), p(d[3]), p(d[4]), p(d[1]), C, H, W,
            wh, ww, p(out), p(a2), st)
    vz.call('vc_patch_concretize', p(d[0]), 0, p(d[1]), p(d[5]), p(d[6]), p(d[7]), B * R, R, C, H,
            W, wh, ww, p(lb2), st)
    # one or two roundings of fp32 terms
    for got, ref in ((out, want), (a2, torch.stack(wacc)), (lb2, torch.stack(wlb))):
        torch.testing.assert_close(got.cpu().double(), ref, rtol=1e-6, atol=1e-6, equal_nan=True)
    assert out.isfinite().logical_not().sum() >= 3 and a2.isfinite().any() and lb2.isfinite().any()
