"""The zonotope relu and fc taken together (vc_zono_relu_lists, vc_zono_fc_split,
vc_zono_fc_cols) against 64-bit sums, at the edges of their tiles and with inputs
that do not vary, and against the forward that takes them one by one."""
import pytest
import torch

from vibecheck_amd import _lib
from vibecheck_amd import verify_zono_bnb as vz

# boxes, widths, inputs held fixed, bytes of parts at a time
CASES = [
    (1, [1, 66, 67, 2], 0, 1 << 20),
    (3, [17, 129, 65, 80, 5], 4, 1 << 20),
    (37, [40, 200, 77, 64, 9], 0, 1 << 20),      # chunks of a few domains
    (5, [300, 257, 130, 3], 299, 1),             # one domain at a time, one input
    (4, [33, 70, 68, 2], 33, 1 << 20),           # a point: no generators
]


def _net(gpu, widths, g):
    ops, prev = [], 'X'
    for i, (a, b) in enumerate(zip(widths, widths[1:])):
        W = torch.randn(b, a, generator=g, device=gpu) * (2.0 / a) ** 0.5
        ops.append({'name': f'fc{i}', 'type': 'fc', 'inputs': [prev], 'W': W,
                    'bias': torch.randn(b, generator=g, device=gpu) * 0.1})
        prev = f'fc{i}'
        if i + 2 < len(widths):
            ops.append({'name': f'r{i}', 'type': 'relu', 'inputs': [prev], 'layer_idx': i})
            prev = f'r{i}'
    return {'ops': ops, 'input_name': 'X', 'input_n': widths[0], 'fork_points': set(),
            'input_shape': (1, widths[0]), 'n_relu': len(widths) - 2}


def _exact(gg, xl, xh, vary):
    lo, hi = xl.double(), xh.double()
    c, G = (lo + hi) / 2, torch.diag_embed((hi - lo) / 2)[:, :, vary]
    sb = {}
    for op in gg['ops']:
        if op['type'] == 'fc':
            W = op['W'].double()
            c, G = c @ W.T + op['bias'].double(), W @ G
            continue
        s = G.abs().sum(2)
        lo, hi = c - s, c + s
        sb[op['layer_idx']] = (lo, hi)
        un = (lo < 0) & (hi > 0)
        gap = torch.where(un, hi - lo, torch.ones_like(lo))
        lam = torch.where(un, hi / gap, (hi > 0).double())
        mu = torch.where(un, -hi * lo / (2 * gap), torch.zeros_like(lo))
        new = torch.zeros(*lo.shape, int(un.sum(1).max()), device=lo.device, dtype=lo.dtype)
        b, n = un.nonzero(as_tuple=True)
        new[b, n, (un.cumsum(1) - 1)[b, n]] = mu[b, n]
        c, G = lam * c + mu, torch.cat([lam.unsqueeze(2) * G, new], 2)
    return sb, c, G


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm().clamp(min=1e-300))


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(map(str, c[1])))
def test_zono_fc_split(gpu, case, monkeypatch):
    B, widths, fixed, work = case
    g = torch.Generator(device=gpu).manual_seed(sum(widths))
    gg = _net(gpu, widths, g)
    mid = torch.randn(B, widths[0], generator=g, device=gpu)
    r = 0.2 * torch.rand(B, widths[0], generator=g, device=gpu)
    r[:, :fixed] = 0.0
    xl, xh = mid - r, mid + r
    vary = ((xh - xl) > 0).any(0)
    sb0, c0, G0 = _exact(gg, xl, xh, vary)
    # a slope hi / (hi - lo) carries its bounds' rounding over their distance
    slope = 1 + max(float(lo.norm() / (hi - lo).norm().clamp(min=1e-30)) if vary.any() else 0
                    for lo, hi in sb0.values())
    monkeypatch.setattr(vz, '_ZONO_WORK_BYTES', work)
    out = {}
    for macs in (0, 1e30):
        monkeypatch.setattr(vz, '_ZONO_SPLIT_MACS', macs)
        sb, (c, G) = vz._forward_zonotope_graph_batched(xl, xh, gg, gpu, torch.float32)
        only = vz._zono_sb(gg, xl, xh, gpu, torch.float32)
        assert G.shape == G0.shape
        for L in sb0:
            for k in (0, 1):
                # a few layers of fp32 sums, each within 3e-7 of its terms' size
                assert _rel(sb[L][k], sb0[L][k]) < 2e-6
                assert torch.equal(only[L][k], sb[L][k])
        assert _rel(c, c0) < 2e-6
        assert _rel(G, G0) < 2e-6 * slope
        out[macs] = sb
    # the first layer's generators are single products: the same bits
    for a, b in zip(out[0][0], out[1e30][0]):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_zono_fc_split_infinities(gpu):
    """Generators that are infinite, NaN or round to infinity in bf16, some under
    a zero slope: what the plain sum gives, in their own columns only."""
    B, n, K, n_out = 2, 70, 90, 33
    g = torch.Generator(device=gpu).manual_seed(5)
    G = torch.randn(B, n, K, generator=g, device=gpu)
    lam = torch.rand(B, n, generator=g, device=gpu)
    W = torch.randn(n_out, n, generator=g, device=gpu) * 0.1
    G[0, 3, 5], G[0, 69, 89], G[1, 20, 64] = float('inf'), float('-inf'), float('nan')
    G[1, 40, 7], G[1, 41, 8] = 3.4e38, float('inf')
    lam[1, 40], lam[1, 41] = 1.0, 0.0
    size = _lib.load().vc_fc_split_pack_bytes
    parts = torch.empty(size(n, n_out), dtype=torch.uint8, device=gpu)
    _lib.call('vc_fc_split_pack', _lib.ptr(W), n, n_out, 1, _lib.ptr(parts), _lib.stream())
    work = torch.empty(size(n, K) * B, dtype=torch.uint8, device=gpu)
    out = torch.empty(B, n_out, K, device=gpu)
    _lib.call('vc_zono_fc_split', _lib.ptr(G), _lib.ptr(lam), B, n, K, _lib.ptr(parts), n_out, K,
              _lib.ptr(out), _lib.ptr(work), work.numel(), _lib.stream())
    want = W.double() @ (G * lam.unsqueeze(2)).double()
    f = want.float()
    assert torch.equal(out.isnan(), f.isnan())
    assert torch.equal(out[f.isinf()], f[f.isinf()])
    big = f.isfinite() & (f.abs() > 1e30)  # sums rounded at their largest term's size
    ok = f.isfinite() & ~big
    assert int((~f.isfinite()).sum()) >= 4 * n_out - 4 and int(big.sum()) > 0
    assert _rel(out[ok], want[ok]) < 2e-7  # as test_fc_split_against_fp64
    assert ((out[big].double() - want[big]).abs() <= 1e-6 * want[big].abs()).all()
