"""Part products taken in slices of their rows (whole domains, rows of one
domain, columns of one zonotope) give the bits of the whole."""
import pytest
import torch

from vibecheck_amd import verify_zono_bnb as vz

F32 = torch.float32


def _net(gpu, widths):
    g = torch.Generator(device=gpu).manual_seed(sum(widths))
    ops, prev = [], 'X'
    for i, (a, b) in enumerate(zip(widths, widths[1:])):
        ops.append({'name': f'fc{i}', 'type': 'fc', 'inputs': [prev],
                    'W': torch.randn(b, a, generator=g, device=gpu) * (2.0 / a) ** 0.5,
                    'bias': torch.randn(b, generator=g, device=gpu) * 0.1})
        prev = f'fc{i}'
        if i + 2 < len(widths):
            ops.append({'name': f'r{i}', 'type': 'relu', 'inputs': [prev], 'layer_idx': i})
            prev = f'r{i}'
    return {'ops': ops, 'input_name': 'X', 'input_n': widths[0], 'fork_points': set(),
            'input_shape': (1, widths[0]), 'n_relu': len(widths) - 2}


# domains, rows of each, bytes of parts at a time (64 rows of 192 values: 73,728)
@pytest.mark.gpu
@pytest.mark.parametrize('B,Q,work', [(70, 9, 100000), (3, 301, 80000), (1, 1030, 1),
                                      (600, 1, 200000)])
@pytest.mark.parametrize('beta', [False, True])
def test_alpha_gradient_in_slices(gpu, monkeypatch, B, Q, work, beta):
    monkeypatch.setattr(vz, '_fc_split_pays', lambda *a: True)
    gg = _net(gpu, [130, 150, 190, 140, 7])
    g = torch.Generator(device=gpu).manual_seed(Q)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=gpu)
    x = rand(B, 130)
    sb, alpha, galpha, bt, gb = {}, {}, {}, {}, {}
    for L, n in enumerate([150, 190, 140]):
        lo = rand(B, n) - 0.5
        sb[L] = (lo, lo + 2)
        alpha[L], galpha[L] = rand(B, n).clamp(0, 1), torch.empty(B, n, device=gpu)
        bt[L], gb[L] = rand(B, n), torch.empty(B, n, device=gpu)
    Wq, bq = rand(Q, 7), rand(Q)
    out = []
    for w, kept in ((work, 0), (1 << 40, 1 << 40)):
        monkeypatch.setattr(vz, '_FC_WORK_BYTES', w)
        monkeypatch.setattr(vz, '_SLOPES_KEPT_BYTES', kept)
        lb, A = vz._alpha_backward_and_grad(sb, x, x + 0.1, gg, Wq, bq, alpha, True, galpha,
                                            beta=bt if beta else None,
                                            gbeta=gb if beta else None, want_A=True)
        out.append([lb, A] + [t.clone() for d in (galpha, gb if beta else {})
                              for t in d.values()])
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize('B,K', [(1, 200), (3, 65), (2, 130)])
def test_zonotope_in_column_slices(gpu, monkeypatch, B, K):
    gg = _net(gpu, [K, 150, 140, 130, 7])
    g = torch.Generator(device=gpu).manual_seed(K)
    xl = torch.randn(B, K, generator=g, device=gpu)
    monkeypatch.setattr(vz, '_ZONO_SPLIT_MACS', 0)
    out = []
    for w in (1, 200000, 1 << 40):  # 64 columns, 128 columns, whole domains
        monkeypatch.setattr(vz, '_ZONO_WORK_BYTES', w)
        sb, (c, G) = vz._forward_zonotope_graph_batched(xl, xl + 0.2, gg, gpu, F32)
        out.append([c, G] + [t for v in sb.values() for t in v])
    for o in out[:2]:
        for a, b in zip(o, out[2]):
            assert torch.equal(a, b)
