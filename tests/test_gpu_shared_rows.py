"""The backward of a merge whose shortcut stands before the main branch in the
op order: the main branch's relu gives every domain its own constant term while
the shortcut's rows are still shared, and its bias belongs to every domain."""
import copy

import pytest
import torch

from oracle import ref_bound as rb
from vibecheck_amd import verify_zono_bnb as vz
from vibecheck_amd import workloads as wk


def _rand(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, dtype=torch.float64) * scale


def _fc(name, inp, a, b, g):
    return {'name': name, 'type': 'fc', 'inputs': [inp], 'W': _rand(g, b, a, scale=a ** -0.5),
            'bias': _rand(g, b)}


def _conv(name, inp, cin, cout, side, k, g):
    return {'name': name, 'type': 'conv', 'inputs': [inp], 'kernel':
            _rand(g, cout, cin, k, k, scale=(cin * k * k) ** -0.5), 'bias': _rand(g, cout),
            'in_shape': (cin, side, side), 'out_shape': (cout, side, side), 'stride': (1, 1),
            'padding': (k // 2, k // 2), 'output_padding': (0, 0), 'n_out': cout * side * side}


def _relu(name, inp, L):
    return {'name': name, 'type': 'relu', 'inputs': [inp], 'layer_idx': L}


def _net(kind):
    """(gg, n_in): [stem relu] shortcut; fc or conv, relu, fc or conv; merge;
    relu; head."""
    g = torch.Generator().manual_seed(4)
    if kind == 'fc':
        ops = [_fc('short', 'X', 40, 70, g), _fc('f1', 'X', 40, 70, g), _relu('r1', 'f1', 0),
               _fc('f2', 'r1', 70, 70, g)]
        n_in, n = 40, 70
    else:  # channels of the image: the fold kernel's, the fp32 product's, the parts' product's
        c = {'conv3': 3, 'conv8': 8}[kind]
        ops = [_conv('short', 'X', c, 6, 7, 3, g), _conv('f1', 'X', c, 5, 7, 3, g),
               _relu('r1', 'f1', 0), _conv('f2', 'r1', 5, 6, 7, 3, g)]
        n_in, n = c * 49, 6 * 49
    ops += [{'name': 'merge', 'type': 'add', 'inputs': ['f2', 'short'], 'is_merge': True,
             'bias': None}, _relu('r2', 'merge', 1), _fc('head', 'r2', n, 5, g)]
    return {'ops': ops, 'input_name': 'X', 'input_n': n_in, 'input_shape': (1, n_in),
            'fork_points': {'X'}, 'relu_names': ['r1', 'r2'], 'n_relu': 2}, n_in


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['fc', 'conv3', 'conv8'])
@pytest.mark.parametrize('split', [False, True])
def test_shortcut_before_main_branch(gpu, kind, split):
    gg64, n_in = _net(kind)
    B = 3
    xl, xh = wk.linf_boxes(B, n_in, 0.05, seed=5)
    sb = rb.ibp_forward_batched(xl.double(), xh.double(), gg64)
    want = rb.crown_intermediate_batched(gg64, xl.double(), xh.double(), sb=sb)
    gg = copy.deepcopy(gg64)
    dev_sb = {L: (lo.float().to(gpu), hi.float().to(gpu)) for L, (lo, hi) in sb.items()}
    if not split:
        got = vz._crown_intermediate_batched(gg, xl.to(gpu), xh.to(gpu), gpu, torch.float32,
                                             sb=dev_sb)
        assert (want[1][0] > sb[1][0] + 1e-4).any()
        for L in want:
            for a, b in zip(got[L], want[L]):
                assert (a.cpu().double() - b).norm() <= 2e-6 * b.norm()
        return
    # rows of the merge itself, seeded below the relu (products may be split)
    n = sb[1][0].shape[1]
    seed = torch.eye(n, dtype=torch.float64).unsqueeze(0).expand(B, n, n)
    ref = rb.spec_backward_batched(sb, xl.double(), xh.double(), gg64, {},
                                   seed_ew_at={'merge': seed})
    s = torch.eye(n, device=gpu).unsqueeze(0).expand(B, n, n)
    lb = vz._spec_backward_graph_batched(dev_sb, xl.to(gpu), xh.to(gpu), gg, {}, gpu,
                                         torch.float32, seed_ew_at={'merge': s})
    ref = ref[0] if isinstance(ref, tuple) else ref
    assert (lb.cpu().double() - ref).norm() <= 2e-6 * ref.norm()


@pytest.mark.gpu
@pytest.mark.parametrize('B', [1, 3])
@pytest.mark.parametrize('bias', [False, True])
def test_callers_constant_terms_stay(gpu, B, bias):
    """The shared rows' constant terms are the caller's: a call leaves them as
    they are, also for one domain, whose own terms would be the same memory."""
    gg, n_in = _net('conv8')
    for op in gg['ops']:
        if op['type'] == 'fc':
            op['bias'] = op['bias'] if bias else None
    xl, xh = (t.to(gpu) for t in wk.linf_boxes(B, n_in, 0.05, seed=5))
    sb = vz._ibp_forward_graph_batched(xl, xh, gg, gpu, torch.float32)
    W, b = torch.randn(4, 5, device=gpu), torch.randn(4, device=gpu)
    keep = b.clone()
    out = [vz._backward(sb, xl, xh, gg, 'head', W, True, b) for _ in range(2)]
    assert torch.equal(b, keep)
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][3], out[1][3])
    spec = {0: (W[0], 1.5)}
    lb = [vz._spec_backward_graph_batched(sb, xl, xh, gg, spec, gpu, torch.float32)
          for _ in range(2)]
    assert torch.equal(lb[0], lb[1])
