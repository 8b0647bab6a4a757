"""Sizes past a kernel's 32-bit limits go to the kernels that take them.  Host
logic only: tensors without storage, launches recorded instead of run."""
import pytest
import torch

from vibecheck_amd import _lib
from vibecheck_amd import verify_zono_bnb as vz

META = torch.device('meta')


@pytest.fixture
def launches(monkeypatch):
    names = []
    monkeypatch.setattr(vz, 'call', lambda name, *a: names.append(name))
    monkeypatch.setattr(vz, 'ptr', lambda t: t)
    monkeypatch.setattr(vz, 'f32', lambda t: t.contiguous())
    monkeypatch.setattr(vz, 'stream', lambda: 0)
    return names


def _net(side, layers):
    """Convs (channels, k) and relus (None) on side x side images."""
    ops, prev, c = [], 'X', 1
    for i, la in enumerate(layers):
        if la is None:
            ops.append({'name': 'relu', 'type': 'relu', 'inputs': [prev], 'layer_idx': 0})
            prev = 'relu'
            continue
        m, k = la
        ops.append({'name': f'conv{i}', 'type': 'conv', 'inputs': [prev], 'bias': None,
                    'kernel': torch.empty(m, c, k, k, device=META), 'stride': (1, 1),
                    'padding': (k // 2, k // 2), 'in_shape': (c, side, side),
                    'out_shape': (m, side, side)})
        prev, c = f'conv{i}', m
    return {'ops': ops, 'input_name': 'X', 'input_n': side * side, 'fork_points': set(),
            'input_shape': (1, 1, side, side), 'n_relu': 1}


@pytest.mark.parametrize('rows,alone', [(64, False), (1100, True)])
def test_shared_rows_past_4_gib(launches, rows, alone):
    """1,100 rows of 2^20 values, shared by two domains: relaxed on their own,
    not in the split conv's loads."""
    gg = _net(64, [(16, 1), (256, 3), None])
    x = torch.empty(2, 64 * 64, device=META)
    n = 256 * 64 * 64
    sb = {0: (torch.empty(2, n, device=META), torch.empty(2, n, device=META))}
    seed = torch.empty(rows, n, device=META).unsqueeze(0).expand(2, rows, n)
    vz._spec_backward_graph_batched(sb, x, x, gg, {}, META, torch.float32,
                                    seed_ew_at={'relu': seed})
    assert ('vc_backward_relu' in launches) == alone
    assert 'vc_backward_conv_split' in launches


@pytest.mark.parametrize('side,entry', [(512, 'vc_ibp_conv_split'), (4097, 'vc_ibp_conv')])
def test_interval_conv_of_many_pixels(launches, monkeypatch, side, entry):
    """2^24 pixels and more."""
    monkeypatch.setattr(vz, '_IBP_SPLIT_MACS', 0)
    gg = _net(side, [(60, 1), None, (33, 3)])
    x = torch.empty(1, side * side, device=META)
    vz._ibp_forward_graph_batched(x, x, gg, META, torch.float32)
    assert launches.count(entry) == (2 if entry == 'vc_ibp_conv' else 1)


def test_split_conv_limits():
    """vc_backward_conv_split_fits follows the rows; the geometry alone is
    vc_backward_conv_split_ok's."""
    lib = _lib.load()
    geom = (256, 64, 64, 16, 64, 64, 3, 3, 1, 1, 1, 1)
    assert lib.vc_backward_conv_split_ok(*geom)
    n = 256 * 64 * 64 * 4
    most = (0xf0000000 - 1) // n
    assert lib.vc_backward_conv_split_fits(2 * most, most, 1, *geom)
    assert not lib.vc_backward_conv_split_fits(2 * (most + 1), most + 1, 1, *geom)
    assert lib.vc_backward_conv_split_fits(2 * (most + 1), most + 1, 0, *geom)
    assert not lib.vc_backward_conv_split_fits(1 << 31, 1, 0, *geom)
