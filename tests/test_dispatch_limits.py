"""Sizes past a kernel's 32-bit limits go to the kernels that take them, and the
part products' scratch stays bounded.  Host logic only: tensors without storage,
launches recorded instead of run."""
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
    monkeypatch.setattr(vz, 'host_array', lambda ctype, values: (values, values))
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


@pytest.mark.parametrize('side,entry', [(256, 'vc_ibp_conv_split'), (4097, 'vc_ibp_conv')])
def test_interval_conv_of_many_pixels(launches, monkeypatch, side, entry):
    """2^24 pixels and more."""
    monkeypatch.setattr(vz, '_IBP_SPLIT_MACS', 0)
    gg = _net(side, [(60, 1), None, (33, 3)])
    x = torch.empty(1, side * side, device=META)
    vz._ibp_forward_graph_batched(x, x, gg, META, torch.float32)
    assert launches.count(entry) == (2 if entry == 'vc_ibp_conv' else 1)


# rows; channels in and out, side, kernel, stride, padding; whether the split conv
# was measured the faster, weights packed and the relu before it included
@pytest.mark.parametrize('M,geom,split', [
    (6, (16, 8, 28, 3, 1, 1), False), (60, (16, 8, 28, 3, 1, 1), False),
    (300, (16, 8, 28, 3, 1, 1), True), (6, (33, 17, 20, 3, 1, 1), False),
    (120, (33, 17, 20, 3, 1, 1), False), (300, (33, 17, 20, 3, 1, 1), True),
    (6, (64, 64, 32, 3, 1, 1), False), (12, (64, 64, 32, 3, 1, 1), False),
    (30, (64, 64, 32, 3, 1, 1), True), (6, (13, 8, 14, 3, 1, 0), True),
    (12, (64, 32, 32, 4, 2, 1), True), (6, (32, 16, 28, 5, 2, 2), True)])
def test_split_conv_rule(launches, M, geom, split):
    co, ci, side, k, s, pad = geom
    out = (side + 2 * pad - k) // s + 1
    p = {'name': 'c', 'geom': (ci, side, side, co, k, k, s, s, pad, pad, out, out),
         'K': torch.empty(co, ci, k, k, device=META), 'n_out': co * out * out,
         'n_in': ci * side * side}
    assert (vz._Packs({'ops': []}, META).conv_split(p, M, M, False, 0) is not None) == split


def test_window_limits():
    """Images of more than 2^30 values are carried whole."""
    assert vz._Window(None, 3, 3, 4, 1 << 14, 1 << 14).worth()
    assert not vz._Window(None, 3, 3, 5, 1 << 14, 1 << 14).worth()


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


# argument of the buffer of parts
WORK = {'vc_backward_fc_split': 14, 'vc_alpha_grad_step_split': 13,
        'vc_alpha_grad_input_split': 10, 'vc_zono_fc_split': 9, 'vc_ibp_conv_split': 20}


@pytest.fixture
def scratch(monkeypatch, launches):
    """(name, bytes of parts, rows) of each part product."""
    rec = []

    def call(name, *a):
        if name in WORK:
            rec.append((name, a[WORK[name]].numel(), a[1 if name == 'vc_backward_fc_split' else
                                                      3 if 'input' in name else 2]))
        elif name == 'vc_unstable_union':
            raise AssertionError(name)
    monkeypatch.setattr(vz, 'call', call)
    return rec


def _mlp(widths):
    ops, prev = [], 'X'
    for i, (a, b) in enumerate(zip(widths, widths[1:])):
        ops.append({'name': f'fc{i}', 'type': 'fc', 'inputs': [prev], 'bias': None,
                    'W': torch.empty(b, a, device=META)})
        prev = f'fc{i}'
        if i + 2 < len(widths):
            ops.append({'name': f'r{i}', 'type': 'relu', 'inputs': [prev], 'layer_idx': i})
            prev = f'r{i}'
    return {'ops': ops, 'input_name': 'X', 'input_n': widths[0], 'fork_points': set(),
            'input_shape': (1, widths[0]), 'n_relu': len(widths) - 2}


@pytest.mark.parametrize('B,Q', [(300000, 9), (3, 700000), (1 << 20, 1)])
def test_alpha_gradient_scratch(scratch, monkeypatch, B, Q):
    """Rows whose relaxed form takes 10 GB and more: the parts 512 MiB at a time,
    every row once, and no slopes held past 32 MiB a layer."""
    gg = _mlp([784, 1000, 1000, 10])
    x = torch.empty(B, 784, device=META)
    sb = {L: (torch.empty(B, 1000, device=META),) * 2 for L in (0, 1)}
    alpha = {L: torch.empty(B, 1000, device=META) for L in (0, 1)}
    monkeypatch.setattr(vz, '_fc_split_pays', lambda *a: True)
    traces = []
    init = vz.BackwardTrace.__init__
    vz.BackwardTrace.__init__ = lambda self: (init(self), traces.append(self))[0]
    try:
        vz._alpha_backward_and_grad(sb, x, x, gg, torch.empty(Q, 10, device=META),
                                    torch.empty(Q, device=META), alpha, True, alpha)
    finally:
        vz.BackwardTrace.__init__ = init
    assert max(n for _, n, _ in scratch) <= 512 << 20
    for name, per in (('vc_backward_fc_split', 2), ('vc_alpha_grad_step_split', 1),
                      ('vc_alpha_grad_input_split', 1)):
        assert sum(m for n, _, m in scratch if n == name) == per * B * Q
    assert sum(t.numel() * 4 for s in traces[0].slopes.values() for t in s) <= 2 * (32 << 20)


def test_interval_conv_scratch(scratch, monkeypatch):
    """One box whose parts would take 7 GB stays with the gathering product."""
    monkeypatch.setattr(vz, '_IBP_SPLIT_MACS', 0)
    for side, n in ((64, 1), (1024, 0)):
        gg = _net(side, [(64, 1), None, (33, 3)])
        x = torch.empty(2, side * side, device=META)
        del scratch[:]
        vz._ibp_forward_graph_batched(x, x, gg, META, torch.float32)
        assert len(scratch) == n and all(b <= 1 << 30 for _, b, _ in scratch)


# rows, values, columns; packed for one pass; a gradient sweep follows: whether
# the parts were measured the faster, weights packed and slopes formed included
@pytest.mark.parametrize('M,K,N,once,sweep,pays', [
    (2304, 64, 128, True, False, False), (4608, 64, 784, False, True, True),
    (4608, 64, 784, True, False, False), (73728, 64, 128, False, False, False),
    (2304, 256, 256, True, False, False), (4608, 256, 256, True, False, False),
    (18432, 256, 256, True, False, True), (73728, 256, 256, False, True, True),
    (288, 256, 256, False, True, True), (288, 256, 256, False, False, False),
    (288, 1024, 1024, False, True, False), (576, 784, 128, False, True, False),
    (2304, 784, 128, False, True, True), (2304, 1024, 64, False, False, False),
    (4608, 1024, 1024, False, True, True), (4608, 1024, 1024, True, False, True),
    (18432, 1024, 64, False, True, True), (73728, 1024, 64, False, True, False),
    (73728, 784, 10, False, False, False), (73728, 300, 5, False, True, True),
    (73728, 65, 128, False, True, True), (73728, 65, 100, False, True, False)])
def test_fc_split_rule(M, K, N, once, sweep, pays):
    assert vz._fc_split_pays(M, K, N, once, sweep) == pays
