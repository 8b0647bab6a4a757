"""The weights' second layouts (bf16 parts, packed taps) belong to one call: they
are made on its stream from the weights as they are then.  Calls on several
streams, writes to a weight between calls (also through ``.data``, which moves
no version counter) and weights made under inference mode are all sound.

On the CPU the library's launches are recorded instead of run: a product's
packed operand has to be one that the same call packed, on the same stream,
from the weights' present values.  On the GPU the results are compared."""
import pytest
import torch

from vibecheck_amd import verify_zono_bnb as vz
from vibecheck_amd import workloads as wk

F32 = torch.float32
# entry point: weights and packed buffers of a pack; packed operands of a product
PACKS = {'vc_fc_split_pack_many': (0, [4]), 'vc_fc_split_pack_abs': (0, [4, 5]),
         'vc_conv_split_pack_many': (0, [2]), 'vc_conv_t_pack_many': (0, [2]),
         'vc_fc_split_pack': (0, [4]), 'vc_conv_split_pack': (0, [7]), 'vc_conv_t_pack': (0, [9])}
READS = {'vc_backward_fc_split': [9], 'vc_alpha_grad_step_split': [9],
         'vc_alpha_grad_input_split': [6], 'vc_zono_fc_split': [5],
         'vc_ibp_conv_split': [6, 7], 'vc_backward_conv_split': [9],
         'vc_backward_conv_packed': [3]}


def _mlp(widths, dtype=F32, dev='cpu'):
    g = torch.Generator().manual_seed(sum(widths))
    ops, prev = [], 'X'
    for i, (a, b) in enumerate(zip(widths, widths[1:])):
        W = torch.randn(b, a, generator=g, dtype=torch.float64) * (2.0 / a) ** 0.5
        ops.append({'name': f'fc{i}', 'type': 'fc', 'inputs': [prev], 'W': W.to(dev, dtype),
                    'bias': torch.zeros(b, device=dev, dtype=dtype)})
        prev = f'fc{i}'
        if i + 2 < len(widths):
            ops.append({'name': f'r{i}', 'type': 'relu', 'inputs': [prev], 'layer_idx': i})
            prev = f'r{i}'
    return {'ops': ops, 'input_name': 'X', 'input_n': widths[0], 'fork_points': set(),
            'input_shape': (1, widths[0]), 'n_relu': len(widths) - 2}


MLP = [70, 140, 130, 150, 9]


def _cnn(dtype=F32, dev='cpu'):
    return wk.cnn_gg([(32, 3, 1, 1), (40, 4, 2, 1), (33, 3, 1, 1)], [20, 9], (3, 17, 16), seed=2,
                     device=dev, dtype=dtype)


def _case(path, dtype=F32, dev='cpu'):
    """(gg, call) of a path whose products take packed weights."""
    cnn = path in ('ibp', 'crown_cnn', 'spec_cnn')
    gg = _cnn(dtype, dev) if cnn else _mlp([5, 50, 50, 9] if path == 'narrow' else MLP, dtype, dev)
    n_in, n_out = gg['input_n'], 9
    B = 4 if path == 'crown_cnn' else 16
    g = torch.Generator().manual_seed(3)
    xl = torch.rand(B, n_in, generator=g).to(dev)
    xh = xl + 0.1
    with torch.inference_mode(False):  # spec rows are kept by their version
        eye = torch.eye(n_out, device=dev)
        spec = {q: (eye[0] - eye[q + 1], 0.0) for q in range(n_out - 1)}
    sb = {}
    widths = vz.validate_gg(gg, n_in)
    for L, n in enumerate(widths[op['name']] for op in gg['ops'] if op['type'] == 'relu'):
        lo = torch.randn(B, n, generator=g).to(dev) - 0.5
        sb[L] = (lo, lo + 2)

    def run():
        if path in ('spec', 'spec_cnn'):
            return [vz._spec_backward_graph_batched(sb, xl, xh, gg, spec, dev, F32)]
        if path == 'alpha':
            return [vz._run_alpha_crown_inputsplit_batched(xl, xh, gg, spec, dev, F32, n_iters=3,
                                                           sb=sb)]
        if path == 'narrow':
            return [t for b in vz._zono_sb(gg, xl, xh, dev, F32).values() for t in b]
        if path == 'ibp':
            bounds = vz._ibp_forward_graph_batched(xl, xh, gg, dev, F32)
            return [t for b in bounds.values() for t in b]
        if path == 'crown_cnn':
            bounds = vz._crown_intermediate_batched(gg, xl, xh, dev, F32, chunk=512, sb=sb)
            return [t for b in bounds.values() for t in b]
        bounds, (c, G) = vz._forward_zonotope_graph_batched(xl, xh, gg, dev, F32)
        return [c, G] + [t for b in bounds.values() for t in b]
    return gg, run


PATHS = ['spec', 'alpha', 'zono', 'ibp', 'crown_cnn', 'spec_cnn']


def _weights(gg):
    return [op.get('W', op.get('kernel')) for op in gg['ops'] if 'W' in op or 'kernel' in op]


@pytest.fixture
def small(monkeypatch):
    """Every product from the smallest sizes on by the packed weights."""
    monkeypatch.setattr(vz, '_ZONO_SPLIT_MACS', 0)
    monkeypatch.setattr(vz, '_IBP_SPLIT_MACS', 0)
    monkeypatch.setattr(vz, '_fc_split_pays', lambda *a: True)


@pytest.fixture
def launches(monkeypatch, small):
    """Records launches on the CPU; the dict's 'stream' is the current one."""
    rec = {'stream': 1, 'packed': {}, 'read': 0, 'packs': 0}

    def call(name, *a):
        if name in PACKS:
            src, outs = PACKS[name]
            for i in outs:
                many = name.endswith('_many')
                for w, out in zip(a[src], a[i]) if many else [(a[src], a[i])]:
                    rec['packed'][id(out)] = (out, a[-1], w, w.clone())
            rec['packs'] += 1
        for i in READS.get(name, []):
            _, st, src, was = rec['packed'][id(a[i])]
            assert st == a[-1], f'{name} reads weights packed on another stream'
            assert torch.equal(src, was), f'{name} reads weights packed before they changed'
            rec['read'] += 1
        # what the host reads back
        if name == 'vc_zono_relu_bounds':
            a[8].fill_(a[3])
        if name == 'vc_unstable_union':
            a[4].fill_(1)
        if name == 'vc_best_update':
            a[4].zero_()

    monkeypatch.setattr(vz, 'call', call)
    monkeypatch.setattr(vz, 'ptr', lambda t: t)
    monkeypatch.setattr(vz, 'host_array', lambda ctype, values: (values, values))
    monkeypatch.setattr(vz, 'f32', lambda t: t.contiguous())
    monkeypatch.setattr(vz, 'stream', lambda: rec['stream'])
    return rec


@pytest.mark.parametrize('path', PATHS)
def test_two_streams_pack_for_themselves(launches, path):
    _, run = _case(path)
    for st in (1, 2, 1):
        launches['stream'] = st
        run()
    assert launches['read'] >= 3


@pytest.mark.parametrize('path', PATHS)
def test_changed_weights_are_packed_again(launches, path):
    gg, run = _case(path)
    run()
    for w in _weights(gg):
        w.data.mul_(1.5)
    run()
    assert launches['read'] >= 2


@pytest.mark.parametrize('path,most', [('spec', 1), ('alpha', 1), ('zono', 1), ('ibp', 1),
                                       ('crown_cnn', 2), ('spec_cnn', 2)])
def test_a_layout_is_one_launch(launches, path, most):
    """The layers' weights go together: one launch for each kind of parts, one
    for each form of the taps."""
    gg, run = _case(path)
    run()
    assert 1 <= launches['packs'] <= most


@pytest.mark.parametrize('path', PATHS)
def test_inference_mode_weights(launches, path):
    with torch.inference_mode():
        gg, run = _case(path, torch.float64)
        run()
    run()
    assert launches['read'] >= 2


def test_copies_are_kept_when_ready(monkeypatch):
    """Copies of weights (another type or device) and the narrow networks' plan
    are kept on the graph only after the stream that makes them has been waited
    for, and not under capture; the caller's own fp32 tensors as they are."""
    from vibecheck_amd import mlp_fused
    waits = []
    ready = [False]

    def settled(dev):
        waits.append(('_vc_amd_params' in op, mlp_fused.PLAN_KEY in narrow))
        return ready[0]
    monkeypatch.setattr(vz._lib, 'settled', settled)
    monkeypatch.setattr(mlp_fused, 'call', lambda *a: None)
    monkeypatch.setattr(mlp_fused, 'ptr', lambda t: t.data_ptr())
    monkeypatch.setattr(mlp_fused, 'stream', lambda: 0)
    narrow = _mlp([5, 50, 50, 5])
    op = _mlp(MLP)['ops'][0]
    cpu = torch.device('cpu')
    p = vz._op_params(op, cpu)
    assert not waits and vz._op_params(op, cpu) is p
    op = _mlp(MLP, torch.float64)['ops'][0]
    for ready[0] in (False, True):
        del waits[:]
        p = vz._op_params(op, cpu)
        assert len(waits) == 1 and not waits[0][0]
        q = mlp_fused.plan_for(narrow, cpu)
        assert len(waits) == 2 and not waits[1][1]
        if not ready[0]:
            assert '_vc_amd_params' not in op and mlp_fused.PLAN_KEY not in narrow
            continue
        assert vz._op_params(op, cpu) is p and mlp_fused.plan_for(narrow, cpu) is q


@pytest.mark.gpu
@pytest.mark.parametrize('path', PATHS)
def test_changed_weights_gpu(gpu, small, path):
    """Writes through ``.data`` and in place: the next call's results are those
    of a graph built from the new weights, bit for bit."""
    gg, run = _case(path, dev=gpu)
    first = run()
    for i, w in enumerate(_weights(gg)):
        (w.data if i % 2 else w).mul_(1.5)
    got = run()
    for op in gg['ops']:  # a graph without anything kept
        for k in [k for k in op if k.startswith('_vc_amd')]:
            del op[k]
    want = run()
    assert not torch.equal(first[0], got[0])
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize('path,dtype', [(p, F32) for p in PATHS]
                         + [('zono', torch.float64), ('narrow', F32)])
def test_two_streams_gpu(gpu, small, path, dtype):
    """A first call that waits behind other work on its stream, and a second one
    on another stream before it has run."""
    _, run = _case(path, dtype, dev=gpu)
    _, ref = _case(path, dtype, dev=gpu)
    want = ref()
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.randn(4096, 4096, device=gpu)
    with torch.cuda.stream(a):
        for _ in range(20):
            big = big @ big * 1e-4
        first = run()
    with torch.cuda.stream(b):
        second = run()
    torch.cuda.synchronize()
    for out in (first, second):
        for x, y in zip(out, want):
            assert torch.equal(x, y)
