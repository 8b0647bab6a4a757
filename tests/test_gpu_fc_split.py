"""The fc products of bf16 parts (vc_backward_fc_split, vc_alpha_grad_step_split,
vc_alpha_grad_input_split) against 64-bit sums, at the edges of their row blocks,
column tiles and 32-deep steps, and what infinities and NaN come to."""
import pytest
import torch

from vibecheck_amd import _lib
from vibecheck_amd import verify_zono_bnb as vz
from vibecheck_amd._lib import call, ptr, stream

# B, R, shared, beta, K, N
CASES = [
    (1, 1, 0, 0, 1, 1),
    (1, 9, 1, 0, 256, 784),
    (7, 9, 0, 1, 64, 65),       # one row block and a row
    (131, 6, 1, 0, 203, 117),   # unaligned, odd
    (3, 43, 0, 0, 68, 16),      # a quad past the last step
    (700, 9, 0, 1, 33, 129),    # 64-row blocks, one column past a tile
    (520, 9, 1, 1, 1024, 250),
]


def _inputs(gpu, B, R, shared, beta, K, N):
    g = torch.Generator(device=gpu).manual_seed(K * 7 + N)
    M = B * R

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=gpu)
    lo = rand(B, K) - 0.5
    hi = lo + 2 * rand(B, K).abs()
    t = {k: torch.empty(B, K, device=gpu) for k in ('ls', 'us', 'ut')}
    call('vc_relax_slopes', ptr(lo), ptr(hi), None, B * K, ptr(t['ls']), ptr(t['us']),
         ptr(t['ut']), stream())
    t.update(x=rand(R if shared else M, K), W=rand(K, N), b=rand(K), bn=rand(N), acc=rand(M),
             g=rand(M, K), beta=rand(B, K) if beta else None, xl=lo, xh=hi)
    return t


def _pack(W, K, N, trans):
    out = torch.empty(_lib.load().vc_fc_split_pack_bytes(K, N), dtype=torch.uint8,
                      device=W.device)
    call('vc_fc_split_pack', ptr(W), K, N, trans, ptr(out), stream())
    return out


def _work(out, K):
    return torch.empty(_lib.load().vc_fc_split_pack_bytes(K, out.shape[0]), dtype=torch.uint8,
                       device=out.device)


def _backward(t, B, R, shared, beta, K, N):
    out, acc = torch.empty(B * R, N, device=t['x'].device), t['acc'].clone()
    parts, work = _pack(t['W'], K, N, 0), _work(out, K)
    call('vc_backward_fc_split', ptr(t['x']), B * R, R, shared, K, ptr(t['ls']), ptr(t['us']),
         ptr(t['ut']), ptr(t['beta']), ptr(parts), ptr(t['b']), N, ptr(out), ptr(acc), ptr(work), stream())
    return out, acc


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm().clamp(min=1e-300))


# Each part product is exact and the sums of 64 of them are added with the
# rounding carried along: what stays is a rounding of the 64-term sums (2^-24
# each) and of the result, 1e-7 in the 2-norm; twice that.  acc: sums in 64 bits of terms formed
# in fp32.
TOL = 2e-7


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(map(str, c)))
def test_fc_split_against_fp64(gpu, case):
    B, R, shared, beta, K, N = case
    t = _inputs(gpu, *case)
    W = t['W'].double()
    x = (t['x'].repeat(B, 1) if shared else t['x']).double()
    ls, us, ut = (t[k].double().repeat_interleave(R, 0) for k in ('ls', 'us', 'ut'))
    e = x.clamp(min=0) * ls + x.clamp(max=0) * us
    if beta:
        e = e + t['beta'].double().repeat_interleave(R, 0)
    out, acc = _backward(t, *case)
    # e itself is formed in fp32 (two roundings): as much again
    assert _rel(out, e @ W) < 2 * TOL
    assert _rel(acc, t['acc'].double() + (x.clamp(max=0) * ut).sum(1)
                + e @ t['b'].double()) < 2 * TOL

    Wt = t['W'].T.contiguous()
    parts = _pack(Wt, K, N, 1)
    got = torch.empty(B * R, N, device=gpu)
    work = _work(got, K)
    call('vc_alpha_grad_step_split', ptr(t['g']), ptr(t['x']), B * R, R, K, ptr(t['ls']),
         ptr(t['us']), ptr(t['ut']), shared, ptr(parts), ptr(t['bn']), N, ptr(got),
         ptr(work), stream())
    e = t['g'].double() * ((x >= 0) * ls + (x <= 0) * us) + (x <= 0) * ut
    assert _rel(got, e @ W + t['bn'].double()) < 2 * TOL

    call('vc_alpha_grad_input_split', ptr(t['g']), ptr(t['xl']), ptr(t['xh']), B * R, R, K,
         ptr(parts), None, N, ptr(got), ptr(work), stream())
    xl, xh = (t[k].double().repeat_interleave(R, 0) for k in ('xl', 'xh'))
    e = (t['g'] >= 0) * xl + (t['g'] <= 0) * xh
    assert _rel(got, e @ W) < TOL


@pytest.mark.gpu
def test_fc_split_infinities(gpu):
    case = (5, 9, 0, 0, 96, 70)
    t = _inputs(gpu, *case)
    t['x'][3, 5], t['x'][17, 95], t['W'][7, 69] = float('inf'), 3.39e38, float('nan')
    out, _ = _backward(t, *case)
    ls, us = (t[k].double().repeat_interleave(9, 0) for k in ('ls', 'us'))
    e = (t['x'].clamp(min=0) * ls.float() + t['x'].clamp(max=0) * us.float()).double()
    want = (e @ t['W'].double()).float()
    assert torch.equal(out.isnan(), want.isnan())
    assert torch.equal(out.isinf(), want.isinf())
    ok = want.isfinite()
    rows = [r for r in range(45) if r not in (3, 17)]
    assert _rel(out[rows][ok[rows]], (e @ t['W'].double())[rows][ok[rows]]) < 2 * TOL


def _mlp(gpu, widths):
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


# boxes on both sides of the rule's lines: 8,192 rows; 1e9 and 4e8 products; 64
# rows with a sweep
@pytest.mark.gpu
@pytest.mark.parametrize('widths,boxes', [([70, 128, 130, 5], (2047, 2048)),
                                          ([70, 500, 510, 5], (1024, 1030)),
                                          ([40, 150, 512, 5], (15, 16)),
                                          ([784, 520, 260, 5], (505, 920))])
def test_backward_with_and_without_parts(gpu, monkeypatch, widths, boxes):
    """The whole backward and its alpha gradient, products as parts and not, each
    against 64 bits: the parts are no further off."""
    gg, Q, F32 = _mlp(gpu, widths), 4, torch.float32
    for B in boxes:
        g = torch.Generator(device=gpu).manual_seed(B)

        def rand(*shape):
            return torch.randn(*shape, generator=g, device=gpu)
        xl = rand(B, widths[0])
        xh = xl + 0.1
        sb, alpha, ga = {}, {}, {}
        for L, n in enumerate(widths[1:-1]):
            lo = rand(B, n) - 0.5
            sb[L] = (lo, lo + 2)
            alpha[L] = torch.rand(B, n, generator=g, device=gpu)
            ga[L] = torch.empty(B, n, device=gpu)
        Wq, bq = rand(Q, widths[-1]), rand(Q)
        a64 = {L: a.double().requires_grad_() for L, a in alpha.items()}
        e = Wq.double().unsqueeze(0).expand(B, Q, -1)
        acc = bq.double().expand(B, Q)
        for op in reversed(gg['ops']):
            if op['type'] == 'fc':
                acc = acc + e @ op['bias'].double()
                e = e @ op['W'].double()
                continue
            lo, hi = (t.double() for t in sb[op['layer_idx']])
            act, dead = lo >= 0, hi <= 0
            un = ~act & ~dead
            us = torch.where(un, hi / (hi - lo), act.double())
            ut = torch.where(un, -lo * us, torch.zeros_like(lo))
            ls = act + un * a64[op['layer_idx']]
            en = e.clamp(max=0)
            acc = acc + (en * ut.unsqueeze(1)).sum(2)
            e = e.clamp(min=0) * ls.unsqueeze(1) + en * us.unsqueeze(1)
        lb64 = acc + (e.clamp(min=0) * xl.double().unsqueeze(1)
                      + e.clamp(max=0) * xh.double().unsqueeze(1)).sum(2)
        g64 = dict(zip(a64, torch.autograd.grad(lb64.sum(), list(a64.values()))))
        err = {}
        rule = _fc_rule
        for how, pays in (('rule', rule), ('parts', lambda *a: True), ('fp32', lambda *a: False)):
            monkeypatch.setattr(vz, '_fc_split_pays', pays)
            monkeypatch.setattr(vz, '_FC_SPLIT_SWEEP_ROWS', 64 if how == 'rule' else
                                1 if how == 'parts' else 1 << 30)
            lb, A = vz._alpha_backward_and_grad(sb, xl, xh, gg, Wq, bq, alpha, True, ga,
                                                want_A=True)
            err[how] = [_rel(lb, lb64.detach()), _rel(A.view(B, Q, -1), e.detach())] + \
                [_rel(ga[L], g64[L]) for L in ga]
        for k in ('rule', 'parts'):
            # three layers of fp32 sums; no further off than the fp32 products but
            # for what their last roundings differ by
            assert all(x <= max(1e-6, 1.5 * y) for x, y in zip(err[k], err['fp32'])), (k, err)


_fc_rule = vz._fc_split_pays
