"""The fc products of bf16 parts (vc_backward_fc_split, vc_alpha_grad_step_split,
vc_alpha_grad_input_split) against 64-bit sums, at the edges of their row blocks,
column tiles and 32-deep steps, and what infinities and NaN come to."""
import pytest
import torch

from vibecheck_amd import _lib
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
