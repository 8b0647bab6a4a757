"""CROWN of narrow MLPs over the hidden widths: the bias row sits at row d of
the d-wide layer's tile, so its dot comes from another accumulator entry for
every width, the last ones of the last tile among them."""
import pytest
import torch

from oracle import ref_bound as rb
from vibecheck_amd import verify_zono_bnb as vz
from vibecheck_amd import workloads as wk

F32 = torch.float32


@pytest.mark.gpu
@pytest.mark.parametrize('B', [9, 1100])  # k_crown_dom, the layer-synchronous rows
@pytest.mark.parametrize('width', [3, 14, 15, 18, 31, 32, 34, 35, 46, 47, 48, 50, 51, 54, 58, 59,
                                   62, 63, 64])
def test_bias_row_every_entry(gpu, width, B):
    widths = [5, width, width, width, 4]
    Ws, bs = wk.mlp_params(widths, seed=width, bias_std=0.3)
    gg_c = wk.mlp_gg(Ws, bs, dtype=torch.float64)
    gg_g = wk.mlp_gg(Ws, bs, device=gpu, dtype=F32)
    xl, xh = wk.acas_boxes(B, seed=2)
    spec = {q: (torch.eye(4)[0] - torch.eye(4)[q + 1], 0.0) for q in range(3)}
    tight_c = rb.crown_intermediate_batched(gg_c, xl.double(), xh.double())
    tight_g = {L: (lo.float().to(gpu), hi.float().to(gpu)) for L, (lo, hi) in tight_c.items()}
    got = vz._crown_intermediate_batched(gg_g, xl.to(gpu), xh.to(gpu), gpu, F32)
    lb, A, acc = vz._spec_backward_graph_batched(
        tight_g, xl.to(gpu), xh.to(gpu), gg_g, {q: (w.to(gpu), b) for q, (w, b) in spec.items()},
        gpu, F32, return_input_linear=True)
    ref = rb.spec_backward_batched(
        {L: (lo.float().double(), hi.float().double()) for L, (lo, hi) in tight_c.items()},
        xl.double(), xh.double(), gg_c, {q: (w.double(), b) for q, (w, b) in spec.items()},
        return_input_linear=True)
    # sums of at most 64 fp32 products per layer through three layers, against
    # 64 bits: a few 2^-24 of the row's size; a wrong bias dot is of the size
    # of the biases themselves (0.3)
    for name, g, r in (('lb', lb, ref[0]), ('A', A, ref[1]), ('acc', acc, ref[2])):
        r = r.reshape(g.shape)
        err = (g.cpu().double() - r).norm() / r.norm()
        assert err < 1e-5, (name, float(err))
    for L, (lo, hi) in tight_c.items():
        for g, r in zip(got[L], (lo, hi)):
            err = (g.cpu().double() - r).norm() / r.norm()
            assert err < 1e-5, (L, float(err))
