"""AdamW over tensors packed end to end in flat buffers (no counterpart in the
reference): every start is some elements past an aligned address, neighbours
share cache lines, and parameter, gradient and moments are offset differently.
Bit-exact against the oracle; the elements around the tensors keep their values.
"""

import numpy as np
import pytest
import torch

import oracle
from triton_muon_adamw.adamw import HipAdamW, solve_adamw_step

pytestmark = pytest.mark.gpu

HP = dict(lr=3e-4, betas=(0.9, 0.95), weight_decay=0.1, eps=1e-8)
SIZES = [1, 2, 3, 4, 5, 255, 1021, 1023, 1024, 1025, 1027, 2047, 4099, 70001]


def _packed(gpu, gen, std, dtype, shift):
    """(flat buffer of `shift` guards, the tensors end to end and 8 guards; its views)."""
    flat = (torch.randn(shift + sum(SIZES) + 8, generator=gen) * std).to(dtype).to(gpu)
    views, at = [], shift
    for n in SIZES:
        views.append(flat[at:at + n])
        at += n
    return flat, views


@pytest.mark.parametrize("pdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("gdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shifts", [(0, 0, 0, 0), (1, 2, 3, 1), (3, 1, 2, 0)])
def test_packed_tensors_bitexact_vs_oracle(gpu, pdt, gdt, shifts):
    gen = torch.Generator().manual_seed(21)
    pf, pv = _packed(gpu, gen, 0.02, pdt, shifts[0])
    gf, gv = _packed(gpu, gen, 1e-3, gdt, shifts[1])
    mf, mv = _packed(gpu, gen, 1.0, torch.float32, shifts[2])
    vf, vv = _packed(gpu, gen, 1.0, torch.float32, shifts[3])
    for t in mv + vv:
        t.zero_()
    before = [f.cpu().clone() for f in (pf, mf, vf)]
    params = [torch.nn.Parameter(t) for t in pv]
    opt = HipAdamW(params, **HP)
    for p, g, m, v in zip(params, gv, mv, vv):
        if pdt != gdt:
            p.grad_dtype = None
        p.grad = g
        opt.m[p], opt.v[p] = m, v
    ref = oracle.adamw.AdamWOracle([p.detach().float().cpu().numpy().copy() for p in params], **HP,
                                   param_bf16=pdt == torch.bfloat16)
    for _ in range(2):
        opt.step()
        ref.step([g.float().cpu().numpy() for g in gv])
    torch.cuda.synchronize()
    for i, p in enumerate(params):
        assert np.array_equal(p.detach().float().cpu().numpy(), ref.params[i]), f"tensor {i} ({p.numel()})"
        assert np.array_equal(mv[i].cpu().numpy(), ref.m[i])
        assert np.array_equal(vv[i].cpu().numpy(), ref.v[i])
    for old, new, s in zip(before, (pf, mf, vf), (shifts[0], shifts[2], shifts[3])):
        new = new.cpu()
        assert torch.equal(old[:s], new[:s]) and torch.equal(old[-8:], new[-8:])


@pytest.mark.parametrize("n", [1, 1023, 1025, 5003])
def test_one_tensor_at_any_offset(gpu, n):
    """The single-tensor function on a view one element into its buffer: the bits of an aligned copy."""
    gen = torch.Generator().manual_seed(n)
    aligned = [torch.randn(n, generator=gen).to(gpu) for _ in range(3)]
    aligned.append(torch.rand(n, generator=gen).to(gpu))
    shifted = [torch.cat([t[:1], t])[1:] for t in aligned]
    for ts in (aligned, shifted):
        solve_adamw_step(*ts, 3e-4, 0.1, 0.0975, 0.9, 0.95, 0.1, 1e-8)
    for a, b in zip(aligned, shifted):
        assert torch.equal(a, b)
