"""Hooks on a projection see its calls, and change what they return, also where a kernel of its own does the projection's work with what follows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [1, 40, 192, 200])
def test_gate_and_up(rows):
    from aphrodite_engine_amd import mixer_ops as mops
    from aphrodite_engine_amd.mixers import GatedMLP
    with torch.device(DEV):
        mlp = GatedMLP(256, 512, mops.ACT_SILU, torch.bfloat16)
    g = torch.Generator(device=DEV).manual_seed(rows)
    for lin in (mlp.gate_up, mlp.down):
        lin.weight.data.copy_(torch.randn(lin.weight.shape, generator=g, device=DEV) * 0.1)
    h = torch.randn(rows, 256, generator=g, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        plain, seen = mlp(h), []
        assert plain.abs().max() > 0
        handle = mlp.gate_up.register_forward_hook(lambda module, args, out: (seen.append(out.shape), out.zero_())[1])
        assert not mlp(h).any() and seen == [(rows, 1024)]
        handle.remove()
        handle = mlp.gate_up.register_forward_pre_hook(lambda module, args: (torch.zeros_like(args[0]), ))
        assert not mlp(h).any()
        handle.remove()
        handle = torch.nn.modules.module.register_module_forward_hook(lambda module, args, out: seen.append(module))
        mlp(h)
        handle.remove()
        assert mlp.gate_up in seen
        assert torch.equal(mlp(h), plain)
        mlp.gate_up.bias = torch.nn.Parameter(torch.full((1024, ), -50.0, dtype=torch.bfloat16, device=DEV))       # (shuts every gate)
        assert mlp(h).abs().max() < 1e-6
