"""What the torch front end's host path decides before any kernel runs: operands it refuses, plans it picks, how it is
loaded.  No GPU is needed; tensors are on the CPU, which the calls refuse last."""

import pytest
import torch
import torch.autograd.forward_ad as fwAD

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import moe


def _routing(tokens, top_k):
    slots = torch.arange(tokens * top_k, dtype=torch.int32)
    return moe.Routing(torch.tensor([tokens * top_k], dtype=torch.int32), slots, slots, tokens, top_k)


@pytest.mark.parametrize("call", ["gmm x", "gmm A", "tgmm x", "tgmm y", "dispatch", "combine y", "combine weights"])
@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_tangents_are_refused(call, grad):
    with fwAD.dual_level():
        plain = lambda *s: torch.randn(*s)
        dual = lambda *s: fwAD.make_dual(torch.randn(*s, requires_grad=grad), torch.randn(*s))
        gs = torch.tensor([4], dtype=torch.int32)
        calls = {
            "gmm x": lambda: rd.gmm(dual(4, 8), plain(1, 8, 8), gs),
            "gmm A": lambda: rd.gmm(plain(4, 8), dual(1, 8, 8), gs),
            "tgmm x": lambda: rd.tgmm(dual(4, 8), plain(4, 8), gs),
            "tgmm y": lambda: rd.tgmm(plain(4, 8), dual(4, 8), gs),
            "dispatch": lambda: moe.dispatch(dual(4, 8), _routing(4, 1)),
            "combine y": lambda: moe.combine(dual(4, 8), _routing(4, 1)),
            "combine weights": lambda: moe.combine(plain(4, 8), _routing(4, 1), dual(4, 1)),
        }
        with pytest.raises(NotImplementedError, match="forward-mode"):
            calls[call]()
