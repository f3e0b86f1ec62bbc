"""The raw C-ABI helpers live in the package (mobulaop_amd/abi.py); tests use them under this name."""
from mobulaop_amd.abi import *   # noqa: F401,F403
from mobulaop_amd.abi import _begin, _end, _geom, _ptr   # noqa: F401


def poison_workspace(nbytes):
    """Leaves NaN in (at least) the first nbytes of the calling thread's workspace: a call that uses what
    it has not written shows it.  (The blocked copy of a map of NaN; enough boxes for all of it to be copied.)"""
    import torch
    x = torch.full((1, 32, (nbytes + (1 << 16) - 1) >> 16, 512), float('nan'), device='cuda')
    forward(x, torch.zeros((33, 5), device='cuda'), (1, 1), 1.0, 0)
