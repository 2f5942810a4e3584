"""Blocks of a stack that are not the plain ones: hooks, replaced methods, wrappers, subclasses."""
import torch

from cosmos_amd import DMBlock


class Wrapped(torch.nn.Module):
    def __init__(self, blk):
        super().__init__()
        self.inner = blk

    def forward(self, *args, **kw):
        return self.inner(*args, **kw)


class Older(DMBlock):
    """Takes the keywords that blocks took before a stack could hand over unjoined runs."""

    def forward(self, hidden_states, temb, image_rotary_emb, modality_segments=None, *, inplace=False, workspace=None, causal_prefix=0,
                prefix=None):
        return super().forward(hidden_states, temb, image_rotary_emb, modality_segments, inplace=inplace, workspace=workspace,
                               causal_prefix=causal_prefix, prefix=prefix)


class Doubled(DMBlock):
    def modulation(self, temb):
        return super().modulation(temb * 2.0)


def alter_block(kind, st, i):
    """Makes block i of the stack another than the plain one; returns what is done to the conditioning of (block 0, block 1):
    a factor on ``temb`` or a replacement for the block's own modulation layer."""
    blk, eff = st.blocks[i], [1.0, 1.0]
    lin = blk.adaLN_modulation
    if kind == "pre-hook on temb":
        blk.register_forward_pre_hook(lambda m, a: (a[0], a[1] * 2.0, *a[2:]))
        eff[i] = 2.0
    elif kind == "forward set on the instance":
        inner = blk.forward
        blk.forward = lambda x, temb, *a, **kw: inner(x, temb * 2.0, *a, **kw)
        eff[i] = 2.0
    elif kind == "modulation overridden":
        blk.__class__ = Doubled
        eff[i] = 2.0
    elif kind == "modulation set on the instance":
        own = blk.modulation
        blk.modulation = lambda temb: own(temb * 2.0)
        eff[i] = 2.0
    elif kind in ("pre-hook loads weights", "hook of the block before loads weights"):
        new = lin.weight.detach() * 3.0

        def load(*_):
            lin.weight.data = new

        if kind == "pre-hook loads weights":
            blk.register_forward_pre_hook(load)
        else:
            st.blocks[i - 1].register_forward_hook(load)
        eff[i] = torch.nn.Linear(lin.in_features, lin.out_features, device="meta")
        eff[i].weight, eff[i].bias = torch.nn.Parameter(new, requires_grad=False), lin.bias
    elif kind == "wrapper":
        st.blocks[i] = Wrapped(blk)
    elif kind == "older signature":
        blk.__class__ = Older
    return eff


ALTERED = [("pre-hook on temb", 0), ("pre-hook on temb", 1), ("forward set on the instance", 1), ("modulation overridden", 0),
           ("modulation overridden", 1), ("modulation set on the instance", 1), ("pre-hook loads weights", 0), ("pre-hook loads weights", 1),
           ("hook of the block before loads weights", 1), ("wrapper", 0), ("wrapper", 1), ("older signature", 0), ("older signature", 1)]
