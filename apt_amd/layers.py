"""GNN layers over sampled blocks without DGL.

The reference's DP models take their layers from DGL (examples/model.py:38-41);
its own layers (python/npc/model/sageconv.py:118-188 MPSAGEConv, Aggregate
:100-114) do A(XW) with the library's SpMM operator and get the backward pass
from the same operator with the edges reversed.  The layers here keep that
arithmetic on a Block of this package: the forward sum reads the sampler's
fixed-stride layout directly (no atomics), the backward sum runs over the
block's edges grouped by source (no atomics either), so both directions are
reproducible.
"""
import torch
from torch import nn
from torch.nn.modules.module import _has_any_global_hook

from . import ops  # noqa: F401  (loads the npc operators)


@torch._disable_dynamo      # (imports the compiler on its first call, which is made while compiling)
def _untraced(op, *args):
    return op(*args)


def _call(op, *args):
    """op(*args).  A compiler cannot look into an operator that launches kernels: it breaks its graph around the call."""
    return _untraced(op, *args) if torch.compiler.is_compiling() else op(*args)


class BlockAggregate:
    """out[d] = sum (or mean) over the block's edges (s -> d) of X[s], in X's dtype (sums are fp32 inside the kernels),
    with its gradient: npc.block_aggregate.  The backward pass takes the block's CSR if it has been emitted and
    otherwise orders the edges by source itself, without reading a size back."""

    @staticmethod
    def apply(block, X, mean):
        f = block.formats or {}
        return _call(torch.ops.npc.block_aggregate, block.relabeled, block.num_dst, block.fanout, X, bool(mean),
                     f.get("csr_indptr"), f.get("csr_indices"))


def _native_rows(x, weight):
    """Whether the library's products can take x (fp32 or bf16 GPU rows of the weight's dtype; autocast picks dtypes of
    its own)."""
    return (x.is_cuda and x.dim() == 2 and x.dtype == weight.dtype and x.dtype in (torch.float32, torch.bfloat16)
            and weight.is_cuda and weight.numel() > 0 and not torch.is_autocast_enabled("cuda"))


def _plain(layer):
    """A plain nn.Linear: no subclass, parametrization, replaced forward or hooks, all of which are the module's to run."""
    return (type(layer) is nn.Linear and "forward" not in layer.__dict__
            and not (layer._forward_hooks or layer._forward_pre_hooks or layer._backward_hooks
                     or layer._backward_pre_hooks or _has_any_global_hook()))


def _linear(layer, x):
    """layer(x), its products and gradients from npc.block_linear where they can be."""
    if _plain(layer) and _native_rows(x, layer.weight) and (layer.bias is None or layer.bias.dtype == x.dtype):
        return _call(torch.ops.npc.block_linear, x, layer.weight, layer.bias, False)
    return layer(x)


_RELU = (torch.relu, nn.functional.relu)      # activations that the kernels apply where they store a layer's result


def _is_relu(activation):
    return any(activation is f for f in _RELU)


class SAGEConv(nn.Module):
    """GraphSAGE layer, mean aggregator, with the reference's arithmetic
    (python/npc/model/sageconv.py:118-188): fc_self(h_dst) + fc_neigh(mean of
    the neighbours), the linear map applied before the aggregation when it
    shrinks the features."""

    def __init__(self, in_feats, out_feats, bias=True, activation=None):
        super().__init__()
        self.in_feats, self.out_feats, self.activation = in_feats, out_feats, activation
        self.fc_neigh = nn.Linear(in_feats, out_feats, bias=False)
        self.fc_self = nn.Linear(in_feats, out_feats, bias=bias)
        gain = nn.init.calculate_gain("relu")
        nn.init.xavier_uniform_(self.fc_self.weight, gain=gain)
        nn.init.xavier_uniform_(self.fc_neigh.weight, gain=gain)

    def forward(self, block, feat):
        """feat: [block.num_src, in_feats]; the first num_dst rows are the destinations."""
        wn, ws, b = self.fc_neigh.weight, self.fc_self.weight, self.fc_self.bias
        if (_plain(self.fc_neigh) and _plain(self.fc_self) and self.fc_neigh.bias is None and feat.is_cuda
                and feat.dim() == 2 and feat.dtype in (torch.float32, torch.bfloat16)
                and feat.dtype == wn.dtype == ws.dtype and (b is None or b.dtype == feat.dtype)
                and wn.shape == ws.shape == (self.out_feats, self.in_feats) and feat.shape[1] == self.in_feats > 0
                and self.out_feats > 0 and feat.shape[0] >= block.num_dst and not torch.is_autocast_enabled("cuda")):
            f = block.formats or {}
            relu = _is_relu(self.activation)
            rst = _call(torch.ops.npc.sage_layer, block.relabeled, block.num_dst, block.fanout, feat, wn, ws, b,
                        f.get("csr_indptr"), f.get("csr_indices"), relu)
            return rst if relu or self.activation is None else self.activation(rst)
        h_self = feat[:block.num_dst]
        if self.in_feats > self.out_feats:
            h_neigh = BlockAggregate.apply(block, _linear(self.fc_neigh, feat), True)
        else:
            h_neigh = _linear(self.fc_neigh, BlockAggregate.apply(block, feat, True))
        rst = _linear(self.fc_self, h_self) + h_neigh
        return self.activation(rst) if self.activation is not None else rst


class GraphConv(nn.Module):
    """GCN layer with the reference's arithmetic (python/npc/model/graphconv.py:
    159-232, MPGraphConv): the fanout stands in for the degrees in the
    normalisation ("both": fanout^-1/2 on either side, "left"/"right": 1/fanout
    on one), the weight is applied before the sum."""

    def __init__(self, in_feats, out_feats, norm="both", bias=True, activation=None):
        super().__init__()
        if norm not in ("none", "both", "right", "left"):
            raise KeyError(f'Invalid norm value. Must be either "none", "both", "right" or "left". But got "{norm}".')
        self.norm, self.activation = norm, activation
        self.weight = nn.Parameter(torch.empty(in_feats, out_feats))
        self.bias = nn.Parameter(torch.zeros(out_feats)) if bias else None
        nn.init.xavier_uniform_(self.weight)

    def forward(self, block, feat):
        fanout = float(block.fanout)
        w, b = self.weight, self.bias
        if (feat.is_cuda and feat.dim() == 2 and feat.dtype in (torch.float32, torch.bfloat16) and feat.dtype == w.dtype
                and w.is_cuda and w.dim() == 2 and feat.shape[1] == w.shape[0] and w.numel() > 0
                and (b is None or (b.is_cuda and b.dtype == feat.dtype and b.shape == w.shape[1:]))
                and not torch.is_autocast_enabled("cuda")):
            f = block.formats or {}
            relu = _is_relu(self.activation)
            rst = _call(torch.ops.npc.gcn_layer, block.relabeled, block.num_dst, block.fanout, feat, w, b,
                        *self._factors(fanout), f.get("csr_indptr"), f.get("csr_indices"), relu)
            return rst if relu or self.activation is None else self.activation(rst)
        left, right = self._factors(fanout)
        if self.norm in ("left", "both"):
            feat = feat * left
        h = (_call(torch.ops.npc.block_linear, feat, self.weight, None, True) if _native_rows(feat, self.weight)
             else torch.matmul(feat, self.weight))
        rst = BlockAggregate.apply(block, h, False)
        if self.norm in ("right", "both"):
            rst = rst * right
        if self.bias is not None:
            rst = rst + self.bias
        return self.activation(rst) if self.activation is not None else rst

    def _factors(self, fanout):
        """What the rows are multiplied with before and after the sum."""
        return {"none": (1.0, 1.0), "left": (1.0 / fanout, 1.0), "right": (1.0, 1.0 / fanout),
                "both": (fanout ** -0.5, fanout ** -0.5)}[self.norm]


class GATConv(nn.Module):
    """GAT layer (python/npc/model/gatconv.py:207-236: fc, attention logits,
    LeakyReLU, edge softmax, weighted sum, bias).  Everything between the dense
    product and the activation is npc.gat_layer, forward and backward: two
    kernels from the fixed-stride block, and for the gradients one over the
    destinations' edges, one over the sources and one for the parameters.
    A bf16 layer without gradients returns the fp32 sum (scores in fp32 too); the
    next bf16 layer takes it as its input."""

    def __init__(self, in_feats, out_feats, num_heads, negative_slope=0.2, bias=True, activation=None):
        super().__init__()
        self.num_heads, self.out_feats, self.negative_slope, self.activation = (num_heads, out_feats,
                                                                                negative_slope, activation)
        self.fc = nn.Linear(in_feats, out_feats * num_heads, bias=False)
        self.attn_l = nn.Parameter(torch.empty(num_heads, out_feats))
        self.attn_r = nn.Parameter(torch.empty(num_heads, out_feats))
        self.bias = nn.Parameter(torch.zeros(num_heads * out_feats)) if bias else None
        gain = nn.init.calculate_gain("relu")
        nn.init.xavier_normal_(self.fc.weight, gain=gain)
        nn.init.xavier_normal_(self.attn_l, gain=gain)
        nn.init.xavier_normal_(self.attn_r, gain=gain)

    def forward(self, block, feat):
        if not torch.is_grad_enabled() and feat.dtype == torch.float32 and self.fc.weight.dtype == torch.bfloat16:
            feat = feat.bfloat16()
        ft = _linear(self.fc, feat).view(block.num_src, self.num_heads, self.out_feats)
        f = block.formats or {}
        inside = self.bias is not None and self.bias.dtype == ft.dtype
        relu = _is_relu(self.activation) and (inside or self.bias is None)
        rst = _call(torch.ops.npc.gat_layer, block.relabeled, block.num_dst, block.fanout, ft, self.attn_l, self.attn_r,
                    self.bias if inside else None, self.negative_slope, f.get("csr_indptr"),
                    f.get("csr_indices"), f.get("csr_eids"), f.get("csc_indptr"), relu, True)
        if self.bias is not None and not inside:      # a bias of another type than the rows: torch's promotion
            rst = rst + self.bias.view(1, self.num_heads, self.out_feats)
        return rst if relu or self.activation is None else self.activation(rst)
