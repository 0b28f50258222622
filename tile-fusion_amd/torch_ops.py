"""The reference's PyTorch operator surface, ``torch.ops.sw_gcn.*``, on ROCm tensors.

The reference registers these operators from C++ for CPU tensors
(binding-project/main.cpp:133-142) and its Python layers call them
(binding-project/gcn-e2e-training/FusedGCNLayer.py:6-45).  Here the same names, argument
orders and meanings are registered by ``lib/libtf_torch.so`` (``csrc/tf_torch.cpp``), which importing
this module loads; the arithmetic is done by
libtilefusion_hip on the tensors' own device memory (nothing is copied: the CSR arrays and
dense operands are wrapped and the
launches go to torch's current stream).  torch is plumbing: it owns the memory, the stream and the autograd graph.

    import importlib; importlib.import_module("tile-fusion_amd.torch_ops")
    adj = torch.sparse_csr_tensor(crow.int(), col.int(), val.float(), device="cuda")
    sched = torch.ops.sw_gcn.inspect_vt_ro(adj, in_dim, out_dim, 500000, threads)
    out = torch.ops.sw_gcn.fusedGeMMSpMM_vt_ro(adj, x, weight, sched, threads, 0)   # adj @ (x @ weight.T)

Differences from the reference, all forced by where the data lives:
  * Operands must be ROCm ("cuda") tensors; CPU tensors raise (there is no CPU path here).
    ``inspect`` / ``inspect_vt_ro`` only read the pattern and also accept CPU tensors.
  * The schedule tensors that the inspectors return describe the schedule in the binding
    project's layout (LevelPtr[3]; MixPtr[2p] = start of a partition's first-op ids,
    MixPtr[2p+1] = start of its second-op ids, MixPtr[2P] = end; Partition = the ids;
    Functions.cpp:588-622).  The executors do not parse them back: the native schedule for an
    adjacency and a pair of widths is built once and cached, so any schedule tensors that were
    made for the same adjacency select the same kernels.  MTileSize, CacheSize, NumThreads and
    MaxTileSize are accepted and ignored (tiles are sized by the LDS, not by a CPU cache).
  * Any widths: the library takes them as they are.
  * The backward pass uses the transpose of the adjacency (the reference multiplies by the
    adjacency itself, Functions.cpp:840-852, which is only right for a symmetric matrix).  Both of a layer's gradients
    come out of one sparse product, T = A^T G: grad X = T W, grad W = T^T X.
  * ``fusedGCN`` runs two layers with a ReLU between, Adj @ (relu(Adj @ (Feature @ Weight1^T)) @ Weight2^T), weights
    [out, in] (gcn-e2e-training/FusedGCNModule.py:14-18; binding-project/src/Functions.cpp:228-290).
  * What is built once per adjacency (host pattern, schedules, transpose) is cached for the last 32 of them, keyed by
    the tensors' addresses and version counters: an in-place change of the values or indices makes a new entry.
    The values themselves are read on every call, so that the forward pass honours writes that no version counter shows (through
    ``.data``, by another library, in the replay of a graph).  The transpose for the backward pass, and whether the matrix is its
    own transpose, are taken from the values once per entry: after such a write call ``clear_cache()`` before the next backward
    pass of a matrix whose transpose changes with it.
"""
import ctypes
import os

import torch

from . import binding as _b

__all__ = ["clear_cache", "SCHEMAS"]

_OPERATORS = ("inspect", "inspect_vt_ro", "executeFusedGeMMSpMM", "fusedGeMMSpMM", "fusedGeMMSpMM_vt_ro", "geMMSpMM_f_bw",
              "cachedSpMMGeMM", "unfused_gcn_forward", "fusedGCN")

_path = os.path.join(os.path.dirname(_b.lib_path()), "libtf_torch.so")
if not os.path.exists(_path):
    raise ImportError(f"{_path} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'`")
_b.lib()  # the library the operators stand on
torch.ops.load_library(_path)

SCHEMAS = {}
for _name in _OPERATORS:
    SCHEMAS[_name] = str(getattr(torch.ops.sw_gcn, _name).default._schema)[len("sw_gcn::" + _name):]


def clear_cache():
    """Drops the per-adjacency schedules, transposes and wrapped handles."""
    ctypes.CDLL(_path).sw_gcn_clear_cache()
