"""Replay of a captured forward for serving loops.

A FLARE model forward on the inference fast path is a fixed sequence of HIP launches (5 to 7 per block) with no host
round trip, so on small point clouds its cost is the launches themselves: an 8-block model of 64 channels at N = 4096 takes
0.32 ms eagerly, with one call into the library per block, and 0.36 ms replayed from a HIP graph, which leaves the
host free.  `GraphedForward` captures that sequence once per input
shape and replays it; there is no tracing compiler behind it and nothing is specialised beyond the shapes.

    fwd = GraphedForward(model, autocast_dtype=torch.bfloat16)
    y = fwd(x)            # first call with a new shape: warm-up + capture; later calls: copy in, replay

The returned tensor is the graph's static output buffer: it is overwritten by the next call with the same shape
(clone it to keep it).  A captured graph reads the 16-bit operand copies that the fused launches cache on the
modules (packed weights, the cast latent queries).  Every graph keeps those tensors alive, so an eager forward
that rebuilds a module's cache (another compute dtype, an optimizer step, `load_state_dict`) can never free
memory a graph still reads; and every call compares the versions and addresses of the module's parameters and
buffers with those seen at capture and captures again when any of them changed, so a replay never computes
with operands packed from old weights.  The parameters' and buffers' memory is held for that comparison until the shape is
captured again or `reset()` is called: a replaced one then never gets the address of the one it replaced.
"""
from __future__ import annotations

import contextlib

import torch

from . import fused

__all__ = ["GraphedForward"]


class GraphedForward:
    def __init__(self, module: torch.nn.Module, autocast_dtype=None, warmup: int = 3):
        self.module = module
        self.autocast_dtype = autocast_dtype
        self.warmup = warmup
        self._graphs = {}

    def reset(self):
        """Drop every captured graph (after a parameter update, or to free their memory pools)."""
        self._graphs.clear()

    def _context(self):
        if self.autocast_dtype is None:
            return contextlib.nullcontext()
        return torch.autocast("cuda", dtype=self.autocast_dtype)

    def _param_key(self):
        """Versions and addresses of everything the forward reads: an in-place update bumps the version, a
        replaced tensor changes the address."""
        return tuple((t.data_ptr(), t._version) for t in self._tensors())

    def _tensors(self):
        return list(self.module.parameters()) + list(self.module.buffers())

    def _cached_operands(self):
        """The operand caches the fused launches left on the modules during warm-up (their tensors' addresses are
        baked into the graph)."""
        keep = []
        for m in self.module.modules():
            for name in ("_flare_packed", "_flare_packed_few", "_q_cache"):
                c = getattr(m, name, None)
                if c is not None:
                    keep.append(c)
            keep += m.__dict__.get("_flare_plans", {}).values()
        return keep

    def _capture(self, x):
        static_x = x.clone()
        with torch.no_grad(), self._context():
            side = torch.cuda.Stream(device=x.device)
            side.wait_stream(torch.cuda.current_stream(x.device))
            with torch.cuda.stream(side):
                for _ in range(self.warmup):      # weight packing, kernel attributes, allocator warm-up
                    self.module(static_x)
            torch.cuda.current_stream(x.device).wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                static_y = self.module(static_x)
        return graph, static_x, static_y, self._param_key(), self._cached_operands(), [fused.hold(t) for t in self._tensors()]

    def __call__(self, x: torch.Tensor):
        if x.device.type != "cuda":
            raise ValueError("GraphedForward replays HIP graphs: the input must live on a HIP device")
        key = (tuple(x.shape), x.dtype, x.device.index)
        entry = self._graphs.get(key)
        if entry is not None and entry[3] != self._param_key():
            entry = None                      # parameters changed since the capture: its packed operands are stale
        if entry is None:
            if self.module.training:
                raise RuntimeError("GraphedForward captures inference forwards: call module.eval() first")
            entry = self._graphs[key] = self._capture(x)
        graph, static_x, static_y = entry[:3]
        static_x.copy_(x)
        graph.replay()
        return static_y
