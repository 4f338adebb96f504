"""Buffers that conv_bubbles keeps for graph replay: one output and one workspace
per box shape and stream, whatever the radii, filters and box lengths of the
calls ask for (the library keeps one graph per plan)."""
from types import SimpleNamespace

import torch

from conftest import pkg


def test_one_entry_per_shape_and_stream(monkeypatch):
    fb = pkg("Programs.find_HII_bubbles")
    monkeypatch.setattr(fb, "_graph_cache", {})
    s, other = SimpleNamespace(cuda_stream=7), SimpleNamespace(cuda_stream=9)
    d = torch.zeros(4, 4, 4)
    ion, work = fb._graph_buffers(d, 1000, s)
    assert ion.shape == d.shape and work.numel() == 1000
    # the same call, and one that asks for less, get the captured buffers
    for n in (1000, 400):
        again = fb._graph_buffers(d, n, s)
        assert again[0] is ion and again[1] is work
    # more replaces them, and a study over sizes leaves one entry
    for n in (1500, 1200, 4000, 700):
        assert fb._graph_buffers(d, n, s)[1].numel() >= n
    assert len(fb._graph_cache) == 1
    e = torch.zeros(4, 4, 4)
    assert fb._graph_buffers(e, 700, s)[1].numel() == 700 and len(fb._graph_cache) == 1
    fb._graph_buffers(d, 700, other)
    assert len(fb._graph_cache) == 2
