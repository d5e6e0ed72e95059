"""Sizes at the edges of the kernels' dispatch rules, against the oracle (bit for bit)."""

from __future__ import annotations

import pytest
import torch

from coffin_amd import _native, synth
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(1, 8), (513, 64), (16385, 64), (31, 72), (8193, 128), (8192, 136), (4097, 256), (17, 264),
                                 (2049, 512), (2048, 520), (5, 1024), (3, 1032)])
def test_quantiser_of_short_rows(orc, m, k):
    """Lane groups of 8 .. 64 per row, one or two rows each; rows that do not fill a workgroup."""
    x = synth.activations(m, k, synth.generator(m + k), outliers=True)
    q_ref, s_ref = orc.quant_act_i8(G.bits(x))
    q, s = G.quant(x.to(G.DEV))
    assert (q.cpu().numpy() == q_ref).all() and (s.cpu().numpy() == s_ref).all()
