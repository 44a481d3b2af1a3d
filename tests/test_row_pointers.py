"""The binding's row addresses are those of the indexed rows, whatever the tensor's strides."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd"))
import nnet_mi355x as nm  # noqa: E402

F = torch.float64


@pytest.mark.parametrize("Y", [torch.zeros(14, 100, dtype=F), torch.zeros(87, 7, dtype=F)[:86], torch.zeros(30, 14, dtype=F).t(),
                               torch.zeros(9, 40, dtype=F)[::2, 3:], torch.zeros(1, 9, dtype=F).expand(4, 9),
                               torch.zeros(14, 0, dtype=F), [torch.zeros(5, dtype=F) for _ in range(3)],
                               tuple(torch.zeros(4, 6, dtype=F))])
def test_row_pointers(Y):
    assert nm._row_pointers(Y) == [Y[s].data_ptr() for s in range(len(Y))]
