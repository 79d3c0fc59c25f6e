"""HyperConnection under a symbolic trace: the logits are recorded as torch operations (no GPU needed)."""
import pytest
import torch

from kernelswift_amd.mhc import HyperConnection


@pytest.mark.parametrize("grad", [False, True])
def test_symbolic_trace_records_the_logits(grad):
    hc = HyperConnection(64).requires_grad_(grad)
    graph = torch.fx.symbolic_trace(hc).graph
    names = [str(n.target) for n in graph.nodes]
    assert any("matmul" in n for n in names) and any("mhc_pre" in n for n in names)
    assert not any("mhc_input" in n for n in names)
