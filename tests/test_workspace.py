"""Workspace sizes of the layer: they never fall as the batch grows (a caller
sizes one buffer for its largest batch), and the no-allocation call takes the
batches that its fixed scratch always held. No GPU call: the checks come before
the device and, with null tensors, before any launch."""
import ctypes as C

import pytest

from inferno_amd import Q2_K, Q4_K, Q6_K, Q8_0, lib, ops
from inferno_amd._lib import LayerDesc


def _desc(H, E, I, k, Is, quant=Q2_K, down=Q2_K, shared=Q8_0, shared_down=Q8_0):
    d = LayerDesc()
    d.hidden, d.experts, d.intermediate, d.top_k = H, E, I, k
    d.quant, d.down_quant, d.score_fn = quant, down, 0
    d.norm_topk_prob, d.routed_scaling_factor = 1, 1.0
    d.gate_bytes = d.up_bytes = ops.matrix_bytes(quant, E * I, H)
    d.down_bytes = ops.matrix_bytes(down, E * H, I)
    d.shared_intermediate, d.shared_quant, d.shared_down_quant = Is, shared, shared_down
    if Is:
        d.shared_gate_bytes = d.shared_up_bytes = ops.matrix_bytes(shared, Is, H)
        d.shared_down_bytes = ops.matrix_bytes(shared_down, H, Is)
    return d


@pytest.mark.parametrize("H", [256, 1280, 2048, 2816, 3328, 6144])
@pytest.mark.parametrize("E,I,k,Is", [(8, 256, 1, 0), (64, 768, 8, 768), (96, 256, 2, 0),
                                      (160, 1280, 6, 512), (256, 512, 10, 2048)])
def test_need_does_not_fall(H, E, I, k, Is):
    for formats in ({}, dict(quant=Q4_K, down=Q6_K, shared=Q4_K, shared_down=Q6_K)):
        d = _desc(H, E, I, k, Is, **formats)
        need = [lib().inferno_moe_layer_workspace_bytes(C.byref(d), T) for T in range(1, 700)]
        assert need == sorted(need)


# The largest batches of these layers (H, E, I, k, Is) that the scratch holds
# when the router logits are in powers of two of chunks and there are no lists
# of 16-row tiles; neither may take room from them.
@pytest.mark.parametrize("shape,T", [
    ((6400, 96, 256, 3, 512), 160), ((1536, 128, 1536, 4, 0), 315), ((3584, 64, 768, 5, 512), 192),
    ((2816, 96, 768, 10, 768), 140), ((1792, 64, 768, 2, 1536), 450), ((5120, 256, 2304, 10, 0), 66),
    ((6400, 256, 1024, 1, 0), 192), ((256, 128, 2304, 8, 0), 195)])
def test_no_alloc_takes_what_fitted(shape, T):
    d = _desc(*shape)
    st = lib().inferno_moe_layer_forward_noalloc(None, C.byref(d), None, 0, None, T, None, None, None)
    assert st != -2, ops.lib().inferno_last_error()  # -2: above the scratch
    st = lib().inferno_moe_layer_forward_noalloc(None, C.byref(d), None, 0, None, 4 * T, None, None, None)
    assert st == -2


def test_need_of_an_unset_layer():
    assert lib().inferno_moe_layer_workspace_bytes(C.byref(LayerDesc()), 4) > 0  # no division by its zeros
