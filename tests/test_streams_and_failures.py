"""Calls on streams of the caller's own, tensors that are none of the plain ones, and resources that fail."""
import numpy as np
import pytest
import torch

import bitnet_hip as bh
from helpers import synth_activations, synth_weights


def _layer(rng, n, k):
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n))
    layer.update_weights(torch.from_numpy(synth_weights(rng, n, k)).cuda())
    return layer


@pytest.mark.gpu
def test_tensors_without_strides_or_storage_are_errors():
    """A sparse tensor refuses to say whether it is contiguous, one inside vmap has no storage: an exception in Python, and the
    process goes on."""
    bh.init(0)
    rng = np.random.default_rng(1)
    layer = _layer(rng, 64, 64)
    dec = bh.DecoderProjections(1, 64, 64, 4, 2, 16, max_tokens=4)
    x = torch.eye(64, device="cuda")[:4]
    sparse = x.to_sparse()
    calls = [lambda t: layer.forward(t), lambda t: layer.forward(x, gamma=t), lambda t: layer.forward(x, residual=t),
             lambda t: layer.forward(x, out=t), lambda t: bh.forward_multi([layer], t), lambda t: bh.forward_multi([layer], x, gamma=t),
             lambda t: dec.decode(t), lambda t: dec.decode(x, out=t), lambda t: bh.abs_max(t),
             lambda t: bh.quantize_activations_scaled(t, bh.QuantizationPrecision.EightBit, 1.0),
             lambda t: bh.DynamicActivationQuantizer(bh.ActivationQuantizationConfig()).quantize_dynamic(t)]
    for call in calls:
        with pytest.raises(RuntimeError):
            call(sparse)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda row: layer.forward(row[None]))(x)
    assert torch.isfinite(layer.forward(x)).all()
