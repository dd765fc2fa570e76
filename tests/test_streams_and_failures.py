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


def _calls(rng):
    """name -> (call(x, stream), inputs): calls that take scratch or make their own results, through the native path and through
    the checked one (a Parameter is not the plain tensor the native path takes)."""
    bh.init(0)
    wide, other = _layer(rng, 640, 2560), _layer(rng, 96, 2560)
    gamma = torch.rand(2560, device="cuda") + 0.5
    checked = torch.nn.Parameter(gamma, requires_grad=False)
    dec = bh.DecoderProjections(2, 256, 512, 4, 2, 64, max_tokens=32)
    for layer in range(2):
        for p in range(7):
            dec.projection(layer, p).update_weights(torch.from_numpy(synth_weights(rng, *dec.proj_shape(p))).cuda())
    return {
        "forward": (lambda x, s: [wide.forward(x, gamma=gamma, stream=s)], (48, 2560)),
        "forward_checked": (lambda x, s: [wide.forward(x, gamma=checked, stream=s)], (48, 2560)),
        "forward_multi": (lambda x, s: bh.forward_multi([wide, other], x, gamma=gamma, stream=s), (48, 2560)),
        "decode": (lambda x, s: [dec.decode(x, stream=s)], (32, 256)),
        "quantize_rows": (lambda x, s: list(bh.quantize_activations_i8(x, gamma, stream=s)[:2]), (48, 2560)),
        "quantize_weights": (lambda x, s: list(bh.quantize_weights(x, stream=s)[:2]), (48, 2560)),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["forward", "forward_checked", "forward_multi", "decode", "quantize_rows", "quantize_weights"])
def test_calls_on_another_stream_share_no_memory_with_the_current_one(name):
    """A call on a stream that is held up: what the current stream allocates, fills and frees meanwhile is not the call's scratch
    or result, before or after it, and a result that the current stream reads and drops is not handed out again too early."""
    rng = np.random.default_rng(2)
    call, shape = _calls(rng)[name]
    xs = [torch.from_numpy(synth_activations(rng, *shape)).cuda() for _ in range(2)]
    want = [[t.clone() for t in call(x, None)] for x in xs]
    current, side = torch.cuda.current_stream(), torch.cuda.Stream()
    hold = lambda: torch.cuda._sleep(20_000_000)
    same = lambda got, ref: all(torch.equal(a, b) for a, b in zip(got, ref))

    def litter(value):  # blocks of every size the call may have used, written by the current stream
        keep = [torch.empty((n,), dtype=torch.uint8, device="cuda") for n in
                [t.numel() * t.element_size() for t in want[0]] + [1 << b for b in range(9, 22)] * 2]
        for t in keep:
            t.fill_(value)
        return keep

    for x, ref in zip(xs, want):
        litter(0)  # the allocator now holds free blocks of the current stream
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            hold()
        got = call(x, side)
        keep = litter(85)
        current.synchronize()
        side.synchronize()
        assert same(got, ref)
        # the result dropped before its kernels have run
        with torch.cuda.stream(side):
            hold()
        call(x, side)
        keep = litter(51)
        torch.cuda.synchronize()
        assert all((t == 51).all() for t in keep)
        # blocks that the current stream has freed but not finished with
        hold()
        del keep, got
        litter(119)
        got = call(x, side)
        torch.cuda.synchronize()
        assert same(got, ref)
    # a result read and dropped on the current stream, and the next call on the other one
    got = call(xs[0], side)
    current.wait_stream(side)
    hold()
    read = [t.clone() for t in got]
    del got
    again = call(xs[1], side)
    torch.cuda.synchronize()
    assert same(read, want[0]) and same(again, want[1])


@pytest.mark.gpu
def test_quantisers_on_another_stream_return_what_their_kernels_wrote():
    """The figures and bytes of a quantiser on a stream that is held up, read on the current stream as soon as the call is back."""
    bh.init(0)
    rng = np.random.default_rng(3)
    x = torch.from_numpy(synth_weights(rng, 96, 512)).cuda()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    weights = bh.BitNetWeightQuantizer()
    for call in (lambda s: (a := bh.absmax_quantize_activations(x, stream=s)) and (a.stats, a.values, a.scales),
                 lambda s: (w := weights.quantize(x, stream=s)) and (w.stats, w.values, w.packed, w.scales),
                 lambda s: ({}, *bh.quantize_weights(x, stream=s)[:2])):
        stats, *tensors = call(None)
        tensors = [t.clone() for t in tensors]
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(20_000_000)
        got, *other = call(side)
        assert got == stats and all(torch.equal(a, b) for a, b in zip(other, tensors))


@pytest.mark.gpu
def test_a_step_is_recorded_while_another_thread_captures():
    """The third, recorded call of a step while another thread is in a capture of its own (torch's default, the global mode): the
    capture is whole afterwards, and so are the step's results."""
    import threading

    bh.init(0)
    rng = np.random.default_rng(4)
    dec = bh.DecoderProjections(3, 256, 512, 4, 2, 64, max_tokens=4)
    for layer in range(3):
        for p in range(7):
            dec.projection(layer, p).update_weights(torch.from_numpy(synth_weights(rng, *dec.proj_shape(p))).cuda())
    x = torch.from_numpy(synth_activations(rng, 2, 256)).cuda()
    want, out, a = dec.decode(x), torch.empty_like(x), torch.ones(1000, device="cuda")
    mine = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(2):
        dec.decode(x, out=out, stream=mine)
    mine.synchronize()
    out.zero_()
    torch.cuda.synchronize()
    inside, stepped, errors = threading.Event(), threading.Event(), []

    def steps():
        try:
            assert inside.wait(30)
            for _ in range(2):  # recorded, replayed
                dec.decode(x, out=out, stream=mine)
        except BaseException as exc:
            errors.append(exc)
        finally:
            stepped.set()

    worker = threading.Thread(target=steps)
    worker.start()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        b = a * 2
        inside.set()
        assert stepped.wait(30)
        b = b + 1
    worker.join()
    assert not errors
    for value in (1.0, 4.0):
        a.fill_(value)
        graph.replay()
        torch.cuda.synchronize()
        assert (b == 2 * value + 1).all() and torch.equal(out, want)
