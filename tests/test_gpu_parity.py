"""Parity of the HIP path (through the C ABI) with the CPU oracle on the same seeded inputs.

Bar: int8 activations, packed bytes and int32 accumulators bit-exact; f32 scales and outputs compared
bit-exact where the oracle and the kernel perform the same IEEE operations, and in any case within
1e-5 relative error (the tolerance the path's specification states)."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import bitnet_hip as bh
from helpers import golden_vectors, rel_err, synth_activations, synth_weights
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
G = golden_vectors()
f32 = np.float32
REL_TOL = 1e-5


@pytest.fixture(scope="module", autouse=True)
def _device():
    bh.init(0)
    info = bh.device_info()
    assert info["arch"].startswith("gfx950")
    yield
    torch.cuda.synchronize()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    return t.detach().cpu().numpy()


# ---- P1 ------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("case", G["unpack_2bit"], ids=lambda c: c["source"].split(":")[0].split("/")[-1])
def test_unpack_reference_bytes(case):
    got = host(bh.unpack_ternary_2bit(dev(np.array(case["bytes"], dtype=np.uint8)), case["count"]))
    assert got.tolist() == case["expected"]


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 1000, 10000, 2560 * 640])
def test_pack_unpack_match_oracle(n):
    rng = np.random.default_rng(n)
    w = rng.integers(-1, 2, size=n).astype(np.int8) if n not in (1000, 10000) else (np.arange(n) % 3 - 1).astype(np.int8)
    packed = bh.BitPacked2BitPacker().pack(dev(w))
    assert np.array_equal(host(packed), orc.pack_2bit(w))
    assert np.array_equal(host(bh.BitPacked2BitPacker().unpack(packed, n)), w)


def test_unpack_every_byte_value():
    allb = np.arange(256, dtype=np.uint8)
    assert np.array_equal(host(bh.unpack_ternary_2bit(dev(allb), 1024)), orc.unpack_2bit(allb, 1024))


@pytest.mark.parametrize("n,k", [(16, 256), (17, 257), (5, 7), (33, 100), (640, 2560), (2560, 6912)])
@pytest.mark.parametrize("layout", [bh.LAYOUT_OUT_IN, bh.LAYOUT_IN_OUT])
def test_retile_is_a_bijection(n, k, layout):
    rng = np.random.default_rng(n * 7 + k)
    w = rng.integers(-1, 2, size=(n, k)).astype(np.int8)
    src = w if layout == bh.LAYOUT_OUT_IN else np.ascontiguousarray(w.T)
    tiled = bh.retile_weights(dev(orc.pack_2bit(src)), n, k, layout)
    assert tiled.numel() == bh.tiled_size(n, k)
    back = host(bh.untile_weights(tiled, n, k))
    assert np.array_equal(back, orc.pack_2bit(w))


def test_retile_canonicalises_code_three():
    # code 3 decodes to weight 0 in every reference decoder; the tiled layout stores it as code 1
    n, k = 16, 256
    packed = np.full((n * k // 4,), 0xFF, dtype=np.uint8)
    tiled = bh.retile_weights(dev(packed), n, k)
    assert np.all(host(tiled) == 0x55)
    a = dev(np.full((1, k), 77, dtype=np.int8))
    acc, _ = bh.matmul_w2a8(tiled, a, n, want_out=False)
    assert not host(acc).any()


# ---- W1 ------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("n,k", [(4, 4), (3, 5), (64, 128), (640, 2560), (2560, 2560)])
def test_quantize_weights_absmean_bit_exact(n, k):
    rng = np.random.default_rng(n + k)
    w = synth_weights(rng, n, k)
    packed, w_scale, q = bh.quantize_weights(dev(w), want_i8=True)
    q_ref, s_ref = orc.quantize_weights_absmean(w)
    assert host(w_scale)[0] == s_ref
    assert np.array_equal(host(q), q_ref)
    assert np.array_equal(host(packed), orc.pack_2bit(q_ref))


@pytest.mark.parametrize("n,k", [(1, 4), (3, 127), (16, 64), (33, 1023), (64, 1024), (65, 1028), (2304, 65), (2305, 260), (4099, 4092), (6912, 3072)])
@pytest.mark.parametrize("method,factor", [(0, 0.5), (1, 0.7), (1, 0.0), (1, -0.25), (1, float("inf"))])
def test_quantize_weights_with_row_scratch_bit_exact(n, k, method, factor):
    """Row sums of the caller's, apart from the codes (the sum and the codes in one launch), against those in the codes' place: sizes around a
    chunk of 1024 weights, around 36 x 64 row sums, and with more chunks than the registers hold; with too little scratch the call is the other one."""
    lib = bh.load_library()
    rng = np.random.default_rng(n + k)
    w = dev(synth_weights(rng, n, k))
    w.view(-1)[::7] = 0.0
    need = lib.bitnet_hip_quantize_weights_scratch(n)
    results = []
    for room in (need, need - 8, None):
        packed, scale = torch.full(((n * k + 3) // 4,), 0xAA, dtype=torch.uint8, device="cuda"), torch.zeros(1, device="cuda")
        scratch = torch.full((need // 8,), float("nan"), dtype=torch.float64, device="cuda")
        args = (w.data_ptr(), n, k, method, factor, packed.data_ptr(), scale.data_ptr(), None)
        stream = torch.cuda.current_stream().cuda_stream
        rc = (lib.bitnet_hip_quantize_weights(*args, stream) if room is None else
              lib.bitnet_hip_quantize_weights_with(*args, scratch.data_ptr(), room, stream))
        assert rc == 0
        results.append((host(packed), host(scale)))
    for packed, scale in results[1:]:
        assert np.array_equal(results[0][0], packed) and results[0][1] == scale
    if method == 0 and n * k < 1 << 20:
        q_ref, s_ref = orc.quantize_weights_absmean(host(w))
        assert results[0][1][0] == s_ref and np.array_equal(results[0][0], orc.pack_2bit(q_ref))


@pytest.mark.parametrize("n,k", [(3, 256), (37, 768), (129, 512), (700, 2560), (33, 8192), (4099, 1024), (4000, 5120), (5130, 4096)])
def test_quantize_weights_of_whole_chunks_bit_exact(n, k):
    """Rows that are a quarter of whole chunks: the chunks dealt out by the die that read them, the last ones in order, up to 21 million weights and above."""
    for method, factor in ((0, 0.5), (1, 0.7)):
        test_quantize_weights_with_row_scratch_bit_exact(n, k, method, factor)


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("bits", [0xFFFFFFFF, 0x7FFFFFFF, 0x7FC00000, 0xFFC00001, 0x7F800000, 0xFF800000])
def test_quantize_weights_with_a_weight_that_is_no_number(bits, method):
    """A NaN of any payload or an infinity among the weights: with row sums of the caller's the same codes as without, byte for byte."""
    lib = bh.load_library()
    rng = np.random.default_rng(bits & 0xFFFF)
    n, k = 24, 1028
    w = synth_weights(rng, n, k)
    w.view(np.uint32)[5, 77] = bits
    w.view(np.uint32)[23, 1027] = bits
    w = dev(w)
    scratch = torch.empty((n,), dtype=torch.float64, device="cuda")
    results = []
    for room in (0, 8 * n):
        packed, scale = torch.full((n * k // 4,), 0xAA, dtype=torch.uint8, device="cuda"), torch.zeros(1, device="cuda")
        assert lib.bitnet_hip_quantize_weights_with(w.data_ptr(), n, k, method, 0.5, packed.data_ptr(), scale.data_ptr(), None, scratch.data_ptr(), room,
                                                    torch.cuda.current_stream().cuda_stream) == 0
        results.append((host(packed), host(scale).view(np.uint32)))
    assert np.array_equal(results[0][0], results[1][0]) and np.array_equal(results[0][1], results[1][1])


def test_quantize_weights_reference_vectors():
    c = G["quantize_batch"]
    w = np.array([c["input"]], dtype=f32)
    # threshold form with the reference's factor 0.5 on its own vector (mean|w| of this vector is 1.2167)
    _, s, q = bh.quantize_weights(dev(w), method=bh.TERNARY_MEAN_THRESHOLD, threshold_factor=0.5, want_i8=True)
    assert host(s)[0] == orc.absmean(w)
    assert host(q)[0].tolist() == orc.ternarize_threshold(w, f32(0.5) * orc.absmean(w))[0].tolist()
    for case in G["absmean"]:
        _, s, _ = bh.quantize_weights(dev(np.array([case["input"]], dtype=f32)))
        assert abs(float(host(s)[0]) - case["expected"]) < 1e-6
    # ties and a zero matrix
    w = np.array([[0.5, -0.5, 0.25, 1.5, -7.0, 0.0, 1.0, -1.0]], dtype=f32)
    _, s, q = bh.quantize_weights(dev(w), want_i8=True)
    assert np.array_equal(host(q), orc.ternarize_roundclip(w, host(s)[0]))
    _, s, q = bh.quantize_weights(dev(np.zeros((4, 8), dtype=f32)), want_i8=True)
    assert host(s)[0] == 0.0 and not host(q).any()


@pytest.mark.parametrize("method", range(5))
@pytest.mark.parametrize("normalize,t,custom", [(True, 3.0, None), (False, 0.0, None), (True, 0.0, 0.45), (False, 2.0, None)])
def test_reference_weight_pipeline_bit_exact(method, normalize, t, custom):
    """BitNetWeightQuantizer::quantize with each TernaryMethod: ternary values, packed bytes, the scale and all twelve
    f32 scalars of the pipeline equal to the oracle's, bit for bit (stated bar: q exact, scale within 1e-6 relative)."""
    rng = np.random.default_rng(method * 10 + int(normalize) + int(t))
    for n, k in ((48, 200), (5, 7), (640, 2560)):
        w = (0.3 + 1.7 * rng.standard_normal((n, k))).astype(f32)
        w[rng.random(w.shape) < 0.01] *= f32(6.0)
        cfg = bh.WeightQuantizationConfig(normalize_weights=normalize, outlier_threshold=t, ternary_method=method,
                                          custom_threshold_factor=custom)
        got = bh.BitNetWeightQuantizer(cfg).quantize(dev(w))
        q_ref, s_ref, _, st_ref = orc.quantize_weights_reference(w, method=method, normalize=normalize, outlier_threshold=t,
                                                                 custom_factor=custom, want_details=True)
        assert np.array_equal(host(got.values), q_ref)
        assert np.array_equal(host(got.packed), orc.pack_2bit(q_ref))
        assert abs(float(host(got.scales)[0]) - float(s_ref)) <= 1e-6 * abs(float(s_ref))
        assert host(got.scales)[0] == s_ref
        for name, v in st_ref.items():
            assert f32(got.stats[name]) == v, (name, got.stats[name], v)


@pytest.mark.parametrize("n,k", [(9, 252), (9, 256), (9, 260), (5, 510), (9, 512), (5, 516), (9, 772), (9, 1284), (2113, 260)])
@pytest.mark.parametrize("kind", ["plain", "constant", "zero_dividend", "far"])
def test_reference_weight_pipeline_groups_of_columns(n, k, kind):
    """Widths around the groups of columns that the passes take at once and rows around the batches of row sums; weights equal to the
    mean (a zero dividend) and dividends out of the short division's range, which take the plain one.  Bit for bit, as above."""
    rng = np.random.default_rng(n + k)
    w = (0.3 + 1.7 * rng.standard_normal((n, k))).astype(f32)
    if kind == "constant":
        w[:] = f32(0.25)
    elif kind == "zero_dividend":  # mean exactly 0: a tensor and its negative, with zeros
        w[rng.random(w.shape) < 0.3] = 0
        w[n // 2 * 2:] = 0
        w[1:n // 2 * 2:2] = -w[0:n // 2 * 2:2]
    elif kind == "far":
        w[n // 2, k // 3] = f32(2.0) ** 64
        w *= f32(2.0) ** -4
    got = bh.BitNetWeightQuantizer().quantize(dev(w))
    q_ref, s_ref, _, st_ref = orc.quantize_weights_reference(w, method=0, normalize=True, outlier_threshold=3.0, want_details=True)
    assert np.array_equal(host(got.values), q_ref)
    assert np.array_equal(host(got.packed), orc.pack_2bit(q_ref))
    assert host(got.scales)[0] == s_ref
    for name, v in st_ref.items():
        assert f32(got.stats[name]) == v, (name, got.stats[name], v)


def test_reference_weight_pipeline_through_the_layer():
    """BitLinear with the reference's default quantiser (MeanThreshold, normalise, clip 3.0: layer.rs:53-63): the layer then
    holds the oracle's codes and scale, and forward follows from them."""
    rng = np.random.default_rng(21)
    n, k = 96, 512
    w = synth_weights(rng, n, k)
    for method, factor in ((bh.TERNARY_REF_MEAN_THRESHOLD, 0.0), (bh.TERNARY_REF_OPTIMAL_THRESHOLD, 0.0),
                           (bh.TERNARY_REF_ADAPTIVE_THRESHOLD, 0.0), (bh.TERNARY_REF_DETSTE, 0.9)):
        layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, ternary_method=method, threshold_factor=factor), "ref")
        layer.update_weights(dev(w))
        q_ref, s_ref = orc.quantize_weights_reference(w, method=method - bh.TERNARY_REF_MEAN_THRESHOLD,
                                                      custom_factor=factor or None)
        packed, ws = layer.get_quantized_weights()
        assert ws == s_ref and np.array_equal(packed.numpy(), orc.pack_2bit(q_ref))
        x = synth_activations(rng, 3, k)
        ref = orc.bitlinear_forward(x, orc.pack_2bit(q_ref), n, float(s_ref))[0]
        assert np.array_equal(host(layer.forward(dev(x))), ref)
    with pytest.raises(bh.BitLinearError) as ei:
        bh.BitNetWeightQuantizer(bh.WeightQuantizationConfig(custom_threshold_factor=2.5))
    assert ei.value.kind == "InvalidConfig"
    with pytest.raises(bh.BitLinearError):
        bh.BitNetWeightQuantizer().quantize(torch.ones(4, device="cuda"))
    # an all-zero tensor: no non-zero code, scale 1.0 (compute_ternary_scale, weights.rs:554-556)
    z = bh.BitNetWeightQuantizer(bh.WeightQuantizationConfig(normalize_weights=False, outlier_threshold=0.0)).quantize(
        torch.zeros(4, 8, device="cuda"))
    assert not host(z.values).any() and host(z.scales)[0] == 1.0


# ---- A2 ------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("precision", [bh.QuantizationPrecision.OneFiveFiveBit, bh.QuantizationPrecision.EightBit])
@pytest.mark.parametrize("shape", [(4,), (32, 128), (3, 5, 7), (300, 4096 + 17), (1, 1)])
def test_absmax_quantize_activations_bit_exact(precision, shape):
    """absmax_quantize_activations (one scale per tensor): values, scale, error, min and max equal to the oracle's."""
    rng = np.random.default_rng(len(shape) * 10 + precision)
    x = (rng.standard_normal(shape) * 3).astype(f32)
    if x.size >= 4:
        x.flat[:4] = [100.0, -50.0, 25.0, -75.0]  # the reference's vector (activations.rs:815-840)
    got = bh.absmax_quantize_activations(dev(x), precision)
    q_ref, st = orc.absmax_quantize_activations(x, precision)
    assert np.array_equal(host(got.values), q_ref) and got.original_shape == shape
    assert f32(got.stats["scale_factor"]) == st["scale"] and host(got.scales)[0] == st["scale"]
    assert f32(got.stats["quantization_error"]) == st["mse"]
    assert f32(got.stats["min_value"]) == st["min"] and f32(got.stats["max_value"]) == st["max"]
    assert got.stats["elements_count"] == x.size and got.stats["compression_ratio"] > 1.0 and got.zero_points is None
    assert got.effective_bit_width() == (1.58 if precision == 0 else 8.0)
    deq = bh.ActivationQuantizer(precision).dequantize(got)
    assert tuple(deq.shape) == shape
    zeros = bh.absmax_quantize_activations(torch.zeros(2, 2, device="cuda"), precision)
    assert not host(zeros.values).any() and zeros.stats["scale_factor"] == 1.0
    with pytest.raises(bh.BitLinearError) as ei:
        bh.absmax_quantize_activations(dev(x), 7)
    assert ei.value.kind == "Unsupported"


@pytest.mark.parametrize("precision", [bh.QuantizationPrecision.OneFiveFiveBit, bh.QuantizationPrecision.EightBit])
@pytest.mark.parametrize("shape", [(5,), (32, 128), (3, 5, 7), (300, 4096 + 17), (1, 1)])
def test_dynamic_activation_quantizer_matches_the_oracle(precision, shape):
    """DynamicActivationQuantizer (activations.rs:203-454) on the device: abs-max and the quantiser with a given scale
    bit-equal to the oracle (signed and the reference's literal u8 form), and the stateful object step by step against
    the oracle driven by the same state machine: the moving average after every quantize_dynamic, the values it yields,
    reset, calibration, attention, and the reference's own assertions (ternary values only for the default precision,
    the scale grows with the magnitude, a reset quantizer scales by the tensor's own abs-max)."""
    rng = np.random.default_rng(len(shape) * 7 + precision)
    x = (rng.standard_normal(shape) * 3).astype(f32)
    assert f32(bh.abs_max(dev(x))) == orc.abs_max(x)
    for scale in (float(orc.abs_max(x)) / 127.0, 0.037, 1.0, 2.5):
        for u8 in (False, True):
            got = bh.quantize_activations_scaled(dev(x), precision, scale, reference_u8=u8)
            want = orc.quantize_activations_scaled(x, precision, scale, reference_u8=u8)
            assert np.array_equal(host(got).view(np.int8), want)
    cfg = bh.ActivationQuantizationConfig(precision=precision, ema_decay=0.8, calibration_warmup=2, moving_average_window=4)
    quant = bh.create_activation_quantizer(cfg)
    model = bh.DynamicScaleState(cfg)
    first = quant.quantize(dev(x))  # no state yet: the tensor's own abs-max is the scale
    assert f32(first.stats["scale_factor"]) == orc.abs_max(x)
    assert np.array_equal(host(first.values), orc.quantize_activations_scaled(x, precision, float(orc.abs_max(x))))
    scales = []
    for step, mag in enumerate((0.1, 1.0, 10.0, 3.0, 0.5)):
        xs = (x * f32(mag)).astype(f32)
        out = quant.quantize_dynamic(dev(xs))
        model.step_count += 1
        ema = model.update(orc.abs_max(xs))
        assert f32(out.stats["scale_factor"]) == ema == quant.state.ema_scale
        assert np.array_equal(host(out.values), orc.quantize_activations_scaled(xs, precision, float(ema)))
        assert out.original_shape == shape and out.stats["elements_count"] == x.size
        assert quant.needs_calibration() == model.needs_calibration()
        assert f32(float(quant.get_dynamic_scales())) == ema
        scales.append(float(ema))
        if precision == bh.QuantizationPrecision.OneFiveFiveBit:
            assert set(np.unique(host(out.values)).tolist()) <= {-1, 0, 1}
    assert scales[0] < scales[1] < scales[2]  # the scale adapts to the magnitude (test_..._dynamic_scaling)
    deq = quant.dequantize(out)
    assert tuple(deq.shape) == shape
    quant.reset_dynamic_state()
    again = quant.quantize_dynamic(dev(x))
    own = orc.abs_max(x) / f32(127.0) if precision == bh.QuantizationPrecision.EightBit else orc.abs_max(x)
    assert f32(again.stats["scale_factor"]) == own and again.stats["scale_factor"] > 0
    quant.calibrate([dev((x * f32(m)).astype(f32)) for m in (1.0, 4.0, 2.0)])
    assert f32(quant.state.ema_scale) == orc.abs_max((x * f32(4.0)).astype(f32)) and quant.state.calibrated
    att = quant.quantize_attention(dev(x), 64)
    assert att.sequence_length == 64
    off = bh.DynamicActivationQuantizer(bh.ActivationQuantizationConfig(quantize_attention=False))
    with pytest.raises(bh.BitLinearError):
        off.quantize_attention(dev(x), 8)
    with pytest.raises(bh.BitLinearError):
        quant.validate_input(torch.zeros((), device="cuda"))
    with pytest.raises(bh.BitLinearError):
        quant.validate_input(torch.zeros((4, 4), dtype=torch.uint8, device="cuda"))


# ---- R1 + A1 -------------------------------------------------------------------------------------------

@pytest.mark.parametrize("m,k", [(1, 2560), (4, 2560), (3, 6912), (2, 1024), (5, 4096), (2, 8192), (2, 12000),
                                 (3, 7), (2, 257), (1, 4), (9, 64), (33, 2560), (40, 6912), (35, 1028), (34, 20000),
                                 (2, 20000), (3, 16384), (33, 5)])
@pytest.mark.parametrize("norm", [False, True])
def test_activation_quant_bit_exact(m, k, norm):
    rng = np.random.default_rng(m * 100003 + k)
    x = synth_activations(rng, m, k, outliers=True)
    g = rng.standard_normal(k, dtype=f32) if norm else None
    q, s, asum, y = bh.quantize_activations_i8(dev(x), dev(g) if norm else None, eps=1e-5, want_sum=True, want_y=norm)
    q_ref, s_ref, rs_ref = orc.rmsnorm_quantize_i8(x, g, 1e-5, orc.SUM_BLOCK256)
    assert np.array_equal(host(s), s_ref)
    assert np.array_equal(host(q), q_ref)
    assert np.array_equal(host(asum), rs_ref)
    if norm:
        assert np.array_equal(host(y), orc.rmsnorm(x, g, 1e-5, orc.SUM_BLOCK256))


@pytest.mark.parametrize("m,k", [(3, 2560), (3, 300), (40, 2560), (40, 6912), (5, 12000), (2, 20000), (40, 301), (64, 8192),
                                 (300, 2560), (16, 6912)])
def test_activation_quant_sequential_order_bit_exact(m, k):
    """The reference's literal summation order (one running f32 sum) is available and also bit-exact: the kernels with
    16 and 4 wavefronts per row (the row's squares staged in LDS, every lane running the chain), unaligned rows, rows
    too long for the staging (the chain then reads global memory) and the wavefront-per-row kernel."""
    rng = np.random.default_rng(k + m)
    x = synth_activations(rng, m, k)
    g = rng.standard_normal(k, dtype=f32)
    q, s, _, y = bh.quantize_activations_i8(dev(x), dev(g), eps=1e-6, sum_order=bh.SUM_SEQUENTIAL, want_y=True)
    q_ref, s_ref, _ = orc.rmsnorm_quantize_i8(x, g, 1e-6, orc.SUM_SEQUENTIAL)
    assert np.array_equal(host(y), orc.rmsnorm(x, g, 1e-6, orc.SUM_SEQUENTIAL))
    assert np.array_equal(host(s), s_ref) and np.array_equal(host(q), q_ref)


@pytest.mark.parametrize("m,k", [(600, 1028), (600, 1536), (600, 2048), (600, 2052), (520, 3072), (520, 3076), (520, 4100), (520, 5124), (513, 6148), (513, 7168), (513, 7172), (513, 8192), (513, 9220), (513, 12292), (514, 14336), (514, 14340),
                                 (40, 4), (40, 256), (40, 260), (35, 508), (35, 512), (35, 516), (33, 1020), (33, 1024), (33, 301)])
def test_activation_quant_with_a_norm_bit_exact(m, k):
    """Row lengths around each count of chunks a thread, with rows whose dividends are zeros, tiny, huge or not finite (the plain division)."""
    rng = np.random.default_rng(k + m)
    x = synth_activations(rng, m, k, outliers=True)
    x[1, ::3] = 0.0
    x[2] = -0.0
    x[3] *= f32(1e-36)
    x[4, k // 2] = f32(1e30)
    x[5, k - 1] = np.inf
    x[6] *= f32(1e12)
    g = rng.standard_normal(k, dtype=f32)
    q, s, asum, y = bh.quantize_activations_i8(dev(x), dev(g), want_sum=True, want_y=True)
    q_ref, s_ref, sum_ref = orc.rmsnorm_quantize_i8(x, g, 1e-5)
    finite = [r for r in range(m) if r != 5]
    assert np.array_equal(host(y)[finite].view(np.uint32), orc.rmsnorm(x, g, 1e-5)[finite].view(np.uint32))
    assert np.array_equal(host(y)[5], orc.rmsnorm(x, g, 1e-5)[5], equal_nan=True)
    assert np.array_equal(host(s), s_ref) and np.array_equal(host(q), q_ref) and np.array_equal(host(asum), sum_ref)


@pytest.mark.parametrize("m,k", [(3100, 2564), (1500, 5124), (1300, 6148), (1400, 6916), (2000, 7940), (1150, 8708), (1080, 9980), (1000, 10500), (700, 12284), (1350, 14332),
                                 (1000, 1020), (1100, 1020), (17000, 644), (1030, 512)])
def test_activation_quant_with_a_norm_held_bit_exact(m, k):
    """As many rows as it takes for a workgroup, or a wavefront, to hold the norm's weights, at each count of chunks a thread (the sizes above have fewer)."""
    test_activation_quant_with_a_norm_bit_exact(m, k)


@pytest.mark.parametrize("m,k", [(33, 1), (33, 2), (33, 3), (40, 5), (40, 6), (40, 7), (35, 509), (35, 1021), (35, 1022), (35, 1023), (600, 1029), (600, 1030), (600, 1031),
                                 (5, 2561), (520, 5121), (513, 7169), (514, 9898), (20, 16385), (513, 16387)])
@pytest.mark.parametrize("how", ["plain", "norm", "gated", "shifted"])
def test_activation_quant_of_rows_at_any_alignment_bit_exact(m, k, how):
    """Rows that are no multiple of four columns, each remainder, and rows that start four bytes past an aligned address: the row's last
    chunk is read as the last four of its elements."""
    rng = np.random.default_rng(k + m)
    x, g, kw = synth_activations(rng, m, k, outliers=True), None, {}
    ref = x
    if how == "norm":
        g = rng.standard_normal(k, dtype=f32)
    elif how == "gated":
        up = synth_activations(rng, m, k)
        kw, ref = {"x2": dev(up), "input_mode": bh.INPUT_RELU2_MUL}, orc.relu2_mul(x, up)
    xd = dev(x)
    if how == "shifted":
        xd = torch.cat([torch.zeros(1, device="cuda"), xd.flatten()])[1:].view(m, k)
    q, s, asum, _ = bh.quantize_activations_i8(xd, None if g is None else dev(g), want_sum=True, **kw)
    q_ref, s_ref, sum_ref = orc.quantize_activations_i8(ref) if g is None else orc.rmsnorm_quantize_i8(x, g, 1e-5)
    assert np.array_equal(host(s), s_ref) and np.array_equal(host(q), q_ref) and np.array_equal(host(asum), sum_ref)


def test_activation_quant_edge_rows():
    x = np.zeros((4, 256), dtype=f32)
    x[1, :9] = [127.0, 0.5, -0.5, 1.5, 2.5, -2.5, 0.49999997, -126.5, 126.4999]
    x[2, 3] = np.nan
    x[2, 4] = 2.0
    x[3, :] = 1e-30
    q, s, asum, _ = bh.quantize_activations_i8(dev(x), want_sum=True)
    q_ref, s_ref, rs_ref = orc.quantize_activations_i8(x)
    assert np.array_equal(host(q), q_ref) and np.array_equal(host(s), s_ref) and np.array_equal(host(asum), rs_ref)
    assert host(s)[0] == 1.0 and not host(q)[0].any()
    assert host(q)[1, :9].tolist() == [127, 1, -1, 2, 3, -3, 0, -127, 126]
    # the reference's own property test (ternary_operations.rs:445-461)
    xin = np.array([G["activation_quant_properties"]["input"]], dtype=f32)
    q, s, _, _ = bh.quantize_activations_i8(dev(xin))
    fq = host(q)[0].astype(f32) / host(s)[0]
    assert fq[1] > fq[0] and fq[2] < 0 and fq[3] < fq[2]
    c = G["absmax_8bit_scale"]
    _, s, _, _ = bh.quantize_activations_i8(dev(np.array([c["input"]], dtype=f32)))
    assert host(s)[0] == f32(127.0) / f32(c["absmax"])


def test_activation_quant_fused_inputs():
    rng = np.random.default_rng(21)
    m, ffn = 3, 6912
    gate, up = synth_activations(rng, m, ffn), synth_activations(rng, m, ffn)
    q, s, _, _ = bh.quantize_activations_i8(dev(gate), x2=dev(up), input_mode=bh.INPUT_RELU2_MUL)
    q_ref, s_ref, _ = orc.quantize_activations_i8(orc.relu2_mul(gate, up))
    assert np.array_equal(host(q), q_ref) and np.array_equal(host(s), s_ref)
    v = synth_activations(rng, m, 640)
    q, s, _, _ = bh.quantize_activations_i8(dev(v), input_mode=bh.INPUT_GQA_BROADCAST, gqa_group=4, head_dim=128)
    q_ref, s_ref, _ = orc.quantize_activations_i8(orc.gqa_broadcast_v(v, 20, 5, 128))
    assert np.array_equal(host(q), q_ref) and np.array_equal(host(s), s_ref)


def test_activation_quant_prefill_size_properties():
    """Full prefill size (2048 x 2560): size-independent properties plus a sampled comparison."""
    rng = np.random.default_rng(22)
    x = synth_activations(rng, 2048, 2560, outliers=True)
    g = np.ones(2560, dtype=f32)
    xd = dev(x)
    q, s, asum, _ = bh.quantize_activations_i8(xd, dev(g), want_sum=True)
    qh = host(q)
    assert np.all(np.abs(qh.astype(np.int32)).max(axis=1) == 127)
    assert np.array_equal(host(asum), qh.astype(np.int64).sum(axis=1))
    qn, sn, _, _ = bh.quantize_activations_i8(-xd, dev(g))
    assert np.array_equal(host(qn), -qh) and np.array_equal(host(sn), host(s))
    rows = rng.choice(2048, size=64, replace=False)
    q_ref, s_ref, _ = orc.rmsnorm_quantize_i8(x[rows], g, 1e-5)
    assert np.array_equal(qh[rows], q_ref) and np.array_equal(host(s)[rows], s_ref)


# ---- G1: reference contract on the reference's byte layout ---------------------------------------------------

@pytest.mark.parametrize("case", G["gemv"], ids=lambda c: f'{c["m"]}x{c["k"]}')
def test_w2a8_gemv_reference_vectors(case):
    w = np.array(case["a"], dtype=np.int8).reshape(case["m"], case["k"])
    out = torch.zeros(case["m"], dtype=torch.int32, device="cuda")
    bh.W2A8Backend().w2a8_gemv(dev(orc.pack_2bit(w)), dev(np.array(case["x"], dtype=np.int8)), out, case["m"], case["k"])
    assert (host(out) * case["scale"]).tolist() == case["expected"]


@pytest.mark.parametrize("n,k", [(1, 1), (3, 5), (7, 33), (64, 256), (100, 1000), (640, 2560), (2560, 6912)])
def test_w2a8_gemv_rowmajor_bit_exact(n, k):
    rng = np.random.default_rng(n * 31 + k)
    w = rng.integers(-1, 2, size=(n, k)).astype(np.int8)
    a = rng.integers(-128, 128, size=k).astype(np.int8)
    packed = orc.pack_2bit(w)
    out = torch.zeros(n, dtype=torch.int32, device="cuda")
    bh.W2A8Backend().w2a8_gemv(dev(packed), dev(a), out, n, k)
    assert np.array_equal(host(out), orc.gemv_w2a8(packed, a, n))


def test_w2a8_gemv_shape_errors():
    b = bh.W2A8Backend()
    w, a, o = dev(np.zeros(32, np.uint8)), dev(np.zeros(16, np.int8)), torch.zeros(8, dtype=torch.int32, device="cuda")
    with pytest.raises(bh.BitLinearError) as ei:
        b.w2a8_gemv(w[:31].contiguous(), a, o, 8, 16)
    assert ei.value.kind == "ShapeMismatch" and ei.value.expected == [32] and ei.value.actual == [31]
    with pytest.raises(bh.BitLinearError):
        b.w2a8_gemv(w, a[:15].contiguous(), o, 8, 16)
    with pytest.raises(bh.BitLinearError):
        b.w2a8_gemv(w, a, o[:7].contiguous(), 8, 16)


# ---- G1 / G2 / E1 on the tiled layout ---------------------------------------------------------------------

SHAPES = [(2560, 2560), (640, 2560), (6912, 2560), (2560, 6912)]


def make_problem(rng, m, n, k, outliers=False, full_range=False):
    w = synth_weights(rng, n, k)
    qw, ws = orc.quantize_weights_absmean(w)
    packed = orc.pack_2bit(qw)
    if full_range:
        a = rng.integers(-128, 128, size=(m, k)).astype(np.int8)
        a_scale = (rng.random(m, dtype=f32) * 50 + 1).astype(f32)
    else:
        a, a_scale, _ = orc.quantize_activations_i8(synth_activations(rng, m, k, outliers))
    return packed, ws, a, a_scale


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("m", [1, 2, 3, 4, 8])
def test_decode_gemv_bit_exact(m, n, k):
    rng = np.random.default_rng(m * 1000 + n + k)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, outliers=True)
    tiled = bh.retile_weights(dev(packed), n, k)
    acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale))
    acc_ref = orc.gemm_w2a8(packed, a, n)
    assert np.array_equal(host(acc), acc_ref)
    out_ref = orc.epilogue(acc_ref, ws, a_scale)
    assert np.array_equal(host(out), out_ref)
    assert rel_err(host(out), out_ref) <= REL_TOL


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 5, 7), (2, 17, 257), (3, 33, 100), (1, 16, 255), (4, 15, 512),
                                   (1, 48, 16384), (8, 31, 3000), (17, 40, 512), (33, 100, 300), (48, 33, 768),
                                   (65, 50, 512), (95, 170, 1024), (20, 7000, 256)])
def test_decode_gemv_ragged_shapes(m, n, k):
    """Token counts 1, 2..16, 17..32, 33..64 and 65..95 take different variants of the decode GEMV (dot-product
    chain, MFMA with 1, 2 or 4 groups of 16 token rows, two launches); k a multiple of 256 or not selects the
    unconditional-load variant or the bounds-checked one."""
    rng = np.random.default_rng(m + 10 * n + 100 * k)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, full_range=True)
    tiled = bh.retile_weights(dev(packed), n, k)
    bias = rng.standard_normal(n, dtype=f32)
    res = rng.standard_normal((m, n), dtype=f32)
    acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale), dev(bias), dev(res))
    acc_ref = orc.gemm_w2a8(packed, a, n)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), orc.epilogue(acc_ref, ws, a_scale, bias, res))


@pytest.mark.parametrize("m,n,k", [(5, 40, 256), (16, 33, 3072), (8, 100, 3328), (8, 17, 8192), (5, 6500, 512),
                                   (16, 13000, 256), (7, 2560, 6912), (16, 6912, 2560), (9, 48, 3328), (4, 48, 2560)])
def test_decode_gemv_lds_staged_activations(m, n, k):
    """5..16 tokens with k a multiple of 256 whose rows fit LDS take the MFMA GEMV that copies the activations into
    LDS first: k <= 3072 (one chunk column per thread) or k <= 8192 with at most 8 tokens (two); n selects 1, 2 or 4
    row blocks per workgroup (400 / 800 row blocks), ragged n the partial last block.  The last two cases fall just
    outside (9 tokens at k > 3072, 4 tokens) and take the gathering variant."""
    rng = np.random.default_rng(m + 10 * n + 100 * k)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, full_range=True)
    tiled = bh.retile_weights(dev(packed), n, k)
    bias = rng.standard_normal(n, dtype=f32)
    res = rng.standard_normal((m, n), dtype=f32)
    acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale), dev(bias), dev(res))
    acc_ref = orc.gemm_w2a8(packed, a, n)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), orc.epilogue(acc_ref, ws, a_scale, bias, res))
    acc2, out2 = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale))
    assert np.array_equal(host(acc2), acc_ref)
    assert np.array_equal(host(out2), orc.epilogue(acc_ref, ws, a_scale))


def test_decode_gemv_extremes_and_identities():
    k, n = 6912, 32
    tiled_neg = bh.retile_weights(dev(orc.pack_2bit(-np.ones((n, k), np.int8))), n, k)
    acc, _ = bh.matmul_w2a8(tiled_neg, dev(np.full((1, k), -128, np.int8)), n, want_out=False)
    assert np.all(host(acc) == 128 * k)
    tiled_pos = bh.retile_weights(dev(orc.pack_2bit(np.ones((n, k), np.int8))), n, k)
    rng = np.random.default_rng(5)
    a = rng.integers(-128, 128, size=(2, k)).astype(np.int8)
    acc, _ = bh.matmul_w2a8(tiled_pos, dev(a), n, want_out=False)
    assert np.array_equal(host(acc), np.repeat(a.astype(np.int64).sum(1)[:, None], n, axis=1))
    # linearity in the activations: acc(a1 + a2) = acc(a1) + acc(a2) while a1 + a2 stays in int8
    w = rng.integers(-1, 2, size=(n, k)).astype(np.int8)
    tiled = bh.retile_weights(dev(orc.pack_2bit(w)), n, k)
    a1 = rng.integers(-60, 60, size=(1, k)).astype(np.int8)
    a2 = rng.integers(-60, 60, size=(1, k)).astype(np.int8)
    r1, _ = bh.matmul_w2a8(tiled, dev(a1), n, want_out=False)
    r2, _ = bh.matmul_w2a8(tiled, dev(a2), n, want_out=False)
    r12, _ = bh.matmul_w2a8(tiled, dev((a1 + a2).astype(np.int8)), n, want_out=False)
    assert np.array_equal(host(r12), host(r1) + host(r2))


@pytest.mark.parametrize("m", [16, 24, 64])
@pytest.mark.parametrize("n,k", [(6912, 2560), (2560, 6912)])
def test_batched_decode_sweep_bit_exact(m, n, k):
    rng = np.random.default_rng(m + n)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, outliers=True)
    tiled = bh.retile_weights(dev(packed), n, k)
    acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale))
    acc_ref = orc.gemm_w2a8(packed, a, n)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), orc.epilogue(acc_ref, ws, a_scale))


@pytest.mark.parametrize("m", [17, 31, 32, 33, 48, 80, 95])
@pytest.mark.parametrize("n,k", [(33, 256), (650, 2560), (6912, 2560), (2560, 6912), (100, 8192), (4000, 3072), (1000, 3328),
                                 (640, 2564)])
def test_token_group_gemv_bit_exact(m, n, k):
    """17 to 95 tokens: token groups of 16 with their rows in LDS (k a multiple of 256 up to 8192; one, two or four row
    blocks per workgroup; a last token group that is not full; output rows that do not fill a row block), with bias and
    residual; k = 2564 takes the gathering kernel instead."""
    rng = np.random.default_rng(m * 131 + n + k)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, outliers=True)
    tiled = bh.retile_weights(dev(packed), n, k)
    bias = rng.standard_normal(n, dtype=f32)
    res = rng.standard_normal((m, n), dtype=f32)
    acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale), bias=dev(bias), residual=dev(res))
    acc_ref = orc.gemm_w2a8(packed, a, n)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), orc.epilogue(acc_ref, ws, a_scale, bias, res))
    acc2, _ = bh.matmul_w2a8(tiled, dev(a), n, want_out=False)
    assert np.array_equal(host(acc2), acc_ref)


@pytest.mark.parametrize("m,n,k", [(96, 2560, 6912), (130, 2560, 6912), (256, 2560, 6912), (128, 6912, 2560), (200, 650, 2560),
                                   (256, 4800, 3072), (257, 2560, 6912), (192, 6912, 2560), (500, 2560, 6912), (700, 2577, 6912),
                                   (384, 6912, 2560), (1000, 2560, 2560), (160, 2560, 2560)])
def test_small_prefill_launches_bit_exact(m, n, k):
    """96 to 257 tokens, where the launch is too small for the 128 x 160 GEMM tiles to fill the chip: the token-group GEMV
    while its workgroups fit one round (96 tokens at 6912 -> 2560, 200 tokens at 650 rows), else the GEMM with narrow
    tiles and four stages of loads in flight (64 x 32 or 64 x 64).  Same results whichever runs."""
    rng = np.random.default_rng(m + n + k)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, outliers=True)
    tiled = bh.retile_weights(dev(packed), n, k)
    res = rng.standard_normal((m, n), dtype=f32)
    a_sum = dev(a.astype(np.int32).sum(axis=1).astype(np.int32))
    acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale), residual=dev(res), a_sum=a_sum)
    acc_ref = orc.gemm_w2a8(packed, a, n)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), orc.epilogue(acc_ref, ws, a_scale, None, res))


@pytest.mark.parametrize("n,k", [(6912, 2560), (2560, 6912)])
@pytest.mark.parametrize("with_sum", [True, False], ids=["lds_direct_kernel", "register_staged_kernel"])
def test_prefill_gemm_full_size(n, k, with_sum):
    """M = 2048 at the two prefill shapes: every one of the 2048 x N accumulators against an f64 BLAS
    product of the unpacked operands (|acc| <= 127 K < 2^24, so every partial sum of the f64 product is an exact
    integer whatever the library's order), sampled rows also against the oracle's own loop, the f32 output of the whole
    matrix against the oracle's epilogue.  Supplying the activation row sums selects the LDS-direct kernel, omitting
    them the register-staged one."""
    m = 2048
    rng = np.random.default_rng(n)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, outliers=False)
    tiled = bh.retile_weights(dev(packed), n, k)
    a_sum = dev(a.astype(np.int32).sum(axis=1).astype(np.int32)) if with_sum else None
    acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale), a_sum=a_sum)
    acc_h, out_h = host(acc), host(out)
    rows = np.sort(rng.choice(m, size=48, replace=False))
    acc_ref = orc.gemm_w2a8(packed, a[rows], n)
    assert np.array_equal(acc_h[rows], acc_ref)
    assert np.array_equal(out_h[rows], orc.epilogue(acc_ref, ws, a_scale[rows]))
    w = orc.unpack_2bit(packed, n * k).reshape(n, k)
    full = a.astype(np.float64) @ w.astype(np.float64).T  # exact: integers below 2^53 throughout
    assert np.array_equal(full[rows], acc_ref.astype(np.float64))  # the f64 product agrees with the oracle's loop
    assert np.array_equal(acc_h.astype(np.float64), full), "an accumulator of the full matrix differs"
    assert np.array_equal(out_h, orc.epilogue(acc_h, ws, a_scale))


@pytest.mark.parametrize("m,n,k", [(96, 160, 512), (100, 33, 512), (257, 170, 768), (130, 6912, 2560), (300, 16, 256),
                                   (128, 48, 300), (200, 200, 2561), (1500, 2602, 768), (1600, 2560, 512),
                                   (4100, 5002, 512)])
def test_gemm_ragged_shapes_both_kernels(m, n, k):
    """Token counts, widths and depths that do not fill the MFMA tiles, with bias and residual; with row sums
    (LDS-direct kernels where k allows it: the sizes cover the 64 x 160 tiles, the eight-wavefront 128 x 160
    workgroups (192..256 tiles) and the four-wavefront 128 x 160 workgroups (640 tiles and more)) and
    without."""
    rng = np.random.default_rng(m + 10 * n + 100 * k)
    packed, ws, a, a_scale = make_problem(rng, m, n, k, full_range=True)
    tiled = bh.retile_weights(dev(packed), n, k)
    bias = rng.standard_normal(n, dtype=f32)
    res = rng.standard_normal((m, n), dtype=f32)
    acc_ref = orc.gemm_w2a8(packed, a, n)
    out_ref = orc.epilogue(acc_ref, ws, a_scale, bias, res)
    for a_sum in (dev(a.astype(np.int32).sum(axis=1).astype(np.int32)), None):
        acc, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale), dev(bias), dev(res),
                                  a_sum=a_sum)
        assert np.array_equal(host(acc), acc_ref)
        assert np.array_equal(host(out), out_ref)


@pytest.mark.parametrize("m,n,k", [(100, 172, 512), (257, 2560, 768), (1600, 2564, 512), (1990, 6900, 768),
                                   (2048, 6912, 512), (1990, 6902, 512), (4100, 5000, 512)])
@pytest.mark.parametrize("extras", [False, True], ids=["plain", "bias_residual"])
def test_gemm_f32_only_epilogue_ragged(m, n, k, extras):
    """f32 output without the int32 accumulators: the straight-line epilogue of the LDS-direct kernels (64 x 160,
    eight-wavefront 128 x 160 and four-wavefront 128 x 160 workgroups), tiles cut by m and n, n not a multiple of 4 (general epilogue), and one activation scale outside the short division's
    range (whole wavefronts fall back to the plain division)."""
    rng = np.random.default_rng(7 * m + 3 * n + k + int(extras))
    packed, ws, a, a_scale = make_problem(rng, m, n, k, full_range=True)
    a_scale = a_scale.copy()
    a_scale[m // 2] = np.float32(2.0) ** 100  # invariant_divisor_ok fails for this row
    tiled = bh.retile_weights(dev(packed), n, k)
    bias = rng.standard_normal(n, dtype=f32) if extras else None
    res = rng.standard_normal((m, n), dtype=f32) if extras else None
    out_ref = orc.epilogue(orc.gemm_w2a8(packed, a, n), ws, a_scale, bias, res)
    a_sum = dev(a.astype(np.int32).sum(axis=1).astype(np.int32))
    _, out = bh.matmul_w2a8(tiled, dev(a), n, dev(np.array([ws], dtype=f32)), dev(a_scale),
                            dev(bias) if extras else None, dev(res) if extras else None, want_acc=False, a_sum=a_sum)
    assert np.array_equal(host(out), out_ref)


@pytest.mark.parametrize("m", [1, 4, 16, 128])
def test_forward_in_hip_graph_replays_match_eager(m):
    """forward() with caller-supplied output and workspace allocates nothing and records no memset, so a caller may
    capture it into a HIP graph: three replays, with eager work and synchronisations between them, each bit-equal
    to the eager result and to the oracle."""
    rng = np.random.default_rng(900 + m)
    n, k = 2560, 6912
    w = synth_weights(rng, n, k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "graph")
    layer.update_weights(dev(w))
    qw, ws_ = orc.quantize_weights_absmean(w)
    x = synth_activations(rng, m, k, outliers=True)
    ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws_)[0]
    xd = dev(x)
    y = torch.empty((m, n), device="cuda", dtype=torch.float32)
    scratch = torch.empty((max(layer.workspace_size(m), 16),), device="cuda", dtype=torch.uint8)
    layer.forward(xd, out=y, workspace=scratch)
    torch.cuda.synchronize()
    assert np.array_equal(host(y), ref)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer.forward(xd, out=y, workspace=scratch)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer.forward(xd, out=y, workspace=scratch)
        layer.forward(xd, out=y, workspace=scratch)
    for _ in range(3):
        y.zero_()
        other = layer.forward(xd)  # eager work between replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(y), ref)
        assert np.array_equal(host(other), ref)


@pytest.mark.parametrize("m,n,k,norm", [(16, 2560, 2048, False), (17, 33, 1284, False), (256, 100, 1540, False), (512, 40, 2048, False), (9, 33, 1280, False),
                                        (16, 300, 1024, True), (96, 33, 260, True), (9, 300, 1024, True)])
def test_recorded_calls_on_short_rows_replay_the_eager_result(m, n, k, norm):
    """Short rows on both sides of the line beyond which a captured call takes two launches: with a workspace, with scratch of the
    graph's own pool (the native call path), in the static scratch and for several layers, three replays each."""
    rng = np.random.default_rng(m + n + k)
    pk = random_packed_ternary(rng, n, k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "recorded")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    x, g = synth_activations(rng, m, k, outliers=True), rng.standard_normal(k, dtype=f32) if norm else None
    ref = orc.bitlinear_forward(x, pk, n, f32(0.02), g=g)[0]
    xd, gd = dev(x), dev(g) if norm else None
    ws = torch.empty((layer.workspace_size(m),), dtype=torch.uint8, device="cuda")
    outs = [torch.empty((m, n), device="cuda") for _ in range(2)]
    layer.forward_noalloc(xd, outs[1], gamma=gd)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer.forward(xd, gamma=gd, out=outs[0], workspace=ws)
        made = [layer.forward(xd, gamma=gd)] + bh.forward_multi([layer, layer], xd, gamma=gd)
        layer.forward_noalloc(xd, outs[1], gamma=gd)
    for _ in range(3):
        for y in outs + made:
            y.zero_()
        other = layer.forward(xd, gamma=gd)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(np.array_equal(host(y), ref) for y in outs + made + [other])


@pytest.mark.parametrize("n", [1, 4, 5, 6, 1000, 10001, 2560 * 640])
def test_base3_pack_unpack_bit_exact(n):
    """Base3PackedPacker on the GPU against the oracle, ragged tails included; decoding every byte value."""
    rng = np.random.default_rng(n)
    q = rng.integers(-1, 2, size=n).astype(np.int8)
    packed = bh.pack_ternary_base3(dev(q))
    assert np.array_equal(host(packed), orc.pack_base3(q))
    assert np.array_equal(host(bh.unpack_ternary_base3(packed, n)), q)
    raw = rng.integers(0, 256, size=(n + 4) // 5).astype(np.uint8)  # any byte, also above 242
    assert np.array_equal(host(bh.unpack_ternary_base3(dev(raw), n)), orc.unpack_base3(raw, n))


@pytest.mark.parametrize("n,k", [(1, 4), (48, 300), (33, 7), (640, 2560)])
@pytest.mark.parametrize("on_device", [False, True])
def test_bitlinear_base3_weights_match_2bit_weights(n, k, on_device):
    """A layer loaded from base-3 bytes holds the same canonical 2-bit bytes and computes the same forward as a
    layer loaded from the 2-bit bytes of the same ternary matrix; short buffers are a shape mismatch."""
    rng = np.random.default_rng(31 * n + k)
    q = rng.integers(-1, 2, size=(n, k)).astype(np.int8)
    ws = np.float32(0.0173)
    b3 = torch.from_numpy(orc.pack_base3(q.ravel()))
    a = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "b3")
    a.set_base3_weights(b3.cuda() if on_device else b3, float(ws))
    b = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "b2")
    b.set_quantized_weights(dev(orc.pack_2bit(q.ravel())), float(ws))
    pa, sa = a.get_quantized_weights()
    pb, sb = b.get_quantized_weights()
    assert sa == sb == float(ws)
    assert np.array_equal(pa.numpy(), pb.numpy())
    assert np.array_equal(pa.numpy(), orc.pack_2bit(q.ravel()))
    x = synth_activations(rng, 3, k)
    ya, yb = host(a.forward(dev(x))), host(b.forward(dev(x)))
    assert np.array_equal(ya, yb)
    assert np.array_equal(ya, orc.bitlinear_forward(x, orc.pack_2bit(q.ravel()), n, ws)[0])
    if b3.numel() > 1:
        with pytest.raises(bh.BitLinearError) as err:
            a.set_base3_weights(b3[:-1].contiguous(), float(ws))
        assert err.value.status == bh.SHAPE_MISMATCH


@pytest.mark.parametrize("n,k", [(16, 320), (1, 5), (33, 7), (48, 300), (640, 2560), (2560, 6912), (100, 2561), (4096, 4096)])
def test_gemv_on_base3_bytes_bit_exact(n, k):
    """bitnet_hip_gemv_base3: the decode GEMV that consumes the base-3 bytes of Base3PackedPacker (packing.rs:421-501)
    themselves.  The streaming layout is built from the oracle's flat base-3 bytes; int32 accumulators equal the oracle's
    contraction of the same ternary matrix (and hence the 2-bit GEMV), the f32 output its epilogue; the reference's
    encoding fixture (140 = [1, 0, -1, 1, 0]) goes through the same path."""
    rng = np.random.default_rng(7 * n + k)
    q = rng.integers(-1, 2, size=(n, k)).astype(np.int8)
    a = rng.integers(-127, 128, size=(1, k)).astype(np.int8)
    b3 = orc.pack_base3(q.ravel())
    tiled = bh.retile_base3(dev(b3), n, k)
    assert tiled.numel() == bh.base3_tiled_size(n, k) == ((n + 15) // 16) * ((k + 319) // 320) * 1024
    ws, a_scale = f32(0.0171), np.array([f32(3.37)], dtype=f32)
    acc, out = bh.gemv_base3(tiled, dev(a.ravel()), n, w_scale=dev(np.array([ws], dtype=f32)), a_scale=dev(a_scale))
    acc_ref = orc.gemm_w2a8(orc.pack_2bit(q.ravel()), a, n)
    assert np.array_equal(host(acc), acc_ref[0])
    assert np.array_equal(host(out), orc.epilogue(acc_ref, ws, a_scale)[0])
    # the streaming layout, byte by byte: slot 16 kq + r of tile (row block, k-tile), byte t = columns 320 kt + 80 kq + 5 t ..
    th = host(tiled).reshape(-1, 64, 16)
    kt_count = (k + 319) // 320
    for _ in range(64):
        row, col = int(rng.integers(n)), int(rng.integers(k))
        kt, rem = divmod(col, 320)
        kq, rem = divmod(rem, 80)
        t, d = divmod(rem, 5)
        byte = int(th[(row // 16) * kt_count + kt, 16 * kq + row % 16, t])
        assert (byte // 3 ** d) % 3 - 1 == q[row, col]


def test_gemv_on_base3_bytes_reference_fixture_and_errors():
    """The reference's own base-3 vector (packing_correctness_tests.rs:159-176: [1, 0, -1, 1, 0] -> 140) as a 1 x 5 matrix,
    and the argument checks of the entry point."""
    b3 = np.array([140], dtype=np.uint8)
    assert np.array_equal(orc.unpack_base3(b3, 5), np.array([1, 0, -1, 1, 0], dtype=np.int8))
    tiled = bh.retile_base3(dev(b3), 1, 5)
    a = np.array([3, -7, 11, 5, 100], dtype=np.int8)
    acc, out = bh.gemv_base3(tiled, dev(a), 1)
    assert out is None and host(acc).tolist() == [3 - 11 + 5]
    with pytest.raises(bh.BitLinearError) as err:
        bh.gemv_base3(tiled[:-16].contiguous(), dev(a), 1)
    assert err.value.status == bh.SHAPE_MISMATCH
    with pytest.raises(bh.BitLinearError) as err:
        bh.retile_base3(dev(b3), 2, 5)
    assert err.value.status == bh.SHAPE_MISMATCH


@pytest.mark.parametrize("kind,cls", [(bh.LOOKUP_TERNARY, bh.HipTernaryLookupKernel), (bh.LOOKUP_I2S, bh.HipI2SLookupKernel)],
                         ids=["ternary", "i2s"])
def test_lookup_kernels_bit_exact(kind, cls):
    """TernaryLookupKernel / I2SLookupKernel::compute on the GPU: bit-identical to the oracle, out-of-table weights,
    non-finite inputs and signed zeros included; the shortest buffer decides the length; empty buffers are errors."""
    rng = np.random.default_rng(kind)
    kernel = cls()
    for n in (1, 5, 1000, 100003):
        w = rng.integers(-3, 4, size=n).astype(np.int8)
        x = rng.standard_normal(n, dtype=f32)
        x[rng.integers(0, n, size=max(1, n // 50))] = np.inf
        x[rng.integers(0, n, size=max(1, n // 50))] = np.nan
        out = torch.zeros((n,), device="cuda", dtype=torch.float32)
        kernel.compute(dev(w), dev(x), out)
        ref = orc.lookup_compute(kind, w, x)
        assert np.array_equal(host(out).view(np.uint32), ref.view(np.uint32))
    out = torch.full((6,), 7.0, device="cuda", dtype=torch.float32)
    kernel.compute(dev(np.array([1, -1, 1, 1], np.int8)), dev(np.array([2.0, 3.0, 4.0], f32)), out)
    assert host(out).tolist() == [2.0, -3.0, 4.0, 7.0, 7.0, 7.0]
    empty_w, empty_x = torch.empty((0,), dtype=torch.int8, device="cuda"), torch.empty((0,), dtype=torch.float32, device="cuda")
    for args in ((empty_w, dev(np.ones(2, f32)), out), (dev(np.ones(2, np.int8)), empty_x, out),
                 (dev(np.ones(2, np.int8)), dev(np.ones(2, f32)), empty_x)):
        with pytest.raises(bh.BitLinearError) as err:
            kernel.compute(*args)
        assert err.value.status == bh.INVALID_CONFIG
    assert kernel.name() and kernel.optimal_batch_size() > 0


def test_bitlinear_forward_prefill_uses_quantiser_row_sums():
    """BitLinear.forward at a prefill token count: quantiser -> row sums -> LDS-direct GEMM, bit-exact."""
    rng = np.random.default_rng(77)
    m, k, n = 384, 2560, 640
    w = synth_weights(rng, n, k)
    x = synth_activations(rng, m, k, outliers=True)
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "prefill")
    layer.update_weights(dev(w))
    out, q, a_scale, acc = layer.forward(dev(x), gamma=dev(g), debug=True)
    qw, ws = orc.quantize_weights_absmean(w)
    out_ref, q_ref, s_ref, acc_ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws, g=g, eps=1e-5)
    assert np.array_equal(host(q), q_ref) and np.array_equal(host(a_scale), s_ref)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), out_ref)


@pytest.mark.parametrize("m,k,n", [(97, 6912, 2560), (128, 6912, 2560), (200, 4096, 1000), (256, 6912, 2560), (130, 8192, 644),
                                   (255, 5120, 1408), (97, 4096, 16), (256, 8192, 2816), (300, 4352, 2240)])
def test_forward_of_long_rows_in_few_tiles_bit_exact(m, k, n):
    """A long k with few output tiles (97 to 256 tokens at 6912 -> 2560).  Checked against the oracle (activations,
    accumulators, f32 output with bias and residual); workspace_size is what the quantised activations take; on a
    workspace of that size full of ones, three times in a row."""
    rng = np.random.default_rng(m + k + n)
    w = synth_weights(rng, n, k)
    x = synth_activations(rng, m, k, outliers=True)
    bias = rng.standard_normal(n, dtype=f32)
    res = rng.standard_normal((m, n), dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "long rows")
    layer.update_weights(dev(w))
    layer.update_bias(dev(bias))
    qw, ws = orc.quantize_weights_absmean(w)
    out_ref, q_ref, s_ref, acc_ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws, bias=bias, residual=res)
    out, q, a_scale, acc = layer.forward(dev(x), residual=dev(res), debug=True)
    assert np.array_equal(host(q), q_ref) and np.array_equal(host(a_scale), s_ref)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), out_ref)
    full = layer.workspace_size(m)
    assert full == ((m * k + 255) // 256) * 256 + 2 * (((4 * m) + 255) // 256) * 256 + 256
    ws = torch.full((full,), 1, dtype=torch.uint8, device="cuda")
    for _ in range(3):
        assert np.array_equal(host(layer.forward(dev(x), residual=dev(res), workspace=ws)), out_ref)


# ---- L1: BitLinear object ----------------------------------------------------------------------------------

def test_bitlinear_forward_config1_bit_exact():
    """M=1, K=2560, N=2560, seed 0, W ~ N(0, 0.02), X ~ N(0, 1)."""
    rng = np.random.default_rng(0)
    w = synth_weights(rng, 2560, 2560)
    x = synth_activations(rng, 1, 2560)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=2560, out_features=2560), "config1")
    layer.update_weights(torch.from_numpy(w))  # host weights, quantised on the GPU
    out, q, a_scale, acc = layer.forward(dev(x), debug=True)
    qw, ws = orc.quantize_weights_absmean(w)
    packed_h, ws_h = layer.get_quantized_weights()
    assert ws_h == ws and np.array_equal(packed_h.numpy(), orc.pack_2bit(qw))
    out_ref, q_ref, s_ref, acc_ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), 2560, ws)
    assert np.array_equal(host(q), q_ref)
    assert np.array_equal(host(a_scale), s_ref)
    assert np.array_equal(host(acc), acc_ref)
    assert np.array_equal(host(out), out_ref)
    assert rel_err(host(out), out_ref) <= REL_TOL
    # the non-debug call gives the same bits
    assert np.array_equal(host(layer.forward(dev(x))), out_ref)


def test_bitlinear_forward_shapes_bias_norm_and_layouts():
    rng = np.random.default_rng(31)
    k, n = 256, 80
    w = synth_weights(rng, n, k)
    qw, ws = orc.quantize_weights_absmean(w)
    packed = orc.pack_2bit(qw)
    bias = rng.standard_normal(n, dtype=f32)
    g = rng.standard_normal(k, dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "t")
    with pytest.raises(bh.BitLinearError) as ei:
        layer.forward(dev(np.zeros((2, k), f32)))
    assert ei.value.kind == "NotInitialized"
    layer.update_weights(dev(w))
    # bias starts at zero, like the reference's Tensor::zeros bias (layer.rs:127-133)
    x = synth_activations(rng, 6, k)
    ref0 = orc.bitlinear_forward(x, packed, n, ws)[0]
    assert np.array_equal(host(layer.forward(dev(x))), ref0)
    layer.update_bias(dev(bias))
    ref = orc.bitlinear_forward(x, packed, n, ws, bias=bias)[0]
    assert np.array_equal(host(layer.forward(dev(x))), ref)
    # rank 3 input is flattened to [b*s, in] and reshaped back (forward.rs:182-207)
    out3 = layer.forward(dev(x.reshape(2, 3, k)))
    assert tuple(out3.shape) == (2, 3, n) and np.array_equal(host(out3).reshape(6, n), ref)
    # fused RMSNorm + residual
    res = rng.standard_normal((6, n), dtype=f32)
    refn = orc.bitlinear_forward(x, packed, n, ws, g=g, eps=1e-5, bias=bias, residual=res)[0]
    assert np.array_equal(host(layer.forward(dev(x), gamma=dev(g), residual=dev(res))), refn)
    # [in, out] orientation (the GGUF-side convention) gives the same layer
    layer_t = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "t_in_out")
    layer_t.update_weights(dev(np.ascontiguousarray(w.T)), layout=bh.LAYOUT_IN_OUT)
    p2, s2 = layer_t.get_quantized_weights()
    assert np.array_equal(p2.numpy(), packed)
    assert abs(s2 - float(ws)) <= 1e-7 * float(ws)  # the declared f64 summation order follows the given orientation
    # pre-quantised weights (forward_with_quantized_weights)
    layer_p = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "t_packed")
    layer_p.set_quantized_weights(torch.from_numpy(packed), float(ws))
    assert np.array_equal(host(layer_p.forward(dev(x))), ref0)


@pytest.mark.parametrize("m", [1, 3, 8, 20, 40, 64, 200, 300, 1100])
def test_forward_multi_matches_single_forwards(m):
    """q/k/v-style: several layers on one input give exactly what each layer gives alone, and what the oracle gives.
    (m = 200: the token-group GEMV, which takes prefill launches too small for the GEMM to fill the chip; m = 300 and
    1100: the projections share launches of the 64 x 160 and of the eight-wavefront prefill GEMM.)"""
    rng = np.random.default_rng(40 + m)
    k = 2560
    ns = [2560, 640, 640, 96]
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32)
    x = synth_activations(rng, m, k, outliers=True)
    layers, refs = [], []
    for i, n in enumerate(ns):
        w = synth_weights(rng, n, k)
        layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), f"multi{i}")
        layer.update_weights(dev(w))
        layers.append(layer)
        qw, ws = orc.quantize_weights_absmean(w)
        refs.append(orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws, g=g, eps=1e-5)[0])
    outs = bh.forward_multi(layers, dev(x), gamma=dev(g))
    for layer, out, ref in zip(layers, outs, refs):
        assert np.array_equal(host(out), ref)
        assert np.array_equal(host(layer.forward(dev(x), gamma=dev(g))), ref)
    other = bh.BitLinear(bh.BitLinearConfig(in_features=k + 4, out_features=8), "other")
    other.update_weights(torch.ones(8, k + 4))
    with pytest.raises(bh.BitLinearError) as ei:
        bh.forward_multi([layers[0], other], dev(x))
    assert ei.value.kind == "ShapeMismatch"


def test_forward_multi_prefill_gate_up_one_launch():
    """gate and up at M = 2048 share one launch of the 128 x 160 prefill GEMM (1408 tiles): sampled rows against the
    oracle, everything against the single-layer forwards."""
    rng = np.random.default_rng(4242)
    m, k, n = 2048, 2560, 6912
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32)
    x = synth_activations(rng, m, k)
    rows = np.sort(rng.choice(m, size=24, replace=False))
    layers, refs = [], []
    for i in range(2):
        w = synth_weights(rng, n, k)
        layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), f"gu{i}")
        layer.update_weights(dev(w))
        layers.append(layer)
        qw, ws = orc.quantize_weights_absmean(w)
        refs.append(orc.bitlinear_forward(x[rows], orc.pack_2bit(qw), n, ws, g=g, eps=1e-5)[0])
    outs = bh.forward_multi(layers, dev(x), gamma=dev(g))
    for layer, out, ref in zip(layers, outs, refs):
        got = host(out)
        assert np.array_equal(got[rows], ref)
        assert np.array_equal(got, host(layer.forward(dev(x), gamma=dev(g))))


def test_forward_multi_prefill_qkv_128x128_tiles():
    """q, k and v at M = 3072 (and a ragged M just below) share one launch of the 128 x 128 instance of the prefill GEMM
    (720 tiles): sampled rows against the oracle, everything against the single-layer forwards, which take other
    instances (q alone 480 tiles, k and v alone 120)."""
    rng = np.random.default_rng(3072)
    k, ns = 2560, [2560, 640, 640]
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32)
    layers, packed = [], []
    for i, n in enumerate(ns):
        w = synth_weights(rng, n, k)
        layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), f"qkv{i}")
        layer.update_weights(dev(w))
        layers.append(layer)
        qw, ws = orc.quantize_weights_absmean(w)
        packed.append((orc.pack_2bit(qw), n, ws))
    for m in (3072, 3072 - 37):
        x = synth_activations(rng, m, k, outliers=True)
        rows = np.sort(rng.choice(m, size=24, replace=False))
        rows[-1] = m - 1
        outs = bh.forward_multi(layers, dev(x), gamma=dev(g))
        for layer, out, (pk, n, ws) in zip(layers, outs, packed):
            got = host(out)
            assert np.array_equal(got[rows], orc.bitlinear_forward(x[rows], pk, n, ws, g=g, eps=1e-5)[0])
            assert np.array_equal(got, host(layer.forward(dev(x), gamma=dev(g))))


@pytest.mark.parametrize("m", [1, 2, 3, 4, 6, 7])
@pytest.mark.parametrize("n,k", [(1, 4), (17, 260), (1000, 2560), (2560, 6912), (6912 + 5, 2560), (40, 8192), (13824, 2560)])
def test_forward_fused_rows_bit_exact(m, n, k):
    """One to six tokens take the 16-wavefront kernel with the quantiser in its prologue and a set of workgroups per
    token, as long as those stay within 512 (otherwise, and from seven tokens on, the stand-alone quantiser and the MFMA
    GEMV run): row-block groups that do not fill the last 8 of the grid, one / two chunks per thread, one / four row
    blocks per workgroup, RMSNorm, bias and residual."""
    rng = np.random.default_rng(31 * m + n + k)
    w = synth_weights(rng, n, k)
    x = synth_activations(rng, m, k, outliers=True)
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32)
    bias = rng.standard_normal(n, dtype=f32)
    res = rng.standard_normal((m, n), dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "rows")
    layer.update_weights(dev(w))
    layer.update_bias(dev(bias))
    qw, ws_ = orc.quantize_weights_absmean(w)
    for norm in (False, True):
        ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws_, g=g if norm else None, eps=1e-5, bias=bias, residual=res)[0]
        got = host(layer.forward(dev(x), gamma=dev(g) if norm else None, residual=dev(res)))
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("m", [1, 2, 3, 5, 8])
def test_bitlinear_forward_decode_debug_outputs(m):
    """At decode token counts the quantiser runs inside the GEMV launch; its int8 row, scale and the int32
    accumulators are still observable and bit-exact, with and without RMSNorm, at both FFN widths."""
    rng = np.random.default_rng(50 + m)
    for k, n, norm in [(2560, 640, True), (6912, 2560, False), (1024, 48, True)]:
        w = synth_weights(rng, n, k)
        x = synth_activations(rng, m, k, outliers=True)
        g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32) if norm else None
        layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "dbg")
        layer.update_weights(dev(w))
        out, q, a_scale, acc = layer.forward(dev(x), gamma=dev(g) if norm else None, debug=True)
        qw, ws = orc.quantize_weights_absmean(w)
        out_ref, q_ref, s_ref, acc_ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws, g=g, eps=1e-5)
        assert np.array_equal(host(q), q_ref) and np.array_equal(host(a_scale), s_ref)
        assert np.array_equal(host(acc), acc_ref) and np.array_equal(host(out), out_ref)
    # the reference's literal summation order inside the fused launch
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=1024, out_features=48, sum_order=bh.SUM_SEQUENTIAL), "seq")
    layer.update_weights(dev(w))
    out_ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws, g=g, eps=1e-5, order=orc.SUM_SEQUENTIAL)[0]
    assert np.array_equal(host(layer.forward(dev(x), gamma=dev(g))), out_ref)


@pytest.mark.parametrize("k,ns", [(2560, (640,)), (6912, (2560,)), (2560, (6912, 6912))], ids=["short", "long_row", "two_row_blocks"])
def test_decode_sequential_sum_order_four_wavefront_kernel(k, ns):
    """One token with RMSNorm in the reference's literal (sequential) summation order: the launch shape that keeps four
    wavefronts per workgroup (every thread runs the whole chain), with short and long rows, one and two row blocks per
    workgroup, one and two projections per launch."""
    rng = np.random.default_rng(k + len(ns))
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32)
    x = synth_activations(rng, 1, k, outliers=True)
    layers, refs = [], []
    for i, n in enumerate(ns):
        w = synth_weights(rng, n, k)
        layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, sum_order=bh.SUM_SEQUENTIAL), f"seq{i}")
        layer.update_weights(dev(w))
        layers.append(layer)
        qw, ws = orc.quantize_weights_absmean(w)
        refs.append(orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws, g=g, eps=1e-5, order=orc.SUM_SEQUENTIAL)[0])
    outs = bh.forward_multi(layers, dev(x), gamma=dev(g)) if len(ns) > 1 else [layers[0].forward(dev(x), gamma=dev(g))]
    for out, ref in zip(outs, refs):
        assert np.array_equal(host(out), ref)


def test_forward_from_several_threads_and_streams():
    """BitLinear is Send + Sync in the reference (layer.rs:427-428): forward on one layer object from several host
    threads, each on a stream of its own, at decode and prefill token counts, while nothing is shared but the
    read-locked weights."""
    import threading

    rng = np.random.default_rng(99)
    k, n = 2560, 640
    w = synth_weights(rng, n, k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "shared")
    layer.update_weights(dev(w))
    qw, ws = orc.quantize_weights_absmean(w)
    packed = orc.pack_2bit(qw)
    cases = []
    for t, m in enumerate([1, 1, 5, 130]):
        x = synth_activations(rng, m, k, outliers=True)
        cases.append((x, orc.bitlinear_forward(x, packed, n, ws)[0]))
    errors = []

    def worker(x, ref):
        try:
            stream = torch.cuda.Stream()  # default priority
            xd = dev(x)
            torch.cuda.current_stream().synchronize()
            for _ in range(25):
                with torch.cuda.stream(stream):
                    out = layer.forward(xd, stream=stream)
                stream.synchronize()
                if not np.array_equal(host(out), ref):
                    errors.append("mismatch")
                    return
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append(repr(e))

    threads = [threading.Thread(target=worker, args=c) for c in cases]
    for th in threads:
        th.start()
    for th in threads:
        th.join(timeout=100)
    assert not errors, errors
    assert not any(th.is_alive() for th in threads)


def test_bitlinear_error_behaviour_matches_reference():
    """forward.rs:304-371: wrong last dimension -> ShapeMismatch; rank other than 2/3 -> ShapeMismatch."""
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=4, out_features=3), "test_layer_shape")
    layer.update_weights(torch.ones(3, 4))
    out = layer.forward(torch.ones(2, 4, device="cuda"))
    assert tuple(out.shape) == (2, 3)
    with pytest.raises(bh.BitLinearError) as ei:
        layer.forward(torch.ones(2, 5, device="cuda"))
    assert ei.value.kind == "ShapeMismatch" and ei.value.expected == [2, 4] and ei.value.actual == [2, 5]
    with pytest.raises(bh.BitLinearError) as ei:
        layer.forward(torch.ones(4, device="cuda"))
    assert ei.value.kind == "ShapeMismatch"
    with pytest.raises(bh.BitLinearError) as ei:
        layer.forward(torch.ones(2, 2, 2, 4, device="cuda"))
    assert ei.value.kind == "ShapeMismatch"
    with pytest.raises(bh.BitLinearError) as ei:
        layer.update_weights(torch.ones(4, 3))
    assert ei.value.kind == "ShapeMismatch" and ei.value.expected == [3, 4]
    with pytest.raises(bh.BitLinearError) as ei:
        layer.update_bias(torch.ones(3))
    assert ei.value.kind == "InvalidConfig" and "Bias is not enabled" in str(ei.value)
    with pytest.raises(bh.BitLinearError):
        layer.forward_batch(torch.ones(4, device="cuda"))
    # empty batch: nothing to do
    assert tuple(layer.forward(torch.ones(0, 4, device="cuda")).shape) == (0, 3)


# ---- L1: decoder layer and stack ----------------------------------------------------------------------------

def build_decoder(rng, layers, hidden, ffn, qh, kvh, hd, max_tokens, eps=1e-5):
    dec = bh.DecoderProjections(layers, hidden, ffn, qh, kvh, hd, eps=eps, max_tokens=max_tokens)
    ref = []
    for l in range(layers):
        packed, scales = [], []
        for p in range(7):
            n, k = dec.proj_shape(p)
            w = synth_weights(rng, n, k)
            dec.projection(l, p).update_weights(dev(w))
            qw, s = orc.quantize_weights_absmean(w)
            packed.append(orc.pack_2bit(qw))
            scales.append(s)
        ga = (1 + 0.1 * rng.standard_normal(hidden, dtype=f32)).astype(f32)
        gf = (1 + 0.1 * rng.standard_normal(hidden, dtype=f32)).astype(f32)
        dec.set_norm(l, 0, torch.from_numpy(ga))
        dec.set_norm(l, 1, torch.from_numpy(gf))
        ref.append((packed, scales, ga, gf))
    return dec, ref


def oracle_stack(ref, x, hidden, ffn, qh, kvh, hd, eps=1e-5):
    q = k = None
    for packed, scales, ga, gf in ref:
        x, q, k = orc.decoder_layer(x, packed, scales, hidden, ffn, qh, kvh, hd, ga, gf, eps)
    return x, q, k


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8])
def test_decoder_layer_config2_bit_exact(m):
    """one decoder layer's seven projections at BitNet-2B shapes."""
    rng = np.random.default_rng(0)
    dec, ref = build_decoder(rng, 1, 2560, 6912, 20, 5, 128, max_tokens=8)
    assert dec.weight_bytes() == 17_367_040
    x = synth_activations(rng, m, 2560)
    out, q, k = dec.decode(dev(x), want_qk=True)
    x_ref, q_ref, k_ref = oracle_stack(ref, x, 2560, 6912, 20, 5, 128)
    assert np.array_equal(host(q), q_ref) and np.array_equal(host(k), k_ref)
    assert np.array_equal(host(out), x_ref)
    assert rel_err(host(out), x_ref) <= REL_TOL


@pytest.mark.parametrize("layers", [2, 3])
def test_decoder_stack_small_bit_exact(layers):
    rng = np.random.default_rng(layers)
    dims = (256, 512, 4, 2, 64)
    dec, ref = build_decoder(rng, layers, *dims, max_tokens=4)
    x = synth_activations(rng, 3, 256)
    out = dec.decode(dev(x))
    assert np.array_equal(host(out), oracle_stack(ref, x, *dims)[0])
    with pytest.raises(bh.BitLinearError) as ei:
        dec.decode(dev(synth_activations(rng, 5, 256)))
    assert ei.value.kind == "ShapeMismatch"


def random_packed_ternary(rng, n, k):
    """[n, k] ternary weights as flat 2-bit bytes drawn directly (code 3 folded onto code 1: weight 0), so a
    30-block stack of 521 MB is generated in a second: P(-1) = P(+1) = 1/4, P(0) = 1/2."""
    b = rng.integers(0, 256, size=n * k // 4, dtype=np.uint8)
    return b & ~((b & (b >> 1) & 0x55) << 1)


def build_decoder_packed(rng, layers, hidden, ffn, qh, kvh, hd, max_tokens, eps=1e-5):
    dec = bh.DecoderProjections(layers, hidden, ffn, qh, kvh, hd, eps=eps, max_tokens=max_tokens)
    ref = []
    for l in range(layers):
        packed, scales = [], []
        for p in range(7):
            n, k = dec.proj_shape(p)
            pk = random_packed_ternary(rng, n, k)
            s = f32(0.016 * (1 + 0.25 * rng.random()))
            dec.projection(l, p).set_quantized_weights(torch.from_numpy(pk), float(s))
            packed.append(pk)
            scales.append(s)
        ga = (1 + 0.1 * rng.standard_normal(hidden, dtype=f32)).astype(f32)
        gf = (1 + 0.1 * rng.standard_normal(hidden, dtype=f32)).astype(f32)
        dec.set_norm(l, 0, torch.from_numpy(ga))
        dec.set_norm(l, 1, torch.from_numpy(gf))
        ref.append((packed, scales, ga, gf))
    return dec, ref


def test_decoder_stack_config5_full_depth_bit_exact():
    """BASELINE config 5 at its real depth: 30 blocks at 2560 / 6912 / 20 / 5 / 128 (521,011,200 packed bytes) on a
    decoder sized for 8 tokens, one token and eight tokens per step, every block checked against the oracle's chain;
    then runs of blocks that start and end inside the stack, in place."""
    dims = (2560, 6912, 20, 5, 128)
    rng = np.random.default_rng(5)
    dec, ref = build_decoder_packed(rng, 30, *dims, max_tokens=8)
    assert dec.weight_bytes() == 521_011_200
    for m in (1, 8):
        x = synth_activations(rng, m, dims[0])
        # the oracle's hidden state after every block
        states, cur = [x], x
        for l in range(30):
            cur, q_ref, k_ref = oracle_stack(ref[l:l + 1], cur, *dims)
            states.append(cur)
        assert np.all(np.isfinite(states[-1]))
        out, q, k = dec.decode(dev(x), want_qk=True)
        assert np.array_equal(host(out), states[30]), f"m={m}: 30-block output differs from the oracle"
        assert np.array_equal(host(q), q_ref) and np.array_equal(host(k), k_ref)
        assert rel_err(host(out), states[30]) <= REL_TOL
        for lo, hi in ((2, 7), (4, 5), (3, 30), (29, 30)):
            buf = dev(states[lo].copy())
            dec.decode(buf, out=buf, layers=(lo, hi))
            assert np.array_equal(host(buf), states[hi]), f"m={m}: blocks {lo}..{hi - 1}"


@pytest.mark.parametrize("dims,layers", [((2560, 6912, 20, 5, 128), 4), ((256, 512, 4, 2, 64), 3),
                                         ((1024, 2816, 8, 8, 128), 2)])
def test_decoder_repeated_calls_subranges_and_streams(dims, layers):
    """One token: repeated calls, sub-ranges of blocks, in-place hidden states, one block at a time (as the benchmark
    does), and calls issued from two streams in turn (the decoder's buffers are shared: the second call waits for the
    first on the GPU)."""
    rng = np.random.default_rng(layers + dims[0])
    dec, ref = build_decoder(rng, layers, *dims, max_tokens=2)
    x = synth_activations(rng, 1, dims[0])
    x_ref, q_ref, k_ref = oracle_stack(ref, x, *dims)
    for _ in range(3):
        out, q, k = dec.decode(dev(x), want_qk=True)
        assert np.array_equal(host(out), x_ref)
        assert np.array_equal(host(q), q_ref) and np.array_equal(host(k), k_ref)
    x1_ref = oracle_stack(ref[:1], x, *dims)[0]
    buf = dev(x1_ref.copy())
    dec.decode(buf, out=buf, layers=(1, layers))
    assert np.array_equal(host(buf), x_ref)
    cur = dev(x)
    for l in range(layers):
        cur = dec.decode(cur, layers=(l, l + 1))
    assert np.array_equal(host(cur), x_ref)
    # two streams in alternation, no host synchronisation in between
    xs = [dev(synth_activations(rng, 2, dims[0])) for _ in range(4)]
    refs = [oracle_stack(ref, host(t), *dims)[0] for t in xs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for i, t in enumerate(xs):
        with torch.cuda.stream(streams[i % 2]):
            outs.append(dec.decode(t, stream=streams[i % 2]))
    torch.cuda.synchronize()
    for o, r in zip(outs, refs):
        assert np.array_equal(host(o), r)


@pytest.mark.parametrize("dims,layers,m", [((2560, 6912, 20, 5, 128), 3, 1), ((2560, 6912, 20, 5, 128), 2, 8),
                                           ((256, 512, 4, 2, 64), 3, 3), ((1024, 2816, 8, 8, 128), 2, 1)])
def test_decoder_recorded_step_replays_match_the_oracle(dims, layers, m):
    """A decode step recorded as a HIP graph (bitnet_hip_decoder_graph_*): every replay, with eager work and host
    synchronisations between the replays and with new inputs written into the recorded input tensor, equals the oracle's
    chain bit for bit; so do a recorded sub-range in place, replays on another stream, replays interleaved with eager
    decode calls on the same decoder, and replays after a weight update (the graph reads the layers' buffers, which an
    update keeps)."""
    rng = np.random.default_rng(17 * layers + m + dims[0])
    dec, ref = build_decoder_packed(rng, layers, *dims, max_tokens=max(m, 2))
    x = dev(synth_activations(rng, m, dims[0]))
    graph = dec.record(x, want_qk=True)
    other = torch.cuda.Stream()
    for round_ in range(4):
        fresh = synth_activations(rng, m, dims[0])
        x_ref, q_ref, k_ref = oracle_stack(ref, fresh, *dims)
        x.copy_(dev(fresh))
        graph.out.zero_()
        if round_ == 2:  # another stream, ordered behind the copy above by an explicit wait
            other.wait_stream(torch.cuda.current_stream())
            graph.replay(stream=other)
            torch.cuda.current_stream().wait_stream(other)
        else:
            graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(graph.out), x_ref), f"replay {round_}"
        assert np.array_equal(host(graph.q), q_ref) and np.array_equal(host(graph.k), k_ref)
        # eager work on the same decoder between the replays
        assert np.array_equal(host(dec.decode(dev(fresh))), x_ref)
    # a sub-range of blocks, in place
    if layers >= 3:
        start = oracle_stack(ref[:1], host(x), *dims)[0]
        want = oracle_stack(ref[1:], start, *dims)[0]
        buf = dev(start.copy())
        sub = dec.record(buf, out=buf, layers=(1, layers))
        for _ in range(2):
            buf.copy_(dev(start))
            sub.replay()
            assert np.array_equal(host(buf), want)
    # new weights in one projection: the recorded step reads them
    n, k = dec.proj_shape(6)  # down
    pk = random_packed_ternary(rng, n, k)
    dec.projection(layers - 1, 6).set_quantized_weights(torch.from_numpy(pk), 0.02)
    packed, scales, ga, gf = ref[-1]
    ref[-1] = (packed[:6] + [pk], scales[:6] + [f32(0.02)], ga, gf)
    x_ref = oracle_stack(ref, host(x), *dims)[0]
    graph.replay()
    assert np.array_equal(host(graph.out), x_ref)


@pytest.mark.parametrize("dims,layers,m,chains", [((2560, 6912, 20, 5, 128), 2, 8, 2), ((2560, 6912, 20, 5, 128), 2, 8, 4),
                                                  ((2560, 6912, 20, 5, 128), 2, 5, 8), ((256, 512, 4, 2, 64), 3, 3, 2),
                                                  ((1024, 2816, 8, 8, 128), 3, 16, 3)])
def test_decoder_row_group_chains_match_the_oracle(dims, layers, m, chains):
    """bitnet_hip_decoder_set_chains: a step of several token rows run as groups of rows side by side, each group a chain
    of launches on a stream of the decoder's own.  Eager calls, a recorded step replayed several times (with eager work
    and host synchronisations between the replays), a sub-range in place and the last block's q / k equal the oracle's
    chain bit for bit; more chains than rows are cut down to one row each; back to one chain afterwards."""
    rng = np.random.default_rng(31 * layers + 7 * m + chains + dims[0])
    dec, ref = build_decoder_packed(rng, layers, *dims, max_tokens=m)
    dec.set_chains(chains)
    xs = synth_activations(rng, m, dims[0])
    x_ref, q_ref, k_ref = oracle_stack(ref, xs, *dims)
    for _ in range(2):
        out, q, k = dec.decode(dev(xs), want_qk=True)
        assert np.array_equal(host(out), x_ref)
        assert np.array_equal(host(q), q_ref) and np.array_equal(host(k), k_ref)
    x = dev(xs)
    graph = dec.record(x, want_qk=True)
    for round_ in range(3):
        fresh = synth_activations(rng, m, dims[0])
        want, q_want, k_want = oracle_stack(ref, fresh, *dims)
        x.copy_(dev(fresh))
        graph.out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(graph.out), want), f"replay {round_}"
        assert np.array_equal(host(graph.q), q_want) and np.array_equal(host(graph.k), k_want)
        assert np.array_equal(host(dec.decode(dev(fresh))), want)  # eager work on the same decoder between the replays
    start = oracle_stack(ref[:1], xs, *dims)[0]
    buf = dev(start.copy())
    dec.decode(buf, out=buf, layers=(1, layers))
    assert np.array_equal(host(buf), x_ref)
    dec.set_chains(1)
    assert np.array_equal(host(dec.decode(dev(xs))), x_ref)
    with pytest.raises(bh.BitLinearError) as ei:
        dec.set_chains(9)
    assert ei.value.kind == "InvalidConfig"


def test_decoder_recorded_step_argument_errors():
    dec = bh.DecoderProjections(2, 256, 512, 4, 2, 64, max_tokens=2)
    x = torch.zeros((1, 256), device="cuda")
    with pytest.raises(bh.BitLinearError) as ei:  # no weights yet: nothing is recorded
        dec.record(x)
    assert ei.value.kind == "NotInitialized"
    with pytest.raises(bh.BitLinearError) as ei:
        dec.record(torch.zeros((3, 256), device="cuda"))
    assert ei.value.kind == "ShapeMismatch"
    with pytest.raises(bh.BitLinearError) as ei:
        dec.record(x, layers=(1, 1))
    assert ei.value.kind == "InvalidConfig"
    lib = bh.load_library()
    assert lib.bitnet_hip_decoder_graph_launch(None, None) == bh.NULL_POINTER
    lib.bitnet_hip_decoder_graph_destroy(None)


@pytest.mark.parametrize("layout", [bh.LAYOUT_OUT_IN, bh.LAYOUT_IN_OUT])
@pytest.mark.parametrize("n,k", [(1, 4), (48, 300), (640, 2560)])
def test_gguf_ternary_tensor_ingestion(n, k, layout):
    """A GGUF BitnetB158 tensor (8-byte header + 2-bit codes, either orientation, code 3 included) loaded straight
    into the layer: the layer then holds what the reference's decoder yields, and its forward matches the oracle."""
    rng = np.random.default_rng(n * 7 + k + layout)
    codes = rng.integers(0, 4, size=(n, k)).astype(np.uint8)  # code 3 decodes to 0 (gguf.rs:1139)
    if (n, k) == (1, 4):
        codes = np.array([[0, 1, 2, 0]], np.uint8)  # the reference's test vector 0x24 (gguf.rs:2421-2436)
    src = codes if layout == bh.LAYOUT_OUT_IN else codes.T
    flat = np.ascontiguousarray(src).reshape(-1)
    flat = np.concatenate([flat, np.zeros((-flat.size) % 4, np.uint8)])
    body = (flat[0::4] | (flat[1::4] << 2) | (flat[2::4] << 4) | (flat[3::4] << 6)).astype(np.uint8)
    scale = np.float32(0.0173)
    tensor = np.concatenate([np.frombuffer(np.array([scale, 0.5], "<f4").tobytes(), np.uint8), body])
    q_ref, s_ref, o_ref = orc.gguf_decode_ternary(tensor, n * k)
    w_ref = q_ref.reshape(src.shape) if layout == bh.LAYOUT_OUT_IN else q_ref.reshape(src.shape).T
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "gguf")
    for data in (torch.from_numpy(tensor.copy()), dev(tensor)):
        got_scale, got_offset = layer.load_gguf_ternary(data, layout)
        assert (got_scale, got_offset) == (s_ref, o_ref)
        packed, ws = layer.get_quantized_weights()
        assert ws == s_ref
        assert np.array_equal(orc.unpack_2bit(packed.numpy(), n * k).reshape(n, k), w_ref)
    x = synth_activations(rng, 3, k)
    out = layer.forward(dev(x))
    ref = orc.bitlinear_forward(x, orc.pack_2bit(np.ascontiguousarray(w_ref).reshape(-1)), n, float(s_ref))[0]
    assert np.array_equal(host(out), ref)
    with pytest.raises(bh.BitLinearError) as ei:
        layer.load_gguf_ternary(torch.from_numpy(tensor[:-1].copy()), layout)
    assert ei.value.kind == "ShapeMismatch"


# ---- inference backend ---------------------------------------------------------------------------------------

def test_inference_backend_execute_batch_matches_per_input_oracle():
    """HipInferenceBackend (InferenceBackend, engine/mod.rs:126-138): a batch of inputs of different row counts, each
    result equal to the oracle's decoder chain on that input alone, however the inputs were grouped into passes."""
    dims = (256, 512, 4, 2, 64)
    rng = np.random.default_rng(77)
    dec, ref = build_decoder(rng, 2, *dims, max_tokens=8)
    backend = bh.create_backend("hip:0")
    caps = backend.capabilities()
    assert caps.supports_batching and not caps.supports_streaming and caps.max_batch_size == 0 and caps.device_type == "hip:0"
    assert backend.get_memory_usage() == 0
    with pytest.raises(bh.BitLinearError) as ei:
        backend.execute_batch([dev(synth_activations(rng, 1, dims[0]))])
    assert ei.value.kind == "NotInitialized"
    backend.optimize_model(dec)
    assert backend.capabilities().max_batch_size == 8 and backend.capabilities().memory_limit > 1 << 30
    assert backend.get_memory_usage() > dec.weight_bytes() * 2
    xs = [synth_activations(rng, r, dims[0]) for r in (1, 3, 2, 4, 8, 1, 1)]  # 1+3+2 | 4 | 8 | 1+1
    outs = backend.execute_batch([dev(x) for x in xs])
    assert len(outs) == len(xs)
    for x, o in zip(xs, outs):
        assert np.array_equal(host(o), oracle_stack(ref, x, *dims)[0])
    one = backend.execute_batch([dev(xs[0][0])])  # a rank-1 input is one row
    assert tuple(one[0].shape) == (dims[0],) and np.array_equal(host(one[0]), oracle_stack(ref, xs[0], *dims)[0][0])
    assert backend.execute_batch([]) == []
    with pytest.raises(bh.BitLinearError) as ei:
        backend.execute_batch([dev(synth_activations(rng, 9, dims[0]))])
    assert ei.value.kind == "ShapeMismatch"
    with pytest.raises(bh.BitLinearError) as ei:
        backend.execute_batch([dev(synth_activations(rng, 2, dims[0] + 4))])
    assert ei.value.kind == "ShapeMismatch"
    empty = bh.DecoderProjections(1, *dims, max_tokens=2)
    with pytest.raises(bh.BitLinearError) as ei:
        bh.HipInferenceBackend().optimize_model(empty)
    assert ei.value.kind == "NotInitialized"


# ---- C++ host mirror -----------------------------------------------------------------------------------------

def test_cpp_host_mirror_selftest():
    """bitnet-mlx.rs_amd/host/bitlinear.hpp (the C++ stand-in for the Rust types) against the reference's own
    BitLinear forward tests and against the other routes through the library."""
    import subprocess
    from pathlib import Path

    exe = Path(bh.LIB_PATH).parents[1] / "bin" / "host_selftest"
    assert exe.exists(), "build first: make -C bitnet-mlx.rs_amd"
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=110)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    assert "all passed" in proc.stdout


def test_mfma_rate_diagnostic_is_plausible():
    """The matrix-unit loop bench.py quotes beside the prefill rates: between a tenth of and the published dense int8
    peak (5.0 POP/s), and constant operands are not slower than switching ones beyond run-to-run noise."""
    rand, const = bh.measure_mfma_i8_rate(True), bh.measure_mfma_i8_rate(False)
    assert 500.0 < rand < 5100.0 and 500.0 < const < 5100.0
    assert const > 0.9 * rand


def test_bitlinear_housekeeping_methods_of_the_reference():
    """clear_cache / cache_stats / to_device / device (layer.rs:223,353-411) and Quantizer::get_stats (weights.rs:638-640)
    as the reference's call sites use them: nothing to clear, the same device is a no-op, another device is refused."""
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=64, out_features=32), "api")
    assert layer.clear_cache() is None and layer.cache_stats() is None
    assert layer.device.startswith("hip")
    assert layer.to_device(layer.device) is None and layer.to_device("cuda") is None
    with pytest.raises(bh.BitLinearError) as ei:
        layer.to_device("cpu")
    assert ei.value.kind == "DeviceError"
    stats = bh.BitNetWeightQuantizer().get_stats()
    assert (stats.elements_count, stats.quantization_error, stats.compression_ratio, stats.scale_factor, stats.zero_point) == (0, 0.0, 1.0, 1.0, None)


# ---- device diagnostics behind the C ABI -----------------------------------------------------------------------------------

def test_launch_chain_and_hand_over_diagnostics():
    """bitnet_hip_measure_launch_chain and bitnet_hip_measure_hop: plausible figures, argument checks, and the bounded
    waits of the hand-over kernel: with a spin limit of one look every wait gives up, the call reports that the vector did
    not arrive intact, and the kernel has ended normally (the next call on the device works)."""
    empty = bh.measure_launch_chain(60, replays=5)
    assert 10.0 < empty < 2000.0  # 60 dependent empty kernels: microseconds each, not nanoseconds and not milliseconds
    buf = torch.zeros(60 * 65536, dtype=torch.uint8, device="cuda")
    reads = bh.measure_launch_chain(60, replays=5, buf=buf, bytes_per_launch=[65536])
    assert reads >= 0.5 * empty
    with pytest.raises(bh.BitLinearError):
        bh.measure_launch_chain(61, replays=5, buf=buf, bytes_per_launch=[65536])  # needs more bytes than the buffer holds
    with pytest.raises(bh.BitLinearError):
        bh.measure_launch_chain(2, replays=5, buf=buf, bytes_per_launch=[24])
    for two_level in (False, True):
        us, intact = bh.measure_hop(640, hops=20, two_level=two_level)
        assert intact and 0.2 < us < 200.0
    us, intact = bh.measure_hop(2560, hops=8, two_level=False, spin_limit=1)
    assert not intact  # every wait gave up after one look; the kernel ended all the same
    us, intact = bh.measure_hop(640, hops=20)
    assert intact
    with pytest.raises(bh.BitLinearError):
        bh.measure_hop(0, hops=5)


@pytest.mark.parametrize("m,n,k", [(1, 33, 256), (8, 100, 2560), (9, 33, 260), (40, 64, 301), (130, 96, 512)])
def test_native_call_path_matches_the_checked_one(m, n, k):
    """The binding's native call path (plain tensors) against the Python one (taken when a workspace is supplied): the same
    bits with every combination of operands, two- and three-dimensional inputs, a given output and a given stream; what the
    native path does not take reaches the Python checks and raises."""
    rng = np.random.default_rng(m + n + k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "native")
    layer.update_weights(dev(synth_weights(rng, n, k)))
    x, g = dev(synth_activations(rng, m, k, outliers=True)), dev(rng.standard_normal(k, dtype=f32))
    res = dev(rng.standard_normal((m, n), dtype=f32))
    ws = torch.empty((layer.workspace_size(m),), dtype=torch.uint8, device="cuda")
    side = torch.cuda.Stream()
    for gamma in (None, g):
        for residual in (None, res):
            want = layer.forward(x, gamma=gamma, residual=residual, workspace=ws)
            assert torch.equal(layer.forward(x, gamma=gamma, residual=residual), want)
            assert torch.equal(layer.forward(x.view(1, m, k), gamma=gamma, residual=residual), want.view(1, m, n))
            out = torch.full((m, n), float("nan"), device="cuda")
            assert layer.forward(x, gamma=gamma, residual=residual, out=out) is out and torch.equal(out, want)
            torch.cuda.synchronize()
            on_side = layer.forward(x, gamma=gamma, residual=residual, stream=side)
            torch.cuda.synchronize()
            assert torch.equal(on_side, want)
    for a, b in zip(bh.forward_multi([layer, layer], x, gamma=g), bh.forward_multi((layer, layer), x, gamma=g, stream=torch.cuda.current_stream())):
        assert torch.equal(a, b) and torch.equal(a, layer.forward(x, gamma=g))
    for bad in (lambda: layer.forward(x.cpu()), lambda: layer.forward(x.double()), lambda: layer.forward(x[:, :-1].contiguous()),
                lambda: layer.forward(x, gamma=g[:-1]), lambda: layer.forward(x, residual=res[:, :-1]), lambda: layer.forward(x[0]),
                lambda: layer.forward(x, out=torch.empty((m + 1, n), device="cuda")), lambda: bh.forward_multi([layer], x.t()),
                lambda: bh.BitLinear(layer.config, "no weights").forward(x)):
        with pytest.raises(bh.BitLinearError):
            bad()


@pytest.mark.parametrize("n,k", [(1, 1), (9000, 8), (1025, 33), (3, 600), (64, 700), (20, 1300), (100, 6404)])
@pytest.mark.parametrize("method", [None, bh.TernaryMethod.MeanThreshold, bh.TernaryMethod.OptimalThreshold])
def test_weight_quantisers_at_the_edges_of_their_batches(n, k, method):
    """Rows shorter and longer than a batch of loads, rows that share bytes, more rows than one round of the final sums, and an
    absmean whose rounding boundary is hit exactly (half the mean, and its neighbours)."""
    rng = np.random.default_rng(n + k)
    w = synth_weights(rng, n, k)
    if method is None:
        w[:] = np.where(rng.random((n, k)) < 0.5, f32(0.0137) * f32(0.5), f32(0.0137) * f32(1.5))
        for _ in range(3):  # the mean settles: half of it and the floats around it, in either sign, replace the small half
            s = orc.quantize_weights_absmean(w)[1]
            half = s * f32(0.5)
            edge = np.array([half, np.nextafter(half, f32(0)), np.nextafter(half, f32(1))], dtype=f32)
            w = np.where(np.abs(w) < s, rng.choice(np.concatenate([edge, -edge]), size=w.shape), w).astype(f32)
        q, s = orc.quantize_weights_absmean(w)
        packed, scale, q_dev = bh.quantize_weights(dev(w), want_i8=True)
        assert np.array_equal(host(q_dev), q) and f32(host(scale)[0]) == s and np.array_equal(host(packed), orc.pack_2bit(q))
        off = torch.empty((n * k + 1,), device="cuda")[1:].view(n, k)  # not 16-byte aligned
        off.copy_(dev(w))
        assert torch.equal(bh.quantize_weights(off)[0], packed)
    else:
        got = bh.BitNetWeightQuantizer(bh.WeightQuantizationConfig(ternary_method=method)).quantize(dev(w))
        q, scale, _, stats = orc.quantize_weights_reference(w, method=method, want_details=True)
        assert np.array_equal(host(got.values), q) and np.array_equal(host(got.packed), orc.pack_2bit(q))
        assert host(got.scales)[0] == scale and all(f32(got.stats[name]) == v for name, v in stats.items())


@pytest.mark.parametrize("n,k", [(1, 1), (17, 257), (40, 1000), (33, 48), (2048, 4100), (1040, 2064)])
@pytest.mark.parametrize("layout", [bh.LAYOUT_OUT_IN, bh.LAYOUT_IN_OUT])
def test_layers_loaded_from_the_host_give_their_bytes_back(n, k, layout):
    """GGUF codes through the pinned chunks (more than one of them, a last one that is not full) and below their size, re-tiled
    from both orientations at widths that are and are not whole dwords, code 3 included: the layer's bytes and tiles."""
    rng = np.random.default_rng(n + k)
    raw = rng.integers(0, 256, size=(n * k + 3) // 4, dtype=np.uint8)
    w = orc.unpack_2bit(raw, n * k)
    w = w.reshape(n, k) if layout == bh.LAYOUT_OUT_IN else np.ascontiguousarray(w.reshape(k, n).T)
    header = np.array([0.75, 0.0], dtype=f32).view(np.uint8)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "loaded")
    for data in (torch.from_numpy(np.concatenate([header, raw])), dev(np.concatenate([header, raw]))):
        assert layer.load_gguf_ternary(data, layout=layout) == (0.75, 0.0)
        packed, scale = layer.get_quantized_weights()
        assert scale == 0.75 and np.array_equal(packed.numpy(), orc.pack_2bit(w))
        tiled = bh.retile_weights(dev(raw), n, k, layout)
        assert np.array_equal(host(bh.untile_weights(tiled, n, k)), orc.pack_2bit(w))
        x = synth_activations(rng, 2, k)
        assert np.array_equal(host(layer.forward(dev(x))), orc.bitlinear_forward(x, orc.pack_2bit(w), n, f32(0.75))[0])


@pytest.mark.parametrize("m,k", [(512, 516), (513, 516), (300, 4096), (300, 4100), (513, 7168), (513, 7172), (3, 8192), (513, 1024), (513, 301)])
@pytest.mark.parametrize("norm", [False, True])
def test_activation_quant_at_the_edges_of_its_kernels(m, k, norm):
    """Rows on both sides of each line between the quantiser's kernels: rows that all run at once and more, one and two chunks per
    thread, rows too long for a 256-thread workgroup's registers, short rows, rows that start unaligned."""
    rng = np.random.default_rng(m + k)
    x = synth_activations(rng, m, k, outliers=True)
    x[1] = 0.0
    x[2, ::7] *= f32(2.0**-70)
    g = rng.standard_normal(k, dtype=f32) if norm else None
    q, s, asum, _ = bh.quantize_activations_i8(dev(x), dev(g) if norm else None, eps=1e-5, want_sum=True)
    q_ref, s_ref, rs_ref = orc.rmsnorm_quantize_i8(x, g, 1e-5, orc.SUM_BLOCK256)
    assert np.array_equal(host(s), s_ref) and np.array_equal(host(q), q_ref) and np.array_equal(host(asum), rs_ref)


@pytest.mark.parametrize("m,n,k", [(3, 40, 301), (130, 96, 441), (100, 330, 260), (300, 200, 3201)])
def test_forward_of_padded_widths_bit_exact(m, n, k):
    """Widths that are no multiple of a tile run on padded int8 rows; a workspace without room for the padding still serves."""
    rng = np.random.default_rng(m + n + k)
    w, x = synth_weights(rng, n, k), synth_activations(rng, m, k, outliers=True)
    g = rng.standard_normal(k, dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "padded")
    layer.update_weights(dev(w))
    qw, ws_ = orc.quantize_weights_absmean(w)
    ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws_, g=g, eps=1e-5)[0]
    up = lambda v: (v + 255) // 256 * 256
    least = torch.empty((up(m * k) + 2 * up(4 * m) + 256,), dtype=torch.uint8, device="cuda")
    assert least.numel() < layer.workspace_size(m)
    for ws in (None, least, torch.empty((layer.workspace_size(m),), dtype=torch.uint8, device="cuda")):
        assert np.array_equal(host(layer.forward(dev(x), gamma=dev(g), workspace=ws)), ref)


@pytest.mark.parametrize("m", [9, 16, 17, 95])
@pytest.mark.parametrize("n,k", [(1, 4), (33, 260), (300, 1025), (700, 2560), (1400, 4352), (260, 8192), (700, 8448), (1400, 8448)])
def test_forward_token_groups_bit_exact(m, n, k):
    """The token GEMV on rows laid out by the quantiser: last token groups of one to sixteen rows, one, two and four row blocks per
    workgroup, one and two k-tiles per wavefront and the loop over more, fewer tiles than wavefronts, row blocks past the end."""
    rng = np.random.default_rng(m + n + k)
    w, x = synth_weights(rng, n, k), synth_activations(rng, m, k, outliers=True)
    bias, res = rng.standard_normal(n, dtype=f32), rng.standard_normal((m, n), dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "groups")
    layer.update_weights(dev(w))
    layer.update_bias(dev(bias))
    qw, ws_ = orc.quantize_weights_absmean(w)
    ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws_, eps=1e-5, bias=bias, residual=res)[0]
    assert np.array_equal(host(layer.forward(dev(x), residual=dev(res))), ref)


@pytest.mark.parametrize("m", [1, 3, 20])
def test_decoder_steps_that_repeat_match_the_oracle(m):
    """The same tensors step after step (recorded on the third call and replayed), other tensors and row counts in between, more of
    them than the decoder keeps recordings for, and weights that change under a recording."""
    dims = (256, 512, 4, 2, 64)
    rng = np.random.default_rng(m)
    dec, ref = build_decoder(rng, 3, *dims, max_tokens=20)
    xs = [synth_activations(rng, m, 256) for _ in range(6)]
    ins, outs = [dev(x) for x in xs], [torch.empty((m, 256), device="cuda") for _ in xs]
    want = [oracle_stack(ref, x, *dims)[0] for x in xs]
    for step in range(5):
        for i in range(6 if step < 4 else 2):
            outs[i].fill_(float("nan"))
            dec.decode(ins[i], out=outs[i])
            assert np.array_equal(host(outs[i]), want[i])
        ins[0].copy_(dev(xs[step]))  # new values in the same buffer
        want[0] = want[step] if step else want[0]
        xs[0] = xs[step]
    w = synth_weights(rng, *dec.proj_shape(0))
    dec.projection(0, 0).update_weights(dev(w))
    dec.set_norm(1, 0, torch.full((256,), 1.25))
    qw, s = orc.quantize_weights_absmean(w)
    ref[0][0][0], ref[0][1][0] = orc.pack_2bit(qw), s
    ref[1] = (ref[1][0], ref[1][1], np.full(256, 1.25, dtype=f32), ref[1][3])
    want[1] = oracle_stack(ref, xs[1], *dims)[0]
    side = torch.cuda.Stream()
    for stream in (None, side, None):
        dec.decode(ins[1], out=outs[1], stream=stream)
        torch.cuda.synchronize()
        assert np.array_equal(host(outs[1]), want[1])


def test_inference_backend_moves_many_unaligned_inputs():
    """More inputs than one launch moves, some at addresses that are no multiple of 16 bytes, rows longer than one workgroup's share."""
    dims = (1280, 512, 20, 5, 64)
    rng = np.random.default_rng(5)
    dec, ref = build_decoder(rng, 1, *dims, max_tokens=64)
    backend = bh.create_backend("hip:0")
    backend.optimize_model(dec)
    xs = [synth_activations(rng, 7 if i == 3 else 1 + i % 2, dims[0]) for i in range(36)]
    ins = []
    for i, x in enumerate(xs):
        flat = torch.empty((x.size + 1,), device="cuda")
        ins.append(flat[i % 2:i % 2 + x.size].view(x.shape).copy_(dev(x)))
    for x, o in zip(xs, backend.execute_batch(ins)):
        assert np.array_equal(host(o), oracle_stack(ref, x, *dims)[0])


@pytest.mark.parametrize("m,n,k", [(96, 33, 256), (130, 2049, 256), (700, 300, 256), (2000, 1600, 200), (1100, 2700, 256), (2500, 8200, 250)])
def test_gemm_of_one_weight_tile_per_row_bit_exact(m, n, k):
    """The shortest contraction of the LDS-direct kernels, two load stages, at each of their tile shapes."""
    rng = np.random.default_rng(m + n)
    w, x = synth_weights(rng, n, k), synth_activations(rng, m, k, outliers=True)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "short")
    layer.update_weights(dev(w))
    qw, ws_ = orc.quantize_weights_absmean(w)
    assert np.array_equal(host(layer.forward(dev(x))), orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws_)[0])


@pytest.mark.parametrize("m", [9, 12, 16, 17, 33, 95])
@pytest.mark.parametrize("n,k", [(1, 4), (33, 260), (300, 1024), (1400, 768), (2200, 512), (5000, 100)])
def test_forward_of_short_rows_in_one_launch_bit_exact(m, n, k):
    """Rows that every workgroup quantises for itself (and their neighbours beyond its lines): one to sixteen rows in the last token
    group, widths that are no multiple of a piece or a tile, one to four row blocks a workgroup, groups past the end; with and
    without norm, a zero row, one too small and one too large for the short division."""
    rng = np.random.default_rng(m + n + k)
    w, x = synth_weights(rng, n, k), synth_activations(rng, m, k, outliers=True)
    x[1] = 0.0
    x[2] *= f32(2.0**-70)
    x[3] *= f32(2.0**70)
    g, bias, res = rng.standard_normal(k, dtype=f32), rng.standard_normal(n, dtype=f32), rng.standard_normal((m, n), dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "short rows")
    layer.update_weights(dev(w))
    layer.update_bias(dev(bias))
    qw, ws_ = orc.quantize_weights_absmean(w)
    ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws_, eps=1e-5, bias=bias, residual=res)[0]
    assert np.array_equal(host(layer.forward(dev(x), residual=dev(res))), ref)
    ref = orc.bitlinear_forward(x, orc.pack_2bit(qw), n, ws_, g=g, eps=1e-5, bias=bias)[0]
    assert np.array_equal(host(layer.forward(dev(x), gamma=dev(g))), ref)
    outs = bh.forward_multi([layer] * 4, dev(x), gamma=dev(g))
    assert all(np.array_equal(host(o), ref) for o in outs)


@pytest.mark.parametrize("dims,m", [((2560, 256, 20, 5, 128), 8), ((192, 320, 12, 3, 16), 9), ((4352, 64, 34, 2, 128), 17), ((4096, 64, 64, 8, 64), 13),
                                    ((1344, 64, 21, 7, 64), 40), ((672, 64, 21, 7, 32), 95)])
def test_decoder_output_projection_reads_distinct_heads(dims, m):
    """The attention output projection on its distinct columns: groups of one to seventeen query heads, one and two k-tiles a
    wavefront, heads of one piece, row counts on both sides of a token group; row blocks that fill the chip but not each of its dies."""
    rng = np.random.default_rng(m)
    dec, ref = build_decoder_packed(rng, 1, *dims, max_tokens=m)
    x = synth_activations(rng, m, dims[0])
    assert np.array_equal(host(dec.decode(dev(x))), oracle_stack(ref, x, *dims)[0])


@pytest.mark.parametrize("m,n,k", [(33, 17100, 256), (49, 12900, 300), (65, 10300, 512), (80, 24700, 1600), (95, 33003, 256), (49, 65540, 260), (90, 103001, 300)])
def test_forward_of_long_outputs_at_few_tokens_bit_exact(m, n, k):
    """Few tokens and many outputs, on both sides of the line from which the GEMM takes over below 96 tokens: incomplete row tiles, its
    loader-fed tiles (1600 columns) and those of its other kernel."""
    rng = np.random.default_rng(m)
    x = synth_activations(rng, m, k, outliers=True)
    pk = random_packed_ternary(rng, n, k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "long")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    assert np.array_equal(host(layer.forward(dev(x))), orc.bitlinear_forward(x, pk, n, f32(0.02))[0])


@pytest.mark.parametrize("precision", [bh.QuantizationPrecision.OneFiveFiveBit, bh.QuantizationPrecision.EightBit])
@pytest.mark.parametrize("count,offset", [(1, 0), (4099, 0), (4099, 1), (32767, 0), (32768, 0), (32769, 0), (32800, 1), (700001, 0), (5000000, 0)])
def test_dynamic_quantiser_step_at_the_edges_of_its_kernels(precision, count, offset):
    """Tensors held by one workgroup and larger ones, addresses that are no multiple of 16 bytes, NaN and zero maxima, both 8-bit
    forms, a step with and without an average before it: scale and values as the state and the oracle have them."""
    rng = np.random.default_rng(count + offset)
    for u8 in (False, True):
        cfg = bh.ActivationQuantizationConfig(precision=precision, ema_decay=0.7)
        quant, model = bh.DynamicActivationQuantizer(cfg, reference_u8=u8), bh.DynamicScaleState(cfg)
        for step, mag in enumerate((2.0, 0.0, 5.0) if step_sizes_fit(count) else (2.0,)):
            x = (rng.standard_normal(count) * mag).astype(f32)
            if step == 2 and count > 1:
                x[count // 2] = np.nan
            t = torch.empty((count + offset,), device="cuda")[offset:].copy_(dev(x))
            out = quant.quantize_dynamic(t)
            ema = model.update(np.nanmax(np.abs(x)))
            assert f32(out.stats["scale_factor"]) == ema == f32(host(out.scales)[0])
            want = orc.quantize_activations_scaled(x, precision, float(ema), reference_u8=u8)
            assert np.array_equal(host(out.values).view(np.int8), want)


def step_sizes_fit(count):
    return count < 1000000  # one step of the largest tensor is enough


@pytest.mark.parametrize("m", [2, 3, 5, 8])
@pytest.mark.parametrize("n,k", [(16384, 256), (10300, 516), (6400, 1024), (9600, 1028)])
def test_forward_of_few_short_rows_and_long_outputs_bit_exact(m, n, k):
    """Two to eight tokens on both sides of the lines at which the launch quantises every row once a workgroup instead of one row a
    workgroup, or is two launches; a zero row, one too small and one too large for the short division."""
    rng = np.random.default_rng(m + n + k)
    x, pk, g = synth_activations(rng, m, k, outliers=True), random_packed_ternary(rng, n, k), rng.standard_normal(k, dtype=f32)
    x[1] *= f32(2.0**-70)
    if m > 3:
        x[2], x[3] = 0.0, x[3] * f32(2.0**70)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "few rows")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    res = rng.standard_normal((m, n), dtype=f32)
    assert np.array_equal(host(layer.forward(dev(x), residual=dev(res))), orc.bitlinear_forward(x, pk, n, f32(0.02), residual=res)[0])
    assert np.array_equal(host(layer.forward(dev(x), gamma=dev(g))), orc.bitlinear_forward(x, pk, n, f32(0.02), g=g, eps=1e-5)[0])


@pytest.mark.parametrize("dims", [(2304, 64, 18, 2, 128), (2560, 64, 20, 5, 128), (3200, 64, 25, 5, 128), (5120, 64, 40, 8, 128), (896, 4864, 14, 2, 64)])
@pytest.mark.parametrize("m", [2, 3, 7, 8])
def test_decoder_blocks_of_two_to_eight_tokens_match_the_oracle(dims, m):
    """The attention output projection by either one-launch kernel, on both sides of the line between them, and gate and up of a
    narrow model where the workgroups of one of them do not fit one round."""
    rng = np.random.default_rng(m + dims[0])
    dec, ref = build_decoder_packed(rng, 1, *dims, max_tokens=m)
    x = synth_activations(rng, m, dims[0])
    assert np.array_equal(host(dec.decode(dev(x))), oracle_stack(ref, x, *dims)[0])


@pytest.mark.parametrize("m,n,k", [(130, 45, 512), (300, 1001, 256), (1000, 2403, 512), (1000, 2564, 512), (700, 5030, 256), (2100, 6901, 256), (130, 643, 4096)])
@pytest.mark.parametrize("extras", [False, True], ids=["plain", "bias_residual"])
def test_gemm_rows_that_begin_inside_a_line(m, n, k, extras):
    """Output widths that are no multiple of 32 floats, odd ones among them, through every LDS-direct kernel: the last group of four
    columns cut, bias and residual read at any alignment.  Exact integers and single IEEE operations: the same bits."""
    rng = np.random.default_rng(m + n)
    x = synth_activations(rng, m, k, outliers=True)
    pk = random_packed_ternary(rng, n, k)
    bias = rng.standard_normal(n, dtype=f32) if extras else None
    res = rng.standard_normal((m, n), dtype=f32) if extras else None
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=extras), "lines")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    if extras:
        layer.update_bias(dev(bias))
    got = host(layer.forward(dev(x), residual=dev(res) if extras else None))
    ref = orc.bitlinear_forward(x, pk, n, f32(0.02), bias=bias, residual=res)[0]
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("m,n,k", [(3100, (6917, 3000), 512), (1030, (32768,), 256), (3073, (16385,), 1024), (3200, (4100, 4100, 33), 2048)])
def test_gemm_128x256_tiles_and_grouped_rows(m, n, k):
    """128 x 256 tiles (launches of 640 and more 128 x 160 tiles where they come out even), the last row and column tile cut, and the
    walk down eight row tiles at a time (24 and more of them, weights above 4 MiB) with an incomplete last group: the same bits as the
    oracle on rows at both ends, in the middle and on either side of a group, and as each layer by itself."""
    rng = np.random.default_rng(m + k)
    x = synth_activations(rng, m, k, outliers=True)
    layers, packs = [], []
    for w in n:
        packs.append(random_packed_ternary(rng, w, k))
        layers.append(bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=w), "wide"))
        layers[-1].set_quantized_weights(torch.from_numpy(packs[-1]), 0.02)
    xd = dev(x)
    outs = bh.forward_multi(layers, xd) if len(n) > 1 else [layers[0].forward(xd)]
    rows = sorted({0, 1, 127, 128, 1023, 1024, m // 2, m - 1})
    for w, pk, out in zip(n, packs, outs):
        ref = orc.bitlinear_forward(x[rows], pk, w, f32(0.02))[0]
        assert np.array_equal(host(out)[rows].view(np.uint32), ref.view(np.uint32))
    single = layers[0].forward(xd[: m // 3].contiguous())
    assert torch.equal(single, outs[0][: m // 3])


ONE_ROUND = [(17, 30000), (64, 33), (65, 4100), (130, 1100), (200, 3000), (257, 6000), (333, 8192), (500, 3073), (700, 6500), (1025, 2500), (2040, 2560),
             (513, 33), (650, 1101), (520, 1100), (650, 2001), (257, 5999), (333, 8170)]
ONE_ROUND_K = [1024, 1280, 2816]


@pytest.mark.parametrize("k", ONE_ROUND_K)
@pytest.mark.parametrize("m,n", ONE_ROUND)
def test_gemm_tiles_of_one_round_bit_exact(m, n, k):
    """Launches that one round of the loader-fed workgroups holds: every tile of its table (64 x 32 to 128 x 160, one or two workgroups per
    compute unit) with its last row and column tile cut, which test_host_side.py checks, four to eleven stages; and, up to 200 tokens,
    neighbours that the token GEMV takes; int32 and f32 output through matmul, f32 through forward."""
    rng = np.random.default_rng(m + n + k)
    x = synth_activations(rng, m, k, outliers=True)
    pk = random_packed_ternary(rng, n, k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "round")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    ref, q, a_scale, acc_ref = orc.bitlinear_forward(x, pk, n, f32(0.02))
    assert np.array_equal(host(layer.forward(dev(x))).view(np.uint32), ref.view(np.uint32))
    acc, out = bh.matmul_w2a8(bh.retile_weights(dev(pk), n, k), dev(q), n, dev(np.array([0.02], dtype=f32)), dev(a_scale),
                              a_sum=dev(q.astype(np.int32).sum(axis=1).astype(np.int32)))
    assert np.array_equal(host(acc), acc_ref) and np.array_equal(host(out).view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("m,ns,k", [(1030, (6913,), 256), (1200, (4096,), 512), (800, (13830,), 256), (3072, (2560, 640, 640), 256), (2048, (5120,), 256), (65, (30000,), 768)])
def test_gemm_launches_between_one_round_and_many_tiles(m, ns, k):
    """64 x 128, 64 x 256, 128 x 128 and 64 x 160 tiles: launches that no single round of the loader-fed workgroups holds, with fewer than
    640 tiles of 128 x 160; several projections, tiles cut by rows and columns, one to three weight tiles a row."""
    rng = np.random.default_rng(m + k)
    x = synth_activations(rng, m, k, outliers=True)
    packs = [random_packed_ternary(rng, n, k) for n in ns]
    layers = []
    for n, pk in zip(ns, packs):
        layers.append(bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "between"))
        layers[-1].set_quantized_weights(torch.from_numpy(pk), 0.02)
    xd = dev(x)
    outs = bh.forward_multi(layers, xd) if len(ns) > 1 else [layers[0].forward(xd)]
    rows = sorted({0, 1, 63, 64, min(127, m - 1), m // 2, m - 2, m - 1})
    for n, pk, out in zip(ns, packs, outs):
        assert np.array_equal(host(out)[rows].view(np.uint32), orc.bitlinear_forward(x[rows], pk, n, f32(0.02))[0].view(np.uint32))
        assert torch.isfinite(out).all()
    assert torch.equal(layers[0].forward(xd[:40].contiguous()), outs[0][:40])


@pytest.mark.parametrize("m,k", [(3, 8196), (512, 8448), (513, 8448), (2, 12288), (40, 12292), (5, 16384), (3, 16388), (600, 16384)])
@pytest.mark.parametrize("norm", [False, True])
def test_activation_quant_of_rows_above_8192_columns(m, k, norm):
    """Four chunks a thread up to 16384 columns, both sides of the row counts and widths where the other kernels take over."""
    rng = np.random.default_rng(m + k)
    x = synth_activations(rng, m, k, outliers=True)
    g = (1.0 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32) if norm else None
    q, s, asum, _ = bh.quantize_activations_i8(dev(x), dev(g) if norm else None, eps=1e-5, want_sum=True)
    q_ref, s_ref, rs_ref = orc.rmsnorm_quantize_i8(x, g, 1e-5, orc.SUM_BLOCK256)
    assert np.array_equal(host(s), s_ref) and np.array_equal(host(q), q_ref) and np.array_equal(host(asum), rs_ref)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("n,k", [(17, 7172), (640, 8192), (4100, 8192), (33, 8196), (640, 12292), (2560, 13824), (100, 16384), (4096, 16384), (40, 16388)])
@pytest.mark.parametrize("norm", [False, True])
def test_forward_of_few_long_rows_bit_exact(m, n, k, norm):
    """One to eight tokens on rows above 7168 columns: quantised in the GEMV launch where one round of workgroups serves it (two or four
    chunks a thread, one to four row blocks a workgroup), by the stand-alone quantiser elsewhere; and through a workspace."""
    rng = np.random.default_rng(m + n + k)
    x = synth_activations(rng, m, k, outliers=True)
    g = (1.0 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32) if norm else None
    pk = random_packed_ternary(rng, n, k)
    res = rng.standard_normal((m, n), dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "long")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    gd = None if g is None else dev(g)
    ref, q_ref, s_ref, acc_ref = orc.bitlinear_forward(x, pk, n, f32(0.02), g=g, residual=res)
    assert np.array_equal(host(layer.forward(dev(x), gamma=gd, residual=dev(res))), ref)
    out, q, a_scale, acc = layer.forward(dev(x), gamma=gd, residual=dev(res), debug=True)
    assert np.array_equal(host(out), ref) and np.array_equal(host(q), q_ref) and np.array_equal(host(a_scale), s_ref) and np.array_equal(host(acc), acc_ref)
    ws = torch.empty((layer.workspace_size(m),), dtype=torch.uint8, device="cuda")
    assert np.array_equal(host(layer.forward(dev(x), gamma=gd, residual=dev(res), workspace=ws)), ref)


@pytest.mark.parametrize("ffn", [7424, 8192, 8448, 13824, 16640])
@pytest.mark.parametrize("m", [1, 2, 3, 5, 8, 20])
def test_decoder_blocks_with_wide_ffn_match_the_oracle(ffn, m):
    """The down projection of blocks whose FFN is wider than 7168 (relu2-gated input): each of its launches on both sides of the lines
    between them."""
    dims = (256, ffn, 4, 2, 64)
    rng = np.random.default_rng(ffn + m)
    dec, ref = build_decoder_packed(rng, 1, *dims, max_tokens=m)
    x = synth_activations(rng, m, dims[0])
    assert np.array_equal(host(dec.decode(dev(x))), oracle_stack(ref, x, *dims)[0])


@pytest.mark.parametrize("m,n,k", [(96, 512, 1024), (97, 33, 4), (132, 412, 416), (400, 640, 1024), (400, 640, 1028), (512, 500, 768), (513, 500, 768),
                                   (9, 2560, 1028), (16, 16384, 2048), (16, 16400, 2048), (40, 5120, 2044), (95, 40, 2052), (2, 9000, 1284), (17, 17, 1540)])
@pytest.mark.parametrize("norm", [False, True])
def test_forward_of_rows_quantised_by_every_workgroup(m, n, k, norm):
    """Up to 512 tokens, and rows of up to 2048 columns, in one launch: both sides of the lines beyond which it is two, one and two rounds
    of workgroups, chunks that no lane has, and several projections of one input."""
    rng = np.random.default_rng(m + 3 * n + k)
    x = synth_activations(rng, m, k, outliers=True)
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32) if norm else None
    gd = dev(g) if norm else None
    pk = random_packed_ternary(rng, n, k)
    bias, res = rng.standard_normal(n, dtype=f32), rng.standard_normal((m, n), dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "workgroup rows")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    layer.update_bias(dev(bias))
    ref, q_ref, s_ref, acc_ref = orc.bitlinear_forward(x, pk, n, f32(0.02), g=g, bias=bias, residual=res)
    assert np.array_equal(host(layer.forward(dev(x), gamma=gd, residual=dev(res))), ref)
    out, q, a_scale, acc = layer.forward(dev(x), gamma=gd, residual=dev(res), debug=True)
    assert np.array_equal(host(out), ref) and np.array_equal(host(q), q_ref) and np.array_equal(host(a_scale), s_ref) and np.array_equal(host(acc), acc_ref)
    other = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=24), "beside")
    pk2 = random_packed_ternary(rng, 24, k)
    other.set_quantized_weights(torch.from_numpy(pk2), 0.03)
    got = bh.forward_multi([other, layer], dev(x), gamma=gd)
    assert np.array_equal(host(got[0]), orc.bitlinear_forward(x, pk2, 24, f32(0.03), g=g)[0])
    assert np.array_equal(host(got[1]), orc.bitlinear_forward(x, pk, n, f32(0.02), g=g, bias=bias)[0])


@pytest.mark.parametrize("n,k", [(1, 4), (3, 258), (64, 260), (513, 64), (4095, 12), (4096, 20), (4097, 20), (4097, 6)])
@pytest.mark.parametrize("method,normalize,t", [(0, True, 3.0), (3, True, 3.0), (2, False, 2.5), (3, False, 0.0), (1, True, 0.0)])
def test_reference_weight_pipeline_with_reductions_finished_by_the_next_pass(n, k, method, normalize, t):
    """Row counts on both sides of the line from which a launch of its own finishes each reduction, fewer and more rows than a wavefront
    adds at a time, and every order of the passes."""
    rng = np.random.default_rng(n + k + method)
    w = (0.2 + 1.3 * rng.standard_normal((n, k))).astype(f32)
    w[rng.random(w.shape) < 0.01] *= f32(7.0)
    cfg = bh.WeightQuantizationConfig(normalize_weights=normalize, outlier_threshold=t, ternary_method=method)
    got = bh.BitNetWeightQuantizer(cfg).quantize(dev(w))
    q_ref, s_ref, _, st_ref = orc.quantize_weights_reference(w, method=method, normalize=normalize, outlier_threshold=t, want_details=True)
    assert np.array_equal(host(got.values), q_ref) and np.array_equal(host(got.packed), orc.pack_2bit(q_ref))
    assert host(got.scales)[0] == s_ref
    for name, v in st_ref.items():
        assert f32(got.stats[name]) == v, (name, got.stats[name], v)


@pytest.mark.parametrize("m,n,k", [(9, 1, 1280), (16, 15, 2560), (17, 40, 2304), (31, 4097, 1536), (33, 2573, 2560), (48, 13827, 2560), (95, 5001, 2304),
                                   (15, 2561, 6912), (30, 3330, 4352), (20, 20000, 4608), (13, 1023, 12288), (40, 6007, 9216), (300, 1030, 2560)])
@pytest.mark.parametrize("extras", [False, True])
def test_token_gemv_outputs_that_end_inside_a_row_block(m, n, k, extras):
    """Four outputs a lane: rows that start at any multiple of four bytes, last row blocks of 1 to 15 rows, token groups of 1 to 16 rows,
    one, two and four row blocks a workgroup, k-tiles in one batch and in several."""
    rng = np.random.default_rng(m + n + k)
    x = synth_activations(rng, m, k, outliers=True)
    x[0] *= f32(1e-30)
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32)
    nbytes = (n * k + 3) // 4
    pk = random_packed_ternary(rng, 1, 4 * nbytes)
    bias, res = (rng.standard_normal(n, dtype=f32), rng.standard_normal((m, n), dtype=f32)) if extras else (None, None)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=extras), "ends")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    if extras:
        layer.update_bias(dev(bias))
    ref = orc.bitlinear_forward(x, pk, n, f32(0.02), g=g, bias=bias, residual=res)[0]
    assert np.array_equal(host(layer.forward(dev(x), gamma=dev(g), residual=dev(res) if extras else None)), ref)


# ---- rows quantised once a die (gemv_die_kernel) -------------------------------------------------------------

def die_scratch(layer, x, gamma=None):
    """Bytes of workspace the layer wants for x on the null stream, and those without the flags of a launch on dies."""
    handles = (ctypes.c_void_p * 1)(layer._h)
    wanted = bh.load_library().bitnet_hip_bitlinear_forward_scratch_on(handles, 1, x.data_ptr(), x.shape[0], gamma.data_ptr() if gamma is not None else None,
                                                                       bh.SUM_BLOCK256, None)
    return wanted, layer.workspace_size(x.shape[0])


@pytest.mark.parametrize("m,k,n,norm", [(9, 2308, 2560, False), (9, 1028, 40, True), (16, 6912, 2560, False), (17, 2564, 650, True), (5, 8192, 8200, False),
                                        (33, 4096, 1000, False), (48, 2560, 2570, True), (31, 8192, 648, True), (95, 1536, 1290, True), (128, 1300, 96, True)])
def test_rows_quantised_once_a_die_bit_exact(m, k, n, norm):
    """Rows and columns left over, one and two tiles a wavefront, one to four row blocks a workgroup, up to eight token groups: the
    oracle's bits, on one workspace through calls with other inputs in between (the flags of an earlier call lie in it)."""
    rng = np.random.default_rng(m + 3 * k + n)
    w = synth_weights(rng, n, k)
    qw, ws = orc.quantize_weights_absmean(w)
    packed = orc.pack_2bit(qw)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "dies")
    layer.update_weights(dev(w))
    bias = rng.standard_normal(n, dtype=f32)
    layer.update_bias(dev(bias))
    gamma = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32) if norm else None
    x = dev(synth_activations(rng, m, k))
    wanted, plain = die_scratch(layer, x, dev(gamma) if norm else None)
    assert wanted > plain  # with flags: the launch this test is about
    scratch = torch.full((wanted,), 255, dtype=torch.uint8, device="cuda")
    for _ in range(3):
        xs = synth_activations(rng, m, k, outliers=True)
        xs[m // 2] = 0.0
        res = rng.standard_normal((m, n), dtype=f32)
        want = orc.bitlinear_forward(xs, packed, n, ws, g=gamma, bias=bias, residual=res)[0]
        g = dev(gamma) if norm else None
        assert np.array_equal(host(layer.forward(dev(xs), gamma=g, residual=dev(res), workspace=scratch)), want)
        assert np.array_equal(host(layer.forward(dev(xs), gamma=g, residual=dev(res))), want)
    least = torch.empty((plain,), dtype=torch.uint8, device="cuda")  # no room for flags: two launches
    assert np.array_equal(host(layer.forward(dev(xs), gamma=g, residual=dev(res), workspace=least)), want)


@pytest.mark.parametrize("k,n,norm", [(4100, 4097, True), (4100, 8193, False), (4356, 8201, True), (7168, 12304, False), (7172, 4100, False), (8192, 4129, True),
                                      (8196, 4112, False), (12288, 8225, False), (16384, 4111, False), (8452, 16401, False), (5120, 20500, True)])
def test_one_token_through_many_row_blocks(k, n, norm):
    """Rows of 17 to 64 k-tiles, a few columns past a tile, workgroups with one row block more than others, fewer and more of them than are in
    flight, last row blocks of 1 to 15 rows, the optional outputs, and two projections that share the row."""
    rng = np.random.default_rng(k + 3 * n)
    x = synth_activations(rng, 1, k, outliers=True)
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32) if norm else None
    gd = dev(g) if norm else None
    pk = random_packed_ternary(rng, 1, (n * k + 3) // 4 * 4)
    bias, res = rng.standard_normal(n, dtype=f32), rng.standard_normal((1, n), dtype=f32)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=True), "many")
    layer.set_quantized_weights(torch.from_numpy(pk), 0.02)
    layer.update_bias(dev(bias))
    ref, q_ref, s_ref, acc_ref = orc.bitlinear_forward(x, pk, n, f32(0.02), g=g, bias=bias, residual=res)
    for _ in range(2):
        assert np.array_equal(host(layer.forward(dev(x), gamma=gd, residual=dev(res))), ref)
    out, q, a_scale, acc = layer.forward(dev(x), gamma=gd, residual=dev(res), debug=True)
    assert np.array_equal(host(out), ref) and np.array_equal(host(q), q_ref) and np.array_equal(host(a_scale), s_ref) and np.array_equal(host(acc), acc_ref)
    other = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=24), "beside")
    pk2 = random_packed_ternary(rng, 24, k)
    other.set_quantized_weights(torch.from_numpy(pk2), 0.03)
    for order in ([other, layer], [layer, other], [other, layer, other]):
        for one, y in zip(order, bh.forward_multi(order, dev(x), gamma=gd)):
            want = orc.bitlinear_forward(x, pk2, 24, f32(0.03), g=g)[0] if one is other else orc.bitlinear_forward(x, pk, n, f32(0.02), g=g, bias=bias)[0]
            assert np.array_equal(host(y), want)


@pytest.mark.parametrize("dims", [(4352, 8448, 34, 2, 128), (8320, 512, 65, 5, 128)])
def test_decoder_blocks_of_many_row_blocks(dims):
    """One token through wide blocks, as it comes and recorded: gate and up, the relu2-gated down projection, and repeated heads."""
    rng = np.random.default_rng(sum(dims))
    dec, ref = build_decoder_packed(rng, 1, *dims, max_tokens=1)
    x = synth_activations(rng, 1, dims[0])
    want = oracle_stack(ref, x, *dims)[0]
    assert np.array_equal(host(dec.decode(dev(x))), want)
    graph = dec.record(dev(x))
    for _ in range(3):
        graph.out.zero_()
        graph.replay()
        assert np.array_equal(host(graph.out), want)


DIE_STACKS = [((512, 1408, 8, 2, 64), 3), ((2560, 6912, 20, 5, 128), 1)]  # dimensions and blocks
DIE_TOKENS = (9, 33, 16, 3, 64, 17)


@pytest.mark.parametrize("dims,layers", DIE_STACKS)
def test_decoder_rows_quantised_once_a_die(dims, layers):
    """Steps of several token counts, one after the other and recorded, with workgroups that wait for their rows and (no looks at all)
    with every one that quantises its rows itself: all equal the oracle's chain bit for bit."""
    rng = np.random.default_rng(sum(dims))
    dec, ref = build_decoder_packed(rng, layers, *dims, max_tokens=64)
    for m in DIE_TOKENS:
        xs = synth_activations(rng, m, dims[0])
        want = oracle_stack(ref, xs, *dims)[0]
        for looks in (0, 4096):
            dec.set_row_wait(looks)
            x = dev(xs)
            for _ in range(4):  # the third on is a replay
                assert np.array_equal(host(dec.decode(x)), want), (m, looks)
            graph = dec.record(x)
            for _ in range(3):
                graph.out.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert np.array_equal(host(graph.out), want), (m, looks)
    for looks in (-1, 4097):
        with pytest.raises(bh.BitLinearError):
            dec.set_row_wait(looks)


@pytest.mark.parametrize("looks", [0, 4096])
def test_decoder_rows_quantised_once_a_die_of_any_magnitude(looks):
    """Rows of zeros, of tiny and of huge values, with an infinity and with a NaN: a workgroup that quantises rows for itself divides plainly, those that it waits
    for by the short division with its own rule, and both give the oracle's bits."""
    dims = (512, 1408, 8, 2, 64)
    rng = np.random.default_rng(looks)
    dec, ref = build_decoder_packed(rng, 3, *dims, max_tokens=64)
    dec.set_row_wait(looks)
    xs = synth_activations(rng, 20, dims[0], outliers=True)
    xs[1] = 0.0
    xs[2] *= f32(1e-36)
    xs[3] *= f32(1e18)
    xs[4, 100] = f32(1e30)
    xs[5, ::2] = -0.0
    xs[17] = 0.0
    xs[18, 7] = np.inf
    xs[19, 3] = np.nan
    want = oracle_stack(ref, xs, *dims)[0]
    for _ in range(4):
        assert np.array_equal(host(dec.decode(dev(xs))), want, equal_nan=True)


def test_calls_on_dies_from_several_threads():
    """Launches whose workgroups wait for each other's rows, from three threads on streams of their own: each call's result is its own."""
    rng = np.random.default_rng(5)
    shapes = [(16, 6912, 2560), (9, 2560, 6912), (48, 2560, 5120)]
    jobs = []
    for m, k, n in shapes:
        packed = random_packed_ternary(rng, 1, n * k)
        layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "threads")
        layer.set_quantized_weights(torch.from_numpy(packed), 0.02)
        xs = [synth_activations(rng, m, k) for _ in range(3)]
        jobs.append((layer, [dev(x) for x in xs], [dev(orc.bitlinear_forward(x, packed, n, f32(0.02))[0]) for x in xs]))
        wanted, plain = die_scratch(layer, jobs[-1][1][0])
        assert wanted > plain
    torch.cuda.synchronize()
    wrong = []

    def work(layer, xs, wants):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for i in range(60):
                y = layer.forward(xs[i % 3])
                if not torch.equal(y, wants[i % 3]):
                    wrong.append((layer.config.in_features, i))

    threads = [threading.Thread(target=work, args=job) for job in jobs]
    for th in threads:
        th.start()
    for th in threads:
        th.join(timeout=100)
    assert not any(th.is_alive() for th in threads) and not wrong


def test_a_captured_call_with_room_for_flags():
    """Flags in the workspace would be up in a second replay: a captured call takes two launches, and every replay multiplies its own rows, with
    calls on the same workspace between the replays."""
    rng = np.random.default_rng(6)
    m, k, n = 16, 6912, 2560
    packed = random_packed_ternary(rng, 1, n * k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n), "captured")
    layer.set_quantized_weights(torch.from_numpy(packed), 0.02)
    x, out = torch.zeros((m, k), device="cuda"), torch.empty((m, n), device="cuda")
    wanted, plain = die_scratch(layer, x)
    scratch = torch.empty((wanted,), dtype=torch.uint8, device="cuda")
    layer.forward(x, out=out, workspace=scratch)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        layer.forward(x, out=out, workspace=scratch)
    for i in range(4):
        xs = synth_activations(rng, m, k)
        want = orc.bitlinear_forward(xs, packed, n, f32(0.02))[0]
        x.copy_(dev(xs))
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(out), want)
        assert np.array_equal(host(layer.forward(x, workspace=scratch)), want)


# ---- outputs over the input ----------------------------------------------------------------------------------

@pytest.mark.parametrize("m,k,norm", [(1, 2560, True), (1, 8192, False), (1, 7424, True), (2, 1024, False), (6, 2560, True), (8, 516, False), (16, 2560, True),
                                      (64, 2560, False), (33, 4096, True), (200, 1028, True)])
def test_forward_with_its_output_over_its_input(m, k, norm):
    """A square layer whose result takes the place of its input, wholly or shifted by one row, with and without a workspace, alone, captured, on the
    static scratch and among several layers: the oracle's bits at every size that a one-launch kernel takes without the overlap."""
    rng = np.random.default_rng(m + k)
    packed = random_packed_ternary(rng, 1, k * k)
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=k), "over")
    layer.set_quantized_weights(torch.from_numpy(packed), 0.02)
    g = (1 + 0.1 * rng.standard_normal(k, dtype=f32)).astype(f32) if norm else None
    gd = dev(g) if norm else None
    x = synth_activations(rng, m, k, outliers=True)
    want = orc.bitlinear_forward(x, packed, k, f32(0.02), g=g)[0]
    roomy = torch.empty((layer.workspace_size(m) + (1 << 17),), dtype=torch.uint8, device="cuda")
    for ws in (None, roomy, roomy[: layer.workspace_size(m)]):
        for _ in range(3):
            buf = dev(x)
            assert np.array_equal(host(layer.forward(buf, gamma=gd, out=buf, workspace=ws)), want)
    rows = torch.empty((m + 1, k), device="cuda")
    rows[1:] = dev(x)
    assert np.array_equal(host(layer.forward(rows[1:], gamma=gd, out=rows[:m])), want)
    buf = dev(x)
    with_residual = orc.bitlinear_forward(x, packed, k, f32(0.02), g=g, residual=x)[0]
    assert np.array_equal(host(layer.forward(buf, gamma=gd, residual=buf, out=buf)), with_residual)
    if m * k <= 1 << 20:
        buf = dev(x)
        assert np.array_equal(host(layer.forward_noalloc(buf, buf, gamma=gd)), want)
    # the C entry without a workspace, and with one of the size that forward_scratch names
    lib = bh.load_library()
    handles = (ctypes.c_void_p * 2)(layer._h, layer._h)
    asked = lib.bitnet_hip_bitlinear_forward_multi_scratch(handles, 2, buf.data_ptr(), m, _pointer(gd), bh.SUM_BLOCK256)
    for ws in (None, torch.empty((max(asked, 1),), dtype=torch.uint8, device="cuda")):
        buf, beside = dev(x), torch.empty((m, k), device="cuda")
        outs = (ctypes.c_void_p * 2)(beside.data_ptr(), buf.data_ptr())
        assert lib.bitnet_hip_bitlinear_forward_multi(handles, 2, buf.data_ptr(), m, _pointer(gd), 1e-5, bh.SUM_BLOCK256, outs, _pointer(ws),
                                                      ws.numel() if ws is not None else 0, None) == 0
        torch.cuda.synchronize()
        assert np.array_equal(host(beside), want) and np.array_equal(host(buf), want)
    source, buf = dev(x), torch.empty((m, k), device="cuda")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        buf.copy_(source)
        layer.forward(buf, gamma=gd, out=buf)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host(buf), want)


def _pointer(t):
    return t.data_ptr() if t is not None else None
