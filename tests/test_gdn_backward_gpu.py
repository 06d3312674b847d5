"""GPU parity of the gated delta-net layer backward
(SequenceDeltaNetLayer::bwd_impl, sequence_delta_net.cc:482-561) with the CPU
oracle, through the C ABI.  Shapes follow sequence_delta_net_test.cc (small odd
widths, grouped heads) and add the 128 x 128 head of the headline config."""
import numpy as np
import pytest

from tests.util import assert_close

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def capi():
    from pluto_amd import capi
    assert torch.cuda.is_available(), "these tests need the GPU"
    capi.lib()
    return capi


def dev(x, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    return t.to(dtype) if dtype is not None else t


def make_case(T, kh, vh, kd, vd, K, seed, batch=1):
    from oracle import pyoracle as po
    rng = np.random.default_rng(seed)
    channels = 2 * kh * kd + vh * vd
    r = lambda *shape: po.bf16_round(rng.standard_normal(shape).astype(np.float32))
    return dict(qkv=r(batch, T, channels), z=r(batch, T, vh * vd), a=r(batch, T, vh),
                b=r(batch, T, vh),
                conv=(0.5 * rng.standard_normal((channels, K))).astype(np.float32),
                a_log=(0.3 * rng.standard_normal(vh)).astype(np.float32),
                dt_bias=(0.3 * rng.standard_normal(vh)).astype(np.float32),
                norm=(1 + 0.2 * rng.standard_normal(vd)).astype(np.float32),
                dy=rng.standard_normal((batch, T, vh * vd)).astype(np.float32))


def run(capi, shape, rounding, seed=0, batch=1, with_parameters=True):
    from oracle import pyoracle as po
    T, kh, vh, kd, vd, K = shape
    kw = dict(key_heads=kh, value_heads=vh, key_head_dim=kd, value_head_dim=vd, conv_kernel_dim=K,
              round_to_bfloat16=rounding)
    p, op = capi.delta_params(**kw), po.delta_params(**kw)
    c = make_case(T, kh, vh, kd, vd, K, seed, batch)
    want = None
    for s in range(batch):
        one = po.gdn_sequence_backward(op, c["qkv"][s], c["z"][s], c["a"][s], c["b"][s], c["conv"],
                                       c["a_log"], c["dt_bias"], c["norm"], c["dy"][s])
        if want is None:
            want = {k: ([v] if k in ("dqkv", "dz", "da", "db") else v.copy()) for k, v in one.items()}
        else:
            for k, v in one.items():
                if k in ("dqkv", "dz", "da", "db"):
                    want[k].append(v)
                else:
                    want[k] += v
    for k in ("dqkv", "dz", "da", "db"):
        want[k] = np.stack(want[k])
    channels = 2 * kh * kd + vh * vd
    grads = None
    if with_parameters:
        grads = dict(conv_weight=torch.zeros(channels, K, device="cuda"),
                     a_log=torch.zeros(vh, device="cuda"), dt_bias=torch.zeros(vh, device="cuda"),
                     norm=torch.zeros(vd, device="cuda"))
    bf = torch.bfloat16
    args = (p, dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
            dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"]))
    dqkv, dz, da, db = capi.gdn_layer_backward(*args, parameter_grads=grads)
    torch.cuda.synchronize()
    got = dict(dqkv=dqkv.cpu().numpy(), dz=dz.cpu().numpy(), da=da.cpu().numpy(),
               db=db.cpu().numpy())
    if grads:
        got.update(d_conv_weight=grads["conv_weight"].cpu().numpy(),
                   d_a_log=grads["a_log"].cpu().numpy(), d_dt_bias=grads["dt_bias"].cpu().numpy(),
                   d_norm=grads["norm"].cpu().numpy())
    return got, want, args, grads


# (T, key heads, value heads, key width, value width, conv taps).  128 x 128
# heads take the chunked kernels (64-token chunks: one full chunk, a ragged
# tail, grouped heads over several chunks, and 1, 2, 3, 4 and 5 chunks: the
# sequential kernels request operands a chunk ahead); the other widths go token
# by token.
SHAPES = [(4, 1, 2, 3, 5, 3), (9, 2, 4, 5, 35, 4), (33, 2, 2, 16, 40, 4), (64, 1, 2, 128, 128, 4),
          (37, 1, 1, 128, 128, 4), (200, 1, 2, 128, 128, 4), (130, 2, 4, 128, 128, 3),
          (100, 1, 1, 128, 128, 2), (300, 1, 1, 128, 128, 4)]


@pytest.mark.parametrize("rounding", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_backward_matches_oracle(capi, shape, rounding):
    got, want, _, _ = run(capi, shape, rounding, seed=sum(shape))
    for name in want:
        what = "%s %s" % (name, shape)
        if not rounding:
            assert_close(got[name], want[name], 2e-4, what)
            continue
        # Rounded forward values enter as operands: where the FP32 and the
        # double-precision forward straddle a bf16 rounding tie an operand differs
        # by one ulp.  The bulk must agree to FP32 accuracy.
        expected = want[name].astype(np.float64)
        diff = np.abs(got[name] - expected)
        scale = np.abs(expected) + np.sqrt(np.mean(expected ** 2))
        print("%s: max-abs error %.3e" % (what, diff.max()))
        assert np.all(diff <= 2e-2 * scale), what
        assert np.mean(diff > 2e-4 * scale) <= 2e-2, what


def test_batch_and_parameter_gradient_accumulation(capi):
    shape = (7, 1, 2, 4, 6, 3)
    got, want, args, grads = run(capi, shape, False, seed=3, batch=3)
    for name in want:
        assert_close(got[name], want[name], 2e-4, name)
    first = {k: v.clone() for k, v in grads.items()}
    again = capi.gdn_layer_backward(*args, parameter_grads=grads)
    torch.cuda.synchronize()
    for k in grads:  # parameter gradients accumulate across calls
        np.testing.assert_allclose(grads[k].cpu().numpy(), 2 * first[k].cpu().numpy(), rtol=1e-5,
                                   atol=1e-6)
    for a, name in zip(again, ("dqkv", "dz", "da", "db")):
        np.testing.assert_array_equal(a.cpu().numpy(), got[name])  # repeatable
    frozen, _, _, _ = run(capi, shape, False, seed=3, batch=3, with_parameters=False)
    for name in ("dqkv", "dz", "da", "db"):
        np.testing.assert_array_equal(frozen[name], got[name])


def test_chunked_and_token_by_token_kernels_agree(capi):
    """128 x 128 heads over 9 chunks: the chunked kernels against the
    token-by-token kernels of the same library (FP32 both, different order of
    summation), at a length the CPU oracle would take minutes for."""
    import os
    shape = (520, 2, 4, 128, 128, 4)
    T, kh, vh, kd, vd, K = shape
    kw = dict(key_heads=kh, value_heads=vh, key_head_dim=kd, value_head_dim=vd, conv_kernel_dim=K,
              round_to_bfloat16=False)
    p = capi.delta_params(**kw)
    c = make_case(T, kh, vh, kd, vd, K, seed=11)
    bf = torch.bfloat16
    args = (p, dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
            dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"]))
    channels = 2 * kh * kd + vh * vd

    def once():
        grads = dict(conv_weight=torch.zeros(channels, K, device="cuda"),
                     a_log=torch.zeros(vh, device="cuda"), dt_bias=torch.zeros(vh, device="cuda"),
                     norm=torch.zeros(vd, device="cuda"))
        out = capi.gdn_layer_backward(*args, parameter_grads=grads)
        torch.cuda.synchronize()
        named = dict(zip(("dqkv", "dz", "da", "db"), out))
        named.update(grads)
        return {k: v.cpu().numpy() for k, v in named.items()}

    chunked = once()
    with capi.force_generic():
        sequential = once()
    for name in sequential:
        assert_close(chunked[name], sequential[name], 2e-4, name)


def test_long_sequence_two_heads_matches_oracle(capi):
    """T=2048 (32 chunks), two 128 x 128 heads: the length bench.py times, at a head
    count the scalar oracle finishes in seconds.  The chunked kernels treat heads
    independently (one workgroup row per head)."""
    shape = (2048, 2, 2, 128, 128, 4)
    got, want, _, _ = run(capi, shape, False, seed=5)
    assert capi.last_path() == capi.PATH_CHUNKED
    for name in want:
        assert_close(got[name], want[name], 2e-4, "%s %s" % (name, shape))


@pytest.mark.parametrize("length,key_heads", [(1, 33), (64, 11), (65, 3), (130, 33)])
def test_two_column_tiles_a_workgroup_match_the_oracle(capi, length, key_heads):
    """More heads than the compute units take one column tile of each: 33 of them, no
    multiple of the XCDs, for one chunk, a full one, one token more and three."""
    shape = (length, key_heads, 33, 128, 128, 4)
    got, want, _, _ = run(capi, shape, False, seed=length)
    for name in want:
        assert_close(got[name], want[name], 2e-4, "%s %s" % (name, shape))


def test_benchmarked_shape_against_token_by_token_kernels(capi):
    """The shape bench.py times (T=2048, sixteen 128 x 128 heads, every parameter
    trains): the chunked kernels against the token-by-token kernels of the same
    library, FP32 both."""
    shape = (2048, 16, 16, 128, 128, 4)
    T, kh, vh, kd, vd, K = shape
    p = capi.delta_params(key_heads=kh, value_heads=vh, key_head_dim=kd, value_head_dim=vd,
                          conv_kernel_dim=K, round_to_bfloat16=False)
    c = make_case(T, kh, vh, kd, vd, K, seed=4)
    bf = torch.bfloat16
    args = (p, dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
            dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"]))
    channels = 2 * kh * kd + vh * vd

    def once():
        grads = dict(conv_weight=torch.zeros(channels, K, device="cuda"),
                     a_log=torch.zeros(vh, device="cuda"), dt_bias=torch.zeros(vh, device="cuda"),
                     norm=torch.zeros(vd, device="cuda"))
        out = capi.gdn_layer_backward(*args, parameter_grads=grads)
        torch.cuda.synchronize()
        named = dict(zip(("dqkv", "dz", "da", "db"), out))
        named.update(grads)
        return {k: v.cpu().numpy() for k, v in named.items()}

    chunked = once()
    assert capi.last_path() == capi.PATH_CHUNKED
    with capi.force_generic():
        sequential = once()
        assert capi.last_path() == capi.PATH_RECURRENCE
    for name in sequential:
        assert_close(chunked[name], sequential[name], 2e-4, name)


@pytest.mark.parametrize("T,kh,vh", [(200, 16, 48), (65, 11, 33), (321, 18, 36), (64, 40, 40), (130, 8, 32)])
def test_many_value_heads_against_token_by_token_kernels(capi, T, kh, vh):
    """Beyond 32 value heads a workgroup of the sequential chunk kernels takes two column
    tiles: the decoder's own 16 key and 48 value heads (three to a key head), counts
    that are and are not multiples of eight (the two numberings of the workgroups), one
    chunk, a ragged one and several; 32 heads are the last with one tile."""
    kw = dict(key_heads=kh, value_heads=vh, key_head_dim=128, value_head_dim=128, conv_kernel_dim=4,
              round_to_bfloat16=False)
    p = capi.delta_params(**kw)
    c = make_case(T, kh, vh, 128, 128, 4, seed=T + vh)
    bf = torch.bfloat16
    args = (p, dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
            dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"]))

    def once():
        grads = dict(conv_weight=torch.zeros((2 * kh + vh) * 128, 4, device="cuda"),
                     a_log=torch.zeros(vh, device="cuda"), dt_bias=torch.zeros(vh, device="cuda"),
                     norm=torch.zeros(128, device="cuda"))
        out = capi.gdn_layer_backward(*args, parameter_grads=grads)
        torch.cuda.synchronize()
        named = dict(zip(("dqkv", "dz", "da", "db"), out))
        named.update(grads)
        return {k: v.cpu().numpy() for k, v in named.items()}

    chunked = once()
    assert capi.last_path() == capi.PATH_CHUNKED
    with capi.force_generic():
        sequential = once()
        assert capi.last_path() == capi.PATH_RECURRENCE
    for name in sequential:
        assert_close(chunked[name], sequential[name], 2e-4, name)


@pytest.mark.parametrize("rounding", [False, True])
def test_tensors_off_sixteen_bytes_give_the_same_bits(capi, rounding):
    """Every tensor one element past a 16-byte boundary: the passes with wide accesses
    (four-tap convolution forward and backward, output backward of rows of 128) take
    their narrow variants, which do the same arithmetic.  Two sequences, whose second
    starts at an odd multiple of the row's bytes."""
    import ctypes
    T, kh, vh, batch = 71, 2, 6, 2
    p = capi.delta_params(key_heads=kh, value_heads=vh, key_head_dim=128, value_head_dim=128,
                          conv_kernel_dim=4, round_to_bfloat16=rounding)
    c = make_case(T, kh, vh, 128, 128, 4, seed=9, batch=batch)
    bf = torch.bfloat16
    inputs = [dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
              dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"])]
    channels = (2 * kh + vh) * 128
    shapes = [inputs[0].shape, inputs[1].shape, inputs[2].shape, inputs[3].shape, (channels, 4), (vh,),
              (vh,), (128,)]  # gradients of the inputs, then of the parameters

    def once(shift):
        def moved(x):
            space = torch.zeros(x.numel() + 8, dtype=x.dtype, device="cuda")
            view = space[shift:shift + x.numel()].view(x.shape)
            view.copy_(x)
            assert view.data_ptr() % 16 == (shift * x.element_size()) % 16
            return view
        given = [moved(x) for x in inputs]
        out = [moved(torch.zeros(s, device="cuda")) for s in shapes]
        size = capi.lib().pluto_hip_gdn_layer_backward_workspace_bytes(ctypes.byref(p), T, 1)
        workspace = torch.empty(size, dtype=torch.uint8, device="cuda")
        capi.check(capi.lib().pluto_hip_gdn_layer_backward(
            capi.current_stream(), ctypes.byref(p), batch, T, *[capi.ptr(x) for x in given],
            *[capi.ptr(x) for x in out], capi.ptr(workspace), size))
        torch.cuda.synchronize()
        assert capi.last_path() == capi.PATH_CHUNKED
        return out

    for name, a, b in zip(("dqkv", "dz", "da", "db", "conv", "a_log", "dt_bias", "norm"), once(0), once(1)):
        assert torch.isfinite(a).all() and a.abs().max() > 0, name
        assert torch.equal(a, b), name


def test_rejects_bad_arguments(capi):
    import ctypes
    p = capi.delta_params(key_heads=1, value_heads=2, key_head_dim=4, value_head_dim=6,
                          conv_kernel_dim=3)
    lib = capi.lib()
    assert lib.pluto_hip_gdn_layer_backward_workspace_bytes(ctypes.byref(p), 0, 0) == 0
    assert lib.pluto_hip_gdn_layer_backward_workspace_bytes(ctypes.byref(p), 70000, 0) == 0
    size = lib.pluto_hip_gdn_layer_backward_workspace_bytes(ctypes.byref(p), 5, 1)
    assert size > 0
    x = torch.zeros(4096, device="cuda")
    ptrs = [capi.ptr(x)] * 13
    rc = lib.pluto_hip_gdn_layer_backward(capi.current_stream(), ctypes.byref(p), 1, 5, *ptrs, None,
                                          None, None, None, capi.ptr(x), 16)
    assert rc != 0  # workspace too small
    rc = lib.pluto_hip_gdn_layer_backward(capi.current_stream(), ctypes.byref(p), 1, 5, None,
                                          *ptrs[1:], None, None, None, None, capi.ptr(x), size)
    assert rc != 0  # null input


def test_values_near_the_top_of_the_range_stay_finite(capi):
    """A value between bf16's largest number and FP32's (2^128 - 2^120 to 2^128) rounds to an
    infinity in bf16: the matrix cores' pieces of it must still add up to it."""
    T, kh, vh = 200, 1, 2
    c = make_case(T, kh, vh, 128, 128, 4, seed=3)
    channel = 2 * kh * 128 + 5
    c["conv"][channel] = [0, 0, 0, 1.003]
    c["qkv"][0, :, channel] = 0
    c["qkv"][0, 100, channel] = 2.0 ** 128 - 2.0 ** 120  # 3.4e38 after the convolution
    c["b"][0, 100, 0] = 60  # and as the state's change
    # decaying slowly the state keeps the outputs so large that their norm's inverse is zero
    c["a_log"][:], c["dt_bias"][:] = 0, -3
    p = capi.delta_params(key_heads=kh, value_heads=vh, key_head_dim=128, value_head_dim=128, conv_kernel_dim=4,
                          round_to_bfloat16=False)
    bf = torch.bfloat16
    args = (p, dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
            dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"]))
    got = capi.gdn_layer_backward(*args)
    with capi.force_generic():
        want = capi.gdn_layer_backward(*args)
    torch.cuda.synchronize()
    for name, a, b in zip(("dqkv", "dz", "da", "db"), got, want):
        a, b = a.cpu().numpy(), b.cpu().numpy()
        assert np.isfinite(b).all() and np.isfinite(a).all(), name
        assert_close(a, b, 2e-4, name)  # the tolerance against the oracle


@pytest.mark.parametrize("T,kh,vh,taps", [(1, 1, 1, 4), (65, 3, 33, 4), (200, 2, 2, 3)])
def test_each_parameter_gradient_alone(capi, T, kh, vh, taps):
    """The chunked backward ends with one launch over whichever parameters have gradients:
    any of them alone has the bits it has with the others, none is a valid call, and what
    a head's time steps share, dt_bias, has the sum of their gradients (256 additions at
    most, each within 2^-24 of the magnitudes so far)."""
    c = make_case(T, kh, vh, 128, 128, taps, seed=T)
    p = capi.delta_params(kh, vh, 128, 128, taps)
    bf = torch.bfloat16
    args = [dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]), dev(c["a_log"]),
            dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"])]
    shapes = dict(conv_weight=c["conv"].shape, a_log=(vh,), dt_bias=(vh,), norm=(128,))
    zeros = lambda *names: {n: torch.zeros(shapes[n], device="cuda") for n in names}
    every = zeros(*shapes)
    activations = capi.gdn_layer_backward(p, *args, parameter_grads=every)
    for name in list(shapes) + [None]:
        one = zeros(*([name] if name else []))
        again = capi.gdn_layer_backward(p, *args, parameter_grads=one)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(activations, again)), name
        if name:
            assert torch.equal(one[name], every[name]), name
    da = activations[2].double()
    assert ((every["dt_bias"].double() - da.sum((0, 1))).abs() <= 256 * 2.0 ** -24 * da.abs().sum((0, 1)) + 1e-30).all()


@pytest.mark.parametrize("T,kh,vh", [(1, 2, 2), (64, 3, 3), (129, 2, 32), (130, 11, 33), (200, 16, 48)])
def test_rows_of_any_scale(capi, T, kh, vh):
    """Where activations are bf16 the chunked kernels multiply by a row of Q or K times a power
    of two and put the rest of its scale with the token's other factors: rows from 2^-100 to
    2^58 (whose squares are 2^127 at most), rows whose squares leave the range (scale zero)
    and rows of zeros, for one and two column tiles a workgroup, against the token-by-token
    kernels.  Tolerances as against the oracle: FP32 accuracy for all but the values behind
    a rounding that fell the other way, which are off by an operand's last bit."""
    c = make_case(T, kh, vh, 128, 128, 4, seed=T + kh)
    rng = np.random.default_rng(T)
    keys = 2 * kh * 128
    c["conv"][:keys] = [0, 0, 0, 1]
    exponent = rng.choice([-100, -60, -13, -1, 0, 1, 12, 40, 58, 90], (1, T, 2 * kh, 1))
    rows = c["qkv"][..., :keys].reshape(1, T, 2 * kh, 128)
    rows *= np.exp2(exponent).astype(np.float32)
    rows[rng.random((1, T, 2 * kh)) < 0.05] = 0
    c["qkv"][..., :keys] = rows.reshape(1, T, keys)
    p = capi.delta_params(kh, vh, 128, 128, 4)
    bf = torch.bfloat16
    args = (p, dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
            dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"]))
    got = capi.gdn_layer_backward(*args)
    assert capi.last_path() == capi.PATH_CHUNKED
    with capi.force_generic():
        want = capi.gdn_layer_backward(*args)
    torch.cuda.synchronize()
    for name, a, b in zip(("dqkv", "dz", "da", "db"), got, want):
        a, b = a.double().cpu().numpy(), b.double().cpu().numpy()
        assert np.isfinite(b).all() and np.isfinite(a).all(), name
        if name == "dqkv":  # a row's gradient is as small as the row is large
            a, b = (x.reshape(T, 2 * kh + vh, 128) for x in (a, b))
            scale = np.abs(b).max(-1, keepdims=True) + 1e-30
        else:
            scale = np.abs(b) + np.sqrt(np.mean(b ** 2))
        diff = np.abs(a - b)
        assert np.all(diff <= 2e-2 * scale), name
        assert np.mean(diff > 2e-4 * scale) <= 2e-2, name


def test_largest_bf16_values_stay_finite(capi):
    """The largest bf16 number among activations that are bf16, written to the state as it is:
    the pieces of what it becomes (U, the states, their gradients' products with K and Q)
    must not leave the range where the numbers do not.  Tolerances as for rows of any scale."""
    T, kh, vh = 200, 1, 2
    c = make_case(T, kh, vh, 128, 128, 4, seed=3)
    channel = 2 * kh * 128 + 5
    c["conv"][channel] = [0, 0, 0, 1]
    c["qkv"][0, :, channel] = 0
    c["qkv"][0, 100, channel] = 2.0 ** 128 - 2.0 ** 120
    c["b"][0, 100, 0] = 60
    c["a_log"][:], c["dt_bias"][:] = 0, -3
    p = capi.delta_params(kh, vh, 128, 128, 4)
    bf = torch.bfloat16
    args = (p, dev(c["qkv"], bf), dev(c["z"], bf), dev(c["a"], bf), dev(c["b"], bf), dev(c["conv"]),
            dev(c["a_log"]), dev(c["dt_bias"]), dev(c["norm"]), dev(c["dy"]))
    got = capi.gdn_layer_backward(*args)
    assert capi.last_path() == capi.PATH_CHUNKED
    with capi.force_generic():
        want = capi.gdn_layer_backward(*args)
    torch.cuda.synchronize()
    for name, a, b in zip(("dqkv", "dz", "da", "db"), got, want):
        a, b = a.double().cpu().numpy(), b.double().cpu().numpy()
        assert np.isfinite(b).all() and np.isfinite(a).all(), name
        scale = np.abs(b) + np.sqrt(np.mean(b ** 2))
        diff = np.abs(a - b)
        assert np.all(diff <= 2e-2 * scale), name
        assert np.mean(diff > 2e-4 * scale) <= 2e-2, name
