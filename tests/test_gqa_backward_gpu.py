"""GPU parity of the whole-sequence Qwen GQA backward
(QwenAttentionLayer::SequenceBackward, qwen_attention.cc:450-499) with the CPU
oracle, through the C ABI.  Shapes follow qwen_attention_test.cc:230-345 (tiny,
FP32 kernels, both rounding modes) and add head widths that take the
matrix-core kernels."""
import numpy as np
import pytest

from tests.util import assert_close, assert_close_bf16_gradient

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def capi():
    from pluto_amd import capi
    assert torch.cuda.is_available(), "these tests need the GPU"
    capi.lib()
    return capi


def values(count, phase, scale=0.8):
    i = np.arange(count, dtype=np.float32)
    return (np.float32(scale) * np.sin(np.float32(phase) + i * np.float32(0.29))).astype(np.float32)


def dev(x, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    return t.to(dtype) if dtype is not None else t


def run_case(capi, T, qh, kh, d, rot, rounding, seed=None, weight_grads=True):
    from oracle import pyoracle as po
    kw = dict(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=rot, capacity=max(T, 1),
              round_to_bfloat16=rounding)
    p, op = capi.attention_params(**kw), po.attention_params(**kw)
    if seed is None:
        qg = po.bf16_round(values(T * qh * 2 * d, .1)).reshape(T, qh, 2, d)
        k = po.bf16_round(values(T * kh * d, 1.2)).reshape(T, kh, d)
        v = po.bf16_round(values(T * kh * d, 2.3)).reshape(T, kh, d)
        qw, kw_ = values(d, .2), values(d, .4)
        dy = values(T * qh * d, .7).reshape(T, qh, d)
    else:
        rng = np.random.default_rng(seed)
        qg = po.bf16_round(rng.standard_normal((T, qh, 2, d)).astype(np.float32))
        k = po.bf16_round(rng.standard_normal((T, kh, d)).astype(np.float32))
        v = po.bf16_round(rng.standard_normal((T, kh, d)).astype(np.float32))
        qw = (0.1 * rng.standard_normal(d)).astype(np.float32)
        kw_ = (0.1 * rng.standard_normal(d)).astype(np.float32)
        dy = rng.standard_normal((T, qh, d)).astype(np.float32)
    want = po.gqa_sequence_backward(op, qg, k, v, qw, kw_, dy, weight_grads=weight_grads)
    dq_norm = torch.zeros(d, device="cuda") if weight_grads else None
    dk_norm = torch.zeros(d, device="cuda") if weight_grads else None
    args = (p, dev(qg, torch.bfloat16), dev(k, torch.bfloat16), dev(v, torch.bfloat16), dev(qw),
            dev(kw_), dev(dy))
    dqg, dk, dv = capi.gqa_prefill_backward(*args, dq_norm=dq_norm, dk_norm=dk_norm)
    torch.cuda.synchronize()
    got = dict(dqg=dqg.cpu().numpy(), dk=dk.cpu().numpy(), dv=dv.cpu().numpy())
    if weight_grads:
        got["dq_norm"], got["dk_norm"] = dq_norm.cpu().numpy(), dk_norm.cpu().numpy()
    return got, want, args, (dq_norm, dk_norm)


@pytest.mark.parametrize("rounding", [False, True])
@pytest.mark.parametrize("shape", [(3, 2, 1, 3, 2), (3, 2, 1, 4, 2), (33, 4, 2, 24, 8),
                                   (128, 6, 2, 32, 8)])
def test_fp32_kernels_match_oracle(capi, shape, rounding):
    T, qh, kh, d, rot = shape
    got, want, _, _ = run_case(capi, T, qh, kh, d, rot, rounding)
    for name in ("dqg", "dk", "dv", "dq_norm", "dk_norm"):
        what = "%s T%d d%d" % (name, T, d)
        if not rounding:
            # 3e-5 is the reference's own bound against finite differences
            # (qwen_attention_test.cc:287); sums over many rows carry FP32 rounding
            assert_close(got[name], want[name], 1e-4, what)
            continue
        # The gate gradient multiplies by bf16(core): where the FP32 and the
        # double-precision core straddle a rounding tie that factor differs by
        # one bf16 ulp.  At most 0.1% of the elements may use the one-ulp bound.
        expected = want[name].astype(np.float64)
        diff = np.abs(got[name] - expected)
        scale = np.abs(expected) + np.sqrt(np.mean(expected ** 2))
        print("%s: max-abs error %.3e" % (what, diff.max()))
        assert np.all(diff <= 8e-3 * scale), what
        assert np.mean(diff > 1e-4 * scale) <= 1e-3, what


@pytest.mark.parametrize("shape", [(33, 4, 2, 64, 16), (128, 6, 2, 128, 32), (200, 8, 1, 64, 64),
                                   (65, 4, 4, 128, 32)])
def test_matrix_core_kernels_match_oracle(capi, shape):
    T, qh, kh, d, rot = shape
    got, want, _, _ = run_case(capi, T, qh, kh, d, rot, True, seed=T + d)
    for name in ("dqg", "dk", "dv", "dq_norm", "dk_norm"):
        assert_close_bf16_gradient(got[name], want[name], "%s T%d d%d" % (name, T, d))


@pytest.mark.parametrize("shape", [(200, 8, 2, 64, 32), (333, 6, 2, 128, 64)])
def test_state_saved_by_forward_gives_the_recomputed_gradients(capi, shape):
    """pluto_hip_gqa_prefill can leave the attention output before the gate and
    the row statistics for the backward pass (the role of the state
    SequenceForward hands to SequenceBackward, qwen_attention.cc:445-447); the
    gradients must be those of the self-contained call."""
    T, qh, kh, d, rot = shape
    got, want, args, _ = run_case(capi, T, qh, kh, d, rot, True, seed=T)
    p, qg, k, v, qw, kw_, dy = args
    cache = capi.KvCache(T, kh, d)
    saved = capi.gqa_prefill_saved(p, T, cache)
    assert saved is not None and saved.numel() >= T * qh * (2 * d + 8)
    capi.gqa_prefill(p, qg, k, v, qw, kw_, cache, saved=saved)
    dq_norm, dk_norm = torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda")
    dqg, dk, dv = capi.gqa_prefill_backward(p, qg, k, v, qw, kw_, dy, dq_norm=dq_norm,
                                            dk_norm=dk_norm, saved=saved)
    torch.cuda.synchronize()
    with_saved = dict(dqg=dqg, dk=dk, dv=dv, dq_norm=dq_norm, dk_norm=dk_norm)
    for name, value in with_saved.items():
        # same kernels, same operands: the forward pass of the two calls differs
        # only in where K and V are read from
        np.testing.assert_allclose(value.cpu().numpy(), got[name], rtol=1e-5, atol=1e-6,
                                   err_msg=name)
        assert_close_bf16_gradient(value.cpu().numpy(), want[name], "%s T%d d%d" % (name, T, d))


@pytest.mark.parametrize("T,qh,kh,d,rot", [(1, 2, 1, 256, 64), (31, 4, 2, 256, 64), (65, 6, 2, 256, 64),
                                           (130, 6, 1, 256, 128), (97, 4, 2, 128, 32), (97, 4, 2, 64, 32)])
def test_saved_block_holds_what_both_passes_need(capi, T, qh, kh, d, rot):
    """The block is filled where it starts (also off a multiple of 256 bytes), whatever the
    output's alignment, and the backward makes of it, bit for bit, what it makes of the
    inputs.  Head width 256: the forward that fills it keeps its softmax weights in FP32, so
    its output is within the rounding of bf16 weights of the other forward's (2^-9 a
    weight, sums of weighted values: 1e-2 of the norm is generous) and its cache the same."""
    import ctypes
    got, _, args, _ = run_case(capi, T, qh, kh, d, rot, True, seed=T + d)
    p, qg, k, v, qw, kw_, dy = args
    plain_cache = capi.KvCache(T, kh, d)
    plain, plain_lse = capi.gqa_prefill(p, qg, k, v, qw, kw_, plain_cache, want_lse=True)
    size = capi.lib().pluto_hip_gqa_prefill_saved_bytes(ctypes.byref(p), T, capi.BF16)
    assert size > 0
    for shift in (0, 2 if d == 256 else 0):
        block = torch.full((size + 64,), 0x7f, dtype=torch.uint8, device="cuda")[48:48 + size]
        space = torch.zeros(T * qh * d + 8, dtype=torch.bfloat16, device="cuda")
        out = space[shift:shift + T * qh * d].view(T, qh, d)
        cache = capi.KvCache(T, kh, d)
        made, lse = capi.gqa_prefill(p, qg, k, v, qw, kw_, cache, saved=block, out=out, want_lse=True)
        torch.cuda.synchronize()
        assert torch.equal(cache.keys, plain_cache.keys) and torch.equal(cache.values, plain_cache.values)
        if d == 256:
            assert capi.last_path() == capi.PATH_MATRIX_F32
            assert (made.float() - plain.float()).norm() <= 1e-2 * plain.float().norm()
            # the bf16 kernel adds up rounded weights: each, and so the sum, is off by at
            # most 2^-9 of itself, and the logarithm by as much
            assert (lse - plain_lse).abs().max() <= 2.0 ** -9 + 1e-5 * (1 + plain_lse.abs().max())
        else:
            assert torch.equal(made, plain) and torch.equal(lse, plain_lse)
        dq_norm, dk_norm = torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda")
        grads = capi.gqa_prefill_backward(p, qg, k, v, qw, kw_, dy, dq_norm=dq_norm, dk_norm=dk_norm, saved=block)
        torch.cuda.synchronize()
        for name, value in zip(("dqg", "dk", "dv", "dq_norm", "dk_norm"), grads + (dq_norm, dk_norm)):
            assert np.array_equal(value.cpu().numpy(), got[name]), name


@pytest.mark.parametrize("T,qh,kh", [(1, 2, 1), (32, 3, 1), (33, 6, 2), (64, 4, 2), (65, 6, 1), (129, 2, 2), (300, 5, 1),
                                     (513, 3, 3)])
def test_gradients_in_one_launch_are_those_of_two(capi, T, qh, kh):
    """Head width 256: the workgroups of query and key tiles in one launch, longest first,
    with tiles of either side that are ragged or the only one.  Bit for bit what launches of
    their own make."""
    d = 256
    p = capi.attention_params(qh, kh, d, 64, capacity=T)
    gen = torch.Generator(device="cuda").manual_seed(T)

    def values(*shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=gen, device="cuda").to(dtype)
    args = (p, values(T, qh, 2, d), values(T, kh, d), values(T, kh, d), values(d, dtype=torch.float32),
            values(d, dtype=torch.float32), values(T, qh, d, dtype=torch.float32))
    together = capi.gqa_prefill_backward(*args)
    with capi.only_kernels(capi.QUERY_KERNEL | capi.AUXILIARY_KERNELS):
        queries = capi.gqa_prefill_backward(*args)
    with capi.only_kernels(capi.MAIN_KERNEL | capi.AUXILIARY_KERNELS):
        keys = capi.gqa_prefill_backward(*args)
    torch.cuda.synchronize()
    assert all(torch.isfinite(g).all() for g in together)
    assert torch.equal(together[0], queries[0])
    assert torch.equal(together[1], keys[1]) and torch.equal(together[2], keys[2])


def test_long_sequence_with_saved_state_matches_oracle(capi):
    """T=1024, one kv group of six 128-wide heads (the grouping of the benchmarked
    shape): eight query tiles, so the unpaired heaviest-first grid, with the block
    the forward pass saves.  Every gradient against the oracle."""
    T, qh, kh, d, rot = 1024, 6, 1, 128, 32
    got, want, args, _ = run_case(capi, T, qh, kh, d, rot, True, seed=77)
    assert capi.last_path() == capi.PATH_FLASH
    p, qg, k, v, qw, kw_, dy = args
    cache = capi.KvCache(T, kh, d)
    saved = capi.gqa_prefill_saved(p, T, cache)
    capi.gqa_prefill(p, qg, k, v, qw, kw_, cache, saved=saved)
    dq_norm, dk_norm = torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda")
    dqg, dk, dv = capi.gqa_prefill_backward(p, qg, k, v, qw, kw_, dy, dq_norm=dq_norm,
                                            dk_norm=dk_norm, saved=saved)
    torch.cuda.synchronize()
    assert capi.last_path() == capi.PATH_FLASH
    with_saved = dict(dqg=dqg, dk=dk, dv=dv, dq_norm=dq_norm, dk_norm=dk_norm)
    for name, value in with_saved.items():
        assert_close_bf16_gradient(got[name], want[name], "%s T%d self-contained" % (name, T))
        assert_close_bf16_gradient(value.cpu().numpy(), want[name], "%s T%d saved" % (name, T))


def test_benchmarked_shape_against_fp32_kernels(capi):
    """The shape bench.py times (T=8192, 24 query / 4 kv heads of 128, saved block):
    the matrix-core kernels against the any-shape FP32-arithmetic kernels of the same
    library.  The CPU oracle would need an hour for this length; it covers the same
    kernels at T=1024 above."""
    T, qh, kh, d, rot = 8192, 24, 4, 128, 32
    p = capi.attention_params(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=rot,
                              capacity=T, round_to_bfloat16=True)
    gen = torch.Generator(device="cuda").manual_seed(2)
    bf = torch.bfloat16
    qg = (0.5 * torch.randn((T, qh, 2, d), generator=gen, device="cuda")).to(bf)
    k = (0.5 * torch.randn((T, kh, d), generator=gen, device="cuda")).to(bf)
    v = (0.5 * torch.randn((T, kh, d), generator=gen, device="cuda")).to(bf)
    dy = torch.randn((T, qh, d), generator=gen, device="cuda")
    qw, kw_ = dev(values(d, 0.2, 0.3)), dev(values(d, 0.8, 0.4))

    def once(saved):
        dq_norm, dk_norm = torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda")
        dqg, dk, dv = capi.gqa_prefill_backward(p, qg, k, v, qw, kw_, dy, dq_norm=dq_norm,
                                                dk_norm=dk_norm, saved=saved)
        torch.cuda.synchronize()
        return dict(dqg=dqg, dk=dk, dv=dv, dq_norm=dq_norm, dk_norm=dk_norm)

    cache = capi.KvCache(T, kh, d)
    saved = capi.gqa_prefill_saved(p, T, cache)
    capi.gqa_prefill(p, qg, k, v, qw, kw_, cache, saved=saved)
    fast = once(saved)
    assert capi.last_path() == capi.PATH_FLASH
    with capi.force_generic():
        slow = once(None)
        assert capi.last_path() == capi.PATH_GENERIC
    for name in fast:
        # (fifty million elements: the tail of the per-element error reaches further
        # than in the small cases: the farthest observed sits at 19.1 times the
        # per-element bound; the max-norm bound still holds for every element)
        assert_close_bf16_gradient(fast[name].cpu().numpy(), slow[name].cpu().numpy(),
                                   "%s T%d vs fp32-arithmetic kernels" % (name, T), far=20.0)


@pytest.mark.parametrize("T,qh,kh,d,rot", [(97, 4, 2, 64, 32), (130, 6, 2, 128, 32)])
def test_saved_block_is_the_output_and_its_statistics(capi, T, qh, kh, d, rot):
    """At head width 64 and 128 a block is held for every layer between the passes: the
    attention output in bf16 and two floats a row and head, each rounded up to 256 bytes."""
    import ctypes
    p = capi.attention_params(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=rot, capacity=T,
                              round_to_bfloat16=True)
    size = capi.lib().pluto_hip_gqa_prefill_saved_bytes(ctypes.byref(p), T, capi.BF16)
    assert T * qh * (2 * d + 8) <= size <= T * qh * (2 * d + 8) + 3 * 255


@pytest.mark.parametrize("T,qh,kh,d,rot", [(97, 4, 2, 64, 32), (130, 6, 2, 128, 32), (130, 6, 2, 256, 64)])
def test_saved_block_can_be_moved(capi, T, qh, kh, d, rot):
    """A block that is copied to an address with another remainder (kept on the host between
    the passes, packed behind other tensors) is read as it was written."""
    import ctypes
    got, _, args, _ = run_case(capi, T, qh, kh, d, rot, True, seed=T + d)
    p, qg, k, v, qw, kw_, dy = args
    size = capi.lib().pluto_hip_gqa_prefill_saved_bytes(ctypes.byref(p), T, capi.BF16)
    for filled_at, read_at in ((0, 16), (16, 0), (48, 208), (240, 4), (12, 128), (0, 100)):
        space = torch.full((size + 512,), 0x7f, dtype=torch.uint8, device="cuda")
        assert space.data_ptr() % 256 == 0
        block = space[filled_at:filled_at + size]
        capi.gqa_prefill(p, qg, k, v, qw, kw_, capi.KvCache(T, kh, d), saved=block)
        kept = block.cpu()
        space.fill_(0x7f)
        block = space[read_at:read_at + size]
        block.copy_(kept)
        dq_norm, dk_norm = torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda")
        grads = capi.gqa_prefill_backward(p, qg, k, v, qw, kw_, dy, dq_norm=dq_norm, dk_norm=dk_norm, saved=block)
        torch.cuda.synchronize()
        for name, value in zip(("dqg", "dk", "dv", "dq_norm", "dk_norm"), grads + (dq_norm, dk_norm)):
            assert np.array_equal(value.cpu().numpy(), got[name]), (name, filled_at, read_at)


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("T", [33, 130])
def test_saved_forward_with_non_finite_values(capi, T, bad):
    """Head width 256: the forward that fills the block gives the numbers (to the 2^-9 of the
    other's bf16 weights), infinities and NaNs that it gives without the block, and the
    block's output before the gate the same."""
    qh, kh, d = 4, 2, 256
    p = capi.attention_params(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=64, capacity=T,
                              round_to_bfloat16=True)
    gen = torch.Generator(device="cuda").manual_seed(T)
    qg = torch.randn((T, qh, 2, d), generator=gen, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn((T, kh, d), generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    v[T // 2, 1, 5] = bad
    w = torch.zeros(d, device="cuda")
    cache = capi.KvCache(T, kh, d)
    saved = capi.gqa_prefill_saved(p, T, cache)
    got = capi.gqa_prefill(p, qg, k, v, w, w, cache, saved=saved)
    assert capi.last_path() == capi.PATH_MATRIX_F32
    want = capi.gqa_prefill(p, qg, k, v, w, w, cache)
    torch.cuda.synchronize()
    core = saved[:T * qh * d * 4].view(torch.float32).view(T, qh, d)
    a, b = got.double(), want.double()
    assert torch.equal(a.isnan(), b.isnan())
    assert torch.equal(torch.where(a.isinf(), a, 0), torch.where(b.isinf(), b, 0))
    assert torch.equal(core.isnan(), b.isnan()) and torch.equal(core.isinf(), b.isinf())
    finite = b.isfinite()
    a, b = torch.where(finite, a, 0), torch.where(finite, b, 0)
    assert ((a - b).norm(dim=-1) <= 1e-2 * b.norm(dim=-1)).all()


def test_saved_block_off_a_word_is_refused_at_head_width_256(capi):
    T, qh, kh, d = 33, 2, 1, 256
    p = capi.attention_params(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=64, capacity=T,
                              round_to_bfloat16=True)
    cache = capi.KvCache(T, kh, d)
    block = torch.zeros(capi.gqa_prefill_saved(p, T, cache).numel() + 2, dtype=torch.uint8, device="cuda")[2:]
    qg = torch.zeros((T, qh, 2, d), dtype=torch.bfloat16, device="cuda")
    k = torch.zeros((T, kh, d), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(d, device="cuda")
    with pytest.raises(capi.PlutoHipError) as info:
        capi.gqa_prefill(p, qg, k, k, w, w, cache, saved=block)
    assert info.value.code == capi.EINVAL
    with pytest.raises(capi.PlutoHipError) as info:
        capi.gqa_prefill_backward(p, qg, k, k, w, w, torch.zeros((T, qh, d), device="cuda"), saved=block)
    assert info.value.code == capi.EINVAL


def test_saved_state_is_refused_where_none_is_kept(capi):
    T, qh, kh, d, rot = 16, 2, 1, 32, 8
    kw = dict(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=rot, capacity=T,
              round_to_bfloat16=True)
    p = capi.attention_params(**kw)
    cache = capi.KvCache(T, kh, d)
    assert capi.gqa_prefill_saved(p, T, cache) is None  # head width without matrix-core backward
    lib = capi.lib()
    import ctypes
    fp32 = capi.attention_params(**dict(kw, head_dim=64, rotary_dim=16, round_to_bfloat16=False))
    assert lib.pluto_hip_gqa_prefill_saved_bytes(ctypes.byref(fp32), T, capi.BF16) == 0
    wide = capi.attention_params(**dict(kw, head_dim=64, rotary_dim=16))
    assert lib.pluto_hip_gqa_prefill_saved_bytes(ctypes.byref(wide), T, capi.F32) == 0
    assert lib.pluto_hip_gqa_prefill_saved_bytes(ctypes.byref(wide), T, capi.BF16) > 0
    # a block offered where none can be filled is an error, not silently ignored
    qg = torch.zeros((T, qh, 2, d), dtype=torch.bfloat16, device="cuda")
    k = torch.zeros((T, kh, d), dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(d, device="cuda")
    bogus = torch.empty(1 << 16, dtype=torch.uint8, device="cuda")
    with pytest.raises(capi.PlutoHipError):
        capi.gqa_prefill(p, qg, k, k, w, w, cache, saved=bogus)
    dy = torch.zeros((T, qh, d), device="cuda")
    with pytest.raises(capi.PlutoHipError):
        capi.gqa_prefill_backward(p, qg, k, k, w, w, dy, saved=bogus)


def test_weight_gradients_accumulate_and_are_optional(capi):
    T, qh, kh, d, rot = 5, 2, 1, 8, 4
    got, want, args, (dq_norm, dk_norm) = run_case(capi, T, qh, kh, d, rot, True)
    again = capi.gqa_prefill_backward(*args, dq_norm=dq_norm, dk_norm=dk_norm)
    torch.cuda.synchronize()
    # shared norm gradients accumulate across calls (qwen_attention_test.cc:291-300)
    np.testing.assert_allclose(dq_norm.cpu().numpy(), 2 * got["dq_norm"], rtol=1e-6, atol=1e-7)
    np.testing.assert_allclose(dk_norm.cpu().numpy(), 2 * got["dk_norm"], rtol=1e-6, atol=1e-7)
    for a, name in zip(again, ("dqg", "dk", "dv")):
        np.testing.assert_array_equal(a.cpu().numpy(), got[name])  # repeatable, bit for bit
    frozen, _, _, _ = run_case(capi, T, qh, kh, d, rot, True, weight_grads=False)
    for name in ("dqg", "dk", "dv"):
        np.testing.assert_array_equal(frozen[name], got[name])


def test_later_rows_reach_earlier_keys_and_values(capi):
    # qwen_attention_test.cc:303-345: a gradient on the last row only still
    # reaches the first token's key and value
    from oracle import pyoracle as po
    T, qh, kh, d, rot = 3, 2, 1, 4, 2
    p = capi.attention_params(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=rot,
                              capacity=T, round_to_bfloat16=True)
    qg = po.bf16_round(values(T * qh * 2 * d, .1)).reshape(T, qh, 2, d)
    k = po.bf16_round(values(T * kh * d, 1.2)).reshape(T, kh, d)
    v = po.bf16_round(values(T * kh * d, 2.3)).reshape(T, kh, d)
    dy = np.zeros((T, qh, d), np.float32)
    dy[2] = 0.5
    _, dk, dv = capi.gqa_prefill_backward(p, dev(qg, torch.bfloat16), dev(k, torch.bfloat16),
                                          dev(v, torch.bfloat16), dev(values(d, .2)),
                                          dev(values(d, .4)), dev(dy))
    assert dk[0].abs().sum().item() > 1e-5 and dv[0].abs().sum().item() > 1e-5


def test_rejects_bad_arguments_before_touching_outputs(capi):
    p = capi.attention_params(query_heads=2, key_value_heads=1, head_dim=4, rotary_dim=2,
                              capacity=4, round_to_bfloat16=True)
    import ctypes
    lib = capi.lib()
    assert lib.pluto_hip_gqa_prefill_backward_workspace_bytes(ctypes.byref(p), 0, 0, 0) == 0
    size = lib.pluto_hip_gqa_prefill_backward_workspace_bytes(ctypes.byref(p), 3, 1, 1)
    assert size > 0
    x = torch.zeros(1024, device="cuda")
    rc = lib.pluto_hip_gqa_prefill_backward(capi.current_stream(), ctypes.byref(p), 3, capi.ptr(x),
                                            capi.ptr(x), capi.ptr(x), capi.ptr(x), capi.ptr(x),
                                            capi.ptr(x), None, capi.ptr(x), capi.ptr(x), capi.ptr(x),
                                            None, None, capi.ptr(x), 16)
    assert rc == capi.EWORKSPACE if hasattr(capi, "EWORKSPACE") else rc != 0
    rc = lib.pluto_hip_gqa_prefill_backward(capi.current_stream(), ctypes.byref(p), 3, None,
                                            capi.ptr(x), capi.ptr(x), capi.ptr(x), capi.ptr(x),
                                            capi.ptr(x), None, capi.ptr(x), capi.ptr(x), capi.ptr(x),
                                            None, None, capi.ptr(x), size)
    assert rc != 0


@pytest.mark.parametrize("T,qh,kh,rot", [(1, 2, 1, 64), (31, 2, 2, 64), (33, 6, 2, 64), (128, 4, 1, 32),
                                         (161, 3, 1, 256), (300, 6, 1, 64)])
def test_split_operand_kernels_keep_fp32_accuracy(capi, T, qh, kh, rot):
    """Head width 256 multiplies FP32 factors as three bf16 pieces each: every
    gradient must be that of the element-at-a-time FP32 kernels to FP32 accuracy (a
    bf16 operand anywhere would show as 1e-3).  Ragged tiles on both sides."""
    d = 256
    got, _, args, _ = run_case(capi, T, qh, kh, d, rot, True, seed=T + rot)
    assert capi.last_path() == capi.PATH_MATRIX_F32
    p, qg, k, v, qw, kw_, dy = args
    dq_norm, dk_norm = torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda")
    with capi.force_generic():
        dqg, dk, dv = capi.gqa_prefill_backward(p, qg, k, v, qw, kw_, dy, dq_norm=dq_norm,
                                                dk_norm=dk_norm)
    want = dict(dqg=dqg, dk=dk, dv=dv, dq_norm=dq_norm, dk_norm=dk_norm)
    for name, value in want.items():
        w = value.double().cpu().numpy()
        # (one token has no score gradient: what is left of dk is rounding)
        error = np.linalg.norm(got[name] - w) / max(np.linalg.norm(w), 0.1 * float(dv.norm()))
        print("%s T%d: %.2e" % (name, T, error))
        assert error <= 2e-5, name


@pytest.mark.parametrize("T,qh,kh,d,rot,with_saved", [(70, 4, 2, 64, 32, True), (70, 4, 2, 64, 32, False),
                                                      (131, 6, 2, 128, 32, True), (65, 6, 2, 256, 64, False)])
def test_tensors_off_sixteen_bytes(capi, T, qh, kh, d, rot, with_saved):
    """The gate's pass and the norm's have wide accesses where every tensor allows it.
    With dy alone moved by one element the gate's narrow variant does the same arithmetic,
    bit for bit; with the gradients moved too the norm's any-width kernel adds up in another
    order (FP32 rounding); with the bf16 inputs moved the preparation's does as well, and an
    element of q or k next to a rounding tie may fall to its other side."""
    import ctypes
    p = capi.attention_params(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=rot, capacity=T,
                              round_to_bfloat16=True)
    gen = torch.Generator(device="cuda").manual_seed(T + d)
    bf = torch.bfloat16
    def normal(*shape):
        return torch.randn(shape, generator=gen, device="cuda")
    qg, k, v = (0.5 * normal(T, qh, 2, d)).to(bf), (0.5 * normal(T, kh, d)).to(bf), (0.5 * normal(T, kh, d)).to(bf)
    q_norm, k_norm, dy = 0.1 * normal(d), 0.1 * normal(d), normal(T, qh, d)
    saved = None
    if with_saved:
        cache = capi.KvCache(T, kh, d)
        saved = capi.gqa_prefill_saved(p, T, cache)
        capi.gqa_prefill(p, qg, k, v, q_norm, k_norm, cache, saved=saved)

    def once(inputs, upstream, outputs):
        def moved(x, shift):
            space = torch.zeros(x.numel() + 8, dtype=x.dtype, device="cuda")
            view = space[shift:shift + x.numel()].view(x.shape)
            view.copy_(x)
            return view
        given = [moved(x, inputs) for x in (qg, k, v)] + [q_norm, k_norm, moved(dy, upstream)]
        out = [moved(torch.zeros(s, device="cuda"), outputs)
               for s in ((T, qh, 2, d), (T, kh, d), (T, kh, d), (d,), (d,))]
        size = capi.lib().pluto_hip_gqa_prefill_backward_workspace_bytes(ctypes.byref(p), T, 1, 1)
        workspace = torch.empty(size, dtype=torch.uint8, device="cuda")
        capi.check(capi.lib().pluto_hip_gqa_prefill_backward(
            capi.current_stream(), ctypes.byref(p), T, *[capi.ptr(x) for x in given], capi.ptr(saved),
            *[capi.ptr(x) for x in out], capi.ptr(workspace), size))
        torch.cuda.synchronize()
        assert capi.last_path() == (capi.PATH_MATRIX_F32 if d == 256 else capi.PATH_FLASH)
        return out

    names = ("dqg", "dk", "dv", "dq_norm", "dk_norm")
    want = once(0, 0, 0)
    for name, a, b in zip(names, want, once(0, 1, 0)):
        assert torch.isfinite(a).all() and a.abs().max() > 0, name
        assert torch.equal(a, b), name
    for name, a, b in zip(names, want, once(0, 1, 1)):
        # sums of d and of T * heads FP32 terms in two orders: about sqrt(terms) 2^-24 each
        assert (a - b).norm() <= 1e-5 * a.norm(), name
    for name, a, b in zip(names, want, once(1, 1, 1)):
        # a bf16 ulp (2^-8) in one element of a thousand: 2^-8 sqrt(1e-3) of the norm
        assert (a - b).norm() <= 2.0 ** -8 * 1e-3 ** 0.5 * a.norm(), name


@pytest.mark.parametrize("T,d", [(1, 128), (9, 256), (1001, 256), (1100, 64), (2750, 128), (5501, 64)])
def test_gate_gradients_of_every_row(capi, T, d):
    """24 heads of lengths whose gate gradients go 8 to 64 rows a workgroup, the last one
    not full.  The gradient is dy core s (1 - s) and the forward's output the product of
    the rounded core and the rounded s, rounded: apart by two roundings to eight bits."""
    gen = torch.Generator(device="cuda").manual_seed(T)
    normal = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    qh, kh = 24, 4
    p = capi.attention_params(query_heads=qh, key_value_heads=kh, head_dim=d, rotary_dim=d // 4, capacity=T,
                              round_to_bfloat16=True)
    qg = normal(T, qh, 2, d).to(torch.bfloat16)
    k, v = normal(T, kh, d).to(torch.bfloat16), normal(T, kh, d).to(torch.bfloat16)
    qw, kw_, dy = 0.1 * normal(d), 0.1 * normal(d), normal(T, qh, d)
    cache = capi.KvCache(T, kh, d)
    saved = capi.gqa_prefill_saved(p, T, cache)
    out = capi.gqa_prefill(p, qg, k, v, qw, kw_, cache, saved=saved)
    dqg = capi.gqa_prefill_backward(p, qg, k, v, qw, kw_, dy, saved=saved)[0]
    torch.cuda.synchronize()
    want = dy.double() * out.double() * (1 - torch.sigmoid(qg[:, :, 1].double()))
    error = (dqg[:, :, 1].double() - want).abs()
    assert (error <= 2.0 ** -6.9 * want.abs() + 1e-6).all(), error.max().item()
