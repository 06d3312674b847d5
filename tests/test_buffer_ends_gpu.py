"""Sequences that fill no whole tile, with nothing but guard bytes around every buffer of the
call: what lies there is neither written nor part of a result."""
import pytest

from tests.util import GuardedBuffers

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def capi():
    from pluto_amd import capi
    assert torch.cuda.is_available(), "these tests need the GPU"
    capi.lib()
    return capi


def check(capi, monkeypatch, what, inputs, call):
    """call(inputs) -> tensors, with ordinary buffers and with guarded ones: the same bits."""
    address = capi.ptr

    def of_the_gpu(tensor):
        assert tensor is None or tensor.is_cuda
        return address(tensor)

    monkeypatch.setattr(capi, "ptr", of_the_gpu)
    plain = [t.clone() for t in call([t.clone() for t in inputs])]
    guards = GuardedBuffers(torch)
    monkeypatch.setattr(capi, "torch", guards)
    print(what, flush=True)
    guarded = call([guards.place(t) for t in inputs])
    torch.cuda.synchronize()
    guards.assert_intact(what)
    for i, (a, b) in enumerate(zip(plain, guarded)):
        assert bool(torch.isfinite(a.float()).all()), "%s: output %d" % (what, i)
        assert torch.equal(a, b), "%s: output %d differs" % (what, i)


def random(seed, *shape, dtype=torch.bfloat16, scale=1.0):
    generator = torch.Generator().manual_seed(seed)
    return (scale * torch.randn(shape, generator=generator)).to(dtype).cuda()


# the last row of a sequence at every place of a 32-row block that matters, one and two
# sequences: behind the last one lies the end of every buffer
@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("T", [1, 33, 61, 129, 500])
def test_attention_of_64_channels(capi, monkeypatch, T, B):
    H, E = 2, 128

    def call(inputs):
        qkv, d_out = inputs
        out, maxima, normalizers = capi.mha_forward(qkv, T, H)
        return out, maxima, normalizers, capi.mha_backward(qkv, out, d_out, maxima, normalizers, T, H)

    check(capi, monkeypatch, "T %d B %d" % (T, B),
          [random(T, B * T, 3 * E), random(T + 1, B * T, E, dtype=torch.float32)], call)


# the four-wave forward kernel's queries and the wide backward kernels
@pytest.mark.parametrize("T", [1, 33, 500])
def test_attention_of_128_channels(capi, monkeypatch, T):
    H, E, B = 3, 384, 2

    def call(inputs):
        qkv, d_out = inputs
        out, maxima, normalizers = capi.mha_forward(qkv, T, H)
        return out, maxima, normalizers, capi.mha_backward(qkv, out, d_out, maxima, normalizers, T, H)

    check(capi, monkeypatch, "T %d" % T,
          [random(T, B * T, 3 * E), random(T + 1, B * T, E, dtype=torch.float32)], call)


# 256 channels: tiles of 64 queries and of 128 keys, whose workgroups share a launch, and what
# prepares and follows them; 64 and 128: the kernels above with grouped queries.  The
# preparation has a row a workgroup.
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("T", [1, 33, 65, 129, 190])
def test_grouped_query_training(capi, monkeypatch, T, d):
    qh, kh = 6, 2
    p = capi.attention_params(qh, kh, d, 32, capacity=T)

    def call(inputs):
        qg, k, v, q_norm, k_norm, dy = inputs
        cache = capi.KvCache(T, kh, d)
        saved = capi.gqa_prefill_saved(p, T, cache)
        out = capi.gqa_prefill(p, qg, k, v, q_norm, k_norm, cache, saved=saved)
        norms = [capi.torch.empty_like(w).zero_() for w in (q_norm, k_norm)]
        grads = capi.gqa_prefill_backward(p, qg, k, v, q_norm, k_norm, dy, *norms, saved=saved)
        return (out, cache.keys, cache.values) + tuple(grads) + tuple(norms)

    check(capi, monkeypatch, "T %d d %d" % (T, d),
          [random(T, T, qh, 2, d, scale=0.5), random(T + 1, T, kh, d), random(T + 2, T, kh, d),
           random(T + 3, d, dtype=torch.float32, scale=0.3), random(T + 4, d, dtype=torch.float32, scale=0.3),
           random(T + 5, T, qh, d, dtype=torch.float32)], call)


# Chunks of 64 tokens.  One tile a workgroup of the sequential backward kernels, with a wave
# that only touches what the others read later, and two (36 value heads); groups of one, two
# and three value heads in the forward's preparation.
@pytest.mark.parametrize("kh,vh", [(2, 2), (1, 2), (1, 3), (12, 36)])
@pytest.mark.parametrize("T", [1, 3, 63, 65, 130])
def test_delta_net_training(capi, monkeypatch, T, kh, vh):
    d, channels = 128, (2 * kh + vh) * 128
    p = capi.delta_params(kh, vh, d, d)
    names = ("conv_weight", "a_log", "dt_bias", "norm")

    def call(inputs):
        qkv, z, a, b, dy = inputs[:5]
        weights = dict(zip(names, inputs[5:]))
        state = capi.torch.empty((1, vh, d, d), dtype=torch.float32, device="cuda").zero_()
        out = capi.gdn_layer_forward(p, qkv, z, a, b, state=state, **weights)
        grads = {n: capi.torch.empty_like(w).zero_() for n, w in weights.items()}
        inputs_grads = capi.gdn_layer_backward(p, qkv, z, a, b, dy=dy, parameter_grads=grads, **weights)
        return (out, state) + tuple(inputs_grads) + tuple(grads.values())

    f32 = dict(dtype=torch.float32)
    check(capi, monkeypatch, "T %d heads %d %d" % (T, kh, vh),
          [random(T, 1, T, channels), random(T + 1, 1, T, vh * d), random(T + 2, 1, T, vh), random(T + 3, 1, T, vh),
           random(T + 4, 1, T, vh * d, **f32), random(T + 5, channels, 4, scale=0.5, **f32), random(T + 6, vh, scale=0.5, **f32),
           random(T + 7, vh, **f32), 1 + random(T + 8, d, scale=0.1, **f32)], call)


# The decode step, whose workgroups walk the heads of several sequences.
@pytest.mark.parametrize("B", [1, 11])
def test_delta_net_step(capi, monkeypatch, B):
    kh, vh, d = 2, 6, 128
    channels = (2 * kh + vh) * d
    p = capi.delta_params(kh, vh, d, d)
    f32 = dict(dtype=torch.float32)
    conv, state = random(1, B, channels, 4, **f32), random(2, B, vh, d, d, scale=0.1, **f32)

    def call(inputs):
        step = capi.DeltaNetStep(p, batch=B)
        step.conv, step.state = inputs[:2]
        return step.step(*inputs[2:]), step.conv, step.state

    check(capi, monkeypatch, "B %d" % B,
          [conv, state, random(3, B, channels), random(4, B, vh * d), random(5, B, vh), random(6, B, vh),
           random(7, channels, 4, scale=0.5, **f32), random(8, vh, scale=0.5, **f32), random(9, vh, **f32),
           1 + random(10, d, scale=0.1, **f32)], call)
