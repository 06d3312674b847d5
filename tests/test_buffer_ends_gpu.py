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
