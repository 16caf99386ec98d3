"""What the layers of the Python mirror keep for the shapes they have seen, without a device: a stand-in context that counts what
is allocated and given back."""
import numpy as np

from mycaffe_amd.layers import Blob, CausalSelfAttentionLayer, InnerProductLayer, LayerNormLayer, TransposeLayer, _Kept


class Context:
    DTYPE = np.float32

    def __init__(self):
        self.live, self.made, self.next, self.calls = {}, 0, 1, []

    def _make(self, kind):
        self.made += 1
        self.next += 1
        self.live[self.next] = kind
        return self.next

    def _free(self, h):
        del self.live[h]          # a second free of a handle fails here

    def AllocMemory(self, src, hStream=0, bHalfSize=False):
        return self._make("memory")

    def CreateLayerNorm(self, *a):
        return self._make("layernorm")

    def CreateRope(self, *a):
        return self._make("rope")

    FreeMemory = FreeLayerNorm = FreeRope = _free

    def __getattr__(self, name):
        return lambda *a, **k: self.calls.append(name) or 0   # every other call is only noted


def test_kept_things_are_bounded_and_given_back():
    freed, kept = [], _Kept(lambda v: None)
    kept._free = freed.append
    for i in range(20):
        assert kept.get_or(i, lambda: i) == i and kept.get_or(i, lambda: "again") == i
    assert len(kept) == _Kept.MAX and freed == list(range(20 - _Kept.MAX))


def test_lengths_in_turn_build_nothing_anew_and_leak_nothing():
    for sdpa in (True, False):
        cuda = Context()
        layer = CausalSelfAttentionLayer(cuda, 2, 16, 64, True, sdpa, enable_rotary_positional_embedding=True)
        norm = LayerNormLayer(cuda)
        x, y = Blob(cuda), Blob(cuda)

        def use(B, T):
            layer._reshape(B, T)
            layer._mask(T)
            x.Reshape(B, T, 16)
            norm.Forward(x, y)

        x.Reshape(4, 64, 16), y.Reshape(4, 64, 16)
        for _ in range(2):
            for B, T in ((4, 40), (4, 64), (2, 50), (3, 40)):
                use(B, T)
        made, live = cuda.made, len(cuda.live)
        for _ in range(5):
            for B, T in ((4, 40), (4, 64), (2, 50), (3, 40)):
                use(B, T)
        assert cuda.made == made and len(cuda.live) == live, sdpa
        for T in range(1, 40):     # more lengths than are kept: what they need is given back
            use(1, T)
        assert len(cuda.live) <= live + 3 * _Kept.MAX, sdpa


def test_transposes_of_many_shapes_are_bounded():
    cuda = Context()
    layer, x, y = TransposeLayer(cuda, (0, 2, 1, 3)), Blob(cuda), Blob(cuda)
    x.Reshape(2, 50, 2, 8), y.Reshape(2, 2, 50, 8)
    for T in list(range(1, 50)) * 2:
        x.Reshape(2, T, 2, 8)
        layer.Forward(x, y)
    assert len(cuda.live) <= 2 + 4 * TransposeLayer.MAX_SHAPES + 1


def test_a_single_fp32_row_goes_through_gemv_whatever_its_layout():
    for half, M, want in ((False, 1, ["gemv", "axpy"]), (False, 2, ["LinearForward"]), (True, 1, ["LinearForward"])):
        cuda = Context()
        layer, x, y = InnerProductLayer(cuda, 16, half=half), Blob(cuda, (1, M, 8), half), Blob(cuda, half=half)
        layer.Setup(x)
        for forward in (lambda: layer.Forward(x, y), lambda: layer.ForwardHeads(x, y, 4)):
            cuda.calls.clear()
            forward()
            assert cuda.calls == want, (half, M, cuda.calls)
