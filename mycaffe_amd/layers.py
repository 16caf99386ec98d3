"""Host-side mirrors of the MyCaffe layers that call the attention hot path.

These follow the C# ``forward`` and ``backward`` methods (cited per class).  Where this library has one call for several of
the reference's - inner product with its bias, projection into heads, gradients of both, a norm with the residual next to it -
the layers make the one call; the reference's own sequences run against the library from the C++ host program and the tests of
the single ids.  Dropout layers are the identity (inference, or training with ratio 0).  ``Backward`` is mirrored for the GPT block
(InnerProduct, Transpose, LayerNorm, activations, CausalSelfAttention with the fused attention handle, TransformerBlock).
"""
import math

import numpy as np

from .cudadnn import DIR, SOFTMAX_ALGORITHM, SOFTMAX_MODE


class Blob:
    """Shape + device handle, the part of MyCaffe/common/Blob.cs the layers use."""

    def __init__(self, cuda, shape=None, half=False):
        self.cuda = cuda
        self.half = half
        self.shape_ = []
        self.gpu_data = 0
        self._capacity = 0
        self._gpu_diff = 0
        self._diff_capacity = 0
        if shape is not None:
            self.Reshape(*shape)

    def Reshape(self, *shape):
        if len(shape) == 1 and isinstance(shape[0], (list, tuple)):
            shape = shape[0]
        shape = list(shape)
        if shape == self.shape_ and self.gpu_data:
            return
        self.shape_ = [int(s) for s in shape]
        n = self.count()
        if n > self._capacity:
            if self.gpu_data:
                self.cuda.FreeMemory(self.gpu_data)
            self.gpu_data = self.cuda.AllocMemory(n, bHalfSize=self.half)
            self._capacity = n

    def ReshapeLike(self, other):
        self.Reshape(*other.shape_)

    def count(self, start=0, end=None):
        return math.prod(self.shape_[start:end])

    def shape(self, i):
        return self.shape_[i]

    num = property(lambda self: self.shape_[0])
    channels = property(lambda self: self.shape_[1] if len(self.shape_) > 1 else 1)
    height = property(lambda self: self.shape_[2] if len(self.shape_) > 2 else 1)
    width = property(lambda self: self.shape_[3] if len(self.shape_) > 3 else 1)
    num_axes = property(lambda self: len(self.shape_))
    mutable_gpu_data = property(lambda self: self.gpu_data)

    @property
    def gpu_diff(self):
        """Gradient buffer of the same size, allocated (zero filled) on first use."""
        n = self.count()
        if n > self._diff_capacity:
            if self._gpu_diff:
                self.cuda.FreeMemory(self._gpu_diff)
            self._gpu_diff = self.cuda.AllocMemory(n, bHalfSize=self.half)
            self._diff_capacity = n
        return self._gpu_diff

    mutable_gpu_diff = gpu_diff

    @property
    def mutable_cpu_diff(self):
        return self.cuda.GetMemoryFloat(self.gpu_diff, self.count()).reshape(self.shape_)

    @mutable_cpu_diff.setter
    def mutable_cpu_diff(self, values):
        self.cuda.SetMemory(self.gpu_diff, np.asarray(values, self.cuda.DTYPE).reshape(-1), nCount=self.count())

    @property
    def mutable_cpu_data(self):
        return self.cuda.GetMemoryFloat(self.gpu_data, self.count()).reshape(self.shape_)

    @mutable_cpu_data.setter
    def mutable_cpu_data(self, values):
        self.cuda.SetMemory(self.gpu_data, np.asarray(values, self.cuda.DTYPE).reshape(-1), nCount=self.count())

    def SetData(self, value):
        self.cuda.set(self.count(), self.gpu_data, float(value))

    def CopyFrom(self, src, bCopyDiff=False, bReshape=True):
        """Blob.cs CopyFrom(src, bCopyDiff, bReshape): copies the data, or with bCopyDiff the diff."""
        if bReshape:
            self.ReshapeLike(src)
        if bCopyDiff:
            self.cuda.copy(self.count(), src.gpu_diff, self.gpu_diff)
        else:
            self.cuda.copy(self.count(), src.gpu_data, self.gpu_data)

    def MatMul(self, blobA, blobB, bReshape=False, bTransA=False, bTransB=False, dfScale=1.0, bADiff=False, bBDiff=False,
               bCDiff=False, bAccumulate=False):
        """Blob.cs:4229-4269: batched row-major matmul over the two leading axes; the flags pick the diff side of each blob."""
        outer = blobA.count(0, 2)
        m = blobA.shape(3) if bTransA else blobA.shape(2)
        n = blobB.shape(2) if bTransB else blobB.shape(3)
        k = blobA.shape(2) if bTransA else blobA.shape(3)
        shape = [blobA.shape(0), blobB.shape(1), m, n]
        if bReshape:
            self.Reshape(*shape)
        elif self.shape_ != shape:
            raise ValueError("This (resulting) blob does not have the correct shape! Expected %s" % shape)
        hA = blobA.gpu_diff if bADiff else blobA.gpu_data
        hB = blobB.gpu_diff if bBDiff else blobB.gpu_data
        hC = self.gpu_diff if bCDiff else self.gpu_data
        self.cuda.matmul(outer, m, n, k, hA, hB, hC, dfScale, bTransA, bTransB, bAccumulate)

    def MatMulGrad(self, blobA, blobB, dfScale=1.0, bAccumulate=False):
        """Blob.cs:4304-4311: from this blob's diff, A.diff = dC B^T and B.diff = A^T dC."""
        if dfScale != 1.0:
            self.scale_diff(dfScale)
        blobA.MatMul(self, blobB, False, False, True, 1.0, True, False, True, bAccumulate)
        blobB.MatMul(blobA, self, False, True, False, 1.0, False, True, True, bAccumulate)

    def scale_data(self, df):
        self.cuda.scal(self.count(), df, self.gpu_data)

    def scale_diff(self, df):
        self.cuda.scal(self.count(), df, self.gpu_diff)

    def Dispose(self):
        if self.gpu_data:
            self.cuda.FreeMemory(self.gpu_data)
            self.gpu_data = 0
            self._capacity = 0
        if self._gpu_diff:
            self.cuda.FreeMemory(self._gpu_diff)
            self._gpu_diff = 0
            self._diff_capacity = 0


class InnerProductLayer:
    """MyCaffe/layers/InnerProductLayer.cs:372-417.  Weights are (num_output, K)."""

    def __init__(self, cuda, num_output, bias_term=True, axis=2, half=False, fused_bias=False):
        self.cuda, self.N, self.bias_term, self.axis, self.half = cuda, num_output, bias_term, axis, half
        # a single row goes through gemv and axpy (:385-392) unless fused_bias asks for the one call there too
        self.fused_bias = fused_bias
        self.fp32_sums = False    # forward on the fp32 matrix cores at every size (CudaDnn.LinearForward)
        self.blobs = []

    def Setup(self, bottom, weight=None, bias=None):
        self.K = bottom.count(self.axis)
        w = Blob(self.cuda, (self.N, self.K), self.half)
        if weight is not None:
            w.mutable_cpu_data = weight
        self.blobs = [w]
        if self.bias_term:
            b = Blob(self.cuda, (self.N,), self.half)
            if bias is not None:
                b.mutable_cpu_data = bias
            self.blobs.append(b)

    def Forward(self, bottom, top):
        M = bottom.count(0, self.axis)
        top.Reshape(*(bottom.shape_[:self.axis] + [self.N]))
        if not self._single_row(M, bottom, top):
            self.cuda.LinearForward(M, self.N, self.K, bottom.gpu_data, self.blobs[0].gpu_data, self.blobs[1].gpu_data if self.bias_term else 0,
                                    top.gpu_data, bFp32Sums=self.fp32_sums)

    def _single_row(self, M, bottom, top):
        """One fp32 row as gemv and axpy, if it is one (768 x 768: 2.5 us and a vector update, against 8.4 as a product)."""
        if M != 1 or self.half or self.fused_bias:
            return False
        self.cuda.gemv(False, self.N, self.K, 1.0, self.blobs[0].gpu_data, bottom.gpu_data, 0.0, top.gpu_data)
        if self.bias_term:
            self.cuda.axpy(self.N, 1.0, self.blobs[1].gpu_data, top.gpu_data)
        return True

    def ForwardHeads(self, bottom, top, heads):
        """Forward with the result written head by head, (B,T,K) -> (B, heads, T, N/heads)."""
        B, T = bottom.shape_[:2]
        top.Reshape(B, heads, T, self.N // heads)
        if self._single_row(B * T, bottom, top):   # the heads of one position lie one after the other
            return
        self.cuda.LinearForward(B * T, self.N, self.K, bottom.gpu_data, self.blobs[0].gpu_data, self.blobs[1].gpu_data if self.bias_term else 0,
                                top.gpu_data, T, heads, self.fp32_sums)

    def Backward(self, top, bottom, accumulate=False):
        """InnerProductLayer.cs:429-494: weight and bias gradients accumulate into their diffs, data gradient = top diff x W
        (``accumulate``: added to what the bottom's diff holds)."""
        self.cuda.LinearBackward(bottom.count(0, self.axis), self.N, self.K, bottom.gpu_data, self.blobs[0].gpu_data, top.gpu_diff,
                                 self.blobs[0].gpu_diff, self.blobs[1].gpu_diff if self.bias_term else 0, bottom.gpu_diff, accumulate)


class _Kept(dict):
    """What a layer builds for a shape and needs again when the shape comes back: the last few, the oldest given back."""

    MAX = 8

    def __init__(self, free):
        super().__init__()
        self._free = free

    def get_or(self, key, make):
        if key not in self:
            while len(self) >= self.MAX:
                self._free(self.pop(next(iter(self))))
            self[key] = make()
        return self[key]


class TransposeLayer:
    """MyCaffe.layers.beta/layers.beta/TransposeLayer.cs:127-232."""

    MAX_SHAPES = 8

    def __init__(self, cuda, dim):
        self.cuda, self.dim = cuda, list(dim)
        # The attention layers send two shapes through one transpose layer in turn, (B,T,H,hs) on the way in and (B,H,T,hs)
        # on the way out, so the blobs of a few shapes are kept: uploading them again on every call cost five allocations
        # and five frees, each waiting for the device (0.5 ms a call).
        self._shapes = {}
        self._buffer, self._buffer_count = 0, 0
        self._handles = []

    def _reshape(self, shape):
        """Reshape (TransposeLayer.cs:127-200): stride arrays of bottom and top, forward and backward axis maps."""
        key = tuple(shape)
        known = self._shapes.get(key)
        if known is None:
            n = len(shape)
            top_shape = [shape[d] for d in self.dim]
            bc = [math.prod(shape[i + 1:]) for i in range(n)]
            tc = [math.prod(top_shape[i + 1:]) for i in range(n)]
            bmap = [0] * n
            for i, d in enumerate(self.dim):
                bmap[d] = i
            if len(self._shapes) >= self.MAX_SHAPES:
                for h in self._shapes.pop(next(iter(self._shapes)))[1]:
                    self.cuda.FreeMemory(h)
            known = self._shapes[key] = (top_shape, [self.cuda.AllocMemory(np.float32(v)) for v in (bc, tc, self.dim, bmap)])
            if math.prod(shape) * n > self._buffer_count:
                if self._buffer:
                    self.cuda.FreeMemory(self._buffer)
                self._buffer_count = math.prod(shape) * n
                self._buffer = self.cuda.AllocMemory(self._buffer_count)
            self._handles = [h for _, hs in self._shapes.values() for h in hs] + [self._buffer]
        self.counts_b, self.counts_t, self.fmap, self.bmap = known[1]
        return known[0]

    def Forward(self, bottom, top):
        if bottom.gpu_data == top.gpu_data:
            raise ValueError("The Transpose layer does not support in-place computation.")
        top.Reshape(*self._reshape(bottom.shape_))
        self.cuda.transpose(bottom.count(), bottom.gpu_data, top.gpu_data, self.counts_b, self.counts_t, self.fmap,
                            len(bottom.shape_), self._buffer)

    def Backward(self, top, bottom):
        """TransposeLayer.cs:223-232: reshape for this bottom, then the same kernel with the count arrays swapped and the
        inverse axis map."""
        self._reshape(bottom.shape_)
        self.cuda.transpose(bottom.count(), top.gpu_diff, bottom.gpu_diff, self.counts_t, self.counts_b, self.bmap,
                            len(bottom.shape_), self._buffer)


class SoftmaxLayer:
    """MyCaffe/layers/SoftmaxLayer.cs: the cuDNN engine (:172-181, 339-367) or, with ``engine="CAFFE"``, the chain of
    primitives of forward_cuda / backward_cuda (:230-330; ``algorithm="LOG"`` for the log-softmax variant)."""

    def __init__(self, cuda, axis=-1, engine="CUDNN", algorithm="ACCURATE"):
        self.cuda, self.axis, self.engine, self.algorithm = cuda, axis, engine, algorithm
        self.hCudnn = cuda.CreateCuDNN()
        self.hBottomDesc = cuda.CreateTensorDesc()
        self.hTopDesc = cuda.CreateTensorDesc()
        self.blobScale = None

    def _forward_caffe(self, bottom, top):
        """SoftmaxLayer.cs:230-273."""
        cuda = self.cuda
        axis = self.axis % bottom.num_axes
        nOuter, nCh, nInner = bottom.count(0, axis), bottom.shape(axis), bottom.count(axis + 1)
        top.ReshapeLike(bottom)
        if self.blobScale is None or self.blobScale.count() != nOuter * nInner or self.blobScale.half != bottom.half:
            self.blobScale = Blob(cuda, (nOuter, nInner), bottom.half)
        self._dims = (nOuter, nCh, nInner)
        hB, hT, hSd, hSf = bottom.gpu_data, top.gpu_data, self.blobScale.gpu_data, self.blobScale.gpu_diff
        n = bottom.count()
        cuda.copy(n, hB, hT)
        cuda.channel_max(nOuter * nInner, nOuter, nCh, nInner, hT, hSd)
        cuda.channel_sub(n, nOuter, nCh, nInner, hSd, hT)
        cuda.exp(n, hT, hT)
        cuda.channel_sum(nOuter * nInner, nOuter, nCh, nInner, hT, hSf)
        if self.algorithm == "LOG":
            cuda.log(nOuter * nInner, hSf, hSf)
            cuda.add(nOuter * nInner, hSd, hSf, hSd)
            cuda.copy(n, hB, hT)
            cuda.channel_sub(n, nOuter, nCh, nInner, hSd, hT)
        else:
            cuda.channel_div(n, nOuter, nCh, nInner, hSf, hT)

    def _backward_caffe(self, top, bottom):
        """SoftmaxLayer.cs:289-330 (the ACCURATE branch: inner1d(top_diff, top_data), subtract, multiply)."""
        cuda = self.cuda
        nOuter, nCh, nInner = self._dims
        n = top.count()
        if self.algorithm == "LOG":
            raise NotImplementedError("log-softmax gradient chain (channel_fillfrom over a reshaped scale blob)")
        cuda.copy(n, top.gpu_diff, bottom.gpu_diff)
        cuda.channel_dot(nOuter * nInner, nOuter, nCh, nInner, top.gpu_diff, top.gpu_data, self.blobScale.gpu_data)
        cuda.channel_sub(n, nOuter, nCh, nInner, self.blobScale.gpu_data, bottom.gpu_diff)
        cuda.mul(n, bottom.gpu_diff, top.gpu_data, bottom.gpu_diff)

    def Forward(self, bottom, top):
        if self.engine == "CAFFE":
            return self._forward_caffe(bottom, top)
        axis = self.axis % bottom.num_axes
        nN, nK, nH = bottom.count(0, axis), bottom.shape(axis), bottom.count(axis + 1)
        mode = SOFTMAX_MODE.INSTANCE if nH == 1 else SOFTMAX_MODE.CHANNEL
        top.ReshapeLike(bottom)
        self.cuda.SetTensorDesc(self.hBottomDesc, nN, nK, nH, 1, bottom.half)
        self.cuda.SetTensorDesc(self.hTopDesc, nN, nK, nH, 1, top.half)
        self.cuda.SoftmaxForward(self.hCudnn, SOFTMAX_ALGORITHM.ACCURATE, mode, 1.0, self.hBottomDesc, bottom.gpu_data, 0.0,
                                 self.hTopDesc, top.gpu_data)
        self._mode = mode

    def Backward(self, top, bottom):
        """SoftmaxLayer.cs:359-367: bottom.diff from top.data and top.diff (descriptors as set by Forward)."""
        if self.engine == "CAFFE":
            return self._backward_caffe(top, bottom)
        self.cuda.SoftmaxBackward(self.hCudnn, SOFTMAX_ALGORITHM.ACCURATE, self._mode, 1.0, self.hTopDesc, top.gpu_data, self.hTopDesc,
                                  top.gpu_diff, 0.0, self.hBottomDesc, bottom.gpu_diff)


class CausalSelfAttentionLayer:
    """MyCaffe.layers.gpt/layers.gpt/CausalSelfAttentionLayer.cs (setup :96-250, forward :526-628).

    ``enable_cuda_scaled_dot_product_attention`` selects the fused attention handle
    (ids 160-163); otherwise the explicit transpose / MatMul / scale / mask /
    softmax / MatMul chain runs, as in the reference.
    """

    def __init__(self, cuda, heads, embed, block_size, bias_term=True, enable_cuda_scaled_dot_product_attention=True,
                 enable_rotary_positional_embedding=False, rope_theta=10000.0, half=False, training=False,
                 fused_qkv_heads=False):
        self.training = training
        # inference with the fused attention handle as three calls: the handle writes its output head-merged
        self.fused_qkv_heads = fused_qkv_heads
        self.cuda, self.nHeads, self.nEmbed, self.nBlockSize = cuda, heads, embed, block_size
        self.nSize = embed // heads
        self.bias_term, self.half = bias_term, half
        self.enable_sdpa = enable_cuda_scaled_dot_product_attention
        self.enable_rope, self.rope_theta = enable_rotary_positional_embedding, rope_theta
        self.dfIgnoreVal = -1e29
        self.c_attn = InnerProductLayer(cuda, 3 * embed, bias_term, 2, half)
        self.c_proj = InnerProductLayer(cuda, embed, bias_term, 2, half, fused_bias=fused_qkv_heads)
        self.transpose = TransposeLayer(cuda, (0, 2, 1, 3))
        self.transposeQ = TransposeLayer(cuda, (0, 1, 3, 2))
        self.softmax = SoftmaxLayer(cuda, -1)
        names = "IpAttn Qt Kt Vt Kt1 AttA AttB Work Y".split()
        self.b = {n: Blob(cuda, half=half) for n in names}
        self.blobMask = Blob(cuda, (1, 1, block_size, block_size))
        mask = np.tril(np.ones((block_size, block_size), np.float32))  # fillMask :276-291
        self.blobMask.mutable_cpu_data = mask
        self._masks, self._ropes = _Kept(Blob.Dispose), _Kept(cuda.FreeRope)
        self.hCudnn = self.hAttn = self.hRope = 0
        self._set_for = None

    def Setup(self, bottom, w_attn, b_attn, w_proj, b_proj):
        self.c_attn.Setup(bottom, w_attn, b_attn)
        y = Blob(self.cuda, bottom.shape_, self.half)
        self.c_proj.Setup(y, w_proj, b_proj)
        y.Dispose()

    def _reshape(self, B, T):
        if self._set_for == (B, T):
            return
        if self.enable_sdpa:
            if not self.hCudnn:
                self.hCudnn = self.cuda.CreateCuDNN()
                self.hAttn = self.cuda.CreateAttn()
            self.cuda.SetAttn(self.hCudnn, self.hAttn, 0, self.training, B, self.nBlockSize, self.nHeads, self.nSize, 0.0)
        if self.enable_rope:
            self.hRope = self._ropes.get_or((B, T), lambda: self.cuda.CreateRope(0, 0, B * T * self.nEmbed, B, T, self.nHeads, self.nSize, self.rope_theta))
        self._set_for = (B, T)

    def _mask(self, T):
        """The causal mask of T positions: the layer's own, or one of the last few of shorter sequences."""
        if T == self.nBlockSize:
            return self.blobMask

        def make():
            m = Blob(self.cuda, (1, 1, T, T))
            m.mutable_cpu_data = np.tril(np.ones((T, T), np.float32))
            return m
        return self._masks.get_or(T, make)

    def Forward(self, blobX, top):
        B, T, C = blobX.shape_[:3]
        if T > self.nBlockSize:
            raise ValueError("sequence longer than block_size")
        self._reshape(B, T)
        b, cuda, H, hs = self.b, self.cuda, self.nHeads, self.nSize
        if self.fused_qkv_heads and (not self.enable_sdpa or self.training):
            raise ValueError("fused_qkv_heads needs the fused attention handle, inference mode")
        # q, k, v = self.c_attn(x).split(self.n_embd, dim=2), rotated, (B, T, nh, hs) -> (B, nh, T, hs): one call for the
        # projection, its bias, three channel copies, two rotations and three transposes (:526-557)
        for name in ("Qt", "Kt", "Vt"):
            b[name].Reshape(B, H, T, hs)
        w = self.c_attn.blobs
        cuda.QkvProjHeads(B, T, H, hs, blobX.gpu_data, w[0].gpu_data, w[1].gpu_data if self.bias_term else 0, b["Qt"].gpu_data, b["Kt"].gpu_data,
                          b["Vt"].gpu_data, self.hRope, self.c_attn.fp32_sums)
        if self.enable_sdpa:
            out = b["Work"]
            if self.fused_qkv_heads:
                out = b["Y"]
                out.Reshape(B, T, C)
            else:
                out.ReshapeLike(b["Vt"])
            mask = self._mask(T)   # the handle reads a (1,1,T,T) mask for the block size it is run with
            if self.fused_qkv_heads:
                cuda.AttnScaledDotProductForward(self.hCudnn, self.hAttn, T, b["Qt"].gpu_data, b["Kt"].gpu_data, b["Vt"].gpu_data,
                                                 mask.gpu_data, out.gpu_data, False, T, True)
                self.c_proj.Forward(out, top)
                return
            cuda.AttnScaledDotProductForward(self.hCudnn, self.hAttn, T, b["Qt"].gpu_data, b["Kt"].gpu_data, b["Vt"].gpu_data,
                                             mask.gpu_data, out.gpu_data, False, bOneWave=self.training and self.c_attn.fp32_sums)
        else:
            self.transposeQ.Forward(b["Kt"], b["Kt1"])
            dfScale = 1.0 / math.sqrt(hs)
            b["AttA"].MatMul(b["Qt"], b["Kt1"], bReshape=True)
            b["AttA"].scale_data(dfScale)
            mask = self._mask(T)
            cuda.mask(b["AttA"].count(), mask.count(), 0.0, self.dfIgnoreVal, b["AttA"].gpu_data, mask.gpu_data, b["AttA"].gpu_data)
            self.softmax.Forward(b["AttA"], b["AttB"])
            b["Work"].MatMul(b["AttB"], b["Vt"], bReshape=True)
        # y.transpose(1, 2).contiguous().view(B, T, C)
        self.transpose.Forward(b["Work"], b["Y"])
        b["Y"].Reshape(B, T, C)
        self.c_proj.Forward(b["Y"], top)

    def Backward(self, top, blobX):
        """CausalSelfAttentionLayer.cs:641-747: top.gpu_diff -> blobX.gpu_diff, parameter gradients accumulate in the
        InnerProduct weight diffs.  Fused handle: its backward call gets mask handle 0, as there.  Explicit chain: the
        two MatMulGrad calls around the softmax gradient (no dropout)."""
        b, cuda = self.b, self.cuda
        B, T, C = blobX.shape_[:3]
        H, hs = self.nHeads, self.nSize
        self.c_proj.Backward(top, b["Y"])
        b["Y"].Reshape(B, T, H, hs)
        self.transpose.Backward(b["Y"], b["Work"])
        b["Y"].Reshape(B, T, C)
        if self.enable_sdpa:
            cuda.AttnScaledDotProductBackward(self.hCudnn, self.hAttn, b["Qt"].gpu_data, b["Qt"].gpu_diff, b["Kt"].gpu_data,
                                              b["Kt"].gpu_diff, b["Vt"].gpu_data, b["Vt"].gpu_diff, 0, b["Work"].gpu_data, b["Work"].gpu_diff)
        else:
            # att' = y' @ v^T, vt' = att^T @ y'; softmax gradient; qt' = att' @ kt, kt1' = qt^T @ att' (scaled)
            b["Work"].MatMulGrad(b["AttB"], b["Vt"])
            self.softmax.Backward(b["AttB"], b["AttA"])
            b["AttA"].MatMulGrad(b["Qt"], b["Kt1"], 1.0 / math.sqrt(hs))
            self.transposeQ.Backward(b["Kt1"], b["Kt"])
        # three transposes, two rotations and three channel copies (:700-740)
        ip = b["IpAttn"]
        ip.Reshape(B, T, 3 * C)
        cuda.QkvHeadsGrad(B, T, H, hs, b["Qt"].gpu_diff, b["Kt"].gpu_diff, b["Vt"].gpu_diff, ip.gpu_diff, self.hRope)
        self.c_attn.Backward(ip, blobX)


class MultiheadAttentionLayer:
    """MyCaffe.layers.gpt/layers.gpt/MultiheadAttentionLayer.cs:643-811.  With ``enable_key_value_cache`` and the
    "position" layer option set, the explicit chain takes the reference's cached decode branch (:713-730, 759-777: one
    token per call, a loop over the cached positions); :meth:`CudaDnn.AttnDecodeForward` is the one-call replacement.

    ``Forward(q, k, v, mask)``: mask is ``None``, a (1,1,T,T) blob (causal), a
    (B,T_k) key-padding blob or a (B,T_q,T_k) blob; the last two take the
    mask_batch route, as in the reference (``fuse_batch_qk_mask`` sends the
    (B,T_q,T_k) mask to the fused handle instead, which the reference's handle
    cannot do).
    """

    def __init__(self, cuda, heads, embed, block_size, bias_term=True, enable_cuda_scaled_dot_product_attention=True,
                 enable_rotary_positional_embedding=False, rope_theta=10000.0, half=False, fuse_batch_qk_mask=False,
                 enable_key_value_cache=False):
        self.cuda, self.nHeads, self.nEmbed, self.nBlockSize = cuda, heads, embed, block_size
        self.fuse_batch_qk_mask = fuse_batch_qk_mask
        self.enable_kv_cache = enable_key_value_cache
        self.nSize = embed // heads
        self.half = half
        self.enable_sdpa = enable_cuda_scaled_dot_product_attention
        self.enable_rope, self.rope_theta = enable_rotary_positional_embedding, rope_theta
        self.c_attnQ = InnerProductLayer(cuda, embed, bias_term, 2, half)
        self.c_attnK = InnerProductLayer(cuda, embed, bias_term, 2, half)
        self.c_attnV = InnerProductLayer(cuda, embed, bias_term, 2, half)
        self.c_proj = InnerProductLayer(cuda, embed, bias_term, 2, half)
        self.transpose = TransposeLayer(cuda, (0, 2, 1, 3))
        self.transposeK = TransposeLayer(cuda, (0, 2, 1, 3))
        self.transposeQ = TransposeLayer(cuda, (0, 1, 3, 2))
        self.softmax = SoftmaxLayer(cuda, -1)
        self.b = {n: Blob(cuda, half=half) for n in "Q K Qt Kt Vt Kt1 AttA AttB Work Y KeyCache ValCache Work2 Work3".split()}
        self.hCudnn = self.hAttn = self.hRope = 0
        self._set_for = None
        self.options = {}

    def SetLayerOption(self, name, value):
        self.options[name] = value

    def Setup(self, q, k, v, weights):
        """weights: dict with wq,bq,wk,bk,wv,bv,wo,bo ([out,in] matrices)."""
        self.c_attnQ.Setup(q, weights["wq"], weights.get("bq"))
        self.c_attnK.Setup(k, weights["wk"], weights.get("bk"))
        self.c_attnV.Setup(v, weights["wv"], weights.get("bv"))
        self.c_proj.Setup(q, weights["wo"], weights.get("bo"))

    def Forward(self, q, k, v, blobMask, top):
        cuda, H, hs, b = self.cuda, self.nHeads, self.nSize, self.b
        B, Tq, C = q.shape_[:3]
        Tk = k.shape_[1]
        nPos = int(self.options.get("position", -1))
        if self.enable_rope:
            self.c_attnQ.Forward(q, b["Q"])
            self.c_attnK.Forward(k, b["K"])
            self.c_attnV.ForwardHeads(v, b["Vt"], H)
            b["Q"].Reshape(B, Tq, H, hs)
            b["K"].Reshape(B, Tk, H, hs)
            if not self.hRope:
                self.hRope = cuda.CreateRope(0, 0, B * self.nBlockSize * C, B, self.nBlockSize, H, hs, self.rope_theta)
            nFreqOffset = nPos * hs // 2 if nPos > 0 else -1
            cuda.RopeForward(self.hRope, b["Q"].count(), b["Q"].gpu_data, b["Q"].gpu_data, nFreqOffset)
            cuda.RopeForward(self.hRope, b["K"].count(), b["K"].gpu_data, b["K"].gpu_data, nFreqOffset)
            self.transpose.Forward(b["Q"], b["Qt"])
            self.transposeK.Forward(b["K"], b["Kt"])
        else:
            # projections written head by head: no transposes behind them; in 16-bit storage one call
            projections = ((self.c_attnQ, q, b["Qt"]), (self.c_attnK, k, b["Kt"]), (self.c_attnV, v, b["Vt"]))
            if self.half:
                for _, x, y in projections:
                    y.Reshape(B, H, x.shape_[1], hs)
                cuda.LinearHeadsGroup(C, C, H, [(x.count(0, 2), x.shape_[1], x.gpu_data, layer.blobs[0].gpu_data,
                                                 layer.blobs[1].gpu_data if layer.bias_term else 0, y.gpu_data) for layer, x, y in projections])
            else:
                for layer, x, y in projections:
                    layer.ForwardHeads(x, y, H)
        is_qk_mask = (blobMask is not None and blobMask.num_axes == 4 and blobMask.num == 1 and blobMask.channels == 1
                      and blobMask.height == Tq and blobMask.width == Tk)
        full_mask = blobMask is not None and not is_qk_mask and blobMask.count() == B * Tq * Tk and Tq > 1
        if self.enable_sdpa and (not full_mask or self.fuse_batch_qk_mask):
            if self._set_for != B:
                if not self.hCudnn:
                    self.hCudnn = cuda.CreateCuDNN()
                    self.hAttn = cuda.CreateAttn()
                cuda.SetAttn(self.hCudnn, self.hAttn, 0, False, B, self.nBlockSize, H, hs, 0.0)
                self._set_for = B
            b["Y"].Reshape(B, Tq, C)
            cuda.AttnScaledDotProductForward(self.hCudnn, self.hAttn, Tq, b["Qt"].gpu_data, b["Kt"].gpu_data, b["Vt"].gpu_data,
                                             blobMask.gpu_data if blobMask is not None else 0, b["Y"].gpu_data,
                                             2 if full_mask else (not is_qk_mask), Tk, True)
            self.c_proj.Forward(b["Y"], top)
            return
        else:
            # the fused handle only understands (1,1,T,T) or (B,T) masks (attn.cu:544-556); a
            # (B,T_q,T_k) mask goes through the explicit chain (MultiheadAttentionLayer.cs:733-742)
            self.transposeQ.Forward(b["Kt"], b["Kt1"])
            dfScale = 1.0 / math.sqrt(hs)
            cached = nPos >= 0 and self.enable_kv_cache
            if cached:
                # one token: append its key / value to the caches (sized for the block size at the first call, as the
                # layer's reshape does), then one MatMul per cached position (:713-730)
                for name in ("KeyCache", "ValCache"):
                    if b[name]._capacity == 0:
                        b[name].Reshape(B, H, self.nBlockSize, hs)
                b["KeyCache"].Reshape(nPos + 1, H, hs, 1)
                b["ValCache"].Reshape(nPos + 1, H, 1, hs)
                nK, nV = b["Kt1"].count(), b["Vt"].count()
                cuda.copy(nK, b["Kt1"].gpu_data, b["KeyCache"].gpu_data, 0, nPos * nK)
                cuda.copy(nV, b["Vt"].gpu_data, b["ValCache"].gpu_data, 0, nPos * nV)
                b["AttA"].Reshape(1, H, 1, nPos + 1)
                for i in range(nPos + 1):
                    cuda.copy(nK, b["KeyCache"].gpu_data, b["Kt1"].gpu_data, i * nK, 0)
                    b["Work2"].MatMul(b["Qt"], b["Kt1"], True)
                    b["Work2"].scale_data(dfScale)
                    cuda.channel_copy(b["Work2"].count(), 1, H, nPos + 1, 1, i, b["AttA"].gpu_data, b["Work2"].gpu_data, DIR.BWD)
            else:
                b["AttA"].MatMul(b["Qt"], b["Kt1"], bReshape=True)
                b["AttA"].scale_data(dfScale)
                if blobMask is not None:
                    if is_qk_mask:
                        cuda.mask(b["AttA"].count(), blobMask.count(), 0.0, -1e29, b["AttA"].gpu_data, blobMask.gpu_data, b["AttA"].gpu_data)
                    else:
                        cuda.mask_batch(b["AttA"].count(), b["AttA"].num, blobMask.count(), 0.0, -1e29, b["AttA"].gpu_data,
                                        blobMask.gpu_data, b["AttA"].gpu_data)
            self.softmax.Forward(b["AttA"], b["AttB"])
            if cached:
                # y = sum over the cached positions of weight_i * v_i, one MatMul and one add per position (:759-777)
                b["Work"].Reshape(1, H, 1, hs)
                b["Work3"].Reshape(1, H, 1, 1)
                b["Work2"].Reshape(1, H, 1, hs)
                nV = b["Vt"].count()
                for i in range(nPos + 1):
                    cuda.copy(nV, b["ValCache"].gpu_data, b["Vt"].gpu_data, i * nV, 0)
                    cuda.channel_copy(b["Work3"].count(), 1, H, nPos + 1, 1, i, b["AttB"].gpu_data, b["Work3"].gpu_data, DIR.FWD)
                    b["Work2"].MatMul(b["Work3"], b["Vt"], True)
                    if i == 0:
                        cuda.copy(b["Work"].count(), b["Work2"].gpu_data, b["Work"].gpu_data)
                    else:
                        cuda.add(b["Work"].count(), b["Work2"].gpu_data, b["Work"].gpu_data, b["Work"].gpu_data)
            else:
                b["Work"].MatMul(b["AttB"], b["Vt"], bReshape=True)
        self.transpose.Forward(b["Work"], b["Y"])
        b["Y"].Reshape(B, Tq, C)
        self.c_proj.Forward(b["Y"], top)


class LayerNormLayer:
    """MyCaffe.layers.gpt/layers.gpt/LayerNormLayer.cs.  ``enable_cuda_impl`` runs the LayerNorm handle (ids 970-976;
    reshape :153-166, forward :211-212, backward :285-286); otherwise the explicit chain of :223-264 runs (channel_mean,
    channel_fillfrom, sub, powx, channel_mean, add_scalar, sqrt, channel_fillfrom, div)."""

    def __init__(self, cuda, epsilon=1e-10, enable_cuda_impl=True):
        self.cuda, self.epsilon, self.enable_cuda_impl = cuda, epsilon, enable_cuda_impl
        self.hLayerNorm = 0
        self._kept = _Kept(cuda.FreeLayerNorm)
        self._shape = None
        self.b = {n: Blob(cuda) for n in "Mu Xmu XmuSq Var Stdev StdevFull Work".split()}

    def _reshape(self, bottom):
        nAxis = len(bottom.shape_) - 1
        self.nCount = bottom.count()
        self.nOuterNum, self.nChannels, self.nInnerNum = bottom.shape_[0], bottom.count(1, nAxis), bottom.count(nAxis)
        if self._shape == bottom.shape_:
            return
        if self.enable_cuda_impl:
            self.hLayerNorm = self._kept.get_or(tuple(bottom.shape_), lambda: self.cuda.CreateLayerNorm(
                0, self.nCount, self.nOuterNum, self.nChannels, self.nInnerNum, self.epsilon))
        else:
            for n in ("Xmu", "XmuSq", "StdevFull"):
                self.b[n].ReshapeLike(bottom)
            for n in ("Mu", "Var", "Stdev"):
                self.b[n].Reshape(self.nOuterNum, self.nChannels, 1, 1)
        self._shape = list(bottom.shape_)

    def Forward(self, bottom, top):
        self._reshape(bottom)
        top.ReshapeLike(bottom)
        cuda, b = self.cuda, self.b
        if self.enable_cuda_impl:
            cuda.LayerNormForward(self.hLayerNorm, bottom.gpu_data, top.gpu_data)
            return
        n, o, c, i = self.nCount, self.nOuterNum, self.nChannels, self.nInnerNum
        cuda.channel_mean(n, o, c, i, bottom.gpu_data, b["Mu"].gpu_data)
        cuda.channel_fillfrom(n, o, c, i, b["Mu"].gpu_data, b["Xmu"].gpu_data, DIR.FWD)
        cuda.sub(n, bottom.gpu_data, b["Xmu"].gpu_data, b["Xmu"].gpu_data)
        cuda.powx(n, b["Xmu"].gpu_data, 2.0, b["XmuSq"].gpu_data)
        cuda.channel_mean(n, o, c, i, b["XmuSq"].gpu_data, b["Var"].gpu_data)
        cuda.add_scalar(o * c, self.epsilon, b["Var"].gpu_data)
        cuda.sqrt(o * c, b["Var"].gpu_data, b["Stdev"].gpu_data)
        cuda.channel_fillfrom(n, o, c, i, b["Stdev"].gpu_data, b["StdevFull"].gpu_data, DIR.FWD)
        cuda.div(n, b["Xmu"].gpu_data, b["StdevFull"].gpu_data, top.gpu_data)

    def ForwardAdd(self, x, add, total, top):
        """total = x + add, top = norm(total)."""
        total.ReshapeLike(x)
        if not self.enable_cuda_impl:
            self.cuda.add(x.count(), x.gpu_data, add.gpu_data, total.gpu_data)
            return self.Forward(total, top)
        self._reshape(x)
        top.ReshapeLike(x)
        self.cuda.NormAddForward(self.hLayerNorm, 0, 0, x.gpu_data, add.gpu_data, total.gpu_data, 0, top.gpu_data)

    def BackwardAdd(self, top, bottom, hAdd):
        """Backward with the values behind hAdd added to the bottom's diff."""
        if not self.enable_cuda_impl:
            self.Backward(top, bottom)
            return self.cuda.add(bottom.count(), hAdd, bottom.gpu_diff, bottom.gpu_diff)
        self.cuda.NormAddBackward(self.hLayerNorm, top.gpu_data, top.gpu_diff, bottom.gpu_diff, hAdd)

    def Backward(self, top, bottom):
        if self.enable_cuda_impl:
            self.cuda.LayerNormBackward(self.hLayerNorm, top.gpu_data, top.gpu_diff, bottom.gpu_diff)
            return
        # LayerNormLayer.cs:292-320, the layer's own chain: dx = (dy - (y * mean(y * dy) + mean(dy))) / (std + eps)
        cuda, b = self.cuda, self.b
        n, o, c, i = self.nCount, self.nOuterNum, self.nChannels, self.nInnerNum
        b["Work"].ReshapeLike(top)
        cuda.mul(n, top.gpu_data, top.gpu_diff, b["Work"].gpu_data)
        cuda.channel_mean(n, o, c, i, b["Work"].gpu_data, b["Var"].gpu_diff)
        cuda.channel_mean(n, o, c, i, top.gpu_diff, b["Stdev"].gpu_diff)
        cuda.channel_fillfrom(n, o, c, i, b["Var"].gpu_diff, b["StdevFull"].gpu_diff, DIR.FWD)
        cuda.mul(n, top.gpu_data, b["StdevFull"].gpu_diff, b["Work"].gpu_data)
        cuda.channel_fillfrom(n, o, c, i, b["Stdev"].gpu_diff, b["StdevFull"].gpu_diff, DIR.FWD)
        cuda.add(n, b["Work"].gpu_data, b["StdevFull"].gpu_diff, b["Work"].gpu_data)
        cuda.sub(n, top.gpu_diff, b["Work"].gpu_data, b["Work"].gpu_data)
        cuda.add_scalar(b["StdevFull"].count(), self.epsilon, b["StdevFull"].gpu_data)
        cuda.div(n, b["Work"].gpu_data, b["StdevFull"].gpu_data, bottom.gpu_diff)


class RMSNormLayer:
    """MyCaffe.layers.gpt/layers.gpt/RMSNormLayer.cs:96-180, the layer's own chain: powx(2), channel_mean, sqrt(+eps),
    invert, channel_duplicate, mul, and with weights channel_copyall + mul.  ``fused`` replaces the chains by the
    single calls RMSNORM_FWD and RMSNORM_BWD (ids 2002, 2008), which have no counterpart in the reference."""

    def __init__(self, cuda, epsilon=1e-5, enable_weights=True, fused=False):
        self.cuda, self.epsilon, self.enable_weights, self.fused = cuda, epsilon, enable_weights, fused
        self.blobs = []
        self.b = {n: Blob(cuda) for n in "Rms Rms1 Out Rms1Full".split()}

    def Setup(self, bottom, weight=None):
        nAxis = len(bottom.shape_) - 1
        if self.enable_weights:
            w = Blob(self.cuda, (bottom.count(nAxis),))
            w.mutable_cpu_data = np.ones(bottom.count(nAxis), np.float32) if weight is None else weight
            self.blobs = [w]

    def Forward(self, bottom, top):
        cuda, b = self.cuda, self.b
        nAxis = len(bottom.shape_) - 1
        n, inner = bottom.count(), bottom.count(nAxis)
        channels, outer = bottom.shape_[nAxis - 1], bottom.count(0, nAxis - 1)
        top.ReshapeLike(bottom)
        if self.fused:
            cuda.RmsNormForward(outer * channels, inner, bottom.gpu_data, self.blobs[0].gpu_data if self.enable_weights else 0,
                                top.gpu_data, self.epsilon)
            return
        b["Rms"].Reshape(outer, channels, 1, 1)
        b["Rms1"].Reshape(outer, channels, 1, 1)
        b["Out"].ReshapeLike(bottom)
        b["Rms1Full"].ReshapeLike(bottom)
        cuda.powx(n, bottom.gpu_data, 2.0, top.gpu_data)
        cuda.channel_mean(n, outer, channels, inner, top.gpu_data, b["Rms"].gpu_data)
        cuda.sqrt(b["Rms"].count(), b["Rms"].gpu_data, b["Rms"].gpu_data, self.epsilon)
        cuda.invert(b["Rms1"].count(), b["Rms"].gpu_data, b["Rms1"].gpu_data)
        cuda.channel_duplicate(n, outer * channels, 1, inner, b["Rms1"].gpu_data, b["Rms1Full"].gpu_data)
        cuda.mul(n, bottom.gpu_data, b["Rms1Full"].gpu_data, b["Out"].gpu_data)
        if self.enable_weights:
            cuda.channel_copyall(n, outer * channels, 1, inner, self.blobs[0].gpu_data, b["Out"].gpu_diff)
            cuda.mul(n, b["Out"].gpu_diff, b["Out"].gpu_data, top.gpu_data)
        else:
            top.CopyFrom(b["Out"])
        self._dims = (n, outer, channels, inner)

    def ForwardAdd(self, x, add, total, top):
        """total = x + add, top = norm(total)."""
        total.ReshapeLike(x)
        if not self.fused:
            self.cuda.add(x.count(), x.gpu_data, add.gpu_data, total.gpu_data)
            return self.Forward(total, top)
        nAxis = len(x.shape_) - 1
        top.ReshapeLike(x)
        self.cuda.NormAddForward(0, x.count(0, nAxis), x.count(nAxis), x.gpu_data, add.gpu_data, total.gpu_data,
                                 self.blobs[0].gpu_data if self.enable_weights else 0, top.gpu_data, self.epsilon)

    def BackwardAdd(self, top, bottom, hAdd):
        """Backward with the values behind hAdd added to the bottom's diff."""
        if self.fused:
            return self.Backward(top, bottom, hAdd=hAdd)
        self.Backward(top, bottom)
        self.cuda.add(bottom.count(), hAdd, bottom.gpu_diff, bottom.gpu_diff)

    def Backward(self, top, bottom, freeze_learning=False, hAdd=0):
        """RMSNormLayer.cs:189-232, the layer's own chain (after a Forward through the chain): top.diff -> bottom.diff and,
        with weights, the weight gradient through channel_sum (which, as there, keeps the sums of the first batch
        entry: the call passes outer = batch and a gradient blob of `inner` values)."""
        cuda, b = self.cuda, self.b
        if self.fused:
            nAxis = len(bottom.shape_) - 1
            hW, hdW = (self.blobs[0].gpu_data, 0 if freeze_learning else self.blobs[0].gpu_diff) if self.enable_weights else (0, 0)
            cuda.RmsNormBackward(bottom.count(0, nAxis), bottom.count(nAxis), bottom.gpu_data, hW, top.gpu_diff, bottom.gpu_diff, hdW,
                                 bottom.shape_[nAxis - 1], self.epsilon, hAdd)
            return
        n, outer, channels, inner = self._dims
        if self.enable_weights:
            if not freeze_learning:
                cuda.mul(n, top.gpu_diff, b["Out"].gpu_data, b["Out"].gpu_data)
                cuda.channel_sum(n, outer, channels, inner, b["Out"].gpu_data, self.blobs[0].gpu_diff)
            cuda.mul(n, top.gpu_diff, b["Out"].gpu_diff, b["Out"].gpu_diff)
        # (without weights the reference reads Out's gradient here although nothing has written it; same here)
        # x6 = x * x5 -> dx and dx5
        cuda.mul(n, b["Out"].gpu_diff, b["Rms1Full"].gpu_data, bottom.gpu_diff)
        cuda.mul(n, b["Out"].gpu_diff, bottom.gpu_data, b["Rms1Full"].gpu_diff)
        cuda.channel_sumEx(n, outer, channels, inner, b["Rms1Full"].gpu_diff, b["Rms1"].gpu_diff, False, DIR.FWD)
        # x5 = 1 / x4 -> dx4
        cuda.powx(b["Rms"].count(), b["Rms"].gpu_data, 2.0, b["Rms"].gpu_diff)
        cuda.invert(b["Rms"].count(), b["Rms"].gpu_diff, b["Rms"].gpu_diff, 0, 0, -1)
        cuda.mul(b["Rms1"].count(), b["Rms1"].gpu_diff, b["Rms"].gpu_diff, b["Rms"].gpu_diff)
        # x4 = sqrt(x2 + eps) -> dx2
        cuda.invert(b["Rms1"].count(), b["Rms"].gpu_data, b["Rms1"].gpu_diff, 0, 0, 1, 2)
        cuda.mul(b["Rms"].count(), b["Rms1"].gpu_diff, b["Rms"].gpu_diff, b["Rms"].gpu_diff)
        # x2 = mean(x1) -> dx1
        cuda.channel_duplicate(n, outer * channels, 1, inner, b["Rms"].gpu_diff, b["Rms1Full"].gpu_diff)
        cuda.scal(b["Rms1Full"].count(), 1.0 / inner, b["Rms1Full"].gpu_diff)
        # x1 = x^2 -> dx, and the sum of both paths
        cuda.scale(n, 2.0, bottom.gpu_data, b["Out"].gpu_diff)
        cuda.mul(n, b["Out"].gpu_diff, b["Rms1Full"].gpu_diff, b["Out"].gpu_diff)
        cuda.add(n, b["Out"].gpu_diff, bottom.gpu_diff, bottom.gpu_diff)


class ActivationLayer:
    """ReLU (MyCaffe/layers/ReLULayer.cs), GELU (MyCaffe.layers.gpt/layers.gpt/GeluLayer.cs, ``enable_bert_version``) or
    SiLU (MyCaffe/layers/SiLULayer.cs) as TransformerBlockLayer selects them (TransformerBlockLayer.cs:316-337)."""

    def __init__(self, cuda, kind="relu"):
        if kind not in ("relu", "gelu", "gelu_bert", "silu"):
            raise ValueError(kind)
        self.cuda, self.kind = cuda, kind
        self.blobX = Blob(cuda)     # GeluLayer.cs:84-87: the input is kept when the layer runs in place

    def Forward(self, bottom, top):
        top.ReshapeLike(bottom)
        n = bottom.count()
        hBottom = bottom.gpu_data
        if self.kind != "relu" and bottom.gpu_data == top.gpu_data:
            self.blobX.CopyFrom(bottom)
            hBottom = self.blobX.gpu_data
        if self.kind == "relu":
            self.cuda.relu_fwd(n, hBottom, top.gpu_data, 0.0)
        elif self.kind == "silu":
            self.cuda.silu_fwd(n, hBottom, top.gpu_data)
        else:
            self.cuda.gelu_fwd(n, hBottom, top.gpu_data, self.kind == "gelu_bert")

    def Backward(self, top, bottom):
        """ReLULayer.cs:203, GeluLayer.cs:110-121, SiLULayer.cs backward."""
        n = bottom.count()
        hBottomData = bottom.gpu_data
        if top.gpu_data == bottom.gpu_data:
            hBottomData = self.blobX.gpu_data
        if self.kind == "relu":
            self.cuda.relu_bwd(n, top.gpu_diff, top.gpu_data, bottom.gpu_diff, 0.0)
        elif self.kind == "silu":
            self.cuda.silu_bwd(n, top.gpu_diff, top.gpu_data, bottom.gpu_diff, hBottomData)
        else:
            self.cuda.gelu_bwd(n, top.gpu_diff, top.gpu_data, bottom.gpu_diff, hBottomData, self.kind == "gelu_bert")


class TransformerBlockLayer:
    """MyCaffe.layers.gpt/layers.gpt/TransformerBlockLayer.cs, block types CAUSAL_SELF_ATTENTION and ENCODER (setup
    :99-170, 252-340, forward :800-902): x + attn(ln1(x)), then + proj(act(fc(ln2(.)))).  The ENCODER type attends
    through MultiheadAttentionLayer(x_1, x_1, x_1, mask), the form the Llama models built by LlamaModelBuilder use
    (rotary embedding, key / value cache, "position" layer option).  Dropout is the identity at inference."""

    def __init__(self, cuda, heads, embed, block_size, activation="relu", bias_term=True, epsilon=1e-10,
                 enable_cuda_scaled_dot_product_attention=True, training=False, enable_llama_style_head=False, hidden_dim=0,
                 multiple_of=64, enable_layernorm_cuda_impl=True, fused_rmsnorm=None, block_type="causal_self_attention",
                 enable_key_value_cache=False):
        if block_type not in ("causal_self_attention", "encoder"):
            raise ValueError(block_type)
        self.cuda = cuda
        self.block_type = block_type
        self.llama = enable_llama_style_head
        if self.llama:
            # RMSNorm, rotary attention without bias, SiLU-gated MLP (TransformerBlockLayer.cs:86-98, 239-247, 860-875)
            # (the norms as single calls, unless fused_rmsnorm is False: then the layer's own chain)
            self.norm1 = RMSNormLayer(cuda, epsilon, True, fused_rmsnorm is not False)
            self.norm2 = RMSNormLayer(cuda, epsilon, True, fused_rmsnorm is not False)
            if hidden_dim == 0:
                hidden_dim = 2 * (4 * embed) // 3
                hidden_dim = multiple_of * ((hidden_dim + multiple_of - 1) // multiple_of)
        else:
            self.norm1 = LayerNormLayer(cuda, epsilon, enable_layernorm_cuda_impl)
            self.norm2 = LayerNormLayer(cuda, epsilon, enable_layernorm_cuda_impl)
            hidden_dim = hidden_dim or 4 * embed
        if block_type == "encoder":
            self.attn1 = MultiheadAttentionLayer(cuda, heads, embed, block_size, bias_term, enable_cuda_scaled_dot_product_attention,
                                                 enable_rotary_positional_embedding=self.llama,
                                                 enable_key_value_cache=enable_key_value_cache)
        else:
            self.attn1 = CausalSelfAttentionLayer(cuda, heads, embed, block_size, bias_term, enable_cuda_scaled_dot_product_attention,
                                                  enable_rotary_positional_embedding=self.llama, training=training)
        self.fc1 = InnerProductLayer(cuda, hidden_dim, bias_term, 2)
        self.fc2 = InnerProductLayer(cuda, hidden_dim, bias_term, 2) if self.llama else None
        self.proj = InnerProductLayer(cuda, embed, bias_term, 2)
        self.act = ActivationLayer(cuda, activation)
        if activation == "relu":
            # The gradient of a ReLU is 0 or 1: what moves a sum across zero in its last bit changes a gradient by its whole value
            # (8192 x 3072: some ten of 25 million, the weight gradient by 5e-4).  Neither mask is the better one - the sums of three
            # bf16 parts are off by less - but so the mask for given inputs stays what it has been with fp32 sums, and the gradient can be
            # compared with theirs.  All products behind it go the faster way (8192 x 768 into 12 heads: 2.5 ms, 2.4 without this).
            for layer in [self.fc1, self.attn1.c_proj] + ([self.attn1.c_attn] if block_type != "encoder" else
                                                          [self.attn1.c_attnQ, self.attn1.c_attnK, self.attn1.c_attnV]):
                layer.fp32_sums = True
        self.b = {n: Blob(cuda) for n in "Norm1 Attn1 X Norm2 Mlp1 Mlp2 Mlp3 MlpOut".split()}

    def Setup(self, bottom, p):
        """``p``: attn_weight, attn_bias, attn_proj_weight, attn_proj_bias (ENCODER type: wq, bq, wk, bk, wv, bv, wo, bo),
        fc_weight, fc_bias, proj_weight, proj_bias; Llama style also fc2_weight, rms1_weight, rms2_weight."""
        if self.block_type == "encoder":
            self.attn1.Setup(bottom, bottom, bottom, p)
        else:
            self.attn1.Setup(bottom, p["attn_weight"], p.get("attn_bias"), p["attn_proj_weight"], p.get("attn_proj_bias"))
        self.fc1.Setup(bottom, p["fc_weight"], p.get("fc_bias"))
        if self.llama:
            self.fc2.Setup(bottom, p["fc2_weight"], p.get("fc2_bias"))
            self.norm1.Setup(bottom, p.get("rms1_weight"))
            self.norm2.Setup(bottom, p.get("rms2_weight"))
        hidden = Blob(self.cuda, bottom.shape_[:2] + [self.fc1.N])
        self.proj.Setup(hidden, p["proj_weight"], p.get("proj_bias"))
        hidden.Dispose()

    def SetLayerOption(self, name, value):
        """Layer options reach the attention layer (TransformerBlockLayer.cs SetLayerOption override)."""
        if self.block_type == "encoder":
            self.attn1.SetLayerOption(name, value)

    def Forward(self, blobX, top, blobXMask=None):
        b, cuda = self.b, self.cuda
        nCount = blobX.count()
        self.norm1.Forward(blobX, b["Norm1"])
        if self.block_type == "encoder":
            self.attn1.Forward(b["Norm1"], b["Norm1"], b["Norm1"], blobXMask, b["Attn1"])
        else:
            self.attn1.Forward(b["Norm1"], b["Attn1"])
        self.norm2.ForwardAdd(blobX, b["Attn1"], b["X"], b["Norm2"])
        # the activation runs in place; those that need their input again get it in a blob of their own instead of a copy of it
        blobPre = b["Mlp1"] if self.act.kind == "relu" else self.act.blobX
        self.fc1.Forward(b["Norm2"], blobPre)
        blobMlp = b["Mlp1"]
        if self.llama:
            blobMlp = b["Mlp3"]
            self.fc2.Forward(b["Norm2"], b["Mlp2"])
            b["Mlp1"].ReshapeLike(blobPre)
            blobMlp.ReshapeLike(blobPre)
            if self.act.kind == "silu":
                cuda.SwigluForward(blobPre.count(), blobPre.gpu_data, b["Mlp2"].gpu_data, blobMlp.gpu_data)
            else:
                self.act.Forward(blobPre, b["Mlp1"])
                cuda.mul(blobMlp.count(), b["Mlp1"].gpu_data, b["Mlp2"].gpu_data, blobMlp.gpu_data)
        else:
            self.act.Forward(blobPre, blobMlp)
        self.proj.Forward(blobMlp, b["MlpOut"])
        top.ReshapeLike(blobX)
        cuda.add(nCount, b["X"].gpu_data, b["MlpOut"].gpu_data, top.gpu_data)

    def Backward(self, top, blobX):
        """TransformerBlockLayer.cs:924-1040, CAUSAL_SELF_ATTENTION block: top.gpu_diff -> blobX.gpu_diff.  The gradients of the
        two residuals are read where they are and added by the norms' calls."""
        if self.block_type != "causal_self_attention":
            raise NotImplementedError("backward is mirrored for the CAUSAL_SELF_ATTENTION block type")
        b, cuda = self.b, self.cuda
        self.proj.Backward(top, b["Mlp3"] if self.llama else b["Mlp1"])
        if self.llama:
            # gate: Mlp3 = act(fc1) * fc2
            n1 = b["Mlp1"].count()
            if self.act.kind == "silu":
                cuda.SwigluBackward(n1, self.act.blobX.gpu_data, b["Mlp2"].gpu_data, b["Mlp3"].gpu_diff, b["Mlp1"].gpu_diff, b["Mlp2"].gpu_diff)
            else:
                cuda.mul(n1, b["Mlp3"].gpu_diff, b["Mlp2"].gpu_data, b["Mlp1"].gpu_diff)
                cuda.mul(n1, b["Mlp3"].gpu_diff, b["Mlp1"].gpu_data, b["Mlp2"].gpu_diff)
                self.act.Backward(b["Mlp1"], b["Mlp1"])
            self.fc2.Backward(b["Mlp2"], b["Norm2"])
        else:
            self.act.Backward(b["Mlp1"], b["Mlp1"])
        self.fc1.Backward(b["Mlp1"], b["Norm2"], self.llama)
        self.norm2.BackwardAdd(b["Norm2"], b["X"], top.gpu_diff)
        self.attn1.Backward(b["X"], b["Norm1"])
        self.norm1.BackwardAdd(b["Norm1"], blobX, b["X"].gpu_diff)
