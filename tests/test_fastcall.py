"""The Python binding's call extension (no GPU): the parameter structures that it fills
are those of the ctypes builders, and bad tensors and arguments raise."""
import ctypes

import pytest


class Fake:
    """A tensor's attributes, on a GPU that is not there."""

    def __init__(self, dtype, shape, ptr, cuda=True, stride=None):
        self.dtype, self.shape, self.is_cuda, self._ptr, self._stride = dtype, tuple(shape), cuda, ptr, stride

    def data_ptr(self):
        return self._ptr

    def stride(self, dim=None):
        s, out = 1, []
        for n in reversed(self.shape):
            out.insert(0, s)
            s *= n
        if self._stride:
            out[0] = self._stride
        return tuple(out) if dim is None else out[dim]

    def numel(self):
        n = 1
        for x in self.shape:
            n *= x
        return n

    def element_size(self):
        return self.dtype.itemsize


@pytest.fixture
def calls(vkv):
    """The extension bound to entry points that keep the structures they are given;
    bound to the library again afterwards."""
    import torch
    fast, got = vkv._calls(), {}
    kinds = {"append": (vkv.AppendParams,), "decode": (vkv.DecodeParams,),
             "decode_append": (vkv.AppendParams, vkv.DecodeParams), "prefill": (vkv.PrefillParams,),
             "rope": (vkv.RopeAppendParams,)}
    keep = []
    for name, types in kinds.items():
        def entry(*args, name=name, types=types):
            got[name] = [bytes(ctypes.string_at(p, ctypes.sizeof(t))) for p, t in zip(args, types)] + [args[-1]]
            return 7
        f = ctypes.CFUNCTYPE(ctypes.c_int, *([ctypes.c_void_p] * (len(types) + 1)))(entry)
        keep.append(f)
    fast.bind(tuple(ctypes.cast(f, ctypes.c_void_p).value for f in keep),
              (torch.float32, torch.float16, torch.uint8, torch.float8_e4m3fn), (lambda: 0, lambda _: 0x55))
    yield fast, got
    vkv._bind_fastcall(vkv.load())


def _tensors(torch, fp8=False, S=3, H=14, Hkv=2, D=64, N=20, bs=16, MB=5):
    f16, i32, f32 = torch.float16, torch.int32, torch.float32
    kv = torch.uint8 if fp8 else f16
    t = dict(out=Fake(f16, (S, H, D), 1 << 12), q=Fake(f16, (S, H, D), 2 << 12, stride=H * D + 8),
             kc=Fake(kv, (N, bs, Hkv, D), 3 << 12), vc=Fake(kv, (N, bs, Hkv, D), 4 << 12),
             bt=Fake(i32, (S, MB), 5 << 12), cl=Fake(i32, (S,), 6 << 12),
             key=Fake(f16, (S, Hkv, D), 7 << 12, stride=1000), value=Fake(f16, (S, Hkv, D), 8 << 12),
             slots=Fake(i32, (S,), 9 << 12), ws=Fake(i32, (4096,), 10 << 12), qsl=Fake(i32, (S + 1,), 11 << 12),
             wl=Fake(i32, (64,), 12 << 12), cs=Fake(f32, (4096, D // 2, 2), 13 << 12))
    t["ks"] = Fake(f32, (N, bs, Hkv), 14 << 12) if fp8 else None
    t["vs"] = Fake(f32, (N, bs, Hkv), 15 << 12) if fp8 else None
    return t


@pytest.mark.parametrize("fp8", [False, True])
def test_structures(vkv, calls, fp8):
    import torch
    fast, got = calls
    t = _tensors(torch, fp8)
    ap = bytes(vkv.append_params(t["key"], t["value"], t["kc"], t["vc"], t["slots"], t["ks"], t["vs"]))
    assert fast.append(t["key"], t["value"], t["kc"], t["vc"], t["slots"], t["ks"], t["vs"], 0x33) == 7
    assert got["append"] == [ap, 0x33]
    for max_ctx, acc, size, ws in ((None, False, 0, None), (70, True, 64, t["ws"])):
        dp = bytes(vkv.decode_params(t["out"], t["q"], t["kc"], t["vc"], t["bt"], t["cl"], 0.125, t["ks"], t["vs"],
                                     max_ctx, acc, size, ws))
        args = (t["out"], t["q"], t["kc"], t["vc"], t["bt"], t["cl"], 0.125, t["ks"], t["vs"], max_ctx, acc, size, ws)
        assert fast.decode(*args, None) == 7
        assert got["decode"] == [dp, 0x55]  # (None: the current stream)
        assert fast.decode_append(*args, t["key"], t["value"], t["slots"], 0x33) == 7
        assert got["decode_append"] == [ap, dp, 0x33]
    pp = vkv.prefill_params(t["out"], t["q"], t["kc"], t["vc"], t["bt"], t["cl"], t["qsl"], 2, 0.125, t["ks"], t["vs"],
                            90, t["ws"], True)
    args = (t["out"], t["q"], t["kc"], t["vc"], t["bt"], t["cl"], t["qsl"], 2, 0.125, t["ks"], t["vs"], 90, t["ws"], True)
    assert fast.prefill(*args, None, 0x33) == 7
    assert got["prefill"] == [bytes(pp), 0x33]
    pp.work_list, pp.work_list_words = t["wl"].data_ptr(), 64
    assert fast.prefill(*args, t["wl"], 0x33) == 7
    assert got["prefill"] == [bytes(pp), 0x33]
    assert fast.rope(t["q"], t["key"], t["value"], t["cs"], None, 11, t["kc"], t["vc"], t["slots"], t["ks"], t["vs"], 0x33) == 7
    rp = vkv.RopeAppendParams.from_buffer_copy(got["rope"][0])
    assert (rp.query, rp.key, rp.value, rp.cos_sin, rp.positions) == (2 << 12, 7 << 12, 8 << 12, 13 << 12, None)
    assert (rp.query_stride, rp.key_stride, rp.value_stride) == (14 * 64 + 8, 1000, 2 * 64)
    assert (rp.start_pos, rp.max_position, rp.num_tokens, rp.num_heads, rp.num_kv_heads, rp.head_dim) == (11, 4096, 3, 14, 2, 64)
    assert (rp.block_size, rp.num_blocks, rp.src_dtype, rp.cache_dtype) == (16, 20, 1, 2 if fp8 else 1)


def test_errors(vkv, calls):
    """Nothing reaches the library: a tensor that is not on the GPU, the wrong rank or
    dtype, arguments of the wrong number or kind."""
    import torch
    fast, got = calls
    t = _tensors(torch)
    decode = [t["out"], t["q"], t["kc"], t["vc"], t["bt"], t["cl"], 0.125, None, None, None, False, 0, None, 0]
    for at in (0, 1, 2, 3, 4, 5):
        bad = Fake(decode[at].dtype, decode[at].shape, 64, cuda=False)
        with pytest.raises(ValueError, match="GPU"):
            fast.decode(*decode[:at], bad, *decode[at + 1:])
    with pytest.raises(ValueError, match="dimensions"):
        fast.decode(Fake(torch.float16, (3, 14 * 64), 64), *decode[1:])
    with pytest.raises(ValueError, match="dimensions"):
        fast.decode(*decode[:2], Fake(torch.float16, (20, 16, 128), 64), *decode[3:])
    with pytest.raises(IndexError):
        fast.decode(*decode[:4], Fake(torch.int32, (3,), 64), *decode[5:])
    with pytest.raises(TypeError, match="dtype"):
        fast.decode(Fake(torch.bfloat16, (3, 14, 64), 64), *decode[1:])
    with pytest.raises(TypeError, match="dtype"):
        fast.decode(*decode[:2], Fake(torch.int64, (20, 16, 2, 64), 64), *decode[3:])
    with pytest.raises(TypeError, match="arguments"):
        fast.decode(*decode[:-1])
    with pytest.raises(TypeError):
        fast.decode(*decode[:6], "scale", *decode[7:])
    with pytest.raises(TypeError):
        fast.decode(*decode[:9], 1.5, *decode[10:])
    with pytest.raises(AttributeError):
        fast.decode(None, *decode[1:])
    with pytest.raises(AttributeError):
        fast.append(t["key"], t["value"], [], t["vc"], t["slots"], None, None, 0)
    for name, n in (("append", 8), ("decode_append", 17), ("prefill", 16), ("rope", 12)):
        with pytest.raises(TypeError, match="arguments"):
            getattr(fast, name)(*[None] * (n + 1))
    assert not got
