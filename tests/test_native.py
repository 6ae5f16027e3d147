"""The CPython binding of the hot entry points (csrc/bind/native.cpp) and the one-copy upload of a batch."""
import ctypes
import types

import pytest
import torch

from aici_amd import _lib, _native, kernels, paged


def test_arguments_are_checked_before_the_call():
    x = torch.zeros((2, 16), dtype=torch.bfloat16)
    with pytest.raises(_lib.HipAttnError, match="out: expected a GPU tensor, got one on cpu"):
        _native.silu_and_mul(x, x)
    with pytest.raises(_lib.HipAttnError, match="input: unsupported dtype torch.bool"):
        _native.gelu_new(None, x.bool())
    with pytest.raises(TypeError, match="weight: expected a torch.Tensor or None, got int"):
        _native.rms_norm(None, None, 3, 1e-5)
    with pytest.raises(TypeError, match="takes 4 arguments"):
        _native.rms_norm(x)
    with pytest.raises(_lib.HipAttnError, match="hipattn_reshape_and_cache: .*NULL"):
        _native.reshape_and_cache(None, None, None, None, None)


@pytest.mark.parametrize("S,Hkv,longest,d", [(1000, 1, 1024, 128), (1000, 1, 1024, 80), (1023, 1, 513, 128), (500, 2, 1024, 112), (250, 4, 1024, 96)])
def test_static_scratch_holds_what_contexts_of_1024_tokens_need(S, Hkv, longest, d):
    """Sixteen query heads per kv head: the partitions of that many contexts would not fit the built-in array."""
    assert kernels.paged_attention_workspace_size(S, 16 * Hkv, Hkv, d, 16, longest, torch.bfloat16) <= 16 << 20


@pytest.mark.parametrize("fn", ["hipattn_linear_workspace_size", "hipattn_linear_rms_norm_workspace_size"])
@pytest.mark.parametrize("shape", [(4096, 14336), (6144, 4096), (16, 256), (512, 512)])
def test_linear_workspace_depends_on_the_weight_alone(fn, shape):
    """An engine asks once, with whatever batch it has then.  (Descriptors of host tensors do: nothing is read.)"""
    desc = lambda t: kernels._desc(t, device=False)
    sizes = set()
    for m in (1, 16, 17, 128):
        n = ctypes.c_int64(-1)
        _lib.call(fn, desc(torch.empty((m, shape[1]), dtype=torch.bfloat16)), desc(torch.empty(shape, dtype=torch.bfloat16)),
                  ctypes.byref(n))
        sizes.add(n.value)
    assert len(sizes) == 1 and sizes.pop() > 0


@pytest.mark.parametrize("mapping", [{-1: [0]}, {0: [-1]}, {4: [0]}, {0: [1, 4]}, {0: [2 ** 31]}, {-(2 ** 40): [1]}])
def test_copy_blocks_refuses_blocks_outside_the_caches(mapping):
    """Before anything is launched (and before the caches are looked at: they need not be on a GPU here)."""
    kc, vc = torch.zeros((4, 2, 1, 16, 8), dtype=torch.float16), torch.zeros((4, 2, 8, 16), dtype=torch.float16)
    with pytest.raises(_lib.HipAttnError, match="out of range"):
        kernels.copy_blocks([kc], [vc], mapping)


@pytest.mark.gpu
@pytest.mark.parametrize("mapping", [{-1: [0]}, {0: [-1]}, {4: [0]}, {0: [1, 4]}, {0: [2 ** 31]}, {-(2 ** 40): [1]}])
def test_copy_blocks_refuses_blocks_outside_caches_on_the_device(device, mapping):
    """The binding's own look at the pairs, before any launch."""
    kc = torch.zeros((4, 2, 1, 16, 8), dtype=torch.float16, device=device)
    vc = torch.zeros((4, 2, 8, 16), dtype=torch.float16, device=device)
    with pytest.raises(_lib.HipAttnError, match="out of range, the caches have 4 blocks"):
        kernels.copy_blocks([kc], [vc], mapping)


@pytest.mark.parametrize("pair,message", [((-1, 0), "pair 1 has block -1"), ((0, -5), "pair 1 has block -5"),
                                          ((0, 2 ** 31), "does not fit 32 bits")])
def test_copy_blocks_host_refuses_bad_numbers_before_any_launch(pair, message):
    ptr = (ctypes.c_void_p * 1)(4096)  # never read: the numbers are looked at first
    with pytest.raises(_lib.HipAttnError, match=message):
        _lib.call("hipattn_copy_blocks_host", ptr, ptr, 1, (ctypes.c_int64 * 4)(0, 1, *pair), 2, 4096, None)


@pytest.mark.parametrize("slots", [torch.tensor([3, 1], dtype=d) for d in (torch.int8, torch.int16, torch.uint8, torch.int64)]
                         + [torch.tensor([3, 0, 1], dtype=torch.int32)[::2], torch.tensor([3, 1], dtype=torch.int32)])
def test_slots_of_every_integer_type_reach_the_kernel(slots, monkeypatch):
    seen = []
    monkeypatch.setattr(kernels, "_native", types.SimpleNamespace(reshape_and_cache=lambda *a: seen.append(a[4])))
    kernels.reshape_and_cache(None, None, None, None, slots)
    (got,) = seen
    assert got.dtype in (torch.int32, torch.int64) and got.is_contiguous() and got.tolist() == [3, 1]
    assert got is slots or slots.dtype not in (torch.int32, torch.int64) or not slots.is_contiguous()


def _batch(lens):
    alloc = paged.BlockAllocator(16, 256)
    b = paged.BatchInfoBuilder(16, 4096, 1)
    for sid, (n, computed) in enumerate(lens, start=1):
        alloc.alloc_seq(sid, n)
        b.sched_out(alloc, sid, list(range(n)), computed)
    return b.finish()


def test_batch_upload_waits_for_its_copy(monkeypatch):
    """No array may still be on its way when `to` returns: a caller uploads on one stream and runs the model on another."""
    asked = []
    empty, copy_ = torch.empty, torch.Tensor.copy_
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, device=None, **kw: empty(*a, **kw))  # there is no GPU here
    monkeypatch.setattr(torch.Tensor, "to", lambda t, *a, **kw: asked.append((a, kw)) or t.clone())
    monkeypatch.setattr(torch.Tensor, "copy_", lambda t, src, *a, **kw: asked.append((a, kw)) or copy_(t, src))
    host = _batch([(37, 0), (5, 4)])
    got = host.to("cuda")
    (args, kw), = asked
    assert not kw.get("non_blocking", False) and not any(a is True for a in args)
    for name, want in host.__dict__.items():
        if isinstance(want, torch.Tensor):
            assert torch.equal(getattr(got, name), want), name


@pytest.mark.gpu
def test_batch_uploaded_behind_queued_work_is_there_for_other_streams(device):
    host = _batch([(37, 0), (5, 4), (300, 299)])
    a = torch.randn((4096, 4096), device=device)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(20):  # some milliseconds in front of the upload
            a @ a
        dev = host.to(device)
    for name, want in host.__dict__.items():  # read on the default stream, which waits for nothing
        if isinstance(want, torch.Tensor):
            assert torch.equal(getattr(dev, name).clone().cpu(), want), name
    side.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[(1, 0)], [(37, 0), (5, 4), (100, 99)], [(64, 17)], [(3, 2), (300, 299)]])
def test_batch_upload_keeps_every_array(device, lens):
    host = _batch(lens)
    for _ in range(3):  # the staging buffer is reused
        dev = host.to(device)
        for name, want in host.__dict__.items():
            got = getattr(dev, name)
            if isinstance(want, torch.Tensor):
                assert got.is_cuda and got.dtype == want.dtype and got.shape == want.shape
                assert got.data_ptr() % 16 == 0 or got.numel() == 0
                assert torch.equal(got.cpu(), want), name
            else:
                assert got == want
