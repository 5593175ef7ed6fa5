"""The native shortcuts of the argument checks (host/launch.cpp kv_valid, attend_valid) against the checks themselves
(cache_fp8._refusal, sage_kv._check): a shortcut may only pass what the check passes, over every single broken
requirement. The tensors are on the CPU, where the device requirement of the store alone differs."""

import itertools

import pytest
import torch

FP8 = torch.float8_e4m3fn


def _call():
    kv = lambda n: torch.zeros(1, n, 2, 128, dtype=torch.bfloat16)
    cache = lambda: torch.zeros(1, 12, 2, 128).to(FP8)
    return dict(Q=kv(4), cache_k=cache(), cache_ks=torch.ones(1, 12, 2, 1), cache_v=cache(),
                cache_vs=torch.ones(1, 12, 2, 1), at=8, K=kv(4), V=kv(4))


BREAKS = {
    "fine": lambda t: t,
    "fp32": lambda t: t.float(),
    "fp16": lambda t: t.half(),
    "uint8": lambda t: t.to(torch.uint8),
    "strided rows": lambda t: torch.cat([t, t], -1)[..., ::2],
    "head stride": lambda t: torch.cat([t, t], -1)[..., :t.shape[-1]],
    "token stride": lambda t: torch.cat([t, t], 1)[:, ::2],
    "one head": lambda t: t[:, :, :1],
    "one token fewer": lambda t: t[:, 1:].contiguous(),
    "three dims": lambda t: t[0],
    "batch 2": lambda t: torch.cat([t, t]),
    "half the channels": lambda t: t[..., :64].contiguous(),
    "empty": lambda t: t[:, :0],
}


def _passes(check, *args):
    try:
        return check(*args) is None
    except (TypeError, ValueError, IndexError):
        return False


@pytest.mark.parametrize("at", [-1, 0, 8, 9, 12, 13])
def test_the_native_checks_pass_only_what_the_checks_pass(at):
    from wdl import _lib, cache_fp8, sage_kv

    host, passed = _lib.host(), 0
    for name, how in itertools.product(("Q", "cache_k", "cache_ks", "cache_v", "cache_vs", "K", "V"), BREAKS):
        c = dict(_call(), at=at)
        c[name] = BREAKS[how](c[name])
        order = (c["Q"], c["cache_k"], c["cache_ks"], c["cache_v"], c["cache_vs"], c["at"], c["K"], c["V"])
        try:
            native = host.attend_valid(*order)
        except IndexError:
            native = False
        want = _passes(sage_kv._check, *order)
        assert native <= want, (name, how)
        passed += native
        assert native == want or how != "fine", name
        store = (c["K"], c["V"], c["cache_k"], c["cache_ks"], c["cache_v"], c["cache_vs"], at)
        assert not host.kv_valid(*store)  # on the CPU: refused there by the device alone
        assert cache_fp8.refusal(*store) is not None
    assert (passed > 0) == (0 <= at <= 12)


@pytest.mark.gpu
@pytest.mark.parametrize("at", [-1, 0, 8, 9])
def test_the_native_store_check_passes_only_what_the_check_passes(gpu, at):
    from wdl import _lib, cache_fp8

    host = _lib.host()
    for name, how in itertools.product(("cache_k", "cache_ks", "cache_v", "cache_vs", "K", "V"), BREAKS):
        c = {key: v.cuda() if isinstance(v, torch.Tensor) else v for key, v in _call().items()}
        c[name] = BREAKS[how](c[name])
        store = (c["K"], c["V"], c["cache_k"], c["cache_ks"], c["cache_v"], c["cache_vs"], at)
        assert host.kv_valid(*store) == (cache_fp8._refusal(*store) is None), (name, how)


FAR = [2 ** 63 - 1, 2 ** 63 - 4, 2 ** 63, 2 ** 64 + 8, -2 ** 63, -2 ** 70]


@pytest.mark.parametrize("at", FAR + [9, -1])
def test_offsets_whose_end_does_not_fit_64_bits_are_refused(at):
    """at + n beyond int64 is past the cache, not a small negative number, and an offset that no int64 holds is the
    ValueError of any other offset outside the cache: in the store's and the attention's checks (the store's over
    tensors that only claim to be on a GPU) and in the C entry, whose pointers are null here."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from wdl import _lib, cache_fp8, sage_kv

    c = _call()
    with pytest.raises(ValueError, match="at outside the cache"):
        order = (c["Q"], c["cache_k"], c["cache_ks"], c["cache_v"], c["cache_vs"])
        sage_kv.attend(*order, at if at != 9 else 13, c["K"], c["V"])
    with FakeTensorMode():
        f = {name: torch.empty(t.shape, dtype=t.dtype, device="cuda:0") for name, t in c.items() if name != "at"}
        store = [f[name] for name in ("K", "V", "cache_k", "cache_ks", "cache_v", "cache_vs")]
        assert _lib.host().kv_valid(*store, 8) and cache_fp8.refusal(*store, 8) is None
        kind, message = cache_fp8.refusal(*store, at)
        assert kind is ValueError and "do not fit a cache of 12 rows" in message
    if -2 ** 63 <= at < 2 ** 63:
        lib, strides = _lib.library(), _lib.i64s([1, 1, 1, 1])
        assert lib.wdl_kv_append_fp8(None, 2, strides, None, 2, strides, 1, 4, 1, 8, None, None, None, None, 12, at, None) == 1
        assert b"exceeds capacity" in lib.wdl_last_error()
