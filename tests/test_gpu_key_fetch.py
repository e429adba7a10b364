"""The kernel-level calls read the key and H on the device's stream order: from
aligned and unaligned device memory, the end of a tensor and the last 16 bytes
of a device allocation, pinned host memory (copied instead of fetched), behind
earlier work that outlasts the host's spin, on a side stream, after the same
buffers took a new key, and from threads with their own streams and keys.  The
library's count of fetches tells a fetched key from a copied one.  Against
OpenSSL, bit-exact."""
import ctypes as ct
import struct
import threading

import numpy as np
import pytest
import torch

import secure_infer_amd as si
from oracle import oracle as O
from secure_infer_amd import _lib

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _dev(b, off=0):
    a = np.frombuffer(bytes(b), np.uint8).copy()
    big = torch.zeros(off + a.size, dtype=torch.uint8, device=DEV)
    big[off:] = torch.from_numpy(a).to(DEV)
    return big[off:]


@pytest.mark.parametrize("where", ["aligned", "unaligned", "tensor_end", "pinned_host", "late", "side_stream"])
def test_key_and_h_are_read_in_stream_order(where):
    rng = np.random.default_rng(41)
    n = 5001
    stream = torch.cuda.Stream() if where == "side_stream" else torch.cuda.current_stream()
    off = {"unaligned": 3, "tensor_end": 512 - 16}.get(where, 0)
    dk, dh = _dev(bytes(16), off), _dev(bytes(16), off)
    if where == "pinned_host":
        dk, dh = (torch.zeros(16, dtype=torch.uint8, pin_memory=True) for _ in range(2))
    out = torch.zeros(n, dtype=torch.uint8, device=DEV)
    tag = torch.zeros(16, dtype=torch.uint8, device=DEV)
    fetches = _lib.load().secure_infer_test_key_fetches()
    for _ in range(3):  # the same buffers, another key each time
        key, iv12, aad, pt = rng.bytes(16), rng.bytes(12), rng.bytes(20), rng.bytes(n)
        want_ct, want_tag = O.ossl_gcm_encrypt(key, iv12, aad, pt)
        newk, newh, dp, da = _dev(key), _dev(O.hash_subkey(key)), _dev(pt), _dev(aad)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            if where == "late":
                torch.cuda._sleep(20_000_000)  # the key arrives after the host began to wait
            dk.copy_(newk)
            dh.copy_(newh)
            si.gcm_encrypt_tag(dp, dk, dh, out, tag, struct.unpack(">III", iv12) + (2,), da)
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), np.frombuffer(bytes(want_ct), np.uint8))
        assert np.array_equal(tag.cpu().numpy(), np.frombuffer(bytes(want_tag), np.uint8))
    assert _lib.load().secure_infer_test_key_fetches() - fetches == (0 if where == "pinned_host" else 3)


def test_key_and_h_in_the_last_bytes_of_an_allocation():
    """The key and H end their own device allocations, where the range check of a
    fetch is at its limit."""
    lib = _lib.load()
    with open("/proc/self/maps") as f:
        hip = ct.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))
    rng = np.random.default_rng(42)
    off, n = 512, 5001
    key, iv12, pt = rng.bytes(16), rng.bytes(12), rng.bytes(n)
    want_ct, want_tag = O.ossl_gcm_encrypt(key, iv12, b"", pt)
    dp, out, tag = _dev(pt), _dev(bytes(n)), _dev(bytes(16))
    torch.cuda.synchronize()
    owned, at = [], []
    try:
        for b in (key, bytes(O.hash_subkey(key))):
            p, base, size = ct.c_void_p(), ct.c_void_p(), ct.c_size_t()
            assert hip.hipMalloc(ct.byref(p), ct.c_size_t(off + 16)) == 0
            owned.append(p)
            assert hip.hipMemGetAddressRange(ct.byref(base), ct.byref(size), p) == 0
            assert base.value == p.value and size.value == off + 16
            at.append(ct.c_void_p(p.value + off))
            assert hip.hipMemcpy(at[-1], b, ct.c_size_t(16), 1) == 0  # host to device
        fetches = lib.secure_infer_test_key_fetches()
        assert lib.secure_infer_gpu_gcm_encrypt_tag_do(
            ct.c_void_p(torch.cuda.current_stream().cuda_stream), ct.c_void_p(dp.data_ptr()), *at,
            ct.c_void_p(out.data_ptr()), ct.c_void_p(tag.data_ptr()), n, *struct.unpack(">III", iv12), 2, None, 0) == 0
        torch.cuda.synchronize()
        assert lib.secure_infer_test_key_fetches() == fetches + 1
    finally:
        for p in owned:
            hip.hipFree(p)
    assert out.cpu().numpy().tobytes() == bytes(want_ct) and tag.cpu().numpy().tobytes() == bytes(want_tag)


def test_threads_with_their_own_streams_and_keys():
    nthreads, calls, n = 4, 25, 5001
    rng = np.random.default_rng(43)
    jobs = []
    for _ in range(nthreads):
        key, iv12, pt = rng.bytes(16), rng.bytes(12), rng.bytes(n)
        want = O.ossl_gcm_encrypt(key, iv12, b"", pt)
        jobs.append(dict(key=_dev(key), h=_dev(O.hash_subkey(key)), iv=struct.unpack(">III", iv12) + (2,), pt=_dev(pt),
                         want=want, out=[_dev(bytes(n)) for _ in range(calls)],
                         tag=[_dev(bytes(16)) for _ in range(calls)], stream=torch.cuda.Stream()))
    torch.cuda.synchronize()
    fetches = _lib.load().secure_infer_test_key_fetches()
    errors = []

    def work(j):
        try:
            with torch.cuda.stream(j["stream"]):
                for o, t in zip(j["out"], j["tag"]):
                    si.gcm_encrypt_tag(j["pt"], j["key"], j["h"], o, t, j["iv"], None)
            j["stream"].synchronize()
        except Exception as e:  # reported by the main thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(j,)) for j in jobs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    assert _lib.load().secure_infer_test_key_fetches() == fetches + nthreads * calls
    for j in jobs:
        for o, t in zip(j["out"], j["tag"]):
            assert o.cpu().numpy().tobytes() == bytes(j["want"][0]) and t.cpu().numpy().tobytes() == bytes(j["want"][1])
