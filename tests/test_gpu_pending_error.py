"""A HIP error that an earlier call left on the thread (here: a device that does
not exist) is not the library's: each launch reports its own status, so the
calls succeed with the right bytes and the error stays with its owner."""
import ctypes as ct
import struct

import numpy as np
import pytest
import torch

import secure_infer_amd as si
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"
KEY, SALT = bytes(range(16)), b"salt"


@pytest.fixture
def pending():
    """Leaves a HIP error on this thread; takes it off afterwards, where it must
    still be."""
    with open("/proc/self/maps") as f:
        hip = ct.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))
    torch.cuda.synchronize()
    left = []

    def leave():
        left.append(hip.hipSetDevice(1000))
        assert left[0] != 0
    yield leave
    assert hip.hipGetLastError() == left[0] and hip.hipGetLastError() == 0


def _dev(b):
    return torch.from_numpy(np.frombuffer(bytes(b), np.uint8).copy()).to(DEV)


def _record_calls(n, key, seed):
    """Device buffers of one record's seal and open, and the expected results."""
    rng = np.random.default_rng(seed)
    iv12, aad, pt = rng.bytes(12), rng.bytes(20), rng.bytes(n)
    want_ct, want_tag = O.ossl_gcm_encrypt(key, iv12, aad, pt)
    s = dict(key=_dev(key), h=_dev(O.hash_subkey(key)), pt=_dev(pt), aad=_dev(aad), ct=_dev(bytes(n)),
             tag=_dev(bytes(16)), back=_dev(bytes(n)), status=torch.zeros(4, dtype=torch.int32, device=DEV))
    iv = struct.unpack(">III", iv12) + (2,)
    seal = lambda: si.gcm_encrypt_tag(s["pt"], s["key"], s["h"], s["ct"], s["tag"], iv, s["aad"])
    opened = lambda: si.gcm_decrypt_verify(s["ct"], s["key"], s["h"], s["tag"], s["back"], s["status"], iv, s["aad"])

    def check():
        assert s["ct"].cpu().numpy().tobytes() == bytes(want_ct)
        assert s["tag"].cpu().numpy().tobytes() == bytes(want_tag)
        assert s["back"].cpu().numpy().tobytes() == pt and int(s["status"][0]) == 1
    return seal, opened, check


def test_single_records_of_two_keys_on_two_streams(pending):
    streams = [torch.cuda.Stream() for _ in range(2)]
    calls = [_record_calls(n, bytes([7 + i]) * 16, 60 + i) for i, n in enumerate((100003, 4096))]
    torch.cuda.synchronize()
    pending()
    for _ in range(3):
        for st, (seal, opened, _check) in zip(streams, calls):
            with torch.cuda.stream(st):
                seal()
                opened()
    for st in streams:
        st.synchronize()
    # (the copies back below go through calls that do not read the last error)
    for _seal, _opened, check in calls:
        check()


@pytest.mark.parametrize("bits,strict", [(0, False), (0, True), (4, False), (8, False)])
def test_layers_sealed_and_reloaded(pending, bits, strict):
    heads, dim, nb, layer = 2, 64, 3, 1
    n = si.codec_width(bits, heads, dim) if bits else 128 * heads * dim * 2
    sess = si.GcmSession(KEY, SALT, 0, max_record_bytes=n)
    g = torch.Generator(device=DEV).manual_seed(5)
    src = [torch.randn((nb, 128, heads, dim), generator=g, device=DEV).to(torch.bfloat16) for _ in range(2)]
    dst = [torch.zeros_like(x) for x in src]
    ref = [torch.zeros_like(x) for x in src]
    slots = torch.arange(nb, device=DEV).repeat(2)
    wire = torch.zeros((2 * nb, si.wire_stride(n)), dtype=torch.uint8, device=DEV)
    fail = torch.zeros(1, dtype=torch.int32, device=DEV)
    staging = torch.zeros(2 * nb * si.wire_tag_offset(n), dtype=torch.uint8, device=DEV) if bits else None
    how = dict(codec_bits=bits, heads=heads, head_dim=dim, layer=layer, staging=staging, fail_count=fail)
    put = sess.prepare_writeback_layer(wire, n, 2 * nb, nb, *src, slots, ticket_base=1, **how)
    plain = sess.prepare_reload_layer(wire, n, 2 * nb, nb, *ref, slots, ticket_base=1, **how)
    get = sess.prepare_reload_layer(wire, n, 2 * nb, nb, *dst, slots, ticket_base=1, verify_before_release=strict, **how)
    put.launch()
    plain.launch()
    wire_ref = wire.clone()
    wire.zero_()
    torch.cuda.synchronize()
    pending()
    put.launch()
    get.launch()
    torch.cuda.current_stream().synchronize()
    off = si.wire_tag_offset(n)
    a, b = wire.cpu(), wire_ref.cpu()
    assert torch.equal(a[:, :off + 16], b[:, :off + 16])
    assert torch.equal(a[:, off + 16:off + 20].contiguous().view(torch.int32), torch.ones((2 * nb, 1), dtype=torch.int32))
    for x, y in zip(dst, ref):
        assert torch.equal(x.cpu(), y.cpu())
    if not bits:
        assert torch.equal(ref[0].cpu(), src[0].cpu()) and torch.equal(ref[1].cpu(), src[1].cpu())
    assert int(fail.cpu()) == 0
