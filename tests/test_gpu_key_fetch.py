"""The kernel-level calls read the key and H on the device's stream order: from
aligned and unaligned device memory, the last bytes of an allocation, pinned
host memory (copied instead of fetched), behind earlier work that outlasts the
host's spin, on a side stream, and after the same buffers took a new key.
Against OpenSSL, bit-exact."""
import struct

import numpy as np
import pytest
import torch

import secure_infer_amd as si
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _dev(b, off=0):
    a = np.frombuffer(bytes(b), np.uint8).copy()
    big = torch.zeros(off + a.size, dtype=torch.uint8, device=DEV)
    big[off:] = torch.from_numpy(a).to(DEV)
    return big[off:]


@pytest.mark.parametrize("where", ["aligned", "unaligned", "allocation_end", "pinned_host", "late", "side_stream"])
def test_key_and_h_are_read_in_stream_order(where):
    rng = np.random.default_rng(41)
    n = 5001
    stream = torch.cuda.Stream() if where == "side_stream" else torch.cuda.current_stream()
    off = {"unaligned": 3, "allocation_end": 512 - 16}.get(where, 0)
    dk, dh = _dev(bytes(16), off), _dev(bytes(16), off)
    if where == "pinned_host":
        dk, dh = (torch.zeros(16, dtype=torch.uint8, pin_memory=True) for _ in range(2))
    ct = torch.zeros(n, dtype=torch.uint8, device=DEV)
    tag = torch.zeros(16, dtype=torch.uint8, device=DEV)
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
            si.gcm_encrypt_tag(dp, dk, dh, ct, tag, struct.unpack(">III", iv12) + (2,), da)
        torch.cuda.synchronize()
        assert np.array_equal(ct.cpu().numpy(), np.frombuffer(bytes(want_ct), np.uint8))
        assert np.array_equal(tag.cpu().numpy(), np.frombuffer(bytes(want_tag), np.uint8))
