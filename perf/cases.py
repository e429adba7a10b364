"""Performance cases of the authenticated KV data plane.

Each case is one call sequence that a serving program makes: a layer of
records reloaded into the paged cache or written back from it (bf16 blocks or
int8 / int4 packets, fused or verify-before-release), one record through the
kernel-level calls, or a layer stored to host memory and reloaded from it.
Shapes come from bench.py's workloads and from the reference's causal group of
16 blocks; one block is 128 tokens of one kind (K or V), and a layer of
`blocks` blocks has 2 * blocks records.  Every output is bytes or whole status
words, so results compare exactly.
"""
import struct

import numpy as np
import torch

import secure_infer_amd as si

TOKENS = 128   # tokens of one block
GROUP = 64     # codec group
AAD = 64


def listed():
    return [
        # One block of an 8 x 128 model becoming resident: the smallest
        # layer call, where launches and latency count.
        dict(name="reload_bf16_block", op="reload", heads=8, dim=128, blocks=1, bits=0, strict=False, ivs=False,
             tampered=0),
        # One causal group of 16 blocks, the unit a layer's reload is
        # submitted in.
        dict(name="reload_bf16_group", op="reload", heads=8, dim=128, blocks=16, bits=0, strict=False, ivs=False,
             tampered=0),
        # A 6,144-token prefix of an 8 x 128 model: the headline workload.
        dict(name="reload_bf16_8b", op="reload", heads=8, dim=128, blocks=48, bits=0, strict=False, ivs=True,
             tampered=0),
        # One tensor-parallel rank (1 head, 32-KiB records), a long prefix.
        dict(name="reload_bf16_tp_rank", op="reload", heads=1, dim=128, blocks=256, bits=0, strict=False, ivs=True,
             tampered=0),
        # int8 packets, 8,192 tokens.
        dict(name="reload_int8_8b", op="reload", heads=8, dim=128, blocks=64, bits=8, strict=False, ivs=True,
             tampered=0),
        # int4 packets of a 4 x 128 model, 8,192 tokens, one record in 128
        # tampered with (it must come back as zeros).
        dict(name="reload_int4_qwen", op="reload", heads=4, dim=128, blocks=64, bits=4, strict=False, ivs=True,
             tampered=1),
        # The headline layer with every tag checked before any release.
        dict(name="reload_strict_bf16_8b", op="reload", heads=8, dim=128, blocks=48, bits=0, strict=True, ivs=True,
             tampered=0),
        # A causal group of bf16 blocks sealed on the device.
        dict(name="writeback_bf16_group", op="writeback", heads=8, dim=128, blocks=16, bits=0),
        # A 32,768-token layer quantised to int4 and sealed: the largest.
        dict(name="writeback_int4_70b", op="writeback", heads=8, dim=128, blocks=256, bits=4),
        # The same at one head per tensor-parallel rank (10,256-B packets).
        dict(name="writeback_int4_tp_rank", op="writeback", heads=1, dim=128, blocks=256, bits=4),
        # The kernel-level calls on one record of an odd size: sealed, then
        # verified and opened.
        dict(name="record_odd", op="record", bytes=100_003, aad=20),
        # A layer of int4 packets stored to host memory and reloaded from it
        # (host crypto and PCIe included), as a prefix cache does.
        dict(name="roundtrip_int4_qwen", op="roundtrip", heads=4, dim=128, blocks=64, bits=4),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choices(["reload", "writeback", "record", "roundtrip"], [6, 4, 2, 1])[0]
    if op == "record":
        return dict(op=op, bytes=_log(rng, 1, 4 << 20), aad=rng.randint(0, AAD))
    heads, dim = rng.randint(1, 8), rng.choice([64, 128])
    bits = rng.choice([0, 0, 8, 4])
    blocks = _log(rng, 1, 256)
    # at most the wire bytes of the largest listed layer (the time of a layer
    # follows them); a round trip at most the listed one's
    most = 2 * 256 * _width(dict(heads=8, dim=128, bits=4))
    if op == "roundtrip":
        most = 2 * 64 * _width(dict(heads=4, dim=128, bits=4))
    width = _width(dict(heads=heads, dim=dim, bits=bits))
    blocks = max(1, min(blocks, most // (2 * width)))
    case = dict(op=op, heads=heads, dim=dim, blocks=blocks, bits=bits)
    if op == "reload":
        case.update(strict=rng.random() < 0.2, ivs=rng.random() < 0.5, tampered=rng.choice([0, 0, 1]))
    return case


# ------------------------------------------------------------------ inputs

def _width(c):
    """Bytes of one record: a bf16 block, or a codec packet."""
    hd = c["heads"] * c["dim"]
    if c["bits"] == 0:
        return TOKENS * hd * 2
    return (TOKENS * hd * c["bits"] // 8 + 16 * hd + 16 + 15) // 16 * 16


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _key(seed):
    rng = np.random.default_rng(seed & 0x7FFFFFFF)
    return rng.integers(0, 256, 16, dtype=np.uint8).tobytes(), rng.integers(0, 256, 4, dtype=np.uint8).tobytes()


def _blocks(c, g):
    """[2, blocks, 128, heads, dim] bf16 ~ N(0, 1): the layer's K and V."""
    return torch.randn((2, c["blocks"], TOKENS, c["heads"], c["dim"]), generator=g, device="cuda").to(torch.bfloat16)


def _quantise(x, kind, bits):
    """The transport codec's asymmetric min / max quantiser over x
    [blocks, 128, heads, dim] float32: K groups 64 tokens, V groups 64 dims.
    Returns q (as floats), scale and low, each shaped to broadcast."""
    n, _, h, d = x.shape
    v = x.view(n, 2, GROUP, h, d) if kind == 0 else x.view(n, TOKENS, h, d // GROUP, GROUP)
    axis = 2 if kind == 0 else 4
    lo, hi = v.amin(axis, keepdim=True), v.amax(axis, keepdim=True)
    top = float((1 << bits) - 1)
    scale = ((hi - lo) / top).clamp_min(1e-12)
    return ((v - lo) / scale).round().clamp(0, top), scale, lo


def _packets(c, x, layer):
    """[2 * blocks, width] uint8 codec packets of x [2, blocks, ...]."""
    out = []
    for kind in (0, 1):
        q, scale, lo = _quantise(x[kind].float(), kind, c["bits"])
        n = c["blocks"]
        q = q.reshape(n, -1).to(torch.uint8)
        if c["bits"] == 4:
            q = q[:, 0::2] | (q[:, 1::2] << 4)
        head = np.array([1, layer, kind, c["bits"]], np.int32).view(np.uint8)
        head = torch.from_numpy(head).to(q.device).expand(n, 16)
        params = [p.reshape(n, -1).contiguous().view(torch.uint8) for p in (scale, lo)]
        row = torch.cat([q, *params, head], 1)
        out.append(torch.nn.functional.pad(row, (0, _width(c) - row.shape[1])))
    return torch.cat(out).contiguous()


def _tickets(c, ivs):
    """Tickets in record order (K blocks, then V): one run, or the order in
    which causal groups of 16 blocks submit them (tail first)."""
    n = c["blocks"]
    if not ivs:
        return 1 + np.arange(2 * n)
    pos = {kb: i for i, kb in enumerate(si.gcm.reference_ticket_order(n, 16))}
    return 1 + np.array([pos[divmod(r, n)] for r in range(2 * n)])


def _iv_words(salt, tickets):
    w = np.zeros((tickets.size, 4), np.uint32)
    w[:, 0] = int.from_bytes(salt, "big")
    w[:, 2] = tickets
    w[:, 3] = 2
    return torch.from_numpy(w.view(np.int32)).to("cuda")


def _wire(c, direction, tickets, layer):
    """Empty wire records of a layer with their AADs in place."""
    n = _width(c)
    stride = si.wire_stride(n)
    off = si.wire_tag_offset(n) + 32
    host = np.zeros((2 * c["blocks"], stride), np.uint8)
    for r in range(2 * c["blocks"]):
        kind, b = divmod(r, c["blocks"])
        aad = b"SFAD" + bytes([1, direction, kind, 0]) + struct.pack(">IQQQQ", layer, b, 0, n, int(tickets[r]))
        host[r, off:off + AAD] = np.frombuffer(aad.ljust(AAD, b"\0"), np.uint8)
    return torch.from_numpy(host).to("cuda")


def _slots(c, g):
    """The layer's slot ids (K then V, the same blocks) in a cache of twice
    as many slots."""
    s = torch.randperm(2 * c["blocks"], generator=g, device="cuda")[:c["blocks"]]
    return torch.cat([s, s]).contiguous()


def _tampered(c, seed):
    return [int(r) for r in
            np.random.default_rng(seed & 0xFFFF).choice(2 * c["blocks"], c.get("tampered", 0), replace=False)]


def _cache(c, x=None, slots=None):
    ck = torch.zeros((2 * c["blocks"], TOKENS, c["heads"], c["dim"]), dtype=torch.bfloat16, device="cuda")
    cv = torch.zeros_like(ck)
    if x is not None:
        ck[slots[:c["blocks"]]] = x[0]
        cv[slots[:c["blocks"]]] = x[1]
    return ck, cv


def prepare(case, seed):
    c, g = case, _gen(seed)
    key, salt = _key(seed)
    if c["op"] == "record":
        return _prepare_record(c, g, key, salt)
    layer, n, nrec = 3, _width(c), 2 * c["blocks"]
    sess = si.GcmSession(key, salt, 0, max_record_bytes=n)
    x = _blocks(c, g)
    slots = _slots(c, g)
    if c["op"] == "roundtrip":
        return _prepare_roundtrip(c, sess, x, slots, layer)
    fail = torch.zeros(1, dtype=torch.int32, device="cuda")
    staging = torch.zeros(nrec * si.wire_tag_offset(n), dtype=torch.uint8, device="cuda") if c["bits"] else None
    how = dict(codec_bits=c["bits"], heads=c["heads"], head_dim=c["dim"], layer=layer, staging=staging,
               fail_count=fail)
    if c["op"] == "writeback":
        tickets = _tickets(c, False)
        wire = _wire(c, 2, tickets, layer)
        ck, cv = _cache(c, x, slots)
        plan = sess.prepare_writeback_layer(wire, n, nrec, c["blocks"], ck, cv, slots, ticket_base=1, **how)
        return dict(op="writeback", plan=plan, sess=sess, out=(wire,))
    tickets = _tickets(c, c["ivs"])
    ivs = _iv_words(salt, tickets)
    wire = _wire(c, 1, tickets, layer)
    # The records as the host seals them: bf16 blocks, or packets.
    rows = _packets(c, x, layer) if c["bits"] else x.reshape(nrec, -1).view(torch.uint8)
    order = torch.arange(c["blocks"], device="cuda").repeat(2)
    sess.writeback_layer(wire, n, nrec, c["blocks"], rows[:c["blocks"]], rows[c["blocks"]:], order, iv_words_dev=ivs)
    for r in _tampered(c, seed):
        wire[r, n // 2] ^= 1
    ck, cv = _cache(c)
    plan = sess.prepare_reload_layer(wire, n, nrec, c["blocks"], ck, cv, slots, ticket_base=1,
                                     iv_words_dev=ivs if c["ivs"] else None, verify_before_release=c["strict"], **how)
    off = si.wire_tag_offset(n) + 16
    return dict(op="reload", plan=plan, sess=sess, out=(ck, cv, wire[:, off:off + 4]))


def _prepare_record(c, g, key, salt):
    def u8(n):
        return torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda", generator=g)
    dev = lambda b: torch.frombuffer(bytearray(b), dtype=torch.uint8).to("cuda")
    sess = si.GcmSession(key, salt, 0, max_record_bytes=16)
    n = c["bytes"]
    s = dict(op="record", key=dev(key), h=dev(sess.hash_subkey), iv=sess.record_iv(1), plain=u8(n),
             aad=u8(c["aad"]) if c["aad"] else None, ct=torch.zeros(n, dtype=torch.uint8, device="cuda"),
             tag=torch.zeros(16, dtype=torch.uint8, device="cuda"),
             back=torch.zeros(n, dtype=torch.uint8, device="cuda"),
             status=torch.zeros(4, dtype=torch.int32, device="cuda"))
    sess.close()
    return s


def _prepare_roundtrip(c, sess, x, slots, layer):
    shape = si.LayerShape(c["heads"], c["dim"], c["bits"])
    nb = c["blocks"]

    def pool():
        if c["bits"]:
            return torch.zeros((nb, _width(c)), dtype=torch.uint8)
        return torch.zeros((nb, TOKENS, c["heads"], c["dim"]), dtype=torch.bfloat16)
    host = (pool(), pool())
    for kind in (0, 1):
        si.register_host_range(host[kind], layer, kind)
    there = torch.stack([slots[:nb].cpu(), torch.arange(nb)], 1).contiguous()
    return dict(op="roundtrip", src=_cache(c, x, slots), dst=_cache(c), host=host, store=there,
                load=there.flip(1).contiguous(), layer=layer, sess=sess, d2h=si.D2HTransfer(sess, shape),
                h2d=si.NativeTransfer(sess, shape, causal_group_blocks=16))


# ------------------------------------------------------------------ one pass

def run(state):
    s = state
    if s["op"] in ("reload", "writeback"):
        s["plan"].launch()
        return s["out"]
    if s["op"] == "record":
        si.gcm_encrypt_tag(s["plain"], s["key"], s["h"], s["ct"], s["tag"], s["iv"], s["aad"])
        si.gcm_decrypt_verify(s["ct"], s["key"], s["h"], s["tag"], s["back"], s["status"], s["iv"], s["aad"])
        return s["ct"], s["tag"], s["back"], s["status"]
    s["d2h"].store([s["src"]], [s["host"]], s["store"], layers=[s["layer"]])
    s["h2d"].layer = s["layer"]
    s["h2d"].single_layer_kv_transfer((s["host"], s["load"]), s["dst"])
    ok = s["h2d"].wait_layer(s["layer"])
    return s["host"][0], s["host"][1], s["dst"][0], s["dst"][1], ok


def work(case):
    c = case
    if c["op"] == "record":
        return dict(bytes=4 * c["bytes"] + 2 * c["aad"] + 36, flops=0)
    width, nrec = _width(c), 2 * c["blocks"]
    block = TOKENS * c["heads"] * c["dim"] * 2
    coded = 2 * (block // 2) if c["bits"] else 0  # a product and a sum, or a difference and a quotient, an element
    one = dict(reload=width + block + 84, writeback=width + block + 80, roundtrip=2 * (width + block) + 164)[c["op"]]
    return dict(bytes=nrec * one, flops=nrec * coded * (2 if c["op"] == "roundtrip" else 1))


def tolerance(case):
    # Cipher text, tags, statuses, packets and bf16 KV are fixed bit for bit
    # by AES-GCM and by the codec's one-rounding-per-step definition.
    return "exact"


def exact(case, seed):
    """A reload's KV from its inputs in float64 (bf16 blocks as they are,
    packets decoded); cipher text, tags and stored packets are bytes."""
    c = case
    if c["op"] != "reload":
        return None
    g = _gen(seed)
    x = _blocks(c, g)
    slots = _slots(c, g)
    bad = _tampered(c, seed)
    out = []
    for kind in (0, 1):
        if c["bits"]:
            q, scale, lo = _quantise(x[kind].float(), kind, c["bits"])
            v = (q.double() * scale.double() + lo.double()).reshape(x[kind].shape)
        else:
            v = x[kind].double()
        for r in bad:
            if r // c["blocks"] == kind:
                v[r % c["blocks"]] = 0
        full = torch.zeros((2 * c["blocks"], *v.shape[1:]), dtype=torch.float64, device=v.device)
        full[slots[:c["blocks"]]] = v
        out.append(full)
    return out[0], out[1], None
