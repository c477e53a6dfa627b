"""Performance cases of the cold-page codec.

Every case is one call of a public entry point on tensors that are already in
HBM: an egress (quantize, encrypt, authenticate) or an ingress (verify,
decrypt, dequantize) of a batch of KV pages.  The listed cases are what a
serving engine asks of the codec: the single page that a decode step evicts
or faults in, the few hundred pages of one request, a whole 1 GiB prefix over
all layers, MLA latent pages, the ragged pages of models whose heads and
widths do not cut into whole 64-byte blocks, both hot dtypes, the reference's
presets and RoPE modes and the extension ones, and the per-page policy on a
prefix with tampered pages.  ``draw`` spreads more cases over the same ranges.

``api`` names the entry point:
  peak_into  native_hip_codec.fused_{en,de}code_cold_pages_peak_into (one layer)
  pages      pages.egress / pages.ingress (descriptors, many layers per call)
  codec      codec.NativeHipFusedColdPageCodec.decode_cold_pages_peak_into
             (session key ring, freshness check)
"""
from __future__ import annotations

import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent


def _package():
    """The product package (its folder's name is not an identifier)."""
    if "vlx_tee_amd" not in sys.modules:
        root = ROOT / "vlx-tee_amd"
        spec = importlib.util.spec_from_file_location("vlx_tee_amd", root / "__init__.py",
                                                      submodule_search_locations=[str(root)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vlx_tee_amd"] = mod
        spec.loader.exec_module(mod)
    import vlx_tee_amd.codec as codec
    import vlx_tee_amd.keyring as keyring
    import vlx_tee_amd.native_hip_codec as hip
    import vlx_tee_amd.pages as pages
    import vlx_tee_amd.spec as spec

    return codec, keyring, hip, pages, spec


# ---- geometries ------------------------------------------------------------------
# tokens, heads, head_dim, rope_dim, MLA single buffer
GQA4 = dict(tokens=16, heads=4, head_dim=128, rope=64, mla=False)      # 16-token pages, 4 KV heads
GQA8 = dict(tokens=16, heads=8, head_dim=128, rope=64, mla=False)      # 16-token pages, 8 KV heads
GQA8_64 = dict(tokens=64, heads=8, head_dim=128, rope=64, mla=False)   # the reference benchmark's 64-token page
MLA = dict(tokens=64, heads=1, head_dim=576, rope=64, mla=True)        # MLA latent page
RAGGED_A = dict(tokens=13, heads=5, head_dim=96, rope=32, mla=False)   # sections end inside 64-byte blocks
RAGGED_B = dict(tokens=7, heads=3, head_dim=80, rope=16, mla=False)
RAGGED_M = dict(tokens=29, heads=1, head_dim=192, rope=32, mla=True)

TENANT, MODEL, SESSION = "tenant-alpha-bank", "Qwen/Qwen3.6-35B-A3B", "session-0"
LAYER, HEAD_GROUP = 7, 0
KEYS = dict(k0=0x0123456789ABCDEF, k1=0xFEDCBA9876543210, mk0=0x1111222233334444,
            mk1=0x5555666677778888, k2=0xDEADBEEFCAFEF00D, k3=0x0BADC0DE12345678)
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, way, api, geo, pages, preset, rope_mode, dtype, *, per_page=False, tamper=0.0,
          asynchronous=False, outliers=0.0):
    c = dict(way=way, api=api, pages=pages, preset=preset, rope_mode=rope_mode, dtype=dtype,
             per_page=per_page, tamper=tamper, asynchronous=asynchronous, outliers=outliers, **geo)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a decode step evicts one full 64-token page: the smallest call, all latency
        _case("egress_one_page", "egress", "peak_into", GQA8_64, 1, 2, 1, "fp16"),
        # a request resumes a short context: four 64-token pages of one layer through the session codec
        _case("ingress_session_4", "ingress", "codec", GQA8_64, 4, 2, 1, "fp16"),
        # one layer's 4096-token context, 256 pages with outlier channels: the reference's peak-256 batch
        _case("egress_int4_256", "egress", "peak_into", GQA4, 256, 1, 1, "bf16", outliers=0.01),
        _case("ingress_int4_256", "ingress", "peak_into", GQA4, 256, 1, 1, "bf16", outliers=0.01),
        # a whole evicted prefix, 4096 tokens x 64 layers: 1 GiB of hot pages in one enqueued call
        _case("egress_prefix_k8v4", "egress", "pages", GQA8, 16384, 2, 1, "bf16", asynchronous=True),
        _case("ingress_prefix_k8v4", "ingress", "pages", GQA8, 16384, 2, 1, "bf16", asynchronous=True),
        # the same prefix at 8 bits with 1 % of its pages tampered, each page judged by itself
        _case("ingress_prefix_int8_tampered", "ingress", "pages", GQA8, 16384, 3, 0, "bf16", per_page=True,
              tamper=0.01),
        # MLA latent pages of a medium prefix (61 layers x 67 pages): a count that fills no launch evenly
        _case("egress_mla_int4", "egress", "pages", MLA, 4087, 1, 1, "bf16", outliers=0.02),
        # MLA latents at int4 per 32 with e4m3 RoPE columns: the extension layouts, a part of a prefix
        _case("ingress_mla_int4g32", "ingress", "pages", MLA, 1777, 6, 3, "bf16"),
        # K int8 asymmetric per 64, V int4 per 32: the extension layouts' encoder on a few layers
        _case("egress_k8v4asym", "egress", "pages", GQA8, 2900, 4, 3, "bf16"),
        # heads and widths that cut into no whole 64-byte block, RoPE columns kept as they are
        _case("egress_ragged_raw", "egress", "peak_into", RAGGED_A, 333, 1, 2, "fp16"),
        _case("ingress_ragged", "ingress", "peak_into", RAGGED_B, 1200, 2, 1, "fp16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    way = rng.choice(["egress", "ingress"])
    geo = rng.choice([GQA4, GQA8, GQA8, GQA8_64, MLA, RAGGED_A, RAGGED_B, RAGGED_M])
    ragged = geo in (RAGGED_A, RAGGED_B, RAGGED_M)
    hot = geo["tokens"] * geo["heads"] * geo["head_dim"] * (2 if geo["mla"] else 4)
    # up to a quarter of the largest listed prefix; the ragged geometries up to 2000 pages
    pages = _log_int(rng, 1, 2000 if ragged else min(9000, (1 << 28) // hot))
    preset, mode = rng.choice([(1, 1), (1, 0), (2, 1), (2, 2), (3, 0), (3, 1)] +
                              ([] if ragged else [(4, 3), (5, 0), (6, 3)]))
    api = rng.choice(["peak_into", "pages"] + (["codec"] if way == "ingress" and preset <= 3 else []))
    per_page = way == "ingress" and api == "pages" and rng.random() < 0.5
    return _case(None, way, api, geo, pages, preset, mode, rng.choice(["bf16", "fp16"]), per_page=per_page,
                 tamper=0.02 if per_page else 0.0, asynchronous=api == "pages" and rng.random() < 0.5,
                 outliers=rng.choice([0.0, 0.01]))


# ---- inputs ------------------------------------------------------------------------

def _hot(case, seed, device="cuda"):
    """K and V pages: N(0, 1), K's RoPE columns x8 (MLA: latent sigma 0.5), some channels x20."""
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    n, T, H, D, R = (case[x] for x in ("pages", "tokens", "heads", "head_dim", "rope"))
    dt = DTYPES[case["dtype"]]
    out = []
    for which in range(1 if case["mla"] else 2):
        t = torch.empty((n, T, H, D), dtype=dt, device=device)
        gain = torch.ones(D, device=device)
        if which == 0:
            gain[:R] = 1.0 if case["mla"] else 8.0
            if case["mla"]:
                gain[R:] = 0.5
        if case["outliers"]:
            m = max(1, math.ceil(case["outliers"] * D))
            gain[torch.randperm(D, generator=gen, device=device)[:m]] *= 20.0
        step = max(1, (1 << 26) // (T * H * D))
        for s in range(0, n, step):
            m = min(step, n - s)
            t[s:s + m] = (torch.randn((m, T, H, D), generator=gen, device=device) * gain).to(dt)
        out.append(t)
    return out[0], (out[1] if len(out) > 1 else None)


def _tampered(case, seed):
    n = case["pages"]
    m = int(round(case["tamper"] * n))
    return np.sort(np.random.default_rng(seed + 1).choice(n, size=m, replace=False)) if m else np.zeros(0, np.int64)


def _geometry(case, spec):
    return spec.ColdPageGeometry(case["tokens"], case["heads"], case["head_dim"], case["rope"], 16, 2, case["mla"])


def _meta(case, seed):
    """Token hashes, sequence nonces and layers of the pages (256 pages a layer)."""
    n = case["pages"]
    rng = np.random.default_rng(seed)
    return (rng.integers(0, 1 << 62, size=n, dtype=np.int64), np.arange(n, dtype=np.uint64) + 1000,
            (np.arange(n) // 256).astype(np.uint16))


def _encode(case, k, v, blobs, th, seq, layers, m):
    """The pages' blobs, as the same entry point's egress makes them."""
    codec, keyring, hip, pages, spec = m
    geo = _geometry(case, spec)
    ext = case["preset"] > 3 or case["rope_mode"] > 2
    payload = geo.payload_bytes(case["preset"], case["rope_mode"])
    if case["api"] == "pages":
        d = pages.build_descriptors(k, v, blobs, th, seq, layers)
        pages.egress(d, case["pages"], num_tokens=case["tokens"], num_heads=case["heads"],
                     head_dim=case["head_dim"], rope_dim=case["rope"], dtype=k.dtype,
                     is_mla_single_buffer=case["mla"], preset=case["preset"], rope_mode=case["rope_mode"],
                     expected_payload_bytes=payload, tenant_id_hash=spec.hash32(TENANT),
                     model_id_hash=spec.hash32(MODEL), ext_layouts=ext, **KEYS)
    else:
        hip.fused_encode_cold_pages_peak_into(
            k, v, torch.from_numpy(th).cuda(), blobs, case["preset"], case["rope_mode"], case["rope"], payload,
            spec.hash32(TENANT), spec.hash32(MODEL), LAYER, HEAD_GROUP, 1000, ext_layouts=ext, **KEYS)


def prepare(case, seed):
    m = _package()
    codec, keyring, hip, pages, spec = m
    n = case["pages"]
    geo = _geometry(case, spec)
    k, v = _hot(case, seed)
    th, seq, layers = _meta(case, seed)
    blobs = torch.empty((n, geo.cold_blob_bytes(case["preset"], case["rope_mode"])), dtype=torch.uint8,
                        device="cuda")
    s = dict(case=case, mods=m, geo=geo, blobs=blobs, th=torch.from_numpy(th).cuda(),
             tenant=spec.hash32(TENANT), model=spec.hash32(MODEL),
             ext=case["preset"] > 3 or case["rope_mode"] > 2,
             payload=geo.payload_bytes(case["preset"], case["rope_mode"]))
    if case["way"] == "egress":
        s.update(k=k, v=v)
        if case["api"] == "pages":
            s["descs"] = pages.build_descriptors(k, v, blobs, th, seq, layers)
        return s
    if case["api"] == "codec":  # the blobs of a session, and the session's codec
        ring = keyring.EphemeralSessionKeyRing(b"deployment-pepper-0123456789abcd")
        s["codec"] = codec.NativeHipFusedColdPageCodec(geo, ring, dtype=k.dtype)
        ring.derive_or_get(TENANT, SESSION)
        aad = spec.ColdPageAAD(s["tenant"], s["model"], LAYER, 0, 1000, spec.QuantPreset(case["preset"]),
                               spec.RoPEMode(case["rope_mode"]))
        s["codec"].encode_cold_pages_peak_into(k, v, torch.from_numpy(th), blobs, TENANT, SESSION, aad)
    else:
        _encode(case, k, v, blobs, th, seq, layers, m)
    bad = _tampered(case, seed)
    if len(bad):  # one flipped bit in the middle of the payload
        rows = torch.from_numpy(bad).cuda()
        blobs[rows, blobs.size(1) // 2] ^= 0x10
    del k, v
    shape = (n, case["tokens"], case["heads"], case["head_dim"])
    s["k"] = torch.empty(shape, dtype=DTYPES[case["dtype"]], device="cuda")
    s["v"] = None if case["mla"] else torch.empty_like(s["k"])
    if case["api"] == "pages":
        s["descs"] = pages.build_descriptors(s["k"], s["v"], blobs, th, seq, layers)
        s["status"] = torch.zeros(n, dtype=torch.int32, device="cuda")
    return s


def run(s):
    c = s["case"]
    codec, keyring, hip, pages, spec = s["mods"]
    if c["api"] == "pages":
        geo = dict(num_tokens=c["tokens"], num_heads=c["heads"], head_dim=c["head_dim"], rope_dim=c["rope"],
                   dtype=DTYPES[c["dtype"]], is_mla_single_buffer=c["mla"])
        if c["way"] == "egress":
            pages.egress(s["descs"], c["pages"], preset=c["preset"], rope_mode=c["rope_mode"],
                         expected_payload_bytes=s["payload"], tenant_id_hash=s["tenant"],
                         model_id_hash=s["model"], ext_layouts=s["ext"], asynchronous=c["asynchronous"],
                         **geo, **KEYS)
            return s["blobs"]
        pages.ingress(s["descs"], c["pages"], s["blobs"].size(1), expected_tenant_hash=s["tenant"],
                      expected_model_hash=s["model"], page_status=s["status"], per_page=c["per_page"],
                      asynchronous=c["asynchronous"], ext_layouts=s["ext"], **geo, **KEYS)
        return [t for t in (s["k"], s["v"], s["status"]) if t is not None]
    if c["way"] == "egress":
        hip.fused_encode_cold_pages_peak_into(
            s["k"], s["v"], s["th"], s["blobs"], c["preset"], c["rope_mode"], c["rope"], s["payload"],
            s["tenant"], s["model"], LAYER, HEAD_GROUP, 1000, ext_layouts=s["ext"], **KEYS)
        return s["blobs"]
    if c["api"] == "codec":
        s["codec"].decode_cold_pages_peak_into(s["blobs"], s["th"], s["k"], s["v"], TENANT, SESSION, MODEL, LAYER)
    else:
        hip.fused_decode_cold_pages_peak_into(
            s["blobs"], s["th"], s["k"], s["v"], c["rope"], c["mla"], s["tenant"], s["model"], LAYER,
            ext_layouts=s["ext"], **KEYS)
    return [t for t in (s["k"], s["v"]) if t is not None]


# ---- what a pass cannot do without, and what it must give ------------------------------

# bits per element and parameter bytes per group of the section kinds, by preset (K, V)
_KIND = {1: ("i4", "i4"), 2: ("i8", "i4"), 3: ("i8", "i8"), 4: ("a8", "i4g"), 5: ("f8", "f8"), 6: ("i4g", "i4g")}
_ROPE = {1: "i8", 2: "raw", 3: "f8"}
_PER_EL = {"i4": 0.5 + 2 / 16, "i8": 1 + 2 / 16, "f8": 1 + 2 / 16, "i4g": 0.5 + 2 / 32, "a8": 1 + 4 / 64, "raw": 2.0}


def _sections(case):
    """(kind, buffer, first column, columns) in payload order."""
    kk, kv = _KIND[case["preset"]]
    R = case["rope"] if case["rope_mode"] else 0
    sec = [(_ROPE[case["rope_mode"]], 0, 0, R)] if R else []
    if case["head_dim"] > R:
        sec.append((kk, 0, R, case["head_dim"] - R))
    if not case["mla"]:
        sec.append((kv, 1, 0, case["head_dim"]))
    return sec


def work(case):
    """Hot pages and blobs once each; the codec's arithmetic is integer, so the
    operations counted are its 32-bit ones: 976 per 64-byte ChaCha20 block and
    46 per 8-byte SipHash word, and about 5 per hot element."""
    vecs = case["tokens"] * case["heads"]
    hot = vecs * case["head_dim"] * (1 if case["mla"] else 2)
    payload = sum(_PER_EL[kind] * vecs * cols for kind, _, _, cols in _sections(case))
    return {"bytes": case["pages"] * (2 * hot + payload + 48),
            "flops": case["pages"] * (payload / 64 * 976 + payload / 8 * 46 + 5 * hot)}


def tolerance(case):
    # blobs are bytes, and the decoded pages follow bit for bit from the wire
    # format (one product and one rounding per element)
    return "exact"


def _dequantized(x, kind):
    """A section's columns after the round trip, in 64 bits: fp16 scale
    amax / 127 (or 7) per 16 elements, codes rounded in fp32 as the wire
    format says, code times scale."""
    if kind == "raw":
        return x.double()
    top = 127.0 if kind == "i8" else 7.0
    g = x.float().reshape(*x.shape[:-1], -1, 16)
    sc = (g.abs().amax(-1, keepdim=True).clamp_min(1e-6) / top).half().float()
    q = torch.round(g * (1.0 / sc)).clamp(-127 if kind == "i8" else -8, top)
    return (q.double() * sc.double()).reshape(x.shape)


def exact(case, seed):
    """Decoded pages of the reference's presets; blobs are bytes (ciphertext)
    and the extension layouts' values have no reference here."""
    if case["way"] == "egress" or case["preset"] > 3 or case["rope_mode"] > 2:
        return None
    if case["pages"] * case["tokens"] * case["heads"] * case["head_dim"] > 1 << 25:
        return None  # hundreds of MB in 64 bits; the smaller batches say the same
    k, v = _hot(case, seed)
    out = [torch.empty(t.shape, dtype=torch.float64, device=t.device) for t in (k, v) if t is not None]
    for kind, buf, col, cols in _sections(case):
        src = (k, v)[buf]
        out[buf][..., col:col + cols] = _dequantized(src[..., col:col + cols], kind)
    bad = _tampered(case, seed)
    if len(bad):
        for t in out:
            t[torch.from_numpy(bad).cuda()] = 0.0
    return out + ([None] if case["api"] == "pages" else [])
