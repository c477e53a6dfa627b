"""Pages that are not cut into whole 64-byte units, in the kernels that keep
their payloads in LDS (ztcp_ragged.hip), and on both sides of the payload
sizes and batches past which the layout-agnostic kernels take over.

Every form that path accepts: each section kind, payloads padded to any
length, blobs and hot pages at odd addresses and strides (descriptors), one
page per workgroup and several, pages of mixed and of invalid header flags in
one workgroup.  Blobs must equal the
oracle's byte for byte, decoded pages bit for bit, and a flipped bit must give
the oracle's verdict for its page alone.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

KEYS = dict(k0=0x243F6A8885A308D3, k1=0x13198A2E03707344, mk0=0xA4093822299F31D0,
            mk1=0x082EFA98EC4E6C89, k2=0x452821E638D01377, k3=0xBE5466CF34E90C6C)
TEN, MOD, LAYER, HG, BASE = 0x5EED5EED, 0x0DDBA11, 11, 2, 77_000
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
bits = lambda t: None if t is None else t.contiguous().view(torch.int16).numpy().view(np.uint16)  # noqa: E731


def _pages(seed, B, T, H, D, R, mla, dt):
    rng = np.random.default_rng(seed)
    k = rng.standard_normal((B, T, H, D)).astype(np.float32)
    k[..., :R] *= 8
    k[0, 0, 0, :16] = 0
    v = None if mla else torch.from_numpy(rng.standard_normal((B, T, H, D)).astype(np.float32) * 0.5).to(DT[dt])
    return torch.from_numpy(k).to(DT[dt]), v, rng.integers(0, 1 << 62, size=B, dtype=np.int64)


def _odt(O, dt):
    return O.BF16 if dt == "bf16" else O.FP16


# tokens, heads, head_dim, rope, MLA, preset, mode, pages, dtype, extra payload bytes
CASES = [
    (5, 3, 48, 16, False, 1, 1, 7, "fp16", 0),
    (5, 3, 48, 16, False, 2, 2, 7, "bf16", 1),
    (13, 5, 96, 32, False, 3, 0, 3, "bf16", 3),
    (7, 3, 80, 16, False, 2, 1, 1300, "fp16", 0),       # two pages per workgroup, the last one partial
    (1, 1, 16, 0, True, 1, 0, 1, "bf16", 0),            # one group: a payload of 10 bytes
    (1, 1, 16, 16, True, 1, 2, 33, "fp16", 61),         # raw only, padded over a block's end
    (3, 1, 64, 64, True, 3, 1, 40000, "bf16", 0),       # 32 pages per workgroup
    (3, 1, 128, 64, True, 4, 3, 5, "bf16", 0),          # asym8 per 64, e4m3 RoPE
    (3, 3, 64, 0, False, 4, 0, 9, "fp16", 2),           # asym8 and int4 per 32
    (29, 1, 192, 32, True, 5, 3, 2050, "bf16", 5),      # e4m3, three pages per workgroup
    (7, 1, 96, 32, False, 6, 1, 4, "fp16", 64),         # int4 per 32
    (16, 8, 128, 64, False, 2, 1, 3, "bf16", 13),       # whole units, but a padded payload
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:4])) + f"-p{c[5]}r{c[6]}-B{c[7]}-{c[8]}+{c[9]}")
def test_every_kind_and_padding(hip, O, case):
    T, H, D, R, mla, preset, rm, B, dt, extra = case
    ext = preset > 3 or rm > 2
    k, v, th = _pages(B + preset, B, T, H, D, R, mla, dt)
    exp = O.payload_bytes(preset, rm, T * H, D, R, not mla) + extra
    want = O.egress_batch(bits(k), bits(v), th, dtype=_odt(O, dt), preset=preset, rope_mode=rm, rope_dim=R,
                          expected_payload_bytes=exp, tenant_id_hash=TEN, model_id_hash=MOD, layer_id=LAYER,
                          head_group_id=HG, base_sequence_nonce=BASE, **KEYS)
    dev = torch.device("cuda")
    blobs = torch.full((B, 48 + exp), 0xA5, dtype=torch.uint8, device=dev)
    hip.fused_encode_cold_pages_peak_into(k.to(dev), None if v is None else v.to(dev), torch.from_numpy(th), blobs,
                                          preset, rm, R, exp, TEN, MOD, LAYER, HG, BASE, ext_layouts=ext, **KEYS)
    assert np.array_equal(blobs.cpu().numpy(), want)
    bad = sorted({0, B // 2, B - 1}) if B > 3 else []
    t = want.copy()
    for i, b in enumerate(bad):
        t[b, (16, 32 + exp - 1, 48 + exp - 1)[i]] ^= 0x20  # token hash, the payload's last byte, the tag's
    ko = torch.full((B, T, H, D), 7.0, dtype=DT[dt], device=dev)
    vo = None if mla else torch.full_like(ko, 7.0)
    st = torch.full((B,), -9, dtype=torch.int32, device=dev)
    try:
        hip.fused_decode_cold_pages_peak_into(torch.from_numpy(t).to(dev), torch.from_numpy(th), ko, vo, R, mla, TEN,
                                              MOD, LAYER, page_status=st, per_page=True, ext_layouts=ext, **KEYS)
        assert not bad
    except RuntimeError as e:
        assert "CROSS_TENANT" in str(e), e  # the lowest failing page's
    rc, ost, ok, ov = O.ingress_batch(t, th, num_tokens=T, num_heads=H, head_dim=D, rope_dim=R,
                                      is_mla_single_buffer=mla, dtype=_odt(O, dt), expected_tenant_hash=TEN,
                                      expected_model_hash=MOD, expected_layer_id=LAYER, all_or_nothing=False, **KEYS)
    assert np.array_equal(st.cpu().numpy(), ost)
    assert np.array_equal(bits(ko.cpu()).ravel(), np.asarray(ok).ravel())
    if not mla:
        assert np.array_equal(bits(vo.cpu()).ravel(), np.asarray(ov).ravel())


@pytest.mark.parametrize("shift", [1, 2, 4, 15])
def test_odd_addresses_and_strides(pkg, hip, O, shift):
    """Descriptors: blobs at odd addresses and strides, hot pages 2 bytes off a 16-byte line."""
    import vlx_tee_amd.pages as P

    T, H, D, R, B, preset, rm = 5, 3, 64, 16, 37, 2, 1
    k, v, th = _pages(shift, B, T, H, D, R, False, "fp16")
    exp = O.payload_bytes(preset, rm, T * H, D, R, True)
    dev = torch.device("cuda")
    n = T * H * D
    hot = [torch.full((B, n + 3), 9.0, dtype=torch.float16, device=dev) for _ in range(4)]
    buf = torch.full((B, 48 + exp + 2 * shift + 1), 0xA5, dtype=torch.uint8, device=dev)
    views = [h[:, 1:1 + n] for h in hot]
    views[0].copy_(k.view(B, n))
    views[1].copy_(v.view(B, n))
    blobs = buf[:, shift:shift + 48 + exp]
    seq, layers = np.arange(B, dtype=np.uint64) + BASE, np.full(B, LAYER, dtype=np.uint16)
    geo = dict(num_tokens=T, num_heads=H, head_dim=D, rope_dim=R, dtype=torch.float16, is_mla_single_buffer=False)
    hgs = np.full(B, HG, dtype=np.uint16)
    P.egress(P.build_descriptors(views[0], views[1], blobs, th, seq, layers, hgs), B, preset=preset, rope_mode=rm,
             expected_payload_bytes=exp, tenant_id_hash=TEN, model_id_hash=MOD, **geo, **KEYS)
    want = O.egress_batch(bits(k), bits(v), th, dtype=O.FP16, preset=preset, rope_mode=rm, rope_dim=R,
                          expected_payload_bytes=exp, tenant_id_hash=TEN, model_id_hash=MOD, layer_id=LAYER,
                          head_group_id=HG, base_sequence_nonce=BASE, **KEYS)
    got = buf.cpu().numpy()
    assert np.array_equal(got[:, shift:shift + 48 + exp], want)
    assert (got[:, :shift] == 0xA5).all() and (got[:, shift + 48 + exp:] == 0xA5).all()
    st = torch.full((B,), -9, dtype=torch.int32, device=dev)
    d = P.build_descriptors(views[2], views[3], blobs, th, seq, layers, hgs)
    assert P.ingress(d, B, 48 + exp, expected_tenant_hash=TEN, expected_model_hash=MOD, page_status=st, **geo,
                     **KEYS) == 0
    _, _, ok, ov = O.ingress_batch(want, th, num_tokens=T, num_heads=H, head_dim=D, rope_dim=R,
                                   is_mla_single_buffer=False, dtype=O.FP16, expected_tenant_hash=TEN,
                                   expected_model_hash=MOD, expected_layer_id=LAYER, **KEYS)
    for h, o in ((hot[2], ok), (hot[3], ov)):
        assert np.array_equal(bits(h.cpu()[:, 1:1 + n]).ravel(), np.asarray(o).ravel())
        assert (h[:, 0] == 9.0).all() and (h[:, 1 + n:] == 9.0).all()


# payloads (2,160 T bytes) below / above what fits: ingress keeps two copies (80 KB
# each), egress one (160 KB)
@pytest.mark.parametrize("T", [37, 38, 75, 77])
def test_payloads_around_the_lds_limits(hip, O, T):
    H, D, R, preset, rm, B = 5, 192, 32, 3, 0, 2
    k, v, th = _pages(T, B, T, H, D, R, False, "bf16")
    exp = O.payload_bytes(preset, rm, T * H, D, R, True)
    want = O.egress_batch(bits(k), bits(v), th, dtype=O.BF16, preset=preset, rope_mode=rm, rope_dim=R,
                          expected_payload_bytes=exp, tenant_id_hash=TEN, model_id_hash=MOD, layer_id=LAYER,
                          head_group_id=HG, base_sequence_nonce=BASE, **KEYS)
    dev = torch.device("cuda")
    blobs = torch.zeros((B, 48 + exp), dtype=torch.uint8, device=dev)
    hip.fused_encode_cold_pages_peak_into(k.to(dev), v.to(dev), torch.from_numpy(th), blobs, preset, rm, R, exp, TEN,
                                          MOD, LAYER, HG, BASE, **KEYS)
    assert np.array_equal(blobs.cpu().numpy(), want)
    ko = torch.empty((B, T, H, D), dtype=torch.bfloat16, device=dev)
    vo = torch.empty_like(ko)
    hip.fused_decode_cold_pages_peak_into(blobs, torch.from_numpy(th), ko, vo, R, False, TEN, MOD, LAYER, **KEYS)
    _, _, ok, ov = O.ingress_batch(want, th, num_tokens=T, num_heads=H, head_dim=D, rope_dim=R,
                                   is_mla_single_buffer=False, dtype=O.BF16, expected_tenant_hash=TEN,
                                   expected_model_hash=MOD, expected_layer_id=LAYER, **KEYS)
    assert np.array_equal(bits(ko.cpu()).ravel(), np.asarray(ok).ravel())
    assert np.array_equal(bits(vo.cpu()).ravel(), np.asarray(ov).ravel())


# last and first batch on each side of the rule (rounds of the pages that fit a
# CU's LDS at once): egress of 84,240-byte payloads (one fits, 10 rounds), ingress
# of 75,600 (one, 4 rounds), 32,400 (two, 6) and 23,760 bytes (three, 10)
@pytest.mark.parametrize("way,T,fit,rounds", [("egress", 39, 1, 10), ("ingress", 35, 1, 4), ("ingress", 15, 2, 6),
                                              ("ingress", 11, 3, 10)])
def test_batches_around_the_rule(hip, O, way, T, fit, rounds):
    H, D, R, preset, rm = 5, 192, 32, 3, 0
    dev = torch.device("cuda")
    k, v, _ = _pages(T, 1, T, H, D, R, False, "bf16")
    exp = O.payload_bytes(preset, rm, T * H, D, R, True)
    line = torch.cuda.get_device_properties(0).multi_processor_count * fit * rounds
    for B in (line, line + 1):
        th = np.arange(B, dtype=np.int64) + 5
        kd, vd = (t.to(dev).expand(B, -1, -1, -1).contiguous() for t in (k, v))
        blobs = torch.full((B, 48 + exp), 0xA5, dtype=torch.uint8, device=dev)
        hip.fused_encode_cold_pages_peak_into(kd, vd, torch.from_numpy(th), blobs, preset, rm, R, exp, TEN, MOD, LAYER,
                                              HG, BASE, **KEYS)
        for b in (0, B // 2, B - 1):
            want = O.egress_batch(bits(k), bits(v), th[b:b + 1], dtype=O.BF16, preset=preset, rope_mode=rm, rope_dim=R,
                                  expected_payload_bytes=exp, tenant_id_hash=TEN, model_id_hash=MOD, layer_id=LAYER,
                                  head_group_id=HG, base_sequence_nonce=BASE + b, **KEYS)
            assert np.array_equal(blobs[b].cpu().numpy(), want[0]), (B, b)
        if way == "egress":
            continue
        _, _, ok, ov = O.ingress_batch(want, th[B - 1:], num_tokens=T, num_heads=H, head_dim=D, rope_dim=R,
                                       is_mla_single_buffer=False, dtype=O.BF16, expected_tenant_hash=TEN,
                                       expected_model_hash=MOD, expected_layer_id=LAYER, **KEYS)
        blobs[B // 3, 40] ^= 1
        kd.fill_(3.0), vd.fill_(3.0)
        st = torch.full((B,), -9, dtype=torch.int32, device=dev)
        with pytest.raises(RuntimeError):
            hip.fused_decode_cold_pages_peak_into(blobs, torch.from_numpy(th), kd, vd, R, False, TEN, MOD, LAYER,
                                                  page_status=st, per_page=True, **KEYS)
        want_st = torch.zeros(B, dtype=torch.int32, device=dev)
        want_st[B // 3] = 3
        assert torch.equal(st, want_st)
        for got, o in ((kd, ok), (vd, ov)):
            page = torch.from_numpy(np.asarray(o).ravel().view(np.int16).reshape(T, H, D).copy()).to(dev)
            good = torch.ones(B, dtype=torch.bool, device=dev)
            good[B // 3] = False
            assert (got.view(torch.int16)[good] == page).all() and (got[B // 3] == 0).all(), B


@pytest.mark.parametrize("per_page", [True, False])
def test_mixed_and_invalid_flags_in_one_workgroup(hip, O, per_page):
    """Pages of several presets and RoPE modes, padded to one blob size, beside
    pages of invalid flags, two and three to a workgroup: each by its own header."""
    T, H, D, R, per = 7, 3, 80, 16, 700
    modes = [(1, 0), (2, 1), (3, 2)]
    exp = max(O.payload_bytes(p, m, T * H, D, R, True) for p, m in modes) + 5
    parts, ths = [], []
    for i, (preset, rm) in enumerate(modes):
        k, v, th = _pages(i, per, T, H, D, R, False, "fp16")
        parts.append(O.egress_batch(bits(k), bits(v), th, dtype=O.FP16, preset=preset, rope_mode=rm, rope_dim=R,
                                    expected_payload_bytes=exp, tenant_id_hash=TEN, model_id_hash=MOD, layer_id=LAYER,
                                    head_group_id=HG, base_sequence_nonce=BASE + i * per, **KEYS))
        ths.append(th)
    order = np.random.default_rng(0).permutation(3 * per)
    blobs, th = np.concatenate(parts)[order], np.concatenate(ths)[order]
    blobs[5, 3] = 0x07    # preset 7: no layout
    blobs[901, 3] = 0x31  # RoPE mode 3: an extension layout, not asked for here
    dev = torch.device("cuda")
    ko = torch.full((3 * per, T, H, D), 7.0, dtype=torch.float16, device=dev)
    vo = torch.full_like(ko, 7.0)
    st = torch.full((3 * per,), -9, dtype=torch.int32, device=dev)
    with pytest.raises(RuntimeError):
        hip.fused_decode_cold_pages_peak_into(torch.from_numpy(blobs).to(dev), torch.from_numpy(th), ko, vo, R, False, TEN,
                                              MOD, LAYER, page_status=st, per_page=per_page, **KEYS)
    _, ost, ok, ov = O.ingress_batch(blobs, th, num_tokens=T, num_heads=H, head_dim=D, rope_dim=R,
                                     is_mla_single_buffer=False, dtype=O.FP16, expected_tenant_hash=TEN,
                                     expected_model_hash=MOD, expected_layer_id=LAYER, all_or_nothing=not per_page, **KEYS)
    ost = np.asarray(ost)
    assert (ost != 0).sum() == 2 and np.array_equal(st.cpu().numpy(), ost)
    for got, o in ((ko, ok), (vo, ov)):
        assert np.array_equal(bits(got.cpu()).ravel(), np.asarray(o).ravel())
        assert per_page or not got.any()
