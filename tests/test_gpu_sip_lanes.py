"""The lanes and page groups of a workgroup, at the edges of every split.

The small-batch kernels (one to four pages per workgroup) and the row-pipeline
kernels of up to 32 pages hash each page in two lanes of the MAC wave, larger
workgroups in one; the row pipeline makes its rows for groups of 16 pages.
The page counts below put each of these in a workgroup, on both sides of every
limit, with the last workgroup full and partial.  Blobs and decoded pages
must equal the oracle's, and a page with one flipped bit (the first, the last
and one in the middle) must be the only one rejected: a word that reaches the
wrong lane, or a lane or page group left out, changes some page's tag.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

KEYS = dict(k0=0x452821E638D01377, k1=0xBE5466CF34E90C6C, mk0=0xC0AC29B7C97C50DD,
            mk1=0x3F84D5B5B5470917, k2=0x9216D5D98979FB1B, k3=0xD1310BA698DFB5AC)
TEN, MOD, LAYER, HG, BASE = 0x5EED5EED, 0x0DDBA11, 3, 1, 9
T, H, D, R = 2, 16, 32, 16
# 256 CUs: one page per workgroup up to 256 pages, then two, three, four
# (small-batch kernels); 5, 16, 17, 32, 33, 48, 49 and 64 pages (row pipeline)
COUNTS = [1, 2, 255, 257, 512, 513, 769, 1023, 1024, 1025, 4096, 4099, 8191, 8193, 12288, 12300, 16384, 16385]


@pytest.mark.parametrize("preset,mode", [(2, 1), (1, 2)])
@pytest.mark.parametrize("B", COUNTS)
def test_every_page_is_hashed_in_its_own_lanes(hip, O, B, preset, mode):
    rng = np.random.default_rng(B * 10 + preset)
    k = torch.from_numpy(rng.standard_normal((B, T, H, D)).astype(np.float32)).to(torch.bfloat16)
    v = torch.from_numpy(rng.standard_normal((B, T, H, D)).astype(np.float32)).to(torch.bfloat16)
    th = rng.integers(0, 1 << 62, size=B, dtype=np.int64)
    exp = O.payload_bytes(preset, mode, T * H, D, R, True)
    bits = lambda t: t.contiguous().view(torch.int16).numpy().view(np.uint16)  # noqa: E731
    want = O.egress_batch(bits(k), bits(v), th, dtype=O.BF16, preset=preset, rope_mode=mode, rope_dim=R,
                          expected_payload_bytes=exp, tenant_id_hash=TEN, model_id_hash=MOD, layer_id=LAYER,
                          head_group_id=HG, base_sequence_nonce=BASE, **KEYS)
    dev = torch.device("cuda")
    blobs = torch.full((B, 48 + exp), 0xA5, dtype=torch.uint8, device=dev)
    hip.fused_encode_cold_pages_peak_into(k.to(dev), v.to(dev), torch.from_numpy(th), blobs, preset, mode, R, exp,
                                          TEN, MOD, LAYER, HG, BASE, **KEYS)
    assert np.array_equal(blobs.cpu().numpy(), want)

    bad = sorted({0, B // 2, B - 1})
    tampered = want.copy()
    for i, b in enumerate(bad):
        tampered[b, 32 + (i * 577) % exp] ^= 1 << (i % 8)
    ko = torch.full((B, T, H, D), 7.0, dtype=torch.bfloat16, device=dev)
    vo = torch.full_like(ko, 7.0)
    st = torch.full((B,), -9, dtype=torch.int32, device=dev)
    with pytest.raises(RuntimeError, match="MAC verification failed"):
        hip.fused_decode_cold_pages_peak_into(torch.from_numpy(tampered).to(dev), torch.from_numpy(th), ko, vo, R,
                                              False, TEN, MOD, LAYER, page_status=st, per_page=True, **KEYS)
    want_st = np.zeros(B, dtype=np.int32)
    want_st[bad] = 3
    assert np.array_equal(st.cpu().numpy(), want_st)
    rc, _, ok, ov = O.ingress_batch(want, th, num_tokens=T, num_heads=H, head_dim=D, rope_dim=R,
                                    is_mla_single_buffer=False, dtype=O.BF16, expected_tenant_hash=TEN,
                                    expected_model_hash=MOD, expected_layer_id=LAYER, **KEYS)
    assert rc == 0
    ok, ov = ok.copy(), ov.copy()
    ok[bad], ov[bad] = 0, 0
    assert np.array_equal(bits(ko.cpu()), ok.reshape(B, T, H, D)) and np.array_equal(bits(vo.cpu()), ov.reshape(B, T, H, D))
