// ztcp_ragged.hip -- egress / ingress of pages whose layout is not cut into
// whole 64-byte units (T*H not a multiple of 32 for some section, payload
// padding, blob sizes that are not multiples of 16, unaligned pointers), with
// the pages' payloads in LDS.
//
// The row pipeline's rows do not exist here: a group's codes and its scale
// lie at any even payload offset.  A workgroup therefore keeps the whole
// payload of each of its pages in LDS, where the two ways of cutting it meet:
//   egress:  thread = group: quantize, codes and scale to their places; then
//            thread = 64-byte block: keystream, XOR, ciphertext to the blob
//            and back to LDS; then one wave hashes the pages from LDS.
//   ingress: thread = 64-byte block: ciphertext to LDS, decrypted to a second
//            copy; then one wave verifies the pages from the first copy while
//            the others dequantize the groups of the second.
// The steps are separated by workgroup barriers, so there are no bounded
// waits.  What lasts is the SipHash chain of a page, two lanes per page
// (SipPair): a workgroup holds one page until every SIMD of the chip has one,
// then more (ragged_pages); its hashing wave is another one of its four with
// every workgroup per CU or so, and those of one CU land on different
// SIMDs.  Against the layout-agnostic kernels (ztcp_generic.hip: one thread
// per page and byte loads for the hash, byte arrays in scratch memory for the
// blocks): 333 pages of 10,708 bytes egress 925 -> 115 us, 1,200 pages of
// 2,988 bytes ingress 238 -> 104 us.  Those remain for pages that do not fit
// the LDS, for batches of many rounds of large pages, and as the definition
// of the path.
#include "ztcp_params.h"
#include "ztcp_ragged.h"

namespace ztcp {

namespace {

constexpr int kRgThreads = 256;
constexpr int kRgZero = 0;                      // [16] zero words: the message of the hashing wave's A lanes
constexpr int kRgPages = 16;                    // egress: the payloads; ingress: the layouts first
constexpr int kRgLayoutWords = (int)((sizeof(Layout) / 4 + 4) & ~3);  // Layout, then its index (or -1)
static_assert(kRgPages * 4 == (int)kRaggedFixed, "LDS beside the pages");

// 16 bytes at any address (the hardware's unaligned access; never outside the
// 16 bytes).
struct __attribute__((packed)) Unaligned16 { uint32_t w[4]; };
typedef __attribute__((address_space(1))) Unaligned16 GlobalUnaligned16;

__device__ __forceinline__ uint4 ldu16(const uint8_t* p) {
    const GlobalUnaligned16* g = (const GlobalUnaligned16*)p;
    return make_uint4(g->w[0], g->w[1], g->w[2], g->w[3]);
}
__device__ __forceinline__ void stu16(uint8_t* p, uint4 v) {
    GlobalUnaligned16* g = (GlobalUnaligned16*)p;
    g->w[0] = v.x;
    g->w[1] = v.y;
    g->w[2] = v.z;
    g->w[3] = v.w;
}
// N words at an even LDS address.
template <int N>
__device__ __forceinline__ void lds_put2(uint8_t* dst, const uint32_t* w) {
    uint16_t* h = reinterpret_cast<uint16_t*>(dst);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        h[2 * i] = (uint16_t)w[i];
        h[2 * i + 1] = (uint16_t)(w[i] >> 16);
    }
}
template <int N>
__device__ __forceinline__ void lds_get2(const uint8_t* src, uint32_t* w) {
    const uint16_t* h = reinterpret_cast<const uint16_t*>(src);
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = (uint32_t)h[2 * i] | ((uint32_t)h[2 * i + 1] << 16);
}

__device__ __forceinline__ void load_chunk(const uint8_t* p, uint32_t (&w)[8]) {
    const uint4 a = ldu16(p), b = ldu16(p + 16);
    w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
    w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
}
__device__ __forceinline__ void store_chunk(uint8_t* p, const uint32_t* o) {
    stu16(p, make_uint4(o[0], o[1], o[2], o[3]));
    stu16(p + 16, make_uint4(o[4], o[5], o[6], o[7]));
}

// Group g of section S quantized from `buf` into the page's payload `pay` (LDS).
template <int DT>
__device__ __forceinline__ void quantize_group(const Section& S, const uint8_t* buf, int32_t head_dim, uint32_t g,
                                               uint8_t* pay) {
    const uint32_t ges = (uint32_t)group_elems(S.kind), gpvec = (uint32_t)S.gpv * 16u / ges;  // groups per vector
    const uint32_t vec = g / gpvec, gi = g - vec * gpvec;
    const uint8_t* src = buf + ((size_t)vec * (uint32_t)head_dim + (uint32_t)S.col + gi * ges) * 2u;
    uint8_t* codes = pay + S.q_off + g * (uint32_t)code_bytes_per_group(S.kind);
    uint8_t* prm = pay + S.s_off + g * (uint32_t)param_bytes_per_group(S.kind);
    uint32_t w[4][8], q[16], sc;
    load_chunk(src, w[0]);
    if (S.kind == kSecRaw) {
        lds_put2<8>(codes, w[0]);
        return;
    }
    if (S.kind == kSecInt8) {
        sc = quant_group_int8<DT>(w[0], q);
        lds_put2<4>(codes, q);
    } else if (S.kind == kSecInt4) {
        sc = quant_group_int4<DT>(w[0], q);
        lds_put2<2>(codes, q);
    } else if (S.kind == kSecE4m3) {
        sc = quant_group_e4m3<DT>(w[0], q);
        lds_put2<4>(codes, q);
    } else if (S.kind == kSecInt4G32) {
        load_chunk(src + 32, w[1]);
        sc = quant_group32_int4<DT>(w[0], w[1], q);
        lds_put2<4>(codes, q);
    } else {
        load_chunk(src + 32, w[1]);
        load_chunk(src + 64, w[2]);
        load_chunk(src + 96, w[3]);
        sc = quant_group64_asym8<DT>(w, q);
        lds_put2<16>(codes, q);
        reinterpret_cast<uint16_t*>(prm)[1] = (uint16_t)(sc >> 16);
    }
    reinterpret_cast<uint16_t*>(prm)[0] = (uint16_t)sc;
}

// SipHash of one page per lane pair: the header's four words, then the
// payload in LDS (`mine`: this lane's page in B lanes, the zero row in A
// lanes; `step` words per 64-byte row).
__device__ __forceinline__ void hash_page(SipPair& s, const uint64_t (&hdr)[4], const uint32_t* mine, int32_t step,
                                          uint32_t payload, uint64_t& lo, uint64_t& hi) {
    s.absorb_words<4>(hdr);
    auto fetch = [&](uint4 (&x)[4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = *reinterpret_cast<const uint4*>(mine + 4 * q);
        mine += step;
    };
    sip_stream64(s, payload / 64u, fetch);
    // the last payload % 64 bytes, then the final word (cpp:458-470)
    const uint32_t tail = payload & 63u;
#pragma unroll 1
    for (uint32_t i = 0; i < tail / 8u; ++i) s.absorb((uint64_t)mine[2 * i] | ((uint64_t)mine[2 * i + 1] << 32));
    uint64_t last = (uint64_t)((kHeader + payload) & 0xFFu) << 56;
    const uint8_t* end = reinterpret_cast<const uint8_t*>(mine + (tail / 8u) * 2u);
#pragma unroll 1
    for (uint32_t b = 0; b < (tail & 7u); ++b) last |= (uint64_t)end[b] << (8 * b);
    s.finish(last, lo, hi);
}

// The wave of the workgroup that hashes: another one with every 2^k
// workgroups, 2^k <= CUs (a division by the CU count costs 1 % of a launch of
// 333 pages).
__device__ __forceinline__ int hash_wave(int cu_count) {
    return (int)(blockIdx.x >> (31 - __builtin_clz((uint32_t)cu_count))) & 3;
}

template <int DT>
__global__ __launch_bounds__(kRgThreads) void egress_ragged_kernel(EgressParams p) {
    extern __shared__ __align__(16) uint32_t lds[];
    const int64_t page0 = (int64_t)blockIdx.x * p.ppw;
    const int np = (int)min((int64_t)p.ppw, p.batch - page0);
    const uint32_t stride = ragged_page_words(p.payload), nblk = (p.payload + 63u) / 64u;
    if (threadIdx.x < 16) lds[kRgZero + threadIdx.x] = 0u;
    // the bytes after the last section (padding, the last block's rest) are zero
    for (int i = 0; i < np; ++i) {
        uint8_t* pay = reinterpret_cast<uint8_t*>(lds + kRgPages + i * stride);
        for (uint32_t b = p.lay.required + threadIdx.x; b < nblk * 64u; b += kRgThreads) pay[b] = 0;
    }
    for (int i = 0; i < np; ++i) {
        const EgressPage pg = egress_page(p, page0 + i);
        uint8_t* pay = reinterpret_cast<uint8_t*>(lds + kRgPages + i * stride);
#pragma unroll 1
        for (int si = 0; si < p.lay.n_sec; ++si) {
            const Section S = pick(si == 0, p.lay.sec[0], pick(si == 1, p.lay.sec[1], p.lay.sec[2]));
            const uint32_t n = (uint32_t)S.n_groups;
#pragma unroll 1
            for (uint32_t g = threadIdx.x; g < n; g += kRgThreads)
                quantize_group<DT>(S, S.src ? pg.v : pg.k, p.head_dim, g, pay);
        }
    }
    __syncthreads();
    for (int i = 0; i < np; ++i) {
        const EgressPage pg = egress_page(p, page0 + i);
#pragma unroll 1
        for (uint32_t b = threadIdx.x; b < nblk; b += kRgThreads) {
            uint32_t ks[16];
            chacha_block(p.key, 1u + b, (uint32_t)pg.seq, (uint32_t)(pg.seq >> 32), pg.nonce2, ks);
            uint32_t* row = lds + kRgPages + i * stride + b * 16u;
            uint8_t* dst = pg.blob + kHeader + 64u * b;
            uint4 x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint4 t = *reinterpret_cast<const uint4*>(row + 4 * q);
                x[q] = make_uint4(t.x ^ ks[4 * q], t.y ^ ks[4 * q + 1], t.z ^ ks[4 * q + 2], t.w ^ ks[4 * q + 3]);
                *reinterpret_cast<uint4*>(row + 4 * q) = x[q];
            }
            const uint32_t n = min(64u, p.payload - 64u * b);
            if (n == 64u) {
#pragma unroll
                for (int q = 0; q < 4; ++q) stu16(dst + 16 * q, x[q]);
            } else {
                const uint8_t* bytes = reinterpret_cast<const uint8_t*>(row);
#pragma unroll 1
                for (uint32_t k = 0; k < n; ++k) dst[k] = bytes[k];
            }
        }
    }
    __syncthreads();
    if ((int)(threadIdx.x >> 6) != hash_wave(p.cu_count)) return;
    __builtin_amdgcn_s_setprio(3);
    const int pl = (int)(threadIdx.x & 63) >> 1;
    const bool b = SipPair::lane_b();
    const EgressPage pg = egress_page(p, page0 + (pl < np ? pl : 0));
    const uint64_t hdr[4] = {p.hdr0, pg.hdr1, pg.token, pg.seq};
    SipPair s;
    s.init(p.mk0, p.mk1);
    uint64_t lo, hi;
    hash_page(s, hdr, b ? lds + kRgPages + (pl < np ? pl : 0) * stride : lds + kRgZero, b ? 16 : 0, p.payload, lo, hi);
    if (b && pl < np) {
        stu16(pg.blob, make_uint4((uint32_t)hdr[0], (uint32_t)(hdr[0] >> 32), (uint32_t)hdr[1], (uint32_t)(hdr[1] >> 32)));
        stu16(pg.blob + 16,
              make_uint4((uint32_t)hdr[2], (uint32_t)(hdr[2] >> 32), (uint32_t)hdr[3], (uint32_t)(hdr[3] >> 32)));
        stu16(pg.blob + kHeader + p.payload,
              make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)));
    }
}

// Group g of section S dequantized from the page's plaintext `pay` (LDS).
template <int DT>
__device__ __forceinline__ void dequantize_group(const Section& S, const uint8_t* pay, uint32_t g, uint8_t* buf,
                                                 int32_t head_dim) {
    const uint32_t ges = (uint32_t)group_elems(S.kind), gpvec = (uint32_t)S.gpv * 16u / ges;
    const uint32_t vec = g / gpvec, gi = g - vec * gpvec;
    uint8_t* dst = buf + ((size_t)vec * (uint32_t)head_dim + (uint32_t)S.col + gi * ges) * 2u;
    const uint8_t* codes = pay + S.q_off + g * (uint32_t)code_bytes_per_group(S.kind);
    const uint8_t* pr = pay + S.s_off + g * (uint32_t)param_bytes_per_group(S.kind);
    uint32_t q[16], o[8];
    if (S.kind == kSecRaw) {
        lds_get2<8>(codes, q);
        store_chunk(dst, q);
        return;
    }
    uint32_t prm = reinterpret_cast<const uint16_t*>(pr)[0];
    const bool nans = (prm & 0x7C00u) == 0x7C00u;  // an inf / NaN scale: NaN outputs as the reference writes them
    if (S.kind == kSecAsym8) {
        prm |= (uint32_t) reinterpret_cast<const uint16_t*>(pr)[1] << 16;
        lds_get2<16>(codes, q);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            dequant_asym8_16<DT>(q + 4 * c, prm, o);
            if (nans) canonical_nans<DT>(o);
            store_chunk(dst + 32 * c, o);
        }
        return;
    }
    if (S.kind == kSecInt4) {
        lds_get2<2>(codes, q);
        dequant_group_int4<DT>(q, prm, o);
    } else {
        lds_get2<4>(codes, q);
        if (S.kind == kSecInt8) dequant_group_int8<DT>(q, prm, o);
        else if (S.kind == kSecE4m3) dequant_group_e4m3<DT>(q, prm, o);
        else dequant_group_int4<DT>(q, prm, o);  // the first half of an int4 group of 32
    }
    if (nans) canonical_nans<DT>(o);
    store_chunk(dst, o);
    if (S.kind == kSecInt4G32) {
        dequant_group_int4<DT>(q + 2, prm, o);
        if (nans) canonical_nans<DT>(o);
        store_chunk(dst + 32, o);
    }
}

// Two words of a blob's header (bytes 16 i .. 16 i + 15).
__device__ __forceinline__ uint4 header_quad(const uint8_t* blob, int i) { return ldu16(blob + 16 * i); }

__device__ __forceinline__ int32_t header_layout(const IngressParams& p, uint32_t h0x) {
    const uint32_t preset = (h0x >> 24) & 0x0Fu, rope_mode = h0x >> 28;
    if (!flags_valid(preset, rope_mode)) return -1;
    const int32_t li = (int32_t)((preset - 1u) * 4u + rope_mode);
    return ((p.lay_ok >> li) & 1u) ? li : -1;
}

// status: one entry per page of the batch.  Failing pages are zeroed by the
// caller's next kernel.
template <int DT>
__global__ __launch_bounds__(kRgThreads) void ingress_ragged_kernel(IngressParams p, int32_t* status) {
    extern __shared__ __align__(16) uint32_t lds[];
    const int64_t page0 = (int64_t)blockIdx.x * p.ppw;
    const int np = (int)min((int64_t)p.ppw, p.batch - page0);
    const uint32_t stride = ragged_page_words(p.payload), nblk = (p.payload + 63u) / 64u;
    uint32_t* cts = lds + kRgPages + p.ppw * kRgLayoutWords;  // ciphertexts, then plaintexts
    uint32_t* pts = cts + p.ppw * stride;
    if (threadIdx.x < 16) lds[kRgZero + threadIdx.x] = 0u;
    if ((int)threadIdx.x < np) {  // every page's layout, from its own header
        const int32_t li = header_layout(p, header_quad(ingress_blob(p, page0 + threadIdx.x), 0).x);
        uint32_t* w = lds + kRgPages + threadIdx.x * kRgLayoutWords;
        if (li >= 0) *reinterpret_cast<Layout*>(w) = ingress_layout(p, li);
        w[sizeof(Layout) / 4] = (uint32_t)li;
    }
    for (int i = 0; i < np; ++i) {
        const uint8_t* blob = ingress_blob(p, page0 + i);
        const uint4 h0 = header_quad(blob, 0), h1 = header_quad(blob, 1);
        const uint32_t n2 = ((h0.w & 0xFFFFu) << 16) | (h0.w >> 16);  // nonce (cpp:2357-2365)
#pragma unroll 1
        for (uint32_t b = threadIdx.x; b < nblk; b += kRgThreads) {
            const uint8_t* src = blob + kHeader + 64u * b;
            uint32_t* ct = cts + i * stride + b * 16u;
            const uint32_t n = min(64u, p.payload - 64u * b);
            uint4 x[4];
            if (n == 64u) {
#pragma unroll
                for (int q = 0; q < 4; ++q) x[q] = ldu16(src + 16 * q);
#pragma unroll
                for (int q = 0; q < 4; ++q) *reinterpret_cast<uint4*>(ct + 4 * q) = x[q];
            } else {
                uint8_t* bytes = reinterpret_cast<uint8_t*>(ct);
#pragma unroll 1
                for (uint32_t k = 0; k < 64u; ++k) bytes[k] = k < n ? src[k] : (uint8_t)0;
#pragma unroll
                for (int q = 0; q < 4; ++q) x[q] = *reinterpret_cast<const uint4*>(ct + 4 * q);
            }
            uint32_t ks[16];
            chacha_block(p.key, 1u + b, h1.z, h1.w, n2, ks);
            uint32_t* pt = pts + i * stride + b * 16u;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<uint4*>(pt + 4 * q) = make_uint4(x[q].x ^ ks[4 * q], x[q].y ^ ks[4 * q + 1],
                                                                   x[q].z ^ ks[4 * q + 2], x[q].w ^ ks[4 * q + 3]);
        }
    }
    __syncthreads();
    const int wave = (int)(threadIdx.x >> 6), hw = hash_wave(p.cu_count);
    if (wave != hw) {  // the other three waves dequantize
        const int t0 = (wave - (wave > hw ? 1 : 0)) * 64 + (int)(threadIdx.x & 63);
        for (int i = 0; i < np; ++i) {
            const uint32_t* w = lds + kRgPages + i * kRgLayoutWords;
            if ((int32_t)w[sizeof(Layout) / 4] < 0) continue;
            const Layout& L = *reinterpret_cast<const Layout*>(w);
            const uint8_t* pay = reinterpret_cast<const uint8_t*>(pts + i * stride);
#pragma unroll 1
            for (int si = 0; si < L.n_sec; ++si) {
                const Section S = L.sec[si];
                uint8_t* buf = S.src ? ingress_v(p, page0 + i) : ingress_k(p, page0 + i);
#pragma unroll 1
                for (uint32_t g = (uint32_t)t0; g < (uint32_t)S.n_groups; g += kRgThreads - 64)
                    dequantize_group<DT>(S, pay, g, buf, p.head_dim);
            }
        }
        return;
    }
    __builtin_amdgcn_s_setprio(3);
    const int pl = (int)(threadIdx.x & 63) >> 1;
    const bool bl = SipPair::lane_b();
    const int64_t page = page0 + (pl < np ? pl : 0);
    const uint8_t* blob = ingress_blob(p, page);
    const uint4 h0 = header_quad(blob, 0), h1 = header_quad(blob, 1), tag = ldu16(blob + kHeader + p.payload);
    const uint64_t tok = ingress_token(p, page);
    const uint32_t layer = ingress_layer(p, page);
    const uint64_t hdr[4] = {lo64(h0), hi64(h0), lo64(h1), hi64(h1)};
    SipPair s;
    s.init(p.mk0, p.mk1);
    uint64_t lo, hi;
    hash_page(s, hdr, bl ? cts + (pl < np ? pl : 0) * stride : lds + kRgZero, bl ? 16 : 0, p.payload, lo, hi);
    if (!bl || pl >= np) return;
    // the reference's order (cpp:2313-2355)
    int32_t st = 0;
    if ((h0.x & 0xFFFFu) != kMagic || ((h0.x >> 16) & 0xFFu) != kVersion) st = 1;
    else if (h0.y != p.exp_tenant || h0.z != p.exp_model || (h0.w & 0xFFFFu) != layer || lo64(h1) != tok) st = 2;
    else if (lo64(tag) != lo || hi64(tag) != hi) st = 3;
    else if (header_layout(p, h0.x) < 0) st = 1;
    status[page] = st;
    if (st != 0) atomicMin(&p.call->fail, ((unsigned long long)page << 8) | (unsigned long long)st);
}

}  // namespace

// False when the batch is not for these kernels (ragged_pages): the caller
// then uses the layout-agnostic ones.
bool launch_egress_ragged(const EgressParams& p0, int dtype, hipStream_t s) {
    EgressParams p = p0;
    const size_t bytes = ragged_page_bytes(p.payload, false, 0);
    p.ppw = ragged_pages(p.batch, bytes, false, p.cu_count);
    if (p.ppw == 0) return false;
    const dim3 g((uint32_t)((p.batch + p.ppw - 1) / p.ppw)), b(kRgThreads);
    const size_t lds = (size_t)kRgPages * 4 + (size_t)p.ppw * bytes;
    if (dtype == kHotBf16) hipLaunchKernelGGL(egress_ragged_kernel<kHotBf16>, g, b, lds, s, p);
    else hipLaunchKernelGGL(egress_ragged_kernel<kHotFp16>, g, b, lds, s, p);
    return true;
}

bool launch_ingress_ragged(const IngressParams& p0, int dtype, int32_t* status, hipStream_t s) {
    IngressParams p = p0;
    const size_t bytes = ragged_page_bytes(p.payload, true, kRgLayoutWords);
    p.ppw = ragged_pages(p.batch, bytes, true, p.cu_count);
    if (p.ppw == 0) return false;
    const dim3 g((uint32_t)((p.batch + p.ppw - 1) / p.ppw)), b(kRgThreads);
    const size_t lds = (size_t)kRgPages * 4 + (size_t)p.ppw * bytes;
    if (dtype == kHotBf16) hipLaunchKernelGGL(ingress_ragged_kernel<kHotBf16>, g, b, lds, s, p, status);
    else hipLaunchKernelGGL(ingress_ragged_kernel<kHotFp16>, g, b, lds, s, p, status);
    return true;
}

}  // namespace ztcp
