"""What a call returns when its kernels did not run (no GPU).

The host side of the C ABI (ztcp_abi.hip) is linked with a stand-in for the HIP
runtime and the launchers, whose launches and synchronisations all succeed
and do only what the test asks for.  A synchronous ingress must then not
report success unless its verdict was written; an asynchronous egress must
not give its kernels a word that a later call reads.
"""
import ctypes as C
import re
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT / "vlx-tee_amd"))
import build as B  # noqa: E402  (vlx-tee_amd/build.py: the library's compiler flags)

CSRC = ROOT / "vlx-tee_amd" / "csrc"
HIPCC = shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if Path("/opt/rocm/bin/hipcc").exists() else None)
pytestmark = pytest.mark.skipif(HIPCC is None, reason="hipcc not available")

STAND_IN = r"""
#include <cstdlib>
#include <cstring>
#include "ztcp_params.h"
using namespace ztcp;
static int g_write = 0;            // the stand-in device leaves a verdict: 1 all pages pass, 2 page 3 has status 2
static void* g_sink = nullptr;     // call_diag of the last egress launch
static int g_expire = 0, g_zeroed = 0;
static CallState* g_calls = nullptr;
static void leave(CallState* h) { h->fail = g_write == 2 ? (3ull << 8 | 2ull) : ~0ull; h->diag = 0u; }
extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipFreeAsync(void*, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (g_write) leave((CallState*)d);
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = calloc(1, 1 << 20); return hipSuccess; }
__attribute__((visibility("default"))) void set_mode(int write, int expire) { g_write = write; g_expire = expire; g_zeroed = 0; }
__attribute__((visibility("default"))) void* last_sink() { return g_sink; }
__attribute__((visibility("default"))) int zeroed() { return g_zeroed; }
}
namespace ztcp {
hipError_t launch_egress_fused(const EgressParams& p, int, hipStream_t) {
    g_sink = p.sink.call_diag;
    if (g_expire && p.sink.call_diag) *p.sink.call_diag = p.sink.call_tag;
    return hipSuccess;
}
hipError_t launch_ingress_fused(const IngressParams&, int, hipStream_t) { return hipSuccess; }
hipError_t launch_egress_generic(const EgressParams&, int, hipStream_t) { return hipSuccess; }
bool launch_egress_ragged(const EgressParams&, int, hipStream_t) { return true; }
bool launch_ingress_ragged(const IngressParams&, int, int32_t*, hipStream_t) { return true; }
hipError_t launch_egress_zero_blobs(const EgressParams&, hipStream_t) { ++g_zeroed; return hipSuccess; }
hipError_t launch_ingress_generic_impl(const IngressParams&, int, int32_t*, hipStream_t) { return hipSuccess; }
hipError_t launch_ingress_finalize(const IngressParams& p, hipStream_t) {
    if (g_write && p.host_call) leave(p.host_call);
    return hipSuccess;
}
hipError_t launch_reset_call(CallState*, hipStream_t) { return hipSuccess; }
hipError_t launch_publish_call(const CallState*, CallState* h, hipStream_t) {
    if (g_write) leave(h);
    return hipSuccess;
}
hipError_t launch_chacha_xor(const uint8_t*, uint8_t*, size_t, ChaKey, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t) { return hipSuccess; }
hipError_t launch_selftest(unsigned int*, hipStream_t) { return hipSuccess; }
hipError_t launch_siphash(const uint8_t*, size_t, uint64_t, uint64_t, uint8_t*, hipStream_t) { return hipSuccess; }
}
"""


class Geo(C.Structure):
    _fields_ = [("num_tokens", C.c_int64), ("num_heads", C.c_int64), ("head_dim", C.c_int64),
                ("rope_dim", C.c_int64), ("hot_dtype", C.c_int32), ("is_mla_single_buffer", C.c_int32)]


class Keys(C.Structure):
    _fields_ = [(n, C.c_uint64) for n in ("k0", "k1", "k2", "k3", "mk0", "mk1")]


class Aad(C.Structure):
    _fields_ = [("tenant_id_hash", C.c_uint32), ("model_id_hash", C.c_uint32), ("layer_id", C.c_uint16),
                ("head_group_id", C.c_uint16)]


@pytest.fixture(scope="module")
def abi(tmp_path_factory):
    d = tmp_path_factory.mktemp("abi")
    (d / "stand_in.hip").write_text(STAND_IN)
    objs = []
    for src in (CSRC / "ztcp_abi.hip", d / "stand_in.hip"):
        o = d / (src.name + ".o")
        subprocess.run([HIPCC, *B.HIPCC_FLAGS, "-I", str(CSRC), "-I", str(ROOT / "include"), "-c", str(src),
                        "-o", str(o)], check=True, capture_output=True)
        objs.append(str(o))
    # -Bsymbolic: every call inside the library binds to the stand-ins
    out = d / "libabi.so"
    subprocess.run([HIPCC, "-shared", "-fPIC", *objs, "-Wl,-Bsymbolic", "-o", str(out)], check=True, capture_output=True)
    L = C.CDLL(str(out))
    L.last_sink.restype = C.c_void_p
    return L


DA, DB, DC, DD = (0x100000000 * i for i in (1, 2, 3, 4))  # device addresses, never dereferenced
GEO = Geo(16, 8, 128, 64, 0, 0)
KEYS = Keys(1, 2, 3, 4, 5, 6)


def _ingress(L, geo=GEO, flags=0, status=None, fn="ztcp_ingress_peak_into", blob=None):
    blob = blob or L.ztcp_blob_bytes(C.byref(geo), C.c_int64(2), C.c_int64(1))
    return getattr(L, fn)(C.c_void_p(DA), C.c_int64(blob), C.c_void_p(DB), C.c_void_p(DC), C.c_void_p(DD), C.c_int64(8),
                          C.byref(geo), C.c_uint32(1), C.c_uint32(2), C.c_uint16(3), C.byref(KEYS), C.c_void_p(status),
                          C.c_uint32(flags), None)


def _egress(L, flags=0):
    pay = L.ztcp_payload_bytes(C.byref(GEO), C.c_int64(2), C.c_int64(1))
    return L.ztcp_egress_peak_into_ext(C.c_void_p(DA), C.c_void_p(DB), C.c_void_p(DC), C.c_void_p(DD), C.c_int64(8),
                                       C.byref(GEO), C.c_int64(2), C.c_int64(1), C.c_int64(pay),
                                       C.byref(Aad(1, 2, 3, 4)), C.c_uint64(5), C.byref(KEYS), C.c_uint32(flags), None)


def _constants():
    t = (ROOT / "include" / "ztcp.h").read_text()
    get = lambda n: int(re.search(rf"{n}\s*=?\s*\(?(-?(?:0x)?[0-9a-fA-F]+)", t).group(1), 0)  # noqa: E731
    return {n: get(n) for n in ("ZTCP_EHIP", "ZTCP_EDEVICE", "ZTCP_ASYNC", "ZTCP_PER_PAGE")}


K = _constants()


@pytest.mark.parametrize("fn", ["ztcp_ingress_peak_into", "ztcp_ingress_peak_into_noalloc"])
@pytest.mark.parametrize("per_page", [False, True])
@pytest.mark.parametrize("aligned", [True, False])
def test_an_unwritten_verdict_is_no_success(abi, fn, per_page, aligned):
    geo = GEO if aligned else Geo(7, 3, 80, 16, 0, 0)
    flags = K["ZTCP_PER_PAGE"] if per_page else 0
    abi.set_mode(1, 0)
    for _ in range(70):  # every slot once: a passing verdict left in each
        assert _ingress(abi, geo, flags, fn=fn) == 0
    abi.set_mode(2, 0)
    assert _ingress(abi, geo, flags, fn=fn) == 2
    abi.set_mode(0, 0)
    for _ in range(70):
        assert _ingress(abi, geo, flags, fn=fn) == K["ZTCP_EHIP"]


def test_asynchronous_egress_leaves_no_word_behind(abi):
    abi.set_mode(1, 1)
    assert _egress(abi) == K["ZTCP_EDEVICE"] and abi.zeroed() == 1  # the expiry is seen by the call that had it
    word = C.cast(abi.last_sink(), C.POINTER(C.c_uint32))
    assert word
    abi.set_mode(1, 0)
    assert _egress(abi) == 0
    assert _egress(abi, K["ZTCP_ASYNC"]) == 0 and not abi.last_sink()
