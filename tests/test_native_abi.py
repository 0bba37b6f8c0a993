"""The C ABI: libnhip.so loads on a machine without a GPU and exports every function include/nhip.h
declares; the ctypes binding names exactly those functions."""

import ctypes as C
import os
import re

from lumen_amd import native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "nhip.h")).read()
    return sorted(set(re.findall(r"^\s*(?:int|const char \*)\s*(nhip_\w+)\(", text, re.M)))


def test_library_exports_every_declared_symbol():
    lib = C.CDLL(native.LIBRARY)
    names = _declared()
    assert len(names) >= 30
    for name in names:
        assert hasattr(lib, name), name


def test_binding_covers_the_header():
    assert sorted(native.SIGNATURES) == _declared()


def test_device_count_without_a_gpu_is_an_answer():
    """nhip_device_count succeeds (0 devices where there is no GPU, as in the build container)."""
    n = native.device_count()
    assert n >= 0


def test_gemm_kernel_says_what_nhip_gemm_would_run():
    """Kinds by dtype, layout, alignment and forced config, with the parameters a generated store needs."""
    def kernel(m, n, k, dt, a=None, b=None, aligned=True, config=-1, z=1):
        d = native.GemmDesc(m=m, n=n, k=k, a_dtype=dt, b_dtype=dt, d_dtype=0, d_m=n, d_n=1, config=config, nbatch=1)
        d.batch[0], d.a_batch[0], d.b_batch[0], d.d_batch[0] = z, m * k, n * k, m * n
        (d.a_m, d.a_k), (d.b_k, d.b_n) = a or (k, 1), b or (1, k)
        out = (C.c_int32 * 3)()
        native.call("nhip_gemm_kernel", C.byref(d), int(aligned), out)
        return tuple(out)

    f32, bf16 = native.NHIP_F32, native.NHIP_BF16
    assert kernel(256, 1024, 512, f32) == (native.NHIP_GEMM_FOLD, 2, 0)
    assert kernel(256, 1024, 512, f32, aligned=False) == (native.NHIP_GEMM_FOLD, 2, 0)
    assert kernel(256, 1024, 512, f32, a=(1024, 2))[0] == native.NHIP_GEMM_EXACT
    for m, n, k, a, b, kind in [(8192, 4096, 31, None, None, "EXACT"), (8192, 4096, 96, None, None, "FOLD"),
                                (1024, 1024, 31, None, None, "EXACT"), (1024, 1024, 32, None, None, "FOLD"),
                                (512, 1024, 1, None, None, "FOLD"), (8192, 8192, 256, None, (8192, 1), "EXACT"),
                                (4096, 4096, 256, None, (4096, 1), "FOLD"), (8192, 4096, 1000, (1, 8192), (4096, 1), "EXACT"),
                                (1024, 1024, 40, (1, 1024), (1024, 1), "FOLD"), (512, 1024, 16, (1, 512), None, "EXACT")]:
        assert kernel(m, n, k, f32, a, b)[0] == getattr(native, f"NHIP_GEMM_{kind}"), (m, n, k)
    assert kernel(16, 4096, 2048, bf16) == (native.NHIP_GEMM_FEW_ROWS, 1, 16)
    few = [(16, 8192, 2048, 1), (16, 2048, 8192, 1), (8, 512, 8192, 1), (32, 4096, 4096, 1), (64, 4096, 2048, 1), (16, 512, 1024, 16),
           (16, 256, 128, 64), (1, 1024, 1024, 64)]
    tiled = [(16, 16384, 4096, 1), (16, 512, 8192, 1), (16, 32000, 2048, 1), (32, 2048, 8192, 1), (64, 2048, 4096, 1), (16, 512, 64, 64),
             (64, 2048, 64, 64), (64, 64, 1024, 64), (32, 512, 128, 64), (8, 512, 64, 64), (65, 512, 512, 1)]
    for cases, kind in ((few, native.NHIP_GEMM_FEW_ROWS), (tiled, native.NHIP_GEMM_TILED)):
        for m, n, k, z in cases:
            assert kernel(m, n, k, bf16, z=z)[0] == kind, (m, n, k, z)
    assert kernel(64, 512, 2048, bf16, config=16) == (native.NHIP_GEMM_FEW_ROWS, 4, 16)
    assert kernel(16, 4096, 2048, bf16, config=3) == (native.NHIP_GEMM_TILED, 3, 0)
    assert kernel(16, 4096, 2048, bf16, aligned=False)[0] == native.NHIP_GEMM_ANY
    assert kernel(4096, 4096, 4096, bf16)[0] == native.NHIP_GEMM_TILED
    assert kernel(300, 5003, 511, bf16)[0] == native.NHIP_GEMM_ANY
    assert kernel(300, 500, 0, bf16)[0] == native.NHIP_GEMM_EXACT


def test_forwards_divide_their_keys_where_the_general_kernel_is_slower():
    """Few query rows over many keys, and not the shapes measured slower that way (many row tiles), nor a forced tile."""
    def divides(b, sq, sk, n, nkv, d, config=-1):
        a = native.AttnDesc(batch=b, heads=n, kv_heads=nkv, sq=sq, sk=sk, head_dim=d, dtype=1, causal=1, scale=1.0, config=config)
        out = C.c_int()
        native.call("nhip_flash_fwd_divides_keys", C.byref(a), C.byref(out))
        return bool(out.value)

    for shape in [(16, 1, 4096, 16, 16, 128), (1, 1, 4096, 16, 16, 128), (3, 1, 27958, 16, 16, 128), (21, 1, 963, 32, 8, 64),
                  (1, 1000, 1000, 4, 1, 64), (1, 333, 2100, 4, 1, 128), (3, 4, 517, 8, 2, 64), (16, 1, 1200, 32, 32, 40)]:
        assert divides(*shape) and not divides(*shape, config=0), shape
    for shape in [(2, 8310, 8310, 4, 1, 40), (26, 599, 1661, 4, 1, 40), (2, 317, 21981, 32, 32, 96), (1, 1156, 1895, 16, 16, 64),
                  (12, 60, 3355, 32, 32, 64), (2, 1194, 23358, 32, 8, 64), (4, 512, 512, 8, 8, 128), (2, 1777, 1777, 16, 4, 64),
                  (2, 58, 58, 16, 16, 64), (1, 1, 1, 1, 1, 64), (1, 1, 4096, 16, 16, 256)]:
        assert not divides(*shape), shape
