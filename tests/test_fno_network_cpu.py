"""The calls of csrc/fno_network.h without a GPU: exported, and bad arguments
refused before any launch."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "copara-cgfd3d_amd", "csrc", "fno_network.h")
LIB = os.path.join(ROOT, "copara-cgfd3d_amd", "libcgfd_fno.so")

pytestmark = pytest.mark.skipif(not os.path.exists(LIB), reason="libcgfd_fno.so not built")


@pytest.fixture(scope="module")
def lib():
    import surrogate
    return surrogate.load_library()


def test_every_declared_call_is_exported(lib):
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    names = re.findall(r"\b(cgfd_fno_\w+)\s*\(", text)
    assert sorted(set(names)) == ["cgfd_fno_encode", "cgfd_fno_fourier_bwd", "cgfd_fno_fourier_fwd", "cgfd_fno_linear_bwd",
                                  "cgfd_fno_linear_fwd", "cgfd_fno_weight_rows"]
    assert all(hasattr(lib, n) for n in names)


def _layer(cls, **over):
    arg = cls(*[v for v in (2, 16, 16, 8, 4, 0)])
    for name, kind in cls._fields_:
        if kind is ctypes.c_void_p:
            setattr(arg, name, 4096)  # never read: every call below is refused first
    for name, v in over.items():
        setattr(arg, name, v)
    return arg


BAD_SIZES = [dict(B=0), dict(C=12), dict(C=264), dict(modes=0), dict(modes=9), dict(H=7), dict(W=6), dict(B=65535)]


@pytest.mark.parametrize("over", BAD_SIZES)
def test_fourier_layers_refuse_sizes(lib, over):
    import surrogate
    for cls, fn in ((surrogate._Forward, lib.cgfd_fno_fourier_fwd), (surrogate._Backward, lib.cgfd_fno_fourier_bwd)):
        assert fn(ctypes.byref(_layer(cls, **over)), None) == -1
        assert fn(None, None) == -1


FREE = {"_Forward": {"w", "bias", "sp"}, "_Backward": {"gy", "pre", "wpart", "bpart", "gw", "gb"}}  # at any element
OPTIONAL = {"_Forward": {"sp", "y", "pre"}, "_Backward": {"pre"}}


@pytest.mark.parametrize("name", ["_Forward", "_Backward"])
def test_fourier_layers_refuse_null_and_misaligned_pointers(lib, name):
    import surrogate
    cls = getattr(surrogate, name)
    fn = lib.cgfd_fno_fourier_fwd if name == "_Forward" else lib.cgfd_fno_fourier_bwd
    for field, kind in cls._fields_:
        if kind is not ctypes.c_void_p:
            continue
        if field not in OPTIONAL[name]:
            assert fn(ctypes.byref(_layer(cls, **{field: None})), None) == -1, field
        if field not in FREE[name]:
            for off in (4, 8):
                assert fn(ctypes.byref(_layer(cls, **{field: 4096 + off})), None) == -1, (field, off)
    if name == "_Forward":  # modes that end in two launches need the buffers between them
        for field in ("sp", "y"):
            assert fn(ctypes.byref(_layer(cls, modes=5, **{field: None})), None) == -1, field


def test_linear_layers_and_encoding_refuse_bad_arguments(lib):
    p = 4096
    fwd = lambda xb=p, wb=p, b=p, pre=p, act=1, yb=p, R=8, K=8, N=8: lib.cgfd_fno_linear_fwd(xb, wb, b, pre, act, yb, R, K, N, None)  # noqa: E731
    for bad in (dict(xb=None), dict(wb=None), dict(b=None), dict(yb=None), dict(R=0), dict(R=64 * 65536), dict(K=0),
                dict(N=0), dict(N=6), dict(act=2), dict(b=p + 4), dict(pre=p + 8), dict(yb=p + 4)):
        assert fwd(**bad) == -1, bad
    ptrs = ("gy", "pre", "xb", "wb", "gz", "gzb", "wpart", "bpart", "gx", "gw", "gb")

    def bwd(R=8, K=8, N=8, **over):
        return lib.cgfd_fno_linear_bwd(*[over.get(n, p) for n in ptrs], R, K, N, None)

    for n in ptrs:
        if n not in ("pre", "gz", "gx"):
            assert bwd(**{n: None}) == -1, n
    for bad in (dict(R=0), dict(R=64 * 65536), dict(K=0), dict(K=64 * 65536), dict(N=0), dict(N=257)):
        assert bwd(**bad) == -1, bad
    for bad in ((0, 8, 8), (8, 0, 8), (8, 8, 0)):
        assert lib.cgfd_fno_weight_rows(*bad) == -1
    enc = lambda src=p, out=p, n=1, wi=4, wj=4, L=1.0: lib.cgfd_fno_encode(src, out, n, 0, 0, wi, wj, 1.0, L, None)  # noqa: E731
    for bad in (dict(src=None), dict(out=None), dict(n=-1), dict(n=65536), dict(wi=0), dict(wj=0), dict(L=0.0)):
        assert enc(**bad) == -1, bad
    assert enc(n=0) == 0  # nothing to do
