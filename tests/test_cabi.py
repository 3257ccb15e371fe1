"""CPU: the C-ABI library loads and exports every symbol declared in include/momoe_hip.h;
host-side argument validation works without a GPU (no compute calls)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "momoe-impl_amd", "momoe_amd", "libmomoe_hip.so")
HEADER = os.path.join(ROOT, "include", "momoe_hip.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(momoe_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        import subprocess, sys
        subprocess.check_call([sys.executable, os.path.join(ROOT, "momoe-impl_amd", "build.py")])
    import torch  # noqa: F401  the HIP runtime the library binds to
    return ctypes.CDLL(LIB)


def test_every_declared_symbol_is_exported(lib):
    names = _declared()
    assert len(names) >= 14
    for n in names:
        assert hasattr(lib, n), n


def test_binding_table_matches_header():
    from momoe_amd import _hip
    assert sorted(_hip.EXPORTED_SYMBOLS) == _declared()
    assert _hip.abi_version() == 3
    assert _hip.status_string(0) == "ok" and "unsupported" in _hip.status_string(2)


def test_size_queries_and_argument_validation(lib):
    lib.momoe_tile_table_ints.restype = ctypes.c_int64
    lib.momoe_index_workspace_bytes.restype = ctypes.c_int64
    i64 = ctypes.c_int64
    assert lib.momoe_tile_table_ints(i64(8192), i64(128), i64(8), 128) == 4 + 4 * (512 + 128)
    assert lib.momoe_index_workspace_bytes(i64(8192), i64(128)) >= (128 * 32 + 8 * 8192) * 4
    # null pointers / bad sizes are rejected on the host before anything is launched
    z = ctypes.c_void_p(0)
    assert lib.momoe_combine(z, z, z, i64(1), i64(8), i64(1), i64(1), z) == 1
    assert lib.momoe_wgrad(z, i64(8), z, z, i64(8), z, z, z, i64(1), i64(1), i64(8), i64(8), i64(1),
                           z, i64(0), z) == 1
    lib.momoe_wgrad_workspace_bytes.restype = ctypes.c_int64
    # at most 8 partial tiles of 256 KiB per workgroup (256), fewer when there are few rows
    assert lib.momoe_wgrad_workspace_bytes(i64(128), i64(2048), i64(2048), i64(65536)) == 2048 * 262144
    assert lib.momoe_wgrad_workspace_bytes(i64(2), i64(64), i64(64), i64(9000)) == 4 * 262144
    assert lib.momoe_wgrad_workspace_bytes(i64(2), i64(64), i64(64), i64(100)) == 0


@pytest.mark.parametrize("H,N,msum,parts", [
    (512, 32, 4096, 8),       # 128 tiles of 256 columns: 64-column parts
    (544, 32, 4096, 5),       # 160 tiles: 128-column parts
    (1024, 128, 65536, 8),
    (64, 8, 256, 1), (96, 8, 256, 2), (2048, 8, 16, 32), (0, 8, 256, -1),
])
def test_parts_of_the_gate_gradient(lib, H, N, msum, parts):
    i64, p = ctypes.c_int64, ctypes.c_void_p
    lib.momoe_gs_parts.restype = i64
    got = lib.momoe_gs_parts(i64(H), i64(N), i64(msum))
    assert got == parts
    if H:  # another number of parts than the two documented ones is refused before any launch
        a = p(4096)
        for n in (0, got + 1, 2 * got + 2):
            if n == -(-H // 128):
                continue
            assert lib.momoe_lin1_swiglu_bwd_parts(a, a, a, a, a, a, i64(1), i64(1), i64(0), a, a, i64(H), a, i64(n),
                                                   i64(256), i64(64), i64(H), i64(N), i64(msum), p(0)) == 1


def test_refusals_of_the_joined_backward_launch(lib):
    """All before any launch."""
    i64, p = ctypes.c_int64, ctypes.c_void_p
    good = dict(Gy=4096, W2=4096, x=4096, W1=4096, idx=4096, table=4096, s=4096, sn=1, sm=1, u=4096, gz=4096, hst=4096, ld=64, gs=4096,
                nparts=1, M=256, D=64, H=64, N=8, msum=512)
    pointers = ("Gy", "W2", "x", "W1", "idx", "table", "s", "u", "gz", "hst", "gs")

    def status(**changed):
        a = {**good, **changed}
        return lib.momoe_dgrad_h_lin1_bwd(*[(p if k in pointers else i64)(v) for k, v in a.items()], p(0))

    fits = lambda **c: lib.momoe_dgrad_h_lin1_bwd_fits(*[i64({**good, **c}[k]) for k in ("M", "D", "H", "N", "msum")])
    assert fits() == 1
    assert all(status(**{k: 0}) == 1 for k in pointers)
    assert all(status(**{k: 4096 + 8}) == 1 for k in ("Gy", "W2", "x", "W1", "u", "gz", "hst"))
    assert status(ld=56) == status(ld=68) == 1
    assert status(M=0) == status(msum=0) == 1 and fits(M=0) == 0
    assert all(status(nparts=n) == 1 for n in (0, 2, -1))
    # the lines: 3072 k-values, one and a half row tiles per expert, one tile per CU; and widths that no kernel takes
    assert fits(D=3040) == 1 and fits(msum=3072) == 1
    for c in (dict(D=3072), dict(msum=3073), dict(H=4096, ld=4096, nparts=64), dict(D=48)):
        assert fits(**c) == 0 and status(**c) == 2, c


def test_host_modules_refuse_cpu_tensors():
    import torch
    import momoe_amd
    layer = momoe_amd.MoMoE(32, 32, 2, 1, Wl1_ND2H=torch.zeros(2, 32, 64), Wl2_NHD=torch.zeros(2, 32, 32))
    with pytest.raises(RuntimeError):
        layer(torch.zeros(1, 4, 32), torch.ones(2, 4, dtype=torch.int32), torch.ones(2, 4))
    with pytest.raises(AssertionError):
        momoe_amd.MoMoE(32, 32, 2, 1, save_percent=101, Wl1_ND2H=torch.zeros(2, 32, 64),
                        Wl2_NHD=torch.zeros(2, 32, 32))
