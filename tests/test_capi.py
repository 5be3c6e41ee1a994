"""CPU checks of the C-ABI boundary: the library loads, exports every symbol the
header declares, and the Python mirror/drop-in reject bad input like the
reference does (no GPU compute here)."""
import ctypes
import os
import re
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "loom_hip.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(loom_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from loom_amd import _lib
    lib = _lib.load()
    syms = declared_symbols()
    assert "loom_paraplex_forward" in syms and len(syms) >= 15
    missing = [s for s in syms if not hasattr(lib, s)]
    assert not missing, missing
    assert lib.loom_abi_version() == 10
    # every declared compute entry point has a ctypes signature
    compute = [s for s in syms if s not in ("loom_last_error", "loom_abi_version")]
    bound = set(_lib.SIGNATURES) | set(_lib.QUERIES)
    assert set(compute) == bound, set(compute) ^ bound
    # chunk records [B, KVH, chunks, record] fp32; chunks = min(~1.5 blocks per CU over
    # the B*KVH rows, ceil(max_len / 128)) = min(96, 3) with no device (256 CUs assumed)
    assert lib.loom_gqa_workspace_bytes(2, 300, 8, 2, 96) == 2 * 2 * 3 * (8 + 2 * 4 * 96) * 4
    # the ctypes mirror of the descriptor struct has the C layout
    assert lib.loom_linear_multi_desc_bytes() == ctypes.sizeof(_lib.LinearMultiDesc)
    assert lib.loom_ffn_decode_desc_bytes() == ctypes.sizeof(_lib.FfnDecodeDesc)


def test_error_channel_reports_argument_errors():
    from loom_amd import _lib
    with pytest.raises(RuntimeError, match="axis must be 0"):
        # argument validation happens before any device work
        _lib.call("loom_tria_depth_forward", 0, ctypes.c_void_p(16), ctypes.c_void_p(16),
                  ctypes.c_void_p(16), None, None, None, None, None, None, None, 1, 1, 1,
                  0.05, 7, None)
    with pytest.raises(RuntimeError, match="K=0"):
        _lib.call("loom_final_ca_sparse_forward", 0, *([ctypes.c_void_p(16)] * 5), None,
                  1, 1, 0, 8, 1.0, None)
    p = ctypes.c_void_p(16)
    with pytest.raises(RuntimeError, match="paraplex_tria_endpoint: bad shape"):
        # H odd: the column pairs need H even
        _lib.call("loom_paraplex_tria_endpoint_forward", 1, p, p, p, p, p, p, 3.0, p, p, None,
                  None, p, p, p, None, 1, 1, 3, 0.0375, 0, None)


def test_linear_ln_checks_its_descriptor_before_any_launch():
    """bf16 rows that no staged tile takes (and zero rows) answer as
    loom_linear_multi does: zero rows are no error, a missing input or weight, a row
    stride below the row and rows that are not dense are, whichever kernel the
    product would take (no device here: a launch would be an error of its own)."""
    from loom_amd import _lib

    def ln(m, ldo=768, null=(), **kw):
        d = _lib.LinearMultiDesc()
        d.x, d.ldx, d.k, d.x2, d.ldx2, d.k2, d.m, d.nseg = 256, 768, 768, 256, 768, 768, m, 1
        s = d.seg[0]
        s.w, s.ldw, s.w2, s.ldw2, s.out, s.ldc, s.n = 256, 768, 256, 768, 256, 768, 768
        for k, v in kw.items():
            setattr(s if hasattr(s, k) else d, k, v)
        p = ctypes.c_void_p(256)
        _lib.call("loom_linear_ln", 1, ctypes.byref(d), p, p, 1e-5, p, ldo, p,
                  _lib.load().loom_linear_ln_workspace_bytes(m, 768), None, None)

    ln(0)
    ln(0, k2=0, x2=None, w2=None)
    for m in (0, 100, 4096):
        for bad in (dict(x2=None), dict(w2=None), dict(x=None), dict(w=None), dict(k=0, k2=0), dict(k2=-64)):
            with pytest.raises(RuntimeError, match="linear_ln: an input or a weight|linear_multi:"):
                ln(m, **bad)
    for bad in (dict(out=None), dict(ldx=760), dict(ldx2=760), dict(ldw=760), dict(ldw2=760)):
        with pytest.raises(RuntimeError, match="linear_multi:"):
            ln(100, **bad)
    for bad in (dict(ldc=776), dict(ldo=776)):
        with pytest.raises(RuntimeError, match="dense rows"):
            ln(100, **bad)


def test_product_kernel_rule():
    """Products whose kernels were timed against each other take the faster one
    (256 CUs: no device here); loom_linear_multi's products of many rows take the
    staged tiles, alone as in one launch."""
    from loom_amd import _lib
    lib = _lib.load()
    kernel = lib.loom_test_gemm_kernel
    kernel.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 4 + [ctypes.c_int]
    def of(*s, hd=0, multi=0, dtype=1, shared=0):
        prev = lib.loom_gemm_shared_tiles(shared)
        try:
            return kernel(dtype, *s, hd, multi)
        finally:
            lib.loom_gemm_shared_tiles(prev)
    # staged tiles faster than direct fragments
    for s in [(1024, 2048, 512), (640, 2048, 512), (512, 4096, 1024), (3072, 512, 2048), (4096, 512, 2048),
              (2048, 1024, 4096), (2048, 1024, 1024), (4096, 512, 512)]:
        assert of(*s) == 2, s
    assert of(8192, 3072, 768) == 3 and of(2048, 768, 3072) == 1
    for M in (768, 777, 1024):
        assert of(M, 3072, 1152, hd=96, shared=1) == 5
    # and slower
    for s in [(999, 768, 3072), (512, 768, 768), (1024, 768, 768), (300, 3072, 768), (1024, 512, 2048), (512, 1024, 1024)]:
        assert of(*s) > 100, s
    assert of(600, 4096, 1536, hd=128) > 100 and of(333, 3072, 1152, hd=96, shared=1) > 100
    # few rows: the skinny kernel up to 24 rows of few k
    assert of(17, 2048, 512) == 0 and of(24, 512, 512) == 0 and of(20, 3072, 768) == 0
    assert of(25, 2048, 512) > 100 and of(17, 768, 768) > 100 and of(17, 768, 3072) > 100
    # two products in one launch, and each by itself
    for M in (384, 512, 768, 1024):
        for N in (3072, 1536, 4608):
            assert of(M, N, 768, multi=1) in (1, 2, 3, 4)
    assert of(300, 3072, 768, multi=1) > 100 and of(256, 6144, 1024, multi=1) < 100


def test_final_ca_tile_rule():
    """The shapes whose both kernels were timed take the faster one (256 CUs: no
    device here), and so does each tile size's test shape."""
    from loom_amd import _lib
    takes = _lib.load().loom_test_final_ca_tiles
    takes.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 4
    faster = {1: [(8, 2048, 15, 768), (2, 130, 16, 768), (300, 2, 32, 768), (2, 300, 48, 768), (1, 300, 64, 512),
                  (8, 512, 256, 1024), (8, 512, 120, 768), (130, 17, 15, 768), (32, 130, 33, 320), (30, 140, 17, 1024),
                  (9, 150, 256, 128), (20, 130, 120, 64)],
              0: [(8, 512, 15, 768), (8, 2048, 4, 256), (8, 512, 64, 1024), (8, 512, 100, 768), (1, 1024, 48, 256),
                  (32, 130, 33, 320), (30, 140, 17, 1024), (9, 150, 256, 128), (20, 130, 120, 64)]}
    slower = {1: [(1, 256, 16, 768), (1, 300, 48, 1024), (2, 130, 48, 768), (300, 2, 100, 768), (2, 300, 100, 512),
                  (1, 1024, 100, 768), (8, 2048, 100, 1024), (8, 2048, 15, 96), (4096, 1, 15, 768), (8, 2048, 300, 768),
                  (8, 300, 128, 1024), (300, 2, 33, 1024)],
              0: [(2, 300, 64, 768), (300, 2, 64, 64), (1, 1024, 32, 1024), (1, 1024, 48, 768), (8, 2048, 2, 1024),
                  (2, 300, 100, 1024), (1, 256, 256, 1024), (1, 1024, 33, 256)]}
    for code in (0, 1):
        assert [s for s in faster[code] if not takes(code, *s)] == []
        assert [s for s in slower[code] if takes(code, *s)] == []


def test_package_imports_without_a_gpu_build_of_torch():
    """The host-only parts (configuration, checkpoints, weights, the library's
    queries) need no GPU backend in torch."""
    code = ("import sys, torch\n"
            "if hasattr(torch._C, '_cuda_getCurrentRawStream'): del torch._C._cuda_getCurrentRawStream\n"
            f"sys.path.insert(0, {os.path.join(ROOT, 'loomformer-paraplex_amd')!r})\n"
            "from loom_amd import _lib, checkpoint, config, ops, weights\n"
            "assert _lib.load().loom_abi_version() == 10\n")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr


def test_drop_in_modules_expose_reference_names():
    from kernels.build import EXPORTS, build_or_load
    for ext, names in EXPORTS.items():
        mod = build_or_load(ext, ["ignored.cu"], ptx_kernels={"x": "y"})
        for n in names:
            assert callable(getattr(mod, n)), (ext, n)
    with pytest.raises(RuntimeError, match="unknown extension"):
        build_or_load("loomformer_chunk_attn", [])


def test_mirror_rejects_cpu_tensors_like_the_reference():
    from loom_amd import ops
    x = torch.zeros(2, 3, 8)
    with pytest.raises(RuntimeError, match="CUDA tensors required"):
        ops.paraplex_forward(x, x, x, torch.zeros(8), torch.zeros(2, 8), torch.zeros(8),
                             torch.empty(0, dtype=torch.bool), torch.ones(()), 0, False, 0.99, 3.0)
    with pytest.raises(RuntimeError, match="must be CUDA"):
        ops.tria_step_forward(x, x, x, torch.zeros(2, 3, 8, 3, 3), 0.05, 0)
    with pytest.raises(RuntimeError, match="training-only"):
        ops.paraplex_backward()


def test_tria_chunked_fires_rejects_bad_boundary_lists():
    """The boundary list is validated on the host before any device work."""
    from loom_amd import _lib
    lib = _lib.load()
    arr = lambda *v: (ctypes.c_int64 * len(v))(*v)
    # T=30, W=8: grid positions 7, 15, 23 must be present
    assert lib.loom_tria_chunked_fires_workspace_bytes(3, 30, 128, arr(7, 15, 23), 3) > 0
    args = lambda b, n: (0, ctypes.c_void_p(16), ctypes.c_void_p(16), ctypes.c_void_p(16), 3 * 30 * 4, 4,
                         None, None, b, n, ctypes.c_void_p(16), None, None, ctypes.c_void_p(16),
                         1 << 30, 3, 30, 4, 8, 0.05, 0.1, 1e-6, None)
    with pytest.raises(RuntimeError, match="lacks 1 of the 3 grid positions"):
        _lib.call("loom_tria_chunked_forward_fires", *args(arr(3, 7, 23), 3))
    with pytest.raises(RuntimeError, match="must increase"):
        _lib.call("loom_tria_chunked_forward_fires", *args(arr(7, 7, 15, 23), 4))
    with pytest.raises(RuntimeError, match="outside"):
        _lib.call("loom_tria_chunked_forward_fires", *args(arr(7, 15, 23, 30), 4))


def test_noalloc_rejects_records_beyond_the_scratch():
    """The static-scratch decode step refuses shapes whose chunk records exceed
    its array before any device call (null tensors: nothing is dereferenced)."""
    from loom_amd import _lib
    lib = _lib.load()
    B, QH, KVH, HD, length = 4096, 8, 1, 128, 4096
    need = lib.loom_gqa_workspace_bytes(B, length, QH, KVH, HD)
    assert need > 4 << 20
    with pytest.raises(RuntimeError, match="static scratch"):
        _lib.call("loom_gqa_decode_step_noalloc", 1, None, None, None, KVH * length * HD, HD,
                  length * HD, None, None, None, None, None, QH * HD, B, length, None, QH, KVH,
                  HD, None)


def test_gemm_shared_tiles_is_a_process_switch():
    """loom_gemm_shared_tiles sets the tile mode and returns the previous one
    (host-side state: no device needed)."""
    from loom_amd import _lib
    lib = _lib.load()
    prev = lib.loom_gemm_shared_tiles(1)
    try:
        assert lib.loom_gemm_shared_tiles(1) == 1
        assert lib.loom_gemm_shared_tiles(0) == 1
        assert lib.loom_gemm_shared_tiles(7) == 0      # any nonzero value turns it on
        assert lib.loom_gemm_shared_tiles(0) == 1
    finally:
        lib.loom_gemm_shared_tiles(prev)
