"""The C-ABI shared library: builds for gfx950 without a GPU, loads, exports every symbol declared in
include/lvar_sparse_attn.h, and validates arguments before touching the device."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "lvar_sparse_attn.h")


@pytest.fixture(scope="module")
def lib():
    from lvar_amd import _lib
    from lvar_amd.build import LIB_PATH, build_library
    if not os.path.exists(LIB_PATH):
        build_library()
    return _lib.load()


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lvar_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported(lib):
    from lvar_amd import _lib
    names = declared_symbols()
    assert set(names) == set(_lib.EXPORTED_SYMBOLS), names
    for n in names:
        assert getattr(lib, n) is not None


def test_version_and_arch(lib):
    assert lib.lvar_version() >= 100
    assert lib.lvar_target_arch() == b"gfx950"
    assert lib.lvar_status_string(0) == b"ok"
    assert b"invalid" in lib.lvar_status_string(-1) and b"unsupported" in lib.lvar_status_string(-2)


def test_argument_validation_without_device(lib):
    """Bad arguments are rejected on the host before any HIP call is made."""
    from lvar_amd._lib import LvarTensor
    null = LvarTensor(None, 0, 0, 0)
    fake = LvarTensor(0x1000, 128 * 16 * 128, 16 * 128, 128)          # aligned, never dereferenced
    odd = LvarTensor(0x1008, 128 * 16 * 128, 16 * 128, 128)           # misaligned base
    one = ctypes.c_void_p(0x2000)
    assert lib.lvar_dense_attn_fwd(null, fake, fake, fake, one, one, None, 1, 1, 1, 16, 16, 128, 1.0, None) == -1
    assert lib.lvar_dense_attn_fwd(odd, fake, fake, fake, one, one, None, 1, 1, 1, 16, 16, 128, 1.0, None) == -1
    assert lib.lvar_dense_attn_fwd(fake, fake, fake, fake, one, one, None, 0, 1, 1, 16, 16, 128, 1.0, None) == -1
    assert lib.lvar_dense_attn_fwd(fake, fake, fake, fake, one, one, None, 1, 1, 1, 16, 16, 128, -1.0, None) == -1
    assert lib.lvar_dense_attn_fwd(fake, fake, null, null, None, None, None, 1, 1, 1, 16, 16, 128, 1.0, None) == -1   # no outputs at all
    assert lib.lvar_dense_attn_fwd(fake, fake, fake, fake, one, one, None, 1, 6, 4, 16, 16, 128, 1.0, None) == -1   # 6 query heads over 4 K/V heads
    assert lib.lvar_colsum_fwd(fake, fake, one, one, None, 1, 6, 0, 16, 16, 128, 192, 1.0, None) == -1
    assert lib.lvar_colsum_fwd(fake, fake, one, one, None, 1, 1, 1, 16, 16, 128, 100, 1.0, None) == -1           # group not a multiple of 32
    assert lib.lvar_colsum_fwd(fake, fake, None, one, None, 1, 1, 1, 16, 16, 128, 192, 1.0, None) == -1
    assert lib.lvar_csp_attn_fwd(fake, fake, fake, null, fake, None, None, one, one, 1, 16, 100, 1, 1, 16, 16, 128, 1.0, 1.0, None) == -2   # groups of 100 rows: no workgroup shape
    assert lib.lvar_csp_attn_fwd(fake, fake, fake, null, fake, None, None, one, one, 1, 16, 0, 1, 1, 16, 16, 128, 1.0, 1.0, None) == -1
    assert lib.lvar_dense_attn_rcp_fwd(fake, fake, fake, fake, None, 1, 1, 1, 16, 16, 128, 1.0, None) == -1                # no place for the row constant
    assert lib.lvar_csp_attn_fwd(fake, fake, fake, null, fake, None, None, None, one, 1, 16, 192, 1, 1, 16, 16, 128, 1.0, 1.0, None) == -1
    assert lib.lvar_block_sparse_attn_fwd(fake, fake, fake, fake, None, None, one, 0, 0, one, 0, 0, 4, 4, 96, 64, 1, 1, 16, 16, 128, 1.0, None) == -2    # 96-row query blocks
    assert lib.lvar_block_sparse_attn_fwd(fake, fake, fake, fake, None, None, one, 0, 0, one, 0, 0, 4, 4, 128, 32, 1, 1, 16, 16, 128, 1.0, None) == -2   # 32-key blocks
    wide = LvarTensor(0x1000, 1 << 30, 1 << 26, 1 << 23)                # row stride of 2^23 elements: beyond the 24-bit gather addressing
    assert lib.lvar_csp_attn_fwd(fake, wide, fake, null, fake, None, None, one, one, 1, 16, 192, 1, 1, 16, 16, 128, 1.0, 1.0, None) == -2
    assert lib.lvar_block_sparse_attn_fwd(fake, fake, fake, fake, None, None, None, 0, 0, one, 0, 0, 4, 4, 128, 64, 1, 1, 16, 16, 128, 1.0, None) == -1


def test_colsum_query_span_limit(lib):
    """The fills of a ragged last 64-row stage form 32-bit offsets of up to 63 rows beyond the last query row: rows of
    2 MiB, of which 2^31 bytes hold 1024: 959 rows pass the check (and nothing can be launched here), more do not."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("the call in range would be launched")
    from lvar_amd._lib import LvarTensor
    wide, fake = LvarTensor(0x1000, 1 << 40, 1 << 32, 1 << 20), LvarTensor(0x1000, 128 * 16 * 128, 16 * 128, 128)
    one = ctypes.c_void_p(0x2000)
    for rows, status in ((959, -3), (960, -1), (1000, -1), (1023, -1), (1024, -1)):
        assert lib.lvar_colsum_fwd(wide, fake, one, one, None, 1, 1, 1, rows, 16, 128, 192, 1.0, None) == status, rows


def test_list_build_and_upsample_argument_validation(lib):
    from lvar_amd._lib import LvarTensor
    null = LvarTensor(None, 0, 0, 0)
    fake = LvarTensor(0x1000, 128 * 16 * 128, 16 * 128, 128)
    one = ctypes.c_void_p(0x2000)
    assert lib.lvar_topk_token_lists(None, 100, one, 100, one, 4, 100, 10, 0, None) == -1            # no scores
    assert lib.lvar_topk_token_lists(one, 100, one, 100, one, 4, 100, 101, 0, None) == -1            # k > Lk
    assert lib.lvar_topk_token_lists(one, 99, one, 100, one, 4, 100, 10, 0, None) == -1              # row stride < Lk
    assert lib.lvar_topk_token_lists(one, 100, one, 5, one, 4, 100, 10, 0, None) == -1               # output row shorter than k
    assert lib.lvar_topk_token_lists(one, 100, one, 100, one, 4, 100, 10, 101, None) == -1           # zero fill beyond the row
    assert lib.lvar_topk_token_lists(one, 100, one, 100, one, 0, 100, 10, 0, None) == 0              # no rows: nothing to launch
    assert lib.lvar_remap_concat_lists(one, 100, 100, None, 0, 8, one, 200, one, 2, 3, 4, 64, 500, 0, None) == -1   # local run without a table
    assert lib.lvar_remap_concat_lists(one, 100, 100, one, 8, 8, one, 70, one, 2, 3, 4, 64, 500, 0, None) == -1     # 64 + 8 > output row
    assert lib.lvar_remap_concat_lists(one, 100, 100, None, 0, 0, one, 64, one, 2, 0, 4, 64, 500, 0, None) == -1    # no source groups
    assert lib.lvar_mask_to_lists(one, 10, one, 10, one, 3, 10, 0, None) == -1                    # multiple_of must be positive
    assert lib.lvar_mask_to_lists(one, 10, one, 9, one, 3, 10, 1, None) == -1                     # output row shorter than n
    assert lib.lvar_mask_to_lists(one, 10, one, 10, one, 0, 10, 1, None) == 0
    # fused upsample: Lq must be dst_side^2 and the cache must exist
    args = (one, one, 1, 16, 192, 1, 1, 16, 16, 128, 1.0, 1.0, None)
    assert lib.lvar_csp_attn_upsample_fwd(fake, fake, fake, fake, 2, 5, fake, None, None, *args) == -1         # 25 != 16
    remap = lib.lvar_csp_attn_remap_fwd   # rows of 16 entries, 12 of them taken, then 4 local ones; 16 = 4 x 4 queries
    rows = (1, 1, 16, 16, 128, 1.0, 1.0, None)
    assert remap(fake, fake, fake, fake, 2, 5, fake, one, 16, 16, 1, 12, one, 4, 4, 192, *rows) == -1           # 25 != 16
    assert remap(fake, fake, fake, fake, 2, 4, fake, None, 16, 16, 1, 12, one, 4, 4, 192, *rows) == -1
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 16, 16, 0, 12, one, 4, 4, 192, *rows) == -1
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 16, 11, 1, 12, one, 4, 4, 192, *rows) == -1           # fewer columns than entries
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 15, 16, 1, 12, one, 4, 4, 192, *rows) == -1
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 16, 16, 1, 12, None, 4, 4, 192, *rows) == -1
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 16, 16, 1, 12, one, 3, 4, 192, *rows) == -1
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 16, 16, 1, 12, one, 4, 4, 0, *rows) == -1
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 16, 16, 1, 12, one, 4, 4, 96, *rows) == -2            # 3-wave workgroups
    assert remap(fake, fake, fake, fake, 2, 4, fake, one, 16, 16, 1, 12, one, 4, 4, 192, 1, 1, 16, 16, 256, 1.0, 1.0, None) == -2
    assert lib.lvar_csp_attn_upsample_fwd(fake, fake, fake, null, 2, 4, fake, None, None, *args) == -1


def test_statistics_score_and_merge_argument_validation(lib):
    from lvar_amd._lib import LvarTensor
    null = LvarTensor(None, 0, 0, 0)
    fake = LvarTensor(0x1000, 128 * 16 * 128, 16 * 128, 128)
    odd = LvarTensor(0x1008, 128 * 16 * 128, 16 * 128, 128)
    far = LvarTensor(0x1000, 1 << 40, 1 << 36, 1 << 27)                  # 16 rows span 2^32 bytes
    one, odd4 = ctypes.c_void_p(0x2000), ctypes.c_void_p(0x2002)
    # row statistics: q, k, lse2, scratch, bytes, B, H, kv_heads, Lq, Lk, head_dim
    for q, k, out, scratch, dims, status in (
            (null, fake, one, None, (1, 1, 1, 16, 16, 128), -1), (fake, odd, one, None, (1, 1, 1, 16, 16, 128), -1),
            (fake, fake, None, None, (1, 1, 1, 16, 16, 128), -1), (fake, fake, one, odd4, (1, 1, 1, 16, 16, 128), -1),
            (fake, fake, one, None, (1, 6, 4, 16, 16, 128), -1), (fake, fake, one, None, (1, 6, 0, 16, 16, 128), -1),
            (fake, fake, one, None, (1, 1, 1, 0, 16, 128), -1), (fake, fake, one, None, (1, 1, 1, 16, -1, 128), -1),
            (fake, far, one, None, (1, 1, 1, 16, 16, 128), -1), (fake, fake, one, None, (1, 1, 1, 16, 16, 96), -2)):
        assert lib.lvar_row_lse_fwd(q, k, out, scratch, 64, *dims, 1.0, None) == status, dims
    assert lib.lvar_row_lse_fwd(fake, fake, one, None, 0, 1, 1, 1, 16, 16, 128, -1.0, None) == -1
    assert lib.lvar_row_lse_scratch_bytes(0, 1, 16, 16) == -1 and lib.lvar_row_lse_scratch_bytes(1, 1, 16, 0) == -1
    for m, l, out, rows in ((None, one, one, 4), (one, None, one, 4), (one, one, None, 4), (one, one, one, 0)):
        assert lib.lvar_lse2_from_stats(m, l, out, rows, None) == -1
    # block scores
    need = lib.lvar_block_scores_scratch_bytes(1, 1, 16, 16, 32, 128)
    assert need > 0
    assert all(lib.lvar_block_scores_scratch_bytes(1, 1, 16, 16, g, b) == -1 for g, b in ((0, 128), (32, 0), (32, 96)))

    def scores(q=fake, k=fake, out=one, target=1, scratch=one, nbytes=need, H=1, kv=1, d=128, group=32, block=128, scale=1.0):
        return lib.lvar_block_scores_fwd(q, k, out, None, target, scratch, nbytes, 1, H, kv, 16, 16, d, group, block, scale, None)
    big = dict(nbytes=1 << 40)
    for bad in (dict(q=null), dict(k=odd), dict(out=None), dict(target=-1), dict(scratch=None), dict(scratch=ctypes.c_void_p(0x2008)),
                dict(nbytes=need - 1), dict(H=6, kv=4, **big), dict(k=far), dict(q=far), dict(group=0), dict(group=33), dict(block=96), dict(scale=0.0)):
        assert scores(**bad) == -1, bad
    for bad in (dict(group=96, **big), dict(group=1088, **big), dict(d=96)):   # group sizes and head sizes without a one-sweep kernel
        assert scores(**bad) == -2, bad
    # merged selection: scores, row stride, listed, how many, out, rows, Lk, k
    for args, status in (((None, 100, one, 4, one, 2, 100, 10), -1), ((one, 100, None, 4, one, 2, 100, 10), -1), ((one, 100, one, 4, None, 2, 100, 10), -1),
                         ((one, 100, one, 0, one, 2, 100, 10), -1), ((one, 99, one, 4, one, 2, 100, 10), -1), ((one, 100, one, 4, one, 2, 100, 101), -1),
                         ((one, 100, one, 4, one, 2, 100, 0), -1), ((one, 100, one, 4, one, -1, 100, 10), -1), ((one, 16385, one, 4, one, 2, 16385, 10), -2),
                         ((one, 100, one, 65536, one, 2, 100, 10), -2), ((one, 100, one, 4, one, 0, 100, 10), 0)):
        assert lib.lvar_topk_union_lists(*args, None) == status, args


def test_header_is_plain_c(tmp_path):
    """The public header must be usable from C (the reference's other bindings are C/C++)."""
    import shutil
    import subprocess
    if shutil.which("gcc") is None:
        pytest.skip("no C compiler")
    src = tmp_path / "use.c"
    src.write_text('#include "lvar_sparse_attn.h"\nint main(void) { lvar_tensor_t t = {0, 0, 0, 0}; (void)t; return lvar_version() ? 0 : 1; }\n')
    r = subprocess.run(["gcc", "-std=c99", "-Wall", "-Wextra", "-pedantic", "-Werror", "-I", os.path.dirname(HEADER), "-c", str(src),
                        "-o", str(tmp_path / "use.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def test_python_wrappers_fail_loudly_without_gpu():
    import torch
    from lvar_amd import sparse_attn_ops as ops
    q = torch.zeros(1, 1, 64, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.dense_attn(q, q, q)
    with pytest.raises(TypeError):
        ops.dense_attn(q.float(), q.float(), q.float())
    with pytest.raises(AssertionError):
        ops.csp_attn(q, q, q, None, torch.zeros(1, 1, 1, 3, dtype=torch.int32), torch.zeros(1, 1, 1, dtype=torch.int32), q, 1)


def test_missing_library_is_an_import_error(monkeypatch):
    from lvar_amd import _lib
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setenv("LVAR_AMD_LIB", "/nonexistent/liblvar.so")
    with pytest.raises(ImportError, match="no CPU or PyTorch fallback"):
        _lib.load()


def test_torch_binding_loads_and_declines_cpu_tensors(lib):
    """The compiled fast path of dense_attn is optional: when it is built it must load, bind to the C-ABI
    library and hand anything but plain device tensors back to the general path (None)."""
    import os
    import torch
    from lvar_amd import _lib
    path = os.path.join(os.path.dirname(_lib.__file__), "_lvar_torch.so")
    if not os.path.exists(path):
        pytest.skip("torch binding not built")
    mod = _lib.torch_binding()
    assert mod is not None and hasattr(mod, "fast_dense_attn") and hasattr(mod, "bind")
    x = torch.zeros(1, 1, 8, 128, dtype=torch.bfloat16)
    assert mod.fast_dense_attn(x, x, x, None) is None            # CPU tensors: not its case, and no GPU call is made
