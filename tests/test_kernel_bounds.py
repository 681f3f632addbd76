"""Host arithmetic that the kernels' memory accesses rest on, checked without a GPU: the functions
are the kernels' own (compiled for host and device from one definition) and are called through
the built library."""
import ctypes
import os
import re
import subprocess

import pytest


@pytest.fixture(scope="module")
def mfma_lib():
    from tuff_amd.csrc import ops
    lib = ops.load("attention_mfma")
    lib.tuff_attention_partition_pages.argtypes = [ctypes.c_int, ctypes.c_int]
    lib.tuff_attention_partition_pages.restype = ctypes.c_int
    return lib


def test_single_token_attention_fetches_every_page_a_partition_touches(mfma_lib):
    """A partition of 256 keys that starts inside a page (page sizes that do not divide 256: 96, 112,
    144, ...) touches one page more than 256 / page size rounded up.  For every page size the kernel
    takes and every partition: lanes that fetch a page number == pages touched, and a wave has enough
    lanes.  (With 256 / page size rounded up, pages of 96 positions left the partition at key 256
    one page short: page number -1 from a lane that fetched nothing, keys read from before the pool.)"""
    from tuff_amd.csrc import ops
    part_keys = ops.ATTN_PARTITION
    short = set()
    for ps in range(16, 513, 16):
        for part in range(0, 2048 if ps <= 128 else 300):
            first = part * part_keys
            touched = (first + part_keys - 1) // ps - first // ps + 1
            assert touched == len({k // ps for k in range(first, first + part_keys, 16)})
            lanes = mfma_lib.tuff_attention_partition_pages(part, ps)
            assert lanes == touched, (ps, part, lanes, touched)
            assert lanes <= 64
            if touched > -(-part_keys // ps):
                short.add(ps)
    assert {96, 112, 144} <= short          # the sizes the old bound was wrong for are among those walked


@pytest.mark.parametrize("blocks, parts, columns, whole", [
    (63, 4, 4, False), (64, 4, 4, True), (64, 5, 4, False), (128, 8, 4, False), (175, 8, 4, False), (176, 8, 4, True), (256, 8, 8, True),
    (257, 8, 4, False), (257, 4, 4, True), (288, 8, 4, False), (384, 4, 4, True), (384, 8, 4, False), (431, 8, 4, False), (432, 8, 4, True),
    (512, 8, 4, True), (512, 8, 8, False), (512, 4, 8, True), (384, 4, 8, False), (128, 4, 8, True), (768, 4, 8, False), (576, 8, 4, False),
    (576, 4, 4, False), (768, 4, 4, True), (256, 9, 4, False), (256, 4, 16, True), (128, 4, 16, False), (512, 4, 16, False), (256, 5, 16, False)])
def test_whole_columns_only_where_the_workgroups_fill_their_rounds(mfma_lib, blocks, parts, columns, whole):
    """The rule's sides as measured: 36 to 48 requests of 8 kv heads and 1,100 to 2,000 keys, a second round half empty, took 2 to 4 % of a
    decode step more."""
    mfma_lib.tuff_attention_takes_whole.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_int]
    assert mfma_lib.tuff_attention_takes_whole(blocks, parts, columns) == int(whole)


def test_partition_pages_refuses_nonsense(mfma_lib):
    assert mfma_lib.tuff_attention_partition_pages(-1, 16) < 0
    assert mfma_lib.tuff_attention_partition_pages(0, 0) < 0
    assert mfma_lib.tuff_attention_partition_pages(2 ** 31 // 256, 16) < 0


@pytest.fixture(scope="module")
def gemm_lib():
    from tuff_amd.csrc import ops
    return ops.load("gemm_bf16")


@pytest.mark.parametrize("M,N,K,groups", [(65, 1 << 25, 64, 1 << 17), (129, 1 << 25, 64, 1 << 17), (300, 3 << 24, 128, 3 << 16),
                                         (65, (1 << 25) - 256, 64, (1 << 17) - 1), (65, (1 << 25) + 64, 64, 174763), (65, (1 << 25) + 128, 64, 0)])
def test_rows_beyond_31_bits_leave_the_next_norm_its_sums(gemm_lib, M, N, K, groups):
    """Sixteen rows of 2^25 float32 columns are 2^31 bytes; whole blocks of columns emit on both sides of that."""
    tiles, rows = ctypes.c_int(), ctypes.c_int()
    assert gemm_lib.tuff_gemm_bf16_emit_layout(M, N, K, ctypes.byref(tiles), ctypes.byref(rows)) == 0
    assert (tiles.value, rows.value) == (groups, M)


@pytest.mark.parametrize("M,N,K,plain,emit", [
    (16, 2048, 8192, False, False),                       # up to 16 rows: one kernel, whatever the sizes
    (17, 2048, 2048, False, True), (20, 1024, 1024, False, False), (20, 2048, 1032, False, True), (17, 256, 64, False, False),
    (20, 2048, 2056, True, True), (20, 512, 2048, True, True), (17, 512, 1024, False, False), (17, 2048, 8192, True, True), (21, 2048, 1024, True, True), (20, 2064, 8192, False, False)])
def test_narrow_products_of_few_rows_take_slices_only_where_they_are_faster(gemm_lib, M, N, K, plain, emit):
    """Work space means partial tiles and a second kernel.  Outputs of up to 2,048 columns and 17 to 20 rows go without up to
    K = 2,048 (of less than 1,024 columns K = 1,024), those that leave the next norm its sums up to K = 1,024."""
    def floats(e):
        out = ctypes.c_longlong(-1)
        assert gemm_lib.tuff_gemm_bf16_workspace(M, N, K, e, ctypes.byref(out)) == 0
        return out.value
    assert (floats(0) > 0) == plain and (floats(1) > 0) == emit
    tiles, rows = ctypes.c_int(), ctypes.c_int()
    assert gemm_lib.tuff_gemm_bf16_emit_layout(M, N, K, ctypes.byref(tiles), ctypes.byref(rows)) == 0
    assert tiles.value == -(-N // (64 if emit else 8 if N <= 2048 else 16)) and rows.value == (16 if M <= 16 else 64)


@pytest.mark.parametrize("T,R,q,keys,window,H,Hkv,hd,want", [
    (1, 1, 1, 1, 0, 32, 8, 64, False), (8, 8, 1, 4, 0, 32, 32, 64, False), (256, 256, 1, 40, 0, 32, 32, 64, False),
    (128, 128, 1, 20, 0, 8, 8, 128, False), (64, 64, 1, 20000, 4, 32, 32, 64, False), (65536, 65536, 1, 600, 0, 16, 1, 64, False),
    (256, 256, 1, 40, 0, 32, 8, 64, True), (1, 1, 1, 300, 0, 32, 32, 64, True), (4, 4, 1, 1000, 0, 32, 8, 64, True),
    (500, 1, 500, 500, 0, 32, 8, 64, True), (2000, 1, 2000, 2000, 64, 8, 8, 128, True), (128, 128, 1, 600, 0, 8, 8, 128, True)])
def test_float32_attention_takes_the_kernel_that_is_faster(T, R, q, keys, window, H, Hkv, hd, want):
    """Sizes that were measured with both kernels (the same bits): few keys and workgroups of few columns go to the general one."""
    from tuff_amd.csrc import ops
    assert ops.attention_f32_pays(T, R, q, keys, window, H, Hkv, hd) is want


@pytest.mark.parametrize("T,R,q,keys,H,Hkv,hd,want", [
    (256, 256, 1, 64, 32, 32, 128, True), (256, 256, 1, 200, 32, 32, 128, True), (32, 32, 1, 40, 16, 16, 128, True),     # 666 / 119, 2,013 / 371, 19.4 / 9.5 us
    (4, 4, 1, 40, 8, 8, 128, True), (256, 256, 1, 200, 32, 32, 16, True), (64, 64, 1, 40, 8, 8, 128, True),              # 17.5 / 6.9, 135 / 66, 19.5 / 9.5
    (256, 256, 1, 16, 32, 32, 32, False), (256, 256, 1, 16, 16, 16, 64, False), (32, 32, 1, 4, 16, 16, 16, False),       # 19.5 / 43.9, 16.5 / 29.1, 4.8 / 5.4
    (1, 1, 1, 4, 32, 8, 16, False)])                                                                                     # 4.9 / 5.4
def test_float32_attention_takes_the_faster_kernel_on_both_sides_of_its_line(T, R, q, keys, H, Hkv, hd, want):
    """Measured points near the line, general kernel / tiles."""
    from tuff_amd.csrc import ops
    assert ops.attention_f32_pays(T, R, q, keys, 0, H, Hkv, hd) is want


def test_float32_attention_of_a_mixer_follows_that_rule(monkeypatch):
    import types

    import torch

    from tuff_amd.csrc import ops
    from tuff_amd.parts.attention import PagedAttention
    taken = []
    for name in ("attention_f32", "attention_general"):
        monkeypatch.setattr(ops, name, lambda *a, _n=name, **k: taken.append(_n))
    mixer = PagedAttention.__new__(PagedAttention)
    mixer.H = mixer.Hkv = 32
    mixer.hd = mixer.vd = 64
    mixer.sinks = mixer.slopes = mixer.window = mixer.scale = None
    cache = types.SimpleNamespace(k=None, v=None, page_size=16)
    group = types.SimpleNamespace(block_table=None)
    for keys in (4, 4000):
        ctx = types.SimpleNamespace(T=8, R=8, max_q_len=1, max_ctx_len=keys, req_info=None, req_of_token=None, positions=None)
        mixer.attend(torch.zeros(8, 32 * 64), None, ctx, cache, group)
    assert taken == ["attention_general", "attention_f32"]


@pytest.mark.parametrize("M,N,K,steps", [
    (4, 2048, 8192, 12), (4, 4096, 2048, 12), (4, 4112, 1536, 6), (8, 4096, 2048, 6), (4, 8192, 2048, 6), (4, 8208, 2048, 4), (4, 24576, 3072, 4),
    (4, 32752, 2048, 4), (4, 32768, 2048, 12), (1, 65536, 2048, 12), (4, 65536, 1024, 4), (4, 65536, 1536, 4), (4, 65536, 2304, 4), (4, 40960, 2560, 4),
    (4, 40960, 2944, 4), (4, 65536, 3072, 12), (4, 65536, 3584, 12), (4, 65536, 4096, 12), (4, 65536, 6144, 12), (1, 65536, 8192, 4), (4, 40960, 8192, 4),
    (4, 65536, 9216, 12), (4, 65536, 16384, 4), (4, 65536, 24576, 12), (5, 8192, 2048, 0), (16, 2048, 8192, 6), (4, 65536, 96, 0), (4, 65536, 128, 0), (17, 2048, 2048, 0)])
def test_steps_in_lds_of_the_float32_product_of_four_rows(M, N, K, steps):
    """Measured points on both sides of each line: twelve steps for products of many columns and a K of 8,192 took 8 to 15 % longer than four."""
    from tuff_amd.csrc import ops
    assert ops.load("gemm_f32").tuff_gemm_f32_quad_steps(M, N, K) == steps


def _early_reads(assembly):
    """The links (v_fmac_f32_dpp) whose DPP operand a vector instruction writes, or may have written on another way to a label, less
    than two wait states before: as (line, what stands there).  Also the number of links."""
    code = [line.split(";")[0].strip() for line in assembly.splitlines()]
    code = [line for line in code if line and not (line.startswith(".") and not line.endswith(":"))]
    links, early = 0, []
    for at, line in enumerate(code):
        if not line.startswith("v_fmac_f32_dpp"):
            continue
        links += 1
        operand = int(re.match(r"v_fmac_f32_dpp v\d+, v(\d+), v\d+ row_newbcast", line).group(1))
        states, back = 0, at - 1
        while states < 2:
            before = code[back]
            written = re.match(r"v_\w+ v(?:(\d+)|\[(\d+):(\d+)\])", before)
            first, last = (int(written.group(1) or written.group(2)), int(written.group(1) or written.group(3))) if written else (0, -1)
            if before.endswith(":") or first <= operand <= last:
                early.append((line, before))
                break
            nop = re.match(r"s_nop (\d+)", before)
            states += 1 + int(nop.group(1)) if nop else 1
            back -= 1
    return links, early


def test_links_of_the_float32_chain_do_not_read_what_was_just_written(tmp_path):
    """The chain of the float32 product of four rows is inline assembly that the compiler's hazard handling does not look into; a move of
    an operand that it puts between two links would be read before it is there.  In the kernels' own assembly, and in texts of
    it with such a move planted."""
    from tuff_amd.csrc import build
    out = str(tmp_path / "gemm_f32.s")
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([build._hipcc()] + flags + ["-I", build.HERE, "--offload-device-only", "-S", "-o", out, os.path.join(build.HERE, build.MODULES["gemm_f32"])],
                   check=True, capture_output=True, env={**os.environ, "HOME": os.environ.get("HOME", str(tmp_path))})
    with open(out) as f:
        assembly = f.read()
    links, early = _early_reads(assembly)
    assert links >= 6 * 4 * 64 and not early, early[:4]            # three rings, with and without SwiGLU, of four steps and more
    lines = assembly.splitlines()
    first = next(i for i, line in enumerate(lines) if "row_newbcast:0" in line)
    assert "s_nop 1" in lines[first - 1]
    for at, between, found in ((first + 1, [], True), (first + 6, [], True), (first + 6, ["s_nop 0"], True), (first + 6, ["s_nop 1"], False), (first - 1, [], False)):
        while "v_fmac_f32_dpp" not in lines[at] and at >= first:
            at += 1
        x = re.search(r"v_fmac_f32_dpp v\d+, (v\d+)", lines[max(at, first)]).group(1)
        planted = lines[:at] + [f"\tv_mov_b32_e32 {x}, v1"] + between + lines[at:]
        assert bool(_early_reads("\n".join(planted))[1]) == found, (at - first, between)
