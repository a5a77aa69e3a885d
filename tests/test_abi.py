"""The C ABI boundary on any host: libferric_hip.so loads, exports every
function include/ferric_hip.h declares with the binding's signature, and its
host-only entry points (speculative helpers, scratch sizing, argument
validation) behave like the reference. No GPU calls are made here."""

import ctypes
import re
from pathlib import Path

import numpy as np
import pytest

import ferric_amd
from ferric_amd import _lib
from ferric_amd.pool import PagePool
from ferric_amd.runner import PagedLimits
from oracle import oracle as orc

ROOT = Path(__file__).resolve().parent.parent
HEADER = ROOT / "include" / "ferric_hip.h"


def declared_functions():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = re.findall(r"^\s*(?:const\s+)?[a-z_0-9]+\s*\*?\s*(fh_[a-z_0-9]+)\s*\(", text, flags=re.M)
    return sorted(set(names))


def test_every_declared_symbol_is_exported_and_bound():
    lib = ferric_amd.load()
    names = declared_functions()
    assert len(names) >= 30
    bound = {n for n, _, _ in _lib.SIGNATURES}
    for n in names:
        assert hasattr(lib, n), f"{n} not exported by libferric_hip.so"
        assert n in bound, f"{n} has no ctypes signature in ferric_amd/_lib.py"
    assert bound <= set(names), f"binding names a function the header does not declare: {bound - set(names)}"


def test_struct_layouts_match_the_header():
    # Field counts and widths of the boundary structs.
    assert ctypes.sizeof(_lib.ModelDesc) == 10 * 4
    assert ctypes.sizeof(_lib.CtxOptions) == 8 * 4
    assert _lib.Row.pages.offset == 16 and ctypes.sizeof(_lib.Row) == 32
    from ferric_amd.runner import ROW_DTYPE
    assert ROW_DTYPE.itemsize == ctypes.sizeof(_lib.Row)
    for name, _ in _lib.Row._fields_:
        assert ROW_DTYPE.fields[name][1] == getattr(_lib.Row, name).offset, name


def u32(a):
    return (ctypes.c_uint32 * len(a))(*a)


def test_verify_greedy_round_matches_the_reference_vectors():
    lib = ferric_amd.load()
    for draft, target, acc, emitted in [([3, 4, 5], [9, 4, 5, 6], 0, [9]), ([3, 4, 5], [3, 4, 9, 6], 2, [3, 4, 9]),
                                        ([3, 4, 5], [3, 4, 5, 6], 3, [3, 4, 5, 6])]:
        a = ctypes.c_uint32()
        e = (ctypes.c_uint32 * 8)()
        n = ctypes.c_uint32()
        st = lib.fh_verify_greedy_round(u32(draft), len(draft), u32(target), len(target), ctypes.byref(a), e,
                                        ctypes.byref(n))
        assert st == 0 and a.value == acc and list(e[: n.value]) == emitted
        assert (acc, emitted) == orc.verify_greedy(draft, target)
    a, e, n = ctypes.c_uint32(), (ctypes.c_uint32 * 8)(), ctypes.c_uint32()
    assert lib.fh_verify_greedy_round(u32([3, 4]), 2, u32([3, 4]), 2, ctypes.byref(a), e, ctypes.byref(n)) == 1
    assert lib.fh_verify_greedy_round(None, 0, None, 0, ctypes.byref(a), e, ctypes.byref(n)) == 1


def test_verify_greedy_batch_settles_each_sequence_like_the_single_call():
    # Every sequence of a round in one call (draft iteration-major [K][S],
    # target [S][K + 1]) against the oracle's per-sequence verify: random
    # rounds over a 3-token alphabet (every acceptance count occurs), K = 0,
    # and the three reference vectors as one round.
    from ferric_amd.speculative import verify_greedy_batch
    lib = ferric_amd.load()
    r = np.random.default_rng(9)
    cases = [(r.integers(0, 3, (k, s)), r.integers(0, 3, (s, k + 1))) for k, s in [(4, 32), (1, 5), (7, 3), (0, 4)]]
    cases.append((np.array([[3, 3, 3], [4, 4, 4], [5, 5, 5]]), np.array([[9, 4, 5, 6], [3, 4, 9, 6], [3, 4, 5, 6]])))
    for draft, target in cases:
        acc, ems = verify_greedy_batch(draft, target)
        for s in range(target.shape[0]):
            want_a, want_e = orc.verify_greedy([int(x) for x in draft[:, s]], [int(x) for x in target[s]])
            assert int(acc[s]) == want_a and [int(x) for x in ems[s, : want_a + 1]] == want_e, (s, draft, target)
    e, acc = (ctypes.c_uint32 * 8)(), (ctypes.c_uint32 * 2)()
    assert lib.fh_verify_greedy_batch(None, u32([1, 2]), 2, 0, acc, e) == 0  # K = 0: the bonus token only
    assert list(e[:2]) == [1, 2] and list(acc) == [0, 0]
    assert lib.fh_verify_greedy_batch(None, u32([1, 2, 3, 4]), 2, 1, acc, e) == 1  # draft missing
    assert lib.fh_verify_greedy_batch(None, None, 0, 4, None, None) == 0  # no sequences


def test_token_assembly_matches_the_oracle():
    lib = ferric_amd.load()
    r = np.random.default_rng(0)
    for s, k in [(1, 4), (8, 4), (32, 4), (3, 0)]:
        anchors = r.integers(0, 151936, s).tolist()
        draft = r.integers(0, 151936, s * k).tolist()
        out = (ctypes.c_uint32 * (s * (k + 1)))()
        assert lib.fh_speculative_token_assembly(u32(anchors), u32(draft) if k else None, s, k, out) == 0
        assert list(out) == orc.token_assembly(anchors, draft if k else [0], s, k).tolist()


def test_scratch_sizes():
    lib = ferric_amd.load()
    # 32 rows x 32 heads x ceil(8320 / 512) partitions x (2 + 128) f32
    assert lib.fh_attention_scratch_bytes(32, 32, 8320) == 32 * 32 * 17 * 130 * 4
    assert lib.fh_argmax_scratch_bytes(32) == 32 * 64 * 8
    # split-K factors keep about 256 workgroups per projection launch
    assert lib.fh_gemm_default_splits(4096, 4096) == 4  # o
    assert lib.fh_gemm_default_splits(6144, 4096) == 2  # packed qkv
    assert lib.fh_gemm_default_splits(4096, 12288) == 4  # down
    assert lib.fh_gemm_default_splits(24576, 4096) == 1  # gate/up
    assert lib.fh_gemm_default_splits(151936, 4096) == 1  # LM head
    assert lib.fh_gemm_default_splits(1024, 2048) == 4  # capped at 16 k-blocks per split


def test_attention_scratch_of_a_batch_serves_every_smaller_one():
    # Few rows take smaller partitions (more records per row) than many.
    lib = ferric_amd.load()
    for heads in (8, 16, 32):
        for context in (1, 256, 257, 512, 513, 1024, 2048, 4097, 8192, 40960):
            sizes = [lib.fh_attention_scratch_bytes(rows, heads, context) for rows in range(1, 65)]
            assert sizes == sorted(sizes), (heads, context)
    assert lib.fh_attention_scratch_bytes(4, 32, 2048) == 4 * 32 * 8 * 130 * 4  # 16-page partitions
    assert lib.fh_attention_scratch_bytes(16, 32, 2048) == 16 * 32 * 4 * 130 * 4  # 32-page ones


def launch_records(rows, heads, kv_heads, context):
    """Partition records one decode attention launch writes (the partition rule of fh_op_paged_attention_noalloc)."""
    small = heads <= 16 or rows * heads <= 64 or rows * max(heads, 4 * kv_heads) * -(-context // 256) <= 1024
    pages = 32 if 256 < context <= 512 or not small else 16
    return rows * heads * -(-context // (16 * pages))


@pytest.mark.parametrize("heads", [8, 16, 17, 24, 32, 40, 64])
def test_attention_scratch_serves_every_smaller_batch_and_context(heads):
    # A shorter context may take smaller partitions than a longer one, as fewer
    # rows may: 8 rows of 32 heads need 1024 records at 1024 tokens, 960 at 1280.
    lib = ferric_amd.load()
    contexts = [1, 255, 256, 257, 511, 512, 513] + [c + d for c in range(768, 40961, 256) for d in (0, 1)]
    need = np.max([[[launch_records(rows, heads, heads // g, c) for c in contexts] for rows in range(1, 33)]
                   for g in (1, 2, 4, 8) if heads % g == 0], axis=0)
    most = np.maximum.accumulate(np.maximum.accumulate(need, axis=0), axis=1)
    got = np.array([[lib.fh_attention_scratch_bytes(rows, heads, c) for c in contexts] for rows in range(1, 33)])
    assert (got >= most * 130 * 4).all()
    # ... and the largest batch at the largest context is not asked for more than it needs itself.
    assert got[-1, -1] == need[-1, -1] * 130 * 4


def test_attention_scratch_of_a_few_rows_is_that_of_small_partitions():
    # At most 64 (row, query head) pairs take 256-token partitions at every capacity above 512 tokens.
    lib = ferric_amd.load()
    for rows, heads, context in [(1, 32, 40960), (2, 32, 8192), (2, 32, 16384), (1, 64, 32768), (3, 20, 24576)]:
        assert lib.fh_attention_scratch_bytes(rows, heads, context) == rows * heads * context // 256 * 130 * 4


def test_attention_scratch_of_nothing_is_nothing():
    lib = ferric_amd.load()
    for sizes in [(0, 32, 2048), (4, 0, 2048), (4, 32, 0), (0, 0, 0)]:
        assert lib.fh_attention_scratch_bytes(*sizes) == 0


def block(m, n, k, epilogue=_lib.EPI_BF16, fused_qkv=0):
    b = ferric_amd.load().fh_gemm_block(m, n, k, epilogue, fused_qkv)
    return b >> 16, b & 0xffff


def test_narrow_projections_take_blocks_that_split_k():
    # One or two 256-row x 128-column blocks would walk all of k on one or two
    # CUs: weights of 128 and 256 rows take the small blocks, whose waves split k.
    for n in (128, 256):
        for m in range(33, 257):
            for k in (64, 512, 1024, 2560, 4096, 12288):
                for epilogue in (_lib.EPI_BF16, _lib.EPI_RESIDUAL, _lib.EPI_SWIGLU, _lib.EPI_F32):
                    assert block(m, n, k, epilogue) < (256, 128), (m, n, k, epilogue)
    assert block(40, 120, 64) == block(40, 128, 48) == block(32, 128, 64) == block(40, 128, 64, _lib.EPI_PARTIAL) == (0, 0)
    assert block(300, 384, 1024, fused_qkv=1) == block(256, 256, 1024, fused_qkv=1) == (0, 0)  # not fused there


def test_projections_of_a_short_k_take_small_blocks():
    # With one to four k-blocks a launch is its prologue, reduction and
    # epilogue, which the smallest blocks spread over the most CUs.
    for k in (32, 64, 128):
        for n in (128, 256, 384, 512, 768, 1152):
            for m in (33, 64, 96, 160, 256, 257, 400, 600):
                for epilogue in (_lib.EPI_BF16, _lib.EPI_RESIDUAL, _lib.EPI_SWIGLU, _lib.EPI_F32):
                    rows, cols = block(m, n, k, epilogue)
                    assert 0 < rows * cols <= 64 * 64, (m, n, k, epilogue)


def test_projections_that_256_x_128_blocks_fit_badly_take_others():
    # 288 such blocks with the work of 240: some CU gets a full block and a last one (7 % slower than 256 x 256 blocks).
    for m in (520, 600, 640):
        assert block(m, 12288, 2048, _lib.EPI_SWIGLU) != (256, 128)
    # Gate/up of 8B at 3000 rows: 2256 of them in nine rounds, 5 % slower than five rounds of 256 x 256 blocks.
    assert block(3000, 24576, 4096, _lib.EPI_SWIGLU) == (256, 256)


def test_projections_of_a_very_long_k_take_64_bit_addresses():
    # From k = 2^24 on the operands of a block of 128 columns are beyond 32-bit byte offsets.
    for epilogue in (_lib.EPI_BF16, _lib.EPI_RESIDUAL, _lib.EPI_SWIGLU, _lib.EPI_F32):
        for n in (128, 384, 4096):
            for m in (33, 200, 300, 2000):
                for k in (1 << 24, (1 << 24) + 32, 1 << 27):
                    assert block(m, n, k, epilogue) in ((32, 32), (256, 256)), (m, n, k, epilogue)


def attention_form(runs, query_heads, kv_heads):
    v = ferric_amd.load().fh_prefill_attention_form(u32([p for p, _ in runs]), u32([n for _, n in runs]), len(runs),
                                                    query_heads, kv_heads)
    return v >> 16, v & 0xffff


def test_prefill_attention_form_follows_the_runs_of_a_chunk():
    # The number of rows alone does not tell: many runs of a row or two take the
    # short blocks (64 query vectors of a KV head), one long run long blocks.
    for heads, kv in [(8, 8), (16, 8), (32, 8), (32, 4)]:
        g = heads // kv
        assert attention_form([(0, 1)] * 300, heads, kv) == (64 // g, 0)
        for rows in (257, 777, 2000, 8000):
            block, form = attention_form([(0, rows)], heads, kv)
            assert form in (1, 2, 4) and block == 128 // form // g
        assert attention_form([(5, 100), (0, 156)], heads, kv) == (64 // g, 0)  # up to 256 rows: short blocks
    for runs in ([(0, 1)] * 1000, [(0, 2)] * 400):
        assert attention_form(runs, 32, 8) == (16, 0)
    for runs in ([(7000, 16)] * 20, [(2000, 32)] * 10, [(300, 1)] * 300):  # 8-row blocks: 1.4 to 1.5 times as long
        assert attention_form(runs, 32, 8) in ((16, 0), (16, 2))
    assert attention_form([(0, 300)], 24, 8) == attention_form([(0, 300)], 32, 0) == (0, 0)  # heads not supported


def measured(name):
    """Rows of a table of measured times, without its comment and heading lines."""
    with open(ROOT / "profiles" / name) as f:
        return [line.rstrip("\n").split(",") for line in f.readlines()[2:]]


def test_projection_estimates_against_the_times_they_are_fitted_to():
    blocks = [(128, 128), (64, 128), (128, 64), (64, 64), (64, 32), (32, 32), (256, 128), (256, 256)]
    codes = {"bf16": 0, "residual": 1, "swiglu": 2, "f32": 3, "qkv": 0}
    worse, against_256 = [], []
    for m, n, k, epilogue, *us in measured("projection_blocks_us.csv"):
        taken = block(int(m), int(n), int(k), codes[epilogue], epilogue == "qkv")
        if taken == (0, 0):
            continue  # the weight stream
        times = dict(zip(blocks, (float(t) if t else np.inf for t in us)))
        worse.append(times[taken] / min(times.values()))
        if int(k) >= 1024:
            against_256.append(times[taken] / times[256, 256])
    assert len(worse) > 3000 and np.mean(worse) <= 1.033 and max(worse) <= 1.7
    assert max(against_256) <= 1.03


def test_prefill_attention_estimates_against_the_times_they_are_fitted_to():
    worse, against_short = [], []
    for heads, kv, runs, *us in measured("prefill_attention_forms_us.csv"):
        rows = [r.replace("@", "x").split("x") for r in runs.split(" ")]
        _, form = attention_form([(int(p), int(n)) for c, n, p in rows for _ in range(int(c))], int(heads), int(kv))
        times = dict(zip((0, 1, 2, 4), map(float, us)))
        worse.append(times[form] / min(times.values()))
        against_short.append(times[form] / times[0])
    assert len(worse) == 1368 and np.mean(worse) <= 1.005 and max(worse) <= 1.18 and max(against_short) <= 1.18


def test_ops_reject_bad_shapes_before_any_launch():
    lib = ferric_amd.load()
    p = ctypes.c_void_p(16)  # never dereferenced: validation fails first
    assert lib.fh_op_gemm(p, p, 0, 64, 64, 0, 1, None, p, 64, None, None) == 1  # m = 0
    assert lib.fh_op_gemm(p, p, 33, 64, 64, 0, 1, None, p, 64, None, None) == 1  # m > 32 needs n % 128
    assert lib.fh_op_gemm(p, p, 257, 128, 64, 4, 1, None, p, 128, None, None) == 1  # partials above 256 rows
    assert lib.fh_op_gemm(p, p, 33, 128, 64, 4, 1, None, p, 130, None, None) == 1  # partials: 16-byte aligned rows
    assert lib.fh_op_gemm(p, p, 33, 128, 64, 0, 1, None, p, 130, None, None) == 1  # m > 32: 8-byte aligned rows
    assert lib.fh_op_gemm(p, p, 4, 60, 64, 0, 1, None, p, 64, None, None) == 1  # n % 16
    assert lib.fh_op_gemm(p, p, 4, 64, 48, 0, 1, None, p, 64, None, None) == 1  # k % 32
    assert lib.fh_op_gemm(p, p, 4, 64, 64, 1, 1, None, p, 64, None, None) == 1  # residual epilogue without residual
    assert lib.fh_op_gemm(p, p, 4, 64, 64, 9, 1, None, p, 64, None, None) == 1  # unknown epilogue
    assert lib.fh_op_gemm(p, p, 4, 64, 64, 0, 2, None, p, 64, None, None) == 1  # splits on a non-partial epilogue
    assert lib.fh_op_gemm(p, p, 4, 64, 64, 4, 3, None, p, 64, None, None) == 1  # more splits than k-blocks
    assert lib.fh_op_tile_weight(p, p, 17, 32, None) == 1
    assert lib.fh_op_tile_activation(p, p, 33, 48, None) == 1  # k % 32
    assert lib.fh_activation_rows(1) == 32 and lib.fh_activation_rows(32) == 32
    assert lib.fh_activation_rows(33) == 256 and lib.fh_activation_rows(257) == 512
    # split-K partial slabs: 32 rows for decode batches, 256 for wide ones, none beyond
    assert [lib.fh_partial_slab_rows(m) for m in (0, 1, 32, 33, 256, 257)] == [0, 32, 32, 256, 256, 0]
    # one-row projections with the norm in their prologue: the Qwen3 shapes only
    E = ferric_amd._lib
    covered = [(6144, 4096, E.EPI_PARTIAL, 2, 0), (6144, 4096, E.EPI_PARTIAL, 2, 4), (24576, 4096, E.EPI_SWIGLU, 1, 4),
               (151936, 4096, E.EPI_F32, 1, 4), (4096, 1024, E.EPI_PARTIAL, 2, 6), (6144, 1024, E.EPI_SWIGLU, 1, 4),
               (151936, 1024, E.EPI_F32, 1, 6)]
    assert all(lib.fh_gemm_rmsnorm_supported(*c) == 1 for c in covered)
    assert lib.fh_gemm_rmsnorm_supported(6144, 4096, E.EPI_PARTIAL, 2, 3) == 0  # slab count
    assert lib.fh_gemm_rmsnorm_supported(4096, 4096, E.EPI_PARTIAL, 4, 4) == 0  # the O projection's tiles
    assert lib.fh_gemm_rmsnorm_supported(6144, 8192, E.EPI_PARTIAL, 2, 4) == 0  # width
    assert lib.fh_gemm_rmsnorm_supported(6144, 4096, E.EPI_BF16, 1, 4) == 0  # epilogue
    rn = lambda h_in, h_out, part, ns, n=6144, k=4096, epi=E.EPI_PARTIAL, splits=2: lib.fh_op_gemm_rmsnorm(  # noqa: E731
        h_in, h_out, part, ns, p, 1e-6, p, n, k, epi, splits, p, n, None, None)
    q = ctypes.c_void_p(32)
    assert rn(p, p, q, 4) == 1  # the folded row would overwrite the row being read
    assert rn(p, q, None, 4) == 1  # slabs missing
    assert rn(p, None, q, 4) == 1  # no output row
    assert rn(p, q, q, 3) == 1 and rn(p, q, q, 4, n=4096, splits=4) == 1  # not covered
    ms = ctypes.c_float()
    assert lib.fh_time_attention(None, 1, ctypes.byref(ms)) == 1  # no context
    assert lib.fh_op_rmsnorm(p, p, p, 1, 8200, 1e-6, None, None) == 1
    assert lib.fh_op_residual_rmsnorm(p, None, 2, p, p, 1, 4, 4096, 1e-6, None, None) == 1  # partials missing
    assert lib.fh_op_residual_rmsnorm(p, p, 2, p, p, 1, 257, 4096, 1e-6, None, None) == 1  # partials above 256 rows
    assert lib.fh_op_paged_attention(p, p, p, p, p, p, 0, p, 1, 32, 6, 4, 4, 64, None, None) == 1  # 32 % 6
    assert lib.fh_op_paged_attention(p, p, p, p, p, p, 0, p, 1, 32, 8, 4, 4, 65, None, None) == 1  # stride*16 < ctx
    # fused QK-norm + attention: 2 slabs, at most 4 query heads per KV head, at most 32 rows
    qkn = lambda splits, rows, qh: lib.fh_op_qknorm_paged_attention(  # noqa: E731
        p, splits, p, p, p, p, p, p, p, p, p, 1, p, rows, qh, 8, 64, 64, 1024, 1e-6, None, None)
    assert qkn(3, 4, 32) == 1 and qkn(1, 4, 32) == 1  # slab count
    assert qkn(2, 4, 64) == 1  # 8 query heads per KV head
    assert qkn(2, 33, 32) == 1 and qkn(2, 0, 32) == 1  # rows


def test_create_rejects_unsupported_shapes_without_touching_the_device():
    lib = ferric_amd.load()
    desc = _lib.ModelDesc(2, 1024, 16, 8, 64, 3072, 151936, 1, 1_000_000, 1e-6)  # head_dim 64
    opts = _lib.CtxOptions(8, 64, 32, 512, 0, 0, 0, 0)
    ctx = ctypes.c_void_p()
    assert lib.fh_create(ctypes.byref(desc), ctypes.byref(opts), ctypes.byref(ctx)) == 1
    assert b"unsupported model shape" in lib.fh_last_error(None)
    desc = _lib.ModelDesc(2, 1024, 16, 8, 128, 3072, 151936, 1, 1_000_000, 1e-6)
    opts = _lib.CtxOptions(33, 64, 32, 512, 0, 0, 0, 0)  # more rows than the 32-row envelope
    assert lib.fh_create(ctypes.byref(desc), ctypes.byref(opts), ctypes.byref(ctx)) == 1
    opts = _lib.CtxOptions(8, 64, 16, 512, 0, 0, 0, 0)  # stride * 16 < context
    assert lib.fh_create(ctypes.byref(desc), ctypes.byref(opts), ctypes.byref(ctx)) == 1


def test_page_pool_reserves_write_slots_and_consecutive_positions():
    limits = PagedLimits(context_tokens=128, physical_page_count=20, page_table_stride=8)
    pool = PagePool(limits, seed=3)
    a = pool.admit(15)
    b = pool.admit(0)
    batch = pool.prepare([(a, 7), (a, 8), (b, 9)])
    rows = batch.rows
    assert [r.position for r in rows] == [15, 16, 0]
    assert list(rows[0].physical_pages) == list(rows[1].physical_pages) and len(rows[0].physical_pages) == 2
    assert rows[0].writable_physical_page == rows[0].physical_pages[0]
    assert rows[1].writable_physical_page == rows[1].physical_pages[1]
    assert rows[1].writable_token_offset == 0
    pool.commit(batch)
    assert pool.sequences[a].length == 17 and pool.sequences[b].length == 1
    all_pages = [p for s in pool.sequences.values() for p in s.pages]
    assert len(all_pages) == len(set(all_pages))
    with pytest.raises(ValueError):
        pool.prepare([(a, 1)] * 120)


def test_page_pool_large_batch_matches_row_loop():
    # Batches above 256 rows are prepared with array operations; they must
    # give the same positions, page lists, write slots and page-allocation
    # order as the row-by-row path, for interleaved sequences with prefixes.
    from ferric_amd.runner import PreparedRows

    limits = PagedLimits(context_tokens=1024, physical_page_count=400, page_table_stride=64)

    def build():
        pool = PagePool(limits, seed=11)
        sids = [pool.admit(n) for n in (0, 15, 16, 33, 300)]
        rng = np.random.default_rng(5)
        rows = [(sids[i], int(t)) for i, t in zip(rng.integers(0, 5, 600), rng.integers(0, 151936, 600))]
        return pool, rows

    # A decode step (every row a different sequence) takes the per-column path,
    # which reuses the previous decode batch's page-list block while the
    # sequences and their page counts are unchanged: 40 steps in a row (page
    # boundaries crossed, a sequence released and another admitted) against
    # the row loop on a twin pool.
    for pick in ([0, 1, 2, 3, 4], [4, 2, 0, 3, 1]):
        pool_a, _ = build()
        pool_b, _ = build()
        sa, sb = sorted(pool_a.sequences), sorted(pool_b.sequences)
        for step in range(40):
            if step == 20:
                pool_a.release(sa[pick[1]])
                pool_b.release(sb[pick[1]])
                sa[pick[1]], sb[pick[1]] = pool_a.admit(3), pool_b.admit(3)
            ba = pool_a._prepare_decode([(sa[i], 100 + step + i) for i in pick])
            states, sid, token, pos, group = pool_b._prepare_loop([(sb[i], 100 + step + i) for i in pick])
            rows = ba.rows
            np.testing.assert_array_equal(rows.token, token)
            np.testing.assert_array_equal(rows.position, pos)
            for i, r in enumerate(rows):
                np.testing.assert_array_equal(r.physical_pages, states[group[i]].pages)
                assert r.writable_physical_page == r.physical_pages[r.position // 16]
                assert not r.physical_pages.flags.writeable
            assert pool_a.free == pool_b.free
            pool_a.commit(ba)
            for s, p in zip(sid.tolist(), pos.tolist()):
                pool_b.sequences[s].length = p + 1
    pool_a, _ = build()
    assert pool_a._prepare_decode([(1, 5), (2, 6), (1, 7)]) is None  # a repeated sequence
    pool_a, rows = build()
    pool_b, _ = build()
    cols_a = pool_a._prepare_vector(rows)
    cols_b = pool_b._prepare_loop(rows)
    assert [st.sequence for st in cols_a[0]] == [st.sequence for st in cols_b[0]]
    for x, y in zip(cols_a[1:], cols_b[1:]):
        np.testing.assert_array_equal(x, y)
    assert pool_a.free == pool_b.free
    for s in pool_a.sequences:
        np.testing.assert_array_equal(pool_a.sequences[s].pages, pool_b.sequences[s].pages)
    batch = pool_a.prepare(rows[:400])
    assert isinstance(batch.rows, PreparedRows) and len(batch.rows) == 400
    r = batch.rows[-1]
    assert r.writable_physical_page == r.physical_pages[r.position // 16]
    assert not r.physical_pages.flags.writeable
    with pytest.raises(ValueError):
        pool_a.prepare([(rows[0][0], -1)] * 300)


def test_page_pool_small_batches_match_the_general_path():
    # Up to 4 rows are prepared and marshalled on a short path (a batch-1
    # decode step runs it every step); it must give the columns, page lists,
    # allocations and fh_row records of the general path.
    import ctypes

    from ferric_amd.runner import _rows_to_c

    limits = PagedLimits(context_tokens=1024, physical_page_count=200, page_table_stride=64)

    def build():
        pool = PagePool(limits, seed=5)
        return pool, [pool.admit(n) for n in (0, 15, 16, 47, 300)]

    for rows_of in ([(0, 7)], [(1, 9)], [(4, 3), (4, 4)], [(2, 1), (1, 2), (2, 3), (0, 4)], [(3, 8), (3, 9)]):
        pool_a, sa = build()
        pool_b, sb = build()
        rows_a = [(sa[i], t) for i, t in rows_of]
        rows_b = [(sb[i], t) for i, t in rows_of]
        small = pool_a.prepare(rows_a).rows
        states, sid, token, pos, group = pool_b._prepare_loop(rows_b)
        assert pool_a.free == pool_b.free
        for s_a, s_b in zip(sa, sb):
            np.testing.assert_array_equal(pool_a.sequences[s_a].pages, pool_b.sequences[s_b].pages)
        np.testing.assert_array_equal(small.token, token)
        np.testing.assert_array_equal(small.position, pos)
        np.testing.assert_array_equal(small.table_index, group)
        assert small.token.dtype == np.uint32 and small.sequence.dtype == np.uint64
        for i, r in enumerate(small):
            np.testing.assert_array_equal(r.physical_pages, states[group[i]].pages)
            assert r.writable_physical_page == r.physical_pages[r.position // 16]
            assert not r.physical_pages.flags.writeable
        ptr, keep = _rows_to_c(small)
        for i, r in enumerate(small):
            c = ptr[i]
            assert (c.sequence, c.token, c.position, c.page_count, c.writable_page) == (
                r.sequence, r.token, r.position, len(r.physical_pages), r.writable_physical_page)
            assert list(c.pages[: c.page_count]) == list(r.physical_pages)
            assert ctypes.addressof(c.pages.contents) == r.physical_pages.__array_interface__["data"][0]
    pool, s = build()
    with pytest.raises(ValueError):
        pool.prepare([(s[0], -1)])
    with pytest.raises(ValueError):
        pool.prepare([(s[0], 1 << 32)])


def test_library_shares_torch_hip_runtime():
    # Importing the package before torch must still leave one HIP runtime in
    # the process (two copies disagree about which devices exist).
    import subprocess
    import sys

    code = ("import ferric_amd, torch\n"
            "maps = open('/proc/self/maps').read().splitlines()\n"
            "print(len({l.split()[-1] for l in maps if 'libamdhip64' in l}))\n")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT, timeout=300)
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip() == "1"
