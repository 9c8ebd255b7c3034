"""The C-ABI library loads and exports every symbol include/cce_hip.h declares; the host-only
queries answer without a GPU.  No compute entry point is called here."""

import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "cce_hip.h")


def _declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(cce_[a-z_0-9]+)\s*\(", text)))


def _lib():
    from cut_cross_entropy import _hip

    if not os.path.exists(_hip.lib_path()):
        pytest.fail(f"{_hip.lib_path()} is missing: run __graft_entry__.build() first")
    return _hip.load()


def test_header_declares_the_expected_entry_points():
    names = _declared_functions()
    for want in ("cce_version", "cce_error_string", "cce_tile_stat_elems", "cce_lse_forward_workspace_bytes",
                 "cce_lse_forward", "cce_indexed_neg_dot", "cce_backward_workspace_bytes", "cce_backward",
                 "cce_backward_dz", "cce_lse_forward_static", "cce_lse_forward_static_init", "cce_backward_dense",
                 "cce_backward_dense_workspace_bytes", "cce_backward_dense_fixed_bytes", "cce_backward_dense_dz_bytes",
                 "cce_count_flagged_cells", "cce_backward_products"):
        assert want in names


def test_library_exports_every_declared_symbol():
    lib = _lib()
    for name in _declared_functions():
        assert hasattr(lib, name), f"libcce_hip.so does not export {name}"


def test_binding_covers_every_declared_symbol():
    from cut_cross_entropy import _hip

    assert sorted(_hip._SIGNATURES) == _declared_functions()


def test_host_only_queries():
    lib = _lib()
    from cut_cross_entropy import _hip

    assert lib.cce_version() == _hip.ABI_VERSION
    assert lib.cce_error_string(0) == b"success"
    assert lib.cce_source_hash().decode() == _hip._hash_of_sources()  # the library matches the sources beside it
    assert b"workspace" in lib.cce_error_string(10003)
    # ceil(8192 / 32) * ceil(256000 / 32)
    assert lib.cce_tile_stat_elems(8192, 256000) == 256 * 8000
    assert lib.cce_tile_stat_elems(33, 129) == 2 * 5
    assert lib.cce_tile_stat_elems(0, 100) == 0
    ws = lib.cce_lse_forward_workspace_bytes(8192, 256000, 2304)
    assert ws > 0 and ws % 8 == 0 and ws <= 16 * 2**20
    # one bit per 32 x 32 sub-tile, rows padded to 32-bit words
    # survivor bits (256 row groups x 250 words) + a count and one id per class group for the second dC pass
    assert lib.cce_backward_workspace_bytes(8192, 256000, 2304) == 256 * 250 * 4 + (1 + 8000) * 4
    assert lib.cce_backward_workspace_bytes(0, 5, 5) == 0
    # rows of more than one slice: room for kept gradients on top, which not every call uses (candidate bits, 40 slots of 2 KB)
    lists = 2048 * 149 * 4 + (1 + 4752) * 4
    assert lib.cce_backward_unkept_workspace_bytes(65536, 152064, 3584) == lists
    kept = 2048 * 149 * 4 + 2048 * 40 * 2048
    assert lib.cce_backward_workspace_bytes(65536, 152064, 3584) == (lists + 15) // 16 * 16 + kept


def test_header_constants_match_binding():
    from cut_cross_entropy import _hip

    text = open(HEADER).read()
    assert int(re.search(r"#define CCE_STAT_ROWS (\d+)", text).group(1)) == _hip.STAT_ROWS
    assert int(re.search(r"#define CCE_STAT_COLS (\d+)", text).group(1)) == _hip.STAT_COLS
    assert int(re.search(r"#define CCE_NUM_COUNTERS (\d+)", text).group(1)) == _hip.NUM_COUNTERS
    assert int(re.search(r"#define CCE_DTYPE_BF16 (\d+)", text).group(1)) == 0
    assert int(re.search(r"#define CCE_DTYPE_F16 (\d+)", text).group(1)) == 1
    m = re.search(r"#define CCE_STATIC_SCRATCH_BYTES \((\d+) \* (\d+) \* (\d+)\)", text)
    assert int(m.group(1)) * int(m.group(2)) * int(m.group(3)) == _hip.STATIC_SCRATCH_BYTES


def test_dense_backward_plans_by_classes_or_by_rows():
    """Host-only size queries of the unfiltered backward: with 16-bit gradients and at least twice as many rows as
    classes the walk goes by blocks of rows and the compensation term in the workspace is [v, d], else [b, d]."""
    lib = _lib()
    a256 = lambda x: (x + 255) // 256 * 256
    # rows few against classes: by classes; fixed part = compensation term of dE
    assert lib.cce_backward_dense_fixed_bytes(8192, 256000, 2304, 1) == a256(8192 * 2304 * 2)
    assert lib.cce_backward_dense_fixed_bytes(8192, 256000, 2304, 0) == 0
    assert lib.cce_backward_dense_dz_bytes(8192, 256000, 2304, 1, 1024) == 8192 * 1024 * 2
    # a vocabulary shard: by rows; fixed part = compensation term of dC; a dz unit is 256 rows of all classes
    B, V, D = 65536, 19008, 3584
    v_pad = a256(V)
    assert lib.cce_backward_dense_fixed_bytes(B, V, D, 1) == a256(V * D * 2)
    assert lib.cce_backward_dense_fixed_bytes(B, V, D, 0) == 0           # fp32 gradients: by classes, nothing fixed
    assert lib.cce_backward_dense_dz_bytes(B, V, D, 1, 1024) == 1024 * v_pad * 2
    assert lib.cce_backward_dense_dz_bytes(B, V, D, 0, 1024) == B * 1024 * 2
    # the whole workspace: fixed part + a dz buffer inside the budget, never below one 256-row block
    for budget in (0, 64 << 20, 256 << 20, 1 << 32):
        total = lib.cce_backward_dense_workspace_bytes(B, V, D, 1, budget)
        dz = total - a256(V * D * 2)
        assert dz % (256 * v_pad * 2) == 0 and dz >= 256 * v_pad * 2
        assert dz <= max(budget, 256 * v_pad * 2)
        assert dz <= a256(B) * v_pad * 2


def test_dense_backward_goes_by_rows_only_where_offsets_reach_a_block():
    """Rows of dz of a walk by rows are a vocabulary apart, and 256 of them are reached by 32-bit byte offsets: up to 2^23 classes.
    More go by classes, in chunks whose 256 rows are reached."""
    lib = _lib()
    a256 = lambda x: (x + 255) // 256 * 256
    D = 64
    for V in (1 << 23, (1 << 23) + 1):
        B = 2 * a256(V)
        by_rows = V == 1 << 23
        assert lib.cce_backward_dense_fixed_bytes(B, V, D, 1) == a256((V if by_rows else B) * D * 2)
        units = 4096
        dz = lib.cce_backward_dense_dz_bytes(B, V, D, 1, units)
        assert dz == units * (a256(V) if by_rows else B) * 2
        row = a256(V) if by_rows else units  # classes from one row of dz to the next
        assert (255 * row + 56) * 2 < 1 << 32
        total = lib.cce_backward_dense_workspace_bytes(B, V, D, 1, dz)
        assert total >= a256((V if by_rows else B) * D * 2) + 256 * (a256(V) if by_rows else B) * 2


@pytest.mark.parametrize("sizes", [(0, 10, 64), (10, 0, 64), (10, 10, 0), (0, 0, 0)])
def test_size_queries_answer_for_empty_matrices(sizes):
    """A query is asked before the call that refuses such sizes, so it has to answer."""
    from cut_cross_entropy import _hip

    lib = _hip.load()
    assert lib.cce_lse_forward_workspace_bytes(*sizes) >= 0
    assert 0 <= lib.cce_backward_workspace_bytes(*sizes) <= 12
    assert lib.cce_backward_dense_workspace_bytes(*sizes, 1, 1 << 20) == 0
    assert lib.cce_fp32_forward_workspace_bytes(*sizes, 6) == 0
    assert lib.cce_fp32_backward_workspace_bytes(*sizes, 6) == 0


@pytest.mark.parametrize("sizes,unit,budget", [
    ((65536, 19008, 3584), 6656, 256 << 20), ((41192, 11918, 4864), 10496, 256 << 20), ((53256, 10706, 3200), 10752, 256 << 20),
    ((5472, 148531, 1856), 11776, 256 << 20), ((3879, 33278, 3840), 12288, 256 << 20), ((3209, 48576, 4992), 15104, 256 << 20),
    ((5824, 134912, 2688), 11264, 256 << 20), ((14400, 9131, 3840), 9216, 256 << 20)])
def test_plans_of_whole_reductions_do_not_go_by_the_estimate_for_cut_ones(sizes, unit, budget):
    """Rows per block (more than twice as many rows as classes) or classes per chunk of shapes whose reductions are not cut:
    where the launches begin decides where the carried 16-bit gradient is rounded."""
    lib = _lib()
    a256 = lambda x: (x + 255) // 256 * 256
    b, v, d = sizes
    by_rows = b >= 2 * a256(v)
    fixed = lib.cce_backward_dense_fixed_bytes(b, v, d, 1)
    assert fixed == a256((v if by_rows else b) * d * 2)
    dz = lib.cce_backward_dense_workspace_bytes(b, v, d, 1, budget) - fixed
    assert dz == a256((unit * a256(v) if by_rows else unit * b) * 2)


def test_a_plan_of_the_fp32_backward_is_searched_once():
    """The size query and the call ask for the plan of the same sizes, every step of a training loop again: the answer to a
    question asked before costs a small part of a search."""
    import time

    lib = _lib()
    b, v, d = 39665, 153856, 160

    def seconds(sizes):
        best = 1.0
        for _ in range(5):
            start = time.perf_counter()
            for n in sizes:
                lib.cce_fp32_backward_workspace_bytes(n, v, d, 6)
            best = min(best, time.perf_counter() - start)
        return best

    searched, known = seconds(range(b, b + 200)), seconds([b] * 200)
    assert known < searched / 4, (known, searched)
    # ... and is the answer of a search of its own
    answer = lib.cce_fp32_backward_workspace_bytes(b, v, d, 6)
    for n in range(1, 20):
        lib.cce_fp32_backward_workspace_bytes(b + n, v, d, 6)
    assert lib.cce_fp32_backward_workspace_bytes(b, v, d, 6) == answer
