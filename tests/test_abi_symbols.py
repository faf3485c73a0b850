"""The C-ABI library loads and exports every symbol include/gs_hip.h declares (no GPU needed)."""
import ctypes
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "gs_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(gs_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_surface():
    syms = _declared_symbols()
    for must in ("gs_slice_count", "gs_slice_fill", "gs_sample_count", "gs_sample_uniform_fill",
                 "gs_sample_one_keepdim", "gs_sample_weighted_fill", "gs_unique_relabel",
                 "gs_random_walk", "gs_metapath_walk", "gs_sddmm_coo", "gs_sddmm_csc",
                 "gs_segment_sum", "gs_coo_sum", "gs_segment_normalize", "gs_e_div_u_sum",
                 "gs_list_sample_uniform", "gs_list_sample_weighted", "gs_row_slice_csc_mark",
                 "gs_row_slice_coo_mark", "gs_csc2coo", "gs_coo2csc"):
        assert must in syms


def test_library_exports_every_declared_symbol():
    from graph_sampling_amd import capi
    lib = ctypes.CDLL(capi.LIB_PATH)
    missing = [s for s in _declared_symbols() if not hasattr(lib, s)]
    assert not missing, missing


def test_status_strings_and_argument_errors_without_a_gpu():
    """Argument validation happens before any HIP call, so it can be exercised on the CPU."""
    from graph_sampling_amd import capi
    lib = capi.lib()
    assert lib.gs_version() >= 100
    assert lib.gs_status_string(0) == b"ok"
    st = lib.gs_slice_count(None, ctypes.c_int64(4), None, 8, ctypes.c_int64(4), None, None,
                            ctypes.c_size_t(0), None)
    assert st == -1 and b"gs_slice_count" in lib.gs_status_string(st)
    buf = (ctypes.c_int64 * 64)()
    st = lib.gs_sample_count(buf, ctypes.c_int64(8), buf, 3, ctypes.c_int64(4), ctypes.c_int64(2), 0,
                             buf, None, ctypes.c_size_t(0), None)
    assert st == -1 and b"id_bytes" in lib.gs_status_string(st)
    # workspace too small / misaligned is reported, not executed
    st = lib.gs_sample_count(buf, ctypes.c_int64(8), buf, 8, ctypes.c_int64(4), ctypes.c_int64(2), 0,
                             buf, None, ctypes.c_size_t(0), None)
    assert st == -2
    assert lib.gs_sample_workspace_bytes(ctypes.c_int64(1000), ctypes.c_int64(5)) > 0


def test_python_binding_rejects_cpu_tensors():
    import pytest
    import torch
    from graph_sampling_amd import capi
    indptr = torch.zeros(3, dtype=torch.int64)
    with pytest.raises(capi.GsError, match="no CPU path"):
        capi.slice_count(indptr, torch.zeros(2, dtype=torch.int64))


def test_every_entry_point_names_what_it_replaces():
    """Each declaration of the header stands under a comment (its own or its section's) that cites
    the reference interface it replaces as file:line, or says that it has no counterpart there."""
    lines = open(os.path.join(ROOT, "include", "gs_hip.h")).read().split("\n")
    uncited = []
    for i, line in enumerate(lines):
        m = re.match(r"^(int|size_t|int64_t|const char\*)\s+(gs_[a-z0-9_]+)\s*\(", line)
        if not m:
            continue
        above = "\n".join(lines[max(0, i - 60):i])
        if not re.search(r"(src/|examples/|tests/|python/)[A-Za-z_/\.]+:\d+|counterpart", above, re.I):
            uncited.append(m.group(2))
    assert not uncited, uncited


def test_walks_make_a_table_of_offsets_where_it_pays():
    """Both sides of every line of the rule: nodes, walkers, walkers for the nodes, steps, edges a node (dense graphs,
    whose hubs' records cost more than they save, and large graphs whose walks end early)."""
    from graph_sampling_amd import capi

    def made(nodes, edges, walkers, length):
        return capi.lib().gs_random_walk_workspace_bytes(*(ctypes.c_int64(v) for v in (nodes, edges, walkers, length))) > 0

    k, M = 1 << 10, 1 << 20
    for yes, no in [((256 * k, 4 * M, 128 * k, 20), (256 * k - 1, 4 * M, 128 * k, 20)),
                    ((256 * k, 4 * M, 128 * k, 20), (256 * k, 4 * M, 128 * k - 1, 21)),
                    ((M, 20 * M, M, 4), (M, 20 * M, M, 3)),  # 2^21 + 1.5 * 2^20 steps
                    ((4 * M, 100 * M, 256 * k, 40), (4 * M, 100 * M, 256 * k - 1, 40)),  # a walker for 16 nodes
                    ((8 * M, 80 * M, 512 * k, 30), (8 * M, 80 * M, 300_000, 200)),
                    ((64 * M, 800 * M, 1_000_000, 120), (64 * M, 800 * M, 999_999, 400)),
                    ((64 * M, 64 * 8 * M, M, 120), (64 * M + 1, 64 * 8 * M, M, 120)),
                    ((111_000_000, 1_600_000_000, M, 200), (111_000_000, 900_000_000, M, 200)),
                    ((128 * M, 128 * 12 * M, M, 200), (128 * M + 1, 128 * 16 * M, M, 200)),
                    ((256 * k, 128 * M - 1, M, 80), (256 * k, 128 * M, M, 80)),  # 512 edges a node
                    ((M, 320 * M - 1, M, 80), (M, 320 * M, M, 80)),
                    ((4 * M, 200 * M, M, 80), (4 * M, 4096 * M, M, 80))]:
        assert made(*yes) and not made(*no), (yes, no)
    assert not made(M, 20 * M, M, 0) and not made(0, 0, M, 4) and not made(M, 20 * M, 0, 80)

    def metapath(relations, nodes, walkers, length):
        return capi.lib().gs_metapath_walk_workspace_bytes(*(ctypes.c_int64(v) for v in (relations, nodes, walkers, length))) > 0

    for yes, no in [((3, 256 * k, 128 * k, 20), (3, 256 * k - 1, 128 * k, 20)),
                    ((16, M, 200_000, 20), (17, M, 200_000, 20)),
                    ((3, 4 * M, 128 * k, 80), (3, 4 * M + 32, 128 * k, 80)),  # a walker for 32 nodes
                    ((3, 32 * M, 1_000_000, 80), (3, 32 * M, 999_999, 80)),
                    ((3, 32 * M, M, 80), (3, 32 * M + 1, M, 80)),
                    ((1, M, M, 4), (1, M, M, 3))]:
        assert metapath(*yes) and not metapath(*no), (yes, no)
    assert not metapath(0, M, M, 80)
