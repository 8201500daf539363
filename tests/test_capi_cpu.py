"""CPU-side checks of the boundary: the shared library loads, exports every symbol the header
declares, and the Python binding's signature table matches the header."""
import ctypes
import os
import re

import pytest

from metaseq_amd import _capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "metaseq_amd.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    decls = {}
    for m in re.finditer(r"\b(msa_\w+)\s*\(([^;{]*?)\)\s*;", text, flags=re.S):
        args = [a.strip() for a in m.group(2).split(",") if a.strip() and a.strip() != "void"]
        decls[m.group(1)] = args
    return decls


def test_library_exports_every_declared_symbol():
    if not os.path.exists(_capi.LIB_PATH):
        from metaseq_amd.csrc.build import build
        build(force=True, verbose=False)
    lib = ctypes.CDLL(_capi.LIB_PATH)
    decls = _declared()
    assert len(decls) >= 12
    for name in decls:
        assert hasattr(lib, name), name


def test_binding_table_matches_header_arity():
    decls = _declared()
    for name, argtypes in _capi.SIGNATURES.items():
        assert name in decls, name
        assert len(argtypes) == len(decls[name]), (name, len(argtypes), decls[name])
    for name in decls:
        assert name in _capi.SIGNATURES or name in _capi.OTHER_SYMBOLS, name


def test_loader_reports_version_and_fails_loudly_without_library(monkeypatch, tmp_path):
    lib = _capi.load()
    assert lib.msa_version() >= 1
    monkeypatch.setattr(_capi, "_lib", None)
    monkeypatch.setattr(_capi, "LIB_PATH", str(tmp_path / "missing.so"))
    with pytest.raises(RuntimeError, match="no non-HIP fallback"):
        _capi.load()


def test_argument_validation_needs_no_gpu():
    """Entry points reject bad arguments before touching the device."""
    lib = _capi.load()
    assert lib.msa_layernorm_f16(None, None, None, None, 1, 64, 1e-5, 0, None) == -1
    assert b"null pointer" in lib.msa_last_error()
    one = ctypes.c_void_p(16)
    assert lib.msa_linear_f16(one, one, None, None, one, 4, 16, 40, 0, None) == -1
    assert b"multiple of 32" in lib.msa_last_error()
    assert lib.msa_attention_f16(one, one, one, None, 0, one, 1, 1, 64, 2, 9, 10, 0, None, None) == -2
    with pytest.raises(ValueError):
        _capi.check(-2, lib)
    # split-K counts that would leave a slice of the partial sums unwritten are refused
    assert lib.msa_linear_partial_f16(one, one, one, 58, 50272, 160, 4, 2, None) == -1
    assert b"leaves a K range empty" in lib.msa_last_error()
    assert lib.msa_linear_partial_w8a16(one, one, one, one, 52, 8000, 768, 8, 2, None) == -1
    assert b"leaves a K range empty" in lib.msa_last_error()


@pytest.mark.parametrize("int8", [0, 1])
@pytest.mark.parametrize("width", [768, 1024, 2048, 4096, 5120, 9216])
def test_a_workspace_for_more_rows_serves_fewer(width, int8):
    """... also where more rows are summed in fewer slices."""
    lib, h, one = _capi.load(), ctypes.c_void_p(), ctypes.c_void_p(4096)
    conf = _capi.DecoderConfig(1, width, width // 128, 4 * width, 512, 40, 1, int8)
    table = (_capi.LayerWeights * 1)()
    for name, _ in _capi.LayerWeights._fields_:
        setattr(table[0], name, 4096)
    assert lib.msa_decoder_create(ctypes.byref(conf), one, one, one, one, one, table, ctypes.byref(h)) == 0
    need = [lib.msa_decoder_step_workspace_bytes(h, b) for b in range(16, 65)]
    lib.msa_decoder_destroy(h)
    assert need == sorted(need) and need[0] > 0


def step_workspaces(width, int8, vocab, positions, rows):
    lib, h, one = _capi.load(), ctypes.c_void_p(), ctypes.c_void_p(4096)
    conf = _capi.DecoderConfig(1, width, width // 128, 4 * width, vocab, positions, 1, int8)
    table = (_capi.LayerWeights * 1)()
    for name, _ in _capi.LayerWeights._fields_:
        setattr(table[0], name, 4096)
    assert lib.msa_decoder_create(ctypes.byref(conf), one, one, one, one, one, table, ctypes.byref(h)) == 0
    need = [lib.msa_decoder_step_workspace_bytes(h, b) for b in rows]
    lib.msa_decoder_destroy(h)
    return need


@pytest.mark.parametrize("int8", [0, 1])
@pytest.mark.parametrize("vocab,positions", [(512, 40), (50272, 2050), (512, 8194)])
@pytest.mark.parametrize("width", [128, 768, 1024, 2048, 4096, 5120, 9216])
def test_every_buffer_of_a_workspace_for_more_rows_serves_fewer(width, vocab, positions, int8):
    """... also where no two launches attend to them, or no projection selects."""
    need = step_workspaces(width, int8, vocab, positions, range(1, 129))
    assert need == sorted(need) and need[0] > 0


FEED_FORWARDS = {"dense": dict(ff_kind=_capi.MSA_FF_DENSE), "relu2": dict(ff_kind=_capi.MSA_FF_RELU2),
                 # hardly a row, some rows and many to an expert; with few experts and with a shared one
                 "routed": dict(ff_kind=_capi.MSA_FF_MOE, experts=64, top=8, ff_expert=1408),
                 "few experts": dict(ff_kind=_capi.MSA_FF_MOE, experts=12, top=2, ff_expert=128),
                 "shared": dict(ff_kind=_capi.MSA_FF_MOE, experts=64, top=4, ff_expert=704, ff_shared=704)}


@pytest.mark.parametrize("dtype", [0, 1], ids=["bf16", "fp32"])
@pytest.mark.parametrize("ff", FEED_FORWARDS)
@pytest.mark.parametrize("width", [128, 512, 1024, 2048, 4096])
def test_a_hybrid_workspace_for_more_rows_serves_fewer(width, ff, dtype):
    """... where more rows are summed in fewer slices, or routed in fewer tiles."""
    lib, h = _capi.load_hybrid(), ctypes.c_void_p()
    t, cfg = _capi.HybridLayer(), _capi.HybridConfigC()
    for s in (t, cfg):
        for name, kind in s._fields_:
            if kind is ctypes.c_void_p:
                setattr(s, name, 4096)      # never followed
    t.kind, t.channels, t.blocks, t.taps, t.ko, t.n_in = _capi.MSA_MIX_RGLRU, width, 1, 4, width, 2 * width
    t.n_groups, t.keep, t.router_scale, t.ff = 1, 1, 1.0, 4 * width
    for name, value in FEED_FORWARDS[ff].items():
        setattr(t, name, value)
    t.n_ff_in = {"dense": 8 * width, "relu2": 4 * width}.get(ff, (2 * t.ff_shared + t.experts + 16) // 16 * 16)
    cfg.dtype, cfg.layers, cfg.D, cfg.Dp, cfg.vocab, cfg.Vp, cfg.eps, cfg.n_runs = dtype, 1, width, width, 16, 16, 1e-6, 0
    assert lib.msa_hybrid_create(ctypes.byref(cfg), (_capi.HybridLayer * 1)(t), ctypes.byref(h)) == 0, lib.msa_last_error()
    need = []
    for rows in list(range(1, 300)) + [384, 511, 512, 513, 768, 769, 1024, 1025, 2048, 2049, 4096, 4097]:
        a = _capi.HybridStepArgs()
        a.batch.M = a.batch.nseg = rows
        a.batch.max_count = a.batch.key_bound = a.capacity = 1
        need.append(lib.msa_hybrid_workspace_bytes(h, ctypes.byref(a)))
    lib.msa_hybrid_destroy(h)
    assert need == sorted(need) and need[0] > 0


def test_decoder_handle_is_host_only_bookkeeping():
    """msa_decoder_create validates and copies a pointer table without touching a GPU; the
    workspace size grows with the row count; a bad configuration or a missing pointer is
    refused."""
    lib = _capi.load()
    conf = _capi.DecoderConfig(2, 128, 2, 512, 64, 40, 1, 0)
    table = (_capi.LayerWeights * 2)()
    for t in table:
        for name, _ in _capi.LayerWeights._fields_:
            setattr(t, name, 4096)
    h = ctypes.c_void_p()
    one = ctypes.c_void_p(4096)
    assert lib.msa_decoder_create(ctypes.byref(conf), one, one, one, one, one, table,
                                  ctypes.byref(h)) == 0
    w8, w40 = (lib.msa_decoder_step_workspace_bytes(h, b) for b in (8, 40))
    w100 = lib.msa_decoder_step_workspace_bytes(h, 100)
    assert 0 < w8 < w40 and w100 > 0 and lib.msa_decoder_step_workspace_bytes(h, 129) == 0
    args = _capi.StepArgs()
    assert lib.msa_decoder_step(h, ctypes.byref(args), None) == -1     # nothing filled in
    lib.msa_decoder_destroy(h)
    table[1].fc2_bias = None
    assert lib.msa_decoder_create(ctypes.byref(conf), one, one, one, one, one, table,
                                  ctypes.byref(h)) == -1
    assert b"layer 1" in lib.msa_last_error()
    bad = _capi.DecoderConfig(2, 160, 2, 512, 64, 40, 1, 0)            # head_dim 80
    assert lib.msa_decoder_create(ctypes.byref(bad), one, one, one, one, one, table,
                                  ctypes.byref(h)) == -1


@pytest.mark.parametrize("N,K,rows,fp16,bf16", [
    (2048, 8192, (1, 4, 8), 4, 8),     # the next product of an fp16 step sums four slices itself
    (2048, 8192, (9, 16), 8, 8),       # but not of more rows,
    (2560, 10240, (1, 8, 16), 8, 8),   # nor of a wider model
    (5120, 20480, (1, 4), 8, 8),
    (5120, 20480, (8, 16), 4, 4),
    (1024, 4096, (1, 8, 16), 4, 4),
])
def test_only_products_that_fold_stop_at_four_slices(N, K, rows, fp16, bf16):
    """(256 compute units: also where there is no device)"""
    core, hybrid = _capi.load(), _capi.load_hybrid()
    for M in rows:
        assert core.msa_linear_default_splits(M, N, K) == fp16, M
        assert hybrid.msa_linear_bf16_splits(M, N, K, 1) == bf16, M


@pytest.mark.parametrize("M,N,K,fp16,int8", [
    # queues of few tiles, or twice the slices in one pass of the shared-activation kernel
    (128, 12288, 12288, 4, 2), (100, 12288, 49152, 4, 2), (128, 9216, 36864, 4, 2), (128, 5120, 20480, 8, 4),
    (64, 12288, 12288, 2, 2), (64, 12288, 49152, 4, 4), (40, 12288, 49152, 4, 4), (57, 4096, 16384, 4, 4),
    # up to 32 rows: as many as the stream kernel takes, unless queues take others
    (9, 6640, 8256, 4, 4), (32, 5120, 5120, 4, 4), (32, 9216, 9216, 2, 2), (16, 9216, 9216, 4, 2), (32, 9216, 36864, 4, 4)])
def test_slices_of_packed_rows(M, N, K, fp16, int8):
    """(256 compute units)"""
    core = _capi.load()
    assert (core.msa_linear_default_splits(M, N, K), core.msa_linear_default_splits_w8a16(M, N, K)) == (fp16, int8)


def tiles(M, N, K, S=0, cus=256):
    f = _capi.TileForm()
    assert _capi.load().msa_linear_tiles(M, N, K, S, cus, ctypes.byref(f)) == 0
    return f


@pytest.mark.parametrize("M,N,K,S,want", [
    (64, 4096, 4096, 0, dict(kind=_capi.MSA_TILES_NONE, main=0)),
    (65, 768, 96, 0, dict(kind=_capi.MSA_TILES_SIMPLE, rows=128, columns=128)),
    (65, 768, 768, 0, dict(kind=_capi.MSA_TILES_WHOLE, columns=64, n_rows=1)),
    (200, 12288, 4096, 0, dict(kind=_capi.MSA_TILES_FEW, rows=128, columns=128, n_rows=2)),
    (66, 50272, 4096, 0, dict(kind=_capi.MSA_TILES_FEW, rows=128, columns=256)),
    (129, 50272, 4096, 0, dict(kind=_capi.MSA_TILES_FEW, rows=160, columns=256)),
    (193, 50272, 4096, 0, dict(kind=_capi.MSA_TILES_FEW, rows=224, columns=256)),
    (2005, 9216, 4096, 0, dict(kind=_capi.MSA_TILES_WHOLE, columns=256, pieces=4, main=2005)),
    (32800, 16384, 4096, 0, dict(kind=_capi.MSA_TILES_WHOLE, columns=256, pieces=1, main=32768)),
    (1607, 16384, 4096, 0, dict(kind=_capi.MSA_TILES_EVEN)),
    (2005, 4096, 16384, 2, dict(columns=256)),
    (200, 4096, 16384, 8, dict(kind=_capi.MSA_TILES_FEW, rows=256, columns=128)),
    (200, 4096, 4096, 4, dict(kind=_capi.MSA_TILES_FEW, rows=256, columns=64))])
def test_tiles_of_a_product(M, N, K, S, want):
    f = tiles(M, N, K, S)
    assert {k: getattr(f, k) for k in want} == want


def test_even_cuts_cover_the_rows():
    seen = set()
    for M in list(range(256, 2100, 7)) + [3000, 5555, 8200]:
        for N, K, S in ((4096, 4096, 0), (12288, 4096, 0), (16384, 4096, 0), (4096, 16384, 1), (2048, 8192, 2), (11392, 1984, 0)):
            f = tiles(M, N, K, S)
            if f.kind != _capi.MSA_TILES_EVEN:
                continue
            low = f.rows - 32
            rows = f.n_tall * f.rows + (f.n_rows - f.n_tall) * low
            last = f.rows if f.n_tall == f.n_rows else low
            assert rows - last < M <= rows and 0 <= f.n_tall <= f.n_rows and 160 <= f.rows <= 32 * (8 if f.columns == 256 else 7)
            assert f.main == M and f.pieces == 1
            seen.add((f.columns, f.rows))
    assert len(seen) > 4


@pytest.mark.parametrize("M,N,K,S,panels", [
    (516, 11392, 1984, 0, 1), (516, 11392, 1984, 1, 1), (1143, 2160, 1856, 0, 1), (669, 12480, 512, 0, 1),
    (1436, 3552, 448, 0, 0),       # columns in fours
    (600, 3424, 9600, 2, 1), (778, 1600, 14720, 2, 0), (1110, 3296, 8576, 2, 0),      # slices
    (640, 12288, 4096, 0, 0), (545, 16400, 704, 0, 1)])
def test_even_cuts_of_odd_columns_are_taken_in_panels(M, N, K, S, panels):
    f = tiles(M, N, K, S)
    assert (f.kind, f.panels) == (_capi.MSA_TILES_EVEN, panels), (f.kind, f.columns, f.n_rows)


def test_sizes_of_the_kernel_tests_reach_the_kernels_that_they_name():
    from tests import test_gpu_hybrid_kernels as H, test_gpu_kernels as C

    def of(M, N, K, S=0):
        f = tiles(M, N, K, S)
        return f.kind, f.columns, f.rows
    for M, N, K, pieces in C.PIECES:
        assert tiles(M, N, K).pieces == pieces, (M, N, K)
    for M, K, rows in C.FEW_ROWS:
        assert of(M, 50272, K) == (_capi.MSA_TILES_FEW, 256, rows), M
    for M, N, columns, rows, tall in C.EVEN_DEEP:
        assert of(M, N, 704) + (tiles(M, N, 704).n_tall,) == (_capi.MSA_TILES_EVEN, columns, rows, tall), (M, N)
    for M, N, K in C.EVEN_ODD:
        assert tiles(M, N, K).kind == _capi.MSA_TILES_EVEN and tiles(M, N, K).panels, (M, N, K)
    for M, N in C.PARTIALS_ODD:
        assert all(tiles(M, N, 1408, S).kind == _capi.MSA_TILES_EVEN and tiles(M, N, 1408, S).panels for S in (1, 2)), (M, N)
    for M, N, columns, rows in C.PARTIALS_DEEP:
        assert of(M, N, 1408, 2) == (_capi.MSA_TILES_EVEN, columns, rows), (M, N)
    for M, heads, columns, rows in C.QKV_DEEP:
        assert of(M, 384 * heads, 704) == (_capi.MSA_TILES_EVEN, columns, rows), (M, heads)
    for M, N, pieces in H.BF16_PIECES:
        assert tuple(tiles(M, N, 1408, S).pieces for S in (0, 1, 2)) == pieces, (M, N)
    for M, N, columns, rows in H.BF16_EVEN:
        assert of(M, N, 1408) == (_capi.MSA_TILES_EVEN, columns, rows), (M, N)
    assert {tiles(M, N, K).columns for M, N, K in C.QUEUE_ROWS} == {16, 32, 48, 64, 80}
    assert all(tiles(M, N, K).kind == _capi.MSA_TILES_QUEUE for M, N, K in C.QUEUE_ROWS)
    assert {tiles(*sizes).columns for sizes in C.QUEUE_SLICES} == {16, 32, 48, 64, 80}
    assert all(tiles(*sizes).kind == _capi.MSA_TILES_QUEUE for sizes in C.QUEUE_SLICES)
    for M, N, K in C.TILES_128:
        assert of(M, N, K) == (_capi.MSA_TILES_FEW, 128, 128), (M, N, K)
    assert {r[2:4] for r in C.EVEN_DEEP} == {(128, 160), (128, 192), (128, 224), (256, 160), (256, 192), (256, 224), (256, 256)}
    assert {r[2:4] for r in C.PARTIALS_DEEP} == {r[2:4] for r in C.EVEN_DEEP}


def test_tiles_refuses_what_the_products_refuse():
    lib, f = _capi.load(), _capi.TileForm()
    for bad in ((0, 64, 64, 0, 256), (4, 8, 64, 0, 256), (4, 64, 48, 0, 256), (300, 64, 256, 4, 256), (300, 64, 256, -1, 256)):
        assert lib.msa_linear_tiles(*bad, ctypes.byref(f)) == -1, bad
    assert lib.msa_linear_tiles(300, 64, 256, 0, 256, None) == -1
