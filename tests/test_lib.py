"""The C-ABI library builds for gfx950, loads, and exports every entry point
include/quail_mi355x.h declares; argument errors are reported without
touching a GPU."""

import ctypes

import pytest

from quail_amd import _lib


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    declared = _lib.declared_symbols()
    assert len(declared) >= 14
    missing = [name for name in declared if not hasattr(lib, name)]
    assert not missing
    assert set(declared) == set(_lib.SIGNATURES)
    assert lib.qx_version() == _lib.ABI_VERSION == _lib.header_abi_version()


def test_direct_lds_loads_compile_without_a_warning(tmp_path):
    """The direct HBM -> LDS loads hand the compiler their M0 operand: named
    as a clobber instead, M0 is a reserved register the compiler does not
    keep track of across the statement, and it says so."""
    from quail_amd import build
    src = tmp_path / "loads.hip"
    src.write_text("""
#include "qx_common.h"
__global__ void loads(const uint8_t* a, float* out, int n) {
  __shared__ __attribute__((aligned(1024))) uint8_t buf[3][1024];
  for (int i = 0; i < n; ++i) {
    qx::lds_dma16(a + threadIdx.x * 16, buf[0]);
    qx::lds_dma16_stream(a + 1024 + threadIdx.x * 16, buf[1]);
    qx::lds_dma4(a + 2048 + threadIdx.x * 4, buf[2]);
    qx::wait_vmcnt<0>();
    qx::lds_barrier();
    out[i * 64 + threadIdx.x] = reinterpret_cast<const float*>(buf)[threadIdx.x * 3];
  }
}
""")
    assert build._compile(src, tmp_path / "loads.o") == ""


def test_argument_errors_return_minus_one_with_a_message():
    with pytest.raises(_lib.QxError, match="null pointer"):
        _lib.call("qx_gemm_fp8_blockscaled", None, None, None, None, None, 1, 256, 128, 128,
                  256, 1, 0, None)
    with pytest.raises(_lib.QxError, match="not a multiple of 128"):
        _lib.call("qx_gemm_fp8_blockscaled", 16, 16, 16, 16, 16, 1, 256, 100, 128, 256, 1, 0,
                  None)
    with pytest.raises(_lib.QxError, match="head_dim"):
        _lib.call("qx_paged_attention", 16, 8, 16, 16, 16, 16, 16, 1, 1, 1, 64, 4, 2, 96, 16,
                  0.1, 1, 16, None, 8, None, 0, None, 0, 0, 1, None)
    with pytest.raises(_lib.QxError, match="query rows per workgroup"):
        _lib.call("qx_paged_attention", 16, 8, 16, 16, 16, 16, 16, 1, 1, 1, 64, 4, 2, 64, 16,
                  0.1, 1, 16, None, 8, None, 0, None, 0, 32, 1, None)
    with pytest.raises(_lib.QxError, match="1..16"):
        _lib.call("qx_answer_head", 16, 8, 16, 8, 17, 1, 8, 0, None, 1.0, None, None, None,
                  None, None)


def test_attention_work_list_is_heaviest_first_and_covers_every_tile():
    import numpy as np
    # 3 sequences of 100, 1, 200 query rows over 150, 40, 260 keys (causal)
    cu_q = np.array([0, 100, 101, 301], dtype=np.int32)
    used = np.array([150, 40, 260], dtype=np.int32)
    work = np.zeros(2 * 16, dtype=np.int32)
    n = _lib.count("qx_paged_attention_work", cu_q.ctypes.data, used.ctypes.data, 3, 32, 8,
                   128, 1, 0, work.ctypes.data, 16)
    items = [tuple(work[2 * i:2 * i + 2]) for i in range(n)]
    # query tiles of 64 rows (G = 4): 2 + 1 + 4 of them
    assert sorted(items) == [(0, 0), (0, 1), (1, 0), (2, 0), (2, 1), (2, 2), (2, 3)]
    keys = {(0, 0): 114, (0, 1): 150, (1, 0): 40, (2, 0): 124, (2, 1): 188, (2, 2): 252,
            (2, 3): 260}
    loads = [keys[it] for it in items]
    assert loads == sorted(loads, reverse=True)
    with pytest.raises(_lib.QxError, match="capacity"):
        _lib.count("qx_paged_attention_work", cu_q.ctypes.data, used.ctypes.data, 3, 32, 8,
                   128, 1, 0, work.ctypes.data, 3)


def test_attention_tile_rows_choice_and_32_row_work_list():
    """qx_paged_attention_tile_rows picks 32 query rows per workgroup for
    packs whose 64-row items read few key tiles (at most 40 on average) and
    the default 64 otherwise; only D = 128 with 4 heads per workgroup offers
    32 (G = 2 keeps its default of 128). A 32-row work list covers every
    32-row tile that holds rows, heaviest first."""
    import numpy as np

    def rows(q_lens, used, hq=32, hk=8, d=128):
        cu_q = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
        used = np.asarray(used, dtype=np.int32)
        return _lib.count("qx_paged_attention_tile_rows", cu_q.ctypes.data, used.ctypes.data,
                          len(used), hq, hk, d, 1)

    # 512-token documents after a 64-token prefix: 5.5 key tiles per item
    assert rows([512] * 4, [576] * 4) == 32
    # 1024- to 4096-token documents: 9.5 to 33.5 key tiles per item, 32-row
    # workgroups measured up to 5% faster (1.00 at 4096); 8000: 63.5, 1-1.6% slower
    for n, want in ((1024, 32), (1536, 32), (2048, 32), (4096, 32), (8000, 64)):
        assert rows([n] * 4, [n + 64] * 4) == want, n
    assert rows([512] * 4, [576] * 4, d=64) == 64
    assert rows([512] * 4, [576] * 4, hq=16, hk=8) == 128
    cu_q = np.array([0, 100, 101, 301], dtype=np.int32)
    used = np.array([150, 40, 260], dtype=np.int32)
    work = np.zeros(2 * 32, dtype=np.int32)
    n = _lib.count("qx_paged_attention_work", cu_q.ctypes.data, used.ctypes.data, 3, 32, 8,
                   128, 1, 32, work.ctypes.data, 32)
    items = [tuple(work[2 * i:2 * i + 2]) for i in range(n)]
    assert sorted(items) == sorted([(0, t) for t in range(4)] + [(1, 0)] +
                                   [(2, t) for t in range(7)])
    keys = [min(u, u - ql + min(qt * 32 + 32, ql)) for s_, qt in items
            for u, ql in [(int(used[s_]), int(cu_q[s_ + 1] - cu_q[s_]))]]
    assert keys == sorted(keys, reverse=True)
    with pytest.raises(_lib.QxError, match="query rows per workgroup"):
        _lib.count("qx_paged_attention_work", cu_q.ctypes.data, used.ctypes.data, 3, 16, 8,
                   128, 1, 32, work.ctypes.data, 32)


def test_attention_tile_rows_for_half_empty_and_few_workgroups():
    """32 query rows per workgroup also for sequences that leave the second
    half of a 64-row workgroup empty (few rows over many keys) and for calls
    whose 64-row workgroups do not outnumber the 256 CUs; 64 where 64-row
    workgroups are full, long and many."""
    import numpy as np

    def rows(q_lens, used, causal=1):
        cu_q = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
        used = np.asarray(used, dtype=np.int32)
        return _lib.count("qx_paged_attention_tile_rows", cu_q.ctypes.data, used.ctypes.data,
                          len(used), 32, 8, 128, causal)

    assert rows([21] * 60, [921] * 60) == 32
    assert rows([21] * 60, [900] * 60, causal=0) == 32
    assert rows([48] * 240, [4096] * 240) == 64
    assert rows([2048], [8192]) == 32       # 32 items x 8 head groups = 256 workgroups
    assert rows([2112], [8192]) == 64
    assert rows([], []) == 64


def test_gemm_config_choice_by_shape(monkeypatch):
    """The arithmetic family is a function of N alone: widths that are a
    multiple of 256 or 320 take the promotion family (config 31's 256 x 320
    tiles where those take fewer full-wave units than 256 x 256 ones, or
    where N is not a multiple of 256; config 30 otherwise), the rest config
    11; the environment variable forces one."""
    from quail_amd.engine import GEMM_CONFIG_ENV, gemm_config
    monkeypatch.delenv(GEMM_CONFIG_ENV, raising=False)
    assert gemm_config(6144, 2560, 16294) == 30     # qkv of a Qwen3-4B pack
    assert gemm_config(6144, 2688, 16294) == 30     # 21 K-blocks
    assert gemm_config(6144, 2560, 256) == 30       # fewer tiles than CUs
    assert gemm_config(4096, 4096, 37) == 30        # Qwen3-8B o_proj, a few final rows
    assert gemm_config(2560, 4096, 16294) == 31     # 512 tiles of 256 x 320, not 640
    assert gemm_config(2560, 9728, 8192) == 31      # 256 tiles, not 320
    assert gemm_config(2560, 4096, 13056) == 30     # 510 tiles of 256 x 256: 2 waves
    assert gemm_config(2560, 4096, 2048) == 30      # 80 tiles: 64 wide ones cost more
    assert gemm_config(2560, 2688, 12000) == 30     # 470 tiles against 376 wide ones
    assert gemm_config(10240, 5120, 16294) == 30    # Qwen3-32B qkv: 10 waves either way
    assert gemm_config(5120, 8192, 16294) == 30     # Qwen3-32B o_proj: 5 waves either way
    assert gemm_config(2688, 2560, 16294) == 11
    assert gemm_config(640, 256, 100) == 31         # a multiple of 320 but not of 256
    monkeypatch.setenv(GEMM_CONFIG_ENV, "11")
    assert gemm_config(6144, 2560, 16294) == 11


def test_gemm_family_depends_on_width_only():
    """Rows never change arithmetic with the number of rows in the launch:
    for every width, all M choose configs of one family."""
    from quail_amd.engine import RESCALE_CONFIGS, gemm_config
    for n in (256, 512, 1280, 2560, 4096, 5120, 6144, 10240, 19456, 2688, 640):
        fams = {gemm_config(n, 2560, m) in RESCALE_CONFIGS
                for m in (1, 37, 255, 2048, 8192, 13056, 16294, 16384, 32768)}
        assert len(fams) == 1, n


def test_promotion_tiles_divide_the_width_and_stay_in_the_family(monkeypatch):
    """The tile the engine launches at any row count: one whose weights divide
    N, of the promotion family exactly where gemm_config is; small for few
    rows, config 30 or 31 for packs; the environment variable forces one."""
    from quail_amd import engine as e
    monkeypatch.delenv(e.GEMM_CONFIG_ENV, raising=False)
    monkeypatch.delenv(e.SWIGLU_CONFIG_ENV, raising=False)
    rows = (1, 15, 16, 17, 46, 97, 255, 333, 1003, 2048, 3600, 8192, 16294, 32768)
    for n in (256, 640, 1280, 1920, 2560, 4096, 5120, 6144, 10240, 2688):
        for k in (128, 2560, 9728, 25600):
            for m in rows:
                config = e.gemm_tiles(n, k, m)
                if e.gemm_config(n, k, m) == e.GEMM_ODD_WIDTH_CONFIG:
                    assert config == e.GEMM_ODD_WIDTH_CONFIG
                else:
                    assert n % e.PROMOTION_TILES[config][1] == 0
    for m in rows:
        assert e.swiglu_config(19456, 2560, m) in e.SWIGLU_TILES
    assert e.gemm_tiles(2560, 9728, 46) == 40
    assert e.gemm_tiles(2560, 9728, 16294) == 31
    assert e.gemm_tiles(6144, 2560, 16294) == 30
    assert e.swiglu_config(19456, 2560, 46) == 48
    monkeypatch.setenv(e.GEMM_CONFIG_ENV, "30")
    assert e.gemm_tiles(2560, 9728, 46) == 30


def test_tile_costs_rise_with_rows_and_narrow_models_keep_the_large_tile(monkeypatch):
    """A launch's predicted time is positive and never falls when rows are
    added, for every tile at every K; full packs run on 256-row tiles also
    where K is small (a round of the CUs is not free there)."""
    from quail_amd import engine as e
    for env in (e.SWIGLU_CONFIG_ENV, e.GEMM_CONFIG_ENV):
        monkeypatch.delenv(env, raising=False)
    for table in (e.PROMOTION_TILES, e.SWIGLU_TILES):
        for tile in table.values():
            for k in (128, 256, 384, 640, 2560, 25600):
                costs = [e._tile_cost(tile, 19456 if table is e.SWIGLU_TILES else 2560, k, m)
                         for m in (1, 64, 65, 257, 1003, 4096, 16384, 1 << 24)]
                assert costs[0] > 0 and costs == sorted(costs)
    for n in (2048, 19456, 51200):
        for k in (128, 256, 640, 2560):
            assert e.swiglu_config(n, k, 16384) == 30
            # no launch of millions of one-tile workgroups
            assert e.swiglu_launches(n, k, 1 << 24) == ((1 << 24, 30),)


def test_swiglu_config_choice_by_shape(monkeypatch):
    from quail_amd.engine import GEMM_CONFIG_ENV, SWIGLU_CONFIG_ENV, swiglu_config
    monkeypatch.delenv(GEMM_CONFIG_ENV, raising=False)
    monkeypatch.delenv(SWIGLU_CONFIG_ENV, raising=False)
    assert swiglu_config(19456, 2560, 16294) == 30
    assert swiglu_config(19456, 2560, 9000) == 30
    assert swiglu_config(19456, 2688, 16294) == 30   # 21 K-blocks
    monkeypatch.setenv(SWIGLU_CONFIG_ENV, "10")
    assert swiglu_config(19456, 2560, 16294) == 10


def test_forced_configs_are_read_from_the_environment_of_the_call(monkeypatch):
    """A forced config is seen wherever the program put it: os.environ set
    after the import, another mapping in os.environ's place, and that
    mapping's own changes; without it the choice is the table's."""
    import os

    from quail_amd import engine as e
    for env in (e.SWIGLU_CONFIG_ENV, e.GEMM_CONFIG_ENV):
        monkeypatch.delenv(env, raising=False)
    assert e.gemm_tiles(2560, 9728, 46) == 40
    monkeypatch.setenv(e.GEMM_CONFIG_ENV, "30")
    assert e.gemm_tiles(2560, 9728, 46) == e.gemm_config(2560, 9728, 46) == 30
    assert e.swiglu_launches(19456, 2560, 1003) == ((1003, 30),)
    mine = {e.GEMM_CONFIG_ENV: "42"}
    monkeypatch.setattr(os, "environ", mine)
    assert e.gemm_tiles(2560, 9728, 46) == e.gemm_config(2560, 9728, 46) == 42
    mine[e.SWIGLU_CONFIG_ENV] = "50"
    assert e.swiglu_config(19456, 2560, 46) == 50
    mine.clear()
    assert e.gemm_tiles(2560, 9728, 46) == 40


def test_stream_handle_where_torch_lacks_the_raw_one(monkeypatch):
    """The launch stream is torch's current one, also in a torch without the
    functions that give its handle alone."""
    import torch

    from quail_amd import engine as e
    stream = type("Stream", (), {"cuda_stream": 1234})()
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: stream)
    monkeypatch.setattr(e, "_raw_stream", None)
    assert e._stream() == 1234


def test_swiglu_launches_cover_the_rows(monkeypatch):
    """gate_up goes out as one launch or as the whole 256-row tiles and the
    rest: every row once, first rows first, the second launch only where a
    few rows past a multiple of 256 would cost another round of the CUs; a
    forced config is one launch."""
    from quail_amd import engine
    for env in (engine.SWIGLU_CONFIG_ENV, engine.GEMM_CONFIG_ENV):
        monkeypatch.delenv(env, raising=False)
    for n, k in ((19456, 2560), (24576, 4096), (51200, 5120), (256, 128)):
        for m in (1, 16, 255, 256, 257, 277, 512, 800, 1003, 1300, 4097, 16384):
            launches = engine.swiglu_launches(n, k, m)
            assert sum(rows for rows, _ in launches) == m
            assert len(launches) == 1 or (launches[0][0] % 256 == 0 and launches[0][1] == 30
                                          and 0 < launches[1][0] < 256)
            if len(launches) == 1:
                assert launches[0][1] == engine.swiglu_config(n, k, m)
    assert engine.swiglu_launches(51200, 5120, 277) == ((256, 30), (21, 48))
    assert engine.swiglu_launches(19456, 2560, 1003) == ((768, 30), (235, 49))
    assert len(engine.swiglu_launches(19456, 2560, 277)) == 1
    assert len(engine.swiglu_launches(19456, 2560, 16384)) == 1
    monkeypatch.setenv(engine.SWIGLU_CONFIG_ENV, "50")
    assert engine.swiglu_launches(51200, 5120, 277) == ((277, 50),)
