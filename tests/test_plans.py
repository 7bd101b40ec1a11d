"""Which kernel form the launch plans choose, on the CPU: the plans' C++ functions (csrc/ns_internal.hpp) called in
the built library, with 256 CUs where there is no GPU.  For rules whose two sides give the same bits."""
import ctypes
import os
import re

import pytest

import nsffn as N

U32, SIZE = ctypes.c_uint32, ctypes.c_size_t


def tuning(**overrides):
    """struct Tuning with its defaults, read from the header."""
    text = open(os.path.join(N.PKG, "csrc", "ns_internal.hpp")).read()
    body = re.search(r"struct Tuning \{(.*?)\n\};", text, re.S).group(1)
    fields = {k: int(v) for k, v in re.findall(r"^\s*int (\w+) = (-?\d+);", body, re.M)}
    assert set(overrides) <= set(fields)
    fields.update(overrides)
    return (ctypes.c_int * len(fields))(*fields.values())


def function(mangled, restype):
    f = getattr(N.lib(), mangled)
    f.restype = restype
    return f


@pytest.mark.parametrize("rows,grid", [(131072, 0), (139264, 0), (163840, 0), (196608, 0), (212992, 416), (262144, 512),
                                       (278528, 0), (327680, 0), (360448, 470), (393216, 512)])
def test_stream_only_with_a_full_last_round(rows, grid):
    """The batch 2-4 kernel streams where its last round of 512 workgroups is more than half full (rows / 256 of them):
    163,840 rows of 3,840 columns, 1.25 rounds, took 1.15-1.2 times as long streamed."""
    f = function("_ZN2ns21gemv_mfma_stream_gridEjjRKNS_6TuningE", U32)
    assert f(U32(3840), U32(rows), tuning()) == grid


@pytest.mark.parametrize("cols,rows,batch,tile", [
    (4096, 163840, 138, 8), (4096, 30720, 1203, 8), (8192, 30720, 1548, 8), (3840, 30720, 1713, 8),
    (3840, 15360, 300, 4), (3840, 3840, 225, 4), (3840, 163840, 300, 4)])
def test_f16_tile_over_many_rounds(cols, rows, batch, tile):
    """The FP16-mode GEMM's tile: of 256 tokens (8) where that makes more than two rounds and 128-token tiles (4) only
    look cheaper by their rounds rounded up; 128-token ones where they fill a round better or pad less."""
    f = function("_ZN2ns13gemm_f16_costEjjjbRKNS_6TuningE", U32)
    cost = {mi: f(U32(cols), U32(rows), U32(batch), ctypes.c_bool(False), tuning(f16_mi=mi)) for mi in (0, 4, 8)}
    assert cost[4] != cost[8]
    assert cost[0] == cost[tile]


class Grid(ctypes.Structure):
    _fields_ = [("tiles", U32), ("kparts", U32), ("tokens", U32)]


@pytest.mark.parametrize("cols,rows,batch,pair,kparts", [
    (15360, 3840, 600, False, 6), (15360, 3840, 740, False, 5), (15360, 3840, 1300, False, 3), (3840, 15360, 300, True, 1),
    (15360, 3840, 512, False, 4), (3840, 15360, 64, True, 4), (3840, 4096, 1500, False, 2), (3840, 3840, 64, False, 4),
    (32768, 3776, 1652, True, 1)])
def test_q4k_parts_leave_no_empty_round(cols, rows, batch, pair, kparts):
    """Q4_K on CDNA4, FP32 mode: fewer K parts than the power of two (8, 8, 4, 2; 8, 4) where two workgroups per CU
    would make a nearly empty second round or share a CU for little; that power of two where it fits.  The pair may walk
    all of K in one chain."""
    f = function("_ZN2ns13gemm_reg_gridEjjjbRKNS_6TuningE", Grid)
    g = f(U32(cols), U32(rows), U32(batch), ctypes.c_bool(pair), tuning())
    assert (g.tokens, g.kparts) == (128, kparts)


@pytest.mark.parametrize("qtype,cols,rows,batch,pair,acc,kparts", [
    (N.Q4_K, 8192, 5120, 64, True, N.ACC_FP32, 4), (N.Q4_K, 8192, 11520, 64, False, N.ACC_FP16, 4),
    (N.Q4_K, 8192, 11520, 64, False, N.ACC_FP32, 8), (N.Q4_K, 2304, 49152, 5, False, N.ACC_FP16, 1),
    (N.Q4_K, 2304, 49152, 5, False, N.ACC_FP32, 2), (N.Q6_K, 32768, 1024, 55, False, N.ACC_FP16, 32),
    (N.Q6_K, 15360, 3840, 600, False, N.ACC_FP16, 5), (N.Q6_K, 15360, 3840, 600, False, N.ACC_FP32, 8)])
def test_lds_tile_parts(qtype, cols, rows, batch, pair, acc, kparts):
    """The LDS-tile GEMM: the pair and the FP16 mode (results rounded to fp16) take fewer K parts where the power of two
    would make a nearly empty second round; plain FP32-mode outputs keep it, as their error grows with the chains."""
    f = function("_ZN2ns9gemm_gridEijjjbiRKNS_6TuningE", Grid)
    g = f(qtype, U32(cols), U32(rows), U32(batch), ctypes.c_bool(pair), acc, tuning())
    assert (g.tokens, g.kparts) == (256, kparts)


@pytest.mark.parametrize("qtype,layout,cols,rows,batch,here", [
    (N.Q6_K, N.ROW_MAJOR, 2304, 21504, 3, True), (N.Q6_K, N.ROW_MAJOR, 15360, 21504, 2, True),
    (N.Q6_K, N.ROW_MAJOR, 1024, 32768, 4, True), (N.Q6_K, N.ROW_MAJOR, 1024, 2048, 4, False),
    (N.Q6_K, N.ROW_MAJOR, 512, 262144, 4, False), (N.Q6_K, N.ROW_MAJOR, 3840, 64, 3, False),
    (N.Q4_K, N.ROW_MAJOR, 3840, 21504, 3, True), (N.Q4_K, N.ROW_MAJOR, 256, 21504, 3, False)])
def test_small_batch_rule(qtype, layout, cols, rows, batch, here):
    """Batch 2-4 on row-major tensors: where the few-token GEMM takes a call from the small-batch kernel, which is 1.2 to
    1.8 times as fast or slow on these."""
    f = function("_ZN2ns18skinny_small_batchEiijjPKvjRKNS_6TuningE", ctypes.c_bool)
    assert f(qtype, layout, U32(cols), U32(rows), ctypes.c_void_p(4096), U32(batch), tuning()) is here


@pytest.mark.parametrize("rows,batch,here", [(32768, 5, True), (32768, 32, True), (32768, 33, False), (65536, 16, False)])
def test_one_super_block_pair(rows, batch, here):
    """The gate/up pair at 256 columns: up to two workgroups per CU run at once (10.8 us, the tile kernel 15.3)."""
    f = function("_ZN2ns20gemm_skinny_eligibleEiiijjjbRKNS_6TuningE", ctypes.c_bool)
    assert f(N.Q4_K, N.CDNA4, N.ACC_FP32, U32(256), U32(rows), U32(batch), ctypes.c_bool(True), tuning()) is here


def test_context_need_covers_every_batch():
    """A context is sized at multiples of 16 tokens: no batch between them needs more, on either kind of kernel."""
    tile = function("_ZN2ns24gemm_tile_workspace_needEiiijjjbRKNS_6TuningEPmS3_", None)
    skinny = function("_ZN2ns26gemm_skinny_workspace_needEijPKjijbiRKNS_6TuningEPmS5_", None)
    t, top = tuning(), {}
    for step in (1, 16):
        most = [0, 0]
        for qtype, cols, rows, pair in ((N.Q4_K, 3840, 15360, True), (N.Q4_K, 15360, 3840, False), (N.Q6_K, 15360, 3840, False)):
            for batch in range(16 if step == 16 else 5, 2049, step):
                for acc in (N.ACC_FP32, N.ACC_FP16):
                    f, c = SIZE(), SIZE()
                    for call in (lambda: tile(qtype, N.CDNA4, acc, U32(cols), U32(rows), U32(batch), ctypes.c_bool(pair), t,
                                              ctypes.byref(f), ctypes.byref(c)),
                                 lambda: skinny(qtype, U32(cols), (U32 * 1)(rows), 1, U32(batch), ctypes.c_bool(pair), acc, t,
                                                ctypes.byref(f), ctypes.byref(c))):
                        call()
                        most = [max(most[0], f.value), max(most[1], c.value)]
        top[step] = most
    assert top[1] == top[16]
