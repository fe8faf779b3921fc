"""Host side of the drop-in boundary, no GPU: launch law, kernarg packing against the reference's
committed manifest, manifest <-> code object validation with negative controls, layouts, and that
the C-ABI library exports every symbol include/saber_iu8.h declares."""
import ctypes
import json
import os
import re
import shutil
import struct
import subprocess

import numpy as np
import pytest

from oracle import ref
from saber_engine_amd import iu8, kbuild, synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GOLD = os.path.join(ROOT, "tests", "golden")


@pytest.fixture(scope="module", autouse=True)
def built():
    if not os.path.exists(iu8.LIB_PATH) or not os.path.exists(os.path.join(iu8.PREBUILT, "macaq_iu8.manifest.toml")):
        kbuild.build_all()


# ------------------------------------------------------------------ the C ABI surface

def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "saber_iu8.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    names = sorted(set(re.findall(r"\b(saber_iu8_[a-z0-9_]+)\s*\(", header)))
    assert len(names) >= 25
    lib = ctypes.CDLL(iu8.LIB_PATH)
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing
    assert lib.saber_iu8_abi_version() == 1


def test_descriptor_struct_layout_matches_the_header():
    # sizes the C side and the ctypes mirror must agree on (a drifted mirror corrupts launches)
    d = iu8.resolve(iu8.W4, 1, 5120, 5120)
    assert d.kernel == b"macaq_iu8_dec_w4_tm1" and d.op == b"gemm_i4a8" and d.plugin == b"macaq_iu8"
    assert d.n_args == 10 and d.kernarg_bytes == 68 and d.n_launches == 1 and d.shared_bytes == 0
    assert [d.args[i].name.decode() for i in range(10)] == ["a", "w", "as", "ws", "decode_partial", "decode_counter", "c", "m", "n", "k"]
    assert (d.arg("m").ival, d.arg("n").ival, d.arg("k").ival) == (1, 5120, 5120)


# ------------------------------------------------------------------ launch law

def test_resolve_refuses_by_name():
    for bad in [(0, 64, 128), (1, 0, 128), (1, 64, 0), (1, 40, 128), (1, 64, 192)]:
        with pytest.raises(iu8.IU8Error) as e:
            iu8.resolve(iu8.W4, *bad)
        assert e.value.code == iu8.E_RULE
    with pytest.raises(iu8.IU8Error):
        iu8.describe("macaq_iu8_dec_w4_tm1", 17, 64, 128)      # 17 rows do not fit one m-tile
    with pytest.raises(iu8.IU8Error):
        iu8.describe("macaq_iu8_pf_w4_tn4_lbk64", 256, 256, 256, ks=2)  # the prefill tile does not split
    with pytest.raises(iu8.IU8Error):
        iu8.describe("no_such_kernel", 1, 64, 128)


@pytest.mark.parametrize("wk,tag", [(iu8.W4, "w4"), (iu8.W8, "w8")])
def test_decode_band_routing(wk, tag):
    for m in (1, 4, 8, 16, 17, 32, 33, 48):
        d = iu8.resolve(wk, m, 5120, 5120)
        tm = (m + 15) // 16
        assert d.kernel.decode().startswith(f"macaq_iu8_dec_{tag}_tm{tm}")
        assert d.ks == 1 and d.grid[2] == 1 and d.n_workspaces == 0
        assert d.arg("decode_partial").kind == iu8.ARG_NULL_BUFFER and d.arg("decode_counter").kind == iu8.ARG_NULL_BUFFER
        assert d.grid[0] * (d.block[0] // 64) >= 5120 // 16 // 4       # the grid covers every 16-column tile
    # the tile GEMM's small cells take over from 49 rows, earlier on wide outputs; the streaming forms
    # stay reachable by name up to 64 rows
    for (m, n) in [(49, 5120), (64, 5120), (65, 5120), (33, 34816), (17, 34816)]:
        assert iu8.resolve(wk, m, n, 5120).kernel.decode().startswith(f"macaq_iu8_pf_{tag}"), (m, n)
    assert iu8.resolve(wk, 16, 34816, 5120).kernel.decode().startswith(f"macaq_iu8_dec_{tag}_tm1")
    assert iu8.describe(f"macaq_iu8_dec_{tag}_tm4", 64, 5120, 5120).grid[0] > 0


def test_activation_rows_are_staged_when_they_fit():
    assert iu8.resolve(iu8.W4, 1, 5120, 17408).kernel == b"macaq_iu8_dec_w4_tm1"        # 17 KiB
    assert iu8.resolve(iu8.W4, 4, 5120, 5120).kernel == b"macaq_iu8_dec_w4_tm1"         # 20 KiB
    assert iu8.resolve(iu8.W4, 8, 5120, 5120).kernel == b"macaq_iu8_dec_w4_tm1_a0"      # past 20 KiB: streamed
    assert iu8.resolve(iu8.W4, 8, 5120, 17408).kernel == b"macaq_iu8_dec_w4_tm1_a0"     # does not fit
    assert iu8.resolve(iu8.W4, 16, 5120, 17408).kernel == b"macaq_iu8_dec_w4_tm1_a0"
    assert iu8.resolve(iu8.W4, 3, 5120, 8704).kernel == b"macaq_iu8_dec_w4_tm1_a0"


def test_sixteen_row_tile_staged_once_a_workgroup_where_it_measured_faster():
    """`_s80`: the persistent GEMV that copies the 16-row tile (K <= 5120: 80 KiB) into LDS once a workgroup.
    W4 at 9-16 rows everywhere it holds; up to 8 rows, and int8 weights, from 64 MiB of weights (5 rows and more) or
    24,576 columns (any row count)."""
    for wk, m, n, k, s80 in ((iu8.W4, 16, 5120, 5120, True), (iu8.W4, 9, 96, 5120, True), (iu8.W4, 16, 16384, 4096, True),
                             (iu8.W4, 8, 5120, 5120, False), (iu8.W4, 8, 34816, 5120, True), (iu8.W4, 5, 28672, 4096, True),
                             (iu8.W4, 4, 34816, 5120, True), (iu8.W4, 1, 24576, 2048, True), (iu8.W8, 2, 34816, 5120, True),
                             (iu8.W4, 4, 16384, 5120, False), (iu8.W8, 3, 14336, 5120, False), (iu8.W4, 16, 5120, 5248, False), (iu8.W4, 17, 34816, 5120, False),
                             (iu8.W4, 4, 5120, 17408, True), (iu8.W4, 2, 5120, 17408, True), (iu8.W4, 1, 5120, 17408, False),
                             (iu8.W4, 4, 5120, 20608, False), (iu8.W4, 2, 256, 32768, True), (iu8.W8, 4, 5120, 17408, False),
                             (iu8.W8, 16, 7168, 5120, False), (iu8.W8, 16, 14336, 5120, True), (iu8.W8, 5, 34816, 5120, True),
                             (iu8.W8, 9, 24576, 2048, True)):
        d = iu8.resolve(wk, m, n, k)
        tag = "w8" if wk == iu8.W8 else "w4"
        # the whole-tile kernel while the 16-row tile fits (K <= 5120); the rows kernel (`_s80r`) for fewer rows of a longer K
        name = f"macaq_iu8_dec_{tag}_tm1_s80" + ("" if k <= 5120 else "r")
        assert (d.kernel.decode() == name) == s80 and d.kernel.decode().startswith(f"macaq_iu8_dec_{tag}_tm1_s80") == s80, (tag, m, n, k, d.kernel)
        if s80:
            blocks = -(-n // 32)
            assert d.block[0] == 1024 and d.ks == 1 and d.n_workspaces == 0
            assert d.grid[0] == (blocks if blocks <= 256 else -(-blocks // min(8, -(-blocks // 256))))
            assert bytes(d) == bytes(iu8.describe(name, m, n, k))
    assert iu8.describe("macaq_iu8_dec_w4_tm1_s80r", 8, 5120, 10240).grid[0] == 160       # by name: whatever fits 80 KiB
    assert iu8.describe("macaq_iu8_dec_w4_tm1_s80", 3, 5120, 5120).grid[0] == 160 and iu8.describe("macaq_iu8_dec_w8_tm1_s80r", 16, 64, 5120).grid[0] == 2
    for bad in (lambda: iu8.describe("macaq_iu8_dec_w4_tm1_s80", 17, 5120, 5120), lambda: iu8.describe("macaq_iu8_dec_w4_tm1_s80", 16, 5120, 5248),
                lambda: iu8.describe("macaq_iu8_dec_w4_tm1_s80", 4, 5120, 17408), lambda: iu8.describe("macaq_iu8_dec_w4_tm1_s80r", 17, 5120, 128),
                lambda: iu8.describe("macaq_iu8_dec_w4_tm1_s80r", 5, 5120, 10368), lambda: iu8.describe("macaq_iu8_dec_w4_tm1_s80r", 3, 5120, 20608),
                lambda: iu8.describe("macaq_iu8_dec_w4_tm1_s80", 16, 5120, 5120, ks=2)):
        with pytest.raises(iu8.IU8Error) as e:
            bad()
        assert e.value.code == iu8.E_RULE
    # a pair's halves stay the streamed geometry, whatever the law gives each alone
    a, b = iu8.resolve(iu8.W4, 16, 12288, 5120), iu8.resolve(iu8.W4, 16, 96, 5120)
    assert a.kernel == b.kernel == b"macaq_iu8_dec_w4_tm1_s80"
    d = iu8.pair(a, b)
    a0, b0 = iu8.describe("macaq_iu8_dec_w4_tm1_a0", 16, 12288, 5120), iu8.describe("macaq_iu8_dec_w4_tm1_a0", 16, 96, 5120)
    assert d.kernel == b"macaq_iu8f_pairb_w4_tm1_a0" and bytes(d) == bytes(iu8.pair(a0, b0))


def test_pair_lays_two_decode_grids_end_to_end():
    """macaq_iu8::pair (crates/saber-kernels/src/macaq_iu8.rs:632-704): each half keeps its own descriptor's
    split and workspaces; refusals by name."""
    a, b = iu8.resolve(iu8.W4, 4, 12288, 5120), iu8.resolve(iu8.W4, 4, 96, 5120)
    d = iu8.pair(a, b)
    # the law's block order is the reference's: the second ("ba") half's workgroups first at every tm
    # (PAIR_BA_FIRST, crates/saber-kernels/src/macaq_iu8.rs:549-553)
    assert d.kernel == b"macaq_iu8f_pairb_w4_tm1" and d.plugin == b"macaq_iu8f" and d.op == b"gemm_i4a8_pair"
    assert iu8.pair_ordered(a, b, False).kernel == b"macaq_iu8f_pair_w4_tm1"
    assert iu8.pair_ordered(a, b, True).kernel == b"macaq_iu8f_pairb_w4_tm1"
    assert bytes(iu8.pair_ordered(a, b, False).args) == bytes(d.args)          # one kernarg list for both orders
    assert tuple(d.grid) == (a.grid[0] + b.grid[0], 1, 1) and d.block[0] == a.block[0] and d.n_launches == 1
    vals = {n: d.arg(n).ival for n in ("m", "k", "n", "ks", "nb", "n_b", "ks_b", "nb_b")}
    assert vals == dict(m=4, k=5120, n=12288, ks=1, nb=a.grid[0], n_b=96, ks_b=1, nb_b=b.grid[0])
    for n in ("decode_partial", "decode_counter", "decode_partial_b", "decode_counter_b"):
        assert d.arg(n).kind == iu8.ARG_NULL_BUFFER
    assert d.n_workspaces == 0 and d.kernarg_bytes == 128
    # rows that stream from L2 pair on the streamed form
    assert iu8.pair(iu8.resolve(iu8.W4, 16, 5120, 5120), iu8.resolve(iu8.W4, 16, 64, 5120)).kernel == b"macaq_iu8f_pairb_w4_tm1_a0"
    assert iu8.pair(iu8.resolve(iu8.W4, 40, 5120, 5120), iu8.resolve(iu8.W4, 40, 64, 5120)).kernel == b"macaq_iu8f_pairb_w4_tm3"
    # explicit splits: the grids multiply, the second half's workspaces take the suffix
    a2, b2 = iu8.describe("macaq_iu8_dec_w4_tm1", 4, 256, 5120, ks=2), iu8.describe("macaq_iu8_dec_w4_tm1", 4, 64, 5120, ks=4)
    d2 = iu8.pair(a2, b2)
    assert d2.grid[0] == a2.grid[0] * 2 + b2.grid[0] * 4 and d2.n_workspaces == 4
    assert d2.workspace("decode_partial").bytes == 2 * 4 * 256 * 4 and d2.workspace("decode_partial_b").bytes == 4 * 4 * 64 * 4
    assert d2.workspace("decode_counter_b").kind == iu8.WS_PERSISTENT and d2.workspace("decode_counter_b").zero_once
    assert d2.arg("decode_partial_b").kind == iu8.ARG_BUFFER and d2.arg("ks_b").ival == 4
    for x, y in [(iu8.resolve(iu8.W4, 4, 256, 5120), iu8.resolve(iu8.W4, 4, 256, 17408)),      # another K
                 (iu8.resolve(iu8.W4, 4, 256, 5120), iu8.resolve(iu8.W4, 5, 256, 5120)),       # another M
                 (iu8.resolve(iu8.W4, 4, 256, 5120), iu8.resolve(iu8.W8, 4, 256, 5120)),       # an int8-row half
                 (iu8.resolve(iu8.W4, 100, 256, 5120), iu8.resolve(iu8.W4, 100, 256, 5120))]:  # prefill cells
        with pytest.raises(iu8.IU8Error) as e:
            iu8.pair(x, y)
        assert e.value.code == iu8.E_RULE and "pair" in str(e.value)


def test_pair_keeps_the_split_of_a_half_at_another_block_width():
    """A `_tm2_n1` / `_tm3_n2` half is paired in the streamed form of the pair kernels with the split count it was given:
    the descriptor is the one its `tm2` / `tm3` twin gives, grid and workspaces with it."""
    for m, wide, twin in ((32, "macaq_iu8_dec_w4_tm2_n1", "macaq_iu8_dec_w4_tm2"), (40, "macaq_iu8_dec_w4_tm3_n2", "macaq_iu8_dec_w4_tm3")):
        for ks_a, ks_b in ((1, 1), (3, 1), (1, 2), (3, 2)):
            for name_b in (wide, twin):
                d = iu8.pair(iu8.describe(wide, m, 4112, 4096, ks=ks_a), iu8.describe(name_b, m, 96, 4096, ks=ks_b))
                want = iu8.pair(iu8.describe(twin, m, 4112, 4096, ks=ks_a), iu8.describe(twin, m, 96, 4096, ks=ks_b))
                assert bytes(d) == bytes(want), (wide, name_b, ks_a, ks_b)
                assert d.arg("ks").ival == ks_a and d.arg("ks_b").ival == ks_b and d.n_workspaces == 2 * ((ks_a > 1) + (ks_b > 1))


def test_pair_variants_share_their_decode_twin_geometry():
    text = open(os.path.join(iu8.PKG, "csrc", "kernels", "iu8_variants.def")).read()
    dec = {m[0]: m[1:] for m in re.findall(r"^IU8_DEC_VARIANT\((\w+), (\d+), (\w+), (\d+), (\d+), (\d+), (\d+), (\d+), (\w+)\)", text, flags=re.M)}
    pairs = re.findall(r"^IU8_PAIR_VARIANT\((\w+), (\d+), (\d+), (\d+), (\d+), (\d+), (\d+), (\w+)\)", text, flags=re.M)
    assert len(pairs) == 10
    for name, tm, nt, kw, wpb, d, alds, bfirst in pairs:
        assert (bfirst == "true") == ("_pairb_" in name)
        twin = dec[name.replace("macaq_iu8f_pairb_", "macaq_iu8_dec_").replace("macaq_iu8f_pair_", "macaq_iu8_dec_")]
        assert twin == (tm, "false", nt, kw, wpb, d, alds, "false"), name


def test_reference_symbol_names_are_answered_by_the_law():
    """Names of the reference's fused object that encode gfx1201 tiles (macaq_iu8.rs:520-546) are
    requests for the op at the shape: the descriptor is the gfx950 law's; the all-reduce forms are
    refused by name."""
    for name, wk, shape in (("macaq_iu8f_dec_w4_tm5", iu8.W4, (80, 5120, 5120)), ("macaq_iu8f_pf_w4_bm128", iu8.W4, (400, 5120, 17408)),
                            ("macaq_iu8f_pf_w8_bm64", iu8.W8, (200, 5120, 5120)), ("macaq_iu8f_pf_w4_t3w8n4k128p", iu8.W4, (384, 34816, 5120)),
                            ("macaq_iu8f_pf_w8_t1w4n2k128", iu8.W8, (300, 5120, 6144))):
        d, law = iu8.describe(name, *shape), iu8.resolve(wk, *shape)
        assert bytes(d) == bytes(law) and d.kernel.decode().startswith("macaq_iu8_pf_"), name
    with pytest.raises(iu8.IU8Error) as e:
        iu8.describe("macaq_iu8f_arnq_hadi8_w4_tm1", 1, 5120, 5120)
    assert e.value.code == iu8.E_RULE and "all-reduce" in str(e.value)
    with pytest.raises(iu8.IU8Error):
        iu8.describe("macaq_iu8f_pf_w4_bm128", 400, 5120, 17408, ks=2)


def test_row_producer_forms_by_law():
    """The activation producers' form for a (rows, width): a wave a row for many narrow rows, 16 waves a row
    for rows wider than 4,096 whose count leaves the card part idle, else the narrowest 256-thread form."""
    for rows, width, quant, act in ((1, 5120, "t1024", "t1024"), (16, 17408, "t1024", "t1024"), (256, 8192, "t1024", "t1024"),
                                    (257, 8192, "t256_g2", "t1024"), (512, 5120, "t256_g2", "t1024"), (513, 5120, "t256_g2", "t256_g2"),
                                    (512, 12288, "t1024", "t1024"), (2048, 17408, "t256_g5", "t1024"), (2048, 12288, "t256_g5", "t1024"),
                                    (8, 4096, "t256_g1", "t256_g1"), (64, 2048, "w64", "w64"), (6, 2048, "t256_g1", "t256_g1"),
                                    (1, 32768, "t1024", "t1024"), (4096, 24576, "t256", "t1024")):
        q, a = iu8.resolve_quant(rows, width), iu8.resolve_silu_mul_quant(rows, width)
        assert q.kernel.decode() == "macaq_i8_quant_" + quant and a.kernel.decode() == "macaq_i8_silu_mul_quant_" + act, (rows, width)
        for d, form in ((q, quant), (a, act)):
            assert d.block[0] == (1024 if form == "t1024" else 256) and d.grid[0] == (rows // 4 if form == "w64" else rows)
    with pytest.raises(iu8.IU8Error):
        iu8.resolve_quant(4, 32832)


def test_gate_up_with_activation_descriptor():
    """saber_iu8_resolve_gate_up_act: the fused forms' grid over inter / 16 column blocks, 1,024 threads, the kernarg list
    (a, w, as, ws, gu, p, m, n, k) with n = the intermediate width; what does not fit is refused by name."""
    d = iu8.resolve_gate_up_act(16, 5120, 17408)
    assert d.kernel == b"macaq_iu8f_gateup_act_w4_s80" and d.plugin == b"macaq_iu8f" and d.op == b"linear_i4a8_gate_up_act"
    assert tuple(d.grid) == (218, 1, 1) and d.block[0] == 1024 and d.n_workspaces == 0 and d.kernarg_bytes == 60
    assert [d.args[i].name.decode() for i in range(d.n_args)] == ["a", "w", "as", "ws", "gu", "p", "m", "n", "k"]
    assert (d.arg("m").ival, d.arg("n").ival, d.arg("k").ival) == (16, 17408, 5120)
    assert iu8.resolve_gate_up_act(3, 17408, 256).grid[0] == 16 and iu8.gate_up_act_holds(4, 20480, 64)
    for m, h, i in ((17, 5120, 17408), (16, 5248, 17408), (5, 10368, 1024), (8, 5120, 17400), (0, 5120, 17408), (16, 5120, 16 * 2049)):
        assert not iu8.gate_up_act_holds(m, h, i), (m, h, i)
        with pytest.raises(iu8.IU8Error) as e:
            iu8.resolve_gate_up_act(m, h, i)
        assert e.value.code == iu8.E_RULE


def test_fused_quant_tile_gemm_descriptors():
    """macaq_iu8_pfq_*: the geometry of the cell the suffix names, the pf kernarg list with `x` for `a`."""
    d = iu8.describe("macaq_iu8_pfq_w4_t256x160", 2048, 5120, 17408)
    u = iu8.describe("macaq_iu8_pf_w4_t256x160", 2048, 5120, 17408)
    assert tuple(d.grid) == tuple(u.grid) and d.block[0] == u.block[0] == 512 and d.kernarg_bytes == 52 and d.op == b"linear_i4a8_pfq"
    assert [d.args[i].name.decode() for i in range(d.n_args)] == ["x", "w", "as", "ws", "c", "m", "n", "k"]
    assert iu8.resolve_prefill_fused(iu8.W4, 2048, 34816, 5120).kernel == b"macaq_iu8_pfq_w4_t256x160"
    assert iu8.resolve_prefill_fused(iu8.W8, 256, 5120, 5120).kernel == b"macaq_iu8_pfq_w8_t128x128"
    for bad in (lambda: iu8.describe("macaq_iu8_pfq_w4_t64x64_s", 256, 256, 256), lambda: iu8.describe("macaq_iu8_pfq_w4_t256x160", 256, 256, 256, ks=2),
                lambda: iu8.resolve_prefill_fused(iu8.W4, 0, 256, 256), lambda: iu8.describe("macaq_iu8_pfq_w4_t128x128", 500000, 128, 5120)):
        with pytest.raises(iu8.IU8Error) as e:
            bad()
        assert e.value.code == iu8.E_RULE


def test_band_table_is_the_launch_law():
    """prebuilt/gfx950/macaq_iu8.band.toml (the law as data, the gfx950 counterpart of the reference's
    PF_BAND / PF_TILES tables, macaq_iu8.rs:150-212) is what the library writes today, and every row
    re-derives from saber_iu8_resolve at both ends and the middle of its run."""
    import tomli

    text = open(iu8.BAND_TABLE).read()
    assert text == iu8.band_toml(), "stale band table: run python -m saber_engine_amd.kbuild"
    t = tomli.loads(text)
    assert t["arch"] == "gfx950" and t["cu_count"] == 256 and t["decode_split"] == 1
    cells = {c["kernel"]: c for c in t["cell"]}
    runs = {}
    for b in t["band"]:
        wk = iu8.W8 if b["w8"] else iu8.W4
        for m in sorted({b["first_m"], (b["first_m"] + b["last_m"]) // 2, b["last_m"]}):
            d = iu8.resolve(wk, m, b["n"], b["k"])
            assert d.kernel.decode() == b["kernel"] and d.ks == b["ks"] and d.block[0] == b["block"], (b, m)
        assert list(iu8.resolve(wk, b["first_m"], b["n"], b["k"]).grid) == b["grid_first"]
        assert list(iu8.resolve(wk, b["last_m"], b["n"], b["k"]).grid) == b["grid_last"]
        c = cells[b["kernel"]]
        assert c["threads"] == b["block"] and c["w8"] == b["w8"]
        if c["regime"] == "prefill" and b["ks"] == 1:     # the persistent grid law the cell row states
            tiles = -(-b["last_m"] // c["block_m"]) * -(-b["n"] // c["block_n"])
            assert b["grid_last"] == [min(tiles, 256 * c["workgroups_per_cu"]), 1, 1]
        runs.setdefault((b["op"], b["w8"]), []).append((b["first_m"], b["last_m"]))
    for key, rr in runs.items():       # the runs of a shape tile 1..band_last_m without gap or overlap
        rr.sort()
        assert rr[0][0] == 1 and rr[-1][1] == t["band_last_m"] and all(x[1] + 1 == y[0] for x, y in zip(rr, rr[1:])), key
    # the reference's whole symbol set is listed, with an answer each
    names = {r["name"]: r["answer"] for r in t["reference_symbol"]}
    assert len(names) == 45 and names["macaq_iu8_pf_w4_tn4_lbk64"].startswith("same name") and names["macaq_iu8f_arnq_hadi8_w4_tm1"] == "none"
    assert t["moe"]["tile_blocks_1_last_tokens"] == 112 and t["moe"]["tile_blocks_8_last_tokens"] == 2047
    assert t["moe"]["fused_back_last_tokens"] == 112 and t["moe"]["fused_back_inter_max"] == 1536
    assert iu8.moe_back_pays(16, 8, 128, 1, 1536) and iu8.moe_back_pays(112, 8, 128, 1, 1536)
    assert not iu8.moe_back_pays(16, 8, 128, 8, 1536) and not iu8.moe_back_holds(1, 1664)
    assert t["pair"]["second_first"] == [True] * 4
    # the fused decode linear's grid law and the chain's, as the tables state them
    f = t["fused_decode_linear"]
    for op, grid in f["grid"].items():
        n, k = next((b["n"], b["k"]) for b in t["band"] if b["op"] == op)
        d = iu8.resolve_fused(iu8.W4, 1, n, k)
        blocks = -(-n // f["column_block"])
        assert d.grid[0] == grid and d.block[0] == f["threads"] and grid * f["column_blocks_per_workgroup_max"] >= blocks
        assert grid == (blocks if blocks <= 256 else -(-blocks // min(8, -(-blocks // 256))))
    assert f["grid"]["gate_up"] == 218 and f["grid"]["down"] == 160
    c = t["mlp_chain"]
    d = iu8.resolve_mlp_chain(1, 5120, 17408)
    assert d.grid[0] == c["grid"]["hidden5120_inter17408"] <= 256 and d.block[0] == c["threads"]
    assert d.workspace("state").bytes == c["state_bytes"] == iu8.MLP_CHAIN_STATE_BYTES and d.arg("spin").ival == c["spin_default"]
    # where the chain measured faster than the three launches: one row of a wide intermediate, two of a wider one
    assert c["pays_one_row_inter_min"] == 12288 and c["pays_two_rows_inter_min"] == 13824
    for m, hid, inter, pays in ((1, 5120, 17408, True), (1, 4096, 12288, True), (1, 8192, 8192, False), (1, 5120, 5120, False),
                                (2, 5120, 17408, True), (2, 5120, 13824, True), (2, 4096, 12288, False), (3, 5120, 17408, False),
                                (4, 5120, 17408, False), (1, 5120, 24576, False), (5, 5120, 17408, False)):
        assert iu8.mlp_chain_pays(m, hid, inter) == pays, (m, hid, inter)
        assert not pays or iu8.mlp_chain_holds(m, hid, inter)
    rp = t["row_producers"]
    assert (rp["t1024_width_over"], rp["t1024_quant_rows_max"], rp["t1024_quant_rows_max_wide"], rp["t1024_silu_rows_max"], rp["t1024_wide"]) == (4096, 256, 512, 512, 12288)


def test_device_profile_is_the_planners_struct_as_data():
    """prebuilt/gfx950/device_profile.toml carries every field of the planner's DeviceProfile
    (crates/saber-plan/src/device.rs:168-193) in its serde shape, is what the library writes today, and
    agrees with the launch law's own constants; no bandwidth is given without its provenance."""
    import tomli

    text = open(iu8.DEVICE_PROFILE).read()
    assert text == iu8.device_profile_toml(), "stale device profile: run python -m saber_engine_amd.kbuild"
    p = tomli.loads(text)
    assert set(p) == {"gfx_target", "name", "cu_count", "wmma_shapes", "lds_bytes", "wave_sizes", "caps", "bandwidths",
                      "infinity_cache_bytes", "vram_bytes"}
    assert p["gfx_target"] == "gfx950" and p["wave_sizes"] == [64] and p["lds_bytes"] == 160 * 1024
    assert p["cu_count"] == tomli.loads(open(iu8.BAND_TABLE).read())["cu_count"] == 256
    assert set(p["caps"]) == {"fp8_wmma", "int8_wmma", "int4_wmma", "sparse_2_4_swmmac", "lds_dma", "nontemporal_loads", "lds_transpose_read"}
    assert p["caps"]["int8_wmma"] and p["caps"]["lds_dma"] and not p["caps"]["int4_wmma"]
    for w in p["wmma_shapes"]:
        assert set(w) == {"m", "n", "k", "a_dtype", "b_dtype", "acc_dtype", "sparse_2_4"}
    dense_i8 = {(w["m"], w["n"], w["k"]) for w in p["wmma_shapes"] if w["a_dtype"] == "iu8" and not w["sparse_2_4"]}
    assert dense_i8 == {(16, 16, 64), (32, 32, 32)}           # the two forms the decode and the tile GEMM are written on
    assert set(p["bandwidths"]) == {"dram", "pcie_h2d", "p2p"}
    dram = p["bandwidths"]["dram"]
    assert 5000 < dram["gbs"] < 8000 and set(dram["source"]["measured_here"]) == {"harness", "when"}
    assert p["bandwidths"]["pcie_h2d"]["source"] == "nominal" and p["bandwidths"]["p2p"]["source"] == "nominal"


def test_operands_past_4_gib_are_refused_by_the_tile_gemm():
    with pytest.raises(iu8.IU8Error) as e:
        iu8.resolve(iu8.W4, 300000, 5120, 17408)            # A: 300,000 x 17,408 bytes
    assert e.value.code == iu8.E_RULE and "4 GiB" in str(e.value)
    with pytest.raises(iu8.IU8Error):
        iu8.resolve(iu8.W8, 256, 262144, 16384)             # W8: 4 GiB of weights
    assert iu8.resolve(iu8.W4, 8192, 34816, 5120).ks == 1


def test_launch_law_shares_k_only_on_deep_narrow_tile_gemms():
    """The one band where the law splits the tile GEMM: K >= 16384, up to 192 rows and at most 128 tiles of the
    64x128 cell (two shares at least); the descriptor then names the `_ks` form, its z grid and both workspaces."""
    for wk, m, n, k, ks in ((iu8.W4, 64, 12288, 17408, 2), (iu8.W4, 128, 8192, 16384, 2), (iu8.W4, 160, 3072, 16384, 3)):
        d = iu8.resolve(wk, m, n, k)
        tiles = -(-m // 64) * (n // 128)
        assert d.kernel == b"macaq_iu8_pf_w4_t64x128_s_ks" and d.ks == ks and tuple(d.grid) == (tiles, 1, ks), (m, n, k)
    for m, ks, tiles in ((33, 4, 40), (48, 4, 40), (49, 4, 40), (64, 4, 40), (65, 3, 80), (128, 3, 80), (129, 2, 120), (192, 2, 120)):
        d = iu8.resolve(iu8.W4, m, 5120, 17408)
        assert d.kernel == b"macaq_iu8_pf_w4_t64x128_s_ks" and d.ks == ks and tuple(d.grid) == (tiles, 1, ks)
        assert d.workspace("decode_partial").bytes == ks * m * 5120 * 4 and d.workspace("decode_partial").kind == iu8.WS_SCRATCH
        c = d.workspace("decode_counter")
        assert c.bytes == tiles * 4 and c.kind == iu8.WS_PERSISTENT and c.zero_once
        assert iu8.gemm_workspace(iu8.W4, m, 5120, 17408) == (ks * m * 5120 * 4, tiles * 4)
    # up to 32 rows the streaming form keeps a deep narrow linear too (18.0 against 22.4 us)
    assert iu8.resolve(iu8.W4, 32, 5120, 17408).kernel == b"macaq_iu8_dec_w4_tm2"
    for wk, m, n, k in ((iu8.W4, 193, 5120, 17408), (iu8.W4, 64, 5120, 16256), (iu8.W4, 64, 16512, 17408), (iu8.W4, 129, 8192, 16384),
                        (iu8.W8, 64, 5120, 17408), (iu8.W4, 2048, 5120, 17408), (iu8.W4, 64, 5120, 5120),
                        (iu8.W4, 4096, 128, 17408), (iu8.W4, 4096, 16, 16384)):       # many rows of a narrow output: few tiles, no split
        d = iu8.resolve(wk, m, n, k)
        assert d.ks == 1 and d.n_workspaces == 0 and not d.kernel.endswith(b"_ks"), (m, n, k)
        assert iu8.gemm_workspace(wk, m, n, k) == (0, 0)


def test_moe_tile_law_thresholds():
    """16-row streaming tiles up to 7 routes an expert, 128-row MFMA tiles up to 96, 256-row above."""
    got = {t: iu8.moe_tile_blocks(t, 8, 128) for t in (1, 16, 112, 113, 256, 1536, 2047, 2048, 4096)}
    assert got == {1: 1, 16: 1, 112: 1, 113: 8, 256: 8, 1536: 8, 2047: 8, 2048: 16, 4096: 16}
    assert iu8.moe_tiles_cap(4096, 8, 128, 16) == 128 + 128 + 1 and iu8.moe_rows_cap(4096, 8, 128) == 32768 + 15 * 128


def test_explicit_split_declares_its_workspaces():
    d = iu8.describe("macaq_iu8_dec_w4_tm1", 4, 5120, 17408, ks=4)
    assert d.ks == 4 and d.grid[2] == 4
    p, c = d.workspace("decode_partial"), d.workspace("decode_counter")
    assert p.kind == iu8.WS_SCRATCH and p.bytes == 4 * 4 * 5120 * 4 and not p.zero_once
    assert c.kind == iu8.WS_PERSISTENT and c.bytes == d.grid[0] * 4 and c.zero_once
    assert d.arg("decode_partial").kind == iu8.ARG_BUFFER


PF_CELLS = {  # tile suffix -> (rows, columns, workgroups a CU, threads)
    "tn4_lbk64": (256, 256, 1, 512), "t256x224": (256, 224, 1, 512), "t256x160": (256, 160, 1, 512),
    "t128x128": (128, 128, 1, 512), "t128x128_o2": (128, 128, 2, 256), "t128x64_o2": (128, 64, 2, 256),
    "t128x64_s": (128, 64, 1, 256), "t64x128_s": (64, 128, 2, 256), "t64x64_s": (64, 64, 2, 256),
    "t256x320": (256, 320, 1, 512), "t128x320": (128, 320, 1, 512), "t128x256": (128, 256, 1, 512)}
PF_CELLS_W8 = dict(PF_CELLS, t128x320=(128, 320, 1, 256), t128x160=(128, 160, 1, 256))  # (one wave a wave tile)



def test_prefill_launch_is_persistent_and_covers_the_output():
    for wk, tag in ((iu8.W4, "w4"), (iu8.W8, "w8")):
        for (m, n, k) in [(256, 5120, 5120), (2048, 34816, 5120), (300, 304, 640), (8192, 7168, 5120), (65, 16, 128), (2048, 5120, 5120),
                          (777, 5120, 17408), (1024, 5120, 17408), (256, 34816, 5120)]:
            d = iu8.resolve(wk, m, n, k)
            name = d.kernel.decode()
            assert name.startswith(f"macaq_iu8_pf_{tag}_")
            bm, bn, occ, thr = (PF_CELLS_W8 if wk == iu8.W8 else PF_CELLS)[name[len(f"macaq_iu8_pf_{tag}_"):]]
            tiles = -(-n // bn) * -(-m // bm)
            # one workgroup (or two) a CU walks the tiles; the kernel derives the tile grid from m, n
            assert d.grid[0] == min(tiles, 256 * occ) and d.grid[1] == 1 and d.grid[2] == 1 and d.block[0] == thr
            assert d.n_workspaces == 0 and d.ks == 1


def test_every_tile_cell_has_its_threads():
    """By name, the threads a workgroup of every cell of the table, those with k-waves among them."""
    for tag, cells in (("w4", PF_CELLS), ("w8", {c: v for c, v in PF_CELLS_W8.items() if c != "t256x224"})):
        for cell, (bm, bn, occ, thr) in cells.items():
            d = iu8.describe(f"macaq_iu8_pf_{tag}_{cell}", 300, 5120, 2176)
            assert d.block[0] == thr and d.grid[0] == min(-(-300 // bm) * -(-5120 // bn), 256 * occ), (tag, cell)


def test_lines_of_the_launch_law_at_17_to_64_rows():
    """Either side of each line that `resolve` draws in rows, columns and K at 17 to 64 rows and for the 128 x 160 cell of
    int8 weights (the bytes of the cells named here: tests/test_gpu_dense.py)."""
    def picks(m, n, k):
        return tuple(iu8.resolve(wk, m, n, k).kernel.decode()[len("macaq_iu8_"):].replace(f"_{tag}_", "_") for wk, tag in ((iu8.W4, "w4"), (iu8.W8, "w8")))

    for (m, n, k), want in {
            # 17-32 rows: a 16-column block a CU, 32-column blocks, tiles
            (16, 4096, 6144): "dec_tm1_a0", (17, 4096, 128): "dec_tm2_n1", (32, 4096, 128): "dec_tm2_n1", (32, 4112, 128): "dec_tm2",
            (32, 16384, 5120): "dec_tm2", (32, 16400, 5120): ("pf_t64x128_s", "pf_t64x64_s"),
            # 33-48: 32-column blocks from K = 4,096, up to 8,192 columns
            (33, 4096, 6144): "dec_tm3", (33, 4112, 4096): "dec_tm3_n2", (33, 8192, 3968): "dec_tm3", (48, 8192, 4096): "dec_tm3_n2",
            (48, 8208, 4096): "pf_t64x64_s",
            # 49-64: streamed from K = 2,048 (up to 4,096 columns) and 6,144 (up to 8,192)
            (49, 4096, 1920): "pf_t64x64_s", (49, 4096, 2048): "dec_tm4_k16", (64, 4096, 2048): "dec_tm4_k16", (64, 4096, 6144): "dec_tm4_k16",
            (64, 4112, 6016): "pf_t64x64_s", (64, 4112, 6144): "dec_tm4_n2", (49, 8192, 6016): "pf_t64x64_s", (49, 8192, 6144): "dec_tm4_n2",
            (64, 8192, 6144): "dec_tm4_n2", (64, 8208, 6144): "pf_t64x64_s", (65, 4096, 2048): "pf_t64x64_s", (65, 8192, 6144): "pf_t64x64_s",
            # one row tile past the band: 64, 128 and 160 columns a CU
            (64, 16384, 640): "pf_t64x64_s", (64, 16400, 640): ("pf_t64x128_s", "pf_t64x64_s"), (32, 32768, 640): ("pf_t64x128_s", "pf_t64x64_s"),
            (32, 32784, 640): ("pf_t32x160_s", "pf_t64x160_s"), (33, 32784, 640): "pf_t64x160_s", (32, 40960, 640): ("pf_t32x160_s", "pf_t64x160_s"),
            (64, 40960, 640): "pf_t64x160_s", (17, 40976, 640): ("pf_t64x128_s", "pf_t64x64_s"), (64, 40976, 640): ("pf_t64x128_s", "pf_t64x64_s"),
            # K shared over workgroups leaves the streaming band to int8 weights
            (33, 4096, 16384): ("pf_t64x128_s_ks", "dec_tm3"), (33, 4096, 16256): "dec_tm3", (48, 8192, 16384): ("pf_t64x128_s_ks", "dec_tm3_n2")}.items():
        assert picks(m, n, k) == ((want, want) if isinstance(want, str) else want), (m, n, k)
    # 128 x 160: one round where 128 x 128 is two, 65 to 1,023 rows
    for m, n, takes in ((64, 40960, False), (65, 40960, True), (65, 40976, False), (65, 32784, True), (65, 32768, False), (128, 40960, True),
                        (129, 40960, False), (129, 20480, True), (129, 20496, False), (129, 16400, True), (129, 16384, False),
                        (1023, 5120, True), (1023, 5136, False), (1023, 4112, True), (1023, 4096, False), (1024, 5120, False)):
        assert (picks(m, n, 5120)[1] == "pf_t128x160") == takes, (m, n)


def test_int8_128x160_cell_only_where_it_measured_faster():
    """The 128 x 160 cell of int8 weights against the estimate's pick: not where a 64-row cell wastes less of a half live
    last row block on a short K, and not on a tile count that leaves the order by XCD at a K of 512 to 2,944."""
    mine = "macaq_iu8_pf_w8_t128x160"
    for m, n, k, takes in ((513, 7168, 128, False), (513, 7168, 2048, False), (385, 9216, 4096, False), (272, 12288, 1024, False),
                           (513, 7168, 4992, False), (513, 7168, 5120, True), (385, 8208, 5120, True), (129, 16400, 8192, True),
                           (784, 5760, 384, True), (784, 5760, 512, False), (784, 5760, 2944, False), (784, 5760, 3072, True),
                           (720, 5632, 1024, True), (777, 5120, 1024, True), (1000, 5120, 512, True), (200, 18432, 1024, True),
                           (200, 17408, 1024, False), (65, 32784, 1024, True), (128, 40960, 2048, True), (100, 34816, 512, True)):
        assert (iu8.resolve(iu8.W8, m, n, k).kernel.decode() == mine) == takes, (m, n, k)
        if not takes:   # what the estimate gives, not another of the law's rules
            assert iu8.resolve(iu8.W8, m, n, k).kernel.decode().startswith(("macaq_iu8_pf_w8_t64x", "macaq_iu8_pf_w8_t256x160")), (m, n, k)


def test_int8_cells_of_one_round_in_place_of_two_of_a_64_row_cell():
    """Int8 weights: 128 x 64 where it is one round and 64 x 64 is not, by K and by whole eighths; else 128 x 128 where that is one and
    64 x 128 is not. 256 rows and launches of no more 64 x 64 tiles than CUs stay with the estimate."""
    for m, n, k, tile in ((200, 5120, 5120, "t128x64_s"), (200, 5120, 2048, "t128x64_s"), (200, 5120, 1920, None), (256, 5120, 17408, None),
                          (257, 5120, 5120, "t128x64_s"), (160, 5120, 5120, None), (192, 5120, 5120, None), (193, 5120, 5120, "t128x64_s"),
                          (384, 5440, 5120, "t128x64_s"), (384, 5456, 5120, "t128x128"), (200, 5136, 4096, "t128x64_s"), (200, 5136, 3968, None),
                          (777, 2048, 17408, "t128x64_s"), (1500, 1152, 5120, "t128x64_s"), (65, 10240, 6144, "t128x64_s"),
                          (160, 16384, 5120, "t128x128"), (256, 16384, 4096, "t128x128"), (160, 16400, 5120, None), (129, 11008, 6144, "t128x128")):
        name = iu8.resolve(iu8.W8, m, n, k).kernel.decode()[len("macaq_iu8_pf_w8_"):]
        assert (name == tile) if tile else name not in ("t128x64_s", "t128x128"), (m, n, k, name)


def test_prefill_cells_of_the_benchmark_shapes():
    # speed data of this card: the cell that was fastest in the sustained sweep of each shape, weights cold (every cell on
    # the four 27B-class shapes x 14 row counts; the law's tables are fitted to those timings, one a weight kind)
    want = {(2048, 34816, 5120): "tn4_lbk64", (2048, 7168, 5120): "tn4_lbk64", (2048, 5120, 17408): "t128x320",
            (2048, 5120, 5120): "t128x320",
            (8192, 34816, 5120): "tn4_lbk64", (8192, 7168, 5120): "tn4_lbk64",
            # N = 5120 is 16 column blocks of 320: two even rounds of 256 x 320 tiles at 8,192 rows
            (8192, 5120, 17408): "t256x320", (8192, 5120, 5120): "t256x320", (4096, 5120, 17408): "t256x320",
            (512, 34816, 5120): "t256x320",
            # up to M of about 512 the launch is bound by what the CUs pull from L2: small tiles on every CU
            (256, 5120, 17408): "t64x128_s", (256, 7168, 5120): "t64x128_s", (256, 5120, 5120): "t64x128_s",
            (128, 5120, 17408): "t64x128_s_ks", (128, 5120, 5120): "t64x64_s",
            # 256 rows of the wide gate+up: 218 tiles of 256 x 160 (52.1 us against 55.6 on 128 x 320 and on 256 x 256)
            (256, 34816, 5120): "t256x160",
            # about a thousand rows of a narrow output: two 128 x 128 workgroups a CU (96.9 us against 117.6 on
            # 128 x 256 for down, 33.2 against 39.7 for O)
            (1024, 5120, 17408): "t128x128_o2", (1024, 5120, 5120): "t128x128_o2", (1024, 7168, 5120): "t128x128_o2",
            (512, 5120, 5120): "t128x128", (128, 34816, 5120): "t128x128_o2"}
    # shapes the fit had not seen: the served 27B graph's own projections (crates/saber-kernels/src/macaq_iu8.rs:931-947),
    # each pick the fastest cell of a cold sweep of all of them (65 / 128 rows of the wide ones: 16.5-18.8 us on 64 x 128
    # against 22.5-23.4 on 128 x 64, which the law chose before the side-by-side term came off the 64-row cells)
    want.update({(65, 16384, 5120): "t64x128_s", (128, 14336, 5120): "t64x128_s", (256, 16384, 5120): "t128x128",
                 (512, 14336, 5120): "t128x128_o2", (2048, 16384, 5120): "tn4_lbk64", (8192, 14336, 5120): "tn4_lbk64",
                 (128, 5120, 6144): "t64x64_s", (256, 5120, 6144): "t64x128_s", (1024, 5120, 6144): "t128x128_o2",
                 (2048, 5120, 6144): "t128x320", (4096, 5120, 6144): "t256x320", (2048, 96, 5120): "t64x64_s",
                 (8192, 96, 5120): "t64x64_s"})
    for (m, n, k), tile in want.items():
        assert iu8.resolve(iu8.W4, m, n, k).kernel.decode() == "macaq_iu8_pf_w4_" + tile, (m, n, k)
    # int8 weights rank the cells differently (twice the bytes a tile, no unpack): the output-side projections
    # of the mixed sequence at 2,048 rows take 256 x 160 (O 51.6 us against 72.6 on 128 x 320, down 158.6 against 224.2)
    # from 4,096 rows the 256 x 320 cell (N = 5120: 16 column blocks, even rounds): O 91.2 us against 104.5 on 256 x 256 at
    # 4,096 rows, down 278.5 against 313.0; at 8,192 rows 176.1 against 190.6 and 560.3 against 635.0; QKV stays (174.8 against 147.9)
    want8 = {(2048, 5120, 5120): "t256x160", (2048, 5120, 17408): "t256x160", (8192, 5120, 17408): "t256x320",
             (8192, 5120, 5120): "t256x320", (4096, 5120, 5120): "t256x320", (4096, 5120, 17408): "t256x320",
             (4096, 7168, 5120): "tn4_lbk64", (8192, 7168, 5120): "tn4_lbk64", (1024, 5120, 17408): "t128x256",
             (512, 5120, 17408): "t128x128", (256, 5120, 5120): "t64x128_s", (128, 5120, 17408): "t64x64_s"}
    for (m, n, k), tile in want8.items():
        assert iu8.resolve(iu8.W8, m, n, k).kernel.decode() == "macaq_iu8_pf_w8_" + tile, (m, n, k)
    with pytest.raises(iu8.IU8Error):
        iu8.describe("macaq_iu8_pf_w4_tn4_lbk64", 256, 5120, 5120, ks=2)   # the prefill tile does not split K


def test_int4_tile_cells_that_a_refit_had_slowed():
    """Shapes, most of a short K, that rates drawn from long ones gave slower cells than the ones before them (us there / on the pick
    here): the launch law is back on the earlier cell, or on one at least as fast."""
    for m, n, k, tile in ((611, 14368, 768, "tn4_lbk64"), (1397, 6784, 640, "tn4_lbk64"),      # 20.2 / 16.0, 17.0 / 14.6
                          (125, 288, 128, "t64x64_s"), (192, 4032, 256, "t64x64_s"),           # 3.6 / 3.2, 4.2 / 3.8
                          (420, 7856, 128, "t128x128"), (66, 30864, 512, "t128x128"), (191, 14080, 384, "t128x128"),  # 5.8 / 5.1, 7.9 / 6.7, 7.1 / 6.3
                          (802, 18368, 256, "t128x128_o2"), (573, 14192, 256, "t64x128_s"),    # 15.7 / 12.7, 12.0 / 9.7
                          (217, 25984, 2304, "t128x128_o2"), (149, 23440, 10368, "t128x256"),  # 26.5 / 21.6, 78.2 / 61.6
                          (777, 5120, 17408, "t128x256"), (200, 34816, 5120, "t256x160")):     # 96.0 / 92.4; as before
        assert iu8.resolve(iu8.W4, m, n, k).kernel.decode() == "macaq_iu8_pf_w4_" + tile, (m, n, k)


def test_256x224_cell_is_reached_by_name_only():
    """The estimate does not hold the 256 x 224 cell, which lost to 256 x 256 wherever it was picked, last at a K past 24,000."""
    for m, n, k in ((718, 13712, 27520), (2270, 4832, 24448), (8221, 1184, 25344), (1317, 16496, 26112), (786, 3632, 29056), (2404, 6032, 29568)):
        assert iu8.resolve(iu8.W4, m, n, k).kernel != b"macaq_iu8_pf_w4_t256x224", (m, n, k)
    d = iu8.describe("macaq_iu8_pf_w4_t256x224", 718, 13712, 27520)
    assert d.block[0] == 512 and d.grid[0] == 186


# ------------------------------------------------------------------ kernarg ABI

def test_signatures_pack_exactly_like_the_reference_manifest():
    table = json.load(open(os.path.join(GOLD, "kernarg_gfx1201.json")))
    checked = 0
    for name, args in table.items():
        slots, nbytes = iu8.signature(name)
        assert [(s[0], s[1], s[2]) for s in slots] == [(a["name"], a["offset"], a["size"]) for a in args], name
        assert [("global_buffer" if s[3] == iu8.ARG_BUFFER else "by_value") for s in slots] == [a["value_kind"] for a in args]
        assert nbytes == max(a["offset"] + a["size"] for a in args)
        checked += 1
    assert checked == 24


def test_routed_layer_signatures_keep_the_reference_lists():
    """The router, the grouped GEMM, the SiLU*up requant and the combine pack their kernargs as the
    reference's kernels of the same role do (prebuilt/gfx1201/moe_route.manifest.toml,
    moe_grouped.manifest.toml): names, offsets, sizes, value kinds."""
    table = json.load(open(os.path.join(GOLD, "kernarg_gfx1201_moe.json")))
    checked = 0
    for ref_name, row in table.items():
        for ours in row["gfx950"]:
            slots, nbytes = iu8.signature(ours)
            assert [(s[0], s[1], s[2]) for s in slots] == [(a["name"], a["offset"], a["size"]) for a in row["args"]], (ref_name, ours)
            assert [("global_buffer" if s[3] == iu8.ARG_BUFFER else "by_value") for s in slots] == [a["value_kind"] for a in row["args"]]
            assert nbytes == max(a["offset"] + a["size"] for a in row["args"])
            checked += 1
    assert checked == 17 and len(table) == 9
    text = open(os.path.join(iu8.PREBUILT, "moe_iu8.manifest.toml")).read() + open(os.path.join(iu8.PREBUILT, "macaq_i8q.manifest.toml")).read()
    for row in table.values():
        for ours in row["gfx950"]:
            assert f'name = "{ours}"' in text, ours


def test_kernarg_image_built_two_ways_is_byte_identical():
    d = iu8.describe("macaq_iu8_dec_w4_tm1", 3, 5120, 17408, ks=2)
    bufs = dict(a=0x7F0000001000, w=0x7F0000002000, ws=0x7F0000004000, decode_partial=0x7F0000005000,
                decode_counter=0x7F0000006000, c=0x7F0000007000)
    bufs["as"] = 0x7F0000003000
    img = iu8.pack_kernarg(d, bufs)
    want = struct.pack("<7Q3i", bufs["a"], bufs["w"], bufs["as"], bufs["ws"], bufs["decode_partial"], bufs["decode_counter"],
                       bufs["c"], 3, 5120, 17408)
    assert img == want and len(img) == 68
    # ks == 1: the workspace pointers are written as NULL whatever is bound
    d1 = iu8.resolve(iu8.W4, 3, 5120, 17408)
    img1 = iu8.pack_kernarg(d1, bufs)
    assert img1[32:48] == b"\0" * 16 and img1[:32] == want[:32]
    # a missing or NULL binding is refused, not packed
    del bufs["ws"]
    with pytest.raises(iu8.IU8Error) as e:
        iu8.pack_kernarg(d, bufs)
    assert e.value.code == iu8.E_ARG
    bufs["ws"] = 0
    with pytest.raises(iu8.IU8Error):
        iu8.pack_kernarg(d, bufs)


# ------------------------------------------------------------------ manifests and code objects

def _copy_plugin(tmp_path, stem="macaq_iu8"):
    for ext in (".hsaco", ".manifest.toml"):
        shutil.copy(os.path.join(iu8.PREBUILT, stem + ext), tmp_path / (stem + ext))
    return str(tmp_path / (stem + ".manifest.toml"))


def test_every_built_manifest_validates_against_its_code_object():
    ms = [f for f in os.listdir(iu8.PREBUILT) if f.endswith(".manifest.toml")]
    assert {"macaq_iu8.manifest.toml", "macaq_i8q.manifest.toml"} <= set(ms)
    for f in ms:
        rc, refusal, msg = iu8.manifest_validate(os.path.join(iu8.PREBUILT, f))
        assert rc == 0 and refusal == 0, msg
        text = open(os.path.join(iu8.PREBUILT, f)).read()
        assert 'arch = "gfx950"' in text and "wavefront_size = 64" in text and "wavefront_size = 32" not in text
        assert "private_segment_fixed_size = 0" in text


def test_reference_symbols_and_lds_budget():
    stems = ("macaq_iu8", "macaq_iu8f", "mxfp4_hadi8", "attn_glue_hadi8")
    text = "".join(open(os.path.join(iu8.PREBUILT, f"{s}.manifest.toml")).read() for s in stems)
    for name in json.load(open(os.path.join(GOLD, "kernarg_gfx1201.json"))):
        assert f'name = "{name}"' in text and f'symbol = "{name}.kd"' in text
    assert max(int(v) for v in re.findall(r"group_segment_fixed_size = (\d+)", text)) <= 160 * 1024
    # no kernel of the shipped objects spills to scratch -- but for one dword that the int8-weight 256 x 320 cell
    # parks across a tile's K loop (stored in front of the loop, read behind it)
    spills = {n: int(b) for n, b in re.findall(r'name = "(\w+)"(?:(?!\[\[kernel\]\]).)*?private_segment_fixed_size = (\d+)', text, flags=re.S) if int(b)}
    assert spills == {"macaq_iu8_pf_w8_t256x320": 8}, spills


@pytest.mark.parametrize("edit,counter", [
    (("offset = 56", "offset = 60", 1), iu8.REFUSED_KERNARG),                  # a drifted kernarg offset
    (("wavefront_size = 64", "wavefront_size = 32", 1), iu8.REFUSED_WAVE),       # mixed wave sizes in one plugin
    (("group_segment_fixed_size = ", "group_segment_fixed_size = 1", 1), iu8.REFUSED_METADATA),  # LDS drift
    (("hsaco_sha256 = \"", "hsaco_sha256 = \"0", 1), iu8.REFUSED_METADATA),       # another build's blob
    (("arch = \"gfx950\"", "arch = \"gfx1201\"", 1), iu8.REFUSED_METADATA),
])
def test_drifted_manifest_is_refused_with_the_right_counter(tmp_path, edit, counter):
    path = _copy_plugin(tmp_path)
    text = open(path).read()
    assert edit[0] in text
    open(path, "w").write(text.replace(edit[0], edit[1], edit[2]))
    rc, refusal, msg = iu8.manifest_validate(path, arch="gfx950")
    assert rc == iu8.E_VALIDATE and refusal == counter, (rc, refusal, msg)


def test_tampered_code_object_is_refused(tmp_path):
    path = _copy_plugin(tmp_path)
    blob = bytearray(open(tmp_path / "macaq_iu8.hsaco", "rb").read())
    blob[len(blob) // 2] ^= 0xFF
    open(tmp_path / "macaq_iu8.hsaco", "wb").write(bytes(blob))
    rc, refusal, _ = iu8.manifest_validate(path)
    assert rc in (iu8.E_VALIDATE, iu8.E_PARSE)


def _elf_with_note(desc, sh_offset=None, sh_size=None):
    """A minimal little-endian ELF64 for EM_AMDGPU whose only real section is one metadata note."""
    note = struct.pack("<III", 7, len(desc), 32) + b"AMDGPU\0\0" + desc + b"\0" * (-len(desc) % 4)
    off = 64
    shoff = off + len(note)
    hdr = bytearray(64)
    hdr[0:6] = b"\x7fELF\x02\x01"
    struct.pack_into("<HH", hdr, 16, 3, 224)
    struct.pack_into("<Q", hdr, 40, shoff)
    struct.pack_into("<HHHHHH", hdr, 52, 64, 0, 0, 64, 2, 0)
    sh = bytearray(128)
    struct.pack_into("<I", sh, 64 + 4, 7)
    struct.pack_into("<QQ", sh, 64 + 24, off if sh_offset is None else sh_offset, len(note) if sh_size is None else sh_size)
    return bytes(hdr) + note + bytes(sh)


@pytest.mark.parametrize("what,blob", [
    ("a note nested 200,000 arrays deep", _elf_with_note(b"\x91" * 200000 + b"\xc0")),
    ("a note nested 200,000 maps deep", _elf_with_note(b"\x81\xa1k" * 200000 + b"\xc0")),
    ("a note section whose offset + size wraps 64 bits", _elf_with_note(b"\x80", sh_offset=2**64 - 8, sh_size=64)),
    ("a section table whose end wraps 64 bits", _elf_with_note(b"\x80")[:40] + struct.pack("<Q", 2**64 - 64) + _elf_with_note(b"\x80")[48:]),
])
def test_crafted_code_objects_are_parse_errors_not_crashes(tmp_path, what, blob):
    """The code-object reader's bounds: a msgpack note that nests without end is refused at a fixed depth
    (it must not recurse down the stack), and section ranges that wrap around 2^64 are not ranges."""
    path = tmp_path / "crafted.hsaco"
    path.write_bytes(blob)
    rc = iu8.lib().saber_iu8_manifest_write(str(path).encode(), b"crafted", b"gfx950", b"crafted.hip", b"0" * 64, b"", b"0" * 64,
                                           str(tmp_path / "crafted.manifest.toml").encode())
    assert rc == iu8.E_PARSE, (what, rc, iu8.lib().saber_iu8_last_error().decode())
    assert not (tmp_path / "crafted.manifest.toml").exists()


def test_schema_version_and_garbage_are_parse_errors(tmp_path):
    path = _copy_plugin(tmp_path)
    text = open(path).read()
    open(path, "w").write(text.replace("schema_version = 1", "schema_version = 2"))
    assert iu8.manifest_validate(path)[0] == iu8.E_PARSE
    open(path, "w").write("this is not a manifest")
    assert iu8.manifest_validate(path)[0] == iu8.E_PARSE
    assert iu8.manifest_validate(str(tmp_path / "absent.manifest.toml"))[0] == iu8.E_IO


def test_source_ladder():
    assert kbuild.candidates("macaq_iu8", "gfx950") == ["macaq_iu8.gfx950.hip", "macaq_iu8.gfx95.hip", "macaq_iu8.hip"]
    assert kbuild.candidates("k", "gfx1201") == ["k.gfx1201.hip", "k.gfx12.hip", "k.hip"]
    assert kbuild.resolve_source("macaq_iu8").endswith("macaq_iu8.gfx950.hip")
    assert kbuild.resolve_source("no_such_kernel") is None


def test_open_without_a_gpu_fails_loudly():
    import torch

    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    with pytest.raises(iu8.IU8Error) as e:
        iu8.Context()
    assert e.value.code == iu8.E_HIP and "no CPU fallback" in str(e.value)


@pytest.fixture(params=["fastcall", "ctypes"])
def op(request):
    """The operators' entry points: the extension's (where this interpreter has it) and those of an interpreter without it."""
    if request.param == "ctypes":
        return iu8._CtypesOperators()
    o = iu8.operators()
    if isinstance(o, iu8._CtypesOperators):
        pytest.skip("_fastcall is not built for this interpreter")
    return o


def test_operator_entry_points_take_what_ctypes_takes(op):
    """The binding's own entry points (csrc/python/fastcall.cpp): ints and None as they are, everything else -- ctypes objects,
    other integer types, a wrong type or count -- as the ctypes function has it. Without a context every call is refused by
    the library itself, before anything is launched."""
    L = iu8.lib()
    args = (0, 1 << 40, 1 << 40, 1 << 40, 1 << 40, None, None, 1, 5120, 5120)
    for a in ((None,) + args + (0,), (None,) + args + (None,), (ctypes.c_void_p(),) + args + (ctypes.c_void_p(0),), (None, True) + args[1:] + (0,),
              (None,) + args[:-1] + (np.int64(5120), 0), (None,) + args[:-1] + ((1 << 32) + 5120, 0), (None, 7) + args[1:] + (0,),
              (None,) + args[:-1] + (5121, 0)):
        assert op.linear_fused(*a) == L.saber_iu8_linear_fused(*a) != 0, a
    assert op.linear_fused(None, 0, -1, 1, 1, 1, None, None, 1, 5120, 5121, 0) == iu8.E_RULE and "5121" in L.saber_iu8_last_error().decode()
    assert op.add_rms_quant_had(None, 1, 1, 1, 1, 1, 1, 4, 5120, 1e-6, 1, 0) == iu8.E_ARG
    assert op.add_rms_quant_had(None, 1, 1, 1, 1, 1, 1, 4, 5120, 1, 1, 0) == iu8.E_ARG      # an int for a float: ctypes takes it
    for bad in ((None,) + args[:-1] + (1.5, 0), (None,) + args[:-1] + ("5120", 0), (None,) + args):
        with pytest.raises((ctypes.ArgumentError, TypeError)):
            op.linear_fused(*bad)
        with pytest.raises((ctypes.ArgumentError, TypeError)):
            L.saber_iu8_linear_fused(*bad)


def test_sizes_at_the_end_of_32_bits_are_refused_not_divided_by():
    """Row and column counts whose tile counts used to wrap to none: refused with a message, and no descriptor without a workgroup."""
    top = 1 << 32
    sizes = [(top - 1, 5120, 128), (top - 15, 16, 128), (top - 16, 5120, 5120), (top - 63, 16, 128), (top - 255, 256, 16384), (1 << 31, 5120, 5120),
             (100, top - 16, 128), (17, top - 128, 16384), (192, top - 16, 16384), (1, top - 16, 16384), (16, top - 32, 5120), (2048, top - 256, 128),
             (top - 1, top - 16, top - 128), (40, top - 48, 4096), (64, top - 16, 6144), (1 << 27, 16, 128)]
    names = [f"macaq_iu8_pf_{t}" for t in ("w4_tn4_lbk64", "w8_tn4_lbk64", "w4_t256x160", "w4_t128x320", "w4_t64x64_s", "w8_t128x160", "w4_t64x128_s_ks")]
    names += ["macaq_iu8_pfq_w4_t128x128", "macaq_iu8_dec_w4_tm1", "macaq_iu8_pf_w4_t48x144_w"]
    calls = [lambda m, n, k, wk=wk, f=f: f(wk, m, n, k) for wk in (iu8.W4, iu8.W8) for f in (iu8.resolve, iu8.resolve_fused, iu8.resolve_prefill_fused)]
    calls += [lambda m, n, k, name=name: iu8.describe(name, m, n, k) for name in names]
    calls += [lambda m, n, k: iu8.resolve_gate_up_act(m, k, n), lambda m, n, k: iu8.resolve_mlp_chain(m, k, n), lambda m, n, k: iu8.resolve_quant(m, k)]
    for m, n, k in sizes:
        for f in calls:
            try:
                d = f(m, n, k)
            except iu8.IU8Error as e:
                assert e.code == iu8.E_RULE and str(e)
            else:
                assert d.grid[0] and d.grid[1] and d.grid[2], (m, n, k, d.kernel)
    for m, n, k in ((top - 1, 5120, 128), (1, 1 << 31, 128), (1, 16, 1 << 31)):
        with pytest.raises(iu8.IU8Error, match="32-bit sizes"):
            iu8.resolve(iu8.W4, m, n, k)
    assert iu8.resolve(iu8.W4, 1, (1 << 31) - 16, 128).grid[0]


OPERATORS = ("quant quant_rowmajor gemm rowscale linear_prefill_fused gemm_static gemm_pair linear_fused mlp_chain gate_up_act quant_had "
             "silu_mul_quant_had silu_mul_quant_had_lut add_rms_quant_had gdn_norm_quant_had attn_gate_quant_had attn_gate_quant_had_lut "
             "moe_route moe_route_quant moe_grouped moe_quant_rows moe_silu_mul_quant moe_gate_up_act moe_down_rows moe_combine").split()


class OtherTables(iu8.MoeTables):
    pass


@pytest.mark.parametrize("name", OPERATORS)
def test_every_operator_takes_the_forms_ctypes_takes(op, name):
    """Every operator, every argument in turn in every form a caller may have it in (the routed ones' tables among them): the
    ctypes function's result, message or exception. Without a context: the library refuses each call before a launch."""
    f, g, T = getattr(op, name), getattr(iu8.lib(), "saber_iu8_" + name), iu8.MoeTables()
    base, forms = [], []
    for t in g.argtypes:
        if t is ctypes.c_void_p:
            base.append(1 << 40 if base else None)
            forms.append([None] if len(base) == 1 else [None, 0, -1, 1 << 63, ctypes.c_void_p(0), ctypes.c_void_p(64), ctypes.byref(T), b"x", True, np.int64(64), 1.5])
        elif t is ctypes.c_float:
            base.append(1e-6)
            forms.append([1, ctypes.c_float(2.0), np.float32(3.0), np.float64(3.0), True, None, "1"])
        elif t is ctypes.POINTER(iu8.MoeTables):
            base.append(T)
            forms.append([ctypes.byref(T), ctypes.pointer(T), (iu8.MoeTables * 1)(), OtherTables(), None, ctypes.addressof(T), ctypes.byref(iu8.Counters()),
                          iu8.Counters(), ctypes.c_void_p(0), bytearray(ctypes.sizeof(T))])
        else:
            base.append(128 if len(base) > 1 else 0)
            forms.append([8, 1, 0, -1, 128 - (1 << 32), (1 << 32) + 128, 1 << 70, np.int64(128), np.uint32(8), True, t(128), 1.5, None, "128"])

    def outcome(fn, a):
        try:
            return fn(*a), iu8.lib().saber_iu8_last_error()
        except Exception as e:
            return type(e), str(e)

    calls = [base, base[:-1], base + [0], []] + [base[:i] + [v] + base[i + 1:] for i, vs in enumerate(forms) for v in vs]
    refused = sum(isinstance(outcome(g, a)[0], int) for a in calls)
    assert refused > len(base)      # the library's own refusals, not the conversions' alone
    for a in calls:
        want = outcome(g, a)
        assert want[0] != 0 and outcome(f, a) == want, (name, a)


def test_routed_operators_of_a_context_take_any_form(op):
    """The routed layer's methods with a count or a stream that is not a plain int (refused for the missing context, by the
    library), on the extension and on ctypes alone; what is not a table is refused as ctypes refuses it."""
    ctx, P = iu8.Context.__new__(iu8.Context), 1 << 40
    ctx._h, ctx._op, ctx._addr = ctypes.c_void_p(), op, None
    calls = (("moe_route", (P, 16, 128, 8, 1), ()), ("moe_route_quant", (P, P, P, P, 16, 128, 8, 4096, 1), ()),
             ("moe_grouped", (P, P, P, P, 4096, 1536, True, 16, 128, 8, 1), ()), ("moe_gate_up_act", (P, P, P, P, 1536, 4096, 16, 128, 8, 1), ()),
             ("moe_down_rows", (P, P, P, 4096, 1536, 16, 128, 8, 1), ()), ("moe_quant_rows", (P, P, P, 4096, 64), ()),
             ("moe_silu_mul_quant", (P, P, P, 1536, 64), ()), ("moe_combine", (P,), (P, 16, 8, 4096)))
    for name, before, after in calls:
        for tables in (iu8.MoeTables(), OtherTables()):
            full = before + (tables,) + after
            ints = [i for i, a in enumerate(full) if type(a) is int and a != P]
            for a in [full] + [full[:i] + (np.int64(full[i]),) + full[i + 1:] for i in ints]:
                for stream in (0, None, ctypes.c_void_p(0)):
                    with pytest.raises(iu8.IU8Error, match="null argument"):
                        getattr(ctx, name)(*a, stream=stream)
        for bad in (None, 0, iu8.Counters()):
            with pytest.raises((ctypes.ArgumentError, TypeError)):
                getattr(ctx, name)(*before, bad, *after)


# ------------------------------------------------------------------ operand orders

def test_a_order_is_a_bijection_with_16_byte_lane_pieces():
    L = iu8.lib()
    M, K = 32, 256
    offs = np.array([[L.saber_iu8_a_offset(m, k, K) for k in range(K)] for m in range(M)])
    assert sorted(offs.ravel().tolist()) == list(range(M * K))
    # lane l of fragment (mt, kt): row mt*16 + l%16, k = kt*64 + (l/16)*16 + 0..15
    for (m, k) in [(0, 0), (5, 17), (17, 130), (31, 255)]:
        mt, kt, lane = m // 16, k // 64, (m % 16) + 16 * ((k % 64) // 16)
        assert offs[m, k] == (mt * (K // 64) + kt) * 1024 + lane * 16 + k % 16
    rng = np.random.default_rng(0)
    a = rng.integers(-127, 128, (21, K), dtype=np.int8)
    frag = iu8.repack_a(a)
    assert frag.size == 32 * K == iu8.a_bytes(21, K)
    np.testing.assert_array_equal(iu8.unpack_a(frag, 21, K), a)
    assert frag.view(np.int8)[offs[7, 33]] == a[7, 33]


def test_w4_order_unpacks_to_natural_k_order():
    L = iu8.lib()
    N, K = 32, 256
    rng = np.random.default_rng(1)
    codes = rng.integers(-8, 8, (N, K), dtype=np.int8)
    frag = iu8.repack_w4(synth.pack_w4(codes))
    seen = set()
    for n in range(N):
        for k in range(K):
            hi = ctypes.c_uint32()
            off = L.saber_iu8_w4_offset(n, k, K, ctypes.byref(hi))
            seen.add((off, hi.value))
            nib = (int(frag[off]) >> 4) if hi.value else (int(frag[off]) & 15)
            assert (nib - 16 if nib >= 8 else nib) == codes[n, k]
    assert len(seen) == N * K
    # the device unpack: lo = (d << 4) & 0xF0F0F0F0, hi = d & 0xF0F0F0F0 of lane l's dwords d0..d3 gives
    # int8 = 16 * code for k = kt*128 + s*64 + (l/16)*16 + 0..15 in order, s = 0 (d0,d1) and 1 (d2,d3)
    d = frag.view(np.uint32).reshape(N // 16, K // 128, 64, 4)
    for (nt, kt, lane) in [(0, 0, 0), (1, 1, 37), (0, 1, 63)]:
        for s in (0, 1):
            regs = []
            for j in (2 * s, 2 * s + 1):
                dj = int(d[nt, kt, lane, j])
                regs += [(dj << 4) & 0xF0F0F0F0, dj & 0xF0F0F0F0]
            vals = np.array(regs, np.uint32).view(np.int8)
            k0 = kt * 128 + s * 64 + (lane // 16) * 16
            np.testing.assert_array_equal(vals, 16 * codes[nt * 16 + lane % 16, k0:k0 + 16])


def test_reference_gfx12_orders_reorder_to_the_same_bytes():
    # build the reference's fragment orders from the canonical form with the oracle's address
    # functions, then let the library re-order them: the result must equal the direct repack
    L = ref.lib()
    N, K = 32, 256
    rng = np.random.default_rng(4)
    codes = rng.integers(-8, 8, (N, K), dtype=np.int8)
    f12 = np.zeros(N * K // 2, np.uint8)
    seen = set()
    for n in range(N):
        for k in range(K):
            nib = ctypes.c_uint32()
            off = L.w4a8_w4_frag_gfx12(n, k, K, ctypes.byref(nib))
            seen.add((off, nib.value))
            f12[off] |= (int(codes[n, k]) & 15) << (4 * nib.value)
    assert len(seen) == N * K
    out = np.empty_like(f12)
    assert iu8.lib().saber_iu8_repack_w4_from_gfx12(f12.ctypes.data_as(ctypes.c_void_p), N, K, out.ctypes.data_as(ctypes.c_void_p)) == 0
    np.testing.assert_array_equal(out, iu8.repack_w4(synth.pack_w4(codes)))
    w8 = rng.integers(-127, 128, (N, K), dtype=np.int8)
    g12 = np.zeros(N * K, np.uint8)
    offs = set()
    for n in range(N):
        for k in range(K):
            off = L.w4a8_a_tiled_gfx12(n, k, K)
            offs.add(off)
            g12[off] = w8[n, k].view(np.uint8)
    assert offs == set(range(N * K))
    out8 = np.empty_like(g12)
    assert iu8.lib().saber_iu8_repack_w8_from_gfx12(g12.ctypes.data_as(ctypes.c_void_p), N, K, out8.ctypes.data_as(ctypes.c_void_p)) == 0
    np.testing.assert_array_equal(out8, iu8.repack_w8(w8))


def test_repack_refuses_ragged_shapes():
    with pytest.raises(iu8.IU8Error):
        iu8.repack_w4(np.zeros((24, 64), np.uint8))
    with pytest.raises(iu8.IU8Error):
        iu8.repack_w8(np.zeros((16, 192), np.int8))


def test_lines_of_the_streamed_cells_past_one_round():
    """Either side of the lines in rows, columns and K: 64-column blocks of the streamed symbols, the wide streamed cells,
    shares of K on deep linears. A launch without workspaces and a pair stay in one piece."""
    def law(w8, m, n, k):
        d = iu8.resolve(iu8.W8 if w8 else iu8.W4, m, n, k)
        return d.kernel.decode()[len("macaq_iu8_"):], d.grid[0], d.ks

    for (w8, m, n, k), want in {
            (0, 32, 8192, 1024): ("dec_w4_tm2", 256, 1), (0, 32, 8208, 1024): ("dec_w4_tm2", 129, 1), (1, 17, 16384, 128): ("dec_w8_tm2", 256, 1),
            (0, 33, 12224, 5120): ("pf_w4_t64x64_s", 191, 1), (0, 33, 12240, 5120): ("dec_w4_tm3", 192, 1), (0, 48, 16384, 2048): ("dec_w4_tm3", 256, 1),
            (0, 48, 16384, 1920): ("pf_w4_t64x64_s", 256, 1), (1, 48, 16384, 4096): ("dec_w8_tm3", 256, 1), (1, 48, 16384, 3968): ("pf_w8_t64x64_s", 256, 1),
            (0, 64, 16384, 3072): ("dec_w4_tm4", 256, 1), (0, 64, 16384, 2944): ("pf_w4_t64x64_s", 256, 1),
            (0, 32, 18336, 1024): ("pf_w4_t64x128_s", 144, 1), (0, 32, 18352, 1024): ("pf_w4_t32x96_w", 192, 1), (0, 48, 24576, 2048): ("pf_w4_t48x96_w", 256, 1),
            (0, 49, 24576, 3968): ("pf_w4_t64x128_s", 192, 1), (0, 49, 24576, 4096): ("pf_w4_t64x96_w", 256, 1), (0, 80, 20480, 3072): ("pf_w4_t80x96_w", 214, 1),
            (0, 96, 20480, 5120): ("pf_w4_t96x96_w", 214, 1), (1, 64, 24576, 2048): ("pf_w8_t64x96_w", 256, 1), (1, 96, 24576, 4096): ("pf_w8_t96x96_w", 256, 1),
            (0, 32, 32768, 4096): ("pf_w4_t32x144_w", 228, 1), (0, 33, 32768, 5120): ("pf_w4_t64x128_s", 256, 1), (1, 33, 32768, 3072): ("pf_w8_t48x144_w", 228, 1),
            (0, 45, 34816, 5120): ("pf_w4_t48x144_w", 242, 1), (0, 64, 36864, 4096): ("pf_w4_t64x144_w", 256, 1), (0, 64, 36880, 5120): ("pf_w4_t64x160_s", 231, 1),
            (0, 96, 34816, 2048): ("pf_w4_t96x144_w", 242, 1), (1, 72, 14336, 2048): ("pf_w8_t80x64_w", 224, 1), (0, 72, 14336, 8192): ("pf_w4_t80x64_w", 224, 1),
            (0, 8, 5120, 17408): ("dec_w4_tm1_a0", 160, 1), (0, 9, 5120, 10240): ("dec_w4_tm1_a0", 80, 3), (0, 16, 5120, 10112): ("dec_w4_tm1_a0", 160, 1),
            (0, 17, 5120, 8192): ("dec_w4_tm2", 80, 3), (1, 48, 5440, 8192): ("dec_w8_tm3_n2", 85, 3), (1, 48, 5456, 8192): ("dec_w8_tm3_n2", 171, 1),
            (1, 49, 5120, 8192): ("dec_w8_tm4_n2", 160, 1), (0, 48, 4096, 12288): ("dec_w4_tm3", 64, 4), (0, 48, 4096, 12160): ("dec_w4_tm3", 256, 1),
            (0, 16, 3024, 12288): ("dec_w4_tm1_a0", 48, 4), (0, 16, 3008, 12288): ("dec_w4_tm1_a0", 94, 1)}.items():
        assert law(w8, m, n, k) == want, (w8, m, n, k, law(w8, m, n, k))
    d = iu8.resolve(iu8.W4, 16, 5120, 17408)
    assert iu8.gemm_workspace(iu8.W4, 16, 5120, 17408) == (3 * 16 * 5120 * 4, 80 * 4) and d.grid[2] == 3
    p = iu8.pair(d, iu8.describe("macaq_iu8_dec_w4_tm1_a0", 16, 9600, 17408, ks=1))
    assert (p.arg("nb").ival, p.arg("ks").ival, p.arg("nb_b").ival, p.arg("ks_b").ival) == (80, 3, 150, 1) and p.grid[0] == 80 * 3 + 150
    assert p.workspace("decode_counter").bytes == 80 * 4
    for name, m, ok in (("macaq_iu8_pf_w4_t48x144_w", 48, True), ("macaq_iu8_pf_w4_t48x144_w", 49, False)):
        if ok:
            assert iu8.describe(name, m, 160, 128).grid[0] == 2
        else:
            with pytest.raises(iu8.IU8Error):
                iu8.describe(name, m, 160, 128)
    with pytest.raises(iu8.IU8Error):
        iu8.describe("macaq_iu8_pf_w4_t48x144_w", 48, 160, 256, ks=2)


def test_lines_of_the_streamed_cells_on_row_tiles():
    """Either side of the lines in rows, columns, K and blocks; such a launch needs no workspace, its grid is whole eighths that
    hold every block, and a half of a pair is described again in the pair's form wherever it was one before."""
    for (w8, m, n, k), want in {
            (0, 16, 96, 5120): None, (0, 17, 96, 5120): "16x16", (0, 17, 96, 640): None, (0, 17, 96, 768): "16x16", (0, 48, 256, 768): "16x16",
            (0, 48, 272, 3968): None, (0, 48, 272, 4096): "16x16", (0, 48, 1024, 4096): "16x16", (0, 48, 1040, 4096): None,
            (1, 48, 512, 4096): "16x16", (1, 48, 512, 3968): None, (1, 48, 528, 5120): None, (1, 17, 96, 3968): None,
            (0, 49, 48, 2048): None, (0, 49, 64, 2048): "16x16", (1, 64, 48, 5120): None, (1, 64, 64, 768): "16x16", (0, 65, 16, 768): "16x16",
            (0, 49, 1024, 768): "16x16", (0, 49, 1040, 768): "16x32", (0, 64, 2048, 768): "16x32", (0, 64, 2064, 5120): None,
            (0, 400, 160, 1024): "16x16", (0, 416, 160, 1024): "16x32", (0, 777, 160, 1024): "16x32", (0, 800, 192, 2048): "32x32",
            (0, 800, 256, 1920): "32x32", (0, 800, 288, 1920): None, (0, 800, 320, 2048): "32x32", (0, 800, 336, 3968): None,
            (0, 800, 336, 4096): "32x64", (0, 800, 512, 4096): "32x64", (0, 800, 528, 4096): None, (0, 97, 3328, 4096): "32x64", (0, 97, 3344, 4096): None, (0, 2047, 96, 5120): "32x32", (0, 2048, 96, 5120): None,
            (0, 96, 5440, 4096): "32x64", (0, 96, 5456, 4096): None, (0, 96, 1024, 16256): "16x32", (0, 96, 1024, 16384): None, (0, 32, 96, 17408): "16x16", (0, 33, 96, 17408): None,
            (0, 193, 96, 17408): "16x16",
            (1, 100, 576, 768): "16x16", (1, 100, 592, 768): None, (1, 200, 304, 5120): "16x16", (1, 200, 320, 5120): None}.items():
        d = iu8.resolve(iu8.W8 if w8 else iu8.W4, m, n, k)
        name = d.kernel.decode()
        assert (name[len("macaq_iu8_pf_w4_t"):-2] if name.endswith("_r") else None) == want, (w8, m, n, k, name)
        if want:
            bm, bn = map(int, want.split("x"))
            assert d.grid[0] % 8 == 0 and 0 <= d.grid[0] - -(-m // bm) * -(-n // bn) < 8 and d.block[0] == 512 and d.n_workspaces == 0 and d.ks == 1
    for m, twin in ((17, "tm2"), (32, "tm2"), (48, "tm3")):
        wide, ba = iu8.resolve(iu8.W4, m, 16384, 5120), iu8.resolve(iu8.W4, m, 96, 5120)
        assert ba.kernel.endswith(b"_r")
        want = iu8.pair(wide, iu8.describe(f"macaq_iu8_dec_w4_{twin}", m, 96, 5120))
        assert bytes(iu8.pair(wide, ba)) == bytes(want)
    for m, k in ((49, 5120), (64, 5120), (33, 16384)):     # no half of a pair before, and none now
        with pytest.raises(iu8.IU8Error):
            iu8.pair(iu8.describe(f"macaq_iu8_dec_w4_tm{-(-m // 16)}", m, 96, k), iu8.resolve(iu8.W4, m, 96, k))
    with pytest.raises(iu8.IU8Error):
        iu8.describe("macaq_iu8_pf_w4_t16x16_r", 100, 96, 1024, ks=2)
    with pytest.raises(iu8.IU8Error):
        iu8.describe("macaq_iu8_pf_w4_t16x16_r", 1 << 20, 96, 1024)   # more blocks than a launch holds


def test_32x32_row_tiles_of_a_short_k():
    """Below K = 1,408 32 x 32 blocks lose to 64 x 64 tiles on outputs of more than 160 rows (192 from K = 1,152) and more than 256 columns
    (204 rows of 752 x 896 5.1 us for 4.5): such a launch is on tiles, either side of each line."""
    for (m, n, k), cell in {(204, 752, 896): "t64x64_s", (510, 368, 896): "t64x64_s", (241, 736, 768): "t64x64_s", (160, 928, 896): "t32x32_r", (161, 928, 896): "t64x64_s",
                            (161, 928, 1024): "t64x64_s", (192, 928, 1152): "t32x32_r", (193, 864, 1152): "t64x64_s", (193, 864, 1280): "t64x64_s", (193, 864, 1408): "t32x32_r",
                            (750, 256, 768): "t32x32_r", (700, 272, 768): "t64x64_s", (700, 272, 1408): "t32x32_r",
                            (1593, 80, 768): "t32x32_r", (66, 2000, 768): "t32x32_r"}.items():
        assert iu8.resolve(iu8.W4, m, n, k).kernel.decode() == "macaq_iu8_pf_w4_" + cell, (m, n, k)


def test_row_tiles_leave_operands_past_4_gib_to_the_other_cells():
    """An operand past 4 GiB, which the tile GEMM refuses by name, is refused for an output of few tiles as for any other, on either
    side of the limit in rows, columns and K; up to 64 rows the streamed form, which has no such limit, has it."""
    for kind, m, n, k in ((iu8.W4, 1518, 112, 13019776), (iu8.W8, 425, 48, 10425088), (iu8.W8, 1181, 48, 4639872), (iu8.W4, 65, 1024, 1 << 23),
                          (iu8.W4, 256, 64, 1 << 24), (iu8.W8, 65, 256, 1 << 24), (iu8.W4, 2000, 16, 1 << 22)):
        with pytest.raises(iu8.IU8Error, match="4 GiB") as e:
            iu8.resolve(kind, m, n, k)
        assert e.value.code == iu8.E_RULE
    for kind, m, n, k in ((iu8.W4, 256, 64, (1 << 24) - 128), (iu8.W4, 2000, 16, 2147328), (iu8.W8, 65, 240, 1 << 24)):
        assert iu8.resolve(kind, m, n, k).kernel.endswith(b"_r"), (m, n, k)
    assert iu8.resolve(iu8.W4, 17, 1024, 1 << 23).kernel == b"macaq_iu8_dec_w4_tm2_n1"
    for m, name in ((48, b"macaq_iu8_dec_w8_tm3"), (49, b"macaq_iu8_dec_w8_tm4_k16"), (64, b"macaq_iu8_dec_w8_tm4_k16")):
        assert iu8.resolve(iu8.W8, m, 256, 1 << 24).kernel == name


def test_thin_tiles_by_weight_kind(tmp_path):
    """The layout rule of the 256 x 256 cell (csrc/kernels/iu8_pf_law.h, compiled here): which launches of 256 workgroups run
    the rows past the last whole 256 as thin tiles -- int8 weights only where they measured no slower than whole tiles. Every
    thin tile is dealt out once, whatever share the workgroups with a tile less take."""
    src, so = tmp_path / "plan.cpp", tmp_path / "plan.so"
    src.write_text(f'#include "{iu8.PKG}/csrc/kernels/iu8_pf_law.h"\n'
                   'extern "C" void plan(int m, int gx, int G, int k, int w8, int *o) {\n'
                   '  const iu8_pf_plan p = iu8_pf_plan256(m, gx, G, k, w8 != 0);\n'
                   '  const int v[] = {p.thin, p.tail, p.gy, p.q, p.rem, p.own, p.own_wgs};\n'
                   '  for (int i = 0; i < 7; ++i) o[i] = v[i];\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    lib, out = ctypes.CDLL(str(so)), (ctypes.c_int * 7)()

    def plan(m, n, k, w8, G=256):
        gx = -(-n // 256)
        lib.plan(m, gx, min(G, gx * -(-m // 256)), k, int(w8), out)
        return list(out)

    for m, n, w4, w8 in ((520, 28672, 1, 0), (1030, 16384, 1, 0), (4105, 8192, 1, 0), (8212, 6144, 1, 0), (520, 34816, 1, 0), (600, 28672, 1, 0),
                         (1290, 28672, 1, 0), (1540, 20480, 1, 0), (4105, 20480, 1, 1), (4200, 20480, 1, 1), (8212, 28672, 1, 1), (777, 34816, 1, 1),
                         (800, 34816, 1, 1), (1030, 28672, 1, 1), (3100, 10240, 1, 1), (897, 34816, 0, 0), (2048, 34816, 0, 0)):
        assert (plan(m, n, 5120, False)[0], plan(m, n, 5120, True)[0]) == (w4, w8), (m, n)
        assert not plan(m, n, 896, False)[0] and not plan(m, n, 896, True)[0]
    rng, seen = np.random.default_rng(7), 0
    for _ in range(3000):
        m, gx, G, w8 = int(rng.integers(257, 9000)), int(rng.integers(1, 140)), int(rng.integers(1, 257)), int(rng.integers(0, 2))
        thin, tail, gy, q, rem, own, own_wgs = plan(m, gx * 256, 5120, w8, G)
        if not thin:
            continue
        seen += 1
        assert gy == m // 256 and 0 < m % 256 <= 128 and q * min(G, gx * -(-m // 256)) + rem == gx * gy
        G, got = min(G, gx * -(-m // 256)), []
        for at in range(G):          # the kernel's walk: iu8_dense_defs.h, iu8_thin_tile_at
            for r in range(200):
                if own_wgs > 0 and at >= rem and r < own:
                    j = at - rem + r * own_wgs
                else:
                    j = own * own_wgs + (G - 1 - at) + (r - (own if own_wgs > 0 and at >= rem else 0)) * G
                if j >= gx:
                    break
                got.append(j)
        assert sorted(got) == list(range(gx)), (m, gx, G, w8)
    assert seen > 200


def test_64_column_blocks_where_they_halve_the_blocks_a_cu():
    """The streamed symbols' block width on both sides of its lines: an even count of 32-column blocks on the busiest of the 256
    CUs, the edges of such a count at up to eight rows, and a K of whole 8,192; the pair's halves by the same rule."""
    for (m, n, k), blocks in {
            (16, 8192, 5376): 256, (16, 8208, 5376): 129, (5, 16384, 5376): 256, (5, 16400, 5376): 513, (16, 24576, 5376): 768,
            (16, 24592, 5376): 385, (16, 32768, 5376): 512, (16, 32784, 5376): 1025, (9, 41008, 5376): 641,
            (8, 25088, 5376): 784, (8, 25104, 5376): 393, (9, 25088, 5376): 392, (8, 29696, 5376): 464, (8, 29712, 5376): 929, (9, 29712, 5376): 465,
            (8, 13312, 8192): 208, (8, 13328, 8192): 417, (9, 13328, 8192): 209, (8, 13328, 8064): 209, (8, 13328, 16384): 417,
            (8, 28672, 8192): 896, (9, 31744, 8192): 496, (9, 31760, 8192): 993, (16, 15360, 8192): 240, (16, 15376, 8192): 481}.items():
        for wk, tag in ((iu8.W4, "w4"), (iu8.W8, "w8")):
            d = iu8.resolve(wk, m, n, k)
            assert (d.kernel.decode(), d.grid[0], d.ks) == (f"macaq_iu8_dec_{tag}_tm1_a0", blocks, 1), (m, n, k, d.grid[0])
        p = iu8.pair(iu8.resolve(iu8.W4, m, n, k), iu8.resolve(iu8.W4, m, 48, k))
        assert (p.arg("nb").ival, p.arg("nb_b").ival) == (blocks, 2), (m, n, k)
    assert iu8.resolve(iu8.W4, 17, 16384, 8192).grid[0] == 256
    for (m, n0, n1, k), blocks in {(16, 9600, 9600, 8192): (300, 300), (16, 9600, 96, 8192): (150, 3), (16, 16384, 16384, 5376): (256, 256),
                                   (16, 16384, 8192, 5376): (256, 256), (8, 16384, 16384, 5376): (512, 512),
                                   (40, 12288, 12288, 8192): (192, 192)}.items():
        p = iu8.pair(iu8.resolve(iu8.W4, m, n0, k), iu8.resolve(iu8.W4, m, n1, k))
        assert (p.arg("nb").ival, p.arg("nb_b").ival) == blocks, (m, n0, n1, k)


def test_arrivals_of_shared_launches_are_counted_at_any_share_count(tmp_path):
    """The arrival counters of a streamed launch that shares K (csrc/kernels/iu8_stream_law.h, compiled here), the blocks' arrivals
    in any order: one last arrival a block, behind all its others, and every word back at zero, in no more words than blocks
    (half of them up to 16 bits of shares, which is what a tile launch's workspaces hold)."""
    src, so = tmp_path / "arrival.cpp", tmp_path / "arrival.so"
    src.write_text(f'#include "{iu8.PKG}/csrc/kernels/iu8_stream_law.h"\n'
                   'extern "C" int run(int blocks, int shares, int odd_first, unsigned *words) {\n'
                   '  for (int i = 0; i < blocks; ++i) {\n'
                   '    const iu8_arrival a = iu8_arrival_of(i, shares);\n'
                   '    if (a.word < 0 || a.word >= (shares <= 0xFFFF ? (blocks + 1) / 2 : blocks)) return 1;\n'
                   '  }\n'
                   '  for (int s = 0; s < shares; ++s)\n'       # the last arrivals of two blocks of a word either way round
                   '    for (int j = 0; j < blocks; ++j) {\n'
                   '      const int i = odd_first ? blocks - 1 - j : j;\n'
                   '      const iu8_arrival a = iu8_arrival_of(i, shares);\n'
                   '      const unsigned before = words[a.word];\n'
                   '      words[a.word] += a.one();\n'
                   '      if (a.last(before, shares) != (s == shares - 1)) return 2;\n'
                   '      if (s == shares - 1) words[a.word] -= a.all(shares);\n'
                   '    }\n'
                   '  return 0;\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    for blocks in (1, 2, 3, 80):
        for shares in (2, 3, 4, 0xFFFE, 0xFFFF, 0x10000, 0x10001, 70000, 1 << 17):
            for odd_first in (0, 1):
                words = (ctypes.c_uint * (blocks + 1))()
                assert lib.run(blocks, shares, odd_first, words) == 0 and not any(words), (blocks, shares, odd_first)


def test_band_table_grids_follow_their_cell_rows():
    """Every decode and wide row of the shipped law table states the grid that its cell row and the table's own rules give: the
    block width, the shares of K, one arrival counter a block."""
    import tomli

    t = tomli.loads(open(iu8.BAND_TABLE).read())
    cells, sp, bw = {c["kernel"]: c for c in t["cell"]}, t["stream_split"], t["decode_block_width"]

    def shares(m, n, k):
        b = -(-n // 64)
        z = min(sp["shares_max"], t["cu_count"] // b)
        k_min = sp["k_min_16_rows"] if m <= 16 else sp["k_min_4096_columns"] if n <= 4096 else sp["k_min"]
        return z if sp["rows_over"] < m <= sp["rows_max"] and z >= sp["shares_min"] and 16 * b >= 3 * t["cu_count"] and k >= k_min else t["decode_split"]

    def width(c, m, n, k, ks):
        if "block_n_wide" not in c or (ks == 1 and c["block_n"] == 16 and n <= bw["round"]):
            return c["block_n"]
        a = -(-n // bw["round"])
        last, aligned = n - (a - 2) * bw["round"], k % bw["aligned_k"] == 0
        if m <= bw["few_rows"]:
            edge = (not aligned or last <= bw["few_last_max"]) if a == 2 else not aligned and bw["few_last_over"] < last <= bw["few_last_max"]
        else:
            edge = m > bw["aligned_rows"] or not aligned or last <= bw["aligned_last_max"]
        return c["block_n_wide"] if ks > 1 or c["block_n"] == 16 or (a % 2 == 0 and edge) else c["block_n"]

    seen = set()
    for b in t["band"]:
        c = cells[b["kernel"]]
        if c["regime"] not in ("decode", "wide") or "persistent" in c["grid"]:
            continue
        for m, grid in ((b["first_m"], b["grid_first"]), (b["last_m"], b["grid_last"])):
            ks = shares(m, b["n"], b["k"]) if "block_n_wide" in c else 1     # (the streamed symbols have one)
            w = width(c, m, b["n"], b["k"], ks) if c["regime"] == "decode" else c["block_n"]
            assert b["ks"] == ks and grid == [-(-b["n"] // w), 1, ks], (b, m, ks, w)
            seen.add((c["regime"], w, ks > 1))
            if ks > 1:
                assert iu8.gemm_workspace(iu8.W8 if b["w8"] else iu8.W4, m, b["n"], b["k"])[1] == 4 * grid[0]
    assert {("decode", 64, True), ("decode", 64, False), ("decode", 32, False), ("decode", 16, False), ("wide", 144, False)} <= seen
    # the width rule away from the table's shapes
    rng = np.random.default_rng(11)
    for _ in range(2000):
        name = str(rng.choice([c for c in cells if cells[c]["regime"] == "decode" and "block_n_wide" in cells[c]]))
        c, n, k, ks = cells[name], int(rng.integers(1, 3500)) * 16, int(rng.choice([128, 5376, 8192, 16384])), int(rng.integers(1, 3))
        m, ks = int(rng.integers(1, c["rows_max"] + 1)), min(ks, k // 128)
        assert iu8.describe(name, m, n, k, ks).grid[0] == -(-n // width(c, m, n, k, ks)), (name, m, n, k, ks)


def test_lines_of_the_calls_that_stream_in_a_tile_launchs_workspaces(tmp_path):
    """What saber_iu8_gemm makes of the law's tile launches that share K (rules.cpp:stream_in_tile_workspaces, called in the library):
    which shapes stream, on which symbol and shares, either side of the lines in rows, columns and K; partials and
    counters are never more than the tile launch's, counting as the kernel does."""
    src, so = tmp_path / "streams.cpp", tmp_path / "streams.so"
    src.write_text(f'#include "{iu8.ROOT}/include/saber_iu8.h"\n#include "{iu8.PKG}/csrc/host/rules.h"\n#include "{iu8.PKG}/csrc/kernels/iu8_stream_law.h"\n'
                   'extern "C" int streams(const saber_iu8_desc *d, saber_iu8_desc *out) { return iu8::stream_in_tile_workspaces(*d, out); }\n'
                   'extern "C" int words(int blocks, int shares) {\n'
                   '  int n = 0;\n'
                   '  for (int i = 0; i < blocks; ++i) n = iu8_arrival_of(i, shares).word + 1;\n'
                   '  return n;\n}\n')
    lib_dir = os.path.dirname(iu8.lib()._name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so), f"-L{lib_dir}", "-lsaber_iu8", f"-Wl,-rpath,{lib_dir}"], check=True)
    lib = ctypes.CDLL(str(so))

    def streamed(m, n, k):
        tiles, out = iu8.resolve(iu8.W4, m, n, k), iu8.Desc()
        return tiles, out if lib.streams(ctypes.byref(tiles), ctypes.byref(out)) else None

    for (m, n, k), want in {(33, 5120, 16384): ("tm3_n2", 3), (48, 5120, 17408): ("tm3_n2", 3), (49, 5120, 17408): ("tm4_n2", 3), (64, 5120, 17408): ("tm4_n2", 3),
                            (65, 5120, 17408): None, (33, 4096, 16384): ("tm3", 4), (48, 4112, 16384): ("tm3_n2", 3), (64, 4096, 16384): ("tm4", 4),
                            (33, 3024, 16384): ("tm3", 4), (33, 3008, 16384): None, (64, 3008, 16384): None, (48, 5440, 16384): ("tm3_n2", 3),
                            (48, 5456, 16384): None, (64, 5456, 16384): None, (45, 8192, 16384): None, (32, 5120, 17408): None, (45, 5120, 16256): None}.items():
        tiles, d = streamed(m, n, k)
        assert (tiles.kernel == b"macaq_iu8_pf_w4_t64x128_s_ks") == (33 <= m and k >= 16384), (m, n, k)
        assert (d and (d.kernel.decode()[len("macaq_iu8_dec_w4_"):], d.ks)) == want, (m, n, k)
    rng = np.random.default_rng(2)
    taken = 0
    for _ in range(4000):
        m, n, k = int(rng.integers(33, 65)), 16 * int(rng.integers(180, 360)), 128 * int(rng.integers(120, 300))
        tiles, d = streamed(m, n, k)
        if d is None:
            continue
        taken += 1
        assert d.grid[2] == d.ks and d.grid[0] == -(-n // 64) and d.ks <= tiles.ks
        assert d.workspace("decode_partial").bytes <= tiles.workspace("decode_partial").bytes
        assert 4 * lib.words(d.grid[0], d.ks) <= tiles.workspace("decode_counter").bytes
    assert taken > 1000


def test_words_are_shared_only_in_a_tile_launchs_workspaces(tmp_path):
    """Two column blocks count in one word only where a streamed launch may stand in a tile launch's workspaces
    (csrc/kernels/iu8_stream_law.h, compiled here): every launch that does so shares its words, and the law's own K shares, which
    list a counter a block, count in a word each (at two in one, 9 to 48 rows lost 2-5 %)."""
    src, so = tmp_path / "shared.cpp", tmp_path / "shared.so"
    src.write_text(f'#include "{iu8.ROOT}/include/saber_iu8.h"\n#include "{iu8.PKG}/csrc/host/rules.h"\n#include "{iu8.PKG}/csrc/kernels/iu8_stream_law.h"\n'
                   'extern "C" int streams(const saber_iu8_desc *d, saber_iu8_desc *out) { return iu8::stream_in_tile_workspaces(*d, out); }\n'
                   'extern "C" int two(int w8, int tm, long k) { return iu8_stream_shared_words(w8, tm, k); }\n'
                   'extern "C" int words(int blocks, int shares, int w8, int tm, long k) {\n'
                   '  return iu8_arrival_of(blocks - 1, shares, iu8_stream_shared_words(w8, tm, k)).word + 1;\n}\n')
    lib_dir = os.path.dirname(iu8.lib()._name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so), f"-L{lib_dir}", "-lsaber_iu8", f"-Wl,-rpath,{lib_dir}"], check=True)
    lib = ctypes.CDLL(str(so))
    rng, called, split = np.random.default_rng(5), 0, 0
    for _ in range(6000):
        m, n, k, kind = int(rng.integers(9, 65)), 16 * int(rng.integers(180, 360)), 128 * int(rng.integers(60, 300)), int(rng.choice([iu8.W4, iu8.W8]))
        d, out = iu8.resolve(kind, m, n, k), iu8.Desc()
        tm = -(-m // 16)
        if kind == iu8.W4 and lib.streams(ctypes.byref(d), ctypes.byref(out)):
            called += 1
            assert lib.two(0, tm, k) and 4 * lib.words(out.grid[0], out.ks, 0, tm, k) <= d.workspace("decode_counter").bytes
        elif d.kernel.startswith(b"macaq_iu8_dec_") and d.ks > 1:
            split += 1
            assert not lib.two(kind == iu8.W8, tm, k) and 4 * lib.words(d.grid[0], d.ks, kind == iu8.W8, tm, k) == d.workspace("decode_counter").bytes
    assert called > 300 and split > 300


def test_routed_items_are_dealt_once_and_level(tmp_path):
    """The deal of the routed tile launches (csrc/kernels/moe_deal.h, compiled here): every light item goes to one position
    once, and no position's share (a heavy item counts `cost`) is more than one heavy item above another's that has light ones."""
    src, so = tmp_path / "deal.cpp", tmp_path / "deal.so"
    src.write_text(f'#include "{iu8.PKG}/csrc/kernels/moe_deal.h"\n'
                   'extern "C" int share(int hi, int li, int G, int cost, int w, int *ids) {\n'
                   '  const moe_deal d = moe_deal_of(hi, li, G, cost);\n'
                   '  int n = 0;\n'
                   '  for (int r = 0; r < (w < d.more ? d.l_more : d.l_rest); ++r)\n'
                   '    if (d.light_id(r, w, G) < li) ids[n++] = d.light_id(r, w, G);\n'
                   '  return n;\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    lib, ids = ctypes.CDLL(str(so)), (ctypes.c_int * 4096)()
    rng = np.random.default_rng(3)
    cases = [(0, 1, 256, 2), (24, 1548, 256, 2), (256, 0, 256, 2), (255, 1, 256, 4), (1, 256, 256, 2), (1, 255, 256, 2), (1536, 700, 256, 4),
             (0, 2048, 256, 2), (5, 3, 3, 2), (1, 2, 1, 4)]
    cases += [(int(rng.integers(0, 3000)), int(rng.integers(0, 3000)), int(rng.choice([1, 3, 16, 255, 256])), int(rng.choice([2, 4]))) for _ in range(60)]
    for hi, li, G, cost in cases:
        got, load = [], []
        for w in range(G):
            n = lib.share(hi, li, G, cost, w, ids) if (li // G + cost + 2) < 4096 else 0
            got += ids[:n]
            load.append((cost * (hi // G + (w < hi % G)) + n, n))
        assert sorted(got) == list(range(li)), (hi, li, G, cost)
        top = max(x for x, n in load if n) if li else 0
        assert all(x >= top - 1 - cost for x, _ in load), (hi, li, G, cost)


def test_routed_items_are_dealt_to_the_level_share(tmp_path):
    """No position that has light items has a larger share (a heavy item counts `cost`) than the level one, all of it over the
    positions rounded up, or one more heavy item than every position has alone. Dealt evenly, the two kinds apart, 31 of
    these 70 cases have."""
    src, so = tmp_path / "deal.cpp", tmp_path / "deal.so"
    src.write_text(f'#include "{iu8.PKG}/csrc/kernels/moe_deal.h"\n'
                   'extern "C" int share(int hi, int li, int G, int cost, int w, int *ids) {\n'
                   '  const moe_deal d = moe_deal_of(hi, li, G, cost);\n'
                   '  int n = 0;\n'
                   '  for (int r = 0; r < (w < d.more ? d.l_more : d.l_rest); ++r)\n'
                   '    if (d.light_id(r, w, G) < li) ids[n++] = d.light_id(r, w, G);\n'
                   '  return n;\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    lib, ids = ctypes.CDLL(str(so)), (ctypes.c_int * 4096)()
    rng = np.random.default_rng(3)
    cases = [(0, 1, 256, 2), (24, 1548, 256, 2), (256, 0, 256, 2), (255, 1, 256, 4), (1, 256, 256, 2), (1, 255, 256, 2), (1536, 700, 256, 4),
             (0, 2048, 256, 2), (5, 3, 3, 2), (1, 2, 1, 4)]
    cases += [(int(rng.integers(0, 3000)), int(rng.integers(0, 3000)), int(rng.choice([1, 3, 16, 255, 256])), int(rng.choice([2, 4]))) for _ in range(60)]
    uneven = 0
    for hi, li, G, cost in cases:
        got, load = [], []
        for w in range(G):
            n = lib.share(hi, li, G, cost, w, ids) if (li // G + cost + 2) < 4096 else 0
            got += ids[:n]
            load.append((cost * (hi // G + (w < hi % G)) + n, n))
        assert sorted(got) == list(range(li)), (hi, li, G, cost)
        level = max(-(-(cost * hi + li) // G), cost * (hi // G + 1))
        assert all(x <= level for x, n in load if n), (hi, li, G, cost)
        even = [(cost * (hi // G + (w < hi % G)) + n, n) for w, n in enumerate(li // G + (G - 1 - w < li % G) for w in range(G))]
        uneven += any(x > level for x, n in even if n)
    assert uneven == 31


def test_routed_launches_keep_both_cells_on_wide_experts(tmp_path):
    """Which tiles of a 256-row routed launch run on the tile cell (csrc/kernels/moe_deal.h, compiled here; a table of 18 light items a
    workgroup): 128 experts of a full tile and a light one keep both cells up to outputs of 9,216 columns, and past the
    table all tiles run on the tile cell, where a launch of up to 64 of its items a workgroup still has them resolved in front."""
    src, so = tmp_path / "cells.cpp", tmp_path / "cells.so"
    src.write_text(f'#include "{iu8.PKG}/csrc/kernels/moe_deal.h"\n'
                   'extern "C" int tiles(int heavy, int nt, int gx, int G, int cost, int lr) { return moe_tile_cell_tiles(heavy, nt, gx, G, cost, lr); }\n'
                   'extern "C" int rounds(int hi, int li, int G, int cost) { return moe_deal_of(hi, li, G, cost).l_rest; }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    for columns, tiles in ((3072, 128), (4096, 128), (7168, 128), (8192, 128), (9216, 128), (9472, 256), (16384, 256)):
        assert lib.tiles(128, 256, columns // 256, 256, 4, 18) == tiles, columns
    assert 256 * (16384 // 256) <= 64 * 256
    rng = np.random.default_rng(11)
    for _ in range(2000):
        nt, gx, G, lr = int(rng.integers(1, 900)), int(rng.integers(1, 70)), int(rng.choice([1, 3, 8, 61, 256])), int(rng.choice([12, 18]))
        heavy = int(rng.integers(0, nt + 1))
        kept = lib.tiles(heavy, nt, gx, G, 4, lr)
        assert kept == (heavy if lib.rounds(heavy * gx, (nt - heavy) * gx, G, 4) <= lr else nt)
        assert lib.rounds(kept * gx, (nt - kept) * gx, G, 4) <= lr           # what the light table is asked to hold
