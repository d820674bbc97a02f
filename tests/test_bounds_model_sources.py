"""The CPU bounds replay (``tests/bounds_model.py``) restates the launchers' tile tables and the
kernels' ring and tile constants.  These tests read the same values out of the HIP sources, so a
change to a kernel's shape that is not mirrored in the replay fails here instead of going unseen.
Each check names the source line it parses; a pattern that no longer matches fails too."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

import bounds_model as bm

CSRC = Path(__file__).resolve().parent.parent / "pymsst_amd" / "csrc"


def _src(name: str) -> str:
    return (CSRC / name).read_text()


def _one(pattern: str, text: str, what: str) -> re.Match:
    found = list(re.finditer(pattern, text))
    assert len(found) == 1, f"{what}: pattern {pattern!r} matched {len(found)} times"
    return found[0]


def _const(name: str, src: str) -> int:
    return int(_one(rf"constexpr int {name} = (\d+);", _src(src), name).group(1))


def _define(name: str, src: str) -> int:
    return int(_one(rf"#define {name} (\d+)", _src(src), name).group(1))


def test_shared_constants():
    assert _const("kChunkK", "mfma.h") == bm.CHUNK_K
    assert _const("kGemmThreads", "gemm.h") == bm.GEMM_THREADS
    assert _const("kRowSumMaxF", "band_split.hip") == bm.ROWSUM_MAX_F


def test_mask_mlp_tile_table_and_ring():
    """mask_mlp.hip launch_mlp_fwd: dim -> launch_dk<T, DK, NT[, WV = 4]>; kMlpJ; mlp_stages."""
    s = _src("mask_mlp.hip")
    table = {int(d): (int(dk), int(nt), int(wv or 4))
             for d, dk, nt, wv in re.findall(r"case (\d+): return launch_dk<T, (\d+), (\d+)(?:, (\d+))?>", s)}
    assert table == bm.MLP_TILES
    assert _const("kMlpJ", "mask_mlp.hip") == 64
    m = _one(r"return DK >= (\d+) \? (\d+) : (\d+);", s, "mlp_stages")
    assert tuple(int(v) for v in m.groups()) == (12, 2, 3)  # S, J = (2 if DK >= 12 else 3), 64 in the replay
    # the row tile rule: full - 32 where the last full tile holds at most an eighth of a tile
    _one(r"const int64_t alt = full - 32;", s, "mlp_row_tile")
    _one(r"if \(M > full && tail <= full / 8 && \(M \+ alt - 1\) / alt == tiles\) return alt;", s, "mlp_row_tile")
    assert bm.mlp_row_tile(1032, 2, 8) == 224 and bm.mlp_row_tile(1024, 2, 8) == 256


def test_grouped_dx_tile_table_and_row_tile():
    """grouped_dx.hip launch_grouped_dx: in_features -> launch<T, DT, NT, S>, the two forms at 192."""
    s = _src("grouped_dx.hip")
    plain = {int(i): (int(dt), int(nt), int(st))
             for i, dt, nt, st in re.findall(r"case (\d+): return launch<T, (\d+), (\d+), (\d+)>", s)}
    assert plain == {k: v for k, v in bm.GDX_TILES.items() if k != 192}
    forms = set(re.findall(r"launch<T, 12, (\d+), (\d+)>", s))
    assert forms == {("3", "3"), ("2", "4")}
    assert bm.GDX_TILES[192] == (12, 2, 4)
    assert bm.gdx_tiles(192, 62, 1032) == (12, 3, 3)
    _one(r"if \(rounds\(192\) \* 3 <= rounds\(128\) \* 2\)", s, "48-row form rule")
    _one(r"const int64_t rb = \(\(M \+ tiles - 1\) / tiles \+ 15\) / 16 \* 16;", s, "gdx_row_tile")
    _one(r"const int64_t slots = 2 \* static_cast<int64_t>\(num_cus\(\)\);", s, "two blocks per CU")
    assert bm.GDX_SLOTS == 2 * 256


def test_mask_dz_ring_and_instances():
    s = _src("mask_dz.hip")
    assert _const("kDzStages", "mask_dz.hip") == 4
    assert set(re.findall(r"return launch<T, (\d+), (\d+)>", s)) == {("12", "2"), ("8", "2")}
    # the replay's block cost: K chunks + 5
    _one(r"\[&\]\(int b\) \{ return \(2 \* dim_inputs\[b\] \+ 31\) / 32 \+ 5; \}", s, "dz block cost")
    src_replay = Path(bm.__file__).read_text()
    assert "lambda b: cdiv(2 * widths[b], 32) + 5" in src_replay
    assert "S, HT = 4, 16 * DT" in src_replay


def test_mask_estimator_dpre_and_dw_rules():
    s = _src("mask_estimator.hip")
    assert _const("kDpreFlatRows", "mask_estimator.hip") == 4
    assert _const("kDpreFlatMaxBands", "mask_estimator.hip") == 4096
    m = _one(r"ring128 = (\d+) \* kChunkK \* 2 \* \(64 \+ 128\), ring192 = (\d+) \* kChunkK \* 2 \* \(64 \+ 192\)",
             s, "dW ring sizes")
    assert m.groups() == ("3", "3")
    _one(r"const int jt = rounds\(192, ring192\) < rounds\(128, ring128\) \? 192 : 128;", s, "dW tile rule")
    assert bm.dw_jt(62, 192, 768) == 192


def test_band_split_dw_ring():
    assert _define("PMSST_BS_DWD_STAGES", "band_split.hip") == 3
    assert _define("PMSST_BS_DWD_KS", "band_split.hip") == 2
    assert "S, KS = 3, 2" in Path(bm.__file__).read_text()


@pytest.mark.parametrize("mistake", ["table", "constant"])
def test_a_planted_mismatch_is_caught(monkeypatch, mistake):
    """A replay table or constant that no longer matches the source fails the checks above."""
    if mistake == "table":
        monkeypatch.setitem(bm.MLP_TILES, 192, (6, 2, 4))
        with pytest.raises(AssertionError):
            test_mask_mlp_tile_table_and_ring()
    else:
        monkeypatch.setattr(bm, "CHUNK_K", 64)
        with pytest.raises(AssertionError):
            test_shared_constants()


def test_fp32_split_rules_and_tiles():
    """gemm.h kSplitRow, kSplitMacs, gemm_lds_elems; the launchers' rules in band_split.hip and
    mask_estimator.hip."""
    assert _const("kSplitRow", "gemm.h") == bm.SPLIT_ROW
    m = _one(r"constexpr int64_t kSplitMacs = ([\d']+);", _src("gemm.h"), "kSplitMacs")
    assert int(m.group(1).replace("'", "")) == bm.SPLIT_MACS
    _one(r"return SPLIT \? \(BR \+ BC\) \* kSplitRow : 2 \* \(BR \+ BC\) \* LdsPitch<T>::value;", _src("gemm.h"), "LDS")
    s = _src("band_split.hip")
    _one(r"constexpr int dw_cols\(bool norm, bool split\) \{ return split && !norm \? 128 : 64; \}", s, "dW columns")
    _one(r"return split_macs\(M, hb\.F, O\) && blocks >= num_cus\(\);", s, "dW rule")
    _one(r"if \(split_macs\(a\.vec4 \? M : M / 2, hb\.F, O\)\) launch\(std::true_type\{\}\);", s, "forward rule")
    _one(r"kF32 && v4 && split_macs\(M, hb\.F, O\) && M > 64 && 5 \* split_blocks >= int64_t\{6\} \* num_cus\(\);", s,
         "grouped dx rule")
    _one(r"const bool split = kF32 && v4 && split_macs\(M, hb\.F, O\);", s, "band split dx rule")
    _one(r"\(M \+ 63\) / 64 \* chunks >= int64_t\{2\} \* 7 \* num_cus\(\)", s, "mixed 128-row rule")
    s = _src("mask_estimator.hip")
    _one(r"kF32 && a\.vec4 && split_macs\(M, 2 \* static_cast<int64_t>\(hm\.F\), H\);", s, "mask backward rule")
    _one(r"if \(kF32 && split_macs\(M, 2 \* static_cast<int64_t>\(hm\.F\), H\)\) \{", s, "mask forward rule")


def test_wide_grouped_tiles_and_rules():
    """grouped_gemm.hip: waves, stages, tiles and the dispatch rules; mask_mlp.hip's choice of form."""
    s = _src("grouped_gemm.hip")
    _one(r"return op == kGgFwd \? 4 : 8; \}", s, "waves")
    _one(r"constexpr int NW = gg_waves\(OP\), S = NW == 8 \? 4 : 3;", s, "stages")
    _one(r"constexpr int WB = NW / WA, TB = 4;", s, "B tiles")
    _one(r"% 256 == 0\) return launch<T, OP, 8, 2>\(a, stream\);\s+return launch<T, OP, 6, 2>\(a, stream\);", s, "tiles")
    assert bm.gg_tile("dx", 512, 64) == (8, 4, 8, 256, 256) and bm.gg_tile("fwd", 64, 192) == (4, 3, 6, 192, 128)
    _one(r"const int64_t quarters = groups >= 24 \? 11 : 16;", s, "dx rule")
    _one(r"return groups \* rows \* in_features >= quarters \* 1024 \* num_cus\(\);", s, "dx rule")
    _one(r"\(in_features == 192 \|\| in_features == 256\) && 5 \* blocks >= 4 \* rounds \* cus;", s, "dx rule at 192, 256")
    _one(r"if \(a_cols == 256\) return other >= 6 \* rounds \* cus && rows >= 64;", s, "dW rule, 256 wide")
    _one(r"\(other >= 6 \* rounds \* cus && rows > 128\) \|\| \(2 \* other >= 9 \* rounds \* cus && rows >= 1400\);", s,
         "dW rule, 192 wide")
    _one(r"return other >= 5 \* rounds \* cus && rows \* other >= 2000 \* rounds \* cus;", s, "dW rule, no whole 64s")
    _one(r"return out_features >= 128 && shape_ok\(", s, "tanh rule")
    s = _src("mask_mlp.hip")
    _one(r"if \(dim >= 384\) return true;", s, "two kernels")
    _one(r"return passes > 2 \* band_count && \(dim >= 256 \|\| rows > \(dim <= 64 \? 768 : 256\)\);", s, "two kernels")


def test_matrix_core_gate_rules():
    s = _src("attn_gate.hip")
    _one(r"return work >= 4096 \|\| rows >= 16384 \|\| \(rows >= 8192 && work >= 1024\);", s, "forward rule")
    _one(r"return work >= 1536 \|\| \(work >= 1024 && s\.rows\(\) >= 2000\);", s, "backward rule")
    _one(r"\(nt <= 4 \|\| nt == 6 \|\| nt == 8\)", s, "dims")
    assert _const("kGateBwdMaxBlocks", "attn_gate.hip") == 1024
    _one(r"std::min<int64_t>\(2 \* static_cast<int64_t>\(num_cus\(\)\), kGateBwdMaxBlocks\)", s, "backward blocks")
