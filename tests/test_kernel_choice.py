"""What the dispatch runs for a call, on the CPU: the names it knows, a tuned
row's kernel, and the instance and split count that the library chooses."""
import math
import os
import random
import re

import pandas as pd
import pytest
import torch

from aiter_amd import config, fused_gemm, gemm_op_a4w4, gemm_op_a8w4, tuned_gemm, tuner
from aiter_amd._lib import gemm_choice, instance_table, kernel_names, kernel_table
from aiter_amd.csrc import build
from tests.test_dispatch import _clear, _row, gfx950  # noqa: F401


def _unlisted():
    try:
        return [r[1] for r in instance_table()[len(kernel_table()):]]
    except RuntimeError:   # not built
        return []


UNLISTED = _unlisted()


def test_instances_outside_the_table():
    """The 96-, 160- and 192-row tiles follow the kernel table's ids."""
    assert instance_table()[:len(kernel_table())] == tuple(kernel_table())
    assert {r[4] for r in instance_table()[len(kernel_table()):]} == {96, 160, 192}
    assert set(UNLISTED) <= kernel_names()


@pytest.mark.parametrize("name", [n for n in UNLISTED if n.startswith("a4w4")])
def test_row_naming_an_instance_outside_the_table(name, tmp_path, monkeypatch, gfx950):
    """A caller's row with such a name runs that kernel with the call's bias,
    alpha and beta (a name the library does not know goes to the CK entry, which
    has none of them)."""
    p = tmp_path / "t.csv"
    pd.DataFrame([_row(300, 512, 512, name, split=1)]).to_csv(p, index=False)
    monkeypatch.setenv("AITER_CONFIG_GEMM_A4W4", str(p))
    _clear()
    seen = []
    monkeypatch.setattr(gemm_op_a4w4, "call", lambda *a: seen.append(a))
    a, w = torch.zeros(300, 256, dtype=torch.uint8), torch.zeros(512, 256, dtype=torch.uint8)
    s = torch.zeros(512, 16, dtype=torch.uint8)
    bias = torch.ones(512)
    gemm_op_a4w4.gemm_a4w4(a, w, s, s, bias=bias, alpha=0.5, beta=2.0)
    (entry, *args), = seen
    assert entry == "gemm_a4w4_asm"
    assert args[5] == name and args[6] is bias and args[7:11] == [0.5, 2.0, 1, 1]
    assert fused_gemm._tuned_a4w4(300, 512, 512, True) == name


def test_tuner_sees_every_instance():
    names = {n for fam in ("a4w4", "a8w4", "a16w16") for pre in (False, True)
             for _, n, _ in tuner.candidates(fam, 150, pre)}
    assert set(UNLISTED) <= names


@pytest.mark.parametrize("fam,m,n,k", [("a16w16", 43, 512, 3904), ("a8w4", 36, 2064, 15616)])
def test_more_splits_of_the_base_instance(fam, m, n, k):
    """The time model's answer may be the simple rule's own split tile with
    another count: here 8 splits, where the rule's count is 4."""
    name, splits = gemm_choice(fam, m, n, k)
    assert "splitk" in name and splits == 8
    assert gemm_choice(fam, m, n, k, kernel_name=name)[1] == 4   # by name: the launcher's own count


def _shapes(n=400, seed=3):
    rng = random.Random(seed)
    log_int = lambda lo, hi, step: max(step, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) // step * step)
    for i in range(n):
        fam, kw = [("a16w16", {"b_pre": False}), ("a16w16", {}), ("a4w4", {}), ("a8w4", {})][i % 4]
        yield fam, kw, log_int(17, 4096, 1), log_int(64, 16384, 16), log_int(512, 28672, 256)


def _base(fam, m, n, k, kw):
    """(name, splits) of the simple rule, which a call with a split request takes as it is"""
    name = gemm_choice(fam, m, n, k, splits=1, **kw)[0]
    return name, gemm_choice(fam, m, n, k, kernel_name=name, **kw)[1] if "splitk" in name else 1


def test_workspace_of_a_choice():
    """Eagerly a choice asks for 64 MiB of partials at most (or what the simple
    rule asks for).  Under capture it is the eager one if the stream holds its
    bytes; otherwise one that needs no more than the simple rule's, and the same
    whatever the stream holds."""
    changed = 0
    for fam, kw, m, n, k in [("a16w16", {"b_pre": False}, 896, 5488, 27968), *_shapes()]:
        need = lambda c: c[1] * m * n * 4 if "splitk" in c[0] and c[1] > 1 else 0
        base = need(_base(fam, m, n, k, kw)) if m > 32 else 0
        eager = gemm_choice(fam, m, n, k, **kw)
        if "skinny" in eager[0]:
            continue
        assert need(eager) <= max(base, 64 << 20)
        assert gemm_choice(fam, m, n, k, held=max(base, 64 << 20), **kw) == eager
        assert gemm_choice(fam, m, n, k, held=need(eager), **kw) == eager
        if need(eager):
            others = {gemm_choice(fam, m, n, k, held=h, **kw) for h in (0, need(eager) // 2, need(eager) - 1)}
            assert len(others) == 1 and need(others.pop()) <= base
            changed += 1
    assert changed > 40


def _chain(choice, k):
    """K that one f32 accumulator sums in a row (the 8 waves of a skinny kernel share K)"""
    stages = -(-(k // 64) // choice[1])
    return -(-stages // 8) if "skinny" in choice[0] else stages


def test_f32_chains_are_no_longer_than_the_simple_rules():
    """f32 outputs: no choice sums K in longer chains than the simple rule's."""
    log_int = lambda rng, lo, hi, step: max(step, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) // step * step)
    rng = random.Random(9)
    shapes = [(4009, 128, 1472)] + [(log_int(rng, 17, 4096, 1), log_int(rng, 32, 512, 16), log_int(rng, 1024, 8192, 64))
                                    for _ in range(400)]
    for m, n, k in shapes:
        for pre in (False, True):
            kw = {"b_pre": pre, "out_f32": True}
            base = gemm_choice("a16w16", m, n, k, splits=1, **kw)[0]
            base = gemm_choice("a16w16", m, n, k, kernel_name=base, **kw)
            choice = gemm_choice("a16w16", m, n, k, **kw)
            if "splitk" in choice[0] and "skinny" in choice[0]:
                continue   # the skinny rule's own split
            assert _chain(choice, k) <= _chain(base, k), (m, n, k, base, choice)


def test_bf16_up_to_32_rows_is_the_skinny_rules():
    log_int = lambda rng, lo, hi, step: max(step, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) // step * step)
    rng = random.Random(4)
    for _ in range(300):
        m, n, k = rng.randint(1, 32), log_int(rng, 32, 16384, 16), log_int(rng, 512, 28672, 64)
        for kw in ({"b_pre": False}, {"b_pre": True}, {"b_pre": False, "out_f32": True}):
            base = gemm_choice("a16w16", m, n, k, splits=1, **kw)[0]
            assert gemm_choice("a16w16", m, n, k, **kw)[0] == base


@pytest.mark.parametrize("m,n,k,row,splits,keeps", [
    (1132, 8192, 28672, "a16w16_tile_256x256_bplain_flat", 0, None),    # 545 us, with 4 splits of 256x128 565
    (150, 14336, 4096, "a16w16_tile_128x128_bplain", 0, True),          # 96x128 within 2 % either way
    (1275, 4096, 4096, "a16w16_tile_256x128_bplain", 0, False),         # 52.7 us, 160x128 42.7
    (145, 8192, 28672, "a16w16_tile_256x128_splitk_bplain", 4, False),  # 115.7 us, 160x128 100.6
])
def test_what_replaces_a_tuned_rows_tile(m, n, k, row, splits, keeps):
    """"~row": an unsplit tile gives way to an unsplit one and a split one to a
    split one, where the model puts it clearly ahead; by its plain name a kernel
    always runs."""
    kw = {"b_pre": False, "splits": splits}
    assert gemm_choice("a16w16", m, n, k, kernel_name=row, **kw)[0] == row
    choice = gemm_choice("a16w16", m, n, k, kernel_name="~" + row, **kw)
    assert keeps is None or (choice[0] == row) == keeps
    assert ("splitk" in choice[0]) == ("splitk" in row)


def _costs():
    """{instance: stage time} of gemm_cost.h, the tiles by (family, split form, row-major)"""
    text = open(os.path.join(build.HERE, "gemm_cost.h")).read()
    out = {}
    for name, stage in re.findall(r'\{"([a-z0-9_]+)", ([\d.e-]+),', text):
        m = re.fullmatch(r"(a\d+w\d+)_tile_(\d+)x(\d+)(_splitk)?(_bplain)?", name)
        if m:
            out[(m[1], bool(m[4]), bool(m[5]), int(m[2]), int(m[3]))] = float(stage)
    return out


def test_cost_table_is_plausible():
    """A larger tile's stage takes no less time than a smaller one's of the same
    form (5 % for the fit), and the forms for the two weight orders of one t32
    tile, which move the same bytes, are within 25 %."""
    costs = _costs()
    assert len(costs) > 50
    for a, ta in costs.items():
        for b, tb in costs.items():
            if a[:3] == b[:3] and a[3] <= b[3] and a[4] <= b[4]:
                assert tb >= 0.95 * ta, (a, ta, b, tb)
        twin = (*a[:2], False, *a[3:])
        if a[2] and twin in costs and not (a[3] >= 128 and a[4] == 256):
            assert 0.8 <= ta / costs[twin] <= 1.25, (a, ta, costs[twin])


TABLES = {"a4w4": ("AITER_CONFIG_GEMM_A4W4", gemm_op_a4w4.get_GEMM_config),
          "a8w4": ("AITER_CONFIG_GEMM_A8W4", gemm_op_a8w4.get_GEMM_A8W4_config),
          "a16w16": ("AITER_CONFIG_GEMM_BF16", lambda m, n, k: tuned_gemm.get_GEMM_A16W16_config(
              m, n, k, False, "torch.bfloat16", "torch.bfloat16"))}


def _table(fam, rows):
    """a tuned CSV of the family with (M, N, K, kernel) rows"""
    extra = {"bias": False, "dtype": "torch.bfloat16", "outdtype": "torch.bfloat16", "scaleAB": False,
             "bpreshuffle": False, "libtype": "aiter_amd", "solidx": 1} if fam == "a16w16" else {}
    return pd.DataFrame([{**_row(m, n, k, name), **extra} for m, n, k, name in rows])


@pytest.mark.parametrize("fam", TABLES)
@pytest.mark.parametrize("shipped", [True, False])
def test_rows_tuned_for_other_row_counts(fam, shipped, tmp_path, monkeypatch, gfx950):
    """A shipped row above 64 rows that serves a call of 1/1.25 of its rows or
    fewer is handed on as "~name"; a row of the caller's own list by its name."""
    name = f"{fam}_tile_128x128" + ("_bplain" if fam == "a16w16" else "")
    path = tmp_path / "t.csv"
    _table(fam, [(512, 512, 512, name), (64, 512, 512, name)]).to_csv(path, index=False)
    env, lookup = TABLES[fam]
    if shipped:
        monkeypatch.delenv(env, raising=False)
        for mod in (gemm_op_a4w4, gemm_op_a8w4, tuned_gemm):
            for const in ("DEFAULT_A4W4_CSV", "DEFAULT_A8W4_CSV", "DEFAULT_BF16_CSV"):
                if hasattr(mod, const):
                    monkeypatch.setattr(mod, const, str(path))
    else:
        monkeypatch.setenv(env, str(path))
    _clear()
    for m, rows in ((512, 512), (410, 512), (409, 512), (257, 512), (64, 64), (33, 64)):
        row = lookup(m, 512, 512)
        assert row["kernelName"] == name and row.rows == (rows if shipped else m)
        assert config.row_kernel(row, m) == ("~" if shipped and rows == 512 and m <= 409 else "") + name


@pytest.mark.parametrize("shipped", [True, False])
def test_the_call_takes_the_hint(shipped, tmp_path, monkeypatch, gfx950):
    """The three entries pass the row's kernel on as row_kernel writes it."""
    m, mark, seen = 300, "~" if shipped else "", []
    for fam, mod in (("a4w4", gemm_op_a4w4), ("a8w4", gemm_op_a8w4), ("a16w16", tuned_gemm)):
        name = f"{fam}_tile_128x128" + ("_bplain" if fam == "a16w16" else "")
        path = tmp_path / f"{fam}.csv"
        _table(fam, [(512, 512, 512, name)]).to_csv(path, index=False)
        if shipped:
            monkeypatch.delenv(TABLES[fam][0], raising=False)
            const = {"a4w4": "DEFAULT_A4W4_CSV", "a8w4": "DEFAULT_A8W4_CSV", "a16w16": "DEFAULT_BF16_CSV"}[fam]
            monkeypatch.setattr(mod, const, str(path))
        else:
            monkeypatch.setenv(TABLES[fam][0], str(path))
        monkeypatch.setattr(mod, "call", lambda *a: seen.append(a))
    _clear()
    u8 = lambda r, c: torch.zeros(r, c, dtype=torch.uint8)
    gemm_op_a4w4.gemm_a4w4(u8(m, 256), u8(512, 256), u8(512, 16), u8(512, 16))
    gemm_op_a8w4.gemm_a8w4_mxfp8(u8(m, 512), u8(512, 256), u8(512, 16), u8(512, 16), a_preshuffle=False)
    tuned_gemm.tgemm.mm(torch.zeros(m, 512, dtype=torch.bfloat16), torch.zeros(512, 512, dtype=torch.bfloat16))
    assert [next(x for x in a[1:] if isinstance(x, str)) for a in seen] == [
        mark + "a4w4_tile_128x128", mark + "a8w4_tile_128x128", mark + "a16w16_tile_128x128_bplain"]


@pytest.mark.parametrize("fam,m,n,k,kw,choice", [
    ("a4w4", 43, 4096, 4096, {}, "a4w4_skinny_m64_n32_alds"), ("a4w4", 150, 14336, 4096, {}, "a4w4_tile_96x128"),
    ("a8w4", 300, 7168, 16384, {}, "a8w4_tile_96x128"),
    ("a16w16", 600, 7168, 2048, {"b_pre": False}, "a16w16_tile_160x128_bplain"),
    ("a16w16", 150, 4096, 14336, {"b_pre": False}, "a16w16_tile_160x128_splitk_bplain"),
    ("a16w16", 4001, 4096, 14336, {"b_pre": False}, "a16w16_tile_256x256_bplain_flat"),
])
def test_instance_chosen(fam, m, n, k, kw, choice):
    """Calls whose choice is not the simple rule's tile, by instance; with a
    split request or a kernel named the model has no say."""
    base = gemm_choice(fam, m, n, k, splits=1, **kw)[0]
    got = gemm_choice(fam, m, n, k, **kw)[0]
    assert got == choice != base
    assert gemm_choice(fam, m, n, k, kernel_name=base, **kw)[0] == base
