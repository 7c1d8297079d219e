"""The tiles for row counts between 64 and 256 (gemm_reg_mid.hip) and the
dispatch that picks them (gemm_cost.h): each tile at its row edges against the
oracle, one pass and split; shapes on both sides of the dispatch's lines; and
a split choice under graph capture, where the workspace cannot grow."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as O
from tests.conftest import announce
from tests.mx_inputs import allclose_report, bf16_operand, mxfp4_operand, mxfp8_operand

pytestmark = pytest.mark.gpu

TILES = ([("a16w16", f"a16w16_tile_{t}{{}}{s}", bm) for bm, t in ((96, "96x128"), (160, "160x128"),
                                                                 (128, "128x64")) for s in ("_bplain", "")] +
         [("a4w4", f"a4w4_tile_{t}{{}}", bm) for bm, t in ((32, "32x128"), (96, "96x128"), (128, "128x64"),
                                                           (192, "192x128"))] +
         [("a8w4", f"a8w4_tile_{t}{{}}", bm) for bm, t in ((32, "32x128"), (96, "96x128"), (128, "128x64"))])


def _dev(x, cuda):
    return torch.from_numpy(np.ascontiguousarray(x)).to(cuda)


def _case(fam, m, n, k, cuda, shuffled=True):
    """(call(name, split) -> out, reference)."""
    from aiter_amd._lib import call

    if fam == "a16w16":
        a, b = bf16_operand(m, k, 5), bf16_operand(n, k, 6)
        ref = O.bf16_bits_to_f32(O.gemm_a16w16_ref(a, b))
        w = O.shuffle_weight(b) if shuffled else b
        A, B = (torch.from_numpy(v.view(np.int16).copy()).to(cuda).view(torch.bfloat16) for v in (a, w))
        sa = sb = None
    else:
        q, s, ss = (mxfp4_operand if fam == "a4w4" else mxfp8_operand)(m, k, 5, *(("triton",) if fam == "a4w4" else ()))
        bq, bs, bss = mxfp4_operand(n, k, 6, "triton")
        ref = O.bf16_bits_to_f32((O.gemm_a4w4_ref if fam == "a4w4" else O.gemm_a8w4_ref)(q, bq, s, bs))
        A, B, sa, sb = _dev(q, cuda), _dev(O.shuffle_weight(bq), cuda), _dev(ss, cuda), _dev(bss, cuda)

    def run(name, split, out):
        if fam == "a16w16":
            call("gemm_a16w16_asm", A, B, out, None, None, split, name, int(shuffled))
        elif fam == "a4w4":
            call("gemm_a4w4_asm", A, B, sa, sb, out, name, None, 1.0, 0.0, 1, {0: 0, 2: 1}[split])
        else:
            call("mxfp8_mxfp4_gemm_asm", A, B, sa, sb, out, name, 0)

    return run, ref


@pytest.mark.parametrize("fam,name,bm", TILES, ids=[t[1] for t in TILES])
@pytest.mark.parametrize("edge", [-1, 0, 1])
def test_tile_row_edges(cuda, fam, name, bm, edge):
    m, n, k = bm + edge, 144, 64 * 9 if fam == "a16w16" else 256 * 9
    run, ref = _case(fam, m, n, k, cuda, "_bplain" not in name)
    for split in (0, 2):
        nm = name.format("_splitk" if split else "")
        announce(f"{nm} {m}x{n}x{k} split {split}")
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=cuda)
        run(nm, split, out)
        torch.cuda.synchronize()
        ok, msg = allclose_report(out.float().cpu().numpy(), ref)
        assert ok, f"{nm}: {msg}"


# (m, n, k): both sides of 16, 32 and 64 rows; grids that split K; a 32-column
# skinny grid of exactly one round; rows that no tile divides
SHAPES = [(16, 256, 1024), (17, 8192, 512), (33, 256, 3584), (64, 1088, 2560), (65, 1088, 2560), (150, 512, 7168),
          (97, 4096, 1280), (161, 2048, 768), (300, 3072, 768), (600, 7168, 512)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("fam", ["a16w16", "a16w16_pre", "a4w4", "a8w4"])
def test_dispatch_shapes(cuda, fam, m, n, k):
    announce(f"dispatch {fam} {m}x{n}x{k}")
    run, ref = _case(fam.split("_")[0], m, n, k, cuda, fam != "a16w16")
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=cuda)
    run(None, 0, out)
    torch.cuda.synchronize()
    ok, msg = allclose_report(out.float().cpu().numpy(), ref)
    assert ok, msg


# both sides of the K from which up to 32 rows are split, per family and rows
@pytest.mark.parametrize("fam,m,n,k", [("a16w16_pre", 9, 80, 7104), ("a16w16_pre", 9, 80, 7168), ("a16w16", 32, 80, 12224),
                                       ("a16w16", 32, 80, 12288), ("a16w16", 16, 80, 12288), ("a16w16", 16, 80, 14336),
                                       ("a4w4", 7, 80, 16128), ("a4w4", 7, 80, 16384), ("a4w4", 25, 80, 16384),
                                       ("a8w4", 16, 80, 16384), ("a8w4", 17, 80, 16384)])
def test_skinny_split_lines(cuda, fam, m, n, k):
    test_dispatch_shapes(cuda, fam, m, n, k)


@pytest.mark.parametrize("m,n,k", [(1, 16, 1024), (16, 80, 2048), (17, 80, 2048), (32, 256, 7168)])
def test_skinny_f32_split_error(cuda, m, n, k):
    """f32 output up to 32 rows, K split where it is long: the sums stay within a
    chain of K / 256 f32 roundings (8 waves, 32 products per step) plus the 8 + 8
    that add the waves and the splits."""
    from aiter_amd import tgemm

    announce(f"skinny f32 {m}x{n}x{k}")
    x = torch.randn(m, k, device=cuda, dtype=torch.bfloat16)
    w = torch.randn(n, k, device=cuda, dtype=torch.bfloat16)
    got = tgemm.mm(x, w, None, otype=torch.float32).double().cpu()
    x, w = x.double().cpu(), w.double().cpu()
    bound = (k / 256 + 16) * 2.0 ** -24 * (x.abs() @ w.abs().t())
    assert ((got - x @ w.t()).abs() <= bound).all()


def test_split_choice_under_capture(cuda):
    """A shape for which the dispatch splits K eagerly: captured on a stream
    without a workspace it runs without the split, and replays give that result."""
    from aiter_amd._lib import lib

    m, n, k = 150, 4096, 14336
    announce(f"dispatch under capture {m}x{n}x{k}")
    run, ref = _case("a16w16", m, n, k, cuda, False)
    st = torch.cuda.Stream()
    out = torch.empty((m, n), dtype=torch.bfloat16, device=cuda)
    with torch.cuda.stream(st):
        run(None, 0, out)
        st.synchronize()
        assert lib().aiter_amd_workspace_bytes(out.device.index, st.cuda_stream) > 0, "expected a split choice"
        assert lib().aiter_amd_workspace_release(out.device.index, st.cuda_stream) == 0
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            run(None, 0, out)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        ok, msg = allclose_report(out.float().cpu().numpy(), ref)
        assert ok, msg
