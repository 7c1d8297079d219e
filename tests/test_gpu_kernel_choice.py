"""The choices of the dispatch as the GPU runs them: split counts through the
workspace that a call leaves, and results against the oracle."""
import numpy as np
import pytest
import torch

from aiter_amd._lib import call, gemm_choice, lib
from oracle import mx_oracle as O
from tests.conftest import announce
from tests.mx_inputs import allclose_report, bf16_operand

pytestmark = pytest.mark.gpu


def _bf16_case(m, n, k, cuda, shuffled):
    a, b = bf16_operand(m, k, 5), bf16_operand(n, k, 6)
    ref = O.bf16_bits_to_f32(O.gemm_a16w16_ref(a, b))
    w = O.shuffle_weight(b) if shuffled else b
    A, B = (torch.from_numpy(v.view(np.int16).copy()).to(cuda).view(torch.bfloat16) for v in (a, w))
    return A, B, ref


@pytest.mark.parametrize("m,n,k", [(43, 512, 3904), (70, 256, 4096)])
def test_choice_is_what_runs(cuda, m, n, k):
    """A split choice leaves its partials' bytes in a released stream's workspace."""
    announce(f"dispatch choice {m}x{n}x{k}")
    name, splits = gemm_choice("a16w16", m, n, k)
    assert "splitk" in name and splits > 1
    A, B, ref = _bf16_case(m, n, k, cuda, True)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=cuda)
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        assert lib().aiter_amd_workspace_release(0, st.cuda_stream) == 0
        call("gemm_a16w16_asm", A, B, out, None, None, 0, None, 1)
    torch.cuda.synchronize()
    assert lib().aiter_amd_workspace_bytes(0, st.cuda_stream) == splits * m * n * 4
    ok, msg = allclose_report(out.float().cpu().numpy(), ref)
    assert ok, msg


def test_reserved_capture_runs_the_eager_kernel(cuda):
    """With 64 MiB reserved a captured call runs the split that the eager call
    runs, bit for bit; the same call captured with a few bytes held runs the form
    without a workspace that it runs with none."""
    import aiter_amd

    m, n, k = 150, 4096, 14336
    announce(f"captured choice {m}x{n}x{k}")
    assert gemm_choice("a16w16", m, n, k, b_pre=False)[1] > 1
    A, B, ref = _bf16_case(m, n, k, cuda, False)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=cuda)
    st = torch.cuda.Stream()

    def run():
        call("gemm_a16w16_asm", A, B, out, None, None, 0, None, 0)
        return out

    def captured(prepare):
        with torch.cuda.stream(st):
            assert lib().aiter_amd_workspace_release(0, st.cuda_stream) == 0
            prepare()
            st.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=st):
                run()
            res = []
            for _ in range(3):
                out.fill_(float("nan"))
                g.replay()
                st.synchronize()
                res.append(out.clone())
        torch.cuda.synchronize()
        assert all(torch.equal(r, res[0]) for r in res)
        return res[0]

    with torch.cuda.stream(st):
        eager = run().clone()
    reserved = captured(aiter_amd.opus_gemm_workspace_init)
    assert torch.equal(reserved, eager)
    none = captured(lambda: None)
    few = captured(lambda: lib().gemm_workspace_reserve(0, st.cuda_stream, 4 * m * n * 4))
    assert torch.equal(none, few)
    for got in (eager, none):
        ok, msg = allclose_report(got.float().cpu().numpy(), ref)
        assert ok, msg


def test_graph_keeps_the_workspace_it_was_captured_with(cuda):
    """A larger split call on the stream gets another block; the graph's replays
    still write to theirs, whatever has been allocated since."""
    m, n, k = 64, 1024, 1280
    announce(f"captured workspace outgrown {m}x{n}x{k}")
    A, B, _ = _bf16_case(m, n, k, cuda, False)
    big = [t.repeat(8, 1) for t in (A, B)]
    out = torch.empty((m, n), dtype=torch.bfloat16, device=cuda)
    out_big = torch.empty((8 * m, 8 * n), dtype=torch.bfloat16, device=cuda)
    st = torch.cuda.Stream()
    name = "a16w16_tile_64x64_splitk_bplain"
    with torch.cuda.stream(st):
        assert lib().aiter_amd_workspace_release(0, st.cuda_stream) == 0
        call("gemm_a16w16_asm", A, B, out, None, None, 4, name, 0)
        eager = out.clone()
        st.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            call("gemm_a16w16_asm", A, B, out, None, None, 4, name, 0)
        held = lib().aiter_amd_workspace_bytes(0, st.cuda_stream)
        call("gemm_a16w16_asm", *big, out_big, None, None, 4, name, 0)
        assert lib().aiter_amd_workspace_bytes(0, st.cuda_stream) == 64 * held
        other = [torch.full((held // 4,), 7.0, device=cuda) for _ in range(16)]
        for _ in range(3):
            out.fill_(float("nan"))
            g.replay()
            st.synchronize()
            assert torch.equal(out, eager)
        assert all(bool((t == 7.0).all()) for t in other)
    torch.cuda.synchronize()
    assert torch.equal(out_big[:m, :n], eager)
    assert lib().aiter_amd_workspace_release(0, st.cuda_stream) == 0


@pytest.mark.parametrize("m,n,k", [(40, 512, 3904), (100, 128, 1024), (1500, 256, 1984), (4009, 128, 1472)])
def test_f32_error_above_32_rows(cuda, m, n, k):
    """f32 output: the error of the dispatch's choice is that of the simple
    rule's kernel, whose chains of f32 roundings it may not exceed (2 % for the
    roundings' signs, over some thousand outputs)."""
    from aiter_amd import tgemm

    announce(f"f32 error {m}x{n}x{k}")
    kw = {"b_pre": False, "out_f32": True}
    base = gemm_choice("a16w16", m, n, k, splits=1, **kw)[0]
    splits = gemm_choice("a16w16", m, n, k, kernel_name=base, **kw)[1]
    x = torch.randn(m, k, device=cuda, dtype=torch.bfloat16)
    w = torch.randn(n, k, device=cuda, dtype=torch.bfloat16)
    ref = x.double().cpu() @ w.double().cpu().t()
    out = torch.empty((m, n), dtype=torch.float32, device=cuda)
    call("gemm_a16w16_asm", x, w, out, None, None, splits if "splitk" in base else 0, base, 0)
    err = lambda got: ((got.double().cpu() - ref).norm() / ref.norm()).item()
    by_rule, by_choice = err(out), err(tgemm.mm(x, w, None, otype=torch.float32))
    print(f"[error] {by_rule:.3g} {base} x{splits}, {by_choice:.3g} {gemm_choice('a16w16', m, n, k, **kw)}", flush=True)
    assert by_choice <= 1.02 * by_rule
