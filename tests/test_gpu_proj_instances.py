"""Every variant of the projection kernels once, at the shapes of proj_instances.py: against the definition in 64 bits, with
nothing written past the outputs, and a row's bits those it has in other company."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import proj_instances as inst  # noqa: E402
from hipml_amd import attn  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def _init():
    attn.init(0)


def inputs(m, k, rows):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m * 1_000_003 + k * 131 + rows)
    q = torch.randint(-128, 128, (m, k // 32, 32), device="cuda", dtype=torch.int8, generator=gen)
    d = (torch.rand((m, k // 32, 1), device="cuda", generator=gen) * 0.05 + 0.001).to(torch.float16)
    w = torch.cat((d.view(torch.uint8), q.view(torch.uint8)), dim=2).contiguous()
    return w, d, q, torch.randn((rows, k), device="cuda", generator=gen) * 0.25


def padded(rows, m):
    return torch.full((rows + 1, m), float("nan"), device="cuda")


@pytest.mark.parametrize("m,k,rows", inst.ROWS)
def test_row_kernel(m, k, rows):
    w, d, q, x = inputs(m, k, rows)
    y = padded(rows, m)
    attn.gemv_q8_0_rows(w, x, y, m, k, rows)
    assert bool(y[rows].isnan().all())
    exact = x.double() @ (d.double() * q.double()).reshape(m, k).T
    err = (y[:rows] - exact).abs().max().item()
    # activations to ~22 bits (24 of their block's largest up to eight rows), fp32 sums over eight chains or up to twelve waves
    assert err <= 2e-6 * exact.abs().max().item() * max(1.0, (k / 8192) ** 0.5) + 1e-5, err
    # the last row among others: the same bits where those take kernels of the same class
    kernel = inst.row_kernel(m, k, rows) // 1_000_000
    for more in (2 * rows, rows + 9, 128):
        if more <= 128 and more > rows and inst.row_kernel(m, k, more) // 1_000_000 == kernel:
            company = torch.cat((torch.randn((more - 1, k), device="cuda"), x[-1:]))
            z = padded(more, m)
            attn.gemv_q8_0_rows(w, company, z, m, k, more)
            assert torch.equal(z[more - 1], y[rows - 1]) and bool(z[more].isnan().all())


@pytest.mark.parametrize("m,k,rows", inst.WIDE)
def test_rows_by_wide_requests(m, k, rows):
    assert inst.row_variant(m, k, rows)[1]
    w, d, q, x = inputs(m, k, rows)
    y = padded(rows, m)
    attn.gemv_q8_0_rows(w, x, y, m, k, rows)
    assert bool(y[rows].isnan().all())
    exact = x.double() @ (d.double() * q.double()).reshape(m, k).T
    err = (y[:rows] - exact).abs().max().item()
    assert err <= 2e-6 * exact.abs().max().item() + 1e-5, err  # as test_row_kernel, k below 8,192
    for first, n in ((0, 9), (rows - 9, 9), (0, rows - 1)):    # a row's bits, whichever tile its company takes
        if n > 8:
            z = padded(n, m)
            attn.gemv_q8_0_rows(w, x[first:first + n], z, m, k, n)
            assert torch.equal(z[:n], y[first:first + n]) and bool(z[n].isnan().all())
    bad = x.clone()                                            # infinite in one row: its own results only
    bad[rows // 2, k - 3] = float("inf")
    z = padded(rows, m)
    attn.gemv_q8_0_rows(w, bad, z, m, k, rows)
    others = [i for i in range(rows) if i != rows // 2]
    assert torch.equal(z[others], y[others]) and not bool(z[rows // 2].isfinite().any())


@pytest.mark.parametrize("m,k,tokens,x16", inst.TILES)
def test_tile(m, k, tokens, x16):
    w, d, q, x = inputs(m, k, tokens)
    h = x.to(torch.float16)
    y, one = padded(tokens, m), padded(1, m)
    if x16:
        attn.output_chunk_q8_0(w, None, None, y, m, k, tokens, h)
    else:
        attn.gemm_q8_0_f16(w, x, y, m, k, tokens)
    attn.gemm_q8_0_f16(w, x[tokens // 2:], one, m, k, 1)
    assert bool(y[tokens].isnan().all()) and bool(one[1].isnan().all())
    # f16 operands, the weights f16(d * q); 2^-24 of every term for each of about sqrt(k) roundings of the fp32 sum
    dense = (d.float() * q.float()).to(torch.float16).double().reshape(m, k)
    terms = h.double().norm(dim=1)[:, None] * dense.norm(dim=1)[None, :]
    err = ((y[:tokens] - h.double() @ dense.T).abs() / terms).max().item()
    assert err <= 2.0 ** -24 * np.sqrt(k), err
    assert torch.equal(y[tokens // 2], one[0])


@pytest.mark.parametrize("m,k,tokens,kind", inst.PACKED)
def test_packed_tile(m, k, tokens, kind):
    w, _, _, x = inputs(m, k, tokens)
    gate = torch.randn((tokens, k), device="cuda") if kind == 1 else None
    rows = x
    if kind == 1:
        rows = torch.empty_like(x)
        attn.q_gate(x, gate, rows, tokens * k)
    y, want = padded(tokens, m), padded(tokens, m)
    scratch = torch.full((tokens + 1, k), 3.0, dtype=torch.float16, device="cuda")
    plain = torch.cuda.current_stream()  # (a stream by name: no scratch, test_tile's kernels)
    attn.gemm_q8_0_f16(w, rows, want, m, k, tokens, stream=plain)
    ready = rows.to(torch.float16)
    if kind == 2:
        assert attn.lib().hipml_gemm_q8_0_f16_rows(plain.cuda_stream, w.data_ptr(), ready.data_ptr(), y.data_ptr(), m, k, tokens,
                                                   scratch.data_ptr()) == 0
    else:
        attn.output_chunk_q8_0(w, x, gate, y, m, k, tokens, scratch)
    assert torch.equal(y[:tokens], want[:tokens]) and bool(y[tokens].isnan().all())
    assert bool((scratch[tokens] == 3.0).all()) and torch.equal(ready, rows.to(torch.float16))


def test_scratch_of_a_call_on_the_current_stream_and_under_capture():
    m, k, tokens = 12380, 3072, 392
    assert attn.lib().hipml_gemm_q8_0_f16_scratch(m, k, tokens) == tokens * k * 2
    w, _, _, x = inputs(m, k, tokens)
    want, y = padded(tokens, m), padded(tokens, m)
    attn.gemm_q8_0_f16(w, x, want, m, k, tokens, stream=torch.cuda.current_stream())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    h, z = x.to(torch.float16), padded(tokens, m)
    assert attn.lib().hipml_gemm_q8_0_f16_rows_scratch(m, k, tokens) == tokens * k * 2
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(3):  # (the scratch of one call is the next one's)
            attn.gemm_q8_0_f16(w, x, y, m, k, tokens)
            attn.output_chunk_q8_0(w, None, None, z, m, k, tokens, h)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(y[:tokens], want[:tokens]) and torch.equal(z[:tokens], want[:tokens])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attn.gemm_q8_0_f16(w, x, y, m, k, tokens)
    for _ in range(3):
        y.fill_(float("nan"))
        junk = torch.randn((tokens, k), device="cuda")  # (eager work in memory that was free at the capture)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y[:tokens], want[:tokens]) and bool(junk.isfinite().all())


@pytest.mark.parametrize("threaded", [False, True])
def test_a_call_beside_another_streams_capture(threaded):
    # the call's scratch may need new memory from the driver: the capture goes on, and so does the call (capture begins with
    # the allocator's cache emptied, so that this one does)
    m, k, tokens = 12380, 3072, 392
    w, _, _, x = inputs(m, k, tokens)
    h = x.to(torch.float16)
    want, y, z = padded(tokens, m), padded(tokens, m), padded(tokens, m)
    attn.gemm_q8_0_f16(w, x, want, m, k, tokens, stream=torch.cuda.current_stream())
    count = torch.zeros(64, device="cuda")
    side = torch.cuda.Stream()
    raised = []

    def body():
        try:
            with torch.cuda.stream(side):
                attn.gemm_q8_0_f16(w, x, y, m, k, tokens)
                attn.output_chunk_q8_0(w, None, None, z, m, k, tokens, h)
        except Exception as e:
            raised.append(e)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        count += 1
        if threaded:
            thread = threading.Thread(target=body)
            thread.start()
            thread.join()
        else:
            body()
        count += 1
    assert not raised
    torch.cuda.synchronize()
    assert torch.equal(y[:tokens], want[:tokens]) and torch.equal(z[:tokens], want[:tokens])
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert count.eq(2 * i + 2).all()


def test_a_captured_call_with_the_callers_scratch():
    # the packed route inside a graph: the scratch is used (nothing behind it is), every replay has the bits of the eager
    # call, and scratch that is too short is refused
    m, k, tokens = 12380, 3072, 392
    w, _, _, x = inputs(m, k, tokens)
    h = x.to(torch.float16)
    want, y, z = padded(tokens, m), padded(tokens, m), padded(tokens, m)
    attn.gemm_q8_0_f16(w, x, want, m, k, tokens, stream=torch.cuda.current_stream())
    need = attn.chunk_projection_scratch(m, k, tokens)
    assert need == attn.chunk_projection_scratch(m, k, tokens, f16_rows=True) == 2 * tokens * k
    scratch = torch.full((need + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    rows = torch.full((need + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    with pytest.raises(ValueError):
        attn.gemm_q8_0_f16(w, x, y, m, k, tokens, scratch=scratch[:need - 16])
    with pytest.raises(ValueError):
        attn.output_chunk_q8_0(w, None, None, z, m, k, tokens, h, scratch=scratch[:need - 16])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attn.gemm_q8_0_f16(w, x, y, m, k, tokens, scratch=scratch)
        attn.output_chunk_q8_0(w, None, None, z, m, k, tokens, h, scratch=rows)
    for _ in range(3):
        for t in (y, z):
            t.fill_(float("nan"))
        for t in (scratch, rows):
            t.fill_(0x5A)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y[:tokens], want[:tokens]) and torch.equal(z[:tokens], want[:tokens])
        assert bool(y[tokens].isnan().all()) and bool(z[tokens].isnan().all())
        assert torch.equal(scratch[:need], rows[:need]) and not bool((scratch[:need] == 0x5A).all())
        assert bool((scratch[need:] == 0x5A).all()) and bool((rows[need:] == 0x5A).all())
    # (a stream by name, with scratch: the packed route too)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    scratch.fill_(0x5A)
    torch.cuda.synchronize()
    attn.gemm_q8_0_f16(w, x, y, m, k, tokens, stream=side, scratch=scratch)
    side.synchronize()
    assert torch.equal(y[:tokens], want[:tokens]) and not bool((scratch[:need] == 0x5A).all())
    # a shape that has no use for scratch leaves it alone
    assert attn.chunk_projection_scratch(64, 320, 3) == 0
    scratch.fill_(0x5A)
    few = torch.empty((3, 64), device="cuda")
    attn.gemm_q8_0_f16(w.flatten()[:64 * 340], x.flatten()[:960], few, 64, 320, 3, scratch=scratch)
    assert bool((scratch == 0x5A).all())
