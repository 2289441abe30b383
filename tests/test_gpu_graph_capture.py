"""vedic_gemm_noalloc under HIP graph capture, the callers it is meant for.

Each case records one vedic_gemm_noalloc call into a graph
(torch.cuda.graph, global capture mode, so any allocating or synchronising
HIP call inside would end the capture with an error), then replays the graph
four times.  Between replays the program does its own eager work: another
vedic_gemm_noalloc call of a different shape, which overwrites the shared
scratch region, a vedic_gemm call, and the reset of C (and of the column
sums) to their starting values, then a device synchronisation.  Every replay
must reproduce the eager call's C (and column sums) bit for bit: a replay
that read scratch contents left by an earlier call, or a captured node that
behaved differently on later replays, shows up here.

The cases use each kind of temporary the entry point carves from its region:
split-K partial slabs (a TN product with beta = 1), the column partials of the
GELU backward, the binary16 copy of an fp32 activation (AMP product wider
than the in-kernel conversion serves), and none (bias + GELU on the 256 x 256
tiles).

The other two tests record the entry points that take their temporaries from
the stream's workspace block: a graph must not hold memory that later calls on
the stream use, outgrow or free, nor allocate any."""
import ctypes

import pytest

torch = pytest.importorskip("torch")

from logos_amd import _lib  # noqa: E402

pytestmark = pytest.mark.gpu

CASES = ["splitk_tn_f16", "gelu_bwd_colsum", "amp_cast", "bias_gelu_f16"]


@pytest.fixture(scope="module")
def lib():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield _lib.load()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()


def _desc(op, in_dtype, M, N, K, A, B, C, *, beta=0.0, epilogue=_lib.EPI_NONE, bias=None, preact=None,
          colsum=None, colsum_beta=0.0):
    return _lib.GemmDesc(op=op, in_dtype=in_dtype, out_dtype=_lib.DT_F32, M=M, N=N, K=K,
                         A=A.data_ptr(), lda=A.shape[1], B=B.data_ptr(), ldb=B.shape[1], C=C.data_ptr(), ldc=N,
                         alpha=1.0, beta=beta, bias=bias.data_ptr() if bias is not None else None,
                         epilogue=epilogue, preact=preact.data_ptr() if preact is not None else None,
                         ld_preact=N if preact is not None else 0,
                         stream=torch.cuda.current_stream().cuda_stream,
                         colsum=colsum.data_ptr() if colsum is not None else None, colsum_beta=colsum_beta)


def _case(case, g):
    r = lambda *s, std=1.0: torch.randn(*s, generator=g, device="cuda") * std  # noqa: E731
    if case == "splitk_tn_f16":  # 1024 x 1024 over K = 8192: four slices into the region
        M, N, K = 1024, 1024, 8192
        A, B = r(K, M).half(), r(K, N, std=1e-2).half()
        return M, N, K, A, B, r(M, N, std=1e-3), dict(op=_lib.OP_TN, in_dtype=_lib.DT_F16, beta=1.0), False
    if case == "gelu_bwd_colsum":  # column partials of every 32-row block in the region
        M, N, K = 2048, 1024, 512
        A, B = r(M, K, std=1e-3).half(), r(N, K, std=0.02).half()
        args = dict(op=_lib.OP_NT, in_dtype=_lib.DT_F16, epilogue=_lib.EPI_GELU_BWD, preact=r(M, N, std=2.0))
        return M, N, K, A, B, torch.zeros(M, N, device="cuda"), args, True
    if case == "amp_cast":  # fp32 activation, N = 2048: cast into the region, then the fp16 product
        M, N, K = 1024, 2048, 1024
        A, B = r(M, K), r(K, N, std=0.02).half()
        args = dict(op=_lib.OP_NN, in_dtype=_lib.DT_F32_F16, epilogue=_lib.EPI_BIAS_GELU, bias=r(N, std=0.01))
        return M, N, K, A, B, torch.zeros(M, N, device="cuda"), args, False
    if case == "bias_gelu_f16":  # no temporaries
        M, N, K = 2048, 2048, 1024
        A, B = r(M, K).half(), r(K, N, std=0.02).half()
        args = dict(op=_lib.OP_NN, in_dtype=_lib.DT_F16, epilogue=_lib.EPI_BIAS_GELU, bias=r(N, std=0.01))
        return M, N, K, A, B, torch.zeros(M, N, device="cuda"), args, False
    raise ValueError(case)


def _bits(t):
    return t.contiguous().view(torch.int32)


@pytest.mark.parametrize("case", CASES)
def test_noalloc_graph_replays(lib, case):
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    M, N, K, A, B, C0, args, want_cs = _case(case, g)
    # the eager work between replays: a split-K product through the same
    # region (other contents), and an ordinary vedic_gemm
    oA, oB = torch.randn(4096, 512, generator=g, device="cuda").half(), \
        torch.randn(4096, 768, generator=g, device="cuda").half()
    oC = torch.zeros(512, 768, device="cuda")
    xA, xB = torch.randn(512, 256, generator=g, device="cuda").half(), \
        torch.randn(256, 384, generator=g, device="cuda").half()
    xC = torch.empty(512, 384, device="cuda")

    C = C0.clone()
    cs = torch.full((N,), 0.5, device="cuda") if want_cs else None
    d = _desc(M=M, N=N, K=K, A=A, B=B, C=C, colsum=cs, colsum_beta=1.0 if want_cs else 0.0, **args)
    assert lib.vedic_gemm_noalloc(ctypes.byref(d)) == _lib.STATUS_OK, case  # eager, and the region's lookup
    torch.cuda.synchronize()
    want, want_sums = C.clone(), cs.clone() if want_cs else None

    graph = torch.cuda.CUDAGraph()
    C.copy_(C0)
    if want_cs:
        cs.fill_(0.5)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        dg = _desc(M=M, N=N, K=K, A=A, B=B, C=C, colsum=cs, colsum_beta=1.0 if want_cs else 0.0, **args)
        status = lib.vedic_gemm_noalloc(ctypes.byref(dg))
    assert status == _lib.STATUS_OK, f"{case}: status {status} under capture"

    for rep in range(4):
        od = _desc(op=_lib.OP_TN, in_dtype=_lib.DT_F16, M=512, N=768, K=4096, A=oA, B=oB, C=oC)
        assert lib.vedic_gemm_noalloc(ctypes.byref(od)) == _lib.STATUS_OK
        xd = _desc(op=_lib.OP_NN, in_dtype=_lib.DT_F16, M=512, N=384, K=256, A=xA, B=xB, C=xC)
        assert lib.vedic_gemm(ctypes.byref(xd)) == _lib.STATUS_OK
        C.copy_(C0)
        if want_cs:
            cs.fill_(0.5)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(_bits(C), _bits(want)), \
            f"{case}: replay {rep}: {int((C != want).sum())} outputs differ from the eager call"
        if want_cs:
            assert torch.equal(_bits(cs), _bits(want_sums)), f"{case}: replay {rep}: column sums differ"
    del graph


def _ordinary(case, g):
    """The call and its output tensors."""
    from logos_amd import vedic

    r = lambda *s, std=1.0: torch.randn(*s, generator=g, device="cuda") * std  # noqa: E731
    if case == "splitk_f32":  # 128 tiles of 128 x 128 in slices of K
        A, B, C = r(2048, 2048), r(2048, 1024, std=0.02), torch.empty(2048, 1024, device="cuda")
        return lambda: vedic.gemm(vedic.OP_NN, A, B, C), [C]
    if case == "splitk_f16_colsum":
        A, B, C = r(8192, 512).half(), r(8192, 512, std=0.01).half(), torch.empty(512, 512, device="cuda")
        cs = torch.empty(512, device="cuda")
        return lambda: vedic.gemm(vedic.OP_TN, A, B, C, colsum=cs), [C, cs]
    if case == "amp_cast":
        A, B, C = r(2100, 4096), r(4096, 1024, std=0.02).half(), torch.empty(2100, 1024, device="cuda")
        return lambda: vedic.amp_gemm(A, B, out=C), [C]
    dh = int(case.split("_")[-1])
    Q, K, V, dO = (r(1500, dh) for _ in range(4))
    O, lse = torch.empty_like(Q), torch.empty(1500, device="cuda")
    if case.startswith("attention_fwd"):  # one head: key chunks from the work queue, partials merged
        return lambda: vedic.flash_attention_fwd(Q, K, V, O, lse=lse), [O, lse]
    vedic.flash_attention_fwd(Q, K, V, O, lse=lse)
    d = [torch.empty_like(Q) for _ in range(3)]
    return lambda: vedic.flash_attention_bwd(Q, K, V, O, dO, lse, *d), d


@pytest.mark.parametrize("case", ["splitk_f32", "splitk_f16_colsum", "amp_cast", "attention_fwd_64", "attention_fwd_128",
                                  "attention_fwd_80", "attention_bwd_64"])
def test_block_of_a_capture(lib, case):
    """One eager call on the stream, then its capture, which takes the block
    over; between the replays the stream serves other calls from a new one."""
    from logos_amd import vedic

    g = torch.Generator(device="cuda")
    g.manual_seed(13)
    call, outs = _ordinary(case, g)
    oA, oB = torch.randn(4096, 640, generator=g, device="cuda"), torch.randn(4096, 512, generator=g, device="cuda")
    oC = torch.empty(640, 512, device="cuda")
    oQ, oK, oV = (torch.randn(2000, 64, generator=g, device="cuda") for _ in range(3))
    oO = vedic.flash_attention_fwd(oQ, oK, oV)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call()
    torch.cuda.synchronize()
    want = [t.clone() for t in outs]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call()
    for rep in range(4):
        with torch.cuda.stream(stream):
            vedic.gemm(vedic.OP_TN, oA, oB, oC)
            got = vedic.flash_attention_fwd(oQ, oK, oV)
        for t in outs:
            t.fill_(7.0)
        torch.cuda.synchronize()
        assert torch.equal(got, oO)
        graph.replay()
        torch.cuda.synchronize()
        for t, w in zip(outs, want):
            assert torch.equal(_bits(t), _bits(w)), f"{case}: replay {rep}: {int((t != w).sum())} outputs differ"
    del graph
    assert lib.vedic_workspace_release(stream.cuda_stream) == _lib.STATUS_OK
    torch.cuda.synchronize()


@pytest.mark.parametrize("case", ["splitk_f32", "splitk_f16_colsum", "amp_cast", "attention_fwd_64", "attention_fwd_80",
                                  "attention_bwd_64"])
def test_capture_without_a_block(lib, case):
    """Captured on a stream that has no block: products and attention run
    without slices, the AMP product converts in the kernel (the same bits), and
    what cannot do without memory is refused, with nothing recorded."""
    g = torch.Generator(device="cuda")
    g.manual_seed(17)
    call, outs = _ordinary(case, g)
    call()
    torch.cuda.synchronize()
    want = [t.clone() for t in outs]
    stream = torch.cuda.Stream()
    lib.vedic_workspace_release(stream.cuda_stream)  # (the handle may have served another test)
    torch.cuda.synchronize()
    x = torch.zeros(4, device="cuda")
    graph = torch.cuda.CUDAGraph()
    refused = False
    with torch.cuda.graph(graph, stream=stream):
        x.add_(1.0)
        try:
            call()
        except RuntimeError:
            refused = True
    assert refused == (case in ("splitk_f16_colsum", "attention_fwd_80", "attention_bwd_64"))
    for t in outs:
        t.fill_(7.0)
    for rep in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert float(x[0]) == rep + 1
        for t, w in zip(outs, want):
            if refused:
                assert bool((t == 7.0).all())
            elif case == "amp_cast":
                assert torch.equal(_bits(t), _bits(w))
            else:  # (the sums in another order)
                assert float((t - w).abs().max()) <= 1e-5 * float(w.abs().max())
    del graph
