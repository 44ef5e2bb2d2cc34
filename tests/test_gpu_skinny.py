"""GPU parity of the few-row split-K GEMM (csrc/gemm_skinny.hip): each row
padding (4, 8, 16) and activation form (fp32 quantized inside, fragments), the
piece counts per wave at their edges (K of one 128-byte piece up to 6144),
ragged columns, segments, and the SwiGLU form. Against the CPU oracle, bit for
bit (the products and the ordered sums round as the oracle's)."""
import numpy as np
import pytest

from golden.gen import make_case

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import q3vl_int8 as q  # noqa: E402


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def assert_bits(got, want, what):
    torch.cuda.synchronize()
    g, w = got.cpu().numpy().view(np.uint32), np.ascontiguousarray(want, np.float32).view(np.uint32)
    bad = np.flatnonzero(g.ravel() != w.ravel())
    assert bad.size == 0, f"{what}: {bad.size} of {g.size} differ, first at {bad[:5]}"


@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("K", [128, 896, 1024, 1152, 2048, 3072, 4096, 5120, 6144])
def test_linear_few_rows(orc, K, gs):
    for M, N in ((2, 33), (4, 70), (5, 16), (8, 50), (9, 47), (16, 70)):
        A, W, S = make_case(M + N + K, M, N, K, gs)
        A[M - 1, :gs] = 0.0
        A[0, gs - 1] = 1e30  # an overflowing group: scale inf
        assert_bits(q.linear_i8(dev(A), dev(W), dev(S), gs), orc.linear(A, W, S, gs), f"{M}x{N}x{K} gs {gs}")


@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("M,N,K", [(6, 40, 4224), (6, 40, 4608), (8, 33, 4864), (9, 47, 3200), (16, 70, 3328)], ids=str)
def test_linear_past_the_pieces(orc, M, N, K, gs):
    """K past the pieces a wave takes with these rows (4096 at 5..8, 3072 at
    9..16): the fragment form."""
    A, W, S = make_case(M + N + K, M, N, K, gs)
    A[0, gs - 1] = 1e30
    assert_bits(q.linear_i8(dev(A), dev(W), dev(S), gs), orc.linear(A, W, S, gs), f"{M}x{N}x{K} gs {gs}")


@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("M,N,K", [(2, 33, 3200), (3, 70, 3584), (4, 40, 3840), (6, 40, 3200)], ids=str)
def test_swiglu_past_the_pieces(orc, M, N, K, gs):
    """K past 3072 under SwiGLU: the integer GEMV; the MLP of such a width too."""
    A, Wg, Sg = make_case(M + N, M, N, K, gs)
    _, Wu, Su = make_case(M + N + 1, M, N, K, gs)
    h = orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs))
    assert_bits(q.linear_i8_swiglu(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), gs), h, f"swiglu {M}x{N}x{K} gs {gs}")
    I = 256
    _, Wg, Sg = make_case(M, M, I, K, gs)
    _, Wu, Su = make_case(M + 1, M, I, K, gs)
    _, Wd, Sd = make_case(M + 2, M, K, I, gs)
    h = orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs)).reshape(M, I)
    assert_bits(q.mlp_i8(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), dev(Wd), dev(Sd), gs), orc.linear(h, Wd, Sd, gs), "mlp")


@pytest.mark.parametrize("M", [3, 8, 16])
def test_multi_few_rows(orc, M):
    K, gs, Ns = 1152, 64, (33, 16, 50)
    cases = [make_case(M + n, M, n, K, gs) for n in Ns]
    A = cases[0][0]
    outs = q.linear_i8_multi(dev(A), [dev(w) for _, w, _ in cases], [dev(s) for _, _, s in cases], gs)
    for o, (_, w, s), n in zip(outs, cases, Ns):
        assert_bits(o, orc.linear(A, w, s, gs), f"segment of {n}")


@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("M,N,K", [(2, 33, 128), (4, 70, 2048), (7, 40, 1152), (8, 100, 2048), (3, 20, 3072)], ids=str)
def test_swiglu_few_rows(orc, M, N, K, gs):
    A, Wg, Sg = make_case(M + N, M, N, K, gs)
    _, Wu, Su = make_case(M + N + 1, M, N, K, gs)
    got = q.linear_i8_swiglu(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), gs)
    assert_bits(got, orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs)), f"swiglu {M}x{N}x{K} gs {gs}")


@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("M,H,I", [(2, 256, 384), (8, 1024, 6144), (13, 128, 6144), (16, 256, 256)], ids=str)
def test_mlp_few_rows(orc, M, H, I, gs):
    A, Wg, Sg = make_case(M + I, M, I, H, gs)
    _, Wu, Su = make_case(M + I + 1, M, I, H, gs)
    _, Wd, Sd = make_case(M + I + 2, M, H, I, gs)
    ws = torch.zeros(q.mlp_workspace_bytes(M, H, I, gs), dtype=torch.uint8, device="cuda")
    got = q.mlp_i8(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), dev(Wd), dev(Sd), gs, workspace=ws)
    h = orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs)).reshape(M, I)
    assert_bits(got, orc.linear(h, Wd, Sd, gs), f"mlp {M}x{H}x{I} gs {gs}")


@pytest.mark.parametrize("M", [6, 8, 12])
def test_multi_empty_segment(orc, M):
    """A segment of no columns among the others, in the fragment form (K past
    what the rows' quantizer leaves of the LDS) as elsewhere."""
    K, gs, Ns = 5120, 64, (33, 0, 50)
    cases = [make_case(M + n, M, n, K, gs) if n else (None, np.zeros((0, K), np.int8), np.zeros((0, K // gs), np.float32))
             for n in Ns]
    A = cases[0][0]
    ws = torch.zeros(q.workspace_bytes(M, max(Ns), K, gs), dtype=torch.uint8, device="cuda")
    outs = q.linear_i8_multi(dev(A), [dev(w) for _, w, _ in cases], [dev(s) for _, _, s in cases], gs, workspace=ws)
    for o, (_, w, s), n in zip(outs, cases, Ns):
        if n:
            assert_bits(o, orc.linear(A, w, s, gs), f"segment of {n}")


def test_small_workspace_still_served(orc):
    """5..8 rows at K = 6144 with a workspace too small for the fragments: the
    integer GEMV, as before."""
    M, N, K = 6, 40, 6144
    A, W, S = make_case(5, M, N, K, 64)
    small = torch.zeros(2 * 8192 * M * 4 + 512, dtype=torch.uint8, device="cuda")  # the argmax partials alone
    assert small.numel() < q.workspace_bytes(M, N, K, 64)
    assert_bits(q.linear_i8(dev(A), dev(W), dev(S), 64, workspace=small), orc.linear(A, W, S, 64), "small workspace")


def test_no_workspace_single_launch(orc):
    """5..8 rows without a workspace keep nothing in the library's own buffer
    (which two streams would share): one launch, no quantized activations ahead
    of it. With a workspace the fragments are a launch of their own."""
    import ctypes
    M, N, K, gs = 6, 40, 6144, 64
    A, W, S = make_case(5, M, N, K, gs)
    a, w, s = dev(A), dev(W), dev(S)
    ws = torch.zeros(q.workspace_bytes(M, N, K, gs), dtype=torch.uint8, device="cuda")
    hip = ctypes.CDLL("libamdhip64.so")
    for workspace, launches in ((None, 1), (ws, 2)):
        out = q.linear_i8(a, w, s, gs, workspace=workspace)
        assert_bits(out, orc.linear(A, W, S, gs), "before the capture")
        g = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(g):
            q.linear_i8(a, w, s, gs, out=out, workspace=workspace)
        n = ctypes.c_size_t()
        assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
        assert n.value == launches
        out.zero_()
        g.instantiate()
        g.replay()
        assert_bits(out, orc.linear(A, W, S, gs), "replayed")


# the wide kernel (csrc/gemm_wide.hip): N * K >= 2^26, each row padding and
# group size, with fewer tiles than waves and more, ragged rows
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,V,K", [(2, 65541, 1024), (4, 32801, 2048), (7, 131075, 512), (9, 262150, 256), (16, 33003, 2048)],
                         ids=str)
def test_wide_few_rows(orc, M, V, K, gs):
    A, W, S = make_case(M + V, M, V, K, gs)
    W[V - 1], S[V - 1] = W[V // 2], S[V // 2]  # a tie across waves: the lower index wins
    A[0, 1] = 1e30  # an overflowing group: scale inf
    want = orc.linear(A, W, S, gs)
    logits = torch.zeros((M, V), device="cuda")
    ids = q.lm_head_argmax(dev(A), dev(W), dev(S), gs, logits=logits)
    assert_bits(logits, want, f"logits {M}x{V}x{K} gs {gs}")
    np.testing.assert_array_equal(ids.cpu().numpy(), orc.argmax_rows(want))
    if M <= 8:  # without stored logits
        np.testing.assert_array_equal(q.lm_head_argmax(dev(A), dev(W), dev(S), gs).cpu().numpy(), ids.cpu().numpy())
    assert_bits(q.linear_i8(dev(A), dev(W), dev(S), gs), want, "plain")


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,V,K", [(6, 18749, 3584), (8, 8205, 8192), (3, 20977, 3200), (2, 14567, 4608), (9, 14567, 4608),
                                   (2, 20977, 3200), (2, 16385, 4096), (2, 20010, 3584)], ids=str)
def test_wide_past_its_lds(orc, M, V, K, gs):
    """Wide weights that the wide kernel does not take -- its LDS does not hold
    the rows, K is no multiple of 256, or 2 rows that are better off on the GEMV
    -- on whichever kernel they go to, with a workspace and without."""
    A, W, S = make_case(M + V, M, V, K, gs)
    W[V - 1], S[V - 1] = W[V // 2], S[V // 2]
    want = orc.linear(A, W, S, gs)
    ws = torch.zeros(q.workspace_bytes(M, V, K, gs), dtype=torch.uint8, device="cuda")
    logits = torch.zeros((M, V), device="cuda")
    for w in (ws, None):
        ids = q.lm_head_argmax(dev(A), dev(W), dev(S), gs, logits=logits, workspace=w)
        assert_bits(logits, want, f"logits {M}x{V}x{K} gs {gs}")
        np.testing.assert_array_equal(ids.cpu().numpy(), orc.argmax_rows(want))
        assert_bits(q.linear_i8(dev(A), dev(W), dev(S), gs, workspace=w), want, "plain")


@pytest.mark.parametrize("M,N,K", [(3, 51000, 2048), (4, 24001, 3072), (2, 8100, 2048), (2, 9000, 3072)], ids=str)
def test_swiglu_one_block_a_cu(orc, M, N, K):
    """SwiGLU where a CU's LDS holds one block of the few-row kernel, on either
    side of where the GEMV takes over."""
    A, Wg, Sg = make_case(M + N, M, N, K, 64)
    _, Wu, Su = make_case(M + N + 1, M, N, K, 64)
    ws = torch.zeros(q.workspace_bytes(M, N, K, 64), dtype=torch.uint8, device="cuda")
    got = q.linear_i8_swiglu(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), 64, workspace=ws)
    assert_bits(got, orc.swiglu(orc.linear(A, Wg, Sg, 64), orc.linear(A, Wu, Su, 64)), f"swiglu {M}x{N}x{K}")
