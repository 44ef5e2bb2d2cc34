"""GPU parity of the fragment-order GEMM (csrc/gemm_t16.hip): every tile that
its size rule picks, at each group size, with ragged rows and columns and with
K of whole loop bodies, of less than one, and of one and a remainder. Against
the CPU oracle, bit for bit (integer sums are exact and the fp32 order is
fixed, so there is no tolerance to derive)."""
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


# rows x columns over the plain tiles (32 x 64, 32 x 128, 64 x 64, 64 x 128,
# 128 x 128), each with ragged last tiles; test_t16_plan.py holds that all of
# them are reached on 256 CUs
PLAIN = [(9, 70), (33, 130), (70, 6001), (70, 14003), (70, 20005), (131, 12801), (70, 21851), (131, 16571),
         (131, 19871), (70, 24821)]
# ... with the K that those need: 128 x 128 in front of a row split at groups 32
# and 64, 64 x 64 at group 128
PLAIN_K = [(257, 13311, 64), (140, 22275, 256), (129, 21905, 320), (33, 33824, 1024), (33, 33620, 1152)]
SWIGLU = [(9, 70), (9, 16571), (40, 16571), (70, 11001), (70, 17003)]
MLP = [(9, 128, 128), (37, 640, 384), (70, 128, 11008), (70, 128, 17024), (130, 192, 320), (9, 128, 16640),
       (40, 128, 16640)]
SPLIT = [(2100, 2048, 512)]


def plain_ks(N, gs):
    """The K of test_linear_tiles: loop bodies' remainders, less than one, one and some."""
    return [K for K in ((128, 640, 1152) if gs == 128 else (64, 320, 576)) if not (N > 10000 and K > 700)]


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,N,K", PLAIN_K, ids=str)
def test_linear_tiles_at_k(orc, M, N, K, gs):
    if K % gs:
        pytest.skip("not whole groups")
    A, W, S = make_case(M + N + K, M, N, K, gs)
    A[0, gs // 2] = 1e30
    assert_bits(q.linear_i8(dev(A), dev(W), dev(S), gs), orc.linear(A, W, S, gs), f"{M}x{N}x{K} gs {gs}")


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,N", PLAIN, ids=str)
def test_linear_tiles(orc, M, N, gs):
    for K in ((128, 640, 1152) if gs == 128 else (64, 320, 576)):
        if N > 10000 and K > 700:
            continue  # (the oracle's time)
        A, W, S = make_case(M + N + K, M, N, K, gs)
        A[min(3, M - 1), :gs] = 0.0
        A[0, gs // 2] = 1e30  # an overflowing group: scale inf
        got = q.linear_i8(dev(A), dev(W), dev(S), gs)
        assert_bits(got, orc.linear(A, W, S, gs), f"{M}x{N}x{K} gs {gs}")


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,N", [(9, 70), (9, 16571), (40, 16571), (70, 11001), (70, 17003)], ids=str)
def test_swiglu_tiles(orc, M, N, gs):
    K = 640 if gs == 128 else 320
    A, Wg, Sg = make_case(M + N, M, N, K, gs)
    _, Wu, Su = make_case(M + N + 1, M, N, K, gs)
    got = q.linear_i8_swiglu(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), gs)
    want = orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs))
    assert_bits(got, want, f"swiglu {M}x{N}x{K} gs {gs}")


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,H,I", [(9, 128, 128), (37, 640, 384), (70, 128, 11008), (70, 128, 17024), (130, 192, 320),
                                   (9, 128, 16640), (40, 128, 16640)],
                         ids=str)
def test_mlp_tiles(orc, M, H, I, gs):
    if H % gs or I % gs:
        pytest.skip("not whole groups")
    A, Wg, Sg = make_case(M + I, M, I, H, gs)
    _, Wu, Su = make_case(M + I + 1, M, I, H, gs)
    _, Wd, Sd = make_case(M + I + 2, M, H, I, gs)
    ws = torch.zeros(q.mlp_workspace_bytes(M, H, I, gs), dtype=torch.uint8, device="cuda")
    got = q.mlp_i8(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), dev(Wd), dev(Sd), gs, workspace=ws)
    h = orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs)).reshape(M, I)
    assert_bits(got, orc.linear(h, Wd, Sd, gs), f"mlp {M}x{H}x{I} gs {gs}")


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,V", [(9, 1030), (70, 6001), (70, 14003), (70, 20005)], ids=str)
def test_argmax_tiles(orc, M, V, gs):
    K = 128 if gs == 128 else 64
    A, W, S = make_case(M + V, M, V, K, gs)
    W[V - 1], S[V - 1] = W[V // 2], S[V // 2]  # a tie across blocks: the lower index wins
    logits = torch.zeros((M, V), device="cuda")
    ids = q.lm_head_argmax(dev(A), dev(W), dev(S), gs, logits=logits)
    want = orc.linear(A, W, S, gs)
    assert_bits(logits, want, "logits")
    np.testing.assert_array_equal(ids.cpu().numpy(), orc.argmax_rows(want))
    ids2 = q.lm_head_argmax(dev(A), dev(W), dev(S), gs) if M > 8 else ids
    np.testing.assert_array_equal(ids2.cpu().numpy(), ids.cpu().numpy())


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M,V", [(17, 200), (70, 20005)], ids=str)
def test_argmax_ties_in_a_tile(orc, M, V, gs):
    """The winning column repeated over the lanes of its own 16-column tile and
    a row that is all zeros: the lowest column wins; a row of NaN has none."""
    K = 128
    A, W, S = make_case(M + V + gs, M, V, K, gs)
    A[1] = 0.0
    A[2] = np.nan
    for r in (0, 5, M - 1):
        best = int(orc.argmax_rows(orc.linear(A[r:r + 1].repeat(9, 0), W, S, gs))[0])
        for x in (1, 2, 4, 8, 15):
            if (best ^ x) < V:
                W[best ^ x], S[best ^ x] = W[best], S[best]
    want = orc.linear(A, W, S, gs)
    ids = q.lm_head_argmax(dev(A), dev(W), dev(S), gs).cpu().numpy()
    np.testing.assert_array_equal(ids, orc.argmax_rows(want))


# what the fragment-order GEMM leaves to csrc/gemm.hip
def test_k_past_its_offsets(orc):
    """K past 2^22 (32-bit offsets into a block's rows): plain and SwiGLU."""
    M, N, K, gs = 3, 2, (1 << 22) + 64, 64
    A, Wg, Sg = make_case(1, M, N, K, gs)
    _, Wu, Su = make_case(2, M, N, K, gs)
    g, u = orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs)
    assert_bits(q.linear_i8(dev(A), dev(Wg), dev(Sg), gs), g, "plain")
    assert_bits(q.linear_i8_swiglu(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), gs), orc.swiglu(g, u), "swiglu")


@pytest.mark.parametrize("gs", [32, 64])
def test_argmax_of_stored_logits(orc, gs):
    """A vocabulary of more argmax partials than the workspace holds (8192, of
    128 columns): the logits are stored and scanned."""
    M, V, K = 9, 8192 * 128 + 65, 64
    A, W, S = make_case(gs, M, V, K, gs)
    W[V - 1], S[V - 1] = W[V // 2], S[V // 2]
    want = orc.linear(A, W, S, gs)
    ids = q.lm_head_argmax(dev(A), dev(W), dev(S), gs).cpu().numpy()
    np.testing.assert_array_equal(ids, orc.argmax_rows(want))
    logits = torch.zeros((M, V), device="cuda")
    q.lm_head_argmax(dev(A), dev(W), dev(S), gs, logits=logits)
    assert_bits(logits, want, "logits")


@pytest.mark.parametrize("M", [1, 4, 40], ids=str)
def test_silu_range(orc, M):
    """Gates from 2^-75 to past expf's range on both sides, 0, infinite and
    NaN: the SwiGLU epilogues' fast division and its other case."""
    N, K, gs = 320, 64, 64
    A, Wg, Sg = make_case(7, M, N, K, gs)
    _, Wu, Su = make_case(8, M, N, K, gs)
    Sg[:, 0] = np.exp2(np.linspace(-75, 12, N)).astype(np.float32)
    Sg[5:9, 0] = 0.0, np.inf, 1e37, np.nan
    got = q.linear_i8_swiglu(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), gs)
    want = orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs)).reshape(M, N)
    torch.cuda.synchronize()
    g, ok = got.cpu().numpy().reshape(M, N), ~np.isnan(want)
    np.testing.assert_array_equal(np.isnan(g), ~ok)
    np.testing.assert_array_equal(g[ok].view(np.uint32), want[ok].view(np.uint32))


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M", [641, 700, 2100], ids=str)
def test_row_split(orc, M, gs):
    """A nearly empty last round runs as a product of its own: 640 + 1 and
    640 + 60 rows of a SwiGLU pair, the same in front of down (group 32 and
    64), and 2048 + 52 rows of a plain product."""
    if M == 2100:
        A, W, S = make_case(M, M, 2048, 512, gs)
        assert_bits(q.linear_i8(dev(A), dev(W), dev(S), gs), orc.linear(A, W, S, gs), f"plain gs {gs}")
        return
    H, I = 128, 6144
    A, Wg, Sg = make_case(M, M, I, H, gs)
    _, Wu, Su = make_case(M + 1, M, I, H, gs)
    _, Wd, Sd = make_case(M + 2, M, H, I, gs)
    h = orc.swiglu(orc.linear(A, Wg, Sg, gs), orc.linear(A, Wu, Su, gs)).reshape(M, I)
    assert_bits(q.linear_i8_swiglu(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), gs), h, f"swiglu gs {gs}")
    ws = torch.zeros(q.mlp_workspace_bytes(M, H, I, gs), dtype=torch.uint8, device="cuda")
    got = q.mlp_i8(dev(A), dev(Wg), dev(Sg), dev(Wu), dev(Su), dev(Wd), dev(Sd), gs, workspace=ws)
    assert_bits(got, orc.linear(h, Wd, Sd, gs), f"mlp gs {gs}")
