"""GPU parity of each stage, called through the C ABI, against the CPU oracle."""

import numpy as np
import pytest
import torch

from fairseq2_amd import _abi
import workloads as W
from oracle import moe_oracle as O
from tests._util import TORCH_DTYPE, assert_output_close, assert_routing_equal, launched, oracle_routing

pytestmark = pytest.mark.gpu

MODES = {
    "reference": W.RoutingMode("sigmoid", False, "input"),
    "softmax_renorm": W.RoutingMode("softmax", True, "output"),
    "softmax_plain": W.RoutingMode("softmax", False, "output"),
    "sigmoid_renorm": W.RoutingMode("sigmoid", True, "output"),
}


def _say(*a):
    print(*a, flush=True)


# ------------------------------------------------------------------------------------------ router
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize(
    "tokens,d,e,k,mode,zipf",
    [
        (333, 64, 8, 2, "reference", None),
        (1000, 256, 128, 8, "softmax_renorm", 1.2),
        (257, 136, 16, 1, "reference", None),
        (100, 512, 200, 16, "softmax_plain", 1.1),
        (64, 72, 5, 5, "sigmoid_renorm", None),  # K == E
        (31, 64, 1, 1, "reference", None),  # E == 1
        (50, 128, 256, 16, "softmax_renorm", 1.0),  # the largest E the matrix-pipe router takes
        (70, 128, 512, 32, "softmax_renorm", 1.0),  # the largest E and K the library takes
        (33, 200, 384, 24, "sigmoid_renorm", None),
        # bf16 with D >= 512 and few tokens: several blocks share a token tile
        (64, 2048, 128, 8, "softmax_renorm", 1.2),   # 8 blocks per tile
        (33, 1024, 256, 16, "softmax_plain", 1.0),   # two-fragment kernel, 8 blocks per tile
        (3000, 576, 24, 3, "reference", None),       # 2 blocks per tile, 9 chunks: uneven shares
        (1, 512, 8, 2, "sigmoid_renorm", None),
    ],
)
def test_router_matches_oracle(gpu_device, dtype, tokens, d, e, k, mode, zipf):
    _say("router", dtype, tokens, d, e, k, mode)
    spec = W.small_spec(tokens=tokens, model_dim=d, num_experts=e, top_k=k, inner_dim=8, dtype=dtype,
                        zipf_s=zipf, mode=MODES[mode], seed=tokens)
    wl = W.make_workload_from_spec(spec, with_weights=False)
    logits, idx, w = oracle_routing(wl)
    dt = TORCH_DTYPE[dtype]
    x = wl.x.reshape(-1, d).to(dt).to(gpu_device)
    bias = None if wl.router_bias is None else wl.router_bias.to(gpu_device)
    gi, gw, gl = _abi.router_topk(
        x, wl.router.to(dt).to(gpu_device), bias, k, _abi.SCORE_SOFTMAX if "softmax" in mode else _abi.SCORE_SIGMOID,
        spec.mode.renormalize, want_logits=True,
    )
    np.testing.assert_allclose(gl.cpu().double().numpy(), logits.numpy(), rtol=1e-5, atol=2e-5)
    assert torch.equal(gi.cpu().long(), idx), "selected experts differ from the oracle"
    np.testing.assert_allclose(gw.cpu().double().numpy(), w.numpy(), rtol=5e-5, atol=1e-6)
    # without the scratch buffer one block per 32 tokens walks all of D: same selection, logits
    # equal up to the f32 summation order
    si, sw, sl = _abi.router_topk(
        x, wl.router.to(dt).to(gpu_device), bias, k, _abi.SCORE_SOFTMAX if "softmax" in mode else _abi.SCORE_SIGMOID,
        spec.mode.renormalize, want_logits=True, split=False,
    )
    np.testing.assert_allclose(sl.cpu().double().numpy(), logits.numpy(), rtol=1e-5, atol=2e-5)
    assert torch.equal(si.cpu().long(), idx), "selected experts differ from the oracle (one block per tile)"
    np.testing.assert_allclose(sw.cpu().double().numpy(), w.numpy(), rtol=5e-5, atol=1e-6)
    splits = _abi.load().fs2moe_router_workspace_bytes(x.shape[0], d, e, _abi.dtype_code(dt)) > 0
    assert splits == (dtype == "bf16" and d >= 512 and tokens <= 4096)
    if not splits:
        assert torch.equal(gl, sl) and torch.equal(gw, sw)


# Numbers of experts that are no multiple of 8 on the matrix-pipe router (rows of the matrix begin anywhere, the
# last chunk ends past it), and the bookkeeping that the router's kernels leave to the whole-layer call: in one
# block (up to 32 tokens), in tiles of 8 (up to 2048), of 16 and of 32, with one step of the model dimension to
# a block (normalised on the way) and with several.
@pytest.mark.parametrize("tokens,d,e,k", [
    (1, 512, 60, 6), (32, 2048, 132, 32), (33, 1024, 60, 8), (257, 2048, 250, 5), (1024, 320, 9, 2),
    (1025, 2048, 60, 4), (40, 5120, 7, 3), (8200, 128, 60, 6),
    # a last block with part of a step: of one chunk, of three, with a tail of a chunk; the most slices, one
    # chunk more than they take at a step each, and with the experts that have two k-groups to a block
    (33, 1600, 60, 8), (1, 576, 16, 2), (40, 2880, 128, 8), (17, 2632, 64, 5), (32, 5120, 128, 8), (3, 5184, 128, 4),
    (9, 2496, 200, 5),
    # the last tile of 8, the first and the last of 16
    (2047, 1024, 60, 4), (2049, 512, 132, 32), (4096, 512, 250, 5),
])
@pytest.mark.parametrize("normed", [False, True])
def test_router_and_bookkeeping_in_the_whole_layer_call(gpu_device, tokens, d, e, k, normed):
    from fairseq2_amd import MoE

    _say("router and bookkeeping", tokens, d, e, k, normed)
    g = torch.Generator().manual_seed(tokens + e)
    x = torch.randn(tokens, d, generator=g).bfloat16().to(gpu_device)
    with torch.device(gpu_device):
        layer = MoE(d, 64, False, e, 1.0, k, inner_dim_scale=1.0, auto_scale=False, score_fn="softmax", scale_on="output")
        norm = torch.nn.RMSNorm(d, eps=1e-6) if normed else None
    layer.bfloat16().requires_grad_(False)
    for p in layer.parameters():
        p.normal_(0.0, 0.05)
    if normed:
        norm.bfloat16().requires_grad_(False).weight.normal_(1.0, 0.1)
    router = layer.router.detach()
    idx, _, logits = _abi.router_topk(x, router, None, k, _abi.SCORE_SOFTMAX, want_logits=True)
    ref = x.double().cpu() @ router.double().cpu()
    np.testing.assert_allclose(logits.cpu().double().numpy(), ref.numpy(), rtol=1e-5, atol=1e-4)
    host, _ = _abi.cpu_router_select(logits, k, _abi.SCORE_SOFTMAX)
    assert torch.equal(idx.cpu(), host)
    with torch.inference_mode():
        whole = layer(x, norm=norm)
        again = layer(x, norm=norm)
        staged = layer._stages(x, None, layer._norm_args(norm, x))[0]
    assert torch.equal(whole, again) and torch.equal(whole, staged)


@pytest.mark.parametrize(
    "tokens,d,e,k,mode,zipf",
    [
        (1, 2048, 128, 8, "softmax_renorm", 1.2),    # the decode step of the benchmark's layer
        (4, 2048, 128, 8, "softmax_renorm", None),
        (3, 4096, 8, 2, "softmax_renorm", None),
        (2, 5120, 16, 1, "sigmoid_renorm", None),
        (4, 2048, 256, 16, "softmax_plain", 1.0),
        (3, 8192, 64, 6, "reference", None),
        (4, 520, 32, 4, "softmax_plain", None),      # 9 chunks of the model dimension over 2 blocks
        (1, 8, 8, 8, "reference", None),             # one 16-byte chunk per row, K == E
        (2, 1024, 24, 3, "softmax_renorm", None),
        (5, 2048, 128, 8, "softmax_renorm", None),
    ],
)
def test_router_of_a_few_tokens(gpu_device, tokens, d, e, k, mode, zipf):
    """The token counts of a decode step at the model and expert counts of the known layers:
    against the oracle, and with the normalisation in front."""
    _say("router, few tokens", tokens, d, e, k, mode)
    spec = W.small_spec(tokens=tokens, model_dim=d, num_experts=e, top_k=k, inner_dim=8, dtype="bf16",
                        zipf_s=zipf, mode=MODES[mode], seed=tokens + d)
    wl = W.make_workload_from_spec(spec, with_weights=False)
    logits, idx, w = oracle_routing(wl)
    x = wl.x.reshape(-1, d).bfloat16().to(gpu_device)
    router = wl.router.bfloat16().to(gpu_device)
    bias = None if wl.router_bias is None else wl.router_bias.to(gpu_device)
    score = _abi.SCORE_SOFTMAX if "softmax" in mode else _abi.SCORE_SIGMOID
    gi, gw, gl = _abi.router_topk(x, router, bias, k, score, spec.mode.renormalize, want_logits=True)
    np.testing.assert_allclose(gl.cpu().double().numpy(), logits.numpy(), rtol=1e-5, atol=2e-5)
    assert torch.equal(gi.cpu().long(), idx), "selected experts differ from the oracle"
    np.testing.assert_allclose(gw.cpu().double().numpy(), w.numpy(), rtol=5e-5, atol=1e-6)
    # the normalisation in front: the rows, and the routing of those rows
    g = torch.Generator().manual_seed(d)
    gamma = (1.0 + 0.3 * torch.randn(d, generator=g)).bfloat16().to(gpu_device)
    xn, ni, nw, nl = _abi.router_topk_norm(x, gamma, 1e-5, router, bias, k, score,
                                           spec.mode.renormalize, want_logits=True)
    want = O.rms_norm(x.cpu(), gamma.cpu(), 1e-5).double()
    assert bool(((xn.cpu().double() - want).abs() <= 2.0 ** -7 * want.abs()).all())
    pi, pw, pl = _abi.router_topk(xn, router, bias, k, score, spec.mode.renormalize, want_logits=True)
    assert torch.equal(ni, pi) and torch.equal(nw, pw) and torch.equal(nl, pl)
    # up to 32 tokens the router's blocks normalise the columns they read; more tokens go through a
    # kernel in front: the same rows among 40 come out with the same bits
    many = torch.cat([x, x.flip(0).repeat(40, 1)[: 40 - tokens]])
    xn40 = _abi.router_topk_norm(many, gamma, 1e-5, router, bias, k, score, spec.mode.renormalize)[0]
    assert torch.equal(xn40[:tokens], xn)


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize(
    "tokens,d,e,k,with_weight",
    [
        (257, 256, 16, 4, True),    # a last block of one row (normalised by the kernel in front)
        (1500, 256, 16, 4, True),   # up to 4096 tokens a small kernel in front normalises the rows
        (1101, 2048, 128, 8, True),
        (1100, 100, 10, 2, True),
        (4100, 256, 16, 4, True),   # beyond 4096 tokens the MFMA routers normalise on the way
        (4133, 128, 8, 2, False),
        (4133, 100, 10, 2, True),   # ... and so does the FMA router
        (8192, 512, 128, 8, True),  # the prefill token count
        (64, 2048, 128, 8, True),   # the decode shape
        (100, 96, 24, 3, False),    # no elementwise weight
        (45, 100, 10, 2, True),     # D, E off the 16-byte grid: element-wise path, FMA router
        (1, 64, 8, 8, True),
    ],
)
def test_router_with_norm_in_front(gpu_device, dtype, tokens, d, e, k, with_weight):
    """fs2moe_router_topk_norm: the normalised rows against the oracle's rms_norm (the reduction
    order of the mean differs, so a value may land on the neighbouring number), and the routing bit
    for bit against the plain router run on those rows."""
    _say("router+norm", dtype, tokens, d, e, k, with_weight)
    td = TORCH_DTYPE[dtype]
    g = torch.Generator().manual_seed(tokens + d)
    x = (3.0 * torch.randn(tokens, d, generator=g) * torch.rand(tokens, 1, generator=g)).to(td)
    x[0] = 0.0  # a zero row: rsqrt(eps) stays finite and the row stays zero
    weight = (1.0 + 0.3 * torch.randn(d, generator=g)).to(td) if with_weight else None
    router = (0.2 * torch.randn(d, e, generator=g)).to(td)
    bias = 0.1 * torch.randn(e, generator=g)
    eps = 1e-5
    xd = x.to(gpu_device)
    xn, idx, w, logits = _abi.router_topk_norm(
        xd, None if weight is None else weight.to(gpu_device), eps, router.to(gpu_device),
        bias.to(gpu_device), k, _abi.SCORE_SOFTMAX, True, want_logits=True)
    idx2, w2, logits2 = _abi.router_topk(xn, router.to(gpu_device), bias.to(gpu_device), k,
                                         _abi.SCORE_SOFTMAX, True, want_logits=True)
    torch.cuda.synchronize()
    assert torch.equal(xd, x.to(gpu_device)), "the input rows are left untouched"
    want = O.rms_norm(x, weight, eps)
    step = 2.0 ** -7 if dtype == "bf16" else 2.0 ** -20
    got = xn.cpu().double()
    assert bool(((got - want.double()).abs() <= step * want.double().abs()).all())
    assert bool((got[0] == 0).all())
    if dtype == "bf16":
        assert (xn.cpu() == want).float().mean() > 0.98
    assert torch.equal(idx, idx2) and torch.equal(w, w2) and torch.equal(logits, logits2)


@pytest.mark.parametrize(
    "tokens,d,e,k,mode,zipf",
    [
        (8192, 2048, 128, 8, "softmax_renorm", 1.2),  # the benchmark's layer
        (33, 128, 8, 2, "reference", None),           # one step, a last block of one token
        (4100, 256, 16, 4, "softmax_plain", None),
        (4200, 1024, 256, 16, "sigmoid_renorm", 1.0),  # two expert fragments per wave
        (4130, 384, 136, 3, "softmax_renorm", None),   # experts off the fragment size
        (5000, 5120, 16, 1, "reference", None),
    ],
)
def test_router_reading_an_expert_major_matrix(gpu_device, tokens, d, e, k, mode, zipf):
    """The router given its matrix as (E, D) (ROUTER_OUT_IN): the same selection as the oracle's,
    logits equal up to summation order, with exact ties, and with the
    normalisation in front bit for bit what the plain call makes of the normalised rows."""
    _say("router (E, D)", tokens, d, e, k, mode)
    lib = _abi.load()
    assert lib.fs2moe_router_takes_out_in(tokens, d, e, _abi.dtype_code(torch.bfloat16)) == 1
    assert lib.fs2moe_router_takes_out_in(tokens, d, e, _abi.dtype_code(torch.float32)) == 0
    assert lib.fs2moe_router_takes_out_in(32, d, e, _abi.dtype_code(torch.bfloat16)) == 0
    # few tokens of a wide model: several blocks share a token tile, and those kernels read (D, E)
    assert lib.fs2moe_router_takes_out_in(64, 2048, 128, _abi.dtype_code(torch.bfloat16)) == 0
    assert lib.fs2moe_router_takes_out_in(tokens, d + 8, e, _abi.dtype_code(torch.bfloat16)) == 0
    spec = W.small_spec(tokens=tokens, model_dim=d, num_experts=e, top_k=k, inner_dim=8, dtype="bf16",
                        zipf_s=zipf, mode=MODES[mode], seed=tokens + e)
    wl = W.make_workload_from_spec(spec, with_weights=False)
    logits, idx, w = oracle_routing(wl)
    x = wl.x.reshape(-1, d).bfloat16().to(gpu_device)
    router = wl.router.bfloat16().to(gpu_device)
    router_t = router.t().contiguous()
    bias = None if wl.router_bias is None else wl.router_bias.to(gpu_device)
    score = _abi.SCORE_SOFTMAX if "softmax" in mode else _abi.SCORE_SIGMOID
    gi, gw, gl = _abi.router_topk(x, router, bias, k, score, spec.mode.renormalize, want_logits=True,
                                  router_t=router_t)
    np.testing.assert_allclose(gl.cpu().double().numpy(), logits.numpy(), rtol=1e-5, atol=2e-5)
    assert torch.equal(gi.cpu().long(), idx), "selected experts differ from the oracle"
    np.testing.assert_allclose(gw.cpu().double().numpy(), w.numpy(), rtol=5e-5, atol=1e-6)
    # the (D, E) form of the same call: the same experts; logits up to the order of the sums
    pi, pw, pl = _abi.router_topk(x, router, bias, k, score, spec.mode.renormalize, want_logits=True)
    assert torch.equal(pi, gi)
    np.testing.assert_allclose(gl.cpu().numpy(), pl.cpu().numpy(), rtol=1e-5, atol=2e-5)
    # with the normalisation in front
    g = torch.Generator().manual_seed(d)
    gamma = (1.0 + 0.3 * torch.randn(d, generator=g)).bfloat16().to(gpu_device)
    xn, ni, nw, nl = _abi.router_topk_norm(x, gamma, 1e-5, router, bias, k, score, spec.mode.renormalize,
                                           want_logits=True, router_t=router_t)
    xn2 = _abi.router_topk_norm(x, gamma, 1e-5, router, bias, k, score, spec.mode.renormalize)[0]
    assert torch.equal(xn, xn2), "the normalised rows do not depend on the router's layout"
    qi, qw, ql = _abi.router_topk(xn, router, bias, k, score, spec.mode.renormalize, want_logits=True,
                                  router_t=router_t)
    assert torch.equal(ni, qi) and torch.equal(nw, qw) and torch.equal(nl, ql)
    # exact ties and special values: small integers make every sum exact
    gi2 = torch.Generator().manual_seed(7)
    xi = torch.randint(-2, 3, (tokens, d), generator=gi2).float()
    ri = torch.randint(-1, 2, (d, e), generator=gi2).float()
    xi[0] = 0.0
    if e > 7:
        ri[:, 7] = ri[:, 3]
    want = xi.double() @ ri.double()
    ti, _, tl = _abi.router_topk(xi.bfloat16().to(gpu_device), ri.bfloat16().to(gpu_device), None, k,
                                 want_logits=True, router_t=ri.t().contiguous().bfloat16().to(gpu_device))
    assert torch.equal(tl.cpu().double(), want)
    assert torch.equal(ti.cpu().long(), O.topk_lowest_index(want, k))


def test_router_refuses_an_expert_major_matrix_where_it_does_not_read_one(gpu_device):
    x = torch.zeros(16, 64, dtype=torch.bfloat16, device=gpu_device)
    r = torch.zeros(8, 64, dtype=torch.bfloat16, device=gpu_device)
    idx = torch.empty(16, 2, dtype=torch.int32, device=gpu_device)
    w = torch.empty(16, 2, dtype=torch.float32, device=gpu_device)
    lib = _abi.load()
    rc = lib.fs2moe_router_topk(x.data_ptr(), r.data_ptr(), None, 16, 64, 8, 2, _abi.dtype_code(x.dtype),
                                _abi.SCORE_SIGMOID | _abi.ROUTER_OUT_IN, 0, idx.data_ptr(), w.data_ptr(),
                                None, None, 0, None)
    assert rc != 0 and b"fs2moe_router_takes_out_in" in lib.fs2moe_last_error()


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
def test_router_ties_resolve_to_lower_expert_id(gpu_device, dtype):
    # Small-integer operands: every partial sum is exact in f32 whatever the order, so exact ties
    # are common and the tie rule is the only thing that decides.
    g = torch.Generator().manual_seed(5)
    t, d, e, k = 512, 64, 24, 6
    x = torch.randint(-2, 3, (t, d), generator=g).float()
    r = torch.randint(-1, 2, (d, e), generator=g).float()
    x[0] = 0.0  # all logits zero: selects experts 0..k-1
    r[:, 7] = r[:, 3]  # two identical experts
    logits = x.double() @ r.double()
    idx = O.topk_lowest_index(logits, k)
    assert idx[0].tolist() == list(range(k))
    dt = TORCH_DTYPE[dtype]
    gi, gw, gl = _abi.router_topk(x.to(dt).to(gpu_device), r.to(dt).to(gpu_device), None, k, want_logits=True)
    assert torch.equal(gl.cpu().double(), logits)
    assert torch.equal(gi.cpu().long(), idx)
    # every selection is sorted by (descending logit, ascending id)
    sel = torch.gather(logits, 1, gi.cpu().long())
    assert bool(((sel[:, :-1] > sel[:, 1:]) | ((sel[:, :-1] == sel[:, 1:]) & (gi.cpu()[:, :-1] < gi.cpu()[:, 1:]))).all())


def test_router_nan_and_inf_order(gpu_device):
    # NaN ranks above +inf (as torch.topk does), -0.0 ties with +0.0.
    d, e = 8, 6
    r = torch.zeros(d, e)
    r[0] = torch.tensor([1.0, -1.0, 0.0, 2.0, 0.5, -0.0])
    x = torch.zeros(4, d)
    x[0, 0] = float("inf")  # logits: inf, -inf, nan, inf, inf, nan
    x[1, 0] = 1.0  # 1, -1, 0, 2, .5, -0
    x[2, 0] = float("nan")  # all nan
    x[3, 0] = -1.0  # -1, 1, -0, -2, -.5, 0
    logits = x @ r
    want = O.topk_lowest_index(logits, 4)
    assert want.tolist() == [[2, 5, 0, 3], [3, 0, 4, 2], [0, 1, 2, 3], [1, 2, 5, 4]]
    gi, _, _ = _abi.router_topk(x.to(gpu_device), r.to(gpu_device), None, 4)
    assert gi.cpu().tolist() == want.tolist()


# ---------------------------------------------------------------------------------------- dispatch
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("tile_m", [1, 16, 128])
@pytest.mark.parametrize("scale_input", [False, True])
def test_dispatch_matches_oracle(gpu_device, dtype, tile_m, scale_input):
    _say("dispatch", dtype, tile_m, scale_input)
    t, d, e, k = 1500, 128, 40, 4
    spec = W.small_spec(tokens=t, model_dim=d, num_experts=e, top_k=k, inner_dim=8, dtype=dtype, zipf_s=1.2, seed=9)
    wl = W.make_workload_from_spec(spec, with_weights=False)
    _, idx, w = oracle_routing(wl)
    r = O.route(idx, e, tile_m)
    assert (r.counts == 0).any(), "the case should contain an expert without tokens"
    dt = TORCH_DTYPE[dtype]
    x = wl.x.reshape(t, d).to(dt).to(gpu_device)
    gi = idx.to(torch.int32).to(gpu_device)
    gw = w.float().to(gpu_device)
    disp = _abi.dispatch(gi, gw, x, e, tile_m, scale_input)
    np.testing.assert_array_equal(disp.counts.cpu().numpy(), r.counts)
    np.testing.assert_array_equal(disp.offsets.cpu().numpy(), r.offsets)
    perm = disp.perm.cpu().numpy()
    np.testing.assert_array_equal(perm[: r.num_rows], r.perm)
    assert (perm[r.num_rows:] == -1).all()
    np.testing.assert_array_equal(disp.inv_perm.cpu().numpy(), r.inv_perm)
    # gathered rows: exact copies (or the f32 product rounded once), zeros on padding rows
    xe = disp.xe[: r.num_rows].float().cpu()
    xs = x.float().cpu()
    want = torch.zeros(r.num_rows, d)
    rows = torch.from_numpy(r.inv_perm.astype(np.int64))
    for s in range(k):
        src = xs * gw.cpu()[:, s : s + 1] if scale_input else xs
        want[rows[:, s]] = src.to(dt).float()
    assert torch.equal(xe, want)


@pytest.mark.parametrize("tokens,e,k", [(1, 8, 2), (200, 256, 16), (256, 128, 8), (257, 128, 8), (700, 24, 4),
                                        (5000, 40, 3), (1100, 384, 24), (16384, 8, 1), (16500, 16, 2)])
def test_dispatch_without_row_copy_matches_oracle(gpu_device, tokens, e, k):
    # at most 256 tokens take the one-kernel path; up to 64 counting blocks (16384 tokens) two kernels,
    # the second doing the scan in every block (with top-3 its blocks of 256 pairs straddle counting
    # blocks); more the three-kernel path: same artefacts
    _say("dispatch index only", tokens, e, k)
    spec = W.small_spec(tokens=tokens, model_dim=64, num_experts=e, top_k=k, inner_dim=8, dtype="bf16",
                        zipf_s=1.1, seed=tokens + e)
    wl = W.make_workload_from_spec(spec, with_weights=False)
    _, idx, w = oracle_routing(wl)
    for tile_m in (1, 16):
        r = O.route(idx.numpy(), e, tile_m)
        x = wl.x.reshape(-1, 64).to(torch.bfloat16).to(gpu_device)
        disp = _abi.dispatch(idx.to(torch.int32).to(gpu_device), w.float().to(gpu_device), x, e, tile_m, False, gather=False)
        assert disp.xe is None
        assert_routing_equal(idx.to(torch.int32), disp, r, f"T={tokens} tile_m={tile_m}")


def test_dispatch_single_token_and_all_to_one(gpu_device):
    # T = 1 and "every token picks the same experts" (maximum collision on the histogram)
    for t in (1, 700):
        idx = torch.tensor([[3, 0]], dtype=torch.int32).repeat(t, 1)
        x = torch.randn(t, 64, generator=torch.Generator().manual_seed(t))
        r = O.route(idx, 5, 16)
        disp = _abi.dispatch(idx.to(gpu_device), None, x.to(gpu_device), 5, 16, False)
        assert disp.counts.cpu().tolist() == [t, 0, 0, t, 0]
        np.testing.assert_array_equal(disp.inv_perm.cpu().numpy(), r.inv_perm)
        np.testing.assert_array_equal(disp.perm.cpu().numpy()[: r.num_rows], r.perm)
        assert torch.equal(disp.xe[r.inv_perm[:, 0].astype(np.int64)].cpu(), x)


# ----------------------------------------------------------------------------------------- experts
def _expert_case(dtype, rows_per_expert, d, f, seed):
    g = torch.Generator().manual_seed(seed)
    e = len(rows_per_expert)
    dt = TORCH_DTYPE[dtype]
    rnd = lambda *s: (torch.randn(*s, generator=g)).to(dt).float()
    counts = torch.tensor(rows_per_expert, dtype=torch.int32)
    tile_m = 16
    padded = (counts + tile_m - 1) // tile_m * tile_m
    offsets = torch.zeros(e + 1, dtype=torch.int32)
    offsets[1:] = torch.cumsum(padded, 0)
    rows = int(offsets[-1])
    xe = rnd(rows, d)
    wg, wu, wd = 0.05 * rnd(e * d, f), 0.05 * rnd(e * d, f), 0.05 * rnd(e * f, d)
    wg, wu, wd = (t.to(dt).float() for t in (wg, wu, wd))
    return counts, offsets, xe, wg, wu, wd


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize(
    "rows_per_expert,d,f",
    [
        ([5, 0, 130, 64, 1, 300], 128, 256),  # ragged, empty expert, several m-tiles
        ([40, 17], 72, 40),  # dims that are not multiples of the tile sizes
        ([128] * 4, 256, 128),  # exact tiles
        ([3] * 32, 64, 64),  # many tiny experts
        ([(5 * i) % 7 for i in range(256)], 64, 64),  # the largest expert count the library takes
        # more tiles than compute units (every persistent block walks several, heavy and light mixed)
        ([(37 * i * i + 11 * i) % 701 for i in range(72)], 128, 384),
    ],
)
def test_grouped_swiglu_matches_oracle(gpu_device, dtype, rows_per_expert, d, f):
    _say("grouped_swiglu", dtype, rows_per_expert[:6], d, f)
    counts, offsets, xe, wg, wu, wd = _expert_case(dtype, rows_per_expert, d, f, seed=d + f)
    e = len(rows_per_expert)
    dt = TORCH_DTYPE[dtype]
    dev = gpu_device
    ye, h = _abi.grouped_swiglu(
        xe.to(dt).to(dev), counts.to(dev), offsets.to(dev), wg.to(dt).to(dev), wu.to(dt).to(dev), wd.to(dt).to(dev), e
    )
    for ex in range(e):
        lo, n = int(offsets[ex]), int(counts[ex])
        if n == 0:
            continue
        u = xe[lo : lo + n].double()
        h_ref = torch.nn.functional.silu(u @ wg[ex * d : (ex + 1) * d].double()) * (u @ wu[ex * d : (ex + 1) * d].double())
        assert_output_close(h[lo : lo + n], h_ref, dtype, f"h of expert {ex}")
        # second GEMM checked from the device's own (rounded) h, so its error is isolated
        y_ref = h[lo : lo + n].double().cpu() @ wd[ex * f : (ex + 1) * f].double()
        assert_output_close(ye[lo : lo + n], y_ref, dtype, f"ye of expert {ex}")
        y_full = O.glu_expert(u, wg[ex * d : (ex + 1) * d].double(), wu[ex * d : (ex + 1) * d].double(), wd[ex * f : (ex + 1) * f].double())
        assert_output_close(ye[lo : lo + n], y_full, dtype, f"expert {ex}")


@pytest.mark.parametrize(
    "bound,rows_per_expert,d,f",
    [
        (1, [1, 0, 1, 1, 0, 0, 1, 1], 2048, 768),   # one decoding sequence at the Qwen3 shape
        (1, [1, 1], 72, 40),                          # K not a multiple of the 128 rows a step takes
        (2, [2, 0, 1, 2], 256, 136),
        (4, [3, 4, 0, 1, 4, 2], 128, 200),
        (8, [8, 5, 0, 7, 1, 8, 3], 320, 192),
        (8, [(3 * i) % 9 for i in range(128)], 64, 64),
        (4, [9, 4, 13, 0, 1], 128, 64),               # counts above the bound: walked again, still right
        (4, [4, 2], 8192, 64),
        (4, [4, 1], 18432, 64),                       # the longest K whose four rows fit LDS
        (1, [1, 0, 1], 128, 4096),                    # a long inner dimension: the second product keeps
        (2, [2, 1, 0, 2], 64, 4352),                  # eight steps of loads in flight (4352: 17 steps)
        # 5 to 16 rows: the same stream with the arithmetic on the matrix pipe
        (16, [16, 9, 0, 12, 1, 5], 2048, 768),       # the Qwen3 shape
        (12, [12, 3, 7], 72, 40),                     # K and N off the kernel's steps
        (5, [5, 0, 2, 5], 256, 136),
        (16, [16, 2], 5112, 64),                      # the longest K whose sixteen rows fit LDS
        (8, [8, 1], 8192, 64),                        # eight rows staged
        (16, [16, 2, 9], 8192, 64),                   # sixteen such rows do not fit: eight at a time
        (8, [20, 8, 9], 128, 136),                    # counts above the bound
        (16, [33, 16, 0, 17], 64, 200),
    ],
)
def test_grouped_swiglu_with_a_bound_on_the_rows_per_expert(gpu_device, bound, rows_per_expert, d, f):
    """``fs2moe_grouped_swiglu_rows``: with a bound of 1..4 rows per expert and bf16 weights the two
    products stream the weights through the vector ALUs, with 5..16 through the matrix pipe (larger
    bounds take the GEMM kernels).  Each expert against the oracle's SwiGLU in f64; rows read
    through a map give the same bits."""
    _say("grouped_swiglu_rows", bound, rows_per_expert[:8], d, f)
    counts, offsets, xe, wg, wu, wd = _expert_case("bf16", rows_per_expert, d, f, seed=bound + d + f)
    e = len(rows_per_expert)
    dev = gpu_device
    bf = torch.bfloat16
    args = (counts.to(dev), offsets.to(dev), wg.to(bf).to(dev), wu.to(bf).to(dev), wd.to(bf).to(dev), e)
    ye, h = _abi.grouped_swiglu(xe.to(bf).to(dev), *args, rows_per_expert=bound)
    for ex in range(e):
        lo, n = int(offsets[ex]), int(counts[ex])
        if n == 0:
            continue
        u = xe[lo : lo + n].double()
        h_ref = torch.nn.functional.silu(u @ wg[ex * d : (ex + 1) * d].double()) * (u @ wu[ex * d : (ex + 1) * d].double())
        assert_output_close(h[lo : lo + n], h_ref, "bf16", f"h of expert {ex}")
        y_ref = h[lo : lo + n].double().cpu() @ wd[ex * f : (ex + 1) * f].double()
        assert_output_close(ye[lo : lo + n], y_ref, "bf16", f"ye of expert {ex}")
        y_full = O.glu_expert(u, wg[ex * d : (ex + 1) * d].double(), wu[ex * d : (ex + 1) * d].double(), wd[ex * f : (ex + 1) * f].double())
        assert_output_close(ye[lo : lo + n], y_full, "bf16", f"expert {ex}")
    # through a row map: rows scattered over a larger matrix, same bits
    total = xe.shape[0]
    g = torch.Generator().manual_seed(5)
    src_rows = torch.randperm(total + 11, generator=g)[:total]
    src = torch.randn(total + 11, d, generator=g).to(bf)
    src[src_rows] = xe.to(bf)
    ye2, h2 = _abi.grouped_swiglu(src.to(dev), *args, row_map=src_rows.to(torch.int32).to(dev), rows_per_expert=bound)
    for ex in range(e):
        lo, n = int(offsets[ex]), int(counts[ex])
        assert torch.equal(ye2[lo : lo + n], ye[lo : lo + n]) and torch.equal(h2[lo : lo + n], h[lo : lo + n])
    # bounds outside 1..16 take the other kernels; a negative bound is refused
    ye3, _ = _abi.grouped_swiglu(xe.to(bf).to(dev), *args, rows_per_expert=17)
    ye4, _ = _abi.grouped_swiglu(xe.to(bf).to(dev), *args)
    for ex in range(e):
        lo, n = int(offsets[ex]), int(counts[ex])
        assert torch.equal(ye3[lo : lo + n], ye4[lo : lo + n])
    with pytest.raises(_abi.Fs2MoeError, match="rows_per_expert"):
        _abi.grouped_swiglu(xe.to(bf).to(dev), *args, rows_per_expert=-1)


def test_grouped_swiglu_row_map_equals_gathered_rows(gpu_device):
    """Reading the rows through dispatch's permutation gives bit for bit what the gathered copy gives."""
    _say("grouped_swiglu row_map")
    t, d, e, k, f = 1500, 128, 24, 4, 192
    spec = W.small_spec(tokens=t, model_dim=d, num_experts=e, top_k=k, inner_dim=f, dtype="bf16", zipf_s=1.2, seed=13)
    wl = W.make_workload_from_spec(spec)
    _, idx, w = oracle_routing(wl)
    dev = gpu_device
    assert _abi.fuses_gather(d, f, torch.bfloat16, torch.bfloat16)
    assert not _abi.fuses_gather(d, f, torch.float32, torch.float32)
    x = wl.x.reshape(-1, d).to(torch.bfloat16).to(dev)
    idx_d, w_d = idx.to(torch.int32).to(dev), w.float().to(dev)
    gathered = _abi.dispatch(idx_d, w_d, x, e, 16, False)
    bare = _abi.dispatch(idx_d, w_d, x, e, 16, False, gather=False)
    assert bare.xe is None and torch.equal(bare.perm, gathered.perm)
    weights = [v.to(torch.bfloat16).to(dev) for v in (wl.gate, wl.up, wl.down)]
    ye_a, h_a = _abi.grouped_swiglu(gathered.xe, gathered.counts, gathered.offsets, *weights, e)
    ye_b, h_b = _abi.grouped_swiglu(x, bare.counts, bare.offsets, *weights, e, row_map=bare.perm)
    valid = (gathered.perm >= 0)
    assert torch.equal(h_a[valid], h_b[valid])
    assert torch.equal(ye_a[valid], ye_b[valid])
    # where the library has no fused path it says so instead of reading garbage
    with pytest.raises(_abi.Fs2MoeError):
        _abi.grouped_swiglu(x.float(), bare.counts, bare.offsets, *(v.float() for v in weights), e, row_map=bare.perm)


def test_grouped_swiglu_beyond_4_gb_of_activations(gpu_device):
    """Rows whose byte offset does not fit 32 bits: the throughput kernel (32-bit offsets) steps
    aside for the general one, and a row map is refused rather than mis-read."""
    _say("grouped_swiglu > 4 GB")
    d, f, e = 2048, 128, 2
    far = 1_090_000  # rows; far * d * 2 bytes = 4.46 GB
    counts = torch.tensor([100, 60], dtype=torch.int32)
    offsets = torch.tensor([0, far, far + 64], dtype=torch.int32)
    g = torch.Generator().manual_seed(9)
    bf = lambda t: t.to(torch.bfloat16)  # noqa: E731
    wg, wu = bf(0.02 * torch.randn(e * d, f, generator=g)), bf(0.02 * torch.randn(e * d, f, generator=g))
    wd = bf(0.02 * torch.randn(e * f, d, generator=g))
    rows = {0: bf(torch.randn(100, d, generator=g)), 1: bf(torch.randn(60, d, generator=g))}
    dev = gpu_device
    xe = torch.empty((far + 64, d), dtype=torch.bfloat16, device=dev)
    xe[:100] = rows[0].to(dev)
    xe[far : far + 60] = rows[1].to(dev)
    ye, h = _abi.grouped_swiglu(xe, counts.to(dev), offsets.to(dev), wg.to(dev), wu.to(dev), wd.to(dev), e)
    for ex, lo in ((0, 0), (1, far)):
        u = rows[ex].double()
        ref = O.glu_expert(u, wg[ex * d : (ex + 1) * d].double(), wu[ex * d : (ex + 1) * d].double(), wd[ex * f : (ex + 1) * f].double())
        assert_output_close(ye[lo : lo + u.shape[0]], ref, "bf16", f"expert {ex}")
    row_map = torch.zeros(far + 64, dtype=torch.int32, device=dev)
    with pytest.raises(_abi.Fs2MoeError, match="4 GB"):
        _abi.grouped_swiglu(xe, counts.to(dev), offsets.to(dev), wg.to(dev), wu.to(dev), wd.to(dev), e, row_map=row_map)


@pytest.mark.parametrize("t,d,e,k,f", [(48, 128, 16, 4, 64), (700, 128, 4, 2, 192)])  # decode / throughput kernel
def test_grouped_swiglu_fp8_row_map_equals_gathered_rows(gpu_device, t, d, e, k, f):
    """The e4m3-weight kernels read rows through the permutation too, with identical results."""
    _say("grouped_swiglu fp8 row_map", t, d, e, k, f)
    spec = W.small_spec(tokens=t, model_dim=d, num_experts=e, top_k=k, inner_dim=f, dtype="bf16",
                        weight_dtype="fp8", zipf_s=1.2, seed=17)
    wl = W.make_workload_from_spec(spec)
    _, idx, w = oracle_routing(wl)
    dev = gpu_device
    assert _abi.fuses_gather(d, f, torch.bfloat16, torch.float8_e4m3fn)
    x = wl.x.reshape(-1, d).to(torch.bfloat16).to(dev)
    idx_d, w_d = idx.to(torch.int32).to(dev), w.float().to(dev)
    gathered = _abi.dispatch(idx_d, w_d, x, e, 16, False)
    bare = _abi.dispatch(idx_d, w_d, x, e, 16, False, gather=False)
    packed = [_abi.pack_fp8_weights(wl.fp8[n + "_q"], e).to(dev) for n in ("gate", "up", "down")]
    scales = tuple(wl.fp8[n + "_scale"].to(dev) for n in ("gate", "up", "down"))
    ye_a, h_a = _abi.grouped_swiglu(gathered.xe, gathered.counts, gathered.offsets, *packed, e, scales=scales)
    ye_b, h_b = _abi.grouped_swiglu(x, bare.counts, bare.offsets, *packed, e, scales=scales, row_map=bare.perm)
    valid = gathered.perm >= 0
    assert int(valid.sum()) == t * k
    assert torch.equal(h_a[valid], h_b[valid])
    assert torch.equal(ye_a[valid], ye_b[valid])


# K off the throughput kernel's units of 64 (8 mod 64 up to 56 mod 64), N off its tiles of 128 and 256
@pytest.mark.parametrize("d,f", [(8, 56), (1032, 8), (120, 184), (200, 1368), (952, 264)])
def test_grouped_swiglu_with_a_k_tail(gpu_device, d, f):
    """bf16 sizes that end inside a unit: every expert against the oracle, the rows through a map bit
    for bit like the copy, and an expert full of NaN, whose weights lie right behind its neighbour's
    last rows of k, reaches no other expert."""
    _say("grouped_swiglu k tail", d, f)
    rows_per_expert = [257, 0, 40, 3, 300, 128]
    counts, offsets, xe, wg, wu, wd = _expert_case("bf16", rows_per_expert, d, f, seed=d + f)
    e, bf, dev = len(rows_per_expert), torch.bfloat16, gpu_device
    args = [v.to(bf).to(dev) for v in (wg, wu, wd)]
    groups = (counts.to(dev), offsets.to(dev))
    ye, h = _abi.grouped_swiglu(xe.to(bf).to(dev), *groups, *args, e)
    for ex in range(e):
        lo, n = int(offsets[ex]), int(counts[ex])
        if n == 0:
            continue
        u = xe[lo : lo + n].double()
        h_ref = torch.nn.functional.silu(u @ wg[ex * d : (ex + 1) * d].double()) * (u @ wu[ex * d : (ex + 1) * d].double())
        assert_output_close(h[lo : lo + n], h_ref, "bf16", f"h of expert {ex}")
        y_ref = h[lo : lo + n].double().cpu() @ wd[ex * f : (ex + 1) * f].double()
        assert_output_close(ye[lo : lo + n], y_ref, "bf16", f"ye of expert {ex}")
    order = torch.randperm(xe.shape[0], generator=torch.Generator().manual_seed(d))
    scattered = torch.empty_like(xe)
    scattered[order] = xe
    ye_map, _ = _abi.grouped_swiglu(scattered.to(bf).to(dev), *groups, *args, e, row_map=order.to(torch.int32).to(dev))
    for w, k in zip(args, (d, d, f)):
        w[3 * k : 4 * k] = float("nan")
    ye_nan, _ = _abi.grouped_swiglu(xe.to(bf).to(dev), *groups, *args, e)
    for ex in range(e):
        sl = slice(int(offsets[ex]), int(offsets[ex]) + int(counts[ex]))
        assert torch.equal(ye_map[sl], ye[sl]), f"expert {ex} through the map"
        assert ex == 3 or torch.equal(ye_nan[sl], ye[sl]), f"expert {ex} next to NaN weights"


# The bf16 products choose their tile by how many of them a launch has (256 CUs): 64 x 64, 64 x 128, 128 x 128 and
# the throughput kernel's 256 x 256, in this order; rows on both sides of a tile's 64 and 128, N off its channels.
TILE_CASES = [
    ([1, 63, 64, 65, 0, 130], 200),
    ([128, 0, 129, 127, 200, 120], 1352),
    ([1290, 0, 129, 1581], 712),
    ([1290, 0, 257, 1581], 2056),
]


def _tile_case(counts, gen, dev):
    counts = torch.tensor(counts, dtype=torch.int32)
    blocks = (counts + 15) // 16 * 16
    offsets = torch.zeros(len(counts) + 1, dtype=torch.int32)
    offsets[1:] = blocks.cumsum(0)
    rows = int(offsets[-1]) + 15 * len(counts)
    return counts.to(dev), offsets.to(dev), rows, torch.randint(0, 500, (rows,), generator=gen, dtype=torch.int32).to(dev)


def _assert_products(got, pairs, what):
    """Every element within its rounding to bf16 and the rounding of a f32 sum of its products."""
    ref = sum(a.double() @ b.double() for a, b in pairs)
    size = sum(a.double().abs() @ b.double().abs() for a, b in pairs)
    terms = sum(a.shape[1] for a, _ in pairs)
    bound = 2.0**-8 * ref.abs() + (terms + 2) * 2.0**-24 * size + 1e-30
    worst = float(((got.double() - ref).abs() / bound).max())
    assert worst <= 1.0, f"{what}: {worst:.3f} of the bound"


@pytest.mark.parametrize("counts,n", TILE_CASES)
@pytest.mark.parametrize("k", [8, 64, 200, 328])
@pytest.mark.parametrize("layout", [_abi.W_IN_OUT, _abi.W_OUT_IN])
def test_products_on_every_tile_size(gpu_device, counts, n, k, layout):
    _say("tile sizes", counts, n, k, layout)
    g = torch.Generator().manual_seed(n + k)
    c, off, rows, row_map = _tile_case(counts, g, gpu_device)
    e = len(counts)
    x = torch.randn(500, k, generator=g).to(torch.bfloat16).to(gpu_device)
    w = torch.randn(e, k, n, generator=g).to(torch.bfloat16).to(gpu_device)
    b = (w if layout == _abi.W_IN_OUT else w.transpose(1, 2).contiguous()).reshape(-1, n if layout == _abi.W_IN_OUT else k)
    mapped = _abi.grouped_gemm(x, b, layout, c, off, e, row_map=row_map, rows=rows)
    copied = _abi.grouped_gemm(x[row_map.long()].contiguous(), b, layout, c, off, e)
    for i in range(e):
        sl = slice(int(off[i]), int(off[i]) + counts[i])
        if counts[i]:
            _assert_products(mapped[sl], [(x[row_map[sl].long()], w[i])], f"expert {i}")
            assert torch.equal(mapped[sl], copied[sl]), f"expert {i}: rows through the map"
    # all rows of one matrix
    _assert_products(_abi.grouped_gemm(x, b[: (k if layout == _abi.W_IN_OUT else n)], layout), [(x, w[0])], "dense")


@pytest.mark.parametrize("counts,n", TILE_CASES)
def test_pair_and_two_sources_on_every_tile_size(gpu_device, counts, n):
    """The gate/up product with both products kept, and the product of two sources; the pair without keeping, bit for
    bit the same."""
    _say("tile sizes, pair", counts, n)
    g = torch.Generator().manual_seed(n)
    c, off, rows, row_map = _tile_case(counts, g, gpu_device)
    e, k, n = len(counts), 192, (n + 63) // 64 * 64
    make = lambda *shape: (0.1 * torch.randn(*shape, generator=g)).to(torch.bfloat16).to(gpu_device)
    x, wg, wu, wd = make(500, k), make(e * k, n), make(e * k, n), make(e * n, k)
    ye, h, gk, uk = _abi.grouped_swiglu_keep(x, c, off, wg, wu, wd, e, row_map=row_map)
    ye2, h2 = _abi.grouped_swiglu(x, c, off, wg, wu, wd, e, row_map=row_map)
    summed = _abi.grouped_gemm_sum(gk, wg, uk, wu, c, off, e)  # (gradients of the same shapes, as it happens)
    for i in range(e):
        sl = slice(int(off[i]), int(off[i]) + counts[i])
        if not counts[i]:
            continue
        xr, ks, ns = x[row_map[sl].long()], slice(i * k, (i + 1) * k), slice(i * n, (i + 1) * n)
        _assert_products(gk[sl], [(xr, wg[ks])], f"g of expert {i}")
        _assert_products(uk[sl], [(xr, wu[ks])], f"u of expert {i}")
        h_ref = torch.nn.functional.silu(xr.double() @ wg[ks].double()) * (xr.double() @ wu[ks].double())
        assert_output_close(h[sl], h_ref.cpu(), "bf16", f"h of expert {i}")
        _assert_products(ye[sl], [(h[sl], wd[ns])], f"ye of expert {i}")
        _assert_products(summed[sl], [(gk[sl], wg[ks].t()), (uk[sl], wu[ks].t())], f"sum of expert {i}")
        assert torch.equal(ye[sl], ye2[sl]) and torch.equal(h[sl], h2[sl]), f"expert {i} without keeping"


# Gate/up of experts that are known to have at most 64 rows, on tiles as wide as the throughput kernel's: the same bits as
# from that kernel.  One stage of 64 k and fewer, as many as the ring's and more with a remainder; channels within a
# tile, past its half and past its end.
@pytest.mark.parametrize("d", [8, 64, 136, 200, 840])
@pytest.mark.parametrize("f", [1032, 1096, 1408])
def test_pair_of_experts_of_at_most_64_rows(gpu_device, d, f):
    _say("at most 64 rows", d, f)
    counts = [1, 32, 0, 33, 64, 63, 17, 5] + [3] * 72
    g = torch.Generator().manual_seed(d + f)
    c, off, rows, row_map = _tile_case(counts, g, gpu_device)
    e = len(counts)
    make = lambda *shape: (0.1 * torch.randn(*shape, generator=g)).to(torch.bfloat16).to(gpu_device)  # noqa: E731
    x, wg, wu, wd = make(500, d), make(e * d, f), make(e * d, f), make(e * f, d)

    def call(hint):
        return _abi.grouped_swiglu(x, c, off, wg, wu, wd, e, row_map=row_map, rows_per_expert=hint)

    (ye, h), (ye0, h0) = call(64), call(0)
    for i in range(e):
        sl = slice(int(off[i]), int(off[i]) + counts[i])
        assert torch.equal(h[sl], h0[sl]) and torch.equal(ye[sl], ye0[sl]), f"expert {i}"
    names = launched(lambda: call(64)), launched(lambda: call(0))
    assert names[0][0].startswith("glu_gemm_half_kernel<64, 256"), names
    assert names[1][0].startswith("glu_gemm_bf16_dma_kernel"), names


# The f32 products take tiles of 64 x 64, on which two groups of waves share the sum over K (the pair one), or of 128 x
# 128 (the pair 128 x 64) by the size of the buffers: the same bits.  Rows on both sides of 32, 64 and 128, experts
# without any, K within a chunk of 32, past its quarters and over several, N off the tiles' channels.
@pytest.mark.parametrize("k", [8, 24, 40, 200])
@pytest.mark.parametrize("n", [1024, 1000])
@pytest.mark.parametrize("layout", [_abi.W_IN_OUT, _abi.W_OUT_IN])
def test_f32_products_are_the_same_on_every_tile_size(gpu_device, k, n, layout):
    rows = [1, 16, 17, 33, 65, 0, 130, 700] + [0] * 16
    _say("f32 tiles", k, n, layout)
    e, g = len(rows), torch.Generator().manual_seed(k + n)
    counts = torch.tensor(rows, dtype=torch.int32, device=gpu_device)
    offsets = torch.zeros(e + 1, dtype=torch.int32, device=gpu_device)
    offsets[1:] = torch.cumsum((counts + 15) // 16 * 16, 0)
    lo = offsets.tolist()
    x, w, wu = torch.randn(20000, k, generator=g), torch.randn(e, k, n, generator=g), torch.zeros(e, k, n)
    # the pair's h is its gate product: a product of 20 and more with an up product of one
    x[:, -1], w[:, -1], wu[:, -1] = 1.0, 20.0 + 16 * k**0.5, 1.0
    x, w, wu = x.to(gpu_device), w.to(gpu_device), wu.to(gpu_device)
    b = (w if layout == _abi.W_IN_OUT else w.transpose(1, 2).contiguous()).reshape(-1, n if layout == _abi.W_IN_OUT else k)
    wd = torch.zeros(e * n, k, device=gpu_device)
    got = []
    for total in (lo[-1], 3000, 20000):
        out = [_abi.grouped_gemm(x[:total], b, layout, counts, offsets, e)]
        if layout == _abi.W_IN_OUT:
            out.append(_abi.grouped_swiglu(x[:total], counts, offsets, b, wu.reshape(-1, n), wd, e)[1])
        got += [torch.cat([o[lo[i] : lo[i] + r] for i, r in enumerate(rows)]) for o in out]
    for i, o in enumerate(got[1:], 1):
        assert torch.equal(o, got[0]), i
    ref = torch.cat([x[lo[i] : lo[i] + r].double() @ w[i].double() for i, r in enumerate(rows)])
    assert_output_close(got[0], ref.cpu(), "fp32")
    # all rows of one matrix: every group of rows in a launch of its own size
    first = b[: (k if layout == _abi.W_IN_OUT else n)]
    dense = [_abi.grouped_gemm(x[:r].contiguous(), first, layout) for r in (32, 33, 9000)]
    assert torch.equal(dense[0], dense[2][:32]) and torch.equal(dense[1], dense[2][:33])


# Tiles of 32 x 64 and of 64 x 64 by the rows and experts of a launch: the same bits, in both orientations of a matrix, for
# one product and two.
@pytest.mark.parametrize("k", [8, 32, 40, 72, 200])
@pytest.mark.parametrize("n", [1024, 1000])
def test_f32_products_on_flat_tiles(gpu_device, k, n):
    rows = [1, 16, 17, 33, 65, 0, 130, 31]
    _say("f32 flat tiles", k, n)
    g, many = torch.Generator(gpu_device).manual_seed(k + n), 128
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu_device)  # noqa: E731
    x, w, wu, wd = rnd(3000, k), rnd(many * k, n), rnd(many * k, n), rnd(many * n, k)
    wt = w.reshape(many, k, n).transpose(1, 2).contiguous().reshape(-1, k)
    kind = lambda name: name.rsplit(", ", 2)[-1] == "1>"  # noqa: E731
    seen, first = set(), None
    for e, total in ((8, 368), (8, 1000), (many, 3000)):
        counts = torch.tensor(rows + [0] * (e - 8), dtype=torch.int32, device=gpu_device)
        offsets = torch.zeros(e + 1, dtype=torch.int32, device=gpu_device)
        offsets[1:] = torch.cumsum((counts + 15) // 16 * 16, 0)
        lo, got = offsets.tolist(), []
        assert lo[-1] <= total
        names = launched(lambda: got.extend([
            _abi.grouped_gemm(x[:total], w[: e * k], _abi.W_IN_OUT, counts, offsets, e),
            _abi.grouped_gemm(x[:total], wt[: e * n], _abi.W_OUT_IN, counts, offsets, e),
            _abi.grouped_swiglu(x[:total], counts, offsets, w[: e * k], wu[: e * k], wd[: e * n], e)[1]]))
        assert all(m.startswith("glu_gemm_f32_kernel<") for m in names), names
        seen |= {(m.split("<")[1].split(",")[0], kind(m)) for m in names[:3]}
        out = [torch.cat([o[lo[i] : lo[i] + r] for i, r in enumerate(rows)]) for o in got]
        first = first or out
        assert all(torch.equal(a, b) for a, b in zip(out, first)), (e, total)
        assert torch.equal(out[0], out[1])
    assert seen == {(dual, flat) for dual in ("true", "false") for flat in (True, False)}, seen
    ref = torch.cat([x[lo[i] : lo[i] + r].double() @ w[i * k : (i + 1) * k].double() for i, r in enumerate(rows)])
    assert_output_close(first[0], ref.cpu(), "fp32")


# Weights of more than 320 MB are loaded past the caches where one block reads them (all experts), others through them (the
# first 8 of these experts alone): the same bits from every kernel that has both kinds of loads.  Which kernels a call
# takes, and which loads, is asked for: where "past the caches" stands among their template arguments, by name.
_PAST = {"glu_gemv_bf16_kernel": 2, "glu_gemv16_bf16_kernel": 2, "glu_gemm_half_kernel": 6, "glu_gemm_bf16_dma_kernel": 6,
         "glu_gemm_fp8w_kernel": 4, "glu_gemm_mx_kernel": 1}


class _PastTheCaches:
    def __init__(self, many, few, device):
        self.many, self.few, self.device, self.seen = many, few, device, set()

    def both(self, rows, total, run, everywhere=True):
        """``run(counts, offsets, experts, total)`` with all experts and with the first few: the same bits; past the
        caches with all of them (in every kernel, or in one) and never with a few."""
        out = []
        for e in (self.many, self.few):
            counts = torch.tensor(rows + [0] * (e - len(rows)), dtype=torch.int32, device=self.device)
            offsets = torch.zeros(e + 1, dtype=torch.int32, device=self.device)
            offsets[1:] = torch.cumsum((counts + 15) // 16 * 16, 0)
            lo, got = offsets.tolist(), []
            assert lo[-1] <= total
            names = [n.rstrip(">").split("<") for n in launched(lambda: got.extend(run(counts, offsets, e, total)))]
            loads = [(n, a.split(", ")) for n, a in (m for m in names if m[0] in _PAST)]
            past = [a[_PAST[n]] == "true" for n, a in loads]
            assert past and ((all if everywhere else any)(past) if e == self.many else not any(past)), (e, loads)
            self.seen |= {(n, ", ".join(a[2:4]) if n == "glu_gemm_half_kernel" else a[0]) for (n, a), p in zip(loads, past) if p}
            out.append([torch.cat([o[lo[i] : lo[i] + n] for i, n in enumerate(rows)]) for o in got])
        assert all(torch.equal(a, b) for a, b in zip(*out))


# K and N of whole units and lines, K off the units, and N off the lines (whose weights go through the caches)
@pytest.mark.parametrize("d,f", [(1024, 512), (1000, 512), (1024, 520)])
def test_weights_past_the_caches_give_the_same_bits(gpu_device, d, f):
    _say("past the caches", d, f)
    many, few, dev, bf = 128, 8, gpu_device, torch.bfloat16
    assert 3 * d * f * 2 * few < 320 << 20 < 3 * d * f * 2 * many
    g = torch.Generator(dev).manual_seed(d + f)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(bf)
    x, mid = rnd(100 * many, d), rnd(102 * many, f)
    wg, wu, wd = rnd(many * d, f) * 0.05, rnd(many * d, f) * 0.05, rnd(many * f, d) * 0.05
    check, whole = _PastTheCaches(many, few, dev), d % 64 == 0 and f % 64 == 0
    w = lambda e: (wg[: e * d], wu[: e * d], wd[: e * f])
    swiglu = lambda **kw: lambda c, o, e, t: _abi.grouped_swiglu(x[:t], c, o, *w(e), e, **kw)
    if whole:
        for bound, rows in ((1, [1] * 8), (2, [2, 1, 2, 0, 2, 2, 2, 2]), (4, [4, 1, 3, 4, 4, 2, 4, 4]),
                            (8, [8, 1, 5, 0, 7, 8, 8, 3]), (16, [16, 9, 1, 0, 12, 16, 5, 16])):
            check.both(rows, 128, swiglu(rows_per_expert=bound))
    rows = [300, 17, 0, 256, 257, 129, 1, 64]
    # buffers that may hold 32 rows besides padding, of a few rows an expert (small tiles), and of more (large ones)
    for total in (32 + 15 * many, 100 * many):
        check.both(rows, total, swiglu(), whole)
        if _abi.keeps_products(d, f, total, bf):
            check.both(rows, total, lambda c, o, e, t: _abi.grouped_swiglu_keep(x[:t], c, o, *w(e), e), whole)
            check.both(rows, total, lambda c, o, e, t: [
                _abi.grouped_gemm_sum(mid[:t], w(e)[0], mid[200 : 200 + t], w(e)[1], c, o, e)], whole)
        if d % 64 == 0:
            check.both(rows, total, lambda c, o, e, t: [_abi.grouped_gemm(x[:t], w(e)[2], _abi.W_OUT_IN, c, o, e)], whole)
    # (small tiles: two products, and the matrices' orientation)
    single = {("glu_gemm_half_kernel", "false, 0"), ("glu_gemm_bf16_dma_kernel", "false")}
    dual = {("glu_gemm_half_kernel", "true, 0"), ("glu_gemm_bf16_dma_kernel", "true")}
    streams = {(n, two) for n in ("glu_gemv_bf16_kernel", "glu_gemv16_bf16_kernel") for two in ("true", "false")}
    assert check.seen >= (single | dual | streams | {("glu_gemm_half_kernel", "false, 1")} if whole else
                          single if f % 64 else dual), check.seen


# The same of e4m3 weights, with rows of bf16 and block-scaled ones: many experts, whose launches take the stream and large
# tiles, and fewer with a long K, whose gate/up takes small ones.
@pytest.mark.parametrize("many,d,f", [(128, 2048, 768), (32, 9216, 384)])
def test_e4m3_weights_past_the_caches_give_the_same_bits(gpu_device, many, d, f):
    _say("e4m3 past the caches", many, d, f)
    few, dev, bf = 8, gpu_device, torch.bfloat16
    assert 3 * d * f * few < 320 << 20 < 3 * d * f * many
    g = torch.Generator(dev).manual_seed(d + f)
    codes = lambda k, n: (torch.randn(many * k, n, generator=g, device=dev) * 0.05).to(torch.float8_e4m3fn)
    packed = [_abi.pack_fp8_weights(codes(k, n), many) for k, n in ((d, f), (d, f), (f, d))]
    scales = [torch.rand(many, n, generator=g, device=dev) + 0.5 for n in (f, f, d)]
    w = lambda e: dict(scales=tuple(s[:e] for s in scales))
    x = torch.randn(5632, d, generator=g, device=dev).to(bf)
    check = _PastTheCaches(many, few, dev)
    swiglu = lambda pairs: lambda c, o, e, t: _abi.grouped_swiglu(
        x[:t], c, o, *(q[:e] for q in packed), e, pairs=pairs(e), **w(e))
    if many == 128:
        for pairs in (96, 480):  # pieces of one and of two groups of channels
            check.both([16, 17, 1, 0, 33, 2, 9, 16], 480, swiglu(lambda e: min(pairs, 26 * e)))
        rows, mx_total = [300, 17, 0, 256, 257, 129, 1, 64], 44 * many
    else:
        rows, mx_total = [60, 17, 0, 100, 64, 129, 1, 65], 31 * many
    check.both(rows, 27 * many + 600, swiglu(lambda e: 27 * many))
    xq, xs = _abi.mx_quantize(x[:mx_total].contiguous())
    check.both(rows, mx_total, lambda c, o, e, t: _abi.grouped_swiglu_w8a8(
        xq, xs, c, o, *(q[:e] for q in packed), w(e)["scales"], e)[:2])
    duals = lambda *names: {(n, dual) for n in names for dual in ("true", "false")}
    assert check.seen >= (duals("glu_gemm_fp8w_kernel", "glu_gemm_bf16_dma_kernel", "glu_gemm_mx_kernel") if many == 128 else
                          {("glu_gemm_half_kernel", "true, 2"), ("glu_gemm_half_kernel", "true, 3"),
                           ("glu_gemm_bf16_dma_kernel", "false"), ("glu_gemm_mx_kernel", "false")}), check.seen


# The shared expert's weights are loaded past the caches where their rows begin on lines: off them a line is read twice.
@pytest.mark.parametrize("d,f,past", [(4096, 8192, True), (4104, 8192, False), (4096, 8200, False), (5160, 8232, False)])
def test_shared_expert_off_the_lines_goes_through_the_caches(gpu_device, d, f, past):
    _say("shared expert on lines", d, f)
    x = torch.randn(3, d, device=gpu_device).bfloat16()
    w = [torch.randn(*s, device=gpu_device).bfloat16() * 0.02 for s in ((f, d), (f, d), (d, f))]
    names = launched(lambda: _abi.dense_swiglu(x, *w))
    flag = str(past).lower()
    assert names == [f"dense_gemv_bf16_kernel<true, {flag}>", f"dense_gemv_bf16_kernel<false, {flag}>"]


# Which tiles products of bf16 take follows from the size of the buffers (one round of small ones, several rounds of
# few rows, the throughput kernel): the same bits, with few experts' tiles about one a compute unit and several a unit,
# rows on both sides of a tile's 64 in one expert, K and N off the units.
@pytest.mark.parametrize("e,d,f", [(8, 1024, 2048), (32, 1000, 1416)])
def test_products_of_few_rows_are_the_same_on_every_tile_size(gpu_device, e, d, f):
    _say("tiles of few rows", e, d, f)
    dev, bf = gpu_device, torch.bfloat16
    g = torch.Generator(dev).manual_seed(e)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(bf)
    rows = [130, 1, 0, 64, 65, 17, 0, 33] + [0, 2] * (e // 2 - 4)
    counts = torch.tensor(rows, dtype=torch.int32, device=dev)
    offsets = torch.zeros(e + 1, dtype=torch.int32, device=dev)
    offsets[1:] = torch.cumsum((counts + 15) // 16 * 16, 0)
    lo = offsets.tolist()
    x, wg, wu, wd = rnd(400 * e, d), rnd(e * d, f) * 0.05, rnd(e * d, f) * 0.05, rnd(e * f, d) * 0.05
    got = []
    for total in (lo[-1], 24 * e + lo[-1], 48 * e + lo[-1], 80 * e + lo[-1], 400 * e):
        out = list(_abi.grouped_swiglu(x[:total], counts, offsets, wg, wu, wd, e))
        out.append(_abi.grouped_gemm(x[:total], wd, _abi.W_OUT_IN, counts, offsets, e))
        got.append([torch.cat([o[lo[i] : lo[i] + n] for i, n in enumerate(rows)]) for o in out])
    assert all(torch.equal(a, b) for o in got[:-1] for a, b in zip(o, got[-1]))
    for i, n in enumerate(rows):
        if n == 0:
            continue
        ref = O.glu_expert(*(t.double() for t in (x[lo[i] : lo[i] + n], wg[i * d : (i + 1) * d], wu[i * d : (i + 1) * d],
                                                  wd[i * f : (i + 1) * f])))
        at = sum(rows[:i])
        assert_output_close(got[0][0][at : at + n], ref.cpu(), "bf16", f"expert {i}")


# How many rows and channels a piece of the e4m3 stream's work has follows from the rows that the caller says: the same
# bits, for rows on both sides of 16 and 32, K within a step, past one and split over two waves, against the oracle.
@pytest.mark.parametrize("d,f", [(512, 1024), (448, 704), (1088, 64)])
def test_e4m3_streams_of_every_chunk_are_the_same(gpu_device, d, f):
    _say("e4m3 stream", d, f)
    e, dev, bf = 32, gpu_device, torch.bfloat16
    g = torch.Generator(dev).manual_seed(d)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(bf)
    rows = [33, 32, 17, 16, 1, 0, 48, 31] + [0] * (e - 10) + [40, 5]
    counts = torch.tensor(rows, dtype=torch.int32, device=dev)
    offsets = torch.zeros(e + 1, dtype=torch.int32, device=dev)
    offsets[1:] = torch.cumsum((counts + 15) // 16 * 16, 0)
    lo = offsets.tolist()
    x = rnd(lo[-1], d)
    codes = [(rnd(e * i, o) * 0.05).to(torch.float8_e4m3fn) for i, o in ((d, f), (d, f), (f, d))]
    packed = [_abi.pack_fp8_weights(c, e) for c in codes]
    scales = [torch.rand(e, n, generator=g, device=dev) + 0.5 for n in (f, f, d)]
    got, variants = [], []
    for pairs in (3 * e, 5 * e, lo[-1], 0):
        def run():
            out = _abi.grouped_swiglu(x, counts, offsets, *packed, e, scales=tuple(scales), pairs=pairs)
            got.append([torch.cat([o[lo[i] : lo[i] + n] for i, n in enumerate(rows)]) for o in out])
        variants.append([n.split("<")[1] for n in launched(run) if n.startswith("glu_gemm_fp8w_kernel")])
    assert 8 * e < lo[-1] <= 23 * e  # (0: what such buffers hold besides padding to 16 may be few rows)
    up, down = (4 if d >= 512 else 2), (4 if f >= 512 else 2)  # waves along K
    groups = (1, 2, 2, 2) if d >= 512 else (1, 1, 1, 1)
    assert variants == [[f"true, {up}, {c}, {fr}, false>", f"false, {down}, {4 if f >= 512 else 2}, {fr}, false>"]
                        for c, fr in zip(groups, (1, 1, 2, 1))]
    assert all(torch.equal(a, b) for o in got[1:] for a, b in zip(o, got[0]))
    for i, n in enumerate(rows):
        if n == 0:
            continue
        w = [c[i * k : (i + 1) * k].double() * s[i].double() for c, s, k in zip(codes, scales, (d, d, f))]
        ref = O.glu_expert(x[lo[i] : lo[i] + n].double(), *w)
        at = sum(rows[:i])
        assert_output_close(got[0][0][at : at + n], ref.cpu(), "bf16", f"expert {i}")


# f32 products of many rounds take large tiles; rows and channels past them, one product, its transpose and two at once:
# the bits of launches of a few rows, which take small ones.
def test_f32_products_on_large_tiles(gpu_device):
    rows, k, n = 8190, 40, 2040
    _say("f32 large tiles", rows, k, n)
    g = torch.Generator(gpu_device).manual_seed(1)
    x, w, wu = (torch.randn(*s, generator=g, device=gpu_device) for s in ((rows, k), (k, n), (k, n)))
    wd = torch.zeros(n, k, device=gpu_device)
    group = lambda m: (torch.tensor([m], dtype=torch.int32, device=gpu_device),
                       torch.tensor([0, m], dtype=torch.int32, device=gpu_device))
    runs = (lambda a: _abi.grouped_gemm(a, w, _abi.W_IN_OUT),
            lambda a: _abi.grouped_gemm(a, w.t().contiguous(), _abi.W_OUT_IN),
            lambda a: _abi.grouped_swiglu(a, *group(a.shape[0]), w, wu, wd, 1)[1])
    for run in runs:
        whole = run(x)
        for lo in (0, 4096, 8126):
            assert torch.equal(run(x[lo : lo + 64].contiguous()), whole[lo : lo + 64])
    assert_output_close(runs[0](x[:300]), (x[:300].double() @ w.double()).cpu(), "fp32")


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize(
    "t,d,f",
    [
        (200, 128, 256), (37, 72, 40), (1, 64, 64), (600, 192, 320),
        # up to 16 bf16 rows stream the weights (K off the 32-wide steps, N off the 16-channel blocks)
        (1, 5120, 1024), (3, 72, 40), (8, 2048, 768), (16, 1000, 200), (16, 8, 8), (17, 256, 128),
    ],
)
def test_dense_swiglu_matches_oracle(gpu_device, dtype, t, d, f):
    _say("dense_swiglu", dtype, t, d, f)
    g = torch.Generator().manual_seed(t)
    dt = TORCH_DTYPE[dtype]
    x = torch.randn(t, d, generator=g).to(dt).float()
    wg, wu, wd = (0.05 * torch.randn(*s, generator=g) for s in ((f, d), (f, d), (d, f)))
    wg, wu, wd = (w.to(dt).float() for w in (wg, wu, wd))
    y = _abi.dense_swiglu(*(v.to(dt).to(gpu_device) for v in (x, wg, wu, wd)))
    ref = O.shared_glu(x.double(), wg.double(), wu.double(), wd.double())
    assert_output_close(y, ref, dtype, "shared expert")


@pytest.mark.parametrize(
    "rows,d,f,experts",
    [
        # tiles of 256 rows x 256 channels on 256 blocks.  Down projection (1 channel tile): 258 row
        # tiles, the last of 208 rows: the two left over by the one whole round go out as halves,
        # the second half of the last one 80 rows; gate/up (2 channel tiles): 516 tiles, 4 left over
        (66000, 256, 256, 1),
        # two experts of 198 + 99 row tiles (the last of each partly filled): 41 left over, as halves
        (76000, 256, 128, 2),
        # 384 + 1 tiles: 129 left over would be 258 halves, one too many: dealt whole
        (98560, 256, 128, 1),
    ],
)
def test_tiles_around_the_last_round_of_the_deal(gpu_device, rows, d, f, experts):
    """The throughput kernel deals its tiles round-robin to one block per CU and splits the heavy
    tiles that do not fill a round into halves when they then fit one round: shapes on both sides of
    that rule, the grouped experts reading their rows through a map and the dense network, checked
    on sampled rows (every row depends on its own tile only)."""
    _say("last round of the deal", rows, d, f, experts)
    g = torch.Generator().manual_seed(rows)
    dev = gpu_device
    tokens = 4096
    x = torch.randn(tokens, d, generator=g).to(torch.bfloat16)
    row_map = torch.randint(0, tokens, (rows,), generator=g, dtype=torch.int32)
    first = rows * 2 // 3 if experts == 2 else rows
    counts = torch.tensor([first, rows - first][:experts], dtype=torch.int32)
    offsets = torch.tensor([0, first, rows][: experts + 1], dtype=torch.int32)
    wg, wu = (0.05 * torch.randn(experts * d, f, generator=g) for _ in range(2))
    wd = 0.05 * torch.randn(experts * f, d, generator=g)
    wg, wu, wd = (w.to(torch.bfloat16) for w in (wg, wu, wd))
    ye, _ = _abi.grouped_swiglu(x.to(dev), counts.to(dev), offsets.to(dev), wg.to(dev), wu.to(dev), wd.to(dev),
                                experts, row_map=row_map.to(dev))
    torch.cuda.synchronize()
    # the first and last rows of every tile boundary region, and a random sample
    pick = torch.cat([torch.arange(0, 3), torch.arange(rows - 400, rows), torch.arange(first - 200, min(first + 200, rows)),
                      torch.randint(0, rows, (300,), generator=g)]).unique()
    got = ye[pick.to(dev)]
    for e in range(experts):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        sel = (pick >= lo) & (pick < hi)
        if not bool(sel.any()):
            continue
        xr = x[row_map[pick[sel]].long()].double()
        ref = O.glu_expert(xr, wg[e * d : (e + 1) * d].double(), wu[e * d : (e + 1) * d].double(),
                           wd[e * f : (e + 1) * f].double())
        assert_output_close(got[sel.to(dev)], ref, "bf16", f"expert {e}")
    if experts == 1:
        # the same rows through the dense network (nn.Linear-oriented weights, no map)
        xs = x[row_map.long()].contiguous()
        y = _abi.dense_swiglu(xs.to(dev), wg.t().contiguous().to(dev), wu.t().contiguous().to(dev),
                              wd.t().contiguous().to(dev))
        ref = O.shared_glu(xs[pick].double(), wg.t().double(), wu.t().double(), wd.t().double())
        assert_output_close(y[pick.to(dev)], ref, "bf16", "dense network")


# ----------------------------------------------------------------------------------------- combine
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("weight_output", [False, True])
@pytest.mark.parametrize("with_base", [False, True])
@pytest.mark.parametrize("k", [4, 3, 7, 12])  # also values below the kernel's compile-time bounds 4, 8, 16
def test_combine_matches_oracle(gpu_device, dtype, weight_output, with_base, k):
    _say("combine", dtype, weight_output, with_base, k)
    g = torch.Generator().manual_seed(21)
    t, d, e = 777, 128, 12
    dt = TORCH_DTYPE[dtype]
    logits = torch.randn(t, e, generator=g)
    idx = O.topk_lowest_index(logits, k)
    w = O.combine_weights(logits, idx, "softmax", True).float()
    r = O.route(idx, e, 16)
    ye = torch.randn(r.num_rows, d, generator=g).to(dt).float()
    base = torch.randn(t, d, generator=g).to(dt).float() if with_base else None
    dev = gpu_device
    out = _abi.combine(
        ye.to(dt).to(dev), torch.from_numpy(r.inv_perm).to(dev), idx.to(torch.int32).to(dev), w.to(dev),
        None if base is None else base.to(dt).to(dev), weight_output,
    )
    # f32 accumulation in ascending expert id from the base, one rounding at the end
    acc = base.clone() if with_base else torch.zeros(t, d)
    order = torch.argsort(idx, dim=1)
    rows = torch.from_numpy(r.inv_perm.astype(np.int64))
    for j in range(k):
        slot = order[:, j]
        y = ye[rows[torch.arange(t), slot]]
        if weight_output:
            acc = torch.addcmul(acc, y, w[torch.arange(t), slot][:, None]) if False else acc + w[torch.arange(t), slot][:, None] * y
        else:
            acc = acc + y
    want = acc.to(dt).float()
    got = out.float().cpu()
    if not weight_output:
        assert torch.equal(got, want), "unweighted combine must be bit-exact"
    else:
        # the device may fuse the multiply-add; allow one ulp of the output type
        assert_output_close(out, acc, dtype)
        assert float((got - want).abs().max()) <= float(want.abs().max()) * (2**-7 if dtype == "bf16" else 2**-22)


# One, two and four waves a token, through the caches and past them, rows off a wave's pieces, lists shorter than the
# compile-time one: without weights the sum is bit-exact.
@pytest.mark.parametrize("t,d,k,dtype", [(2048, 512, 3, "bf16"), (2049, 2056, 6, "bf16"), (2300, 2048, 8, "bf16"),
                                         (4100, 1032, 9, "bf16"), (2048, 4096, 5, "bf16"), (2050, 1028, 4, "fp32"),
                                         (2047, 4096, 2, "bf16")])
def test_combine_by_rows_and_tokens(gpu_device, t, d, k, dtype):
    _say("combine", t, d, k, dtype)
    g, dev, dt = torch.Generator(gpu_device).manual_seed(t + d), gpu_device, TORCH_DTYPE[dtype]
    idx = torch.rand(t, 32, generator=g, device=dev).argsort(dim=1)[:, :k]
    inv = torch.randperm(t * k, generator=g, device=dev).view(t, k)
    ye, base = (torch.randn(n, d, generator=g, device=dev).to(dt) for n in (t * k, t))
    out = _abi.combine(ye, inv.to(torch.int32), idx.to(torch.int32).contiguous(), torch.rand(t, k, device=dev), base, False)
    acc, order = base.float(), idx.argsort(dim=1)
    for j in range(k):
        acc = acc + ye[inv.gather(1, order[:, j : j + 1])[:, 0]].float()
    assert torch.equal(out, acc.to(dt))


# Pairs without a row (-1), first, in between, last and all of a token's, in lists of every compile-time length: what they
# load in a row's place is not ye's first row, and adds nothing.
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("t", [3, 2100])
@pytest.mark.parametrize("k", [1, 2, 3, 5, 8, 9, 10, 11, 17])
def test_combine_of_pairs_without_rows(gpu_device, t, k, dtype):
    _say("combine without rows", t, k, dtype)
    d, dev, dt = 520, gpu_device, TORCH_DTYPE[dtype]
    g = torch.Generator(dev).manual_seed(t + k)
    idx = torch.rand(t, 32, generator=g, device=dev).argsort(dim=1)[:, :k].to(torch.int32).contiguous()
    inv = 1 + torch.randperm(t * k, generator=g, device=dev).view(t, k).to(torch.int32)
    order = idx.argsort(dim=1)
    inv[0] = -1
    inv[1, order[1, 0]] = -1
    inv[2::2, order[2, k // 2]] = -1
    ye = torch.randn(t * k + 1, d, generator=g, device=dev).to(dt)
    ye[0] = float("nan")
    base = torch.randn(t, d, generator=g, device=dev).to(dt)
    out = _abi.combine(ye, inv, idx, torch.rand(t, k, device=dev), base, False)
    acc = base.float()
    for j in range(k):
        row = inv.gather(1, order[:, j : j + 1])
        acc = acc + torch.where(row >= 0, ye[row[:, 0].clamp(min=0)].float(), 0.0)
    assert torch.equal(out, acc.to(dt))
    assert torch.equal(_abi.combine(ye[1:2], torch.full_like(inv, -1), idx, None, base, False), base)
    assert float(_abi.combine(ye[1:2], torch.full_like(inv, -1), idx, None, None, False).float().abs().max()) == 0.0


# ------------------------------------------------------------------------ experts, fp8 weights
@pytest.mark.parametrize(
    "rows_per_expert,d,f",
    [
        ([5, 0, 17, 64, 1, 11, 0, 33], 128, 192),  # decode-like: few rows, empty experts
        ([100, 3], 64, 64),  # more than 64 rows: weights re-streamed per 64-row chunk
        # 64 or more rows per expert on average: the throughput kernel (codes turned into bf16 on
        # the way to LDS, scales in its epilogue); ragged last tiles, an empty expert, F and D that
        # leave the last channel tile partly (192 = 128 + 64) or mostly (128 of 256) empty
        ([300, 0, 70, 513, 1, 129, 256, 40], 128, 192),
        ([700, 260], 64, 64),
        ([257, 255, 31, 1000], 320, 448),
    ],
)
def test_grouped_swiglu_fp8_weights_match_oracle(gpu_device, rows_per_expert, d, f):
    _say("grouped_swiglu fp8", rows_per_expert, d, f)
    counts, offsets, xe, wg, wu, wd = _expert_case("bf16", rows_per_expert, d, f, seed=3 * d + f)
    e = len(rows_per_expert)
    qs = [W.quantize_fp8_per_channel(w, e) for w in (wg, wu, wd)]
    deq = [W.dequantize_fp8_per_channel(q, s) for q, s in qs]
    dev = gpu_device

    def kernel_layout(q, k, n):  # (E*k, n) -> 1 KB tiles (E, n/16, k/64, 16, 64)
        packed = _abi.pack_fp8_weights(q, e)
        assert packed.shape == (e, n // 16, k // 64, 16, 64)
        # tile [t, c, b] row i, byte j is weight (in = 64 b + j, out = 16 c + i) of expert t
        ref = q.view(torch.uint8).view(e, k, n)
        pk = packed.view(torch.uint8)
        assert int(pk[e - 1, 1, 0, 3, 5]) == int(ref[e - 1, 5, 16 + 3])
        return packed.to(dev)

    ye, h = _abi.grouped_swiglu(
        xe.to(torch.bfloat16).to(dev), counts.to(dev), offsets.to(dev),
        kernel_layout(qs[0][0], d, f), kernel_layout(qs[1][0], d, f), kernel_layout(qs[2][0], f, d), e,
        scales=tuple(s.to(dev) for _, s in qs),
    )
    for ex in range(e):
        lo, n = int(offsets[ex]), int(counts[ex])
        if n == 0:
            continue
        u = xe[lo : lo + n].double()
        g_, u_, d_ = (deq[0][ex * d : (ex + 1) * d].double(), deq[1][ex * d : (ex + 1) * d].double(), deq[2][ex * f : (ex + 1) * f].double())
        h_ref = torch.nn.functional.silu(u @ g_) * (u @ u_)
        assert_output_close(h[lo : lo + n], h_ref, "bf16", f"h of expert {ex}")
        assert_output_close(ye[lo : lo + n], O.glu_expert(u, g_, u_, d_), "bf16", f"expert {ex}")
