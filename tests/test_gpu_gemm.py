"""W4A16 linears of more than 16 rows (the matrix-core GEMM) against the float64
oracle, at the edges of its tiles and of its dispatch."""
import numpy as np
import pytest
import torch

from gemmainfer_amd import _lib as L
from gemmainfer_amd import ops, synth
from oracle import moe_oracle as O

from helpers import assert_dtype_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _f64(t):
    return t.float().cpu().numpy().astype(np.float64)


def _operands(m, k, n, gs, dtype, seed=0):
    B, S = synth.linear_weights(k, n, gs, seed=seed)
    x = synth.activations(m, k, seed=seed)
    return x.to(dtype).to(DEV), B.to(DEV), S.to(dtype).to(DEV)


def _check(y, ref, dtype):
    assert_dtype_close(y, ref, "bf16" if dtype == torch.bfloat16 else "fp16")


# rows: one past 16, the 16-, 32- and 64-row tiles' edges, several row blocks;
# one and two k blocks per unit at each row tile count; columns: N = 4 mod 64 and
# mod 256, one tile; K: 8 mod 32, less than a unit, a last group cut short, one
# past a chunk; enough tiles for the large kernel
SHAPES = [(17, 64, 64, 64), (17, 264, 132, 32), (32, 200, 68, 96), (32, 136, 68, 64), (33, 512, 200, 64),
          (64, 2816, 260, 64), (65, 704, 132, 128), (40, 96, 68, 32), (70, 200, 36, 64), (61, 1000, 300, 192),
          (16 * 5 + 1, 264, 4, 96), (129, 8200, 64, 64), (1281, 264, 2052, 64), (1300, 520, 2304, 32),
          (2049, 200, 1284, 128), (640, 2816, 4096, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,n,gs", SHAPES)
def test_gemm_parity(m, k, n, gs, dtype):
    x, B, S = _operands(m, k, n, gs, dtype, seed=m)
    y = ops.w4a16_linear(x, B, S, gs)
    ref = O.w4a16_linear(_f64(x), B.cpu().numpy(), _f64(S), gs)
    _check(y, ref, dtype)
    assert torch.equal(y, ops.w4a16_linear(x, B, S, gs))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m", [33, 1100])
def test_gemm_softcap_and_floor_groups(m, dtype):
    """Softcap epilogue; scales with fewer groups than K spans (the rows past
    the last group are dropped, an infinity or NaN in a dropped column with
    them), on the small tiles and on the large ones; scales with more groups."""
    k, n, gs = 320, 2560, 128
    x, B, S = _operands(m, k, n, gs, dtype, seed=3)
    full = ops.w4a16_linear(x, B, S, gs, softcap=3.0)
    assert torch.equal(full, ops.w4a16_linear(x, B, torch.cat([S, S + 1]), gs, softcap=3.0))
    S = S[: k // gs].contiguous()
    x[3, 256], x[m - 1, 319], x[m // 2, 300] = float("inf"), float("nan"), float("-inf")
    y = ops.w4a16_linear(x, B, S, gs, softcap=3.0)
    kk = (k // gs) * gs
    ref = O.w4a16_linear(_f64(x)[:, :kk], B[: kk // 8].cpu().numpy(), _f64(S), gs)
    _check(y, 3.0 * np.tanh(ref / 3.0), dtype)


@pytest.mark.parametrize("m", [40, 1100])
def test_gemm_multi_unequal_group_counts(m):
    """Projections of one call whose scales end at different groups: each drops
    its own columns, with an infinity in one that only the first keeps."""
    k, gs = 456, 64
    x = synth.activations(m, k, seed=m).to(DEV)
    x[5, 450] = float("inf")
    ws = [tuple(t.to(DEV) for t in synth.linear_weights(k, n, gs, seed=n)) for n in (1092, 256, 520)]
    ws[1] = (ws[1][0], ws[1][1][:7].contiguous())
    ws[2] = (ws[2][0], ws[2][1][:4].contiguous())
    ys = ops.w4a16_linear_multi(x, ws, gs)
    keep = [i for i in range(m) if i != 5]
    for i, (y, (B, S)) in enumerate(zip(ys, ws)):
        kk = min(k, S.shape[0] * gs)
        xi, yi = (x[keep], y[keep]) if i == 0 else (x, y)
        _check(yi, O.w4a16_linear(_f64(xi)[:, :kk], B[: kk // 8].cpu().numpy(), _f64(S), gs), torch.bfloat16)
    assert not torch.isfinite(ys[0][5].float()).any()


def _check_gated(got, g, u):
    """gelu(g) * u of the projections' bf16 outputs, as the torch statements round it."""
    want = torch.nn.functional.gelu(g.float(), approximate="tanh").to(torch.bfloat16) * u
    # the two may sum K in different orders, so the rounding of a gate or up
    # value may fall the other way: an ulp (at most 2^-7 of the value) of the
    # gate through gelu's largest slope 1.13, of gelu's own rounding, of the up
    # value, and of the result
    g, u, w = g.float(), u.float(), want.float()
    gel = torch.nn.functional.gelu(g, approximate="tanh")
    bound = 2.0 ** -7 * ((1.13 * g.abs() + 2 * gel.abs()) * u.abs() + w.abs()) + 1e-6
    assert torch.all((got.float() - w).abs() <= bound)


@pytest.mark.parametrize("m", [24, 50, 1500])
def test_gemm_multi_and_gated(m):
    """Several projections in one grid against the oracle; the gated form keeps the torch statements' roundings."""
    k, gs = 456, 64
    x = synth.activations(m, k, seed=m).to(DEV)
    ws = [tuple(t.to(DEV) for t in synth.linear_weights(k, n, gs, seed=n)) for n in (1092, 256, 4)]
    for y, (B, S) in zip(ops.w4a16_linear_multi(x, ws, gs), ws):
        _check(y, O.w4a16_linear(_f64(x), B.cpu().numpy(), _f64(S), gs), torch.bfloat16)
    gate, up = (tuple(t.to(DEV) for t in synth.linear_weights(k, 1092, gs, seed=s)) for s in (7, 8))
    g, u = (ops.w4a16_linear(x, *w, gs) for w in (gate, up))
    _check_gated(ops.gated_mlp_act(x, gate, up, gs), g, u)


@pytest.mark.parametrize("gs", [64, 32])
@pytest.mark.parametrize("m", [24, 50, 1500])
def test_gated_unequal_group_counts(m, gs):
    """Gate and up scales with different group counts (one covers all of K, the
    other drops the rows of the last, partial group): every token row keeps
    each projection's own rows, on the small tiles and on the large ones."""
    k, n = 456, 1092
    x = synth.activations(m, k, seed=m + gs).to(DEV)
    gate, up = (tuple(t.to(DEV) for t in synth.linear_weights(k, n, gs, seed=s)) for s in (17, 18))

    def short(w):
        return w[0], w[1][: k // gs].contiguous()

    def oracle(w):
        kk = min(k, w[1].shape[0] * gs)
        y = O.w4a16_linear(_f64(x)[:, :kk], w[0][: kk // 8].cpu().numpy(), _f64(w[1]), gs)
        return torch.from_numpy(y).to(torch.bfloat16)

    for gt, u in ((short(gate), up), (gate, short(up)), (short(gate), short(up))):
        _check_gated(ops.gated_mlp_act(x, gt, u, gs).cpu(), oracle(gt), oracle(u))


def test_gemm_output_at_any_element():
    """An output that starts at an odd element (2-byte aligned only), and one
    whose rows are strided, through the drop-in's write semantics."""
    for m in (30, 1200):
        k, n, gs = 264, 2564, 64
        x, B, S = _operands(m, k, n, gs, torch.bfloat16, seed=1)
        want = ops.w4a16_linear(x, B, S, gs)
        flat = torch.zeros(m * n + 3, dtype=torch.bfloat16, device=DEV)
        C = flat[3:].view(m, n)
        ops.marlin_w4a16(x, B, S, C, gs)
        assert torch.equal(C, want) and not flat[:3].any()
        wide = torch.zeros(m, n + 5, dtype=torch.bfloat16, device=DEV)
        ops.marlin_w4a16(x, B, S, wide[:, 3:n + 3], gs)
        assert torch.equal(wide[:, 3:n + 3], want) and not wide[:, :3].any() and not wide[:, n + 3:].any()


def test_gemm_rows_with_inf_stay_apart():
    """A row with an infinity, and padding rows, leave the other rows alone."""
    for m in (19, 1200):
        k, n, gs = 256, 2304, 64
        x, B, S = _operands(m, k, n, gs, torch.bfloat16, seed=2)
        want = ops.w4a16_linear(x, B, S, gs)
        x[5, 7] = float("inf")
        y = ops.w4a16_linear(x, B, S, gs)
        keep = [i for i in range(m) if i != 5]
        assert torch.equal(y[keep], want[keep])
        assert not torch.isfinite(y[5].float()).all()


def test_gemm_without_its_workspace():
    """A caller whose workspace holds less than the query is still served where
    the general kernel needs none."""
    m, k, n, gs = 20, 64, 65536 + 64, 64
    x, B, S = _operands(m, k, n, gs, torch.bfloat16, seed=4)
    y = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    p = lambda t: t.data_ptr()  # noqa: E731
    st = L.load().gi_w4a16_linear(p(x), L.DTYPE_BF16, p(B), p(S), S.shape[0], p(y), m, k, n, gs, 0.0, None, 0,
                                  torch.cuda.current_stream().cuda_stream)
    assert st == L.GI_OK
    ref = O.w4a16_linear(_f64(x), B[:, :512].cpu().numpy(), _f64(S[:, :512]), gs)
    _check(y[:, :512], ref, torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("most", [320, 512, 1024])
def test_one_workspace_for_the_largest_call(dtype, most):
    """One workspace, sized for a program's largest row count, serves calls of
    every smaller one, linear and gated, whatever their K
    split: the same results as with a workspace of their own."""
    k, n, gs = 2816, 4096, 64
    lib, stream = L.load(), torch.cuda.current_stream().cuda_stream
    p = lambda t: t.data_ptr()  # noqa: E731
    code = L.DTYPE_BF16 if dtype == torch.bfloat16 else L.DTYPE_FP16
    ws = torch.zeros(max(lib.gi_w4a16_workspace_bytes(most, k, n, gs),
                         lib.gi_w4a16_gated_mlp_workspace_bytes(most, k, n, gs)) + 256, dtype=torch.uint8, device=DEV)
    base = p(ws) + -p(ws) % 256
    for m in (64, 17, 3, 192, 16, 64):
        x, B, S = _operands(m, k, n, gs, dtype, seed=m)
        y = torch.empty(m, n, dtype=dtype, device=DEV)
        size = lib.gi_w4a16_workspace_bytes(most, k, n, gs)
        assert lib.gi_w4a16_linear(p(x), code, p(B), p(S), S.shape[0], p(y), m, k, n, gs, 0.0, base, size,
                                   stream) == L.GI_OK, (m, lib.gi_last_error())
        assert torch.equal(y, ops.w4a16_linear(x, B, S, gs))
        if dtype == torch.bfloat16:
            size = lib.gi_w4a16_gated_mlp_workspace_bytes(most, k, n, gs)
            S2 = S.flip(0).contiguous()
            assert lib.gi_w4a16_gated_mlp(p(x), code, p(B), p(S), S.shape[0], p(B), p(S2), S.shape[0], p(y), m, k, n,
                                          gs, base, size, stream) == L.GI_OK, (m, lib.gi_last_error())
            assert torch.equal(y, ops.gated_mlp_act(x, (B, S), (B, S2), gs))


def test_gemm_rows_past_32_bit_offsets():
    """2^19 + 400 rows of K 65536 at group size 32: the rows' offset table is
    larger than 4 GiB (one offset per row and 32 k).  Rows from both ends and
    around the 64-row blocks, the others zero."""
    m, k, n, gs = 2 ** 19 + 400, 65536, 4, 32
    if torch.cuda.mem_get_info()[0] < 180 * 2 ** 30:
        pytest.skip("needs 180 GiB of free device memory")
    _, B, S = _operands(1, k, n, gs, torch.bfloat16, seed=5)
    rows = [0, 1, 63, 64, 2 ** 18 + 9, m - 81, m - 80, m - 6, m - 1]
    xr = synth.activations(len(rows), k, seed=6)
    lib = L.load()
    size = lib.gi_w4a16_workspace_bytes(m, k, n, gs)
    x = ws = None
    try:
        x = torch.zeros(m, k, dtype=torch.bfloat16, device=DEV)
        x[torch.tensor(rows, device=DEV)] = xr.to(DEV)
        ws, y = torch.zeros(size, dtype=torch.uint8, device=DEV), torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
        assert lib.gi_w4a16_linear(x.data_ptr(), L.DTYPE_BF16, B.data_ptr(), S.data_ptr(), S.shape[0], y.data_ptr(), m,
                                   k, n, gs, 0.0, ws.data_ptr(), size,
                                   torch.cuda.current_stream().cuda_stream) == L.GI_OK
        y = y.cpu()
    finally:
        del x, ws
        torch.cuda.empty_cache()
    _check(y[rows], O.w4a16_linear(_f64(xr), B.cpu().numpy(), _f64(S), gs), torch.bfloat16)
    y[rows] = 0
    assert not y.any()
