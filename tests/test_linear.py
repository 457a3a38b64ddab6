"""Non-expert compact3 linears (compact3_linear_forward / _dual_ / _qkv_, TriSMoE_cuda.cpp:497-700,
kernel.cu:2146-3744 and 10781-11740): the oracle's composition on the CPU, and on the GPU the single, dual
and Q/K/V bindings against the oracle, with input and output scales, bias, the matrix-mode null-space
term, and ragged batches."""
import numpy as np
import pytest
import torch

from tris_moe_amd import synthetic
from tris_moe_amd.packing import pack_4bit

MODULE_KEYS = ("qweight1", "qweight2_sparse", "qweight2_sparse_prefix", "q_gmap_gr_words", "q_gmap_gr_offsets",
               "q_gmap_gr_meta", "c_map", "g_idx", "col_pack3", "row_pack3")


def _modules(ext, count, n, k, seed):
    """count one-matrix modules (a synthetic projection's experts, each without its expert dimension)."""
    rng = np.random.default_rng(seed)
    col_norm = rng.random(k).astype(np.float32) + 0.5
    proj = synthetic.make_projection(rng, count, n, k, 0.15, col_norm, ext.gr_encode)
    return [{key: np.ascontiguousarray(proj[key][e]) for key in MODULE_KEYS} for e in range(count)], rng


def _ns(rng, n, k, ns_rank, gs):
    c2 = pack_4bit(rng.standard_normal((ns_rank, k)).astype(np.float32) * 0.05, gs)
    c1 = pack_4bit(rng.standard_normal((n, ns_rank)).astype(np.float32) * 0.05, min(ns_rank, gs))
    return c2, c1


def test_oracle_linear_is_the_composition(oracle_mod, tris):
    """oracle.compact3_linear against the same products taken by torch on the CPU: (x' W^T + C1 (C2 x)) *
    output_scale + bias in fp32, one rounding; without extras it is the grouped oracle over one segment.
    Two plausible slips (the null-space term after the output scale; the input scale applied to the term's
    input too) give other bits on this data, so the check sees them."""
    import torch.nn.functional as F

    mods, rng = _modules(tris["ext"], 1, 96, 128, 5)
    m = mods[0]
    x = (rng.standard_normal((6, 128)) * 2).astype(np.float16)
    s_in = (rng.random(128) + 0.5).astype(np.float16)
    s_out = (rng.random(96) * 2 + 0.25).astype(np.float16)
    bias = rng.standard_normal(96).astype(np.float16)
    c2p, c1p = _ns(rng, 96, 128, 16, 32)
    c2 = oracle_mod.packed4_dequant(c2p["qweight"], c2p["qzeros"], c2p["scales"], c2p["g_idx"], 16, 128)
    c1 = oracle_mod.packed4_dequant(c1p["qweight"], c1p["qzeros"], c1p["scales"], c1p["g_idx"], 96, 16)
    got = oracle_mod.compact3_linear(x, m, s_in, s_out, bias, c2, c1)
    w = torch.from_numpy(oracle_mod.dequant_grouped_expert(oracle_mod.module_as_payload(m), 0)).float()
    xt, xs = torch.from_numpy(x).float(), (torch.from_numpy(x) * torch.from_numpy(s_in)).float()
    ns = F.linear(F.linear(xt, torch.from_numpy(c2).float()), torch.from_numpy(c1).float())
    want = ((F.linear(xs, w) + ns) * torch.from_numpy(s_out).float() + torch.from_numpy(bias).float()).half().numpy()
    np.testing.assert_array_equal(got, want)
    slip1 = ((F.linear(xs, w) * torch.from_numpy(s_out).float() + ns) + torch.from_numpy(bias).float()).half().numpy()
    ns2 = F.linear(F.linear(xs, torch.from_numpy(c2).float()), torch.from_numpy(c1).float())
    slip2 = ((F.linear(xs, w) + ns2) * torch.from_numpy(s_out).float() + torch.from_numpy(bias).float()).half().numpy()
    assert not np.array_equal(slip1, want) and not np.array_equal(slip2, want)
    plain = oracle_mod.compact3_linear(x, m)
    grouped = oracle_mod.grouped_forward(oracle_mod.module_as_payload(m), x, np.asarray([0]), np.asarray([0, 6]))
    np.testing.assert_array_equal(plain, grouped)


# ------------------------------------------------------------------------------------------------ GPU
def _dev(mod, cuda):
    return {k: torch.from_numpy(v).to(cuda) for k, v in mod.items()}


def _linear(ext, x, m, s_in=None, s_out=None, bias=None, ns=None):
    empty = x.new_empty((0,))
    ns_args = ([ns[1]["qweight"], ns[1]["qzeros"], ns[1]["scales"], ns[1]["g_idx"], ns[0]["qweight"],
                ns[0]["qzeros"], ns[0]["scales"], ns[0]["g_idx"], True] if ns is not None else [empty] * 8 + [False])
    return ext.compact3_linear_forward(
        x, m["qweight1"], m["qweight2_sparse"], m["qweight2_sparse_prefix"], empty, empty, m["q_gmap_gr_words"],
        m["q_gmap_gr_offsets"], m["q_gmap_gr_meta"], m["c_map"], m["g_idx"], m["col_pack3"], m["row_pack3"],
        s_in if s_in is not None else empty, s_out if s_out is not None else empty,
        bias if bias is not None else empty, s_in is not None, s_out is not None, bias is not None, *ns_args, 1, False)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 7, 70])
@pytest.mark.parametrize("extras", ["plain", "scales_bias", "ns"])
def test_linear_matches_oracle(tris, oracle_mod, cuda, batch, extras):
    """compact3_linear_forward: one row, a ragged tile and several tiles; no extras, input / output scales
    with bias, and all of them with a null-space term (act-order-free groups of 32 and 16)."""
    from test_gpu_parity import assert_close, note

    note(f"compact3 linear batch={batch} extras={extras}")
    ext = tris["ext"]
    n, k = 200, 192
    mods, rng = _modules(ext, 1, n, k, 40 + batch)
    m = mods[0]
    x = (rng.standard_normal((batch, k)) * 1.5).astype(np.float16)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    s_in = s_out = bias = ns = None
    c2 = c1 = None
    if extras != "plain":
        s_in = (rng.random(k) + 0.5).astype(np.float16)
        s_out = (rng.random(n) * 2 + 0.25).astype(np.float16)
        bias = rng.standard_normal(n).astype(np.float16)
    if extras == "ns":
        c2p, c1p = _ns(rng, n, k, 24, 32)
        c2 = oracle_mod.packed4_dequant(c2p["qweight"], c2p["qzeros"], c2p["scales"], c2p["g_idx"], 24, k)
        c1 = oracle_mod.packed4_dequant(c1p["qweight"], c1p["qzeros"], c1p["scales"], c1p["g_idx"], n, 24)
        ns = ({kk: t(v) for kk, v in c2p.items()}, {kk: t(v) for kk, v in c1p.items()})
    got = _linear(ext, t(x), _dev(m, cuda), *(t(a) if a is not None else None for a in (s_in, s_out, bias)), ns=ns)
    want = oracle_mod.compact3_linear(x, m, s_in, s_out, bias, c2, c1)
    assert_close(got.cpu().numpy(), want, f"compact3_linear_forward {extras}")


@pytest.mark.gpu
def test_dual_and_qkv_match_single_calls(tris, oracle_mod, cuda):
    """compact3_dual_linear_forward and compact3_qkv_linear_forward (with biases): the bits of single calls,
    within tolerance of the oracle; a sparse-format payload is refused with a message."""
    from test_gpu_parity import assert_close, note

    note("compact3 dual / qkv")
    ext = tris["ext"]
    n, k, batch = 128, 256, 9
    mods, rng = _modules(ext, 3, n, k, 77)
    dm = [_dev(m, cuda) for m in mods]
    x = torch.from_numpy((rng.standard_normal((batch, k)) * 1.5).astype(np.float16)).to(cuda)
    args = lambda m: [m[key] for key in MODULE_KEYS]
    dual = ext.compact3_dual_linear_forward(x, *args(dm[0]), *args(dm[1]), 1, False)
    for i in range(2):
        assert torch.equal(dual[i], _linear(ext, x, dm[i]))
        assert_close(dual[i].cpu().numpy(), oracle_mod.compact3_linear(x.cpu().numpy(), mods[i]), f"dual[{i}]")
    biases = [torch.from_numpy(rng.standard_normal(n).astype(np.float16)).to(cuda) for _ in range(3)]
    qkv = ext.compact3_qkv_linear_forward(x, *args(dm[0]), biases[0], *args(dm[1]), biases[1], *args(dm[2]), biases[2],
                                          1, False)
    for i in range(3):
        assert torch.equal(qkv[i], _linear(ext, x, dm[i], bias=biases[i]))
        want = oracle_mod.compact3_linear(x.cpu().numpy(), mods[i], bias=biases[i].cpu().numpy())
        assert_close(qkv[i].cpu().numpy(), want, f"qkv[{i}]")
    sparse = dict(dm[0], q_gmap_gr_offsets=dm[0]["q_gmap_gr_offsets"][:-1])
    with pytest.raises(RuntimeError, match="block-GR"):
        _linear(ext, x, sparse)


@pytest.mark.gpu
def test_module_and_fused_runners(tris, oracle_mod, cuda):
    """qlinear.Compact3Linear (mode-4 QuantLinear) with every extra, and the Q/K/V and shared-expert gate/up
    runners: the bits of the modules run one by one; a module with scales is left to the caller (None)."""
    from test_gpu_parity import assert_close, note

    note("Compact3Linear module and fused runners")
    ext, ql = tris["ext"], tris["qlinear"]
    n, k = 160, 128
    mods, rng = _modules(ext, 3, n, k, 91)
    c2p, c1p = _ns(rng, n, k, 16, 32)
    full = ql.Compact3Linear(k, n).load_tensors(dict(mods[0], input_scale=(rng.random(k) + 0.5).astype(np.float16),
                                                     output_scale=(rng.random(n) + 0.5).astype(np.float16),
                                                     bias=rng.standard_normal(n).astype(np.float16),
                                                     ns_c1=c1p, ns_c2=c2p)).to(cuda)
    x = torch.from_numpy((rng.standard_normal((2, 3, k)) * 1.5).astype(np.float16)).to(cuda)
    y = full(x)
    assert y.shape == (2, 3, n)
    c2 = oracle_mod.packed4_dequant(c2p["qweight"], c2p["qzeros"], c2p["scales"], c2p["g_idx"], 16, k)
    c1 = oracle_mod.packed4_dequant(c1p["qweight"], c1p["qzeros"], c1p["scales"], c1p["g_idx"], n, 16)
    want = oracle_mod.compact3_linear(x.reshape(-1, k).cpu().numpy(), mods[0], full.input_scale.cpu().numpy(),
                                      full.output_scale.cpu().numpy(), full.bias.cpu().numpy(), c2, c1)
    assert_close(y.reshape(-1, n).cpu().numpy(), want, "Compact3Linear")
    plain = [ql.Compact3Linear(k, n).load_tensors(dict(m, bias=rng.standard_normal(n).astype(np.float16))).to(cuda)
             for m in mods]
    q, kk, v = ql.run_compact3_qkv_block_gr_forward(*plain, x)
    for got, m in zip((q, kk, v), plain):
        assert torch.equal(got, m(x))
    nobias = [ql.Compact3Linear(k, n).load_tensors(m).to(cuda) for m in mods[:2]]
    g, u = ql.run_compact3_shared_expert_gate_up_forward(*nobias, x)
    assert torch.equal(g, nobias[0](x)) and torch.equal(u, nobias[1](x))
    assert ql.run_compact3_qkv_block_gr_forward(full, plain[1], plain[2], x) is None


@pytest.mark.gpu
@pytest.mark.parametrize("n,k,batch,groups", [
    (64, 64, 1, "uniform"),         # the smallest matrix
    (130, 1152, 16, "uniform"),     # columns no multiple of 4; a last chunk of two K tiles
    (192, 1024, 17, "uniform"),     # 32-row tiles, one row past the 16-row ones
    (64, 2048, 70, "uniform"),      # more than eight groups; three row tiles, the last ragged
    (136, 640, 33, "split"),        # groups changing inside a K tile of the second chunk only
    (68, 192, 5, "shuffled"),       # a group per column
    (96, 96, 3, "uniform"),         # rank no multiple of 64: the exact kernel
])
def test_linear_matrix_core_shapes(tris, oracle_mod, cuda, n, k, batch, groups):
    """The linears' GEMM at the edges of its tiles, chunks and slices and with g_idx it has to walk column by column,
    with an input scale, output scale and bias, against the oracle."""
    from test_gpu_parity import assert_close, note

    note(f"compact3 linear n={n} k={k} batch={batch} groups={groups}")
    ext = tris["ext"]
    rng = np.random.default_rng(n + k)
    gidx = np.arange(k) // 128
    if groups == "shuffled":
        gidx = rng.permutation(gidx)
    elif groups == "split":
        gidx[600:610] = 0
    proj = synthetic.make_projection(rng, 1, n, k, 0.15, rng.random(k).astype(np.float32) + 0.5, ext.gr_encode,
                                     g_idx=gidx.astype(np.int32))
    m = {key: np.ascontiguousarray(proj[key][0]) for key in MODULE_KEYS}
    x = (rng.standard_normal((batch, k)) * 1.5).astype(np.float16)
    s_in, s_out = (rng.random(k) + 0.5).astype(np.float16), (rng.random(n) * 2 + 0.25).astype(np.float16)
    bias = rng.standard_normal(n).astype(np.float16)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    got = _linear(ext, t(x), _dev(m, cuda), t(s_in), t(s_out), t(bias))
    assert_close(got.cpu().numpy(), oracle_mod.compact3_linear(x, m, s_in, s_out, bias), f"linear n={n} k={k}")


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 16, 33])
def test_linear_infinite_activations(tris, oracle_mod, cuda, batch):
    """An infinity in a salient column, in a plain one and in none, a row each, and a NaN: the outputs are infinite with
    the oracle's signs, NaN or finite exactly where the oracle's are."""
    from test_gpu_parity import assert_close, note

    n, k = 80, 640
    note(f"compact3 linear with infinities, batch={batch}")
    ext = tris["ext"]
    mods, rng = _modules(ext, 1, n, k, 12)
    m = mods[0]
    salient = (m["c_map"].view(np.uint32)[np.arange(k) // 32] >> (np.arange(k) % 32)) & 1
    x = rng.standard_normal((batch, k)).astype(np.float16)
    x[0, np.flatnonzero(salient)[-1]] = np.inf
    if batch > 3:
        x[1, np.flatnonzero(salient == 0)[0]] = -np.inf
        x[2, 5] = np.nan
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    got = _linear(ext, t(x), _dev(m, cuda)).cpu().numpy()
    want = oracle_mod.compact3_linear(x, m)
    assert np.isinf(want[0]).all()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(want), want, 0))
    rows = np.isfinite(want).all(1)
    if rows.any():
        assert_close(got[rows], want[rows], f"finite rows, batch={batch}")


def test_linears_stay_on_the_current_device(tris, monkeypatch):
    """The matrix-core linears are refused on any device but the current one (the exact kernel takes those), and only
    there."""
    from types import SimpleNamespace

    st = SimpleNamespace(outfeatures=64, qweight2_sparse_rows=1, num_groups=2)
    x = SimpleNamespace(size=lambda d: (4, 256)[d], data_ptr=lambda: 4096, device=torch.device("cuda", 1))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 1, raising=False)
    assert tris["ext"]._linears_ok(x, (st,))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    assert not tris["ext"]._linears_ok(x, (st,))


@pytest.mark.gpu
def test_linear_without_split_columns(tris, oracle_mod, cuda):
    """A matrix with no split column at all codes to no GR words (an empty tensor): single and Q/K/V calls take it, as
    the exact kernel does."""
    from test_gpu_parity import assert_close, note

    note("compact3 linear with an empty GR stream")
    ext = tris["ext"]
    n, k, batch = 72, 128, 5
    rng = np.random.default_rng(31)
    proj = synthetic.make_projection(rng, 3, n, k, 0.0, rng.random(k).astype(np.float32) + 0.5, ext.gr_encode)
    mods = [{key: np.ascontiguousarray(proj[key][e]) for key in MODULE_KEYS} for e in range(3)]
    assert all(m["q_gmap_gr_words"].size == 0 for m in mods)
    dm = [_dev(m, cuda) for m in mods]
    x = (rng.standard_normal((batch, k)) * 1.5).astype(np.float16)
    xd = torch.from_numpy(x).to(cuda)
    zero = torch.zeros(n, dtype=torch.float16, device=cuda)
    qkv = ext.compact3_qkv_linear_forward(xd, *(a for m in dm for a in [*(m[key] for key in MODULE_KEYS), zero]))
    for i in range(3):
        want = oracle_mod.compact3_linear(x, mods[i])
        assert_close(_linear(ext, xd, dm[i]).cpu().numpy(), want, f"empty stream {i}")
        assert_close(qkv[i].cpu().numpy(), want, f"empty stream qkv {i}")


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 20])
def test_linear_unused_scales_not_finite(tris, oracle_mod, cuda, batch):
    """Row scales that no column picks may hold anything (a mean over no column): R_nd where every plain column is
    split, R0 and R1 of a group without salient columns, the first among them.  The outputs stay the oracle's."""
    from test_gpu_parity import assert_close, note

    note(f"compact3 linear with unused scales not finite, batch={batch}")
    ext = tris["ext"]
    n, k, group = 72, 640, 128
    rng = np.random.default_rng(33)
    norm = np.where(np.arange(k) // group == 2, 9.0, 1.0)  # every salient column in group 2
    proj = synthetic.make_projection(rng, 1, n, k, 1.0, norm, ext.gr_encode, salient_counts=[9])
    m = {key: np.ascontiguousarray(proj[key][0]) for key in MODULE_KEYS}
    rp = m["row_pack3"].view(np.uint16).reshape(n, k // group, 4)  # R0, R1, R_d, R_nd
    rp[:, :, 3] = 0x7C00                     # inf
    rp[:, [0, 1, 3, 4], 0] = 0x7E00          # NaN
    rp[:, [0, 1, 3, 4], 1] = 0xFC00          # -inf
    x = (rng.standard_normal((batch, k)) * 1.5).astype(np.float16)
    want = oracle_mod.compact3_linear(x, m)
    assert np.isfinite(want).all()
    got = _linear(ext, torch.from_numpy(x).to(cuda), _dev(m, cuda)).cpu().numpy()
    assert_close(got, want, f"unused scales, batch={batch}")


def test_linears_workspace_is_bounded(tris):
    """The linears' workspace holds the bitmaps, and partial sums only while the K slices fill the GPU: at most 12 MiB a
    matrix above the bitmaps, none once the tiles do."""
    import ctypes

    from tris_moe_amd import _lib

    size = _lib.load().tris_compact3_linears_workspace_bytes
    for rank, n in ((2048, 2048), (4096, 4096), (14336, 1024), (640, 200)):
        bitmaps = rank // 64 * -(-n // 64) * 512
        for count in (1, 3):
            widths = (ctypes.c_int32 * count)(*[n] * count)
            for batch in (1, 16, 17, 64, 300, 1024, 4096, 100000, 1 << 20):
                sums = size(batch, rank, widths, count) - count * bitmaps
                assert 0 <= sums <= count * (12 << 20)
                assert batch < 32768 or sums == 0


@pytest.mark.gpu
@pytest.mark.parametrize("groups", ["uniform", "split", "infinite"])
def test_linear_prompt_sizes(tris, oracle_mod, cuda, groups):
    """Enough rows and columns that a workgroup takes both chunks of a matrix itself (no slices): the staging between
    chunks, one chunk of two with split K tiles or with an infinity, scales and bias; the last row tile is ragged."""
    from test_gpu_parity import assert_close, note

    n, k, batch = 1540, 1024, 1010
    note(f"compact3 linear prompt sizes groups={groups}")
    ext = tris["ext"]
    rng = np.random.default_rng(63)
    gidx = np.arange(k) // 128
    if groups == "split":
        gidx[700:710] = 0  # the second chunk
    proj = synthetic.make_projection(rng, 1, n, k, 0.15, rng.random(k).astype(np.float32) + 0.5, ext.gr_encode,
                                     g_idx=gidx.astype(np.int32))
    m = {key: np.ascontiguousarray(proj[key][0]) for key in MODULE_KEYS}
    x = rng.standard_normal((batch, k)).astype(np.float16)
    if groups == "infinite":
        x[5, 17] = np.inf  # the first chunk
    s_out, bias = (rng.random(n) * 2 + 0.25).astype(np.float16), rng.standard_normal(n).astype(np.float16)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    got = _linear(ext, t(x), _dev(m, cuda), None, t(s_out), t(bias)).cpu().numpy()
    want = oracle_mod.compact3_linear(x, m, None, s_out, bias)
    if groups == "infinite":
        np.testing.assert_array_equal(got[5], want[5])
        got, want = np.delete(got, 5, 0), np.delete(want, 5, 0)
    assert_close(got, want, f"prompt sizes {groups}")


def test_linears_refuse_a_misaligned_input_scale(tris):
    """The linears' C entry reads input_scale 16 bytes at a time: it refuses one off a 16-byte boundary (before it
    touches any tensor, so the addresses here need not be real)."""
    import ctypes

    from tris_moe_amd import _lib

    lib = _lib.load()
    at = 1 << 20
    pay = _lib.TrisPayload(1, 64, 64, 1, 1, 4, *[at] * 10, None, None, 0, 0, 1)
    outs = (ctypes.c_void_p * 1)(at)
    call = lambda scale: (lib.tris_compact3_linears_forward(at, 4, (_lib.TrisPayload * 1)(pay), 1, scale, None, outs, at,
                                                            0, None), lib.tris_last_error().decode())
    rc, msg = call(at + 2)
    assert rc < 0 and "aligned" in msg
    rc, msg = call(at)  # (the workspace is too small)
    assert rc < 0 and "workspace too small" in msg


@pytest.mark.gpu
def test_linear_longer_than_one_launch(tris, oracle_mod, cuda):
    """A batch past the row tiles of one launch (65535 of 32 rows) goes in two: rows at the start, on both sides of the
    seam and at the ragged end are the oracle's."""
    from test_gpu_parity import assert_close, note

    n, k, seam = 64, 64, 65535 * 32
    batch = seam + 33
    note("compact3 linear in two launches")
    ext = tris["ext"]
    m = _modules(ext, 1, n, k, 71)[0][0]
    x = torch.randn((batch, k), generator=torch.Generator(device=cuda).manual_seed(5), device=cuda).to(torch.float16)
    rows = [0, 1, 31, 32, seam - 33, seam - 1, seam, seam + 1, seam + 31, seam + 32]
    got = _linear(ext, x, _dev(m, cuda))
    assert got.shape == (batch, n)
    assert_close(got[rows].cpu().numpy(), oracle_mod.compact3_linear(x[rows].cpu().numpy(), m), "two launches")


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [3, 70])
def test_exact_kernel_entries(tris, oracle_mod, cuda, batch):
    """A rank that is no multiple of 64 takes the exact kernel in every entry: the single linear with scales, bias and the
    null-space term, the dual linear, and Q / K / V (a pair and a single launch), with an uneven g_idx on one of them."""
    from test_gpu_parity import assert_close, note

    n, k = 136, 160
    note(f"exact linears batch={batch}")
    ext = tris["ext"]
    mods, rng = _modules(ext, 3, n, k, 55)
    mods[1]["g_idx"] = (np.arange(k) % 2).astype(np.int32)
    dm = [_dev(m, cuda) for m in mods]
    x = (rng.standard_normal((batch, k)) * 1.5).astype(np.float16)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    assert not ext._linears_ok(t(x), ())
    args = lambda m: [m[key] for key in MODULE_KEYS]
    dual = ext.compact3_dual_linear_forward(t(x), *args(dm[0]), *args(dm[1]))
    biases = [rng.standard_normal(n).astype(np.float16) for _ in range(3)]
    qkv = ext.compact3_qkv_linear_forward(t(x), *(a for m, b in zip(dm, biases) for a in [*args(m), t(b)]))
    for i in range(3):
        if i < 2:
            assert_close(dual[i].cpu().numpy(), oracle_mod.compact3_linear(x, mods[i]), f"exact dual[{i}]")
        assert_close(qkv[i].cpu().numpy(), oracle_mod.compact3_linear(x, mods[i], bias=biases[i]), f"exact qkv[{i}]")
    s_in, s_out = (rng.random(k) + 0.5).astype(np.float16), (rng.random(n) * 2 + 0.25).astype(np.float16)
    c2p, c1p = _ns(rng, n, k, 24, 32)
    c2 = oracle_mod.packed4_dequant(c2p["qweight"], c2p["qzeros"], c2p["scales"], c2p["g_idx"], 24, k)
    c1 = oracle_mod.packed4_dequant(c1p["qweight"], c1p["qzeros"], c1p["scales"], c1p["g_idx"], n, 24)
    got = _linear(ext, t(x), dm[0], t(s_in), t(s_out), t(biases[0]),
                  ns=({kk: t(v) for kk, v in c2p.items()}, {kk: t(v) for kk, v in c1p.items()}))
    want = oracle_mod.compact3_linear(x, mods[0], s_in, s_out, biases[0], c2, c1)
    assert_close(got.cpu().numpy(), want, "exact single with every extra")
