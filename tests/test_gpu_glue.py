"""The steps between the operators (mask bias, axis swap, residual update, transposed pair-bias producer) and the
triangle-attention block assembled from them, on a real MI355X through the C ABI.

The copies and the residual update are checked bit for bit against torch's own indexing and bf16 addition; the
block is checked against the CPU oracle's LayerNorm, Linear and gated attention composed in numpy (fp32, no
intermediate rounding) at the tolerance of the bf16 path, and, at a full-size pair tensor, through the identity
ending_node(z, mask) == starting_node(z^T, mask^T)^T, which must hold bit for bit.
"""
import ctypes
import math

import numpy as np
import pytest

from kutacc_amd import capi
from kutacc_amd.workloads import round_to_bf16

import helpers

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "these tests need the GPU"
    capi.set_stream(None)
    capi.set_blocking(True)
    return torch


def code(torch, t):
    return capi.K_BF16 if t.dtype == torch.bfloat16 else capi.K_FP32


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("transposed", [0, 1])
def test_mask_bias(torch_cuda, dtype, transposed):
    torch = torch_cuda
    dt = getattr(torch, dtype)
    n0, n1 = 37, 52
    g = torch.Generator(device="cuda").manual_seed(3)
    mask_ij = (torch.rand(n0, n1, device="cuda", generator=g) > 0.3).to(dt)
    stored = mask_ij.t().contiguous() if transposed else mask_ij
    bias = torch.full((n0, n1), 7.0, dtype=dt, device="cuda")
    rc = capi.lib().kutacc_hip_mask_bias(stored.data_ptr(), bias.data_ptr(), n0, n1, transposed, code(torch, bias), None)
    torch.cuda.synchronize()
    assert rc == 0
    want = (mask_ij.float() * 1e9 - 1e9).to(dt)
    assert helpers.same_bits(bias, want)
    assert float(bias.max()) == 0.0 and float(bias.min()) < -9e8


@pytest.mark.parametrize("shape,dtype", [((40, 24, 128), "bfloat16"), ((9, 31, 5), "bfloat16"), ((17, 6, 12), "float32"),
                                         ((384, 384, 128), "bfloat16")])
def test_swap_leading_axes_and_residual_add(torch_cuda, shape, dtype):
    torch = torch_cuda
    dt = getattr(torch, dtype)
    n0, n1, c = shape
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(n0, n1, c, device="cuda", generator=g).to(dt)
    out = torch.zeros(n1, n0, c, dtype=dt, device="cuda")
    L = capi.lib()
    assert L.kutacc_hip_swap_leading_axes(x.data_ptr(), out.data_ptr(), n0, n1, c, code(torch, x), None) == 0
    torch.cuda.synchronize()
    assert helpers.same_bits(out, x.transpose(0, 1).contiguous())
    # acc[i, j] += delta[i, j] and acc[i, j] += delta[j, i]
    acc = torch.randn(n0, n1, c, device="cuda", generator=g).to(dt)
    want_plain = (acc.float() + x.float()).to(dt)
    want_swapped = (acc.float() + out.transpose(0, 1).float()).to(dt)
    a1, a2 = acc.clone(), acc.clone()
    assert L.kutacc_hip_residual_add(a1.data_ptr(), x.data_ptr(), n0, n1, c, 0, code(torch, x), None) == 0
    assert L.kutacc_hip_residual_add(a2.data_ptr(), out.data_ptr(), n0, n1, c, 1, code(torch, x), None) == 0
    torch.cuda.synchronize()
    assert helpers.same_bits(a1, want_plain)
    assert helpers.same_bits(a2, want_swapped)
    assert L.kutacc_hip_swap_leading_axes(x.data_ptr(), x.data_ptr(), n0, n1, c, code(torch, x), None) == capi.EINVAL


@pytest.mark.parametrize("n_i,n_j,c_z,heads,dtype", [(48, 48, 128, 4, "bfloat16"), (40, 56, 128, 8, "bfloat16"),
                                                      (9, 14, 64, 3, "bfloat16"), (7, 5, 32, 2, "float32")])
def test_pair_bias_transposed_equals_pair_bias_of_the_swapped_tensor(torch_cuda, n_i, n_j, c_z, heads, dtype):
    torch = torch_cuda
    dt = getattr(torch, dtype)
    g = torch.Generator(device="cuda").manual_seed(9)
    z_t = torch.randn(n_j, n_i, c_z, device="cuda", generator=g).to(dt)  # stored transposed: [j, i, c]
    z = z_t.transpose(0, 1).contiguous()
    w = (torch.randn(heads, c_z, device="cuda", generator=g) / math.sqrt(c_z)).to(dt)
    gamma = torch.rand(c_z, device="cuda", generator=g) + 0.5
    beta = torch.randn(c_z, device="cuda", generator=g) * 0.1
    L = capi.lib()
    res = []
    for fn, src in ((L.kutacc_hip_pair_bias, z), (L.kutacc_hip_pair_bias_transposed, z_t)):
        nb = torch.zeros(heads, n_i, n_j, dtype=dt, device="cuda")
        zn = torch.zeros(n_i, n_j, c_z, dtype=dt, device="cuda")
        assert fn(src.data_ptr(), gamma.data_ptr(), beta.data_ptr(), w.data_ptr(), nb.data_ptr(), zn.data_ptr(), n_i, n_j, c_z,
                  heads, 1e-5, code(torch, z), None) == 0
        torch.cuda.synchronize()
        res.append((nb, zn))
    assert helpers.same_bits(res[0][0], res[1][0]) and helpers.same_bits(res[0][1], res[1][1])


@pytest.mark.parametrize("n_i,n_j,heads", [(1, 1, 4), (5, 7, 8), (33, 31, 4), (64, 512, 8), (1024, 32, 4)])
@pytest.mark.parametrize("transposed", [False, True])
def test_pair_bias_of_few_rows_equals_that_of_many(torch_cuda, n_i, n_j, heads, transposed):
    """Few rows of z are shared by the waves of a workgroup (up to 1024 units of 32 on 256 CUs: the last two sizes are the most), many are not:
    the same bits for the rows that both have."""
    torch = torch_cuda
    more = n_i + 33000 // n_j + 1
    g = torch.Generator(device="cuda").manual_seed(17)
    z = torch.randn(more, n_j, 128, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(heads, 128, device="cuda", generator=g) / math.sqrt(128)).to(torch.bfloat16)
    gamma = torch.rand(128, device="cuda", generator=g) + 0.5
    beta = torch.randn(128, device="cuda", generator=g) * 0.1
    L = capi.lib()
    res = []
    for rows in (n_i, more):
        src = z[:rows].transpose(0, 1).contiguous() if transposed else z[:rows].contiguous()
        nb = torch.full((heads, rows, n_j), 7.0, dtype=torch.bfloat16, device="cuda")
        zn = torch.full((rows, n_j, 128), 7.0, dtype=torch.bfloat16, device="cuda")
        fn = L.kutacc_hip_pair_bias_transposed if transposed else L.kutacc_hip_pair_bias
        assert fn(src.data_ptr(), gamma.data_ptr(), beta.data_ptr(), w.data_ptr(), nb.data_ptr(), zn.data_ptr(), rows, n_j, 128, heads, 1e-5,
                  capi.K_BF16, None) == 0
        torch.cuda.synchronize()
        res.append((nb, zn))
    assert helpers.same_bits(res[0][0], res[1][0][:, :n_i].contiguous()) and helpers.same_bits(res[0][1], res[1][1][:n_i])


# ---- the block ---------------------------------------------------------------------------------------------------
@pytest.fixture(params=["fused", "separate"])
def layernorm_placement(request):
    """Both placements of the blocks' LayerNorm: inside the attention kernel's row staging (where that kernel can) and as a
    pass of its own.  The setting must hold while the block object is built (it sizes its workspace) and run."""
    assert capi.set_tuning("layernorm", request.param) == 0
    yield request.param
    capi.set_tuning("layernorm", "auto")


def block_case(seed, n, heads):
    rng = np.random.Generator(np.random.PCG64(seed))
    c = heads * 32
    w = lambda o, i: round_to_bf16((rng.standard_normal((o, i)) / math.sqrt(i)).astype(np.float32))  # noqa: E731
    mask = (rng.random((n, n)) > 0.1).astype(np.float32)
    mask[:, -3:] = 0.0  # padded residues: masked as keys for the starting node, whole rows for the ending node
    return dict(z=round_to_bf16(rng.standard_normal((n, n, c)).astype(np.float32)), mask=mask,
                gamma=(rng.random(c) + 0.5).astype(np.float32), beta=(rng.standard_normal(c) * 0.1).astype(np.float32),
                bias_w=w(heads, c), wq=w(c, c), wk=w(c, c), wv=w(c, c), wg=w(c, c), wo=w(c, c),
                bg=np.ones(c, np.float32), bo=(rng.standard_normal(c) * 0.1).astype(np.float32), heads=heads)


def block_oracle(c, ending):
    """AlphaFold's TriangleAttention in numpy on the oracle's operators: orientation swap, LayerNorm, pair bias from
    the normalised tensor, mask bias, gated attention, swap back, residual."""
    from oracle import oracle
    z, mask = c["z"], c["mask"]
    if ending:
        z, mask = z.transpose(1, 0, 2), mask.T
    n, _, ch = z.shape
    zn = oracle.layernorm_rows_f32(np.ascontiguousarray(z).reshape(-1, ch), c["gamma"], c["beta"], 1e-5).reshape(n, n, ch)
    nb = oracle.linear_f32(zn.reshape(-1, ch), c["bias_w"]).reshape(n, n, c["heads"]).transpose(2, 0, 1)
    bias = (mask * np.float32(1e9) - np.float32(1e9)).astype(np.float32)
    out = oracle.gating_attention_f32(zn, c["wq"], c["wk"], c["wv"], c["wg"], c["bg"], c["wo"], c["bo"], bias,
                                      np.ascontiguousarray(nb), c["heads"])
    if ending:
        out = out.transpose(1, 0, 2)
    return c["z"] + out


def run_block(torch, c, ending, z=None, mask=None):
    dev = lambda a, dt=torch.bfloat16: torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=dt)  # noqa: E731
    pair = dev(c["z"]) if z is None else z.clone()
    dmask = dev(c["mask"]) if mask is None else mask
    f32 = torch.float32
    blk = capi.TriangleAttentionBlock(pair, dmask, dev(c["gamma"], f32), dev(c["beta"], f32), dev(c["bias_w"]), dev(c["wq"]),
                                      dev(c["wk"]), dev(c["wv"]), dev(c["wg"]), dev(c["bg"], f32), dev(c["wo"]),
                                      dev(c["bo"], f32), c["heads"], ending)
    rc = blk.run()
    torch.cuda.synchronize()
    assert rc == 0, rc
    return pair


@pytest.mark.parametrize("ending", [False, True], ids=["starting node", "ending node"])
# 64, 96 and 160: whole key tiles, where the producer of the pair bias also writes the copy the attention kernels read
# (96 and 160: an odd tile count, padded with a zero tile)
@pytest.mark.parametrize("n,heads", [(48, 4), (70, 4), (40, 8), (64, 4), (96, 4), (160, 4), (64, 8), (32, 4), (128, 8)])
def test_triangle_attention_block_against_the_oracle(torch_cuda, layernorm_placement, n, heads, ending):
    c = block_case(600 + n, n, heads)
    got = run_block(torch_cuda, c, ending)
    helpers.check_close(helpers.to_numpy(got), block_oracle(c, ending), "bf16", f"block n={n} ending={ending}")


profiled_kernels = helpers.profiled_kernels


@pytest.mark.parametrize("ending", [False, True], ids=["starting node", "ending node"])
@pytest.mark.parametrize("n", [32, 64, 96, 160, 352])
def test_triangle_attention_block_on_the_two_row_kernel(torch_cuda, n, ending):
    """Whole key tiles and the two-row kernel forced wherever it can run: the producer of the pair bias writes the fp32
    tiles that kernel reads (no pre-pass of the operator), one to eleven key tiles, odd counts padded with a zero tile,
    one or several rows per workgroup."""
    c = block_case(900 + n, n, 4)
    assert capi.set_tuning("row_pairs", "1") == 0
    try:
        got = {}
        names = profiled_kernels(torch_cuda, lambda: got.setdefault("z", run_block(torch_cuda, c, ending)))
    finally:
        capi.set_tuning("row_pairs", None)
    assert "persistent_pair_kernel" in names and "pair_bias_tiles_kernel" not in names and "pair_bias_fragments_kernel" not in names, names
    helpers.check_close(helpers.to_numpy(got["z"]), block_oracle(c, ending), "bf16", f"block n={n} ending={ending}, two-row kernel")


@pytest.mark.parametrize("index,n", [(i, int(n)) for i, n in enumerate(np.random.Generator(np.random.PCG64(57)).integers(8, 200, size=8))])
def test_triangle_attention_block_seeded_sweep(torch_cuda, layernorm_placement, index, n):
    """Eight seeded pair sizes between 8 and 199 (ragged key tiles, odd tile counts), four heads, node alternating."""
    ending = bool(index & 1)
    c = block_case(3000 + index, n, 4)
    got = run_block(torch_cuda, c, ending)
    helpers.check_close(helpers.to_numpy(got), block_oracle(c, ending), "bf16", f"block sweep {index}: n={n} ending={ending}")


def test_triangle_attention_block_full_size_orientation_identity(torch_cuda, layernorm_placement):
    """384 residues: the ending-node block equals the starting-node block on the transposed pair tensor and mask,
    transposed back -- the two orientations differ only in which element is read or written where."""
    torch = torch_cuda
    c = block_case(700, 384, 4)
    z = torch.from_numpy(c["z"]).to(device="cuda", dtype=torch.bfloat16)
    mask = torch.from_numpy(c["mask"]).to(device="cuda", dtype=torch.bfloat16)
    end = run_block(torch, c, True, z, mask)
    start_t = run_block(torch, c, False, z.transpose(0, 1).contiguous(), mask.t().contiguous())
    assert helpers.same_bits(end, start_t.transpose(0, 1).contiguous())
    assert not helpers.same_bits(end, z)


def block_oracle_rows(c, ending, rows):
    """block_oracle for the batch rows `rows` of the attention only (rows i of the pair tensor for the starting node,
    columns for the ending node): rows of the attention are independent, so the oracle's LayerNorm and pair bias run on
    the whole tensor and its attention on the sample.  Returns the updated pair_act entries [len(rows), n, c] in the
    orientation of the attention (entry [a, k] is pair_act[rows[a], k] or, ending node, pair_act[k, rows[a]])."""
    from oracle import oracle
    z, mask = c["z"], c["mask"]
    if ending:
        z, mask = z.transpose(1, 0, 2), mask.T
    n, _, ch = z.shape
    zn = oracle.layernorm_rows_f32(np.ascontiguousarray(z).reshape(-1, ch), c["gamma"], c["beta"], 1e-5).reshape(n, n, ch)
    nb = np.ascontiguousarray(oracle.linear_f32(zn.reshape(-1, ch), c["bias_w"]).reshape(n, n, c["heads"]).transpose(2, 0, 1))
    bias = (np.ascontiguousarray(mask[rows]) * np.float32(1e9) - np.float32(1e9)).astype(np.float32)
    out = oracle.gating_attention_f32(np.ascontiguousarray(zn[rows]), c["wq"], c["wk"], c["wv"], c["wg"], c["bg"], c["wo"],
                                      c["bo"], bias, nb, c["heads"])
    return z[rows] + out


@pytest.mark.parametrize("n", [17, 32, 65, 96, 129, 160, 257, 288, 321, 385, 544])
def test_triangle_attention_block_of_odd_numbers_of_key_tiles(torch_cuda, n):
    """1, 3, 5, 9, 11, 13 and 17 tiles of 32 keys, whole and of one key: behind them the kernels have a tile of zeros that is not attended.  The
    oracle on a sample of rows, every other entry checked for finiteness."""
    torch = torch_cuda
    c = block_case(7300 + n, n, 4)
    rows = sorted({0, 1, n // 2, n - 2, n - 1})
    for ending in (False, True):
        got = run_block(torch, c, ending)
        assert bool(torch.isfinite(got).all())
        sample = got[:, rows].transpose(0, 1) if ending else got[rows]
        helpers.check_close(helpers.to_numpy(sample.contiguous()), block_oracle_rows(c, ending, rows), "bf16", f"block n={n} ending={ending}")


@pytest.mark.parametrize("n_seq,n_res", [(40, 32), (40, 33), (40, 96), (130, 65), (130, 160), (64, 161), (600, 224), (24, 257)])
def test_msa_row_attention_of_odd_numbers_of_key_tiles(torch_cuda, n_seq, n_res):
    torch = torch_cuda
    c = msa_case(7700 + n_seq + n_res, n_seq, n_res, 8, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]), "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    assert capi.MsaAttentionBlock(msa, dev(c["mask"]), w, 8, pair).run() == 0
    torch.cuda.synchronize()
    rows = sorted({0, 1, n_seq // 2, n_seq - 2, n_seq - 1})
    want = msa_oracle(dict(c, m=np.ascontiguousarray(c["m"][rows]), mask=np.ascontiguousarray(c["mask"][rows])), False)
    assert bool(torch.isfinite(msa).all())
    helpers.check_close(helpers.to_numpy(msa[rows].contiguous()), want, "bf16", f"msa rows {n_seq}x{n_res}")


@pytest.mark.parametrize("n", [384, 1024])
def test_triangle_attention_block_full_size_sampled_rows(torch_cuda, n):
    """The pair sizes the block is benchmarked at, both orientations: the oracle on a sample of attention rows (first,
    last, the padded residues, rows on either side of 32-row tile edges), every other entry checked for finiteness."""
    torch = torch_cuda
    c = block_case(7000 + n, n, 4)
    rows = sorted({0, 1, 31, 32, 33, n // 2 - 1, n // 2, n - 34, n - 33, n - 32, n - 4, n - 3, n - 2, n - 1})
    for ending in (False, True):
        res = {}
        names = profiled_kernels(torch, lambda: res.setdefault("z", run_block(torch, c, ending)))
        got = res["z"]
        # 384 residues: the two-row kernel on tiles the producer wrote; 1024: the long-sequence kernel on its fragments
        assert ("persistent_pair_kernel" if n == 384 else "fused_head_kernel") in names, names
        assert "pair_bias_tiles_kernel" not in names and "pair_bias_fragments_kernel" not in names, names
        assert bool(torch.isfinite(got).all())
        want = block_oracle_rows(c, ending, rows)
        sample = got[:, rows].transpose(0, 1) if ending else got[rows]
        helpers.check_close(helpers.to_numpy(sample.contiguous()), want, "bf16", f"block n={n} ending={ending}, sampled rows")


@pytest.mark.parametrize("n", [33, 95, 290, 361, 385, 449])
def test_producer_writes_the_attention_s_pair_bias_copy_at_ragged_lengths(torch_cuda, n):
    """Lengths that are no multiple of 32 (one row past a tile, one short of it, odd and even tile counts), on the single-row, the
    two-row and the long-row kernel: no pass of its own for the copy, and the last query block's and key tile's rows against the
    oracle, both orientations."""
    torch = torch_cuda
    c = block_case(7500 + n, n, 4)
    rows = sorted({0, 1, 31, 32, n // 2, n - 2, n - 1})
    for ending in (False, True):
        res = {}
        names = profiled_kernels(torch, lambda: res.setdefault("z", run_block(torch, c, ending)))
        got = res["z"]
        assert "pair_bias_tiles_kernel" not in names and "pair_bias_fragments_kernel" not in names, names
        assert bool(torch.isfinite(got).all())
        sample = got[:, rows].transpose(0, 1) if ending else got[rows]
        helpers.check_close(helpers.to_numpy(sample.contiguous()), block_oracle_rows(c, ending, rows), "bf16", f"block n={n} ending={ending}")


@pytest.mark.parametrize("n", [65, 96, 97, 128])
def test_short_rows_take_a_workgroup_per_unit(torch_cuda, n):
    """Three and four blocks of 32, whole and ragged, with two rows to a CU and head: the long-row kernel, every row against the oracle."""
    torch = torch_cuda
    c = block_case(7800 + n, n, 4)
    for ending in (False, True):
        res = {}
        names = profiled_kernels(torch, lambda: res.setdefault("z", run_block(torch, c, ending)))
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert "fused_head_kernel" in names, names
        helpers.check_close(helpers.to_numpy(res["z"]), block_oracle(c, ending), "bf16", f"block n={n} ending={ending}")


@pytest.mark.parametrize("n_seq,n_res", [(33, 64), (63, 33), (40, 127)])
def test_short_msa_rows_take_a_workgroup_per_unit(torch_cuda, n_seq, n_res):
    """256 channels, two to four blocks, two rows to a CU and head: the long-row kernel, the whole block against the oracle."""
    torch = torch_cuda
    c = msa_case(9600 + n_seq + n_res, n_seq, n_res, 8, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]), "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    blk = capi.MsaAttentionBlock(msa, dev(c["mask"]), w, 8, pair)
    res = {}
    names = profiled_kernels(torch, lambda: res.setdefault("rc", blk.run()))
    torch.cuda.synchronize()
    assert res["rc"] == 0
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert "fused_head_kernel" in names, names
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, False), "bf16", f"msa rows {n_seq}x{n_res}")


@pytest.mark.parametrize("n,pairs", [(129, False), (192, False), (193, True), (257, False)])
def test_odd_numbers_of_rows_per_workgroup_take_the_single_row_kernel(torch_cuda, n, pairs):
    """Three, three, four and five rows a workgroup (256 CUs), both orientations, first and last rows against the oracle."""
    torch = torch_cuda
    c = block_case(7700 + n, n, 4)
    rows = [0, 1, n - 2, n - 1]
    for ending in (False, True):
        res = {}
        names = profiled_kernels(torch, lambda: res.setdefault("z", run_block(torch, c, ending)))
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert ("persistent_pair_kernel" in names) == pairs, names
        got = res["z"]
        assert bool(torch.isfinite(got).all())
        sample = got[:, rows].transpose(0, 1) if ending else got[rows]
        helpers.check_close(helpers.to_numpy(sample.contiguous()), block_oracle_rows(c, ending, rows), "bf16", f"block n={n} ending={ending}")


def test_triangle_attention_block_beyond_1024_residues(torch_cuda):
    """1088 residues: past the fused head kernels' longest row, the block runs the same chain with the attention that keeps q, k, v
    and gate in memory.  Both orientations against the oracle on a sample of attention rows."""
    torch = torch_cuda
    n = 1088
    c = block_case(9100, n, 4)
    rows = sorted({0, 1, 31, 32, 127, 128, n // 2, n - 65, n - 64, n - 2, n - 1})
    assert capi.lib().kutacc_hip_triangle_attention_workspace(n, 4) > 4 * n * n * 128 * 2  # q, k, v and gate
    for ending in (False, True):
        res = {}
        names = profiled_kernels(torch, lambda: res.setdefault("z", run_block(torch, c, ending)))
        got = res["z"]
        assert "streamed_attention_kernel" in names and "output_projection_kernel<residual>" in names, names
        assert bool(torch.isfinite(got).all())
        want = block_oracle_rows(c, ending, rows)
        sample = got[:, rows].transpose(0, 1) if ending else got[rows]
        helpers.check_close(helpers.to_numpy(sample.contiguous()), want, "bf16", f"block n={n} ending={ending}, sampled rows")


def test_triangle_attention_block_past_the_pair_bias_producer_s_rows(torch_cuda):
    """2912 residues: more rows than the producer of the pair bias counts in 32 bits, so the copy that the attention reads has to
    come from a pass of its own.  Single queries against plain fp32 torch: a query of a row needs that row, its own row of the
    pair activation for the bias, and nothing else."""
    torch = torch_cuda
    n, heads, C = 2912, 4, 128
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, device="cuda", generator=g) * scale).to(torch.bfloat16)  # noqa: E731
    act = rnd(n, n, C)
    w = {k: rnd(C, C, scale=C ** -0.5) for k in ("q", "k", "v", "g", "o")}
    bias_w, ones, zeros = rnd(heads, C, scale=4 * C ** -0.5), torch.ones(C, device="cuda"), torch.zeros(C, device="cuda")
    picks = [(0, 5), (1234, 2900), (n - 1, 700)]
    norm = lambda t: torch.nn.functional.layer_norm(t.float(), (C,)).to(torch.bfloat16).float()  # noqa: E731
    want = []
    for b, q in picks:
        x = norm(act[b])
        proj = lambda m, rows: (rows @ w[m].float().T).view(-1, heads, 32).transpose(0, 1)  # noqa: E731
        nb = (norm(act[q]) @ bias_w.float().T).T
        p = torch.softmax((proj("q", x[q:q + 1]) @ proj("k", x).transpose(1, 2))[:, 0] * 32 ** -0.5 + nb, dim=1)
        avg = (p[:, None] @ proj("v", x))[:, 0].reshape(C) * torch.sigmoid(x[q] @ w["g"].float().T + 1.0)
        want.append(act[b, q].float() + avg @ w["o"].float().T)
    blk = capi.TriangleAttentionBlock(act, torch.ones(n, n, device="cuda", dtype=torch.bfloat16), ones, zeros, bias_w, w["q"], w["k"],
                                      w["v"], w["g"], ones, w["o"], zeros, heads, False)
    assert blk.run() == 0
    torch.cuda.synchronize()
    for (b, q), ref in zip(picks, want):
        helpers.check_close(helpers.to_numpy(act[b, q]), ref.cpu().numpy(), "bf16", f"row {b}, query {q}")


@pytest.mark.parametrize("n,heads", [(72, 3), (100, 5), (45, 1)])
def test_triangle_attention_block_with_other_channel_counts(torch_cuda, n, heads):
    """96, 160 and 32 channels (heads of 32): no fused head kernel takes them, the block's tiled route does; whole result
    against the oracle's composition, both orientations, lengths that are and are not multiples of 8."""
    for ending in (False, True):
        c = block_case(9200 + n, n, heads)
        got = run_block(torch_cuda, c, ending)
        helpers.check_close(helpers.to_numpy(got), block_oracle(c, ending), "bf16", f"block n={n} heads={heads} ending={ending}")


@pytest.fixture
def streamed_everywhere():
    assert capi.set_tuning("streamed", "1") == 0
    yield
    capi.set_tuning("streamed", None)


@pytest.mark.parametrize("n,heads", [(1, 4), (31, 4), (33, 8), (64, 4), (97, 8), (128, 4), (130, 4), (161, 8), (290, 4)])
def test_triangle_attention_block_on_the_streamed_kernels(torch_cuda, streamed_everywhere, n, heads):
    """The attention that keeps q, k, v and gate in memory, at lengths on either side of its key tiles (32), workgroups (four
    query blocks) and placement groups (eight of those), odd numbers of rows, whole and ragged tiles (the producer writes
    the tiles of the pair bias, or a pass of its own does); 128 and 256 channels, whole result against the oracle."""
    for ending in (False, True):
        c = block_case(9400 + n, n, heads)
        print(f"streamed block n={n} heads={heads} ending={ending}", flush=True)
        got = run_block(torch_cuda, c, ending)
        helpers.check_close(helpers.to_numpy(got), block_oracle(c, ending), "bf16", f"streamed block n={n} heads={heads} ending={ending}")


@pytest.mark.parametrize("n,heads", [(33, 4), (70, 8)])
def test_streamed_block_adds_its_result_in_a_pass_of_its_own_where_it_must(torch_cuda, streamed_everywhere, n, heads):
    """An output bias that does not start on 16 bytes keeps the projection from adding into the activation itself: the same
    bits by way of the workspace."""
    torch = torch_cuda
    for ending in (False, True):
        c = block_case(9450 + n, n, heads)
        want = run_block(torch, c, ending)
        dev = lambda a, dt=torch.bfloat16: torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=dt)  # noqa: E731
        f32 = torch.float32
        bo = torch.cat([torch.zeros(1, device="cuda"), dev(c["bo"], f32)])[1:]
        pair = dev(c["z"])
        blk = capi.TriangleAttentionBlock(pair, dev(c["mask"]), dev(c["gamma"], f32), dev(c["beta"], f32), dev(c["bias_w"]),
                                          dev(c["wq"]), dev(c["wk"]), dev(c["wv"]), dev(c["wg"]), dev(c["bg"], f32), dev(c["wo"]),
                                          bo, heads, ending)
        assert bo.data_ptr() % 16 == 4 and blk.run() == 0
        torch.cuda.synchronize()
        assert helpers.same_bits(pair, want)


def drawn_block(torch, seed, kind, n_seq, n_res, heads):
    """A block whose inputs are drawn on the device: kind "triangle" (n_res residues, ending node), "row" or "column" (MSA).  Returns
    the activation, its weights as a dict and a function (activation, weights) -> block."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, device="cuda", generator=g) * scale).to(torch.bfloat16)  # noqa: E731
    around = lambda centre, size: centre + 0.1 * torch.randn(size, device="cuda", generator=g)  # noqa: E731
    C = 32 * heads
    act = rnd(n_res if kind == "triangle" else n_seq, n_res, C)
    w = {k: rnd(C, C, scale=C ** -0.5) for k in ("wq", "wk", "wv", "wg", "wo")}
    w.update(ln_gamma=around(1.0, C), ln_beta=around(0.0, C), bg=around(1.0, C), bo=around(0.0, C))
    mask = (torch.rand(act.shape[:2], device="cuda", generator=g) > 0.1).to(torch.bfloat16)
    if kind == "triangle":
        bias_w = rnd(heads, C, scale=C ** -0.5)
        return act, w, lambda z, v: capi.TriangleAttentionBlock(z, mask, v["ln_gamma"], v["ln_beta"], bias_w, v["wq"], v["wk"], v["wv"], v["wg"],
                                                                v["bg"], v["wo"], v["bo"], heads, True)
    pair = None
    if kind == "row":
        pair = dict(pair_act=rnd(n_res, n_res, 64), pair_ln_gamma=around(1.0, 64), pair_ln_beta=around(0.0, 64), bias_w=rnd(heads, 64, scale=0.125))
    return act, w, lambda z, v: capi.MsaAttentionBlock(z, mask, v, heads, pair)


@pytest.mark.parametrize("kind,n_seq,n_res,heads", [("triangle", 0, 1025, 4), ("row", 3, 1057, 4), ("column", 1056, 3, 8)])
def test_blocks_beyond_1024_keys_replay_from_a_hip_graph(torch_cuda, kind, n_seq, n_res, heads):
    """Captured on a side stream and replayed three times, with eager work (the activation and the workspace overwritten) between the
    replays: every replay gives the eager result bit for bit."""
    torch = torch_cuda
    act, w, block = drawn_block(torch, 177 + n_res, kind, n_seq, n_res, heads)
    z = act.clone()
    blk = block(z, w)
    print(f"graph {kind} {n_seq}x{n_res} heads={heads}", flush=True)
    assert blk.run() == 0  # eager; also takes first-call set-up out of the capture
    torch.cuda.synchronize()
    want = z.clone()
    assert bool(torch.isfinite(want).all()) and not helpers.same_bits(want, act)
    z.copy_(act)
    torch.cuda.synchronize()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        assert blk.run(torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(3):
        z.copy_(act)
        blk.workspace.fill_(255)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert helpers.same_bits(z, want)


def test_triangle_attention_block_of_1025_residues(torch_cuda):
    """The first length past the fused head kernels' longest row, one key into its last tile and one row without a partner: both
    orientations against the oracle on a sample of attention rows."""
    torch = torch_cuda
    n = 1025
    c = block_case(9150, n, 4)
    rows = [0, 1, 31, 32, 512, n - 3, n - 2, n - 1]
    for ending in (False, True):
        got = run_block(torch, c, ending)
        assert bool(torch.isfinite(got).all())
        sample = got[:, rows].transpose(0, 1) if ending else got[rows]
        helpers.check_close(helpers.to_numpy(sample.contiguous()), block_oracle_rows(c, ending, rows), "bf16", f"block n={n} ending={ending}, sampled rows")


# rows without a partner; whole tiles and one key more or less; four and five query blocks to the last workgroup; sixteen workgroups
# and one more to a row; a pair bias whose producer does not write the tiles
@pytest.mark.parametrize("n,ending", [(1, False), (33, True), (1025, True), (1056, False)])
def test_streamed_triangle_block_stays_within_its_workspace(torch_cuda, streamed_everywhere, n, ending):
    """The size asked for, NaN beforehand and a guard behind it: the same bits as with any other contents, and the guard untouched; a
    byte less is refused."""
    torch = torch_cuda
    act, w, block = drawn_block(torch, 400 + n, "triangle", 0, n, 4)
    blk = block(act, w)
    blk.args.ending_node = int(ending)
    start, size = act.clone(), blk.args.workspace_bytes
    res = []
    for fill in (255, 0):
        act.copy_(start)
        room = torch.full((size + 4096,), fill, dtype=torch.uint8, device="cuda")
        room[size:] = 90
        blk.args.workspace = room.data_ptr()
        print(f"n={n} ending={ending} fill={fill}", flush=True)
        assert blk.run() == 0
        torch.cuda.synchronize()
        assert bool((room[size:] == 90).all())
        res.append(act.clone())
    assert bool(torch.isfinite(res[0]).all()) and helpers.same_bits(res[0], res[1]) and not helpers.same_bits(res[0], start)
    blk.args.workspace_bytes = size - 1
    assert blk.run() == capi.EINVAL


@pytest.mark.parametrize("column,n_seq,n_res,heads,c_z", [(False, 1, 1056, 4, 128), (True, 1055, 3, 4, 1), (True, 1057, 5, 8, 1), (True, 1152, 2, 4, 1),
                                                          (True, 1153, 1, 8, 1), (True, 2048, 2, 8, 1), (True, 2049, 3, 4, 1), (False, 2, 1281, 8, 16)])
def test_msa_attention_blocks_beyond_1024_keys(torch_cuda, column, n_seq, n_res, heads, c_z):
    torch = torch_cuda
    c = msa_case(9700 + n_seq + n_res, n_seq, n_res, heads, c_z)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = None if column else {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]),
                                "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    res = {}
    names = profiled_kernels(torch, lambda: res.setdefault("rc", capi.MsaAttentionBlock(msa, dev(c["mask"]), w, heads, pair).run()))
    torch.cuda.synchronize()
    assert res["rc"] == 0 and "streamed_attention_kernel" in names and ("pair_bias_tiles_kernel" in names) == (c_z == 16), (res, names)
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, column), "bf16", f"msa block {n_seq}x{n_res} heads={heads} column={column}")


# two rows a wave (with and without pair bias), four (at least three workgroups to two CUs), one to three of a set's rows missing
@pytest.mark.parametrize("column,n_seq,n_res,heads", [(False, 6, 70, 8), (True, 70, 7, 4), (False, 193, 33, 8), (False, 194, 65, 8), (False, 195, 32, 8)])
def test_streamed_rows_of_one_mask_beside_others(torch_cuda, streamed_everywhere, column, n_seq, n_res, heads):
    """Rows whose every key is masked attend uniformly, beside rows with some keys masked, or none, in one wave."""
    torch = torch_cuda
    c = msa_case(9800 + n_seq + n_res, n_seq, n_res, heads, 128)
    mask = c["mask"].T if column else c["mask"]
    mask[:] = 1.0
    mask[1::3] = 0.0
    mask[2::4, -(mask.shape[1] // 3):] = 0.0
    mask[-1] = 0.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = None if column else {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]),
                                "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    print(f"streamed rows of one mask {n_seq}x{n_res} heads={heads} column={column}", flush=True)
    assert capi.MsaAttentionBlock(msa, dev(c["mask"]), w, heads, pair).run() == 0
    torch.cuda.synchronize()
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, column), "bf16", f"rows of one mask {n_seq}x{n_res} heads={heads} column={column}")


# five and six blocks of queries: one and two left over, whose rows the last workgroup's waves share; three, which they do not; sets of four rows and
# of one to three
@pytest.mark.parametrize("n_seq,n_res", [(97, 129), (98, 160), (99, 161), (100, 190), (99, 192), (98, 200)])
def test_streamed_rows_of_left_over_query_blocks(torch_cuda, streamed_everywhere, n_seq, n_res):
    test_streamed_rows_of_one_mask_beside_others(torch_cuda, streamed_everywhere, False, n_seq, n_res, 8)


# without a pair bias: one block of queries and two a wave, three waves a workgroup (3 to 6, 9 to 12, 17 and 18 blocks) and four, the
# last workgroup full, with an odd block, and with waves that have none
@pytest.mark.parametrize("n_seq,n_res,heads", [(1, 5, 8), (33, 3, 4), (96, 2, 8), (193, 3, 4), (256, 2, 8), (257, 3, 8), (390, 2, 4), (520, 2, 8)])
def test_streamed_rows_without_pair_bias_at_the_edges_of_a_workgroup(torch_cuda, streamed_everywhere, n_seq, n_res, heads):
    torch = torch_cuda
    c = msa_case(9900 + n_seq, n_seq, n_res, heads, 128)
    c["mask"][:] = 1.0
    c["mask"][-(n_seq // 4):, n_res // 2] = 0.0  # masked keys at the end of one residue's row, anywhere in the next, everywhere in the last
    c["mask"][::3, (n_res // 2 + 1) % n_res] = 0.0
    c["mask"][:, -1] = 0.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    print(f"streamed column {n_seq}x{n_res} heads={heads}", flush=True)
    assert capi.MsaAttentionBlock(msa, dev(c["mask"]), w, heads, None).run() == 0
    torch.cuda.synchronize()
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, True), "bf16", f"streamed column {n_seq}x{n_res} heads={heads}")


# both sides of each line: more than 256 keys, from 129 sequences row-wise and 33 residues column-wise the first sixteen of every 32, from 257
# on all, 8 heads
@pytest.mark.parametrize("column,n_seq,n_res,heads,streamed", [
    (False, 129, 257, 8, True), (False, 128, 257, 8, False), (False, 129, 256, 8, False), (False, 129, 257, 4, False), (False, 130, 1024, 8, True),
    (True, 257, 33, 8, True), (True, 257, 32, 8, False), (True, 256, 33, 8, False), (True, 257, 33, 4, False), (True, 1023, 34, 8, True),
    (True, 257, 48, 8, True), (True, 257, 49, 8, False), (True, 257, 256, 8, False), (True, 257, 257, 8, True), (False, 145, 257, 8, False),
    (False, 281, 257, 8, True)])
def test_msa_blocks_that_prefer_the_streamed_kernels(torch_cuda, column, n_seq, n_res, heads, streamed):
    """The workspace decides where both kernels take a block: three activations are still enough, for the fused kernels, less is
    refused as before, and so are weights that the fused kernels refuse.  Both give the oracle's result within the parity bar, and so each
    other's within twice that."""
    torch = torch_cuda
    c = msa_case(9950 + n_seq + n_res, n_seq, n_res, heads, 64)
    c["mask"][1::2] *= np.where(c["mask"][1::2].cumsum(1) % 5 == 0, 0.5, 1.0).astype(np.float32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = None if column else {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]),
                                "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    up = lambda x: (x + 255) // 256 * 256  # noqa: E731
    fused_bytes = 3 * up(n_seq * n_res * heads * 64) + up(n_seq * n_res * 2) + (0 if column else up(heads * n_res * n_res * 2))
    mask = dev(c["mask"])
    res = []
    for size in (None, fused_bytes, fused_bytes - 256):
        msa = dev(c["m"])
        blk = capi.MsaAttentionBlock(msa, mask, w, heads, pair)
        assert (blk.args.workspace_bytes > fused_bytes) == streamed and blk.args.workspace_bytes >= fused_bytes
        if size is not None:
            blk.args.workspace_bytes = size
        rc = {}
        print(f"msa {n_seq}x{n_res} heads={heads} column={column} workspace={size}", flush=True)
        names = profiled_kernels(torch, lambda: rc.setdefault("rc", blk.run()))  # noqa: B023
        torch.cuda.synchronize()
        if size == fused_bytes - 256:
            assert rc["rc"] == capi.EINVAL and helpers.same_bits(msa, dev(c["m"]))
            continue
        assert rc["rc"] == 0 and ("streamed_attention_kernel" in names) == (streamed and size is None), (rc, names)
        res.append(helpers.to_numpy(msa))
    if n_seq * n_res < 40000:
        want = msa_oracle(c, column)
        for got in res:
            helpers.check_close(got, want, "bf16", f"msa {n_seq}x{n_res} heads={heads} column={column}")
    helpers.assert_within(res[0], res[1], 2 * (2e-2 + 1e-2 * np.abs(res[1])), f"routes {n_seq}x{n_res} heads={heads} column={column}")
    moved = {k: t if k.startswith("ln_") else torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape) for k, t in w.items()}
    msa = dev(c["m"])
    assert capi.MsaAttentionBlock(msa, mask, moved, heads, pair).run() == capi.EUNSUPPORTED
    torch.cuda.synchronize()
    assert helpers.same_bits(msa, dev(c["m"]))


@pytest.mark.parametrize("kind,n_seq,n_res,heads", [("triangle", 0, 1025, 4), ("row", 3, 1050, 8), ("column", 1030, 2, 4)])
def test_blocks_beyond_1024_keys_take_weights_on_any_address(torch_cuda, kind, n_seq, n_res, heads):
    """The route of these blocks asks nothing of the weights' alignment: the same bits with every matrix and both biases one element
    past a 16-byte boundary."""
    torch = torch_cuda
    act, w, block = drawn_block(torch, 77 + n_res, kind, n_seq, n_res, heads)
    moved = {k: t if k.startswith("ln_") else torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape) for k, t in w.items()}
    assert all(moved[k].data_ptr() % 16 == w[k].element_size() for k in ("wq", "wk", "wv", "wg", "wo", "bg", "bo"))
    res = []
    for weights in (w, moved):
        z = act.clone()
        print(f"{kind} {n_seq}x{n_res} heads={heads} moved={weights is moved}", flush=True)
        rc = block(z, weights).run()
        torch.cuda.synchronize()
        assert rc == 0, rc
        res.append(z)
    assert bool(torch.isfinite(res[0]).all()) and not helpers.same_bits(res[0], act)
    assert helpers.same_bits(res[0], res[1])


def test_fused_layernorm_drops_the_normalised_copy_from_the_workspace(torch_cuda):
    """With the LayerNorm inside the attention kernel the blocks keep no normalised activation: the workspace is one
    activation smaller wherever the persistent kernel runs (384 residues), and unchanged where it does not (1024)."""
    L = capi.lib()
    sizes = {}
    for mode in ("fused", "separate"):
        assert capi.set_tuning("layernorm", mode) == 0
        sizes[mode] = (L.kutacc_hip_triangle_attention_workspace(384, 4), L.kutacc_hip_triangle_attention_workspace(1024, 4),
                       L.kutacc_hip_msa_attention_workspace(512, 256, 8, 0))
    capi.set_tuning("layernorm", "auto")
    assert sizes["separate"][0] - sizes["fused"][0] == 384 * 384 * 128 * 2
    assert sizes["separate"][1] == sizes["fused"][1]
    assert sizes["separate"][2] - sizes["fused"][2] == 512 * 256 * 256 * 2


def test_triangle_attention_block_rejects_bad_arguments(torch_cuda):
    torch = torch_cuda
    L = capi.lib()
    assert L.kutacc_hip_triangle_attention(None, None) == capi.EINVAL
    assert L.kutacc_hip_triangle_attention_workspace(0, 4) == -1
    c = block_case(1, 40, 4)
    dev = lambda a, dt=torch.bfloat16: torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=dt)  # noqa: E731
    blk = capi.TriangleAttentionBlock(dev(c["z"]), dev(c["mask"]), dev(c["gamma"], torch.float32), dev(c["beta"], torch.float32),
                                      dev(c["bias_w"]), dev(c["wq"]), dev(c["wk"]), dev(c["wv"]), dev(c["wg"]),
                                      dev(c["bg"], torch.float32), dev(c["wo"]), dev(c["bo"], torch.float32), 4, False)
    blk.args.workspace_bytes -= 1
    assert blk.run() == capi.EINVAL
    blk.args.workspace_bytes += 1
    blk.args.nheads = 3  # 96 channels: no MFMA attention kernel
    assert blk.run() in (capi.EUNSUPPORTED, capi.EINVAL)
    torch.cuda.synchronize()


# ---- channel-first LayerNorm and the triangle-multiplication block ------------------------------------------------
@pytest.mark.parametrize("channels,positions,dtype", [(128, 4096, "bfloat16"), (128, 1000, "bfloat16"), (128, 40, "bfloat16"),
                                                      (96, 77, "bfloat16"), (20, 33, "float32")])
def test_layernorm_channel_first(torch_cuda, channels, positions, dtype):
    """Against the oracle's row LayerNorm on the transposed tensor: fast path (128 channels, ragged position counts) and
    the generic kernel."""
    from oracle import oracle
    torch = torch_cuda
    dt = getattr(torch, dtype)
    rng = np.random.Generator(np.random.PCG64(31 + positions))
    x = (rng.standard_normal((channels, positions)) * 2 + rng.standard_normal((1, positions))).astype(np.float32)
    if dtype == "bfloat16":
        x = round_to_bf16(x)
    gamma = (rng.random(channels) + 0.5).astype(np.float32)
    beta = (rng.standard_normal(channels) * 0.2).astype(np.float32)
    dx = torch.from_numpy(x).to(device="cuda", dtype=dt)
    out = torch.full((positions, channels + 8), 9.0, dtype=dt, device="cuda")
    g, b = torch.from_numpy(gamma).cuda(), torch.from_numpy(beta).cuda()
    rc = capi.lib().kutacc_hip_layernorm_channel_first(dx.data_ptr(), positions, g.data_ptr(), b.data_ptr(), out.data_ptr(),
                                                       channels + 8, channels, positions, 1e-5, code(torch, dx), None)
    torch.cuda.synchronize()
    assert rc == 0
    ref = oracle.layernorm_rows_f32(np.ascontiguousarray(x.T), gamma, beta, 1e-5)
    helpers.check_close(helpers.to_numpy(out[:, :channels]), ref, "bf16" if dtype == "bfloat16" else "fp32", "channel-first LN")
    assert bool((out[:, channels:] == 9.0).all())


def tm_block_case(seed, n, c_z, c_i):
    rng = np.random.Generator(np.random.PCG64(seed))
    w = lambda o, i: round_to_bf16((rng.standard_normal((o, i)) / math.sqrt(i)).astype(np.float32))  # noqa: E731
    b = lambda k: (rng.standard_normal(k) * 0.3).astype(np.float32)  # noqa: E731
    g = lambda k: (rng.random(k) + 0.5).astype(np.float32)  # noqa: E731
    return dict(z=round_to_bf16(rng.standard_normal((n, n, c_z)).astype(np.float32)),
                mask=(rng.random((n, n)) > 0.15).astype(np.float32),
                ln_in_gamma=g(c_z), ln_in_beta=b(c_z), left_proj_w=w(c_i, c_z), left_proj_b=b(c_i), left_gate_w=w(c_i, c_z),
                left_gate_b=b(c_i), right_proj_w=w(c_i, c_z), right_proj_b=b(c_i), right_gate_w=w(c_i, c_z), right_gate_b=b(c_i),
                ln_center_gamma=g(c_i), ln_center_beta=b(c_i), output_w=w(c_z, c_i), output_b=b(c_z), gating_w=w(c_z, c_z),
                gating_b=b(c_z))


def tm_block_oracle(c, incoming):
    """AlphaFold's TriangleMultiplication in numpy on the oracle's operators (fp32, no intermediate rounding)."""
    from oracle import oracle
    n, _, c_z = c["z"].shape
    c_i = c["left_proj_w"].shape[0]
    act = oracle.layernorm_rows_f32(c["z"].reshape(-1, c_z), c["ln_in_gamma"], c["ln_in_beta"], 1e-5).reshape(n, n, c_z)
    left = oracle.tm_calc_proj_f32(act, c["mask"], c["left_proj_w"], c["left_proj_b"], c["left_gate_w"], c["left_gate_b"])
    right = oracle.tm_calc_proj_f32(act, c["mask"], c["right_proj_w"], c["right_proj_b"], c["right_gate_w"], c["right_gate_b"])
    center = oracle.tm_equation_f32(left, right, incoming)
    center = oracle.layernorm_rows_f32(np.ascontiguousarray(center.transpose(1, 2, 0)).reshape(-1, c_i), c["ln_center_gamma"],
                                       c["ln_center_beta"], 1e-5)
    gate, out = oracle.tm_gate_and_out_f32(act, center, c["gating_w"], c["gating_b"], c["output_w"], c["output_b"])
    return c["z"] + oracle.tm_last_f32(out, gate).reshape(n, n, c_z)


@pytest.mark.parametrize("incoming", [False, True], ids=["outgoing", "incoming"])
# 48: the last kernel takes the centre channel-first, normalises it and projects the gate itself; 46 (positions not in
# whole 16-byte runs): it still projects the gate, behind the stand-alone channel-first LayerNorm; the others: separate passes
@pytest.mark.parametrize("n,c_z,c_i", [(48, 128, 128), (46, 128, 128), (40, 64, 32), (9, 12, 6)])
def test_triangle_multiplication_block_against_the_oracle(torch_cuda, n, c_z, c_i, incoming):
    torch = torch_cuda
    c = tm_block_case(800 + n, n, c_z, c_i)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    pair = dev(c["z"])
    w = {k: dev(v) for k, v in c.items() if k not in ("z", "mask")}
    blk = capi.TriangleMultiplicationBlock(pair, dev(c["mask"]), w, incoming)
    rc = blk.run()
    torch.cuda.synchronize()
    assert rc == 0, rc
    helpers.check_close(helpers.to_numpy(pair), tm_block_oracle(c, incoming), "bf16", f"TM block n={n} incoming={incoming}")


@pytest.mark.parametrize("index,n", [(i, int(n)) for i, n in enumerate(np.random.Generator(np.random.PCG64(31)).integers(8, 90, size=8))])
def test_triangle_multiplication_block_seeded_sweep(torch_cuda, index, n):
    """Eight seeded pair sizes between 8 and 89 at 128 channels (positions in and out of whole 16-byte runs, so both forms of
    the block's last kernel and the stand-alone centre LayerNorm), orientation alternating, against the oracle."""
    torch = torch_cuda
    incoming = bool(index & 1)
    c = tm_block_case(2000 + index, n, 128, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    pair = dev(c["z"])
    w = {k: dev(v) for k, v in c.items() if k not in ("z", "mask")}
    assert capi.TriangleMultiplicationBlock(pair, dev(c["mask"]), w, incoming).run() == 0
    torch.cuda.synchronize()
    helpers.check_close(helpers.to_numpy(pair), tm_block_oracle(c, incoming), "bf16", f"TM block sweep {index}: n={n} incoming={incoming}")


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 33, 63, 64, 65, 127, 129, 200])
def test_triangle_multiplication_block_at_any_length(torch_cuda, n):
    """128 channels, lengths around the padded pitch (8), the steps of the block's first and last kernel (64 positions) and the
    tiles of the product (128), both orientations; a guard behind the activation shows a store past the last row."""
    torch = torch_cuda
    case = tm_block_case(3000 + n, n, 128, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    w = {k: dev(v) for k, v in case.items() if k not in ("z", "mask")}
    for incoming in (False, True):
        guarded = torch.full((n * n + 64, 128), 7.0, device="cuda", dtype=torch.bfloat16)
        pair = guarded[:n * n].view(n, n, 128)
        pair.copy_(dev(case["z"]))
        print(f"n={n} incoming={incoming}", flush=True)
        assert capi.TriangleMultiplicationBlock(pair, dev(case["mask"]), w, incoming).run() == 0
        torch.cuda.synchronize()
        want = tm_block_oracle(case, incoming)
        # Values behind the roundings of the normalised row, projections, their products and the centre (0.2 % each, two sides): the
        # normalised centre, of order one, is off by 0.5 % rms, and so is the update at most; 5 million of them lie within five
        # times that.  The sum with the activation is rounded once more, by at most 2^-8.
        got = helpers.to_numpy(pair)
        helpers.assert_within(got, want, 2.5e-2 + 2.0 ** -8 * np.abs(want), f"TM block n={n} incoming={incoming}")
        assert np.sqrt(np.mean((got - want) ** 2)) < 5e-3
        assert bool((guarded[n * n:] == 7.0).all())


@pytest.mark.parametrize("n,mode", [(257, "direct"), (290, "direct"), (480, "direct"), (509, "direct"), (674, None), (765, None)])
def test_triangle_multiplication_block_on_tiles_over_the_edge(torch_cuda, n, mode):
    """Lengths that are no multiple of 256 on the 256 x 256 tiles, which read past the planes' edges: the same bits as on the
    128 x 128 tiles, in a workspace that holds NaN beforehand."""
    torch = torch_cuda
    case = tm_block_case(3500 + n, n, 128, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    w = {k: dev(v) for k, v in case.items() if k not in ("z", "mask")}
    for incoming in (False, True):
        got = {}
        for tile in ("128", mode):
            assert capi.set_tuning("gemm_tile", tile) == 0
            try:
                pair = dev(case["z"])
                blk = capi.TriangleMultiplicationBlock(pair, dev(case["mask"]), w, incoming)
                blk.workspace.fill_(255)
                assert blk.run() == 0
                torch.cuda.synchronize()
            finally:
                capi.set_tuning("gemm_tile", None)
            got[tile] = pair
        assert bool(torch.isfinite(got[mode]).all()) and helpers.same_bits(got["128"], got[mode]), (n, incoming)


# three tiles a side with an even number of 128 x 128 tiles and with an odd one, four with an odd one up to whole tiles, 14 % of padding
# with an odd number, six
@pytest.mark.parametrize("n,outgoing,incoming", [(640, False, False), (641, True, True), (769, False, True), (896, False, True), (1122, False, True),
                                                 (1130, True, True), (1281, True, True)])
def test_lengths_at_which_the_equation_runs_over_the_edge(torch_cuda, n, outgoing, incoming):
    """The same bits on either tiles, in a workspace that holds NaN beforehand."""
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *sh, scale=1.0: torch.randn(*sh, device="cuda", generator=g) * scale  # noqa: E731
    case = tm_block_case(3700 + n, 8, 128, 128)
    w = {k: torch.from_numpy(np.ascontiguousarray(v)).to(device="cuda", dtype=torch.bfloat16 if v.ndim >= 2 else torch.float32)
         for k, v in case.items() if k not in ("z", "mask")}
    act = rnd(n, n, 128).to(torch.bfloat16)
    mask = (torch.rand(n, n, device="cuda", generator=g) > 0.1).to(torch.bfloat16)
    for edge, direct in ((False, outgoing), (True, incoming)):
        got = []
        for tile in (None, "128"):
            assert capi.set_tuning("gemm_tile", tile) == 0
            try:
                pair = act.clone()
                blk = capi.TriangleMultiplicationBlock(pair, mask, w, edge)
                blk.workspace.fill_(255)
                print(f"n={n} incoming={edge} tile={tile}", flush=True)
                names = profiled_kernels(torch, lambda: blk.run())  # noqa: B023
                torch.cuda.synchronize()
            finally:
                capi.set_tuning("gemm_tile", None)
            assert any(k.startswith("pair_gemm_direct_kernel") for k in names) == (direct and tile is None), names
            got.append(pair)
        assert bool(torch.isfinite(got[0]).all()) and helpers.same_bits(got[0], got[1]), (n, edge)
        assert not helpers.same_bits(got[0], act)


@pytest.mark.parametrize("n", [8, 64, 72, 200, 384])
@pytest.mark.parametrize("kind", ["ones", "one zero", "padding", "halves"])
def test_triangle_multiplication_block_of_steps_without_a_mask(torch_cuda, n, kind):
    """Steps of 64 positions whose masks are all one are not multiplied by them: the streaming kernel's bits with no such step, with all, and with both."""
    torch = torch_cuda
    case = tm_block_case(3900 + n, n, 128, 128)
    mask = np.ones((n, n), np.float32)
    if kind == "one zero":
        mask[n // 2, n // 3] = 0
    elif kind == "padding":
        mask[:, n - n // 10 - 1:] = mask[n - n // 10 - 1:, :] = 0
    elif kind == "halves":
        mask[n // 2:] = 0.5
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    w = {k: dev(v) for k, v in case.items() if k not in ("z", "mask")}
    got = []
    for mode in (None, "streaming"):
        assert capi.set_tuning("gated_projection", mode) == 0
        try:
            pair = dev(case["z"])
            assert capi.TriangleMultiplicationBlock(pair, dev(mask), w, True).run() == 0
            torch.cuda.synchronize()
        finally:
            capi.set_tuning("gated_projection", None)
        got.append(pair)
    assert bool(torch.isfinite(got[0]).all()) and helpers.same_bits(got[0], got[1])


@pytest.mark.parametrize("n", [48, 72, 384])
def test_triangle_multiplication_block_on_each_gated_projection_kernel(torch_cuda, n):
    """The block's two gated projections go out in one launch.  Its default kernel (weights in registers, both sides in
    one pass over the activation) must give the block's result bit for bit as the streaming kernel does, and within the
    rounding of the intermediates as the tiled kernel does."""
    torch = torch_cuda
    case = tm_block_case(900 + n, n, 128, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    w = {k: dev(v) for k, v in case.items() if k not in ("z", "mask")}
    want = {None: "triangle_front_kernel", "streaming": "gated_projection_kernel<2>", "tiled": "pair_gemm_kernel<gated>"}
    res = {}
    for mode in want:
        assert capi.set_tuning("gated_projection", mode) == 0
        try:
            pair = dev(case["z"])
            capi.lib().kutacc_hip_profile_enable(1)
            assert capi.TriangleMultiplicationBlock(pair, dev(case["mask"]), w, False).run() == 0
            torch.cuda.synchronize()
            names = []
            for i in range(16):
                name = ctypes.create_string_buffer(96)
                ms, cnt, fl = ctypes.c_double(), ctypes.c_int64(), ctypes.c_double()
                if capi.lib().kutacc_hip_profile_read(i, name, 96, ctypes.byref(ms), ctypes.byref(cnt), ctypes.byref(fl)) != 0:
                    break
                names.append(name.value.decode())
        finally:
            capi.lib().kutacc_hip_profile_enable(0)
            capi.set_tuning("gated_projection", None)
        assert want[mode] in names, (mode, names)
        res[mode] = pair
    assert helpers.same_bits(res[None], res["streaming"])
    tiled = helpers.to_numpy(res["tiled"])
    helpers.assert_within(helpers.to_numpy(res[None]), tiled, 4e-2 + 2e-2 * np.abs(tiled), "weights in registers vs tiled kernel")


@pytest.mark.parametrize("incoming", [False, True], ids=["outgoing", "incoming"])
@pytest.mark.parametrize("n", [384, 512, 768])  # 768: the equation on the 256 x 256 tiles
def test_triangle_multiplication_block_full_size(torch_cuda, incoming, n):
    """384 residues, 128 channels, the real shape, 512 and 768 (both gated projections in one pass over the activation).  The oracle follows a sample of output positions (i, j) through the
    whole block: their centre needs the left projections of row i and the right projections of row j (columns for the
    incoming form), which the oracle computes for just those rows."""
    from oracle import oracle
    torch = torch_cuda
    c = 128
    case = tm_block_case(900 + n, n, c, c)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    w = {k: dev(v) for k, v in case.items() if k not in ("z", "mask")}
    pair = dev(case["z"])
    assert capi.TriangleMultiplicationBlock(pair, dev(case["mask"]), w, incoming).run() == 0
    torch.cuda.synchronize()
    got = helpers.to_numpy(pair)
    I, J = [0, 77, 200, n - 1], [5, 100, n - 1]
    act = oracle.layernorm_rows_f32(case["z"].reshape(-1, c), case["ln_in_gamma"], case["ln_in_beta"], 1e-5).reshape(n, n, c)
    proj = lambda side, x, m: oracle.tm_calc_proj_f32(x, m, case[side + "_proj_w"], case[side + "_proj_b"],  # noqa: E731
                                                       case[side + "_gate_w"], case[side + "_gate_b"])
    if not incoming:  # center[c, i, j] = sum_k left[c, i, k] right[c, j, k]
        left, right = proj("left", act[I], case["mask"][I]), proj("right", act[J], case["mask"][J])
        center = np.einsum("cik,cjk->ijc", left.astype(np.float64), right.astype(np.float64))
    else:             # center[c, i, j] = sum_k right[c, k, i] left[c, k, j]
        right = proj("right", np.ascontiguousarray(act[:, I]), np.ascontiguousarray(case["mask"][:, I]))
        left = proj("left", np.ascontiguousarray(act[:, J]), np.ascontiguousarray(case["mask"][:, J]))
        center = np.einsum("cki,ckj->ijc", right.astype(np.float64), left.astype(np.float64))
    center = oracle.layernorm_rows_f32(center.reshape(-1, c).astype(np.float32), case["ln_center_gamma"], case["ln_center_beta"], 1e-5)
    act_ij = act[np.ix_(I, J)].reshape(-1, c)
    gate, out = oracle.tm_gate_and_out_f32(act_ij, center, case["gating_w"], case["gating_b"], case["output_w"], case["output_b"])
    want = case["z"][np.ix_(I, J)].reshape(-1, c) + oracle.tm_last_f32(out, gate)
    helpers.check_close(got[np.ix_(I, J)].reshape(-1, c), want, "bf16", f"TM block {n} incoming={incoming}")
    assert not np.array_equal(got, case["z"])


@pytest.mark.parametrize("m,n,k", [(1000, 128, 128), (333, 256, 128), (520, 128, 256)])
def test_gated_residual_projection(torch_cuda, m, n, k):
    """acc += bf16(a . w^T + bias) * sigmoid(gate) in one kernel, against the same three steps in float64."""
    torch = torch_cuda
    rng = np.random.Generator(np.random.PCG64(40 + m))
    a = round_to_bf16(rng.standard_normal((m, k)).astype(np.float32))
    w = round_to_bf16((rng.standard_normal((n, k)) / math.sqrt(k)).astype(np.float32))
    bias = (rng.standard_normal(n) * 0.3).astype(np.float32)
    gate = round_to_bf16(rng.standard_normal((m, n)).astype(np.float32) * 2)
    acc = round_to_bf16(rng.standard_normal((m, n)).astype(np.float32))
    dev = lambda x, dt=torch.bfloat16: torch.from_numpy(x).to(device="cuda", dtype=dt)  # noqa: E731
    d_acc = dev(acc)
    t = [dev(a), dev(w), dev(bias, torch.float32), dev(gate)]
    rc = capi.lib().kutacc_hip_gated_residual_projection(t[0].data_ptr(), k, t[1].data_ptr(), t[2].data_ptr(), t[3].data_ptr(), n,
                                                         d_acc.data_ptr(), n, m, n, k, capi.K_BF16, None)
    torch.cuda.synchronize()
    assert rc == 0, rc
    o = a.astype(np.float64) @ w.astype(np.float64).T + bias
    want = acc + o / (1.0 + np.exp(-gate.astype(np.float64)))
    helpers.check_close(helpers.to_numpy(d_acc), want, "bf16", "gated residual projection")
    rc = capi.lib().kutacc_hip_gated_residual_projection(t[0].data_ptr(), k, t[1].data_ptr(), t[2].data_ptr(), t[3].data_ptr(), n,
                                                         d_acc.data_ptr(), n, m, 96, k, capi.K_BF16, None)
    assert rc == capi.EUNSUPPORTED


# 65536 + 20000 rows: more than one round of workgroups plus a partial one
@pytest.mark.parametrize("rows,c_o,c_i", [(300, 128, 512), (200, 256, 1024), (64 * 64, 128, 512), (50, 24, 40),
                                          (65536 + 20000, 128, 256)])
def test_transition_block(torch_cuda, rows, c_o, c_i):
    """act += transition(LN(act)) in place: the one-kernel form (pair and MSA channel counts, ragged row counts) and the
    separate-pass form through a workspace, against the oracle's LayerNorm and transition composed in numpy."""
    from oracle import oracle
    torch = torch_cuda
    rng = np.random.Generator(np.random.PCG64(70 + rows))
    x = round_to_bf16((rng.standard_normal((rows, c_o)) * 1.5 + 0.3).astype(np.float32))
    gamma, beta = (rng.random(c_o) + 0.5).astype(np.float32), (rng.standard_normal(c_o) * 0.2).astype(np.float32)
    w1 = round_to_bf16((rng.standard_normal((c_i, c_o)) / math.sqrt(c_o)).astype(np.float32))
    w2 = round_to_bf16((rng.standard_normal((c_o, c_i)) / math.sqrt(c_i)).astype(np.float32))
    b1, b2 = (rng.standard_normal(c_i) * 0.3).astype(np.float32), (rng.standard_normal(c_o) * 0.3).astype(np.float32)
    dev = lambda a, dt=torch.bfloat16: torch.from_numpy(a).to(device="cuda", dtype=dt)  # noqa: E731
    f32 = torch.float32
    act = dev(x)
    t = [dev(gamma, f32), dev(beta, f32), dev(w1), dev(b1, f32), dev(w2), dev(b2, f32)]
    L = capi.lib()
    nbytes = L.kutacc_hip_transition_block_workspace(rows, c_o, c_i)
    assert (nbytes == 0) == (c_o in (128, 256))
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device="cuda")
    rc = L.kutacc_hip_transition_block(act.data_ptr(), t[0].data_ptr(), t[1].data_ptr(), 1e-5, t[2].data_ptr(), t[3].data_ptr(),
                                       t[4].data_ptr(), t[5].data_ptr(), ws.data_ptr() if nbytes else None, nbytes, rows, c_o, c_i,
                                       capi.K_BF16, None)
    torch.cuda.synchronize()
    assert rc == 0, rc
    want = x + oracle.transition_f32(oracle.layernorm_rows_f32(x, gamma, beta, 1e-5), w1, b1, w2, b2)
    helpers.check_close(helpers.to_numpy(act), want, "bf16", f"transition block {rows}x{c_o}->{c_i}")
    if nbytes:  # without its workspace the separate-pass form must refuse
        assert L.kutacc_hip_transition_block(act.data_ptr(), t[0].data_ptr(), t[1].data_ptr(), 1e-5, t[2].data_ptr(),
                                             t[3].data_ptr(), t[4].data_ptr(), t[5].data_ptr(), None, 0, rows, c_o, c_i,
                                             capi.K_BF16, None) == capi.EINVAL


# one row; a row past a wave's 32; the last row count of the kernel for few rows (32 per CU) and the first past it; whole
# rounds of workgroups and a remainder, for each width; the narrowest and the widest hidden layer
@pytest.mark.parametrize("rows,c_o,c_i", [(1, 64, 64), (1, 256, 64), (33, 128, 2048), (33, 64, 2048), (31, 256, 2048), (8192, 128, 192),
                                          (8193, 128, 192), (8192, 256, 64), (8193, 256, 64), (98304 + 4133, 128, 64),
                                          (65536 + 33, 256, 64), (131072 + 33, 64, 128)])
def test_transition_block_at_the_edges_of_its_kernels(torch_cuda, rows, c_o, c_i):
    from oracle import oracle
    torch = torch_cuda
    print(rows, c_o, c_i, flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + c_i)
    draw = lambda *s, scale=1.0, centre=0.0: torch.randn(*s, device="cuda", generator=g) * scale + centre  # noqa: E731
    act = draw(rows, c_o, scale=1.5, centre=0.3).to(torch.bfloat16)
    gamma, beta, b1, b2 = draw(c_o, scale=0.1, centre=1.0), draw(c_o, scale=0.2), draw(c_i, scale=0.3), draw(c_o, scale=0.3)
    w1, w2 = draw(c_i, c_o, scale=c_o ** -0.5).to(torch.bfloat16), draw(c_o, c_i, scale=c_i ** -0.5).to(torch.bfloat16)
    num = helpers.to_numpy
    x = num(act)
    want = x + oracle.transition_f32(oracle.layernorm_rows_f32(x, num(gamma), num(beta), 1e-5), num(w1), num(b1), num(w2), num(b2))
    L = capi.lib()
    nbytes = L.kutacc_hip_transition_block_workspace(rows, c_o, c_i)
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device="cuda")
    res = {}
    names = profiled_kernels(torch, lambda: res.setdefault("rc", L.kutacc_hip_transition_block(
        act.data_ptr(), gamma.data_ptr(), beta.data_ptr(), 1e-5, w1.data_ptr(), b1.data_ptr(), w2.data_ptr(), b2.data_ptr(), ws.data_ptr(),
        nbytes, rows, c_o, c_i, capi.K_BF16, None)))
    assert res["rc"] == 0
    few = c_o != 64 and (rows + 31) // 32 <= torch.cuda.get_device_properties(0).multi_processor_count
    assert names == ["transition_split_kernel<block>" if few else "transition_rows_kernel<block>"], names
    helpers.check_close(num(act), want, "bf16", f"transition block {rows}x{c_o}->{c_i}")


# one workgroup of eight waves a CU (with 256 channels from 128 rows a CU on, with 128 from 32, up to 256): first and last row counts, few hidden
# units and many; and b2 behind b1 in the LDS and in its place
@pytest.mark.parametrize("rows,c_o,c_i", [(20011, 128, 512), (65536, 128, 64), (32768, 256, 64), (32769, 256, 64), (32769, 256, 128), (40011, 256, 192), (65536, 256, 1024),
                                          (98304 + 4133, 128, 192), (65536 + 33, 256, 320), (131072 + 33, 64, 64)])
def test_transition_block_with_one_workgroup_a_cu(torch_cuda, rows, c_o, c_i):
    test_transition_block_at_the_edges_of_its_kernels(torch_cuda, rows, c_o, c_i)


# ---- MSA attention blocks ------------------------------------------------------------------------------------------
def msa_case(seed, n_seq, n_res, heads, c_z):
    rng = np.random.Generator(np.random.PCG64(seed))
    c = heads * 32
    w = lambda o, i: round_to_bf16((rng.standard_normal((o, i)) / math.sqrt(i)).astype(np.float32))  # noqa: E731
    mask = (rng.random((n_seq, n_res)) > 0.1).astype(np.float32)
    mask[:, -2:] = 0.0  # padded residues
    mask[-1, :] = 0.0   # a padded sequence: a fully masked row for the row-wise form
    return dict(m=round_to_bf16(rng.standard_normal((n_seq, n_res, c)).astype(np.float32)), mask=mask,
                z=round_to_bf16(rng.standard_normal((n_res, n_res, c_z)).astype(np.float32)),
                ln_gamma=(rng.random(c) + 0.5).astype(np.float32), ln_beta=(rng.standard_normal(c) * 0.1).astype(np.float32),
                pair_ln_gamma=(rng.random(c_z) + 0.5).astype(np.float32),
                pair_ln_beta=(rng.standard_normal(c_z) * 0.1).astype(np.float32), bias_w=w(heads, c_z),
                wq=w(c, c), wk=w(c, c), wv=w(c, c), wg=w(c, c), wo=w(c, c), bg=np.ones(c, np.float32),
                bo=(rng.standard_normal(c) * 0.1).astype(np.float32), heads=heads)


def msa_oracle(c, column):
    """AlphaFold's MSARowAttentionWithPairBias / MSAColumnAttention in numpy on the oracle's operators."""
    from oracle import oracle
    m, mask = c["m"], c["mask"]
    if column:
        m, mask = m.transpose(1, 0, 2), mask.T
    B, S, ch = m.shape
    mn = oracle.layernorm_rows_f32(np.ascontiguousarray(m).reshape(-1, ch), c["ln_gamma"], c["ln_beta"], 1e-5).reshape(B, S, ch)
    nb = None
    if not column:
        n_res, _, cz = c["z"].shape
        zn = oracle.layernorm_rows_f32(c["z"].reshape(-1, cz), c["pair_ln_gamma"], c["pair_ln_beta"], 1e-5)
        nb = np.ascontiguousarray(oracle.linear_f32(zn, c["bias_w"]).reshape(n_res, n_res, c["heads"]).transpose(2, 0, 1))
    bias = (np.ascontiguousarray(mask) * np.float32(1e9) - np.float32(1e9)).astype(np.float32)
    out = oracle.gating_attention_f32(mn, c["wq"], c["wk"], c["wv"], c["wg"], c["bg"], c["wo"], c["bo"], bias, nb, c["heads"])
    if column:
        out = out.transpose(1, 0, 2)
    return c["m"] + out


@pytest.mark.parametrize("column", [False, True], ids=["row-wise with pair bias", "column-wise"])
@pytest.mark.parametrize("n_seq,n_res,heads,c_z", [(24, 40, 8, 128), (50, 20, 8, 128), (33, 33, 4, 64), (24, 64, 8, 128),
                                                   (20, 96, 8, 128)])
def test_msa_attention_block_against_the_oracle(torch_cuda, layernorm_placement, n_seq, n_res, heads, c_z, column):
    torch = torch_cuda
    c = msa_case(1000 + n_seq, n_seq, n_res, heads, c_z)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = None if column else {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]),
                                "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    blk = capi.MsaAttentionBlock(msa, dev(c["mask"]), w, heads, pair)
    rc = blk.run()
    torch.cuda.synchronize()
    assert rc == 0, rc
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, column), "bf16", f"msa block {n_seq}x{n_res} column={column}")


@pytest.mark.parametrize("n_seq,n_res", [(24, 64), (20, 96), (70, 128), (9, 32)])
def test_msa_row_attention_block_on_the_two_row_kernel(torch_cuda, n_seq, n_res):
    """Row-wise MSA attention (256 channels, eight heads) with whole key tiles and the two-row kernel forced: the
    producer of the pair bias writes that kernel's fp32 tiles, and the operator runs no pre-pass."""
    torch = torch_cuda
    heads, c_z = 8, 128
    c = msa_case(1200 + n_seq, n_seq, n_res, heads, c_z)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]), "pair_ln_beta": dev(c["pair_ln_beta"]),
            "bias_w": dev(c["bias_w"])}
    assert capi.set_tuning("row_pairs", "1") == 0
    try:
        blk = capi.MsaAttentionBlock(msa, dev(c["mask"]), w, heads, pair)
        names = profiled_kernels(torch, lambda: blk.run())
    finally:
        capi.set_tuning("row_pairs", None)
    assert "persistent_pair_kernel" in names and "pair_bias_tiles_kernel" not in names and "pair_bias_fragments_kernel" not in names, names
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, False), "bf16", f"msa row block {n_seq}x{n_res}, two-row kernel")


def test_layernorm_rows_transposed(torch_cuda):
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(4)
    for rows_i, rows_j, size, dt in ((20, 36, 256, torch.bfloat16), (7, 9, 24, torch.float32)):
        x_t = torch.randn(rows_j, rows_i, size, device="cuda", generator=g).to(dt)
        gamma = torch.rand(size, device="cuda", generator=g) + 0.5
        beta = torch.randn(size, device="cuda", generator=g) * 0.1
        a, b = torch.zeros(rows_i, rows_j, size, dtype=dt, device="cuda"), torch.zeros(rows_i, rows_j, size, dtype=dt, device="cuda")
        L = capi.lib()
        x = x_t.transpose(0, 1).contiguous()
        assert L.kutacc_hip_layernorm_rows(x.data_ptr(), size, gamma.data_ptr(), beta.data_ptr(), a.data_ptr(), size,
                                           rows_i * rows_j, size, 1e-5, code(torch, x), None) == 0
        assert L.kutacc_hip_layernorm_rows_transposed(x_t.data_ptr(), gamma.data_ptr(), beta.data_ptr(), b.data_ptr(), rows_i,
                                                      rows_j, size, 1e-5, code(torch, x), None) == 0
        torch.cuda.synchronize()
        assert helpers.same_bits(a, b)


def test_pair_stack_blocks_replay_from_a_hip_graph(torch_cuda):
    """The three pair-stack blocks (triangle multiplication, triangle attention, transition) captured into one HIP graph
    on a side stream and replayed three times, with eager work (restoring the pair tensor) between the replays; every
    replay must reproduce the eager result bit for bit.  Nothing in the launch path allocates, frees, memsets or
    synchronises, which is what makes the blocks capturable."""
    torch = torch_cuda
    n, heads = 64, 4
    c = heads * 32
    ca, ct = block_case(1200, n, heads), tm_block_case(1201, n, c, c)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    z0 = dev(ca["z"])
    z = z0.clone()
    mask = dev(ca["mask"])
    tm = capi.TriangleMultiplicationBlock(z, mask, {k: dev(v) for k, v in ct.items() if k not in ("z", "mask")}, False)
    ta = capi.TriangleAttentionBlock(z, mask, dev(ca["gamma"]), dev(ca["beta"]), dev(ca["bias_w"]), dev(ca["wq"]), dev(ca["wk"]),
                                     dev(ca["wv"]), dev(ca["wg"]), dev(ca["bg"]), dev(ca["wo"]), dev(ca["bo"]), heads, True)
    rng = np.random.Generator(np.random.PCG64(5))
    w1 = dev(round_to_bf16((rng.standard_normal((4 * c, c)) / math.sqrt(c)).astype(np.float32)))
    w2 = dev(round_to_bf16((rng.standard_normal((c, 4 * c)) / math.sqrt(4 * c)).astype(np.float32)))
    b1, b2 = dev((rng.standard_normal(4 * c) * 0.1).astype(np.float32)), dev((rng.standard_normal(c) * 0.1).astype(np.float32))
    gam, bet = dev(ca["gamma"]), dev(ca["beta"])
    L = capi.lib()

    def blocks(stream_ptr):
        assert tm.run(stream_ptr) == 0
        assert ta.run(stream_ptr) == 0
        assert L.kutacc_hip_transition_block(z.data_ptr(), gam.data_ptr(), bet.data_ptr(), 1e-5, w1.data_ptr(), b1.data_ptr(),
                                             w2.data_ptr(), b2.data_ptr(), None, 0, n * n, c, 4 * c, capi.K_BF16, stream_ptr) == 0

    blocks(None)  # eager, also takes every first-call set-up (kernel attributes) out of the capture
    torch.cuda.synchronize()
    want = z.clone()
    assert not helpers.same_bits(want, z0)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    z.copy_(z0)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        blocks(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        z.copy_(z0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert helpers.same_bits(z, want)


@pytest.mark.parametrize("column,n_seq,n_res,heads", [(True, 1088, 24, 8), (False, 20, 1040, 8), (False, 24, 56, 3), (True, 40, 24, 5)])
def test_msa_attention_blocks_on_the_tiled_route(torch_cuda, column, n_seq, n_res, heads):
    """Attention rows of more than 1024 keys (column-wise over 1088 sequences, row-wise over 1040 residues) and channel
    counts other than 128 and 256: the attention that keeps q, k, v and gate in memory for the former, the block's separate passes with
    the operator on the tiled MFMA route for the latter; whole result against the oracle's composition."""
    torch = torch_cuda
    c = msa_case(9300 + n_seq + n_res, n_seq, n_res, heads, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = None if column else {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]),
                                "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    blk = capi.MsaAttentionBlock(msa, dev(c["mask"]), w, heads, pair)
    res = {}
    names = profiled_kernels(torch, lambda: res.setdefault("rc", blk.run()))
    torch.cuda.synchronize()
    assert res["rc"] == 0 and ("streamed_attention_kernel" if heads == 8 else "attention_tiles_kernel") in names, (res, names)
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, column), "bf16", f"msa block {n_seq}x{n_res} heads={heads} column={column}")


@pytest.mark.parametrize("column,n_seq,n_res,heads", [(True, 100, 7, 8), (False, 5, 70, 8), (False, 6, 64, 4), (True, 257, 3, 4), (True, 32, 1, 8)])
def test_msa_attention_blocks_on_the_streamed_kernels(torch_cuda, streamed_everywhere, column, n_seq, n_res, heads):
    torch = torch_cuda
    c = msa_case(9500 + n_seq + n_res, n_seq, n_res, heads, 128)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
        device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
    msa = dev(c["m"])
    w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
    pair = None if column else {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]),
                                "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
    print(f"streamed msa {n_seq}x{n_res} heads={heads} column={column}", flush=True)
    assert capi.MsaAttentionBlock(msa, dev(c["mask"]), w, heads, pair).run() == 0
    torch.cuda.synchronize()
    helpers.check_close(helpers.to_numpy(msa), msa_oracle(c, column), "bf16", f"streamed msa block {n_seq}x{n_res} heads={heads} column={column}")


def test_msa_attention_blocks_full_size_sampled_rows(torch_cuda):
    """The MSA shapes the blocks are benchmarked at -- row-wise with pair bias at 512 sequences x 256 residues, column-wise
    at 1024 sequences x 384 residues -- against the oracle on a sample of attention rows (sequences for the row-wise
    form, residues for the column-wise one), every other entry checked for finiteness."""
    from oracle import oracle
    torch = torch_cuda
    for column, n_seq, n_res in ((False, 512, 256), (True, 1024, 384)):
        c = msa_case(8000 + n_seq, n_seq, n_res, 8, 128)
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(  # noqa: E731
            device="cuda", dtype=torch.bfloat16 if a.ndim >= 2 else torch.float32)
        msa = dev(c["m"])
        w = {k: dev(c[k]) for k in ("ln_gamma", "ln_beta", "wq", "wk", "wv", "wg", "bg", "wo", "bo")}
        pair = None if column else {"pair_act": dev(c["z"]), "pair_ln_gamma": dev(c["pair_ln_gamma"]),
                                    "pair_ln_beta": dev(c["pair_ln_beta"]), "bias_w": dev(c["bias_w"])}
        blk = capi.MsaAttentionBlock(msa, dev(c["mask"]), w, 8, pair)
        rc = blk.run()
        torch.cuda.synchronize()
        assert rc == 0, rc
        assert bool(torch.isfinite(msa).all())
        m, mask = (c["m"].transpose(1, 0, 2), c["mask"].T) if column else (c["m"], c["mask"])
        B = m.shape[0]
        rows = sorted({0, 1, 7, 8, 9, B // 2, B - 10, B - 9, B - 8, B - 3, B - 2, B - 1})
        ch = m.shape[-1]
        mn = oracle.layernorm_rows_f32(np.ascontiguousarray(m[rows]).reshape(-1, ch), c["ln_gamma"], c["ln_beta"], 1e-5)
        mn = mn.reshape(len(rows), -1, ch)
        nb = None
        if not column:
            cz = c["z"].shape[-1]
            zn = oracle.layernorm_rows_f32(c["z"].reshape(-1, cz), c["pair_ln_gamma"], c["pair_ln_beta"], 1e-5)
            nb = np.ascontiguousarray(oracle.linear_f32(zn, c["bias_w"]).reshape(n_res, n_res, 8).transpose(2, 0, 1))
        bias = (np.ascontiguousarray(mask[rows]) * np.float32(1e9) - np.float32(1e9)).astype(np.float32)
        out = oracle.gating_attention_f32(mn, c["wq"], c["wk"], c["wv"], c["wg"], c["bg"], c["wo"], c["bo"], bias, nb, 8)
        want = m[rows] + out
        sample = msa[:, rows].transpose(0, 1) if column else msa[rows]
        helpers.check_close(helpers.to_numpy(sample.contiguous()), want, "bf16",
                            f"msa block {n_seq}x{n_res} column={column}, sampled rows")
