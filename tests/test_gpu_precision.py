"""What is computed in 32 bits stays so: calls whose inputs make one operand's rounding the largest error by far, against float64 on
the same bf16 inputs.  A value rounded to bf16 is off by at most 2^-8 of itself, and in the root mean square over values of any
leading digit by 2^-7 / sqrt(12) * sqrt(0.375 / ln 2) = 0.17 %; a result behind n such roundings, each independent, by 0.17 % sqrt(n).
The bars leave a quarter above that."""
import numpy as np
import pytest

import helpers
from kutacc_amd import capi
from kutacc_amd.workloads import MASK_BIAS, round_to_bf16
from test_gpu_tiled_attention import draw_workload

pytestmark = pytest.mark.gpu

BF16_RMS = 2.0 ** -7 / 12 ** 0.5 * (0.375 / np.log(2.0)) ** 0.5


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "these tests need the GPU"
    capi.set_stream(None)
    capi.set_blocking(True)
    return torch


def gated_average_f64(w):
    """softmax(q.k^T / sqrt(d) + bias + nb) . v * sigmoid(gate) of a workload, [B, S, C]."""
    f = lambda a: np.asarray(a, dtype=np.float64)  # noqa: E731
    heads = lambda m: (f(w.x) @ f(m).T).reshape(w.B, w.S, w.H, w.d).transpose(0, 2, 1, 3)  # noqa: E731
    x = heads(w.wq) @ heads(w.wk).transpose(0, 1, 3, 2) / w.d ** 0.5 + f(w.bias)[:, None, None, :]
    x = x + (f(w.nb)[None] if w.nb is not None else 0.0)
    p = np.exp(x - x.max(axis=-1, keepdims=True))
    avg = (p / p.sum(axis=-1, keepdims=True)) @ heads(w.wv)
    return avg.transpose(0, 2, 1, 3).reshape(w.B, w.S, w.C) / (1.0 + np.exp(-(f(w.x) @ f(w.wg).T + f(w.bg))))


def relative_error(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


@pytest.mark.parametrize("B,S,H", [
    (135, 135, 4),  # three rows a workgroup, one at a time
    (140, 33, 4), (190, 80, 4), (130, 97, 4), (128, 128, 4),  # short rows, a workgroup per row and head
    (70, 100, 8), (96, 256, 8),  # 256 channels, three rows a workgroup
    (128, 160, 4),  # two rows, together
])
def test_pair_bias_keeps_32_bits(torch_cuda, B, S, H):
    """A pair bias around 50, whose bf16 steps are a quarter: times log2(e) in 11 bits the probabilities would be off by 1.2 %.  Two
    queries sit at 200 and -200, where the softmax is repeated with the row maxima subtracted, and some keys are masked."""
    w = draw_workload(40 + B + S, B, S, H, 32, masked=0.05)
    w.nb = w.nb * np.float32(0.5) + np.float32(50.0)
    w.nb[:, S // 2, :] += np.float32(150.0)
    w.nb[:, S - 1, :] -= np.float32(250.0)
    w.nb = round_to_bf16(w.nb)
    print(f"B={B} S={S} H={H}", flush=True)
    ten, scratch = helpers.to_device(w)
    assert helpers.run_hip(w, ten, scratch) == 0 and capi.last_path() == "fused_mfma"
    err = relative_error(helpers.to_numpy(scratch["avg"]).reshape(B, S, -1), gated_average_f64(w))
    # q, k, v, probabilities, gate and result are rounded; q and k move a logit by 0.002 of its size, which is about one
    assert err < 1.25 * 6 ** 0.5 * BF16_RMS, err


@pytest.mark.parametrize("heads", [4, 8])
def test_gate_of_long_rows_keeps_32_bits(torch_cuda, heads):
    """Column-wise MSA attention over 1030 sequences of zeros: every normalised row is the LayerNorm's beta, a unit vector, every
    probability is one, the values are the first column of the value weights, the output projection is the identity.  What is
    left is bf16(v * sigmoid(gate)), one rounding of at most 2^-8."""
    torch = torch_cuda
    C, n_seq, n_res = 32 * heads, 1030, 2
    g = torch.Generator(device="cuda").manual_seed(heads)
    zeros = torch.zeros(C, C, device="cuda", dtype=torch.bfloat16)
    v = (torch.rand(C, device="cuda", generator=g) + 0.5).to(torch.bfloat16)
    gate = (2.0 * torch.randn(C, device="cuda", generator=g)).to(torch.bfloat16).float()
    wv, beta = zeros.clone(), torch.zeros(C, device="cuda")
    wv[:, 0], beta[0] = v, 1.0
    w = dict(ln_gamma=torch.ones(C, device="cuda"), ln_beta=beta, wq=zeros, wk=zeros, wv=wv, wg=zeros, bg=gate,
             wo=torch.eye(C, device="cuda").to(torch.bfloat16), bo=torch.zeros(C, device="cuda"))
    act = torch.zeros(n_seq, n_res, C, device="cuda", dtype=torch.bfloat16)
    assert capi.MsaAttentionBlock(act, torch.ones(n_seq, n_res, device="cuda", dtype=torch.bfloat16), w, heads).run() == 0
    torch.cuda.synchronize()
    want = v.double() * torch.sigmoid(gate.double())
    err = float(((act.double() - want).abs() / want).max())
    assert err < 2.0 ** -8 * (1 + 2.0 ** -7), err  # 2^-15: what 32-bit sums, sigmoid and quotient add, and to spare


def halves_to_the_nearest_even(kept):
    """Averages of `kept` values, half of them 1 and half 1 + 2^-7, or 1 + 2^-7 and 1 + 2^-6: halfway between two bf16.  As the sum (exact)
    times the rounded reciprocal of the sum of the probabilities gives them, [low, high][row]."""
    n = np.asarray(kept, dtype=np.float32)
    inv = np.float32(1.0) / n
    return [round_to_bf16(n * np.float32(1.0 + k / 256.0) * inv) for k in (1, 3)]


@pytest.mark.parametrize("heads,n_seq,n_res,column", [
    (4, 1030, 512, True), (8, 1030, 512, True), (8, 400, 300, True),  # two blocks of queries a wave
    (8, 24, 1030, False), (8, 64, 1030, False), (4, 128, 1030, False),  # two rows a wave, four
])
def test_sums_of_long_rows_keep_32_bits(torch_cuda, heads, n_seq, n_res, column):
    """Every probability is one, every average halfway between two bf16: one unit of 32 bits more or less in 1 / sum, as a hardware
    reciprocal has it, is a bf16 more or less.  Normalised rows are 1, -1, s, -s over and over, s the parity of the key."""
    torch = torch_cuda
    C, keys, rows = 32 * heads, n_seq if column else n_res, n_res if column else n_seq
    kept = np.minimum(2 * (1 + np.arange(rows)), keys // 2 * 2)
    zeros = torch.zeros(C, C, device="cuda", dtype=torch.bfloat16)
    wv = zeros.clone()
    wv[:, 0], wv[:, 2], wv[:, 4] = 1.0, 2.0 ** -8, 2.0 ** -8
    wv[C // 2:, 4] = 3.0 * 2.0 ** -8
    w = dict(ln_gamma=torch.ones(C, device="cuda"), ln_beta=torch.zeros(C, device="cuda"), wq=zeros, wk=zeros, wv=wv, wg=zeros,
             bg=torch.full((C,), 100.0, device="cuda"), wo=torch.eye(C, device="cuda").to(torch.bfloat16), bo=torch.zeros(C, device="cuda"))
    parity = 1.0 - 2.0 * (torch.arange(keys, device="cuda") % 2)
    x = torch.ones(keys, C // 4, 4, device="cuda")
    x[:, :, 1], x[:, :, 2], x[:, :, 3] = -1.0, parity[:, None], -parity[:, None]
    there = torch.arange(keys, device="cuda")[None, :] < torch.from_numpy(kept).to("cuda")[:, None]
    act = x.reshape(1, keys, C).expand(rows, keys, C).to(torch.bfloat16)
    if column:
        act, there = act.transpose(0, 1), there.transpose(0, 1)
    act, mask, pair = act.contiguous(), there.to(torch.bfloat16).contiguous(), None
    if not column:
        pair = dict(pair_act=torch.zeros(keys, keys, 128, device="cuda", dtype=torch.bfloat16), pair_ln_gamma=torch.ones(128, device="cuda"),
                    pair_ln_beta=torch.zeros(128, device="cuda"), bias_w=torch.zeros(heads, 128, device="cuda", dtype=torch.bfloat16))
    print(f"heads={heads} n_seq={n_seq} n_res={n_res} column={column}", flush=True)
    assert capi.MsaAttentionBlock(act, mask, w, heads, pair).run() == 0
    torch.cuda.synchronize()
    got = helpers.to_numpy(act.transpose(0, 1) if column else act)[:, :, 1::4] + 1.0  # channels of -1: the sum with the average is exact
    for half, want in enumerate(halves_to_the_nearest_even(kept)):
        wrong = (got[:, :, half * C // 8:(half + 1) * C // 8] != want[:, None, None]).any(axis=(1, 2))
        assert not wrong.any(), (half, kept[wrong])


@pytest.mark.parametrize("heads,n_seq,n_res,column", [(4, 1030, 3, True), (8, 300, 300, True), (8, 24, 1030, False)])
def test_small_gates_of_long_rows_beside_large_sums(torch_cuda, heads, n_seq, n_res, column):
    """Logits of 45 on all keys, sums of 2^75, and gates of -45: the average times 3e-20, which the output weights take back to 0.5.
    Every fourth gate is -100, whose sigmoid is no normal number: no update."""
    torch = torch_cuda
    C, keys = 32 * heads, n_seq if column else n_res
    wq = torch.zeros(C, C, device="cuda", dtype=torch.bfloat16)
    wq[::32, 0] = 16.0
    wv = torch.zeros(C, C, device="cuda", dtype=torch.bfloat16)
    wv[:, 0] = 1.0
    bg = torch.full((C,), -45.0, device="cuda")
    bg[3::4] = -100.0
    w = dict(ln_gamma=torch.ones(C, device="cuda"), ln_beta=torch.zeros(C, device="cuda"), wq=wq, wk=wq, wv=wv, wg=torch.zeros_like(wv),
             bg=bg, wo=(torch.eye(C, device="cuda") * 2.0 ** 64).to(torch.bfloat16), bo=torch.zeros(C, device="cuda"))
    x = torch.ones(n_seq, n_res, C, device="cuda", dtype=torch.bfloat16)
    x[:, :, 1::2] = -1.0
    act, pair = x.clone(), None
    if not column:
        pair = dict(pair_act=torch.zeros(keys, keys, 128, device="cuda", dtype=torch.bfloat16), pair_ln_gamma=torch.ones(128, device="cuda"),
                    pair_ln_beta=torch.zeros(128, device="cuda"), bias_w=torch.zeros(heads, 128, device="cuda", dtype=torch.bfloat16))
    print(f"heads={heads} n_seq={n_seq} n_res={n_res} column={column}", flush=True)
    assert capi.MsaAttentionBlock(act, torch.ones(n_seq, n_res, device="cuda", dtype=torch.bfloat16), w, heads, pair).run() == 0
    torch.cuda.synchronize()
    update = 2.0 ** 64 * torch.sigmoid(bg.double())
    err = float(((act.double() - (x.double() + update)).abs() / (1.0 + 2.0 * update)).max())
    assert err < 2.0 ** -8, err  # the update and the sum, each rounded once to bf16


def run_heads_of_eight(w):
    print(w.name, flush=True)
    ten, scratch = helpers.to_device(w)
    assert helpers.run_hip(w, ten, scratch) == 0 and capi.last_path() == "tiled_mfma"
    err = relative_error(helpers.to_numpy(scratch["avg"]).reshape(w.B, w.S, w.C), gated_average_f64(w))
    # q, k, v, probabilities, gate, weighted average and result are rounded
    assert err < 1.25 * 7 ** 0.5 * BF16_RMS, err


@pytest.mark.parametrize("S", [33, 128, 301])
def test_queries_of_heads_of_eight_keep_32_bits(torch_cuda, S):
    """The first channel of every query is 127, that of the keys a whole number below 256: logits of up to 11 000, which the pair bias and
    the mask together take back to within 0.1, leaving those of the other seven channels.  127 log2(e) / sqrt(8) in 16 bits is off
    by enough to move a probability by up to 8 %."""
    w = draw_workload(700 + S, 5, S, 8, 8, masked=0.0)
    c = np.random.Generator(np.random.PCG64(S)).integers(1, 256, S).astype(np.float32)
    for m in (w.wq, w.wk, w.wv, w.wg):
        m[:, :2] = 0.0
    w.wq[::8], w.wk[::8] = 0.0, 0.0
    w.wq[::8, 0], w.wk[::8, 1] = 1.0, 1.0
    w.x[:, :, 0], w.x[:, :, 1] = 127.0, c
    logit = 127.0 * c.astype(np.float64) / 8.0 ** 0.5
    nb = round_to_bf16(-logit.astype(np.float32))
    w.nb[:], w.bias[:] = nb, round_to_bf16((-logit - nb).astype(np.float32))
    run_heads_of_eight(w)


@pytest.mark.parametrize("S", [33, 128, 301])
def test_masks_of_heads_of_eight_keep_32_bits(torch_cuda, S):
    """Mask biases of up to 4000 on all keys, one set for all rows, which the pair bias takes back: the softmax of the logits alone."""
    w = draw_workload(800 + S, 5, S, 8, 8, masked=0.0)
    w.bias[:] = round_to_bf16(np.random.Generator(np.random.PCG64(S)).uniform(-4000.0, 4000.0, S).astype(np.float32))
    w.nb[:] = -w.bias[0]
    run_heads_of_eight(w)


def test_sums_of_heads_of_eight_keep_32_bits(torch_cuda):
    """As for the long rows: averages halfway between two bf16, 200 rows of 2 .. 400 keys.  The fourth gate of every head is -100: zero."""
    B, S = 200, 401
    w = draw_workload(900, B, S, 8, 8, masked=0.0)
    kept = 2 * (1 + np.arange(B))
    for m in (w.wq, w.wk, w.wv, w.wg):
        m[:] = 0.0
    w.x[:, :, 0], w.x[:, :, 1] = 1.0, 1.0 - 2.0 * (np.arange(S) % 2)
    w.wv[:, 0], w.wv[:, 1] = 1.0 + 2.0 ** -7, 2.0 ** -8
    w.x[:, :, 2], w.wv[:32, 2], w.wv[32:, 2] = 1.0, -(2.0 ** -8), 2.0 ** -8
    w.bg[:], w.bg[3::8], w.nb[:] = 100.0, -100.0, 0.0
    w.bias[:] = np.where(np.arange(S)[None, :] < kept[:, None], np.float32(0.0), round_to_bf16(np.full(1, MASK_BIAS, dtype=np.float32)))
    ten, scratch = helpers.to_device(w)
    assert helpers.run_hip(w, ten, scratch) == 0 and capi.last_path() == "tiled_mfma"
    got = helpers.to_numpy(scratch["avg"])
    assert not got[:, :, :, 3].any()
    for half, want in enumerate(halves_to_the_nearest_even(kept)):
        wrong = (got[:, :, 4 * half:4 * half + 4, [0, 1, 2, 4, 5, 6, 7]] != want[:, None, None, None]).any(axis=(1, 2, 3))
        assert not wrong.any(), (half, kept[wrong])


def test_centre_layernorm_of_the_triangle_multiplication_is_exact_to_32_bits(torch_cuda):
    """One residue whose normalised row is the input LayerNorm's beta, small whole numbers, as are then the left projections and, with
    ones to the right, the centre: its sums are exact, and gamma = 2^20 with beta = -2^20 t, t the centre normalised in 32 bits
    with a correctly rounded square root and quotient, leaves zeros, where one bit more or less would leave 1/16."""
    torch = torch_cuda
    C, f = 128, np.float32
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda")  # noqa: E731
    vec = lambda value: torch.full((C,), float(value), device="cuda")  # noqa: E731
    eye, zeros = torch.eye(C, device="cuda").to(torch.bfloat16), torch.zeros(C, C, device="cuda", dtype=torch.bfloat16)
    for seed in range(24):
        row = np.random.Generator(np.random.PCG64(seed)).integers(-9, 10, C).astype(f)
        mean, var = f(row.mean(dtype=np.float64)), f(row.var(dtype=np.float64))
        rstd = f(1) / np.sqrt(var + f(1e-5))
        t = (row.astype(np.float64) * rstd + (-rstd * mean)).astype(f)
        w = dict(ln_in_gamma=vec(0), ln_in_beta=dev(row), ln_center_gamma=vec(2.0 ** 20), ln_center_beta=dev(-t * f(2.0 ** 20)),
                 left_proj_w=eye, left_proj_b=vec(0), right_proj_w=zeros, right_proj_b=vec(1), output_w=eye, output_b=vec(0),
                 left_gate_w=zeros, right_gate_w=zeros, gating_w=zeros, left_gate_b=vec(100), right_gate_b=vec(100), gating_b=vec(100))
        act = torch.zeros(1, 1, C, device="cuda", dtype=torch.bfloat16)
        assert capi.TriangleMultiplicationBlock(act, torch.ones(1, 1, device="cuda", dtype=torch.bfloat16), w, False).run() == 0
        torch.cuda.synchronize()
        assert not bool(act.any()), (seed, float(act.abs().max()))


@pytest.mark.parametrize("B,S,H", [(130, 97, 4), (135, 135, 4), (70, 100, 8)])
def test_infinite_pair_bias_and_masked_rows_on_fp32_tiles(torch_cuda, B, S, H):
    """The single-row kernels that read the pair bias as fp32 tiles: pairs excluded by -inf, a row with every key masked, a query whose
    logits leave the range of the unshifted softmax."""
    w = draw_workload(60 + B, B, S, H, 32)
    drop = np.random.Generator(np.random.PCG64(B)).random(w.nb.shape) < 0.3
    drop[:, :, 0] = False
    w.nb[:, S // 2, :] += np.float32(150.0)
    w.nb = round_to_bf16(w.nb)
    w.nb[drop] = -np.inf
    w.bias[B // 2, :] = round_to_bf16(np.full(S, MASK_BIAS, dtype=np.float32))
    print(f"B={B} S={S} H={H}", flush=True)
    ten, scratch = helpers.to_device(w)
    assert helpers.run_hip(w, ten, scratch) == 0 and capi.last_path() == "fused_mfma"
    ref_out, ref_avg = helpers.oracle_out(w, return_avg=True)
    helpers.check_close(helpers.to_numpy(scratch["avg"]).reshape(B, S, -1), ref_avg, "bf16", "gated average")
    helpers.check_close(helpers.to_numpy(ten["out"]), ref_out, "bf16", "out")
