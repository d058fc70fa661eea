"""The tiled MFMA route of the gated-attention operator (kutacc_amd/csrc/tiled_attention.hip): the bf16 shapes the fused
head kernels do not take -- rows longer than 1024 positions, head sizes other than 32, channel counts other than 128 and
256 -- against the fp32 oracle, to the bf16 bar (2e-2 absolute + 1e-2 relative); the scratch tensors it leaves against
the oracle's bf16 model of the reference (reference src/attention/gating_attention.cpp:47-66)."""
import ctypes

import numpy as np
import pytest

import helpers
from kutacc_amd import capi
from kutacc_amd.workloads import MASK_BIAS, Workload, layernorm_np, make_workload, round_to_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    assert torch.cuda.is_available(), "these tests need the GPU"
    capi.set_stream(None)
    capi.set_blocking(True)
    return torch


def draw_workload(seed, B, S, H, d, pair_bias=True, masked=0.1, nb_scale=1.0) -> Workload:
    """A seeded problem of any head size: layer-normalised input rows, weights of variance 1 / fan_in, a key mask on
    about `masked` of the positions (never the first), a pair bias of standard deviation `nb_scale`."""
    rng = np.random.Generator(np.random.PCG64(seed))
    C = H * d
    x = round_to_bf16(layernorm_np(round_to_bf16(rng.standard_normal((B, S, C), dtype=np.float32))))
    weight = lambda: round_to_bf16(rng.standard_normal((C, C), dtype=np.float32) / np.float32(np.sqrt(C)))  # noqa: E731
    wq, wk, wv, wg, wo = (weight() for _ in range(5))
    bg = np.ones(C, dtype=np.float32) + 0.1 * rng.standard_normal(C, dtype=np.float32)
    bo = 0.1 * rng.standard_normal(C, dtype=np.float32)
    keep = rng.random((B, S)) >= masked
    keep[:, 0] = True
    bias = round_to_bf16((MASK_BIAS * (1.0 - keep.astype(np.float32))))
    nb = round_to_bf16(nb_scale * rng.standard_normal((H, S, S), dtype=np.float32)) if pair_bias else None
    return Workload(0, f"drawn B={B} S={S} H={H} d={d}", "bf16", B, S, H, d, x, wq, wk, wv, wg, wo, bg, bo, bias, nb)


def run_and_check(w, path=capi.PATH_AUTO, expect="tiled_mfma"):
    print(f"{w.name} path={path}", flush=True)
    ten, scratch = helpers.to_device(w)
    rc = helpers.run_hip(w, ten, scratch, path)
    assert rc == 0 and capi.last_path() == expect, (rc, capi.last_path())
    ref_out, ref_avg = helpers.oracle_out(w, return_avg=True)
    helpers.check_close(helpers.to_numpy(scratch["avg"]).reshape(w.B, w.S, w.C), ref_avg, "bf16", "gated average")
    helpers.check_close(helpers.to_numpy(ten["out"]), ref_out, "bf16", "out")
    return ten, scratch


@pytest.mark.parametrize("B,S,H,d", [
    (3, 200, 8, 8),    # the extra-MSA shape: 64 channels, head size 8 (one k-step, half of it padding)
    (2, 150, 4, 16),   # the template stack's: head size 16
    (2, 96, 3, 24),    # two k-steps, the second half padding; 72 channels
    (1, 70, 3, 40),    # three k-steps, two blocks of values
    (2, 100, 2, 64),   # four k-steps
    (2, 130, 4, 32),   # a shape the fused kernels take as well, forced onto this route
    (9, 64, 2, 32),    # one whole chunk of keys; nine batch rows: a second group of rows with one member
    (2, 65, 2, 32),    # one key into the second chunk
    (1, 1, 2, 32),     # a single position
    (2, 77, 8, 8),     # a length that is no multiple of 8: the rows of v and of the pair bias are read element by element
    (3, 1000, 5, 16),  # eight query blocks, sixteen chunks, 80 channels
])
def test_shapes_beyond_the_fused_kernels(torch_cuda, B, S, H, d):
    w = draw_workload(100 * d + S, B, S, H, d)
    run_and_check(w, capi.PATH_TILED)
    if d != 32 or H * d not in (128, 256):
        run_and_check(w, capi.PATH_AUTO)   # the automatic choice comes here too ...
        run_and_check(w, capi.PATH_FUSED)  # ... and "MFMA kernels only" includes this route


@pytest.mark.parametrize("B,S,H,d", [(2, 1536, 4, 32), (9, 1100, 4, 32), (1, 2048, 8, 8)])
def test_rows_longer_than_1024_positions(torch_cuda, B, S, H, d):
    """Twelve, nine and sixteen query blocks (a second group of query blocks), 24 / 18 / 32 key chunks; the first two are
    triangle-attention shapes past the fused kernels' longest row."""
    w = draw_workload(7 + S, B, S, H, d)
    run_and_check(w, capi.PATH_AUTO)


@pytest.mark.parametrize("B,S,H,d", [(2048, 2048, 4, 32), (5120, 384, 8, 8)])
def test_benchmarked_shapes_on_sampled_rows(torch_cuda, B, S, H, d):
    """The shapes `bench.py --tiled-route` times (triangle attention at 2048 residues, the extra-MSA row attention), drawn
    on the device: the oracle on a sample of batch rows -- first and last, both sides of the 8-row groups the kernel's
    placement forms, one fully masked -- and finiteness of every other entry."""
    import ctypes
    torch = torch_cuda
    C = H * d
    g = torch.Generator(device="cuda").manual_seed(4000 + S)
    bf = lambda *sh, scale=1.0: (torch.randn(*sh, device="cuda", generator=g) * scale).to(torch.bfloat16)  # noqa: E731
    x = torch.nn.functional.layer_norm(torch.randn(B, S, C, device="cuda", generator=g), (C,)).to(torch.bfloat16)
    ws = [bf(C, C, scale=C ** -0.5) for _ in range(5)]
    bg, bo = torch.ones(C, device="cuda"), torch.randn(C, device="cuda", generator=g) * 0.1
    keep = torch.rand(B, S, device="cuda", generator=g) >= 0.1
    keep[:, 0] = True
    bias = ((~keep).float() * MASK_BIAS).to(torch.bfloat16)
    rows = sorted({0, 1, 7, 8, 9, B // 2 - 1, B // 2, B - 9, B - 8, B - 2, B - 1})
    bias[rows[3], :] = MASK_BIAS  # a fully masked row: a uniform average
    nb = bf(H, S, S)
    out = torch.empty(B, S, C, device="cuda", dtype=torch.bfloat16)
    q, k, gate, avg = (torch.empty(B, S, C, device="cuda", dtype=torch.bfloat16) for _ in range(4))
    v = torch.empty(C, B * S, device="cuda", dtype=torch.bfloat16)
    a = capi.HipAttentionArgs()
    a.batch, a.seq_len, a.nheads, a.head_size, a.dtype, a.path = B, S, H, d, capi.K_BF16, capi.PATH_AUTO
    a.input, a.input_ld = x.data_ptr(), C
    a.query_w, a.key_w, a.value_w, a.gating_w, a.output_w = (w.data_ptr() for w in ws)
    a.gating_b, a.output_b = bg.data_ptr(), bo.data_ptr()
    a.bias, a.bias_stride_b = bias.data_ptr(), S
    a.nonbatched_bias, a.nb_stride_h, a.nb_stride_q = nb.data_ptr(), S * S, S
    a.q, a.k, a.v, a.gate, a.avg = q.data_ptr(), k.data_ptr(), v.data_ptr(), gate.data_ptr(), avg.data_ptr()
    for n in ("q", "k", "gate", "avg"):
        setattr(a, f"{n}_stride_b", S * C), setattr(a, f"{n}_stride_s", C), setattr(a, f"{n}_stride_h", d)
    a.v_stride_h, a.v_stride_e, a.v_stride_b = d * B * S, B * S, S
    a.out, a.out_ld = out.data_ptr(), C
    print(f"B={B} S={S} H={H} d={d}", flush=True)
    assert capi.lib().kutacc_hip_gating_attention(ctypes.byref(a), None) == 0
    torch.cuda.synchronize()
    assert capi.last_path() == "tiled_mfma"
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(avg).all())
    from oracle import oracle
    num = lambda t: helpers.to_numpy(t)  # noqa: E731
    ref_out, ref_avg = oracle.gating_attention_f32(num(x[rows]), *(num(w) for w in ws[:4]), num(bg), num(ws[4]), num(bo),
                                                   num(bias[rows]), num(nb), H, return_avg=True)
    helpers.check_close(num(avg[rows]), ref_avg, "bf16", f"gated average, sampled rows of B={B} S={S}")
    helpers.check_close(num(out[rows]), ref_out, "bf16", f"out, sampled rows of B={B} S={S}")


def test_without_pair_bias_and_with_fully_masked_rows(torch_cuda):
    w = draw_workload(5, 4, 300, 8, 8, pair_bias=False)
    w.bias[1, :] = round_to_bf16(np.full(w.S, MASK_BIAS, dtype=np.float32))  # every key of row 1 masked: a uniform average
    run_and_check(w)
    w = draw_workload(6, 3, 1200, 4, 32, pair_bias=True, masked=0.5)
    w.bias[2, :] = round_to_bf16(np.full(w.S, MASK_BIAS, dtype=np.float32))
    run_and_check(w)


def test_large_pair_bias_and_logit_offsets(torch_cuda):
    """A pair bias of standard deviation 10 (what a trained pair representation reaches) and rows whose logits sit
    150 above or below zero: the running maximum absorbs both."""
    w = draw_workload(8, 3, 260, 4, 16, nb_scale=10.0)
    w.nb[:, 5, :] += np.float32(150.0)
    w.nb[:, 9, :] -= np.float32(150.0)
    w.nb = round_to_bf16(w.nb)
    run_and_check(w)


@pytest.mark.parametrize("B,S", [(1, 1), (2, 7), (4, 32), (5, 33), (3, 128), (9, 130), (4, 385), (1, 1120), (2, 1121)])
@pytest.mark.parametrize("pair_bias", [True, False])
def test_heads_of_eight_at_tile_edges(torch_cuda, B, S, pair_bias):
    """One position, less than one piece of eight, whole blocks of 32 and one key past them, four to eight waves, sets of
    four batch rows with one to four members, the longest row whose keys lie in the LDS and the first past it; keys masked
    from a late tile on, a fully masked row, and queries whose logits leave the range of the unshifted softmax."""
    w = draw_workload(60 + S, B, S, 8, 8, pair_bias=pair_bias, masked=0.0)
    w.bias[B // 2, max(1, 2 * S // 3):] = MASK_BIAS
    w.bias[B - 1, :] = MASK_BIAS if B > 1 else 0.0
    if pair_bias:
        w.nb[:, S // 2, :] += np.float32(150.0)
        w.nb[:, S - 1, :] -= np.float32(150.0)
        w.nb = round_to_bf16(w.nb)
    w.bias = round_to_bf16(w.bias)
    names = helpers.profiled_kernels(torch_cuda, lambda: run_and_check(w))
    assert ("small_head_attention_kernel" if S <= 1120 else "attention_tiles_kernel") in names, names


@pytest.mark.parametrize("B,S", [(1, 9), (2, 63), (3, 64), (4, 65), (5, 97), (6, 193)])
def test_heads_of_eight_stage_their_keys_in_units_of_64(torch_cuda, B, S):
    """Units whole, short of a key and with one, half units behind an odd number of tiles, fewer waves than rows, and the last eight keys
    of a row read in one piece."""
    test_heads_of_eight_at_tile_edges(torch_cuda, B, S, True)


# sets of four rows, whole and with one to three; one tile and several, ragged and not, a wave with one tile, two and three, eight waves; rows and averages
# with a pitch.  projects: whether the kernel forms the projections itself: no where the scratch does not hold its queries and gates (5 rows of
# 64, rows of 40), is not dense, or the average or the input lies where the other of the two or a scratch tensor does
@pytest.mark.parametrize("B,S,form,projects", [(8, 64, "", True), (65, 48, "", True), (12, 97, "", True), (11, 128, "", True), (33, 150, "", True), (8, 301, "", True),
                                               (12, 385, "", True), (10, 77, "pitch", True), (5, 64, "", False), (40, 40, "", False), (10, 77, "q", False), (10, 77, "k", False),
                                               (10, 77, "in place", False), (65, 96, "avg over q", False), (65, 96, "avg over k", False),
                                               (65, 96, "avg over gate", False), (65, 96, "input over q", False), (65, 96, "input over k", False),
                                               (65, 96, "input over gate", False)])
@pytest.mark.parametrize("pair_bias", [True, False])
def test_heads_of_eight_with_the_projections_inside(torch_cuda, B, S, form, projects, pair_bias):
    """The kernel that projects against the one that reads q, k, v and gate: the same roundings, sums of products in another order."""
    torch = torch_cuda
    w = draw_workload(300 + S, B, S, 8, 8, pair_bias=pair_bias)
    w.bias[B - 1, :] = MASK_BIAS
    w.bias = round_to_bf16(w.bias)
    got = {}
    for path in (capi.PATH_TILED, capi.PATH_AUTO):
        ten, scratch = helpers.to_device(w)
        a = helpers.hip_args(w, ten, scratch, path)
        wide = torch.full((B, S, 72), 7.0, device="cuda", dtype=torch.bfloat16)
        out_wide, avg = wide.clone(), scratch["avg"].view(B, S, 64)
        if form == "pitch":
            wide[..., :64] = ten["x"]
            a.input, a.input_ld = wide.data_ptr(), 72
            a.avg, a.avg_stride_b, a.avg_stride_s, avg = out_wide.data_ptr(), 72 * S, 72, out_wide[..., :64]
        elif form in ("q", "k"):
            setattr(a, form, wide.data_ptr()), setattr(a, form + "_stride_b", 72 * S), setattr(a, form + "_stride_s", 72)
        elif form == "in place":
            a.avg, avg = ten["x"].data_ptr(), ten["x"]
        elif form.startswith("avg over"):
            a.avg, avg = getattr(a, form.split()[2]), scratch[form.split()[2]].view(B, S, 64)
        elif form.startswith("input over"):
            setattr(a, form.split()[2], ten["x"].data_ptr())
        print(f"{w.name} {form} path={path}", flush=True)
        names = helpers.profiled_kernels(torch, lambda: capi.lib().kutacc_hip_gating_attention(ctypes.byref(a), None))  # noqa: B023
        torch.cuda.synchronize()
        assert capi.last_path() == "tiled_mfma" and "small_head_attention_kernel" in names
        assert ("projections_kernel" in names) == (path == capi.PATH_TILED or not projects), names
        assert form != "pitch" or bool((out_wide[..., 64:] == 7.0).all())
        got[path] = (ten["out"].float(), avg.float().clone())
    ref_out, ref_avg = helpers.oracle_out(w, return_avg=True)
    helpers.check_close(helpers.to_numpy(got[capi.PATH_AUTO][0]), ref_out, "bf16", "out")
    helpers.check_close(helpers.to_numpy(got[capi.PATH_AUTO][1]), ref_avg, "bf16", "gated average")
    for x, y in zip(*got.values()):
        # q, k, v and gate are rounded to bf16 on both sides: a sum in another order moves a few of them, and the results with them, by a unit (2^-8)
        assert float((x - y).norm() / y.norm()) <= 2.0 ** -9 and float((x - y).abs().max()) <= 2.0 ** -6 * float(y.abs().max())


@pytest.mark.parametrize("B,S", [(304, 311), (480, 253), (482, 255), (2005, 100), (2003, 97), (1880, 127), (7600, 64), (7599, 63)])
@pytest.mark.parametrize("offset", [0.0, 150.0])
def test_heads_of_eight_with_the_bias_in_the_lanes_order(torch_cuda, B, S, offset):
    """A bias whose rows start on any address, brought into the order of the logits by a pass of its own, against the same bias in rows of 16 bytes,
    which the kernel reads as they lie: the same bits.  Masked keys, a fully masked row, entries of -inf and, with the offset, rows that are repeated."""
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(500 + S)
    bf16 = lambda *shape, scale=1.0: (torch.randn(*shape, device="cuda", generator=g) * scale).to(torch.bfloat16)  # noqa: E731
    x = torch.nn.functional.layer_norm(torch.randn(B, S, 64, device="cuda", generator=g), (64,)).to(torch.bfloat16)
    wq, wk, wv, wg, wo = (bf16(64, 64, scale=0.125) for _ in range(5))
    bg, bo = 1 + 0.1 * torch.randn(64, device="cuda", generator=g), 0.1 * torch.randn(64, device="cuda", generator=g)
    bias = torch.zeros(B, S, device="cuda", dtype=torch.bfloat16)
    bias[:, S - S // 10:] = -1e9
    bias[B // 2, 3:7] = -1e9
    bias[B - 1] = -1e9
    pitch = (S + 7) // 8 * 8 + 8
    wide = torch.zeros(8, S, pitch, device="cuda", dtype=torch.bfloat16)
    wide[..., :S] = bf16(8, S, S) + offset * (torch.arange(S, device="cuda") % 2 * 2 - 1)[None, :, None]
    wide[3, 5, 2] = -float("inf")
    # rows on any address: dense where the length does so, else a pitch of an odd number
    narrow = torch.zeros(8, S, S + 1 if S % 8 == 0 else S, device="cuda", dtype=torch.bfloat16)
    narrow[..., :S] = wide[..., :S]
    got = []
    for nb in (wide[..., :S], narrow[..., :S]):
        out = torch.full_like(x, 7.0)
        scratch = {k: torch.zeros(B, S, 8, 8, device="cuda", dtype=torch.bfloat16) for k in ("q", "k", "gate", "avg")}
        scratch["v"] = torch.zeros(8, 8, B, S, device="cuda", dtype=torch.bfloat16)
        capi.GatedAttention(x, wq, wk, wv, wg, bg, wo, bo, bias, nb, 8, out, scratch).run()
        torch.cuda.synchronize()
        assert not capi.error_flag() and capi.last_path() == "tiled_mfma"
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            # the seeds of the keys past the end lie in the gate tensor: 64-bit pairs of fp32 -inf, which no stash of queries and gates holds
            assert S % 32 in (0, 31) or bool((scratch["gate"].view(torch.int64) == -0x007fffff00800000).any()) == (nb.stride(1) % 8 != 0)
        assert bool((scratch["v"] == 0).all()) and bool(torch.isfinite(out).all())
        got.append((out, scratch["avg"]))
    assert helpers.same_bits(got[0][0], got[1][0]) and helpers.same_bits(got[0][1], got[1][1])


# (the last three: the fewest sets that pay for the pass on 256 CUs, one set less, and no room for it in the gate tensor)
@pytest.mark.parametrize("B,S,passes", [(304, 311, True), (480, 253, True), (482, 255, True), (2005, 100, True), (2003, 97, True), (1880, 127, True),
                                        (7600, 64, True), (7599, 63, True), (300, 301, True), (296, 301, False), (64, 1001, False)])
def test_which_biases_of_heads_of_eight_come_through_the_pass(torch_cuda, B, S, passes):
    """The pass runs, by its name, where the bias's rows start on any address and sets and tiles pay for it; the bits are those of the bias in rows of 16 bytes."""
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(600 + S)
    bf16 = lambda *shape, scale=1.0: (torch.randn(*shape, device="cuda", generator=g) * scale).to(torch.bfloat16)  # noqa: E731
    x = torch.nn.functional.layer_norm(torch.randn(B, S, 64, device="cuda", generator=g), (64,)).to(torch.bfloat16)
    wq, wk, wv, wg, wo = (bf16(64, 64, scale=0.125) for _ in range(5))
    bg, bo = torch.ones(64, device="cuda"), torch.zeros(64, device="cuda")
    bias = torch.zeros(B, S, device="cuda", dtype=torch.bfloat16)
    wide = torch.zeros(8, S, (S + 7) // 8 * 8 + 8, device="cuda", dtype=torch.bfloat16)
    wide[..., :S] = bf16(8, S, S)
    narrow = torch.zeros(8, S, S + 1 if S % 8 == 0 else S, device="cuda", dtype=torch.bfloat16)
    narrow[..., :S] = wide[..., :S]
    got = []
    for nb, unaligned in ((wide[..., :S], False), (narrow[..., :S], True)):
        out = torch.full_like(x, 7.0)
        scratch = {k: torch.zeros(B, S, 8, 8, device="cuda", dtype=torch.bfloat16) for k in ("q", "k", "gate", "avg")}
        scratch["v"] = torch.zeros(8, 8, B, S, device="cuda", dtype=torch.bfloat16)
        names = helpers.profiled_kernels(torch, capi.GatedAttention(x, wq, wk, wv, wg, bg, wo, bo, bias, nb, 8, out, scratch).run)
        torch.cuda.synchronize()
        assert not capi.error_flag() and "small_head_attention_kernel" in names, names
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert ("seed_tiles_kernel" in names) == (passes and unaligned), names
        got.append((out, scratch["avg"]))
    assert helpers.same_bits(got[0][0], got[1][0]) and helpers.same_bits(got[0][1], got[1][1])


def test_pair_bias_entries_of_minus_infinity(torch_cuda):
    """Pairs excluded by a -inf pair bias get zero weight; a row keeps at least one finite key."""
    w = draw_workload(9, 2, 140, 4, 16)
    rng = np.random.Generator(np.random.PCG64(99))
    drop = rng.random(w.nb.shape) < 0.3
    drop[:, :, 0] = False
    w.nb[drop] = -np.inf
    run_and_check(w)


def test_matches_the_fused_kernels_where_both_run(torch_cuda):
    """Config 3 at 384 positions on both routes: each within the bar of the oracle (checked elsewhere), and within the bar
    of each other on every batch row."""
    import torch
    w = make_workload(3, batch=24)
    ten, scratch = helpers.to_device(w)
    assert helpers.run_hip(w, ten, scratch, capi.PATH_TILED) == 0 and capi.last_path() == "tiled_mfma"
    ten2, scratch2 = helpers.to_device(w)
    assert helpers.run_hip(w, ten2, scratch2, capi.PATH_FUSED) == 0 and capi.last_path() == "fused_mfma"
    a, b = ten["out"].float(), ten2["out"].float()
    assert bool(torch.isfinite(a).all())
    assert float(((a - b).abs() - (2e-2 + 1e-2 * b.abs())).max()) <= 0.0


def test_leaves_q_k_v_gate_as_the_reference_does(torch_cuda):
    """q, k, gate as [B, S, H, d] and v as [H, d, B, S], rounded to bf16 where the reference stores them; the oracle's bf16
    model of the reference holds the same tensors."""
    from oracle import oracle
    w = draw_workload(11, 3, 90, 4, 16)
    ten, scratch = run_and_check(w)
    bits = lambda a: oracle.to_bf16_bits(np.asarray(a, dtype=np.float32))  # noqa: E731
    _, ref = oracle.gating_attention_bf16(bits(w.x), bits(w.wq), bits(w.wk), bits(w.wv), bits(w.wg), w.bg, bits(w.wo), w.bo,
                                          bits(w.bias), bits(w.nb), w.H, return_scratch=True)
    for name in ("q", "k", "gate"):
        got = helpers.to_numpy(scratch[name]).reshape(w.B, w.S, w.C)
        helpers.check_close(got, oracle.from_bf16_bits(ref[name]).reshape(w.B, w.S, w.C), "bf16", name)
    helpers.check_close(helpers.to_numpy(scratch["v"]), oracle.from_bf16_bits(ref["v"]), "bf16", "v")


def test_replays_from_a_hip_graph(torch_cuda):
    """The route's seven launches (five products, the attention, nothing that allocates, clears memory or synchronises)
    captured into a HIP graph on a side stream and replayed three times, with eager work between the replays (the results
    and the scratch tensors overwritten); every replay reproduces the eager result bit for bit."""
    import ctypes
    torch = torch_cuda
    w = draw_workload(21, 5, 200, 8, 8)
    ten, scratch = helpers.to_device(w)
    a = helpers.hip_args(w, ten, scratch, capi.PATH_TILED)
    assert capi.lib().kutacc_hip_gating_attention(ctypes.byref(a), None) == 0  # eager: also takes first-call set-up out of the capture
    torch.cuda.synchronize()
    want_out, want_avg = ten["out"].clone(), scratch["avg"].clone()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        assert capi.lib().kutacc_hip_gating_attention(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(3):
        ten["out"].fill_(7.0)
        for t in scratch.values():
            t.fill_(-3.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert helpers.same_bits(ten["out"], want_out) and helpers.same_bits(scratch["avg"], want_avg)


@pytest.mark.parametrize("B,S,H,d", [(1, 1, 8, 8), (3, 33, 8, 8), (5, 77, 4, 16)])
def test_output_projection_of_64_channels_on_every_form_of_its_operands(torch_cuda, B, S, H, d):
    """Dense results on any address take the row kernel; a wider pitch, weights off the 16-byte grid the products' kernels.  All within
    the parity bar, and so within twice that of each other."""
    import ctypes
    torch = torch_cuda
    w = draw_workload(70 + S, B, S, H, d)
    want = helpers.oracle_out(w)
    for form in ("dense", "dense, one element on", "pitch 72", "weights one element on"):
        ten, scratch = helpers.to_device(w)
        a = helpers.hip_args(w, ten, scratch, capi.PATH_TILED)
        room = torch.full((B * S * 72 + 8,), 5.0, device="cuda", dtype=torch.bfloat16)
        shift, pitch = int(form == "dense, one element on"), 72 if form == "pitch 72" else 64
        a.out, a.out_ld = room.data_ptr() + 2 * shift, pitch
        moved = torch.cat([ten["wo"].new_zeros(1), ten["wo"].flatten()])
        if form == "weights one element on":
            a.output_w = moved.data_ptr() + 2
        print(f"64 channels B={B} S={S} H={H} d={d} {form}", flush=True)
        names = helpers.profiled_kernels(torch, lambda: expect_success(capi.lib().kutacc_hip_gating_attention(ctypes.byref(a), None)))  # noqa: B023
        assert ("linear_rows_kernel" in names) == form.startswith("dense"), (form, names)
        used = room[shift:shift + B * S * pitch].view(B, S, pitch)
        helpers.check_close(helpers.to_numpy(used[..., :64]), want, "bf16", form)
        assert bool((room[:shift] == 5.0).all()) and bool((room[shift + B * S * pitch:] == 5.0).all()) and bool((used[..., 64:] == 5.0).all())


def expect_success(rc):
    assert rc == 0, rc


def test_unsupported_layouts_fall_back_to_the_generic_kernels(torch_cuda):
    """A head size that is no multiple of 8 is not this route's: the automatic choice takes the scalar kernels, the forced
    routes refuse."""
    w = draw_workload(12, 2, 50, 4, 12)
    ten, scratch = helpers.to_device(w)
    assert helpers.run_hip(w, ten, scratch, capi.PATH_TILED) == capi.EUNSUPPORTED
    assert helpers.run_hip(w, ten, scratch, capi.PATH_FUSED) == capi.EUNSUPPORTED
    assert helpers.run_hip(w, ten, scratch, capi.PATH_AUTO) == 0 and capi.last_path() == "generic"
    helpers.check_close(helpers.to_numpy(ten["out"]), helpers.oracle_out(w), "bf16", "out")


def test_handle_based_entry_point_takes_the_route(torch_cuda):
    """kutacc_af2_gating_attention with 64 channels and head size 8 (device tensors), and the same call on host pointers
    (staged): same bits."""
    w = draw_workload(13, 4, 120, 8, 8)
    op, ten, scratch = helpers.make_op(w)
    op.run()
    assert not capi.error_flag() and capi.last_path() == "tiled_mfma"
    helpers.check_close(helpers.to_numpy(ten["out"]), helpers.oracle_out(w), "bf16", "out")
    hten, hscratch = helpers.host_arrays(w)
    hop = capi.GatedAttention(hten["x"], hten["wq"], hten["wk"], hten["wv"], hten["wg"], hten["bg"], hten["wo"], hten["bo"],
                              hten["bias"], hten["nb"], w.H, hten["out"], hscratch)
    hop.run()
    assert not capi.error_flag() and capi.last_path() == "tiled_mfma"
    np.testing.assert_array_equal(hten["out"], ten["out"].view(torch_cuda.int16).cpu().numpy().view(np.uint16))


LOWEST = float(np.float32(np.array(0xff7f0000, dtype=np.uint32).view(np.float32)))  # of bf16


# the persistent kernels on single rows (fragments, tiles, neither) and on pairs, a workgroup per unit, the streamed kernels, the tiles, heads of 8
@pytest.mark.parametrize("B,S,H,d", [(9, 301, 4, 32), (16, 384, 4, 32), (130, 96, 4, 32), (66, 200, 4, 32), (40, 200, 4, 32), (6, 64, 4, 32), (3, 385, 4, 32),
                                     (64, 64, 8, 32), (20, 259, 8, 32), (2, 1200, 4, 32), (64, 77, 8, 8), (6, 70, 8, 8), (3, 200, 4, 16), (1, 70, 3, 40)])
@pytest.mark.parametrize("pair_bias", [True, False])
def test_rows_masked_with_the_types_lowest_value(torch_cuda, B, S, H, d, pair_bias):
    """The lowest value of bf16 times log2(e) is past fp32's range: a batch row with such a mask throughout gave NaN.  It is an even average, as with a mask
    of -1e9, and a key with such a mask among others has no weight."""
    w = draw_workload(9100 + S, B, S, H, d, pair_bias=pair_bias, masked=0.0)
    w.bias[B - 1] = LOWEST
    w.bias[0, S // 3:] = LOWEST
    op, ten, scratch = helpers.make_op(w)
    op.run()
    torch_cuda.cuda.synchronize()
    assert not capi.error_flag() and capi.last_path() != "generic"
    ref_out, ref_avg = helpers.oracle_out(w, return_avg=True)
    helpers.check_close(helpers.to_numpy(scratch["avg"]).reshape(w.B, w.S, w.C), ref_avg, "bf16", "gated average")
    helpers.check_close(helpers.to_numpy(ten["out"]), ref_out, "bf16", "out")


@pytest.mark.parametrize("B,S,H,d", [(2, 1200, 4, 32), (64, 77, 8, 8), (6, 64, 8, 8), (5, 7, 8, 8), (3, 200, 4, 16), (2, 96, 3, 24), (2, 100, 2, 64)])
def test_pair_bias_rows_of_the_types_lowest_value(torch_cuda, B, S, H, d):
    """The same of a query whose row of the pair bias has it throughout, on the kernels that read the bias as it lies."""
    w = draw_workload(9200 + S, B, S, H, d, masked=0.0)
    w.nb[:, S // 2] = LOWEST
    w.nb[1, S - 1] = LOWEST
    w.nb[0, 0, :S // 2] = LOWEST
    run_and_check(w, capi.PATH_TILED)


def test_pair_bias_rows_of_the_types_lowest_value_in_the_lanes_order(torch_cuda):
    """The same where the bias of heads of 8 is brought into the order of the logits by a pass of its own: the bits of the kernel that reads it as it lies."""
    torch = torch_cuda
    B, S = 1880, 127
    g = torch.Generator(device="cuda").manual_seed(9300)
    bf16 = lambda *shape, scale=1.0: (torch.randn(*shape, device="cuda", generator=g) * scale).to(torch.bfloat16)  # noqa: E731
    x = torch.nn.functional.layer_norm(torch.randn(B, S, 64, device="cuda", generator=g), (64,)).to(torch.bfloat16)
    wq, wk, wv, wg, wo = (bf16(64, 64, scale=0.125) for _ in range(5))
    bg, bo = torch.ones(64, device="cuda"), torch.zeros(64, device="cuda")
    bias = torch.zeros(B, S, device="cuda", dtype=torch.bfloat16)
    bias[B - 1] = LOWEST
    wide = torch.zeros(8, S, 136, device="cuda", dtype=torch.bfloat16)
    wide[..., :S] = bf16(8, S, S)
    wide[:, S // 2, :S] = LOWEST
    wide[1, S - 1, :S] = LOWEST
    got = []
    for nb, passes in ((wide[..., :S], False), (wide[..., :S].contiguous(), True)):
        out = torch.full_like(x, 7.0)
        scratch = {k: torch.zeros(B, S, 8, 8, device="cuda", dtype=torch.bfloat16) for k in ("q", "k", "gate", "avg")}
        scratch["v"] = torch.zeros(8, 8, B, S, device="cuda", dtype=torch.bfloat16)
        names = helpers.profiled_kernels(torch, capi.GatedAttention(x, wq, wk, wv, wg, bg, wo, bo, bias, nb, 8, out, scratch).run)
        torch.cuda.synchronize()
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert ("seed_tiles_kernel" in names) == passes, names
        assert not capi.error_flag() and bool(torch.isfinite(out).all()) and bool(torch.isfinite(scratch["avg"]).all())
        got.append((out, scratch["avg"]))
    assert helpers.same_bits(got[0][0], got[1][0]) and helpers.same_bits(got[0][1], got[1][1])


@pytest.mark.parametrize("B,S,H,d", [(9, 301, 4, 32), (66, 200, 4, 32), (40, 200, 4, 32), (6, 64, 4, 32), (3, 385, 4, 32), (20, 259, 8, 32), (2, 1200, 4, 32),
                                     (64, 77, 8, 8), (3, 200, 4, 16)])
@pytest.mark.parametrize("bits", [0x7fc0, 0xffc0])
def test_a_mask_that_is_no_number_is_not_taken_for_a_low_one(torch_cuda, B, S, H, d, bits):
    """A NaN of either sign in a batch row's mask shows in all of that row's averages, and in no other row's."""
    w = draw_workload(9400 + S, B, S, H, d, masked=0.0)
    op, ten, scratch = helpers.make_op(w)
    ten["bias"].view(torch_cuda.int16)[1, S // 3] = bits - 0x10000 if bits > 0x7fff else bits
    op.run()
    torch_cuda.cuda.synchronize()
    avg = scratch["avg"].float().reshape(B, S, H * d)
    assert not capi.error_flag() and capi.last_path() != "generic"
    assert bool(torch_cuda.isnan(avg[1]).all()) and bool(torch_cuda.isfinite(avg[[b for b in range(B) if b != 1]]).all())
