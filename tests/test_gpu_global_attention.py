"""GPU parity of kutacc_af2_global_attention (reference src/attention/global_attention.cpp:30-205) against the CPU
oracle, through the C ABI.  bf16 storage; tolerance as for the gated attention: 2e-2 absolute + 1e-2 relative
against the fp32 oracle on the same bf16-rounded inputs."""
import math
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import helpers  # noqa: E402
from kutacc_amd import capi  # noqa: E402
from kutacc_amd.workloads import round_to_bf16  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    capi.lib()
    return torch


def make_case(seed, B, S, H, d, mask_mode="random"):
    rng = np.random.Generator(np.random.PCG64(seed))
    C = H * d
    f = lambda *s: round_to_bf16(rng.standard_normal(s).astype(np.float32))  # noqa: E731
    w = lambda *s: round_to_bf16((rng.standard_normal(s) / math.sqrt(s[-1])).astype(np.float32))  # noqa: E731
    mask = np.ones((B, S), dtype=np.float32)
    if mask_mode == "random":
        mask = (rng.random((B, S)) > 0.25).astype(np.float32)
        mask[:, 0] = 1
        if B > 2:
            mask[B - 1] = 0  # one row with every token masked
    return dict(x=f(B, S, C), mask=mask, wq=w(C, C), wk=w(d, C), wv=w(d, C), wg=w(C, C),
                bg=np.ones(C, dtype=np.float32), wo=w(C, C), bo=rng.standard_normal(C).astype(np.float32), nheads=H)


def oracle_out(c):
    from oracle import oracle
    return oracle.global_attention_f32(c["x"], c["mask"], c["wq"], c["wk"], c["wv"], c["wg"], c["bg"], c["wo"], c["bo"],
                                       c["nheads"], return_q_avg=True)


def device_op(torch, c, device="cuda"):
    B, S, C = c["x"].shape
    d = C // c["nheads"]
    bf = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch.bfloat16).to(device)  # noqa: E731
    f32 = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    ten = dict(x=bf(c["x"]), mask=bf(c["mask"].reshape(B, S, 1)), wq=bf(c["wq"]), wk=bf(c["wk"]), wv=bf(c["wv"]),
               wg=bf(c["wg"]), bg=f32(c["bg"]), wo=bf(c["wo"]), bo=f32(c["bo"]),
               out=torch.zeros((B, S, C), dtype=torch.bfloat16, device=device))
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16, device=device)  # noqa: E731
    scratch = dict(q=z(B, C), k=z(B * S, d), v=z(d, B * S), gate=z(B, S, C), avg=z(B, C))
    op = capi.GlobalAttention(ten["x"], ten["mask"], ten["wq"], ten["wk"], ten["wv"], ten["wg"], ten["bg"], ten["wo"],
                              ten["bo"], c["nheads"], ten["out"], scratch)
    return op, ten, scratch


SHAPES = [
    # B, S, H, d, mask
    (4, 128, 8, 8, "random"), (3, 97, 8, 8, "random"), (2, 1024, 8, 8, "random"), (5, 33, 4, 16, "random"),
    (2, 200, 2, 32, "ones"), (3, 1, 8, 8, "ones"), (6, 7, 16, 4, "random"), (2, 1500, 8, 8, "random"),
    # both workgroup sizes of the kernel: eight waves while a row has a CU to itself (at most 256 rows) or is streamed,
    # four when two rows share a CU
    (300, 512, 8, 8, "random"), (257, 1024, 4, 16, "random"), (256, 640, 8, 8, "random"), (3, 2100, 4, 16, "random"),
    # streamed rows on either side of what the eight-wave layout's LDS holds (7808 positions), and the longest row
    (2, 7808, 8, 8, "random"), (2, 8192, 8, 8, "random"), (1, 12288, 8, 8, "random"),
]


@pytest.mark.parametrize("B,S,H,d,mask_mode", SHAPES)
def test_global_attention_matches_oracle(torch_cuda, B, S, H, d, mask_mode):
    c = make_case(100 + S, B, S, H, d, mask_mode)
    op, ten, scratch = device_op(torch_cuda, c)
    op.run()
    assert not capi.error_flag() and capi.last_path() == "global_mfma"
    rows = list(range(B)) if B <= 8 else sorted({0, 1, B // 2, B - 2, B - 1})  # large batches: the oracle on a few rows
    ref, ref_qavg = oracle_out(dict(c, x=c["x"][rows], mask=c["mask"][rows]))
    helpers.check_close(helpers.to_numpy(ten["out"][rows]), ref, "bf16", "global attention out")
    helpers.assert_within(helpers.to_numpy(scratch["avg"][rows]), ref_qavg, 2.0 ** -8 * np.abs(ref_qavg) + 1e-6, "masked mean q_avg")


@pytest.mark.parametrize("B,S,H,d", [(2, 1025, 8, 8), (2, 2048, 8, 8), (2, 2049, 4, 16), (2, 2305, 8, 8), (2, 2590, 2, 32), (2, 3201, 16, 4)])
def test_global_attention_rows_past_the_kept_tiles(torch_cuda, B, S, H, d):
    """The first length past the rows that are kept whole; all tiles kept by eight waves; one wave with one tile that is read
    again, one with two (the depth of its ring) and the others with one, all with two and a partial third, four to five."""
    c = make_case(300 + S, B, S, H, d)
    op, ten, scratch = device_op(torch_cuda, c)
    op.run()
    assert not capi.error_flag() and capi.last_path() == "global_mfma"
    ref, ref_qavg = oracle_out(c)
    helpers.check_close(helpers.to_numpy(ten["out"]), ref, "bf16", "global attention out")
    helpers.assert_within(helpers.to_numpy(scratch["avg"]), ref_qavg, 2.0 ** -8 * np.abs(ref_qavg) + 1e-6, "masked mean q_avg")


def device_case(torch, B, S, H, d):
    """make_case on the device, for batches too large to draw and convert on the host quickly."""
    g = torch.Generator(device="cuda").manual_seed(B * 10007 + S)
    bf = lambda *s, scale=1.0: (torch.randn(*s, device="cuda", generator=g) * scale).to(torch.bfloat16)  # noqa: E731
    C = H * d
    mask = (torch.rand(B, S, device="cuda", generator=g) > 0.25).to(torch.bfloat16)
    mask[:, 0] = 1
    mask[B - 1] = 0
    ten = dict(x=bf(B, S, C), mask=mask[..., None].contiguous(), wq=bf(C, C, scale=C ** -0.5), wk=bf(d, C, scale=C ** -0.5), wv=bf(d, C, scale=C ** -0.5),
               wg=bf(C, C, scale=C ** -0.5), bg=torch.ones(C, device="cuda"), wo=bf(C, C, scale=C ** -0.5), bo=torch.randn(C, device="cuda", generator=g))
    return ten, torch.full((B, S, C), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((B, C), -3.0, dtype=torch.bfloat16, device="cuda")


def run_device_case(torch, ten, out, avg, H):
    small = torch.zeros(1, out.shape[2], dtype=torch.bfloat16, device="cuda")  # the device library leaves these alone
    op = capi.GlobalAttention(ten["x"], ten["mask"], ten["wq"], ten["wk"], ten["wv"], ten["wg"], ten["bg"], ten["wo"], ten["bo"], H, out,
                              dict(q=small, k=small, v=small, gate=small, avg=avg))
    op.run()
    assert not capi.error_flag() and capi.last_path() == "global_mfma"


@pytest.mark.parametrize("rows,S", [
    (-1, 513), (-1, 2561),                 # one row short of the CUs: a workgroup each
    (0.5, 481), (0.5, 1024), (0.5, 1057), (0.5, 5121),  # two workgroups a row: first and last length kept whole, first read again, most with tiles of
                                           # the first part all kept and one wave of the second with one more
    (0.3, 2600), (0.2, 700), (7, 2600),    # three, five, eight
    (1.25, 1100), (1.004, 1056),           # rows with a workgroup each, and a rest that shares four, and eight
])
def test_global_attention_rows_shared_by_workgroups(torch_cuda, rows, S):
    torch = torch_cuda
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    B = rows if isinstance(rows, int) and rows > 0 else cus + rows if isinstance(rows, int) else int(rows * cus)
    ten, out, avg = device_case(torch, B, S, 8, 8)
    run_device_case(torch, ten, out, avg, 8)
    checked = sorted({0, 1, B // 2, B - 7, B - 2, B - 1} if B > 7 else set(range(B)))
    c = dict(nheads=8, **{k: helpers.to_numpy(ten[k]) for k in ("wq", "wk", "wv", "wg", "bg", "wo", "bo")})
    c["x"], c["mask"] = helpers.to_numpy(ten["x"][checked]), helpers.to_numpy(ten["mask"][checked][..., 0])
    ref, ref_qavg = oracle_out(c)
    helpers.check_close(helpers.to_numpy(out[checked]), ref, "bf16", "global attention out")
    helpers.assert_within(helpers.to_numpy(avg[checked]), ref_qavg, 2.0 ** -8 * np.abs(ref_qavg) + 1e-6, "masked mean q_avg")
    # every row alone against the call: a workgroup's sums may be in another order, nothing else
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(avg).all())
    one_out, one_avg = torch.empty_like(out[:1]), torch.empty_like(avg[:1])
    for b in checked:
        run_device_case(torch, dict(ten, x=ten["x"][b:b + 1].clone(), mask=ten["mask"][b:b + 1].clone()), one_out, one_avg, 8)
        helpers.check_close(helpers.to_numpy(out[b]), helpers.to_numpy(one_out[0]), "bf16", "a row among others and alone")


def test_global_attention_in_place_keeps_a_workgroup_per_row(torch_cuda):
    """The result over the input: the same as into memory of its own, within the order of the sums."""
    torch = torch_cuda
    ten, out, avg = device_case(torch, 20, 2600, 8, 8)
    run_device_case(torch, ten, out, avg, 8)
    again = ten["x"].clone()
    run_device_case(torch, dict(ten, x=again), again, avg, 8)
    helpers.check_close(helpers.to_numpy(again), helpers.to_numpy(out), "bf16", "global attention in place")


@pytest.mark.parametrize("rows,S", [(0.5, 1024), (0.5, 1057), (0.5, 5121), (0.3, 2600), (0.2, 700), (7, 2600), (1.25, 1100), (1.004, 1056)])
def test_global_attention_rows_shared_by_workgroups_keep_their_bits(torch_cuda, rows, S):
    """Rows of the same values, some of them shared by two to eight workgroups, have the same bits, and the bits of rows with a workgroup each
    (the result over the input): every workgroup of a row forms the same mean and the same average."""
    torch = torch_cuda
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    B = rows if isinstance(rows, int) else int(rows * cus)
    ten, out, avg = device_case(torch, B, S, 8, 8)
    ten["x"], ten["mask"] = ten["x"][:1].expand(B, -1, -1).contiguous(), ten["mask"][:1].expand(B, -1, -1).contiguous()
    run_device_case(torch, ten, out, avg, 8)
    alone, alone_avg = ten["x"].clone(), torch.empty_like(avg)
    run_device_case(torch, dict(ten, x=alone), alone, alone_avg, 8)
    for got, one in ((out, alone), (avg, alone_avg)):
        assert helpers.same_bits(one, one[:1].expand_as(one).contiguous())
        assert helpers.same_bits(got, one)


def test_global_attention_replays_from_a_hip_graph(torch_cuda):
    """Rows past the kept tiles, whose rest comes through the ring in the LDS: captured on a side stream and replayed three times, with
    eager work (the results overwritten) between the replays; every replay gives the eager result bit for bit."""
    torch = torch_cuda
    c = make_case(11, 3, 2590, 8, 8)
    op, ten, scratch = device_op(torch, c)
    op.run()
    torch.cuda.synchronize()
    want, want_avg = ten["out"].clone(), scratch["avg"].clone()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    capi.set_blocking(False)
    try:
        with torch.cuda.graph(graph, stream=side):
            capi.set_stream(torch.cuda.current_stream().cuda_stream)
            op.run()
    finally:
        capi.set_stream(None)
        capi.set_blocking(True)
    assert not capi.error_flag()
    for _ in range(3):
        ten["out"].fill_(7.0)
        scratch["avg"].fill_(-3.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert helpers.same_bits(ten["out"], want) and helpers.same_bits(scratch["avg"], want_avg)


def test_global_attention_full_extra_msa_shape(torch_cuda):
    """An extra-MSA sized call (N_res = 256 batch rows of 1024 extra sequences): spot-check rows against the oracle."""
    c = make_case(7, 256, 1024, 8, 8, "random")
    op, ten, _ = device_op(torch_cuda, c)
    op.run()
    assert not capi.error_flag()
    rows = [0, 100, 255]
    sub = dict(c, x=c["x"][rows], mask=c["mask"][rows])
    ref, _ = oracle_out(sub)
    helpers.check_close(helpers.to_numpy(ten["out"][rows]), ref, "bf16", "global attention, extra-MSA shape")


def test_global_attention_host_pointers_match_device_pointers(torch_cuda):
    c = make_case(9, 3, 70, 8, 8)
    op, ten, scratch = device_op(torch_cuda, c)
    op.run()
    from kutacc_amd.workloads import bf16_bits
    B, S, C = c["x"].shape
    hb = lambda a: bf16_bits(np.ascontiguousarray(a))  # noqa: E731
    hten = dict(x=hb(c["x"]), mask=hb(c["mask"].reshape(B, S, 1)), wq=hb(c["wq"]), wk=hb(c["wk"]), wv=hb(c["wv"]),
                wg=hb(c["wg"]), bg=c["bg"].copy(), wo=hb(c["wo"]), bo=c["bo"].copy(), out=np.zeros((B, S, C), np.uint16))
    hz = lambda *s: np.zeros(s, dtype=np.uint16)  # noqa: E731
    hscratch = dict(q=hz(B, C), k=hz(B * S, 8), v=hz(8, B * S), gate=hz(B, S, C), avg=hz(B, C))
    hop = capi.GlobalAttention(hten["x"], hten["mask"], hten["wq"], hten["wk"], hten["wv"], hten["wg"], hten["bg"],
                               hten["wo"], hten["bo"], 8, hten["out"], hscratch)
    hop.run()
    assert not capi.error_flag()
    out_bits = ten["out"].view(torch_cuda.int16).cpu().numpy().view(np.uint16)
    np.testing.assert_array_equal(hten["out"], out_bits)
    np.testing.assert_array_equal(hscratch["avg"], scratch["avg"].view(torch_cuda.int16).cpu().numpy().view(np.uint16))


def test_global_attention_rejects_other_channel_counts(torch_cuda, capfd):
    c = make_case(3, 2, 16, 4, 8)  # 32 channels
    op, ten, _ = device_op(torch_cuda, c)
    op.run()
    assert capi.error_flag()
    assert "invalid int value" in capfd.readouterr().err


def test_global_attention_rejects_rows_beyond_the_lds(torch_cuda):
    c = make_case(5, 1, 12320, 8, 8)
    op, ten, _ = device_op(torch_cuda, c)
    op.run()
    assert capi.error_flag()
    capi.clear_error()
