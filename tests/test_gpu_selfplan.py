"""Device-length decode planned by the kernel itself (the reference's launch_batched_paged /
qk_batched_paged_decode_attn take the lengths in device memory: batched.cu:140-147,
qwen_kernels.cu:293-326).

Every workgroup derives the host planner's units from the device lengths, so the
outputs must equal the host-planned launch's bit for bit (same chunks, same merge
order), whatever order the units run in and however many workgroups serve them; and
they must match the CPU oracle within the path's tolerance.  On the VALU kernel,
sequences of at most self_lead_tokens tokens are attended whole by the waves that
wait while wave 0 plans, and the plan leaves them out: the other sequences still
equal the host plan bit for bit, the short ones match the oracle, and paged equals
contiguous bit for bit.  No length is truncated:
a stated cap only sizes the launch, and the explicit-split path (whose grid is sized
by the cap) gives NaN rows, never a partial attention, for a sequence longer than it.
"""
import numpy as np
import pytest

from kvcache_amd import KVC_F16, KVC_F32, ops
from kvcache_amd import workloads as W
from kvcache_amd._native import KVC_ERR_ARG, KvcError
from kvcache_amd.device import DeviceBuffer
from kvcache_amd.engine import BlockAllocator
from kvcache_amd.workloads import build_tables

from _helpers import as_np, dev, host, normal, paged_layout, say, tol, tuning

pytestmark = pytest.mark.gpu


def inputs(lens, Hq, Hkv, D, dtype, seed):
    nt = as_np(dtype)
    S = max(int(max(lens)), 1)
    N = len(lens)
    return (normal((N, Hq, D), seed, nt), normal((N, Hkv, S, D), seed + 1, nt), normal((N, Hkv, S, D), seed + 2, nt))


def self_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype, cap=0, workspace=None):
    N, Hq, D = q.shape
    out = DeviceBuffer(q.nbytes)
    ops.launch_batched_paged(dev(q), dev(kp), dev(vp), dev(table), dev(tab_off), dev(np.asarray(lens, np.int32)), out,
                             N, Hq, D, B, cap, float(1.0 / np.sqrt(D)), Hkv=Hkv, dtype=dtype, workspace=workspace)
    return host(out, q.dtype, q.shape).astype(np.float64)


def host_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype):
    N, Hq, D = q.shape
    work, nu, nr = ops.decode_plan(lens, Hq, Hkv, D, B, tab_off=tab_off, table=table, dtype=dtype)
    out = DeviceBuffer(q.nbytes)
    ops.launch_batched_paged_planned(dev(q), dev(kp), dev(vp), dev(table), len(table), out, N, Hq, Hkv, D, B,
                                     float(1.0 / np.sqrt(D)), dev(work), nu, nr, dtype=dtype)
    return host(out, q.dtype, q.shape).astype(np.float64)


def oracle(orc, q, K, V, lens):
    return orc.batched_contig(q, K, V, np.asarray(lens, np.int32), float(1.0 / np.sqrt(q.shape[2])))


CASES = {
    # name: (lengths, Hq, Hkv, D, dtype)
    "c2_reference": (W.ref_lengths(), 8, 8, 64, KVC_F16),
    "c2_loguniform": (W.loguniform_lengths(128, 16, 2048, 7), 8, 8, 64, KVC_F16),
    "gqa_mfma_long": (np.array([8192, 16384, 300, 1, 0, 2500, 700, 1025], np.int32), 14, 2, 64, KVC_F16),
    "gqa_mfma_d128": (np.array([5, 1500, 4097, 33, 900], np.int32), 16, 2, 128, KVC_F16),
    "mha_fp32": (np.array([1, 17, 640, 961, 2000, 3000, 0, 64], np.int32), 8, 8, 64, KVC_F32),
    "gqa_valu_fp32": (np.array([1000, 15, 16, 17, 3000, 1], np.int32), 14, 2, 64, KVC_F32),
    "group2_fp16": (np.array([2048, 1024, 333, 5000, 7], np.int32), 8, 4, 64, KVC_F16),
    # every length within the largest short-sequence threshold: the plan has no units at all
    "short_mha": (np.array([1, 0, 700, 1024, 33, 64, 65, 1000], np.int32), 8, 8, 64, KVC_F16),
}


@pytest.mark.parametrize("case", list(CASES))
def test_self_planned_equals_host_planned(orc, case):
    lens, Hq, Hkv, D, dtype = CASES[case]
    say(f"self-planned vs host-planned: {case}")
    B = 16
    q, K, V = inputs(lens, Hq, Hkv, D, dtype, 300)
    nb = sum((int(x) + B - 1) // B for x in lens)
    kp, vp, table, tab_off = paged_layout(K, V, lens, B, np.random.default_rng(8).permutation(nb))
    with tuning("self_lead_tokens", 0):
        got = self_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype, cap=int(max(lens)))
    ref = host_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype)
    np.testing.assert_array_equal(got, ref)
    want = oracle(orc, q, K, V, lens)
    assert np.abs(got - want).max() <= tol(dtype)
    assert np.all(got[np.asarray(lens) == 0] == 0)
    lead = self_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype, cap=int(max(lens)))  # short ones while planning
    assert np.abs(lead - want).max() <= tol(dtype)
    assert np.all(lead[np.asarray(lens) == 0] == 0)
    planned = np.asarray(lens) > 320  # (the default threshold; matrix-core shapes plan every sequence)
    np.testing.assert_array_equal(lead[planned], ref[planned])


@pytest.mark.parametrize("grid", [1, 7, 100])
def test_small_grids_serve_every_rank_once(orc, grid):
    """With fewer workgroups than units, each workgroup serves several ranks (rounds in
    alternating direction): the same outputs, bit for bit, on a first and a second
    launch over a never-cleared workspace (epoch-tagged arrival counters)."""
    say(f"self-planned, grid {grid}")
    lens, Hq, Hkv, D, dtype = np.array([1, 700, 2048, 90, 5000, 16, 1300], np.int32), 14, 2, 64, KVC_F16
    q, K, V = inputs(lens, Hq, Hkv, D, dtype, 310)
    kp, vp, table, tab_off = paged_layout(K, V, lens, 16)
    ws = DeviceBuffer(ops.decode_workspace_size(len(lens), Hq, Hkv, D, 16, 0, 0, dtype))
    ws.upload(np.random.default_rng(1).integers(0, 256, ws.nbytes, dtype=np.uint8))
    with tuning("self_lead_tokens", 0):  # (small grids run without lead chunks)
        ref = self_planned(q, kp, vp, table, tab_off, lens, Hkv, 16, dtype)
    with tuning("self_grid", grid):
        a = self_planned(q, kp, vp, table, tab_off, lens, Hkv, 16, dtype, workspace=ws)
        b = self_planned(q, kp, vp, table, tab_off, lens, Hkv, 16, dtype, workspace=ws)
    np.testing.assert_array_equal(a, ref)
    np.testing.assert_array_equal(b, ref)
    assert np.abs(ref - oracle(orc, q, K, V, lens)).max() <= 2e-3


def test_paged_and_contiguous_agree_bit_for_bit_gqa():
    """The reference's paged-vs-contiguous check (bench_throughput.cu:124-128) on the
    default launchers: both plan the same chunks from the device lengths."""
    say("self-planned paged vs contiguous, GQA fp16")
    lens = np.array([1, 16, 17, 1000, 4000, 2500, 64, 1023], np.int32)
    N, Hq, Hkv, D = len(lens), 14, 2, 64
    q, K, V = inputs(lens, Hq, Hkv, D, KVC_F16, 320)
    nb = sum((int(x) + 15) // 16 for x in lens)
    kp, vp, table, tab_off = paged_layout(K, V, lens, 16, np.random.default_rng(2).permutation(nb + 40))
    paged = self_planned(q, kp, vp, table, tab_off, lens, Hkv, 16, KVC_F16)
    out = DeviceBuffer(q.nbytes)
    S = K.shape[2]
    ops.launch_batched_decode(dev(q), dev(K), dev(V), dev(lens), out, N, Hq, D, S, int(lens.max()),
                              float(1.0 / np.sqrt(D)), Hkv=Hkv, dtype=KVC_F16)
    np.testing.assert_array_equal(paged, host(out, np.float16, q.shape).astype(np.float64))


def test_lengths_past_the_stated_cap_are_attended_whole(orc):
    """qk_batched_paged_decode_attn has no cap (qwen_kernels.h:35-37) and a cap is only a
    hint to launch_batched_paged: a 40k-token context (past the 32768 a fixed bound
    would have cut it at) and lengths above a cap of 100 are attended over their whole
    length."""
    say("no truncation past cap")
    lens = np.array([40000, 3, 1200], np.int32)
    Hq, Hkv, D = 14, 2, 64
    q, K, V = inputs(lens, Hq, Hkv, D, KVC_F16, 330)
    kp, vp, table, tab_off = paged_layout(K, V, lens, 16)
    out = DeviceBuffer(q.nbytes)
    ops.qk_batched_paged_decode_attn(dev(q), out, dev(kp), dev(vp), dev(table), dev(tab_off), dev(lens), len(lens),
                                     Hq, Hkv, D, 16, float(1.0 / np.sqrt(D)))
    got = host(out, np.float16, q.shape).astype(np.float64)
    ref = oracle(orc, q, K, V, lens)
    assert np.abs(got - ref).max() <= 2e-3
    hinted = self_planned(q, kp, vp, table, tab_off, lens, Hkv, 16, KVC_F16, cap=100)
    np.testing.assert_array_equal(hinted, got)
    # a prefix-only attention would differ from the whole-length one
    cut = oracle(orc, q, K[:, :, :32768], V[:, :, :32768], np.minimum(lens, 32768))
    assert np.abs(cut[0] - ref[0]).max() > 1e-2


def test_long_mean_context_within_the_stated_cap(orc):
    """One- and two-head units take chunks of at most 64 blocks and 64 partial records
    per (sequence, head) by default, so a batch whose mean context passes 63 x 1024
    tokens (BLOCK 16) cannot be planned without a bound: it gets NaN rows.  With the
    reference's own cap argument stated the record budget grows with it and the batch
    is attended whole."""
    say("mean context above the default record budget, MHA fp16")
    lens = np.array([70000, 75000], np.int32)
    Hq = Hkv = 2
    D = 64
    q, K, V = inputs(lens, Hq, Hkv, D, KVC_F16, 345)
    kp, vp, table, tab_off = paged_layout(K, V, lens, 16)
    got = self_planned(q, kp, vp, table, tab_off, lens, Hkv, 16, KVC_F16, cap=int(lens.max()))
    assert np.abs(got - oracle(orc, q, K, V, lens)).max() <= 2e-3
    unbounded = self_planned(q, kp, vp, table, tab_off, lens, Hkv, 16, KVC_F16, cap=0)
    assert np.all(np.isnan(unbounded))
    expect_device_error()


def test_explicit_split_past_cap_gives_nan_rows(orc):
    """The explicit-split path sizes its grid by cap: a longer sequence gets NaN rows
    (loud), the others their attention."""
    say("explicit split, length past cap")
    lens = np.array([50, 500, 80], np.int32)
    Hq, Hkv, D = 8, 8, 64
    q, K, V = inputs(lens, Hq, Hkv, D, KVC_F16, 340)
    kp, vp, table, tab_off = paged_layout(K, V, lens, 16)
    out = DeviceBuffer(q.nbytes)
    ops.launch_batched_paged(dev(q), dev(kp), dev(vp), dev(table), dev(tab_off), dev(lens), out, 3, Hq, D, 16, 100,
                             float(1.0 / np.sqrt(D)), dtype=KVC_F16, split=64)
    got = host(out, np.float16, q.shape).astype(np.float64)
    assert np.all(np.isnan(got[1]))
    ref = oracle(orc, q, K, V, lens)
    assert np.abs(got[[0, 2]] - ref[[0, 2]]).max() <= 2e-3
    expect_device_error(b"longer than its stated cap")


def test_contiguous_length_past_its_cache_gives_nan():
    say("contiguous length past MAXS")
    lens = np.array([10, 40], np.int32)
    Hq, Hkv, D, S = 8, 8, 64, 32
    q, K, V = normal((2, Hq, D), 350, np.float16), normal((2, Hkv, S, D), 351, np.float16), normal((2, Hkv, S, D), 352, np.float16)
    out = DeviceBuffer(q.nbytes)
    ops.launch_batched_decode(dev(q), dev(K), dev(V), dev(lens), out, 2, Hq, D, S, S, 0.125, Hkv=Hkv, dtype=KVC_F16)
    assert np.all(np.isnan(host(out, np.float16, q.shape).astype(np.float64)))
    expect_device_error()


def expect_device_error(text=b"NaN"):
    """The launch that wrote NaN rows also reported it: kvc_check_device_errors returns
    KVC_ERR_ARG once, then the report is cleared."""
    from kvcache_amd._native import lib
    with pytest.raises(KvcError) as e:
        ops.check_device_errors()
    assert e.value.status == KVC_ERR_ARG
    assert text in lib().kvc_last_error()
    ops.check_device_errors()


def test_device_error_fails_the_next_device_length_call(orc):
    """Without an explicit check, the next device-length decode call returns the report
    (KVC_ERR_ARG, nothing launched) and clears it; the call after that runs normally."""
    say("device error report surfaces at the next call")
    lens = np.array([50, 500, 80], np.int32)
    Hq, Hkv, D = 8, 8, 64
    q, K, V = inputs(lens, Hq, Hkv, D, KVC_F16, 341)
    kp, vp, table, tab_off = paged_layout(K, V, lens, 16)
    args = (dev(q), dev(kp), dev(vp), dev(table), dev(tab_off), dev(lens))
    out = DeviceBuffer(q.nbytes)
    ops.launch_batched_paged(*args, out, 3, Hq, D, 16, 100, float(1.0 / np.sqrt(D)), dtype=KVC_F16, split=64)
    host(out, np.float16, q.shape)  # the launch has finished: its report is in host memory
    with pytest.raises(KvcError) as e:
        ops.launch_batched_paged(*args, out, 3, Hq, D, 16, 0, float(1.0 / np.sqrt(D)), dtype=KVC_F16)
    assert e.value.status == KVC_ERR_ARG
    ops.launch_batched_paged(*args, out, 3, Hq, D, 16, 0, float(1.0 / np.sqrt(D)), dtype=KVC_F16)
    got = host(out, np.float16, q.shape).astype(np.float64)
    assert np.abs(got - oracle(orc, q, K, V, lens)).max() <= 2e-3
    ops.check_device_errors()


@pytest.mark.parametrize("case", ["gqa_mfma_600", "mha_valu_1100"])
def test_dropin_batches_past_one_launch(orc, case):
    """qk_batched_paged_decode_attn takes any N (a grid of N x Hq in the reference,
    qwen_kernels.cu:326-334) and no cap: more sequences than one self-planned launch plans
    (512 on the matrix cores, 1024 otherwise) run as consecutive launches, each attended
    whole."""
    rng = np.random.default_rng(370)
    N, Hq, Hkv, D, hi = (600, 14, 2, 64, 700) if case == "gqa_mfma_600" else (1100, 2, 2, 64, 200)
    say(f"drop-in batch of {N} sequences, {Hq}q/{Hkv}kv D{D}, cap 0")
    lens = rng.integers(0, hi, N).astype(np.int32)
    q, K, V = inputs(lens, Hq, Hkv, D, KVC_F16, 371)
    kp, vp, table, tab_off = paged_layout(K, V, lens, 16)
    out = DeviceBuffer(q.nbytes)
    ops.qk_batched_paged_decode_attn(dev(q), out, dev(kp), dev(vp), dev(table), dev(tab_off), dev(lens), N, Hq, Hkv,
                                     D, 16, float(1.0 / np.sqrt(D)))
    got = host(out, np.float16, q.shape).astype(np.float64)
    assert np.abs(got - oracle(orc, q, K, V, lens)).max() <= 2e-3
    ops.check_device_errors()


@pytest.mark.parametrize("B", [48, 4])
def test_dropin_block_without_self_plan_needs_no_cap(orc, B):
    """A BLOCK the self-planned kernel does not page (not a power of two, or smaller than a
    wave-load) with cap 0: the longest length is read from the device and sizes the grid,
    so every sequence is attended whole, as in the reference."""
    say(f"drop-in BLOCK {B}, cap 0")
    lens = np.array([1, 47, 48, 49, 1000, 3000, 0, 333], np.int32)
    Hq, Hkv, D = 14, 2, 64
    q, K, V = inputs(lens, Hq, Hkv, D, KVC_F16, 380 + B)
    kp, vp, table, tab_off = paged_layout(K, V, lens, B)
    out = DeviceBuffer(q.nbytes)
    ops.qk_batched_paged_decode_attn(dev(q), out, dev(kp), dev(vp), dev(table), dev(tab_off), dev(lens), len(lens),
                                     Hq, Hkv, D, B, float(1.0 / np.sqrt(D)))
    got = host(out, np.float16, q.shape).astype(np.float64)
    assert np.abs(got - oracle(orc, q, K, V, lens)).max() <= 2e-3
    ops.check_device_errors()


def test_device_position_variants(orc):
    """qkcuda_rope / qkcuda_write_kv / qkcuda_paged_causal_attn (qwen_kernels.h:42-47):
    positions read from device memory give the host-position results (rope and writes
    bit for bit; the prompt attention within tolerance of the CPU restatement)."""
    say("device-position rope / write / causal attention")
    rng = np.random.default_rng(360)
    Hq, Hkv, D, B, base, Nq = 14, 2, 64, 16, 1234, 5
    x = rng.standard_normal((Nq, Hq, D)).astype(np.float16)
    a, b = dev(x), dev(x)
    pos = dev(np.array([base], np.int32))
    ops.qk_rope(a, Nq, Hq, D, base, 1e6)
    ops.qkcuda_rope(b, Nq, Hq, D, pos, 1e6)
    np.testing.assert_array_equal(host(a, np.float16, x.shape), host(b, np.float16, x.shape))
    total = base + Nq
    nbk = (total + B - 1) // B
    table = rng.permutation(nbk + 7)[:nbk].astype(np.int32)
    kv = [rng.standard_normal((nbk + 7, Hkv, B, D)).astype(np.float16) for _ in range(2)]
    knew, vnew = (rng.standard_normal((Nq, Hkv, D)).astype(np.float16) for _ in range(2))
    p1, p2 = [dev(t) for t in kv], [dev(t) for t in kv]
    ops.qk_write_kv(dev(knew), dev(vnew), p1[0], p1[1], dev(table), base, Nq, Hkv, D, B)
    ops.qkcuda_write_kv(dev(knew), dev(vnew), p2[0], p2[1], dev(table), pos, Nq, Hkv, D, B)
    kp, vp = (host(t, np.float16, kv[0].shape) for t in p1)
    np.testing.assert_array_equal(kp, host(p2[0], np.float16, kv[0].shape))
    np.testing.assert_array_equal(vp, host(p2[1], np.float16, kv[0].shape))
    q = rng.standard_normal((Nq, Hq, D)).astype(np.float16)
    out = DeviceBuffer(q.nbytes)
    ops.qkcuda_paged_causal_attn(dev(q), out, p2[0], p2[1], dev(table), pos, Nq, Hq, Hkv, D, B, 0.125)
    got = host(out, np.float16, q.shape).astype(np.float64)
    ref = orc.paged_causal(q, kp, vp, table, base, Hkv, B, 0.125)
    assert np.abs(got - ref).max() <= 2e-3


@pytest.mark.parametrize("case", ["c2_reference", "gqa_mfma_long", "mha_fp32"])
def test_read_ahead_changes_no_output(case):
    """While the kernel plans, wave 1 of every workgroup reads the first blocks of every
    sequence ahead into an LDS sink (self_prefetch): no output may change, bit for bit,
    whatever the read-ahead budget -- none, the default, or one that covers whole
    sequences -- and with the minimum length at 0 (short sequences read ahead too)."""
    lens, Hq, Hkv, D, dtype = CASES[case]
    say(f"self-planned read-ahead on/off: {case}")
    B = 16
    q, K, V = inputs(lens, Hq, Hkv, D, dtype, 340)
    nb = sum((int(x) + B - 1) // B for x in lens)
    kp, vp, table, tab_off = paged_layout(K, V, lens, B, np.random.default_rng(9).permutation(nb))
    with tuning("self_lead_tokens", 0):  # (the read-ahead runs when there are no lead chunks)
        with tuning("self_prefetch_kib", 0):
            ref = self_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype)
        for kib, min_len in ((32768, 256), (1 << 20, 0), (64, 1)):
            with tuning("self_prefetch_kib", kib), tuning("self_prefetch_min_len", min_len):
                got = self_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype)
            np.testing.assert_array_equal(got, ref)


LEAD_CASES = ["c2_reference", "c2_loguniform", "mha_fp32", "gqa_valu_fp32", "group2_fp16", "short_mha"]


@pytest.mark.parametrize("case", LEAD_CASES)
def test_short_sequences_while_planning(orc, case):
    """Short-sequence thresholds -- one block, the default, more than most sequences,
    and the largest (a chunk's 64 blocks; larger requests are cut to it) -- against the
    oracle, on a first and a second launch over one never-cleared workspace; and paged
    against contiguous caches bit for bit (both cut the same chunks)."""
    lens, Hq, Hkv, D, dtype = CASES[case]
    say(f"self-planned, short sequences while planning: {case}")
    B = 16
    lens = np.asarray(lens, np.int32)
    N = len(lens)
    q, K, V = inputs(lens, Hq, Hkv, D, dtype, 350)
    nb = sum((int(x) + B - 1) // B for x in lens)
    kp, vp, table, tab_off = paged_layout(K, V, lens, B, np.random.default_rng(10).permutation(nb + 7))
    want = oracle(orc, q, K, V, lens)
    ws = DeviceBuffer(ops.decode_workspace_size(N, Hq, Hkv, D, B, 0, 0, dtype))
    ws.upload(np.random.default_rng(11).integers(0, 256, ws.nbytes, dtype=np.uint8))
    for lead in (16, 64, 1000, 1 << 20):
        with tuning("self_lead_tokens", lead):
            a = self_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype, workspace=ws)
            b = self_planned(q, kp, vp, table, tab_off, lens, Hkv, B, dtype, workspace=ws)
            out = DeviceBuffer(q.nbytes)
            ops.launch_batched_decode(dev(q), dev(K), dev(V), dev(lens), out, N, Hq, D, K.shape[2], 0,
                                      float(1.0 / np.sqrt(D)), Hkv=Hkv, dtype=dtype)
            contig = host(out, q.dtype, q.shape).astype(np.float64)
        err = np.abs(a - want).max()
        say(f"  threshold {lead}: max |err| {err:.2e}")
        assert err <= tol(dtype)
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, contig)
        assert np.all(a[lens == 0] == 0)


@pytest.mark.parametrize("n,causal", [(1, False), (5, False), (3, True)])
def test_block_table_at_the_end_of_its_allocation(orc, n, causal):
    # device-length launches carry no table length: every table read has to stay within
    # the blocks of the chunk it is for (each lane of a wave reads one entry of a chunk
    # that may have fewer than 64), also where the table's allocation ends with it
    say(f"table at the end of its allocation n={n} causal={causal}")
    Hq = Hkv = 8
    D, B, base = 64, 16, 4000
    lens = np.array([4001 - 300 * i for i in range(n)], np.int32) if not causal else np.array([base + n], np.int32)
    alloc = BlockAllocator(int(sum((int(x) + B - 1) // B for x in lens)))
    alloc.shuffle(3)
    table, off = build_tables(lens, B, alloc)
    kp, vp = (normal((alloc.total_blocks, Hkv, B, D), 40 + i, np.float16) for i in range(2))
    q = normal((n, Hq, D), 42, np.float16)
    room = 2 << 20  # a whole allocation unit: the table's last entry is its last four bytes
    buf = DeviceBuffer(room)
    full = np.zeros(room // 4, np.int32)
    full[-len(table):] = table
    buf.upload(full)
    tab = buf.ptr + room - 4 * len(table)
    out = DeviceBuffer(q.nbytes)
    if causal:
        pos = DeviceBuffer.from_numpy(np.array([base], np.int32))
        ops.qkcuda_paged_causal_attn(dev(q), out, dev(kp), dev(vp), tab, pos, n, Hq, Hkv, D, B, 0.125)
        ref = orc.batched_paged(q, kp, vp, np.tile(table, n), np.arange(n + 1, dtype=np.int32) * len(table),
                                base + 1 + np.arange(n, dtype=np.int32), Hkv, B, 0.125)
    else:
        ops.launch_batched_paged(dev(q), dev(kp), dev(vp), tab, DeviceBuffer.from_numpy(off),
                                 DeviceBuffer.from_numpy(lens), out, n, Hq, D, B, 0, 0.125, Hkv=Hkv, dtype=KVC_F16)
        ref = orc.batched_paged(q, kp, vp, table, off, lens, Hkv, B, 0.125)
    got = host(out, np.float16, q.shape).astype(np.float64)
    assert np.abs(got - ref).max() <= 2e-3


# wide: sequences far above the mean among 768 (sequence, KV head) pairs
@pytest.mark.parametrize("D,Hq,Hkv,n,wide", [(64, 14, 2, 3, 0), (64, 28, 4, 70, 0), (64, 32, 8, 96, 0), (64, 32, 8, 96, 1),
                                             (128, 8, 2, 5, 0), (128, 32, 8, 33, 0), (128, 16, 1, 7, 0),
                                             (128, 16, 1, 9, 0)])
def test_grouped_units_host_and_device_plans(orc, D, Hq, Hkv, n, wide):
    # the grouped-query units' rules on the batch (gqa_chunk_target): chunks of a twelfth of the
    # longest sequence, of a 176th of the batch, the largest target of four-wave units, and the
    # waves per unit; device lengths and host plan agree bit for bit
    say(f"grouped units D={D} Hq={Hq} Hkv={Hkv} n={n}")
    rng = np.random.default_rng(n)
    lens = rng.integers(1, 400, n).astype(np.int32)
    lens[:3] = (4200, 1549, 900)
    if wide:
        lens[4::8] = 3500
    B = 16
    nb = int(sum((int(x) + B - 1) // B for x in lens))
    alloc = BlockAllocator(nb)
    alloc.shuffle(n)
    table, off = build_tables(lens, B, alloc)
    kp, vp = (normal((nb, Hkv, B, D), 60 + i, np.float16) for i in range(2))
    q = normal((n, Hq, D), 62, np.float16)
    scale = float(1.0 / np.sqrt(D))
    got = self_planned(q, kp, vp, table, off, lens, Hkv, B, KVC_F16)
    work, nu, nr = ops.decode_plan(lens, Hq, Hkv, D, B, tab_off=off, table=table)
    out = DeviceBuffer(q.nbytes)
    ops.launch_batched_paged_planned(dev(q), dev(kp), dev(vp), dev(table), len(table), out, n, Hq, Hkv, D, B, scale,
                                     dev(work), nu, nr)
    np.testing.assert_array_equal(got, host(out, np.float16, q.shape))
    ref = orc.batched_paged(q, kp, vp, table, off, lens, Hkv, B, scale, nthreads=8)
    assert np.abs(got.astype(np.float64) - ref).max() <= tol(KVC_F16)


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 28, 4), (128, 8, 2)])
@pytest.mark.parametrize("longest", [1000, 1536, 1537])
def test_short_grouped_batches_stay_whole(orc, D, Hq, Hkv, longest):
    # up to one and a half chunks of 1024 nothing is split (a split's merge costs more than it
    # saves); both planners draw the line at the same length
    say(f"short grouped batch D={D} longest={longest}")
    lens = np.array([longest, 800, 33, 1, 700], np.int32)
    n, B = len(lens), 16
    nb = int(sum((int(x) + B - 1) // B for x in lens))
    alloc = BlockAllocator(nb)
    alloc.shuffle(longest)
    table, off = build_tables(lens, B, alloc)
    work, nu, nr = ops.decode_plan(lens, Hq, Hkv, D, B, tab_off=off, table=table)
    assert (nr == 0) == (longest <= 1536)
    kp, vp = (normal((nb, Hkv, B, D), 70 + i, np.float16) for i in range(2))
    q = normal((n, Hq, D), 72, np.float16)
    scale = float(1.0 / np.sqrt(D))
    got = self_planned(q, kp, vp, table, off, lens, Hkv, B, KVC_F16)
    out = DeviceBuffer(q.nbytes)
    ops.launch_batched_paged_planned(dev(q), dev(kp), dev(vp), dev(table), len(table), out, n, Hq, Hkv, D, B, scale,
                                     dev(work), nu, nr)
    np.testing.assert_array_equal(got, host(out, np.float16, q.shape))
    ref = orc.batched_paged(q, kp, vp, table, off, lens, Hkv, B, scale)
    assert np.abs(got.astype(np.float64) - ref).max() <= tol(KVC_F16)


# ---- prompt queries at a device position in prompt_stream_kernel (8 grouped queries and more) ----
def prompt_chunk(base, n, Hq, D):
    """The kernel's chunk of keys (prompt_stream_kernel, blocks of 16 tokens)."""
    lall = base + n
    nch = 1 if lall < 3072 else min(max(lall // (512 if D == 64 else 1024), 1), min(64, max(1, 256 // ((n + 31) // 32 * Hq))))
    return (lall // nch + 256) // 256 * 256


def split_bases(n, Hq, D):
    """Positions: whole; a chunk's edge between the first and the last query; few and many chunks."""
    edges = [b for b in range(3200, 9000) if (b + n // 2) % prompt_chunk(b, n, Hq, D) == 0]
    return [700, 3072 - n, edges[0], edges[-1] + 1, 5 * 1024]


@pytest.mark.parametrize("D,Hq,Hkv,n", [(64, 14, 2, 8), (64, 14, 2, 70), (128, 8, 2, 8), (128, 8, 2, 40), (128, 16, 1, 33)])
def test_device_position_merges_in_the_launch(orc, D, Hq, Hkv, n):
    # split prefixes: partials, arrival counter, last arriver's merge and its counter's reset, call
    # after call on one workspace, without one where the static scratch allows, and as one captured
    # launch replayed at every position with eager calls on the same workspace between
    import ctypes as C

    from kvcache_amd._native import check, lib
    say(f"device position, merge in the launch D={D} Hq={Hq} Hkv={Hkv} n={n}")
    B, L = 16, lib()
    bases = split_bases(n, Hq, D)
    assert any(b // prompt_chunk(b, n, Hq, D) != (b + n - 1) // prompt_chunk(b, n, Hq, D) for b in bases)
    nb = (max(bases) + n + B - 1) // B
    table = np.random.default_rng(n).permutation(nb).astype(np.int32)
    kp, vp = normal((nb, Hkv, B, D), 300, np.float16), normal((nb, Hkv, B, D), 301, np.float16)
    q = normal((n, Hq, D), 302, np.float16)
    scale = float(1.0 / np.sqrt(D))
    dq, dk, dv, dt = dev(q), dev(kp), dev(vp), dev(table)
    pos, out = dev(np.array([0], np.int32)), DeviceBuffer(q.nbytes)
    ws = DeviceBuffer(int(L.kvc_paged_causal_attn_dev_workspace_size(n, Hq, Hkv, D, B, KVC_F16)))
    want = {b: orc.batched_paged(q, kp, vp, table, np.zeros(n + 1, np.int32), b + 1 + np.arange(n, dtype=np.int32), Hkv, B,
                                 scale, nthreads=8) for b in bases}

    def call(stream=None, noalloc=False):
        if noalloc:
            check(L.kvc_paged_causal_attn_dev_noalloc(dq.ptr, out.ptr, dk.ptr, dv.ptr, dt.ptr, pos.ptr, n, Hq, Hkv, D, B,
                                                      C.c_float(scale), KVC_F16, stream))
        else:
            check(L.kvc_paged_causal_attn_dev(dq.ptr, out.ptr, dk.ptr, dv.ptr, dt.ptr, pos.ptr, n, Hq, Hkv, D, B,
                                              C.c_float(scale), KVC_F16, ws.ptr, ws.nbytes, stream))

    def result():
        return host(out, np.float16, q.shape)

    eager = {}
    for b in bases + bases[::-1]:
        pos.upload(np.array([b], np.int32))
        call()
        got = result()
        assert np.abs(got.astype(np.float64) - want[b]).max() <= tol(KVC_F16), b
        np.testing.assert_array_equal(got, eager.setdefault(b, got))
        if n == 8:
            call(noalloc=True)
            np.testing.assert_array_equal(result(), got)
    st, ex = C.c_void_p(), C.c_void_p()
    check(L.kvc_stream_create(C.byref(st)))
    check(L.kvc_graph_begin(st))
    call(st)
    check(L.kvc_graph_end(st, C.byref(ex)))
    for b in bases * 2:
        pos.upload(np.array([b], np.int32))
        check(L.kvc_graph_launch(ex, st))
        check(L.kvc_stream_synchronize(st))
        np.testing.assert_array_equal(result(), eager[b])
        call()  # (the same counters under another call's epoch)
        np.testing.assert_array_equal(result(), eager[b])
    check(L.kvc_graph_destroy(ex))
    check(L.kvc_stream_destroy(st))


@pytest.mark.parametrize("D", [64, 128])
def test_device_position_outside_the_keys(orc, D):
    # queries at negative positions have no keys (zero rows); a position past the planning budget
    # gives NaN rows and a report, and reads nothing
    say(f"device position negative and past the budget D={D}")
    Hq, Hkv, B, n = 8, 2, 16, 9
    kp, vp = normal((2, Hkv, B, D), 310, np.float16), normal((2, Hkv, B, D), 311, np.float16)
    q = normal((n, Hq, D), 312, np.float16)
    table, pos, out = np.array([1, 0], np.int32), dev(np.array([0], np.int32)), DeviceBuffer(q.nbytes)
    for base in (-4, -40):
        pos.upload(np.array([base], np.int32))
        ops.qkcuda_paged_causal_attn(dev(q), out, dev(kp), dev(vp), dev(table), pos, n, Hq, Hkv, D, B, 0.125)
        got = host(out, np.float16, q.shape)
        lens = np.maximum(base + 1 + np.arange(n), 0).astype(np.int32)
        want = orc.batched_paged(q, kp, vp, table, np.zeros(n + 1, np.int32), lens, Hkv, B, 0.125)
        assert np.all(got[lens == 0] == 0)
        assert np.abs(got.astype(np.float64) - want)[lens > 0].max(initial=0) <= tol(KVC_F16)
    pos.upload(np.array([63 * 1024 * B], np.int32))
    ops.qkcuda_paged_causal_attn(dev(q), out, dev(kp), dev(vp), dev(table), pos, n, Hq, Hkv, D, B, 0.125)
    assert np.isnan(host(out, np.float16, q.shape)).all()
    expect_device_error()
