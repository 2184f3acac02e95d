"""GPU: batches around one and two matrices a CU, where a plan's tiles and the LDS its
workgroups claim change (256 CUs in 8 XCDs: 256 and 512 matrices, fewer where several groups
go round the XCDs), and beyond, of one element type and of several. Every member is bit for
bit clm_expm_*'s result on the same input; two plans on two streams do not disturb each other.
"""
import numpy as np
import pytest
import torch

import calaman_g_amd as cg
from calaman_g_amd.expm import BatchPlan, expm_cm

pytestmark = pytest.mark.gpu

TYPES = [torch.float32, torch.float64, torch.complex64, torch.complex128]


def _inputs(dtype, orders, dev):
    """per order: the matrix (column-major) and its exponential by the single call"""
    out = {}
    for n in orders:
        gen = torch.Generator(device="cuda").manual_seed(n)
        a = torch.randn((n, n), generator=gen, device=dev, dtype=dtype)
        a = a * (3.0 / float(a.abs().sum(1).max()))
        e = torch.empty_like(a)
        work = torch.empty(cg.expm_buffer_size(n, dtype), dtype=torch.uint8, device=dev)
        assert expm_cm(n, a, n, e, n, work)[0] == 0
        out[n] = (a, e)
    return out


@pytest.mark.parametrize("types", [[t] for t in TYPES] + [TYPES[:1] + TYPES[2:3], TYPES],
                         ids=["f32", "f64", "c64", "c128", "f32+c64", "all"])
@pytest.mark.parametrize("count,lo,hi", [(1, 33, 33), (40, 100, 210), (255, 2, 40), (256, 33, 64),
                                         (257, 20, 70), (300, 40, 44), (512, 2, 40), (513, 33, 64),
                                         (577, 2, 50), (900, 2, 12)])
def test_members_are_the_single_results(dev, types, count, lo, hi):
    rng = np.random.default_rng(count)
    orders = sorted(set(rng.integers(lo, hi + 1, size=9).tolist()))
    known = {t: _inputs(t, orders, dev) for t in types}
    picks = [(types[int(rng.integers(len(types)))], int(rng.choice(orders))) for _ in range(count)]
    entries = [(n, known[t][n][0], n, torch.empty_like(known[t][n][0]), n) for t, n in picks]
    print(f"batch of {count}, orders {lo}..{hi}, {len(types)} types", flush=True)
    plan = BatchPlan(entries)
    work, res = plan.workspace(), plan.results_buffer()
    assert plan.launch(work, res) == 0
    assert all(r["status"] == 0 for r in BatchPlan.decode_results(res))
    for (t, n), (_, _, _, e, _) in zip(picks, entries):
        want = known[t][n][1]
        assert torch.equal(e.view(torch.uint8), want.view(torch.uint8)), (t, n)


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("count,lo,hi", [(200, 33, 64), (260, 4, 40)])
def test_two_plans_on_two_streams(dev, dtype, count, lo, hi):
    known = _inputs(dtype, range(lo, hi + 1, 5), dev)
    orders = list(known)
    torch.cuda.synchronize()
    runs = []
    for k in range(2):
        picks = [orders[(i + k) % len(orders)] for i in range(count)]
        entries = [(n, known[n][0], n, torch.empty_like(known[n][0]), n) for n in picks]
        plan = BatchPlan(entries)
        runs.append((plan, plan.workspace(), torch.cuda.Stream(), picks, entries))
    torch.cuda.synchronize()
    for plan, work, stream, _, _ in runs:
        assert plan.launch(work, stream=stream) == 0
    torch.cuda.synchronize()
    for _, _, _, picks, entries in runs:
        for n, (_, _, _, e, _) in zip(picks, entries):
            assert torch.equal(e.view(torch.uint8), known[n][1].view(torch.uint8)), n


def test_the_tuner_times_complex128_with_a_cu_to_itself(dev):
    """tile 2 is a launch of its own for complex128 (one workgroup a CU), tile 3 is not"""
    saved = cg.batched_tuning(torch.complex128)
    try:
        table, ms = cg.batched_autotune(torch.complex128, nmax=40)
        for b in (0, 1):
            assert all(ms[b][t] > 0 for t in (0, 1, 2, 4)) and ms[b][3] == 0
            assert ms[b][table[b]] == min(t for t in ms[b] if t > 0)
    finally:
        cg.set_batched_tuning(torch.complex128, saved)
