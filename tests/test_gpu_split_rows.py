"""Every split of a row's live units over waves (1, 2 and 4, chosen by the launch's
rows: B H 2 ceil(T/64) against 2048 and 1024 for fp32, half of that for the 2-byte
types) against the float64 oracle, at D = 128, where the passes' LDS and register
layouts differ by the split.  T = 70 leaves a ragged last unit; some keys are
masked.  Tolerances as in test_gpu_parity.py."""

import numpy as np
import pytest
import torch

import screening_oracle as O
from helpers import correlated_qkv, errors, head_sum_err, np64, rel_err, rw64

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 5e-3}


@pytest.mark.parametrize("drop", [(), (0.25, 99)], ids=["plain", "dropout"])
@pytest.mark.parametrize("B", [20, 60, 100, 132])  # 16 B rows: S = 4, 4 / 2, 2 / 1, 1 (fp32 / 2-byte)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
def test_split_rows_d128(dtype, B, drop):
    from multiscreen import ops
    T, H, D = 70, 4, 128
    r, w = [1.1, 1.3, 1.6, 1.2], [20.0, 40.0, 1e4, 70.0]
    q, k, v = correlated_qkv(B, T, T, H, D, seed=B, dtype=dtype, rho=0.45)
    dy = torch.randn(B, T, H, D, generator=torch.Generator().manual_seed(B + 1)).to(dtype)
    kpm = torch.zeros(B, T, dtype=torch.bool)
    kpm[:, 11::17] = True
    rg, wg = torch.tensor(r, device=DEV), torch.tensor(w, device=DEV)
    args = [x.to(DEV) for x in (q, k, v)]
    y, hnorm, bits = ops.fwd_raw(*args, rg, wg, True, 1e-8, kpm.to(DEV), *drop)
    grads = ops.bwd_raw(*args, rg, wg, True, 1e-8, y, hnorm, bits, dy.to(DEV), kpm.to(DEV), *drop)
    ref_args = (np64(q), np64(k), np64(v), rw64(r), rw64(w))
    kw = {"key_padding_mask": kpm.numpy(), "dropout": drop or None}
    ref = (O.forward(*ref_args, True, **kw),) + tuple(O.backward(*ref_args, np64(dy), True, **kw))
    for name, got, want in zip(("y", "dq", "dk", "dv", "dr", "dw"), (y, *grads), ref):
        e = rel_err(np64(got), want)
        assert e <= TOL[dtype], f"{name}: rel err {e:.3e} > {TOL[dtype]}"


@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.float32, 64), (torch.bfloat16, 64), (torch.float16, 32)])
def test_rows_of_few_units(dtype, D):
    """Rows and columns with 0, 1, 2, 3, 4 and more live units under a split over
    four waves: those of one unit are wave 0's alone, others add up as many parts as
    have units.  Query unit u repeats the keys of u mod 7 key units, all else is far
    below the threshold."""
    from multiscreen import ops
    B, T, H, r, w = 2, 320, 2, [6.0, 7.0], [1e4, 1e5]
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(B, T, H, D, generator=g) for _ in range(3))
    for u in range(10):
        for n in range(min(u, u % 7)):  # key unit n, earlier than the query unit
            q[:, 32 * u + n] = k[:, 32 * n + u] + 0.3 * torch.randn(B, H, D, generator=g)
    q, k, v = (x.to(dtype) for x in (q, k, v))
    dy = torch.randn(B, T, H, D, generator=g).to(dtype)
    rg, wg = torch.tensor(r, device=DEV), torch.tensor(w, device=DEV)
    args = [x.to(DEV) for x in (q, k, v)]
    y, hnorm, bits = ops.fwd_raw(*args, rg, wg, True, 1e-8, None)
    grads = ops.bwd_raw(*args, rg, wg, True, 1e-8, y, hnorm, bits, dy.to(DEV))
    ref_args = (np64(q), np64(k), np64(v), rw64(r), rw64(w))
    near = O.live_pairs(*ref_args[:2], *ref_args[3:], True)
    counts = {len(set(near["j"][(near["i"] // 32 == u) & (near["b"] == 0) & (near["h"] == 0)] // 32)) for u in range(10)}
    assert {0, 1, 2, 3, 4, 5} <= counts, counts
    _, ref, P = O.sparse_forward_backward(*ref_args, np64(dy), True)
    for name, got, want in zip(("dq", "dk", "dv"), grads, ref):
        e = errors(np64(got), want)
        assert e["max"] <= TOL[dtype] and e["fro"] <= TOL[dtype], f"{name}: {e}"
    for name, got, want, scale in (("dr", grads[3], ref[3], P["dr_abs"]), ("dw", grads[4], ref[4], P["dw_abs"])):
        e = head_sum_err(np64(got), want, scale)
        assert e <= TOL[dtype], f"{name}: per-head error {e:.3e}"
