"""fp16 rows around the length 2^-15, where 1/|x| leaves fp16's powers of two.

The fp16 kernels split 1/|x| into a power of two, which goes to the row, and a
rest, which goes to the pair weight; below 2^-15 the power of two takes two
factors.  Each 32-row unit of one tensor here holds rows of one length, 2^-13
to 2^-17 (components +-|x|/8, exact in fp16), so a unit has no shorter row that
would bring the second factor in for all of it.  Outputs are compared with the
float64 oracle, the gradient of the short rows times |x| (it is the gradient of
the unit vector over |x|).  Tolerance as in the other fp16 tests: 5e-3."""

import numpy as np
import pytest
import torch

import screening_oracle as O
from helpers import errors, head_sum_err, np64, rel_err, rw64

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = 5e-3


@pytest.mark.parametrize("B", [1, 40], ids=["shared_rows", "one_wave_a_row"])
@pytest.mark.parametrize("short", ["q", "k", "v"])
def test_rows_around_two_to_the_minus_15(short, B):
    from multiscreen import ops
    T, H, D = 192, 2, 64
    r, w = [1.1, 1.3], [40.0, 1e4]
    g = torch.Generator().manual_seed(21)
    base = torch.randn(B, T, H, D, generator=g)
    x = {n: torch.sign(0.6 * base + 0.8 * torch.randn(B, T, H, D, generator=g)) for n in "qk"}
    x["v"] = torch.sign(torch.randn(B, T, H, D, generator=g))
    length = torch.tensor([2.0 ** e for e in (-15, -14, -16, -15, -17, -13)]).repeat_interleave(32).view(1, T, 1, 1)
    x[short] = x[short] * (length / 8.0)
    dy = (0.05 * torch.randn(B, T, H, D, generator=g)).half()
    q, k, v = (x[n].half() for n in "qkv")
    assert torch.equal(x[short].half().float(), x[short])
    rg, wg = torch.tensor(r, device=DEV), torch.tensor(w, device=DEV)
    args = [t.to(DEV) for t in (q, k, v)]
    y, hnorm, bits = ops.fwd_raw(*args, rg, wg, True, 1e-8, None)
    grads = ops.bwd_raw(*args, rg, wg, True, 1e-8, y, hnorm, bits, dy.to(DEV))
    rr, ww = rw64(r), rw64(w)
    ref = (O.forward(np64(q), np64(k), np64(v), rr, ww, True),) + tuple(
        O.backward(np64(q), np64(k), np64(v), rr, ww, np64(dy), True))
    for name, got, want in zip(("y", "dq", "dk", "dv"), (y, *grads), ref):
        got, want = np64(got), np.asarray(want)
        if name == "d" + short:
            got, want = got * np64(length), want * np64(length)
        e = rel_err(got, want)
        print(f"fp16 rows {short} B={B} {name}: rel err {e:.3e}", flush=True)
        assert e <= TOL, f"{name}: rel err {e:.3e} > {TOL}"


@pytest.mark.parametrize("B", [1, 40], ids=["shared_rows", "one_wave_a_row"])
@pytest.mark.parametrize("dy_rms,r,size", [(1e-5, [8.0, 30.0], 2.0 ** -9), (2000.0, [2.0, 4.0], 1.0)],
                         ids=["small_dy", "large_dy"])
def test_gradients_at_the_ends_of_the_range(dy_rms, r, size, B):
    """ds = 2 r a m dP is an fp16 operand of dq and dk.  At dy about 1e-5 the
    plain product a m dP is about 1e-6, 17 of fp16's smallest steps (a step is
    6e-8, so its rounding is 2% of it); 2r takes it out of there.  What is left
    is dh's own rounding to fp16: 0.29 steps of 168, 2e-3.  At dy about 2000
    the largest ds is above 32752, where another factor 2 is past the range.
    q, k and v are short for the small dy, so that dq, dk and dv are not."""
    from multiscreen import ops
    T, H, D = 160, 2, 64
    w = [24.0, 40.0]
    g = torch.Generator().manual_seed(5)
    centre = torch.randn(1, 1, H, D, generator=g)
    noise = torch.tensor([(0.6 / x) ** 0.5 for x in r]).view(1, 1, H, 1)  # 1 - s about 0.6/r, a about 0.4
    q, k = ((size * (centre + noise * torch.randn(B, T, H, D, generator=g))).half() for _ in range(2))
    v = (size * torch.randn(B, T, H, D, generator=g)).half()
    dy = (dy_rms * torch.randn(B, T, H, D, generator=g)).half()
    rg, wg = torch.tensor(r, device=DEV), torch.tensor(w, device=DEV)
    args = [t.to(DEV) for t in (q, k, v)]
    y, hnorm, bits = ops.fwd_raw(*args, rg, wg, True, 1e-8, None)
    grads = ops.bwd_raw(*args, rg, wg, True, 1e-8, y, hnorm, bits, dy.to(DEV))
    _, ref, P = O.sparse_forward_backward(np64(q), np64(k), np64(v), rw64(r), rw64(w), np64(dy), True)
    for name, got, want in zip(("dq", "dk", "dv"), grads, ref):
        e = errors(np64(got), want)
        print(f"fp16 dy {dy_rms} B={B} {name}: {e['max']:.3e} {e['fro']:.3e}", flush=True)
        assert e["max"] <= TOL and e["fro"] <= TOL, f"{name}: {e}"
    for name, got, want, scale in (("dr", grads[3], ref[3], P["dr_abs"]), ("dw", grads[4], ref[4], P["dw_abs"])):
        e = head_sum_err(np64(got), want, scale)
        assert e <= TOL, f"{name}: per-head error {e:.3e}"
