"""The int8 screen (2-byte inputs, heads whose window is at least 4096
positions, launches of one wave a row over at least 7000 positions at D = 64,
4096 at D = 128) against the float64 live-pair oracle.

Every unit with a live pair must be marked; the live pass takes back the bits
of units without one, so in int8 heads a marked unit holds a pair with
1 - r(1 - s) > 0 up to the fp32 rounding of s (2e-5 in s).  Lengths are ragged,
windows lie on both sides of 4096 (both operand types in one launch), and the
rows include ones that quantise badly: one component 40 times the others', zero
rows, rows of length 1e-6 and 1e4.  The backward walks the bitmap that is left:
y and all gradients meet the 2-byte types' tolerance, dq and dk times |q| and |k|
(the gradients of the unit vectors), so that a row of length 1e-6 weighs as much
as any other.  Left out: in fp16, dq of the rows of length 1e4 times the others',
about ten of fp16's smallest steps."""

import numpy as np
import pytest
import torch

import screening_oracle as O
from helpers import errors, head_sum_err, np64, rel_err, rw64

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {torch.bfloat16: 2e-2, torch.float16: 5e-3}


def _units(bits, B, H, Tq, Tk):
    nqu, nku = 2 * ((Tq + 63) // 64), 2 * ((Tk + 63) // 64)
    words = (nku + 31) // 32
    b = bits.cpu().numpy().view(np.uint32)[:B * H * nqu * words].reshape(B, H, nqu, words)
    out = np.zeros((B, H, nqu, words * 32), dtype=bool)
    for e in range(32):
        out[..., e::32] = (b >> e) & 1
    return out[..., :nku]


@pytest.mark.parametrize("dtype,D,Tq,Tk,causal,padded", [
    (torch.bfloat16, 64, 7013, 7013, True, False),
    (torch.float16, 64, 7013, 7013, True, True),
    (torch.bfloat16, 64, 7040, 2100, False, True),
    (torch.float16, 64, 7000, 7000, False, False),
    (torch.bfloat16, 128, 4131, 4131, True, True),
    (torch.float16, 128, 4100, 4500, False, False),
])
def test_int8_screen_marks_the_live_units(dtype, D, Tq, Tk, causal, padded):
    from multiscreen import ops
    B, H = 1, 8
    g = torch.Generator().manual_seed(Tq + D)
    q, k, v = (torch.randn(B, t, H, D, generator=g) for t in (Tq, Tk, Tk))
    k[:, 7::97, :, 5] *= 40.0
    q[:, 11::89, :, 5] *= 40.0
    k[:, 64:96] *= 1e-6
    k[:, 130::131] = 0.0
    q[:, 200:240] *= 1e-6
    q[:, 300:332] *= 1e4
    k[:, 1000:1016] = q[:, 1010:1026]
    kpm = None
    if padded:
        kpm = torch.zeros(B, Tk, dtype=torch.bool)
        kpm[:, Tk - Tk // 5:] = True
        kpm[:, 1004] = True
    q, k, v = (x.to(dtype) for x in (q, k, v))
    # dq and dk of the rows of length 1e-6 stay in fp16's range at this dy
    dy = (0.05 * torch.randn(B, Tq, H, D, generator=g)).to(dtype)
    r = [2.0, 1.7, 2.2, 2.0, 1.05, 1.9, 2.0, 3.0] if D > 64 else [2.0, 1.9, 2.2, 2.0, 2.1, 1.9, 2.0, 3.0]
    w = [4095.5, 4096.0, 4100.0, 1e5, 5000.0, 300.0, float("inf"), 4500.0]
    rg, wg = torch.tensor(r, device=DEV), torch.tensor(w, device=DEV)
    args = [x.to(DEV) for x in (q, k, v)]
    kd = None if kpm is None else kpm.to(DEV)
    y, hnorm, bits = ops.fwd_raw(*args, rg, wg, causal, 1e-8, kd)
    grads = ops.bwd_raw(*args, rg, wg, causal, 1e-8, y, hnorm, bits, dy.to(DEV), kd)
    units = _units(bits, B, H, Tq, Tk)

    rr, ww = rw64(r), np.minimum(rw64(w), 1e30)
    kp = None if kpm is None else kpm.numpy()
    slack = 2e-5
    near = O.live_pairs(np64(q), np64(k), 1.0 / (1.0 / rr + slack), ww, causal, key_padding_mask=kp)
    a = 1.0 - rr[near["h"]] * (1.0 - near["s"])
    live = {n: x[a > 0.0] for n, x in near.items()}
    missed = ~units[live["b"], live["h"], live["i"] // 32, live["j"] // 32]
    assert len(live["i"]) > 0 and not missed.any(), f"{int(missed.sum())} live pairs in unmarked units"
    cover = np.zeros_like(units)
    cover[near["b"], near["h"], near["i"] // 32, near["j"] // 32] = True
    int8 = [h for h in range(H) if w[h] >= 4096]
    stray = (units & ~cover)[:, int8]
    assert not stray.any(), f"{int(stray.sum())} marked units hold no live pair"

    yref, gref, P = O.sparse_forward_backward(np64(q), np64(k), np64(v), rr, ww, np64(dy), causal,
                                              key_padding_mask=kp, pairs=live)
    assert rel_err(np64(y), yref) <= 2e-2
    assert rel_err(np64(grads[2]), gref[2]) <= 2e-2
    tol = TOL[dtype]
    for name, x, got, want in (("dq", q, grads[0], gref[0]), ("dk", k, grads[1], gref[1])):
        length = np.linalg.norm(np64(x), axis=-1, keepdims=True)
        got, want = np64(got) * length, want * length
        if name == "dq" and dtype == torch.float16:
            got[:, 300:332] = want[:, 300:332] = 0.0
        e = errors(got, want)
        print(f"int8 screen {dtype} D={D} {name}: {e['max']:.3e} {e['fro']:.3e}", flush=True)
        assert e["max"] <= tol and e["fro"] <= tol, f"{name}: {e}"
    for name, got, want, scale in (("dr", grads[3], gref[3], P["dr_abs"]), ("dw", grads[4], gref[4], P["dw_abs"])):
        e = head_sum_err(np64(got), want, scale)
        assert e <= tol, f"{name}: per-head error {e:.3e} > {tol}"


@pytest.mark.parametrize("D,T", [(64, 7040), (128, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_pairs_at_the_threshold_keep_their_unit(dtype, D, T):
    """Each head's r is the largest fp32 value at which its most similar pair is
    live in float64 (a = 1 - r(1 - s) below 2e-7): the fp32 a of such a pair is
    as often 0 as not, and its unit stays marked either way."""
    from multiscreen import ops
    H = 16
    for seed in range(3):
        g = torch.Generator(device=DEV).manual_seed(seed)
        q, k, v = (torch.randn(1, T, H, D, device=DEV, generator=g).to(dtype) for _ in range(3))
        later = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)
        r, at = [], []
        for h in range(H):
            qh, kh = (torch.nn.functional.normalize(x[0, :, h].double(), dim=-1) for x in (q, k))
            s = (qh @ kh.T).masked_fill_(later, -1.0)
            at.append(divmod(int(s.argmax()), T))
            bound = 1.0 / (1.0 - float(s.max()))
            x = np.float32(bound)
            r.append(float(x if x < bound else np.nextafter(x, np.float32(0))))
        rg, wg = torch.tensor(r, device=DEV), torch.full((H,), 1e5, device=DEV)
        y, hnorm, bits = ops.fwd_raw(q, k, v, rg, wg, True, 1e-8, None)
        units = _units(bits, 1, H, T, T)
        missed = [h for h, (i, j) in enumerate(at) if not units[0, h, i // 32, j // 32]]
        assert not missed, f"heads {missed} of {H}: the unit of the live pair is not marked"
