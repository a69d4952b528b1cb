"""GPU parity of the rotary embedding kernels against the CPU checker,
through the C ABI.  Tolerance: the reference's own acceptance interval
(tests/kernel/rope.cc:57,95-137): every value within ref (1 +- eps) +- eps with
eps = 2 x the type's epsilon (fp32 2^-23, fp16 2^-10, bf16 2^-7)."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa, synth
from . import helpers as H
from .test_oracle_rope import reference_case, within_reference_interval

pytestmark = pytest.mark.gpu

EPS = {"fp32": 2.0 ** -23, "fp16": 2.0 ** -10, "bf16": 2.0 ** -7}


def _tile(x, dtype):
    t, f = H.rounded(x, dtype)
    return t.cuda(), f


def _run(sin, cos, src, dtype, backward=False, inplace=False):
    S, sf = _tile(sin, dtype)
    C, cf = _tile(cos, dtype)
    X, xf = _tile(src, dtype)
    D = X if inplace else torch.full_like(X, float("nan"))
    hip_sdpa.rope(S, C, X, D, backward=backward)
    torch.cuda.synchronize()
    return H.to_np(D), sf, cf, xf


@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("m,n", [(0, 5), (1, 10), (10, 100)])
def test_reference_kernel_test_cases(oracle, dtype, m, n):
    print("case rope reference", dtype, m, n, flush=True)
    sin, cos, src = reference_case(m, n)
    got, sf, cf, xf = _run(sin, cos, src, dtype)
    if m == 0:
        return
    assert within_reference_interval(got, sf, cf, xf, 2 * EPS[dtype])


@pytest.mark.parametrize("dtype", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("backward", [False, True])
@pytest.mark.parametrize("shape", [
    (64, 1024, 2, 8),       # Llama: head 128, seq 1024, batch 2 | 8 heads: sin is [64, 1024, 2]
    (32, 333, 1, 5),        # m a multiple of 4, odd sizes
    (5, 77, 1, 3),          # m odd: one pair per thread
    (2, 3, 1, 1),
])
def test_against_checker(oracle, dtype, backward, shape):
    print("case rope", dtype, backward, shape, flush=True)
    half, seq, batch, n = shape
    m = half * seq * batch
    ang = synth.randn(70, 0, m).astype(np.float64) * 2.0
    sin, cos = np.sin(ang).astype(np.float32), np.cos(ang).astype(np.float32)
    src = synth.randn(71, 0, 2 * m * n)
    got, sf, cf, xf = _run(sin, cos, src, dtype, backward=backward)
    want = oracle.rope(sf, cf, xf, backward=backward)
    assert np.all(np.isfinite(got))
    err = np.abs(got.reshape(-1) - want.reshape(-1))
    assert np.all(err <= 2 * EPS[dtype] * (np.abs(want.reshape(-1)) + 1.0))
    # in place gives the same bits
    again, _, _, _ = _run(sin, cos, src, dtype, backward=backward, inplace=True)
    assert np.array_equal(again, got)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_unaligned_addresses_and_round_trip(oracle, dtype):
    """Tensors that start one element into an allocation take the
    pair-per-thread kernel; backward(forward(x)) returns x for unit (sin, cos)
    up to the two roundings."""
    m, n = 64 * 50, 6
    ang = synth.randn(72, 0, m).astype(np.float64)
    sin, cos = np.sin(ang).astype(np.float32), np.cos(ang).astype(np.float32)
    src = synth.randn(73, 0, 2 * m * n)
    S, sf = _tile(np.concatenate([[0.0], sin]), dtype)
    C, cf = _tile(np.concatenate([[0.0], cos]), dtype)
    X, xf = _tile(np.concatenate([[0.0], src]), dtype)
    Y = torch.zeros_like(X)
    Z = torch.zeros_like(X)
    hip_sdpa.rope(S[1:], C[1:], X[1:], Y[1:])
    hip_sdpa.rope(S[1:], C[1:], Y[1:], Z[1:], backward=True)
    torch.cuda.synchronize()
    want = oracle.rope(sf[1:], cf[1:], xf[1:])
    got = H.to_np(Y)[1:]
    assert np.all(np.abs(got - want) <= 2 * EPS[dtype] * (np.abs(want) + 1.0))
    assert H.to_np(Y)[0] == 0.0 and H.to_np(Z)[0] == 0.0
    back = H.to_np(Z)[1:]
    assert np.all(np.abs(back - xf[1:]) <= 6 * EPS[dtype] * (np.abs(xf[1:]) + 1.0))


def test_errors():
    x = torch.zeros(8, device="cuda")
    s = torch.zeros(2, device="cuda")
    fn = hip_sdpa.lib().nntile_hip_rope_fp32
    assert fn(None, -1, 1, s.data_ptr(), s.data_ptr(), x.data_ptr(), x.data_ptr()) == hip_sdpa.EINVAL
    assert fn(None, 2, 2, None, s.data_ptr(), x.data_ptr(), x.data_ptr()) == hip_sdpa.EINVAL
    assert fn(None, 0, 7, None, None, None, None) == hip_sdpa.OK
    with pytest.raises(hip_sdpa.SdpaError):
        hip_sdpa.rope(s, s, x[:6], x[:6])       # 6 is not a multiple of 2 m = 4


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("m,n", [(4, 1), (1020, 3), (1024, 5), (262148, 9), (1048576, 4)])
@pytest.mark.parametrize("backward", [False, True])
def test_columns_per_thread(dtype, m, n, backward):
    """One and two columns a thread, rows that end inside a workgroup, an odd
    number of columns: against torch in fp32."""
    print("case rope columns", dtype, m, n, backward, flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    dt = H.TORCH_DT[dtype]
    x = torch.randn(n, m, 2, generator=g, device="cuda").to(dt)
    sin, cos = (torch.randn(m, generator=g, device="cuda").to(dt) for _ in range(2))
    y = torch.full_like(x, float("nan"))
    hip_sdpa.rope(sin, cos, x, y, backward=backward)
    s, c = sin.float() * (-1 if backward else 1), cos.float()
    a, b = x[..., 0].float(), x[..., 1].float()
    want = torch.stack((c * a - s * b, s * a + c * b), dim=-1)
    torch.cuda.synchronize()
    bound = 2 * torch.finfo(dt).eps * (x.float().abs().sum(-1, keepdim=True)
                                       * (s.abs() + c.abs())[None, :, None])
    assert ((y.float() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("backward", [False, True])
@pytest.mark.parametrize("m", [4, 8, 16, 64, 252, 1020, 1024, 1028, 4100])
@pytest.mark.parametrize("n", [1, 3, 258, "many"])
def test_columns_of_any_length_give_the_bits_of_the_pairwise_kernel(dtype, backward, m, n):
    """Four pairs a thread, one column or two ("many": an odd number of them),
    columns shorter and longer than a workgroup and no multiple of it, against
    one pair a thread, which addresses off by one pair take."""
    if n == "many":
        n = (1 << 22) // m | 1
    print("case rope columns", dtype, backward, m, n, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m * 1000 + n)
    dt = H.TORCH_DT[dtype]
    sin, cos = (torch.randn(m, generator=g, device="cuda").to(dt) for _ in range(2))
    size = 2 * m * n
    src = torch.randn(size + 2, generator=g, device="cuda").to(dt)
    out = []
    for shift in (0, 2):
        x = src[shift:shift + size]
        x.copy_(src[:size].clone())
        y = torch.full((size + 18,), 7.0, dtype=dt, device="cuda")
        hip_sdpa.rope(sin, cos, x, y[shift + 8:shift + 8 + size], backward=backward)
        torch.cuda.synchronize()
        assert (y[:shift + 8] == 7.0).all() and (y[shift + 8 + size:] == 7.0).all()
        out.append(y[shift + 8:shift + 8 + size].clone())
    assert torch.equal(out[0], out[1])
