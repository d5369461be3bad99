"""The DeltaNet recurrence of a prefill pass against the token-by-token recurrence in 64 bits.

The launch is called in the built library itself, so its inputs (q, k, v, beta, decay after the convolution)
are read back and the 64-bit recurrence starts from the same 32-bit values: what differs is its own rounding.
"""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sense-nova-server_amd", "libsnl.so")
# snl::launch_deltanet_prefill(const snl::DnPrefillArgs&, int M, hipStream_t), snl::dn_block_floats(int M, int n_v)
LAUNCH = "_ZN3snl23launch_deltanet_prefillERKNS_13DnPrefillArgsEiP12ihipStream_t"
BLOCK_FLOATS = "_ZN3snl15dn_block_floatsEii"
P, D = ctypes.c_void_p, 128


class Args(ctypes.Structure):  # DnPrefillArgs (csrc/kernels.h)
    _fields_ = [("proj", P), ("proj_stride", ctypes.c_int), ("lw", P), ("conv_state", P), ("state", P), ("q", P),
                ("k", P), ("v", P), ("gz", P), ("beta", P), ("decay", P), ("out", P), ("ssq", P), ("blocks", P),
                ("conv_dim", ctypes.c_int), ("n_k", ctypes.c_int), ("n_v", ctypes.c_int)]


def _inputs(torch, n_k, n_v, rows, alike, seed):
    """`alike`: positive convolution inputs and weights, so that the keys point much the same way."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    conv, heads = (2 * n_k + n_v) * D, n_v
    proj = torch.randn(rows, conv + n_v * D + 2 * heads, generator=g, device="cuda")
    w = torch.rand(conv * 4, generator=g, device="cuda") * 0.5 if alike else \
        torch.rand(conv * 4, generator=g, device="cuda") - 0.5
    if alike:
        proj[:, :2 * n_k * D] += 1.0
    a_log = torch.log(torch.rand(heads, generator=g, device="cuda") * 0.05 + 1e-3)  # decays near 1
    dt = torch.randn(heads, generator=g, device="cuda") * 0.5 - 2
    norm = 1 + 0.1 * torch.randn(D, generator=g, device="cuda")
    lw = torch.cat([w, a_log, dt, norm])
    conv_state = torch.randn(3, conv, generator=g, device="cuda")
    state = 0.1 * torch.randn(n_v, D, D, generator=g, device="cuda")
    return proj, lw, norm, conv_state, state


@pytest.mark.parametrize("alike", [False, True])
@pytest.mark.parametrize("n_k,n_v,rows", [(2, 2, 17), (2, 4, 16), (2, 6, 49), (1, 8, 3), (2, 10, 33), (16, 32, 17)])
def test_recurrence_against_64_bits(n_k, n_v, rows, alike):
    """1, 2, 3, 5 and 8 value heads a key head (a lane group of the block matrices takes one, four at a time),
    blocks of 16 tokens whole and in part.  The bound is 1.5 times what the recurrence left token by token, in
    blocks of 4 with each sum in pairs (1.3e-7 of outputs and state, keys alike or not); sums of 128 in one
    f32 chain leave 2.7e-7 of the outputs where the keys are alike."""
    import torch

    lib = ctypes.CDLL(LIB)
    launch, floats = getattr(lib, LAUNCH), getattr(lib, BLOCK_FLOATS)
    launch.argtypes, floats.restype = [ctypes.POINTER(Args), ctypes.c_int, P], ctypes.c_size_t
    errors = []
    for seed in range(4):
        proj, lw, norm, conv_state, state0 = _inputs(torch, n_k, n_v, rows, alike, seed)
        z = lambda *s: torch.zeros(*s, device="cuda")  # noqa: E731
        buf = dict(conv_state=conv_state, state=state0.clone(), q=z(rows, n_k, D), k=z(rows, n_k, D), v=z(rows, n_v, D),
                   gz=z(rows, n_v, D), beta=z(rows, n_v), decay=z(rows, n_v), out=z(rows, n_v, D), ssq=z(rows, n_v, 8),
                   blocks=z(floats(rows, n_v)))
        a = Args(proj=proj.data_ptr(), proj_stride=proj.shape[1], lw=lw.data_ptr(), conv_dim=(2 * n_k + n_v) * D, n_k=n_k,
                 n_v=n_v, **{n: t.data_ptr() for n, t in buf.items()})
        print(f"recurrence {n_k}/{n_v} heads, {rows} rows, alike {alike}, seed {seed}", flush=True)
        assert launch(ctypes.byref(a), rows, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        q, k = (buf[n].double().repeat_interleave(n_v // n_k, 1) for n in "qk")
        v, beta, decay, s = buf["v"].double(), buf["beta"].double(), buf["decay"].double(), state0.double()
        out = []
        for t in range(rows):
            s = s * decay[t][:, None, None]
            u = beta[t][:, None] * (v[t] - (k[t][:, :, None] * s).sum(1))
            s = s + k[t][:, :, None] * u[:, None, :]
            out.append((q[t][:, :, None] * s).sum(1))
        out = torch.stack(out)
        ref = out * norm.double() * buf["gz"].double()
        errors.append([float((buf["out"].double() - ref).norm() / ref.norm()),
                       float((buf["state"].double() - s).norm() / s.norm())])
        ssq = buf["ssq"].double().sum(2)  # sums of squares of 128 outputs, 16 of a group in one f32 sum
        assert float(((ssq - (out * out).sum(2)) / (out * out).sum(2)).abs().max()) < 1e-5
    mean = [sum(e[i] for e in errors) / len(errors) for i in (0, 1)]
    print(f"errors {mean[0]:.2e} (outputs) {mean[1]:.2e} (state)", flush=True)
    assert max(mean) < 2e-7
