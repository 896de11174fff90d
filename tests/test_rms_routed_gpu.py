"""The residual pass over routed rows: every count of them that has a form of its own, one beyond, odd widths, with and
without the token shift, at the batch sizes where the rows a workgroup walks change -- against the reference."""
import pytest
import torch

from kubernetes_cloud_amd.ops.rms_shift import Branch, rms_shift

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("T,d", [(1, 64), (5, 1028), (600, 66), (4100, 32), (9, 8192)])
@pytest.mark.parametrize("shift", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_routed_rows(top, T, d, shift, dtype):
    g = torch.Generator().manual_seed(T + top)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x, a, y, gain = r(T, d), r(T, d).to(dtype), r(T * top, d).to(dtype), torch.tensor(1.5, dtype=dtype)
    inv = torch.randperm(T * top, generator=g).view(T, top).int()
    kw = {}
    if shift:  # one entry
        fl = torch.zeros(T, dtype=torch.int32)
        fl[0] |= 1   # (one after the other: of one token they are the same element)
        fl[-1] |= 2
        kw = dict(shift=torch.rand(d, generator=g).to(dtype), prev=r(2, d), prev_idx=torch.zeros(T, dtype=torch.int32),
                  pos=torch.arange(T, dtype=torch.int32) + 3, flags=fl, state=torch.zeros(2, d),
                  slots=torch.ones(T, dtype=torch.int32))
    want = rms_shift(x, Branch(a, y, inv), 0.5, gain, 1e-5, **{k: v.clone() for k, v in kw.items()})
    c = lambda t: t.cuda()  # noqa: E731
    got = rms_shift(c(x), Branch(c(a), c(y), c(inv)), 0.5, c(gain), 1e-5, **{k: c(v) for k, v in kw.items()})
    # fp32 sums in another order; h and hs rounded once to the type
    for p, q, tol in zip(got, want, (1e-6, 1e-6 if dtype == torch.float32 else 2.0 ** -8, 1e-6 if dtype == torch.float32 else 2.0 ** -8)):
        if q is not None:
            assert (p.float().cpu() - q.float()).norm() <= tol * q.float().norm()
