"""The hand-scheduled GEMM tile behind the projections and their gradients, against float64: contractions that end
inside a 64-deep stage (and inside its first), rows and columns around one tile, all three sizes of the
tile, both weight layouts and element types, with and without the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (rows, model width, heads, head_dim).  On 256 CUs the tile is 224 x 256 for K and V of 6404 and 12700 rows and dX of
# 2300 rows x 4104, 256 x 256 for K and V of 8190 rows and dX of 4090 x 4096, and 256 x 128 for the others
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("w_in_major", [True, False])
@pytest.mark.parametrize("M,Dm,H,D", [(1, 136, 2, 128), (33, 64, 9, 32), (100, 1000, 3, 128), (255, 32, 2, 128),
                                      (257, 512, 4, 128), (300, 264, 10, 16), (1601, 72, 4, 128), (2300, 136, 32, 128),
                                      (2300, 4104, 2, 128), (6404, 72, 8, 128), (12700, 32, 8, 128),
                                      (8190, 136, 8, 128), (4090, 4096, 1, 128)])
def test_projection_and_gradients(dtype, w_in_major, M, Dm, H, D):
    from lv_xattn import ops
    g = torch.Generator(device=DEV).manual_seed(M * 7 + Dm)
    N = H * D

    def normal(*shape, std=1.0):
        return torch.empty(*shape, dtype=dtype, device=DEV).normal_(0, std, generator=g)

    # a result is an exact product sum rounded once to 16 bits (half an ulp: 2^-9 or 2^-12 of the value), so the
    # relative 2-norm error stays below that; fp32 accumulation is two orders below it
    bound = 2 ** -9 if dtype == torch.bfloat16 else 2 ** -12

    def check(got, ref, what, factor=1.0):
        rel = ((got.double() - ref).norm() / ref.norm()).item()
        assert rel <= factor * bound, f"{what}: relative error {rel:.2e}"

    x = normal(1, M, Dm)
    shape = (Dm, N) if w_in_major else (N, Dm)
    w = [normal(*shape, std=Dm ** -0.5) for _ in range(2)]
    wd = [t.double() if w_in_major else t.double().T.contiguous() for t in w]
    k, v = ops.kv_proj(x, *w, H, w_in_major)
    raw = [x[0].double() @ t for t in wd]
    for got, ref, what in ((k, raw[0], "K"), (v, raw[1], "V")):
        check(got.transpose(1, 2).reshape(M, N), ref, what)
    d = [normal(1, M, H, D).transpose(1, 2) for _ in range(2)]
    dd = [t.transpose(1, 2).reshape(M, N).double() for t in d]
    check(ops.dx_vis(*d, *w, w_in_major)[0], dd[0] @ wd[0].T.contiguous() + dd[1] @ wd[1].T.contiguous(), "dX")
    for got, ref, what in zip(ops.dw_kv(x, *d, w_in_major), dd, ("dW_k", "dW_v")):
        ref = x[0].double().T.contiguous() @ ref
        check(got, ref if w_in_major else ref.T, what)
    if D == 128:
        wn = (1 + 0.2 * normal(128)).to(dtype)
        k, v, k_raw, rstd = ops.kv_proj(x, *w, H, w_in_major, wn, 1e-5, True)
        heads = raw[0].view(M, H, 128)
        r = torch.rsqrt(heads.square().mean(-1, keepdim=True) + 1e-5)
        check(k_raw.transpose(1, 2)[0], heads, "raw K")
        check(v.transpose(1, 2).reshape(M, N), raw[1], "V beside the norm")
        check(k.transpose(1, 2)[0], wn.double() * heads * r, "K", factor=3.0)       # three roundings
        check(rstd.view(M, H, 1), r, "r", factor=1.0)
