"""Grouped-GEMM microbench at Qwen3-30B bench shapes (gpurun)."""
import sys, os
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import torch, time
from automodel_amd.ops._backend import hip_ops
from automodel_amd.ops.grouped_gemm import make_group_plan

ops = hip_ops()
E, T, K8 = 128, 16384, 8
M = T * K8
H, I = 2048, 768
counts = torch.full((E,), M // E, dtype=torch.int32, device="cuda")
x = torch.randn(M, H, device="cuda", dtype=torch.bfloat16)
g = torch.randn(M, I, device="cuda", dtype=torch.bfloat16)
w = torch.randn(E, I, H, device="cuda", dtype=torch.bfloat16) * 0.02
offs, tm, ntl = make_group_plan(counts, M)

def timeit(name, fn, flops, iters=10):
    for _ in range(3): fn()
    torch.cuda.synchronize(); t0 = time.perf_counter()
    for _ in range(iters): fn()
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / iters
    print(f"{name}: {dt*1e3:.2f} ms  {flops/dt/1e12:.0f} TF/s")

fl = 2 * M * I * H
timeit("nt  (y=x@wT)", lambda: ops.grouped_gemm_nt(x, w, offs, tm, ntl), fl)
offs_b, tm_b, ntl_b = ops.build_group_plan(counts, M, 256)
w3 = torch.randn(E, 1024, H, device="cuda", dtype=torch.bfloat16) * 0.02
fl3 = 2 * M * 1024 * H
timeit("nt-big 256x256 (N=1024)", lambda: ops.grouped_gemm_nt(x, w3, offs_b, tm_b, ntl_b, 256), fl3)
y_big = ops.grouped_gemm_nt(x, w3, offs_b, tm_b, ntl_b, 256)
y_ref = ops.grouped_gemm_nt(x, w3, offs, tm, ntl)
print("big-vs-128 maxdiff:", float((y_big.float()-y_ref.float()).abs().max()))
timeit("nn  (dx=g@w)", lambda: ops.grouped_gemm_nn(g, w, offs, tm, ntl), fl)
timeit("tn  (dw=gTx)", lambda: ops.grouped_gemm_tn(g, x, offs, E), fl)
# hipBLASLt ceiling: one dense GEMM of the same FLOPs
xb = torch.randn(M, H, device="cuda", dtype=torch.bfloat16)
wb = torch.randn(I, H, device="cuda", dtype=torch.bfloat16)
timeit("hipBLASLt NT same-FLOPs", lambda: xb @ wb.t(), fl)

# ---- fp8 grouped forward (tensorwise-scaled e4m3, BK=128 bytes) ----
sx = torch.ones(1, device="cuda")
dummy = torch.zeros(1, device="cuda")
amax = 448.0 / float(x.abs().amax())
sx8 = torch.full((1,), amax, device="cuda")
x8 = ops.fp8_cast(x, sx8, dummy, False)
wamax = 448.0 / float(w.abs().amax())
sw8 = torch.full((1,), wamax, device="cuda")
w8 = ops.fp8_cast(w.view(-1, H), sw8, dummy, False).view(E, I, H)
deq = (sx8 * sw8).reciprocal()
timeit("nt-fp8 128 (y=x8@w8T)", lambda: ops.grouped_gemm_nt_fp8(x8, w8, offs, tm, deq, ntl), fl)
w38 = ops.fp8_cast(w3.view(-1, H), sw8, dummy, False).view(E, 1024, H)
timeit("nt-fp8 256x256 (N=1024)", lambda: ops.grouped_gemm_nt_fp8(x8, w38, offs_b, tm_b, deq, ntl_b, 256), fl3)
# numerics vs fp32 reference on a slice
y8 = ops.grouped_gemm_nt_fp8(x8, w8, offs, tm, deq, ntl)
ybf = ops.grouped_gemm_nt(x, w, offs, tm, ntl)
ref = (x[:128].float() @ w[0].float().t())
err8 = (y8[:128].float() - ref).abs().max() / ref.abs().max()
errb = (ybf[:128].float() - ref).abs().max() / ref.abs().max()
print(f"fp8 rel-err {float(err8):.4f} (bf16 path {float(errb):.4f})")
