"""Stage timeline of the backbone segment launches (csrc/bb_chain.hip): o_proj -> gate_up -> down_proj -> next qkv, wave 0 of every
workgroup stamps the 100 MHz counter at 8 points per stage (debug library).  Prints the LAST layer-launch of a decode step: its o_proj, gate_up,
down_proj and, where it has one, the head.  BB_STAMPS=eng: the loader / consumer engine (bb_engine.hip, 64 rows of the 1.7B talker).
usage: OMNI_TALKER_DEBUG=1 python scripts/bb_timeline.py [--model tts-1.7b] [--batch 64] [--kv fp8] [--ctx 352]"""
import argparse, ctypes as C, os, sys, types
os.environ["OMNI_TALKER_DEBUG"] = "1"
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import torch
import bench
ap = argparse.ArgumentParser()
ap.add_argument("--model", default="tts-1.7b")
ap.add_argument("--batch", type=int, default=64)
ap.add_argument("--kv", default="fp8")
ap.add_argument("--ctx", type=int, default=352)
cl = ap.parse_args()
args = types.SimpleNamespace(allreduce="rccl", model=cl.model, kv=cl.kv, batch=cl.batch, num_blocks=8192, device_weights=True, parallel="tp", sub_batches=1,
                             tp_force=False, prefill_gemm="tile", warmup=0, steps=64, ttfa_steps=0, ctx_extra=0, target_ctx=cl.ctx)
torch.cuda.set_device(0)
d, w, eng = bench.build_engine(args, 0, 1)
lib = eng.lib
_mode = os.environ.get("BB_STAMPS", "bb")
_f = lib.omni_debug_bb_engine; _f.argtypes = [C.c_int]; _f.restype = None
_f(int(_mode == "eng"))
eng.set_sampling(greedy=0, temperature=0.9, top_k=50, rep_penalty=1.05, seed=42, cp_greedy=0, cp_temperature=0.9, cp_top_k=50)
bench.setup_requests(d, eng, args)
B = cl.batch
for _ in range(4):
    eng.decode_step(B)
torch.cuda.synchronize()
NST, NW = 8, 256
buf = torch.zeros(40 * NST * NW, dtype=torch.int64, device="cuda")
STAMPS = getattr(lib, f"omni_debug_{_mode}_stamps"); STAMPS.argtypes = [C.c_void_p]; STAMPS.restype = None
STAMPS(buf.data_ptr())
eng.decode_step(B)
torch.cuda.synchronize()
STAMPS(None)
t = buf.view(40, NST, NW).cpu().double() * 0.01
names = {0: "o", 1: "gate_up", 2: "down", 4: "head"}
seg = ["W issue", "first look", "operands", "MFMA", "barrier", "epilogue"] if _mode == "bb" else ["W issue", "flag wait", "slabs->rstd", "x+MFMA", "barrier", "epilogue", "drain+flag"]
print(f"{cl.model}, {B} rows, the step's last layer launch, us, medians over the workgroups that run the stage; from .. to: since the launch's first stamp")
print(f"{'stage':8s} {'wgs':>4s} " + " ".join(f"{s:>11s}" for s in seg) + f" {'total':>8s} {'from':>7s} {'to':>7s}")
start = t[0][0][t[0][0] > 0].min().item()
for s, name in names.items():
    m = (t[s][0] >= start) & (t[s][7] > 0)
    if not m.any():
        continue
    x = t[s][:, m]
    d_ = [(x[k + 1] - x[k]).median().item() for k in range(len(seg))]
    print(f"{name:8s} {int(m.sum()):4d} " + " ".join(f"{v:11.2f}" for v in d_) + f" {sum(d_):8.2f} {x[0].min().item() - start:7.2f} {x[7].max().item() - start:7.2f}")
t = t[:4]

if _mode == "eng":
    L_ = buf.view(40, NST, NW)[32].cpu().double()
    ts = L_[:5] * 0.01
    print("loader wave 8 (medians, us): issue o %.2f | gate_up %.2f | down %.2f | (qkv %.2f); polls spent waiting for FIFO space: median %d, max %d" % (
        (ts[1] - ts[0]).median(), (ts[2] - ts[1]).median(), (ts[3] - ts[2]).median(), (ts[4] - ts[3]).median(), int(L_[5].median()), int(L_[5].max())))
    print("loader start -> compute-wave o-stage entry (us): %.2f; loader end vs down-stage end: %.2f" % (
        (t[0][0] - ts[0]).median(), (t[2][7] - ts[3]).median()))
