"""Measured workloads of the sparse-coding path, through its public entry points.

A case is a dict of plain values; its "kind" names the entry points it calls:

  column    lca.LCAColumn: whole timesteps of the Input -> Residual <-> V1 -> Recon
            column, replayed from a hipGraph, or driven by lca.run_column
            (eager steps with the energy probe read after each)
  gather    runtime.PostsynapticPerspectiveGPUDelivery.deliver, one dense delivery
  scatter   runtime.ActiveList.compact and a sparse
            runtime.PresynapticPerspectiveGPUDelivery.deliver over the list
  hebbian   runtime.HebbianUpdater.update_dw with its activation counts
  learn     lca.LCAColumn.update_weights: dW, W += dW, NormalizeL2 and the
            deliveries' weights derived again
  adjoint   adjoint.LCAAdjoint forward and backward through unrolled timesteps
  update    one layer update (HyPerLCA, MomentumLCA or ISTA)

Geometry throughout: a fine layer (image side) `s` times the coarse one (V1
side) along x and y, joined by patches of p fine positions, so the window of
coarse x starts at fine s*x - (p - s)/2.  `exact` restates each computation in
64 bits with unfold, matmul and fold.
"""
import numpy as np
import torch
import torch.nn.functional as F

from openpv_amd import abi, lca, runtime
from openpv_amd.adjoint import LCAAdjoint

DEV = "cuda"
ARITH = {"exact": abi.ARITH_EXACT, "fp32": abi.ARITH_FP32, "bf16": abi.ARITH_BF16,
         "fp8": abi.ARITH_FP8}
FLT_MAX = float(np.finfo(np.float32).max)
DENSITY = 0.07      # active share of an LCA layer in the middle of a run


# ------------------------------------------------------------------ the cases

def _column(name, arith, nb, nyv, nxv, nfv, s, p, nf, vt, steps, vwidth=0.0, host=False, probe=False):
    return {"name": name, "kind": "column", "arith": arith, "nb": nb, "nyv": nyv, "nxv": nxv, "nfv": nfv,
            "s": s, "p": p, "nf": nf, "vt": vt, "vwidth": vwidth, "steps": steps, "host": host, "probe": probe}


def listed():
    return [
        # The smallest call: the two-to-one column of the reference's LCA tests (one
        # 128x64 image, 18x18 patches, firm threshold, host summation order), stepped
        # by run_column with its energy read after every step.  Launches and latency.
        _column("column_small_exact", "exact", 1, 32, 64, 24, 2, 18, 1, 0.025, 4, vwidth=0.025, host=True),
        # The batched workload in the default, bit-exact form.
        _column("column_batch_exact", "exact", 64, 32, 32, 512, 4, 16, 1, 0.15, 2),
        # The same in FP32, the form a params file gets with receiveGpu.
        _column("column_batch_fp32", "fp32", 64, 32, 32, 512, 4, 16, 1, 0.15, 5),
        # The same in BF16 as it is run for throughput: 25 timesteps in one graph,
        # then the sparse code is read.
        _column("column_batch_bf16", "bf16", 64, 32, 32, 512, 4, 16, 1, 0.15, 25),
        # Colour images at stride 2 with the energy probe: other patch rows, another
        # route of the reconstruction, a medium size.
        _column("column_colour_bf16", "bf16", 16, 32, 32, 256, 2, 8, 3, 0.1, 5, probe=True),
        # One full-size delivery, many features into many: the inner layer of a
        # deeper network, BF16 and FP32.
        {"name": "gather_wide_bf16", "kind": "gather", "arith": "bf16", "nb": 1, "ny": 128, "nx": 128,
         "nf": 256, "s": 2, "p": 12, "nfp": 16},
        {"name": "gather_wide_fp32", "kind": "gather", "arith": "fp32", "nb": 1, "ny": 128, "nx": 128,
         "nf": 256, "s": 2, "p": 12, "nfp": 16},
        # The sparse delivery of the same pair of layers, 2 % of the source active:
        # publishing the active list, then the scatter over it.
        {"name": "scatter_sparse_fp32", "kind": "scatter", "arith": "fp32", "nb": 1, "ny": 128, "nx": 128,
         "nf": 256, "s": 2, "p": 12, "nfp": 16, "density": 0.02},
        # dW of a colour dictionary in FP32, ragged sizes.
        {"name": "hebbian_colour_fp32", "kind": "hebbian", "arith": "fp32", "nb": 7, "ny": 37, "nx": 45,
         "nf": 200, "s": 2, "p": 8, "nfp": 3},
        # One weight update of large-image dictionary learning (BF16 column, FP64
        # normalisation), the largest state.
        {"name": "learn_large_bf16", "kind": "learn", "arith": "bf16", "nb": 8, "ny": 128, "nx": 128,
         "nf": 1024, "s": 4, "p": 16, "nfp": 1},
        # Gradients through ten unrolled timesteps, checkpoints every five.
        {"name": "adjoint_colour_fp32", "kind": "adjoint", "arith": "fp32", "nb": 8, "ny": 32, "nx": 32,
         "nf": 256, "s": 2, "p": 8, "nfp": 3, "steps": 10, "checkpoint": 5},
        # The layer update of a MomentumLCA column (its delivery writes GSyn).
        {"name": "update_momentum", "kind": "update", "rule": "momentum", "nb": 64, "ny": 32, "nx": 32,
         "nf": 512, "halo": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["column", "column", "column", "gather", "gather", "scatter", "hebbian", "learn",
                       "adjoint", "update"])
    s = rng.choice([2, 4])
    q = rng.choice([2, 3, 4])                # coarse positions that share a fine one, per axis
    nfp = rng.choice([1, 3])
    if kind == "column":
        arith = rng.choice(["exact", "fp32", "bf16", "fp8"])
        nyv, nxv = _log_int(rng, 8, 48), _log_int(rng, 8, 48)
        nfv = rng.choice([rng.randint(20, 200), 32 * rng.randint(1, 16), 128, 256, 512])
        steps = rng.randint(1, 5)
        # at most the products of two steps of the batched workload
        one = nyv * nxv * nfv * (q * s) ** 2 * nfp * steps
        nb = _log_int(rng, 1, max(1, min(64, (1 << 34) // one)))
        host = nb * nyv * nxv * nfv < 1 << 20 and rng.random() < 0.5
        return dict(kind=kind, arith=arith, nb=nb, nyv=nyv, nxv=nxv, nfv=nfv, s=s, p=q * s, nf=nfp,
                    vt=rng.choice([0.05, 0.1, 0.15]), vwidth=rng.choice([0.0, 0.05]),
                    steps=steps, host=host, probe=rng.random() < 0.3)
    if kind in ("gather", "scatter"):
        nfp = rng.choice([1, 3, 8, 16])
        ny, nx = _log_int(rng, 16, 128), _log_int(rng, 16, 128)
        case = dict(kind=kind, arith=rng.choice(["exact", "fp32", "bf16", "fp8"] if kind == "gather" else
                                                ["exact", "fp32"]),
                    nb=1, ny=ny, nx=nx, nf=rng.choice([rng.randint(30, 200), 64, 128, 256]), s=2,
                    p=2 * rng.choice([2, 3, 4, 6]), nfp=nfp)
        if kind == "scatter":
            case["density"] = rng.choice([0.01, 0.02, 0.05])
        return case
    if kind == "hebbian":
        return dict(kind=kind, arith=rng.choice(["fp32", "bf16"]), nb=_log_int(rng, 1, 8),
                    ny=_log_int(rng, 12, 64), nx=_log_int(rng, 12, 64), nf=_log_int(rng, 32, 512), s=s,
                    p=q * s, nfp=nfp)
    if kind == "learn":
        return dict(kind=kind, arith=rng.choice(["fp32", "bf16", "fp8"]), nb=_log_int(rng, 1, 8),
                    ny=_log_int(rng, 16, 64), nx=_log_int(rng, 16, 64), nf=32 * _log_int(rng, 1, 16), s=4,
                    p=16, nfp=1)
    if kind == "adjoint":
        return dict(kind=kind, arith="fp32", nb=_log_int(rng, 1, 8), ny=_log_int(rng, 8, 24),
                    nx=_log_int(rng, 8, 24), nf=32 * rng.randint(1, 6), s=2, p=8, nfp=3,
                    steps=rng.randint(2, 10), checkpoint=rng.choice([2, 5]))
    return dict(kind=kind, rule=rng.choice(["lca", "momentum", "ista"]), nb=_log_int(rng, 1, 64),
                ny=_log_int(rng, 8, 32), nx=_log_int(rng, 8, 32), nf=_log_int(rng, 24, 512),
                halo=rng.randint(0, 3))


# ------------------------------------------------------------------ inputs

def _images(nb, ny, nx, nf, seed):
    """1/f amplitude spectrum, random phase, zero mean, unit variance per channel."""
    rng = np.random.default_rng(seed)
    f = np.hypot(np.fft.fftfreq(ny)[:, None], np.fft.rfftfreq(nx)[None, :])
    amp = np.divide(1.0, f, out=np.zeros_like(f), where=f > 0)
    ph = np.exp(2j * np.pi * rng.random((nb, nf) + f.shape, dtype=np.float32))
    img = np.fft.irfft2(amp * ph, s=(ny, nx))
    img /= img.std(axis=(2, 3), keepdims=True)
    return np.ascontiguousarray(img.transpose(0, 2, 3, 1)).astype(np.float32)


def _dictionary(nf, p, nfp, seed):
    """N(0,1) features of unit L2 norm, [nf][p][p][nfp]."""
    w = np.random.default_rng([seed, 2]).standard_normal((nf, p, p, nfp))
    return (w / np.sqrt((w * w).sum(axis=(1, 2, 3), keepdims=True))).astype(np.float32)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _pad(case):
    """Fine positions a patch reaches past the stride on each side."""
    return (case["p"] - case["s"]) // 2


def _extended(x, loc_):
    """[nb][ny][nx][nf] into the layer's extended buffer with a zero halo, flat."""
    h = loc_.halo
    return F.pad(x, (0, 0, h.lt, h.rt, h.up, h.dn)).contiguous().reshape(-1)


def _column_inputs(case, seed):
    nfv = case["nfv"]
    img = _images(case["nb"], case["nyv"] * case["s"], case["nxv"] * case["s"], case["nf"], seed)
    W = _dictionary(nfv, case["p"], case["nf"], seed)
    # a membrane potential as in the middle of a run: about DENSITY of it above threshold
    V0 = torch.randn((case["nb"], case["nyv"], case["nxv"], nfv), device=DEV, generator=_gen(seed))
    V0 *= case["vt"] / 1.5
    return img, W, V0


def _delivery_inputs(case, seed):
    g = _gen(seed)
    s, nf, nfp, p = case["s"], case["nf"], case["nfp"], case["p"]
    x = torch.randn((case["nb"], case["ny"] * s, case["nx"] * s, nfp), device=DEV, generator=g)
    if "density" in case:       # sparse, positive
        on = torch.rand(x.shape, device=DEV, generator=g) < case["density"]
        x = torch.where(on, torch.empty_like(x).exponential_(1.0, generator=g), 0.0)
    W = 0.05 * torch.randn((nf, p, p, nfp), device=DEV, generator=g)
    return x, W


def _plastic_inputs(case, seed):
    """Sparse coarse activity and a fine residual."""
    g = _gen(seed)
    shape = (case["nb"], case["ny"], case["nx"], case["nf"])
    on = torch.rand(shape, device=DEV, generator=g) < DENSITY
    a = torch.where(on, torch.empty(shape, device=DEV).exponential_(1.0, generator=g), 0.0)
    r = torch.randn((case["nb"], case["ny"] * case["s"], case["nx"] * case["s"], case["nfp"]), device=DEV,
                    generator=g)
    return a, r


def _update_inputs(case, seed):
    g = _gen(seed)
    shape = (case["nb"], case["ny"], case["nx"], case["nf"])
    G, V, prev = (0.1 * torch.randn(shape, device=DEV, generator=g) for _ in range(3))
    return G, V, prev


def _scatter_weights(W, s, p):
    """The pre-perspective weights of the delivery whose post-perspective ones are
    W [F][p][p][f]: one patch per source feature and phase, [s*s*f][p/s][p/s][F]."""
    nf, nfp, q = W.shape[0], W.shape[3], p // s
    out = torch.empty((s, s, nfp, q, q, nf), device=W.device)
    # source x reaches targets ceil((x - (p - 1 - pad))/s) ..; the one at patch
    # column wx sees it at post-perspective column x + pad - s*(first + wx)
    pad = (p - s) // 2
    at = []
    for x in range(s):
        first = -((p - 1 - pad - x) // s)
        at.append([x + pad - s * (first + w) for w in range(q)])
    for py in range(s):
        for px in range(s):
            out[py, px] = W[:, at[py]][:, :, at[px]].permute(3, 1, 2, 0)
    return out.reshape(s * s * nfp, q, q, nf).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "column":
        img, W, V0 = _column_inputs(case, seed)
        col = lca.LCAColumn(img, W, case["nxv"], case["nyv"], case["nfv"], case["p"], case["p"],
                            VThresh=case["vt"], VWidth=case["vwidth"], timeConstantTau=100.0, dt=1.0,
                            AShift=case["vt"], arith=ARITH[case["arith"]], fused=not case["host"], V0=V0,
                            device=DEV)
        if not case["host"]:
            torch.cuda.synchronize()
            side = torch.cuda.Stream()
            col.capture(side, steps=case["steps"])
            side.synchronize()
        return {"case": case, "col": col}
    if kind == "learn":
        a, r = _plastic_inputs(case, seed)
        W = _dictionary(case["nf"], case["p"], case["nfp"], seed)
        img = torch.zeros((case["nb"], case["ny"] * case["s"], case["nx"] * case["s"], case["nfp"]))
        col = lca.LCAColumn(img, W, case["nx"], case["ny"], case["nf"], case["p"], case["p"], VThresh=0.15,
                            arith=ARITH[case["arith"]], fused=True, device=DEV)
        col.enable_learning(1e-3, normalize_dw=True)
        col.v1_A.copy_(_extended(a, col.v1_loc))        # the state a display period leaves
        col.res_A.copy_(_extended(r, col.res_loc))
        return {"case": case, "col": col}
    if kind == "adjoint":
        img = _images(case["nb"], case["ny"] * case["s"], case["nx"] * case["s"], case["nfp"], seed)
        W = _dictionary(case["nf"], case["p"], case["nfp"], seed)
        adj = LCAAdjoint(case["nb"], case["nx"] * case["s"], case["ny"] * case["s"], case["nfp"], case["nx"],
                         case["ny"], case["nf"], case["p"], case["p"], VThresh=0.05, timeConstantTau=20.0,
                         arith=ARITH[case["arith"]], checkpoint=case["checkpoint"], device=DEV)
        return {"case": case, "adj": adj, "x": torch.as_tensor(img, device=DEV),
                "W": torch.as_tensor(W, device=DEV)}
    if kind == "update":
        G, V, prev = _update_inputs(case, seed)
        loc_ = runtime.loc(case["nb"], case["nx"], case["ny"], case["nf"], case["halo"])
        t = runtime.make_transfer(0.15, 0.0, FLT_MAX, 0.15, 0.0)
        args = dict(timeConstantTau=100.0, dt=1.0, activity_from_v=True, device=DEV)
        if case["rule"] == "momentum":
            upd = runtime.MomentumLCAUpdate(loc_, t, LCAMomentumRate=0.4, **args)
            upd.prev_drive.copy_(prev.reshape(-1))
        elif case["rule"] == "ista":
            upd = runtime.ISTAUpdate(loc_, t, 0.15, **args)
        else:
            upd = runtime.HyPerLCAUpdate(loc_, t, **args)
        V = V.reshape(-1)
        A = torch.zeros(loc_.nbatch * loc_.num_ext, device=DEV)
        runtime.ann_activity(loc_, t, V, A)
        return {"case": case, "upd": upd, "G": G.reshape(-1), "V": V, "A": A}
    s, nb, ny, nx = case["s"], case["nb"], case["ny"], case["nx"]
    if kind == "hebbian":
        a, r = _plastic_inputs(case, seed)
        H = abi.host()
        pre = runtime.loc(nb, nx, ny, case["nf"], H.pvhost_required_margin(nx, nx * s, case["p"]))
        post = runtime.loc(nb, nx * s, ny * s, case["nfp"], H.pvhost_required_margin(
            nx * s, nx, H.pvhost_post_patch_size(case["p"], nx, nx * s)))
        upd = runtime.HebbianUpdater(pre, post, case["p"], case["p"], 1e-3, normalize_dw=True, device=DEV)
        return {"case": case, "upd": upd, "a": _extended(a, pre), "r": _extended(r, post)}
    x, W = _delivery_inputs(case, seed)
    margin = _pad(case)
    pre = runtime.loc(nb, nx * s, ny * s, case["nfp"], margin + margin % 2)
    post = runtime.loc(nb, nx, ny, case["nf"], 0)
    arith = ARITH[case["arith"]]
    state = {"case": case, "x": _extended(x, pre), "G": torch.zeros(nb * post.num_res, device=DEV)}
    if kind == "gather":
        d = runtime.PostsynapticPerspectiveGPUDelivery(pre, post, case["p"], case["p"], W.reshape(-1),
                                                       arith=arith)
        if case["arith"] == "fp8":
            d.set_source_scale(runtime.fp8_scale_for(float(x.abs().max())))
    else:
        q = case["p"] // s
        d = runtime.PresynapticPerspectiveGPUDelivery(pre, post, q, q, _scatter_weights(W, s, case["p"]).reshape(-1),
                                                      arith=arith)
        d.mode = "ordered"      # the sparse delivery, what a layer this sparse is tuned to
        state["active"] = runtime.ActiveList(pre, torch.device(DEV))
    state["delivery"] = d
    return state


# ------------------------------------------------------------------ one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "column":
        col = state["col"]
        out = {}
        if case["host"]:
            out["energies"] = lca.run_column(col, case["steps"], energy_cost="firm" if case["vwidth"] else "l1")
        else:
            col.replay(torch.cuda.current_stream())
            if case["probe"]:
                out["energy"] = col.probe_energy(cost="firm" if case["vwidth"] else "l1")
        out.update(V=col.v1_V, A=col.v1_activity(), residual=col.res_A, reconstruction=col.rec_A)
        return out
    if kind == "learn":
        state["col"].update_weights()
        return {"weights": state["col"].weights, "dw": state["col"].learner.dw,
                "counts": state["col"].learner.counts}
    if kind == "adjoint":
        adj = state["adj"]
        E, ck = adj.forward(state["x"], state["W"], case["steps"])
        gW, gx = adj.backward(state["x"], case["steps"], ck)
        return {"energy": E, "grad_weights": gW, "grad_input": gx}
    if kind == "update":
        upd = state["upd"]
        upd.update(state["G"], state["V"], state["A"])
        out = {"V": state["V"], "A": state["A"]}
        if case["rule"] == "momentum":
            out["drive"] = upd.prev_drive
        return out
    if kind == "hebbian":
        upd = state["upd"]
        upd.update_dw(state["a"], state["r"], arith=ARITH[case["arith"]])
        return {"dw": upd.dw, "counts": upd.counts}
    if kind == "gather":
        state["delivery"].deliver(state["x"], state["G"])
        return state["G"]
    state["active"].compact(state["x"])
    state["delivery"].deliver(state["G"], active=state["active"])
    return {"gsyn": state["G"], "num_active": state["active"].num_active,
            "pos_start": state["active"].pos_start}


def work(case):
    kind = case["kind"]
    if kind == "column":
        n = case["nb"] * case["nyv"] * case["nxv"] * case["nfv"]
        fine = case["nb"] * case["nyv"] * case["nxv"] * case["s"] ** 2 * case["nf"]
        K = case["p"] ** 2 * case["nf"]
        act = 2 if case["arith"] in ("bf16", "fp8") else 4
        # per step: V read and written, the activity written and read; input,
        # residual and reconstruction read and written once each
        nbytes = n * (8 + 2 * act) + 16 * fine
        flops = 2.0 * n * K * (1.0 + DENSITY)
        return {"bytes": float(case["steps"]) * nbytes + 4.0 * n, "flops": case["steps"] * flops}
    coarse = case["nb"] * case["ny"] * case["nx"] * case["nf"]
    if kind == "update":
        return {"bytes": coarse * {"lca": 16.0, "momentum": 24.0, "ista": 16.0}[case["rule"]],
                "flops": 10.0 * coarse}
    fine = case["nb"] * case["ny"] * case["nx"] * case["s"] ** 2 * case["nfp"]
    K = case["p"] ** 2 * case["nfp"]
    if kind == "gather":
        return {"bytes": 4.0 * (coarse + fine + case["nf"] * K), "flops": 2.0 * coarse * K}
    if kind == "scatter":
        # the source scanned, its list written and read, the weights, GSyn written
        return {"bytes": 4.0 * (fine + coarse + case["nf"] * K) + 16.0 * case["density"] * fine,
                "flops": 2.0 * coarse * K * case["density"]}
    if kind in ("hebbian", "learn"):
        w = case["nf"] * K
        return {"bytes": 4.0 * (coarse + fine) + w * (12.0 if kind == "hebbian" else 28.0),
                "flops": 2.0 * coarse * K * DENSITY}
    # a forward step is one gather and one scatter; the backward recomputes it and
    # adds a gather, a scatter and two correlations
    steps = case["steps"]
    return {"bytes": steps * (coarse * 4.0 * 16 + fine * 4.0 * 12), "flops": steps * 2.0 * coarse * K * 8}


# ------------------------------------------------------------------ 64 bits

def _patches(x, s, p):
    """Windows of fine [nb][ny][nx][f]: [nb*positions][p*p*f] in (ky, kx, f) order."""
    nb, f = x.shape[0], x.shape[3]
    u = F.unfold(x.permute(0, 3, 1, 2), p, padding=(p - s) // 2, stride=s)
    return u.view(nb, f, p * p, -1).permute(0, 3, 2, 1).reshape(-1, p * p * f)


def _overlap_add(y, nb, ny, nx, f, s, p):
    """Transpose of _patches onto a fine layer of ny x nx: [nb][ny][nx][f]."""
    u = y.view(nb, -1, p * p, f).permute(0, 3, 2, 1).reshape(nb, f * p * p, -1)
    return F.fold(u, (ny, nx), p, padding=(p - s) // 2, stride=s).permute(0, 2, 3, 1)


def _f32(x):
    return float(np.float32(x))


def _transfer(V, vt, vwidth):
    """The threshold with a linear ramp of width vwidth from 0 to its shifted value."""
    top = vt + vwidth
    a = torch.where(V < vt, torch.zeros_like(V), V - vt)
    if top > vt:
        ramp = (top - vt) * (V - vt) / vwidth
        a = torch.where((V >= vt) & (V < top), ramp, a)
    return a


def _ext_shape(x, halo):
    return F.pad(x, (0, 0, halo, halo, halo, halo)).reshape(-1)


def _margins(case):
    """Halo of the fine layer (residual) and of the coarse one (V1)."""
    q = case["p"] // case["s"]
    return (q - 1) * case["s"] // 2, q // 2


def _exact_column(case, seed):
    img, W, V0 = _column_inputs(case, seed)
    nb, nyv, nxv, nfv, s, p, nf = (case[k] for k in ("nb", "nyv", "nxv", "nfv", "s", "p", "nf"))
    x = torch.as_tensor(img, device=DEV).double()
    Wm = torch.as_tensor(W, device=DEV).double().reshape(nfv, -1)
    V = V0.double().reshape(-1, nfv)
    vt, vw = _f32(case["vt"]), _f32(case["vwidth"])
    e = float(np.exp(-0.01))
    rec = torch.zeros_like(x)
    A = _transfer(V, vt, vw)
    energies = []
    for _ in range(case["steps"]):
        res = x - rec
        V = e * V + (1.0 - e) * (_patches(res, s, p) @ Wm.T + A)
        A = _transfer(V, vt, vw)
        rec = _overlap_add(A @ Wm, nb, nyv * s, nxv * s, nf, s, p)
        cost = A.abs()
        if vw > 0:
            top = vt + vw
            cost = torch.where(cost < top, cost * (1.0 - 0.5 / top * cost), torch.full_like(cost, 0.5 * top))
        energies.append(0.5 * (res * res).view(nb, -1).sum(1) + vt * cost.view(nb, -1).sum(1))
    mres, mv1 = _margins(case)
    out = {}
    if case["host"]:
        out["energies"] = torch.stack(energies)
    elif case["probe"]:
        out["energy"] = energies[-1]
    out.update(V=V.reshape(-1), A=_ext_shape(A.view(nb, nyv, nxv, nfv), mv1),
               residual=_ext_shape(res, mres), reconstruction=rec.reshape(-1))
    return out


def _exact_dw(case, a, r):
    """Correlation of the activity with the residual's windows, [nf][p*p*f]."""
    am = a.double().reshape(-1, case["nf"])
    return am.T @ _patches(r.double(), case["s"], case["p"])


def _exact_counts(case, a, r):
    """The active source neurons whose window holds each weight inside the image."""
    on = (a != 0).double().reshape(-1, case["nf"])
    return on.T @ _patches(torch.ones_like(r, dtype=torch.float64), case["s"], case["p"])


def _exact_adjoint(case, seed):
    nb, ny, nx, nf, s, p, nfp = (case[k] for k in ("nb", "ny", "nx", "nf", "s", "p", "nfp"))
    img = torch.as_tensor(_images(nb, ny * s, nx * s, nfp, seed), device=DEV).double()
    W = torch.as_tensor(_dictionary(nf, p, nfp, seed), device=DEV).double().reshape(nf, -1)
    x, Wm = img.requires_grad_(True), W.requires_grad_(True)
    vt, e = _f32(0.05), float(np.exp(-1.0 / 20.0))
    V = torch.zeros((nb * ny * nx, nf), dtype=torch.float64, device=DEV)
    A, rec = _transfer(V, vt, 0.0), torch.zeros_like(img)
    for _ in range(case["steps"]):
        V = e * V + (1.0 - e) * (_patches(x - rec, s, p) @ Wm.T + A)
        A = _transfer(V, vt, 0.0)
        rec = _overlap_add(A @ Wm, nb, ny * s, nx * s, nfp, s, p)
    E = 0.5 * ((x - rec) ** 2).reshape(nb, -1).sum(1) + vt * A.abs().view(nb, -1).sum(1)
    gx, gW = torch.autograd.grad(E.sum(), (x, Wm))
    return {"energy": E.detach(), "grad_weights": gW.reshape(-1), "grad_input": gx.reshape(-1)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "column":
        return _exact_column(case, seed)
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    if kind == "update":
        G, V, prev = (t.double() for t in _update_inputs(case, seed))
        vt, e = _f32(0.15), float(np.exp(-0.01))
        A = _transfer(V, vt, 0.0)
        out = {}
        if case["rule"] == "ista":
            V = V + 0.01 * (G - vt * torch.sign(A))
        else:
            drive = (1.0 - e) * (G + A)
            V = e * V + drive
            if case["rule"] == "momentum":
                V = V + _f32(0.4) * prev
                out["drive"] = drive.reshape(-1)
        out.update(V=V.reshape(-1), A=_ext_shape(_transfer(V, vt, 0.0), case["halo"]))
        return out
    if kind in ("hebbian", "learn"):
        a, r = _plastic_inputs(case, seed)
        dw = _f32(1e-3) * _exact_dw(case, a, r)
        if kind == "hebbian":
            return {"dw": dw.reshape(-1), "counts": None}
        n = _exact_counts(case, a, r)
        dw = torch.where(n > 0, dw / n.clamp(min=1.0), torch.zeros_like(dw))
        W = torch.as_tensor(_dictionary(case["nf"], case["p"], case["nfp"], seed), device=DEV).double()
        W = W.reshape(case["nf"], -1) + dw
        W = W / W.square().sum(1, keepdim=True).sqrt()
        return {"weights": W.reshape(-1), "dw": dw.reshape(-1), "counts": None}
    x, W = _delivery_inputs(case, seed)
    G = _patches(x.double(), case["s"], case["p"]) @ W.double().reshape(case["nf"], -1).T
    if kind == "gather":
        return G.reshape(-1)
    return {"gsyn": G.reshape(-1), "num_active": None, "pos_start": None}
