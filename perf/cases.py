"""The work a user of this framework has it do, as timed cases.

Three kinds of program use it: the driver's time loop over three levels (one
chunk of N2 x N3 toolpath rows at a time, single rows after a layer change or
a jump, dwell rows while the laser is off), parameter studies that advance
many instances together (L3 windows, or whole three-level stacks), and the
learned operator of the L3 window (its single convolution layers, one jump of
one window, the gradient of a training batch).

A case is a dict of plain values; ``kind`` names the program:

  l1_step   TimeLoop.step_chunk: moveEverything + subcycleGOMELT
  row       moveEverything + stepGOMELT of one toolpath row
  dwell     stepGOMELTDwellTime (the L1-only step)
  windows   Batch.step: one L3 step of n windows
  stacks    Stacks.step: one L1 step of n three-level runs in lockstep
  conv      one convolution layer, forward and backward
  jump      window_input + apply_jump: the operator on one window
  grad      UNet forward, loss and backward of a batch of windows
"""

from __future__ import annotations

import json
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "go-melt_amd"))

import workloads as W  # noqa: E402


def listed():
    return [
        # the 5 mm single track on 41 x 41 x 21 nodes a level: an L1 step of
        # some 300 small dependent launches
        {"name": "track_l1_step", "kind": "l1_step", "deck": "track"},
        # the part-scale raster with property tables: 2.06 M L1 nodes, 520 k
        # on L2 and L3; the framework's headline run
        {"name": "part_l1_step", "kind": "l1_step", "deck": "part"},
        # one toolpath row of the single-step mode on both decks: the first
        # chunk of every layer, jumps and the end of a file run row by row
        {"name": "track_row", "kind": "row", "deck": "track"},
        {"name": "part_row", "kind": "row", "deck": "part"},
        # a row of dwell between layers: the part-scale mesh alone
        {"name": "part_dwell", "kind": "dwell", "deck": "part"},
        # a parameter study's L3 windows (32^3 to 96 x 96 x 48 elements), one
        # step of all
        {"name": "windows_32", "kind": "windows", "n": 32, "ex": 0, "ey": 0, "ez": 0},
        # eight three-level runs of such a study in lockstep
        {"name": "stacks_8", "kind": "stacks", "n": 8},
        # a full-resolution layer of the operator on four windows
        {"name": "conv_fine", "kind": "conv", "nb": 4, "D": 32, "H": 64, "W": 64, "ci": 32,
         "co": 32},
        # a half-resolution layer of a training batch
        {"name": "conv_half", "kind": "conv", "nb": 16, "D": 16, "H": 32, "W": 32, "ci": 64,
         "co": 64},
        # a layer of odd extents and channel counts off the powers of two
        {"name": "conv_odd", "kind": "conv", "nb": 3, "D": 13, "H": 27, "W": 35, "ci": 48,
         "co": 80},
        # the operator in the loop: one window per jump
        {"name": "jump", "kind": "jump", "channels": "32,64,128,128", "nx": 64, "ny": 64,
         "nz": 32},
        # the gradient of one training batch
        {"name": "gradient_16", "kind": "grad", "channels": "32,64,128,128", "nb": 16, "D": 32,
         "H": 64, "W": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["l1_step", "l1_step", "row", "dwell", "windows", "windows", "stacks",
                       "conv", "conv", "conv", "jump", "grad"])
    if kind in ("l1_step", "row", "dwell"):
        # three-level decks of 16 to 96 elements along an axis
        return {"kind": kind, "deck": "stack", "ex": _log_int(rng, 16, 96),
                "ey": _log_int(rng, 16, 96), "ez": _log_int(rng, 8, 48)}
    if kind == "windows":
        if rng.random() < 0.5:  # the study's own mesh sizes
            return {"kind": kind, "n": _log_int(rng, 1, 32), "ex": 0, "ey": 0, "ez": 0}
        return {"kind": kind, "n": _log_int(rng, 1, 32), "ex": _log_int(rng, 16, 96),
                "ey": _log_int(rng, 16, 96), "ez": _log_int(rng, 8, 48)}
    if kind == "stacks":
        return {"kind": kind, "n": rng.randint(2, 8)}
    if kind == "conv":
        # 1 k to 524 k voxels, channels of 16 to 192
        D, H, Wd = _log_int(rng, 4, 32), _log_int(rng, 8, 64), _log_int(rng, 8, 64)
        nb = max(1, min(16, _log_int(rng, 1, 16), 524288 // (D * H * Wd)))
        return {"kind": kind, "nb": nb, "D": D, "H": H, "W": Wd,
                "ci": 16 * rng.choice([1, 2, 2, 3, 4, 6, 8, 12]),
                "co": 16 * rng.choice([1, 2, 2, 3, 4, 5, 8])}
    chans = rng.choice(["16,32", "16,32,64", "16,32,64,64", "32,64,128", "32,64,128,128"])
    if kind == "jump":
        return {"kind": kind, "channels": chans, "nx": 8 * rng.randint(3, 8),
                "ny": 8 * rng.randint(3, 8), "nz": 8 * rng.randint(2, 4)}
    return {"kind": kind, "channels": chans, "nb": rng.randint(1, 12), "D": 8 * rng.randint(2, 4),
            "H": 8 * rng.randint(3, 8), "W": 8 * rng.randint(3, 8)}


# ---------------------------------------------------------------------------
# Decks of the time loop
# ---------------------------------------------------------------------------

def _deck(case, seed):
    """(solver input, one closed lap of G-code): out and back along a track,
    so that a run can go on for any number of laps.  The seed draws the laser
    power (and the stack decks' speed and radius)."""
    rng = np.random.default_rng(seed)
    if case["deck"] == "stack":
        inp, g = W.stack_decks(n=1, seed=seed, sizes=[(case["ex"], case["ey"], case["ez"])])[0]
        first, second = g.split("\n")[:2]
        return inp, f"{first}\n{second}\n{first.replace('G0', 'G1')}\n"
    if case["deck"] == "track":
        inp, _ = W.single_track()
        inp["properties"]["laser_power"] = float(rng.uniform(150.0, 250.0))
        return inp, "G0 X2.5 Y5 Z0\nG1 X7.5 Y5 Z0\nG1 X2.5 Y5 Z0\n"
    inp, _ = W.production()
    inp["properties"]["laser_power"] = float(rng.uniform(200.0, 300.0))
    # two lines of the raster; the hatch jump stays below the single-step limit
    return inp, W.raster_gcode(7.5, 12.5, 9.0, 0.1, 2)


def _write(inp, gcode, where):
    with open(W.write_deck(inp, gcode, where)) as fh:
        return json.load(fh)


_STREAM = []


def _stream():
    """The one stream of a program's runs: its steps follow one another."""
    import _native as N
    if not _STREAM:
        _STREAM.append(N.Stream())
    return _STREAM[0]


def _time_loop(case, seed):
    """A run after its first (single-step) chunk, and the lap's other chunks."""
    import computeFunctions as cf
    import go_melt as G
    tmp = tempfile.TemporaryDirectory(prefix="gomelt_perf_")
    inp, g = _deck(case, seed)
    with cf.engines_on_stream(_stream()):
        run = G.TimeLoop(_write(inp, g, tmp.name), quiet=True, write_outputs=False)
    n = run.subcycle[2]
    lap = [c for c in run.chunks() if len(c) == n]
    run.step_chunk(lap[0])
    return {"run": run, "lap": lap, "at": 0, "tmp": tmp, "views": {}, "owner": run}


class _Device:
    """A device buffer of the framework as torch takes it (no copy).  The
    tensor keeps this object and with it the buffer's owner."""

    def __init__(self, a, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {
            "shape": (a.n,), "typestr": np.dtype(a.dtype).str, "data": (int(a.ptr), False),
            "version": 2, "strides": None}


def _view(state, a):
    key = (int(a.ptr), a.n)
    v = state["views"].get(key)
    if v is None:
        v = state["views"][key] = torch.as_tensor(_Device(a, state["owner"]), device="cuda")
        v.owner = state["owner"]
    return v


def _levels_out(state, L, level0=True):
    """The levels' state after a pass."""
    out = {"T1": L[1]["T0"], "S1_1": L[1]["S1"], "T2": L[2]["T0"], "Tp2": L[2]["Tprime0"],
           "S1_2": L[2]["S1"], "T3": L[3]["T0"], "Tp3": L[3]["Tprime0"], "S1_3": L[3]["S1"],
           "S2_3": L[3]["S2"]}
    if level0:
        out.update({"S1_0": L[0]["S1"], "accum": L[0]["accum_time"],
                    "max_accum": L[0]["max_accum_time"]})
    return {k: _view(state, a) for k, a in out.items()}


# ---------------------------------------------------------------------------
# Windows of the learned operator
# ---------------------------------------------------------------------------

T_SCALE, P_SCALE, H3 = 1000.0, 400.0, 0.0125


def _window(seed, nx, ny, nz):
    """A window's temperature field with a moving melt pool (FP32, x fastest),
    the laser row and the properties."""
    rng = np.random.default_rng(seed)
    P, r = float(rng.uniform(150.0, 350.0)), 0.05
    vx = float((0.4 + 0.2 * rng.random()) * nx * H3)
    vy = float((0.4 + 0.2 * rng.random()) * ny * H3)
    x = torch.arange(nx, device="cuda", dtype=torch.float64) * H3 - vx
    y = torch.arange(ny, device="cuda", dtype=torch.float64) * H3 - vy
    z = torch.arange(nz, device="cuda", dtype=torch.float64) * H3 - (nz - 1) * H3
    X, Y, Z = x[None, None, :], y[None, :, None], z[:, None, None]
    d = torch.sqrt(X * X + Y * Y + Z * Z + (0.5 * r) ** 2)
    T = 300.0 + 2500.0 * P / 350.0 * (0.5 * r / d) * torch.exp(-(d + X) / 0.08)
    row = [vx, vy, 0.0, 1.0, 1.0, 1e-6, P]
    return T.float().reshape(-1).contiguous(), row, {"T_amb": 300.0, "laser_radius": r,
                                                     "laser_depth": r}


def _net(case, seed):
    import surrogate as S
    return S.UNet(channels=tuple(int(c) for c in case["channels"].split(",")), seed=seed)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _conv_inputs(case, seed):
    g = _gen(seed)
    sh = (case["nb"], case["D"], case["H"], case["W"])
    ci, co = case["ci"], case["co"]
    rn = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    return {"X": rn(*sh, ci).clamp_min_(0).to(torch.bfloat16),  # a ReLU layer's output
            "W": (rn(27, co, ci) * (2.0 / (27 * ci)) ** 0.5).to(torch.bfloat16),
            "b": rn(co) * 0.1,
            # backward: the layer's stored activation and the gradient from above
            "A": rn(*sh, co).clamp_min_(0), "dA": rn(*sh, co) / (sh[0] * sh[1] * sh[2] * sh[3])}


# ---------------------------------------------------------------------------
# prepare, run, work
# ---------------------------------------------------------------------------

WARM_STEPS = 10  # steps that give every window of a study a melt pool


def _sizes(case):
    """Element counts of a study's instances: one size, or the study's own in
    turn (ex = 0)."""
    if case.get("ex"):
        return [(case["ex"], case["ey"], case["ez"])] * case["n"]
    return [W.BATCH_SIZES[i % len(W.BATCH_SIZES)] for i in range(case["n"])]


def _instances(case, seed):
    return [W.batch_instances(n=1, seed=1000 * seed + i, sizes=[el])[0]
            for i, el in enumerate(_sizes(case))]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("l1_step", "row", "dwell"):
        st = _time_loop(case, seed)
        st["rows"] = np.array([r for c in st["lap"] for r in c], np.float64)
    elif kind == "windows":
        import batch as B
        inst = _instances(case, seed)
        bt = B.Batch.from_instances(inst, stream=_stream())
        rows = [W.batch_rows(inst, s) for s in range(64)]
        for s in range(WARM_STEPS):
            bt.step(rows[s])
        st = {"bt": bt, "rows": rows, "at": WARM_STEPS, "n": case["n"], "views": {},
              "owner": bt}
    elif kind == "stacks":
        import batch as B
        from createPath import parsingGcode
        import computeFunctions as cf
        tmp = tempfile.TemporaryDirectory(prefix="gomelt_perf_")
        decks = []
        for i, el in enumerate(_sizes(case)):
            inp, g = W.stack_decks(n=1, seed=1000 * seed + i, sizes=[el])[0]
            first, second = g.split("\n")[:2]
            d = _write(inp, f"{first}\n{second}\n{first.replace('G0', 'G1')}\n",
                       os.path.join(tmp.name, f"s{i}"))
            # many laps of the toolpath: the runs read it chunk by chunk
            nm = cf.SetupNonmesh(d["nonmesh"])
            n = parsingGcode(nm, cf.SetupProperties(d["properties"]), 0.0)
            with open(nm["toolpath"]) as fh:
                lap = fh.read()
            with open(nm["toolpath"], "w") as fh:
                fh.write(lap * (60000 // n + 1))
            d["nonmesh"]["use_txt"] = 1
            decks.append(d)
        stacks = B.Stacks(decks)
        stacks.step()  # the single-step chunk
        st = {"stacks": stacks, "tmp": tmp, "views": {}, "owner": stacks}
    elif kind == "conv":
        st = _conv_inputs(case, seed)
        st["dW"] = torch.zeros(st["W"].shape, device="cuda")
        st["db"] = torch.zeros(case["co"], device="cuda")
    elif kind == "jump":
        import _native as N
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        T, row, props = _window(seed, nx, ny, nz)
        st = {"net": _net(case, seed), "T": T, "row": row, "inst": {"properties": props},
              "grid": N.gm_grid.make([nx, ny, nz], [0.0, 0.0, -(nz - 1) * H3], [H3] * 3),
              "face": torch.full_like(T, 300.0),
              "X": torch.empty((1, nz, ny, nx, 16), dtype=torch.bfloat16, device="cuda")}
    else:
        net = _net(case, seed)
        X, t = _batch(case, seed)
        st = {"net": net, "X": X, "target": t,
              "loss": torch.zeros(1, dtype=torch.float64, device="cuda")}
    st["kind"] = kind
    return st


def _batch(case, seed):
    """Training windows (bf16, channels last) and their targets: the change
    of the window's field as a pool moves on."""
    nb, D, H, Wd = case["nb"], case["D"], case["H"], case["W"]
    X = torch.zeros((nb, D, H, Wd, 16), dtype=torch.bfloat16, device="cuda")
    t = torch.empty((nb, D * H * Wd), device="cuda")
    for b in range(nb):
        T, row, _ = _window(1000 * seed + b, Wd, H, D)
        x = (T - 300.0) / T_SCALE
        X[b, ..., 0] = x.reshape(D, H, Wd).to(torch.bfloat16)
        X[b, ..., 2] = _intensity(row, Wd, H, D).to(torch.bfloat16)
        X[b, ..., 3] = row[6] / P_SCALE
        t[b] = torch.roll(x, 1) - x
    return X, t.reshape(-1)


def _intensity(row, nx, ny, nz, r=0.05):
    x = torch.arange(nx, device="cuda", dtype=torch.float64) * H3 - row[0]
    y = torch.arange(ny, device="cuda", dtype=torch.float64) * H3 - row[1]
    z = torch.arange(nz, device="cuda", dtype=torch.float64) * H3 - (nz - 1) * H3
    e = lambda a: torch.exp(-3.0 * a * a / r ** 2)  # noqa: E731
    return e(z)[:, None, None] * e(y)[None, :, None] * e(x)[None, None, :]


def run(state):
    kind = state["kind"]
    if kind == "l1_step":
        state["at"] = state["at"] % (len(state["lap"]) - 1) + 1
        state["run"].step_chunk(state["lap"][state["at"]])
        return _levels_out(state, state["run"].Levels)
    if kind == "row":
        import computeFunctions as cf
        r = state["run"]
        pos = state["rows"][(r.subcycle[2] + state["at"]) % len(state["rows"])]
        state["at"] += 1
        _, r.Shapes, r.LInterp, r.move_hist = cf.moveEverything(
            pos, r.laser_start, r.Levels, r.move_hist, r.LInterp, r.eng.r12, r.eng.r23,
            r.Properties["layer_height"])
        _, reset = cf.stepGOMELT(r.Levels, r.ne_nn, r.tmp_ne_nn, r.Shapes, r.LInterp, pos,
                                 r.Properties, pos[5], pos[6], r.substrate)
        return dict(_levels_out(state, r.Levels), reset=_view(state, reset))
    if kind == "dwell":
        import computeFunctions as cf
        r = state["run"]
        cf.stepGOMELTDwellTime(r.Levels, r.tmp_ne_nn, r.ne_nn, r.Properties, 1e-4, r.substrate)
        return {"T1": _view(state, r.Levels[1]["T0"]), "S1_1": _view(state, r.Levels[1]["S1"])}
    if kind == "windows":
        bt = state["bt"]
        bt.step(state["rows"][state["at"] % len(state["rows"])])
        state["at"] += 1
        return [_view(state, bt._field(i, f)) for i in range(state["n"]) for f in (0, 1)]
    if kind == "stacks":
        if not state["stacks"].step():
            raise RuntimeError("the toolpath has ended")
        keep = ("T1", "T2", "Tp2", "T3", "Tp3", "S1_3", "S2_3")
        return [{k: v for k, v in _levels_out(state, r.Levels, False).items() if k in keep}
                for r in state["stacks"].runs]
    import surrogate as S
    if kind == "conv":
        Y, Yb = S.conv3d(state["X"], state["W"], state["b"], relu=True)
        S.zero(state["dW"])
        S.zero(state["db"])
        dZ = S.relu_bias_bwd(state["dA"], state["A"], state["db"])
        S.conv3d_bwd_weight(state["X"], dZ, state["dW"])
        dX, _ = S.conv3d_bwd_data(dZ, state["W"], want_bf16=False)
        return {"Y": Y, "Yb": Yb, "dZ": dZ, "dW": state["dW"], "db": state["db"], "dX": dX}
    if kind == "jump":
        S.window_input(state["inst"], state["grid"], state["T"], state["face"], state["row"],
                       state["X"][0])
        Tn = S.apply_jump(state["net"], state["X"], state["T"], state["face"], state["grid"])
        return {"T": Tn, "Y": state["net"].head.A}
    net = state["net"]
    for c in net.layers():
        for g in c.grads:
            S.zero(g)
    S.zero(state["loss"])
    Y = net.forward(state["X"])
    net.backward(S.mse(Y, state["target"], state["loss"]))
    return {"Y": Y, "grads": [list(c.grads) for c in net.layers()]}


def _nodes(case):
    """(L1, L2, L3 nodes, L1 steps' N2, N3) of a deck."""
    if case["deck"] == "track":
        return 41 * 41 * 21, 41 * 41 * 21, 41 * 41 * 21
    if case["deck"] == "part":
        return 201 * 201 * 51, 101 * 101 * 51, 101 * 101 * 51
    n = (case["ex"] + 1) * (case["ey"] + 1) * (case["ez"] + 1)
    return n, n, n


def _conv_flops(nvox, ci, co):
    return 2.0 * 27.0 * nvox * ci * co


def _net_flops(case, nvox):
    """Forward operations of the network, and those of its first layer."""
    ch = [int(c) for c in case["channels"].split(",")]
    f = first = _conv_flops(nvox, 16, ch[0])
    w = 27 * 16 * ch[0]
    for l, c in enumerate(ch):
        nv = nvox / 8 ** l
        if l:
            f += _conv_flops(nv, ch[l - 1], c)
            w += 27 * ch[l - 1] * c
        f += _conv_flops(nv, c, c)
        w += 27 * c * c
        if l + 1 < len(ch):
            f += _conv_flops(nv, c + ch[l + 1], c) + _conv_flops(nv, c, c)
            w += 27 * c * (2 * c + ch[l + 1])
    f += _conv_flops(nvox, ch[0], 16)
    w += 27 * ch[0] * 16
    return f, first, w


# operations of one node of an explicit step: the 27-point product with
# element-mean conductivity, the lumped mass and the two property laws
NODE_FLOPS = 100.0


def work(case):
    kind = case["kind"]
    if kind in ("l1_step", "row"):
        n1, n2, n3 = _nodes(case)
        # T and S1 of L1; T, T' and the phase bytes of L2 and L3; melt time
        # of the L3 window: each read and written once
        b = 2.0 * (8 * n1 + 9 * n2 + (8 + 2 + 8) * n3)
        # predictor and corrector: 2 L1, 2 N2 L2 and 2 N2 N3 L3 solves
        k2, k3 = (20, 200) if kind == "l1_step" else (2, 2)
        return {"bytes": b, "flops": NODE_FLOPS * (2 * n1 + k2 * n2 + k3 * n3)}
    if kind == "dwell":
        n1 = _nodes(case)[0]
        return {"bytes": 2.0 * 8 * n1, "flops": NODE_FLOPS * n1}
    if kind == "windows":
        n = sum((a + 1) * (b + 1) * (c + 1) for a, b, c in _sizes(case))
        return {"bytes": 10.0 * n, "flops": NODE_FLOPS * n}
    if kind == "stacks":
        n = sum((a + 1) * (b + 1) * (c + 1) for a, b, c in _sizes(case))
        return {"bytes": 2.0 * (8 + 9 + 18) * n, "flops": NODE_FLOPS * 222 * n}
    if kind == "conv":
        ci, co = case["ci"], case["co"]
        nv = case["nb"] * case["D"] * case["H"] * case["W"]
        return {"bytes": nv * (2.0 * ci + 4 * ci + (4 + 2 + 4 + 4 + 2) * co) + 27.0 * ci * co * 6,
                "flops": 3 * _conv_flops(nv, ci, co)}
    if kind == "jump":
        nv = case["nx"] * case["ny"] * case["nz"]
        f, _, w = _net_flops(case, nv)
        return {"bytes": nv * (4.0 * 3 + 32 + 64) + 2.0 * w, "flops": f}
    nv = case["nb"] * case["D"] * case["H"] * case["W"]
    f, first, w = _net_flops(case, nv)
    return {"bytes": nv * (32.0 + 4 + 64) + 6.0 * w, "flops": 3 * f - first}


# ---------------------------------------------------------------------------
# The same results in 64 bits, from the definitions alone
# ---------------------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind == "windows":
        out = []
        for inst in _instances(case, seed):
            out += [_window_steps(inst, WARM_STEPS + 1), None]
        return out
    if kind == "conv":
        return _conv_exact(_conv_inputs(case, seed))
    if kind == "jump":
        return _jump_exact(case, seed)
    if kind == "grad":
        return _grad_exact(case, seed)
    return None  # a whole L1 step or row of three coupled levels


def _along(a, axis, lo, mid, hi):
    """sum of a 3-point stencil along an axis; lo/mid/hi: one value per node"""
    a = a.movedim(axis, -1)
    out = mid * a
    out[..., 1:] += lo[1:] * a[..., :-1]
    out[..., :-1] += hi[:-1] * a[..., 1:]
    return out.movedim(-1, axis)


def _window_steps(inst, steps):
    """`steps` explicit lumped-mass steps of one window from T_amb: constant
    k and rho cp (the study's material), Gaussian source and convection on the
    top, faces and floor at T_amb.  T is (z, y, x)."""
    p = inst["properties"]
    h, dt, Ta = inst["h"], inst["dt"], p["T_amb"]
    k = p["thermal_conductivity_bulk_a0"] * 1e-3
    rc = p["density"] * p["heat_capacity_solid_a0"]
    n = [e + 1 for e in inst["elements"]]

    def oned(m):
        end = torch.ones(m, dtype=torch.float64, device="cuda")
        end[0] = end[-1] = 0.5
        off = torch.ones_like(end)
        return ((-off / h, 2 * end / h, -off / h), (off * h / 6, 4 * end * h / 6, off * h / 6),
                end * h)

    (Kx, Mx, lx), (Ky, My, ly), (Kz, Mz, lz) = (oned(m) for m in n)
    lump = lz[:, None, None] * ly[None, :, None] * lx[None, None, :]

    def axis_source(m, x0, c, r):
        """nodal integrals of exp(-3 (x - c)^2 / r^2), two Gauss points an element"""
        f = torch.zeros(m, dtype=torch.float64, device="cuda")
        e = torch.arange(m - 1, dtype=torch.float64, device="cuda")
        for g in (-1.0, 1.0):
            s = 0.5 * (1.0 + g / 3.0 ** 0.5)
            v = torch.exp(-3.0 * (x0 + (e + s) * h - c) ** 2 / r ** 2) * h / 2
            f[:-1] += (1 - s) * v
            f[1:] += s * v
        return f

    T = torch.full((n[2], n[1], n[0]), float(Ta), dtype=torch.float64, device="cuda")
    for s in range(steps):
        row = [float(v) for v in W.batch_rows([inst], s)[0]]
        r, d = p["laser_radius"], p["laser_depth"]
        q0 = 6 * np.sqrt(3) * row[6] * p["laser_absorptivity"] / (r * r * d * np.pi ** 1.5)
        F = q0 * (axis_source(n[2], -(n[2] - 1) * h, row[2], d)[:, None, None]
                  * axis_source(n[1], 0.0, row[1], r)[None, :, None]
                  * axis_source(n[0], 0.0, row[0], r)[None, None, :])
        F[-1] += p["h_conv"] * _along(_along(Ta - T[-1], 0, *My), 1, *Mx)
        mx, my = _along(T, 2, *Mx), _along(T, 1, *My)
        KT = k * (_along(_along(_along(T, 2, *Kx), 1, *My), 0, *Mz)
                  + _along(_along(mx, 1, *Ky), 0, *Mz)
                  + _along(_along(my, 2, *Mx), 0, *Kz))
        Tn = (T + row[5] * (F - KT) / (rc * lump)).clamp_min(Ta)
        Tn[0] = Ta
        Tn[:, 0] = Tn[:, -1] = Ta
        Tn[:, :, 0] = Tn[:, :, -1] = Ta
        T = Tn
    return T.reshape(-1)


def _shifted(X, tap):
    """X moved by a tap of the 3 x 3 x 3 kernel, zero outside: (nvox, C)."""
    dz, dy, dx = tap // 9 - 1, (tap // 3) % 3 - 1, tap % 3 - 1
    out = torch.zeros_like(X)
    cut = lambda d, n: (slice(max(0, -d), n - max(0, d)), slice(max(0, d), n - max(0, -d)))  # noqa: E731
    (oz, iz), (oy, iy), (ox, ix) = (cut(d, X.shape[1 + a]) for a, d in enumerate((dz, dy, dx)))
    out[:, oz, oy, ox] = X[:, iz, iy, ix]
    return out.reshape(-1, X.shape[4])


def _conv64(X, Wk):
    Y = sum(_shifted(X, t) @ Wk[t].t().contiguous() for t in range(27))
    return Y.reshape(X.shape[:4] + (Wk.shape[1],))


def _conv64_data(dY, Wk):
    dX = sum(_shifted(dY, 26 - t) @ Wk[t] for t in range(27))
    return dX.reshape(dY.shape[:4] + (Wk.shape[2],))


def _conv64_weight(X, dY):
    d = dY.reshape(-1, dY.shape[4]).t().contiguous()
    return torch.stack([d @ _shifted(X, t) for t in range(27)])


def _conv_exact(s):
    X, Wk, b, A, dA = (s[k].double() for k in ("X", "W", "b", "A", "dA"))
    Y = (_conv64(X, Wk) + b).clamp_min(0)
    g = torch.where(A > 0, dA, torch.zeros_like(dA))
    dZ = g.to(torch.bfloat16).double()  # the layer's gradient as the products take it
    return {"Y": Y, "Yb": Y, "dZ": g, "dW": _conv64_weight(X, dZ), "db": g.sum((0, 1, 2, 3)),
            "dX": _conv64_data(dZ, Wk)}


def _pool64(X):
    nb, D, H, Wd, c = X.shape
    return X.reshape(nb, D // 2, 2, H // 2, 2, Wd // 2, 2, c).mean((2, 4, 6))


def _up64(X):
    return X.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)


def _net64(net, X, keep=None):
    """Forward pass of the network in 64 bits on its bf16 weights; `keep`
    collects (layer, input, pre-activation sign) for the backward pass."""
    def layer(c, x):
        y = _conv64(x, c.wb.double()) + c.b.double()
        y = y.clamp_min(0) if c.relu else y
        if keep is not None:
            keep[c] = (x, y)
        return y

    x, skips = X, []
    for l, (c1, c2) in enumerate(net.enc):
        x = layer(c2, layer(c1, x))
        skips.append(x)
        if l + 1 < len(net.enc):
            x = _pool64(x)
    for k, (c1, c2) in enumerate(net.dec):
        x = torch.cat([skips[len(net.ch) - 2 - k], _up64(x)], 4)
        x = layer(c2, layer(c1, x))
    return layer(net.head, x)


def _grad_exact(case, seed):
    net = _net(case, seed)
    X, t = _batch(case, seed)
    keep, grads = {}, {}
    Y = _net64(net, X.double(), keep)
    nv = t.numel()
    dY = torch.zeros_like(Y)
    dY[..., 0] = (Y[..., 0] - t.double().reshape(Y.shape[:4])) / nv

    def back(c, dA, need=True):
        x, y = keep.pop(c)
        dZ = torch.where(y > 0, dA, torch.zeros_like(dA)) if c.relu else dA
        grads[c] = [_conv64_weight(x, dZ), dZ.sum((0, 1, 2, 3))]
        return _conv64_data(dZ, c.wb.double()) if need else None

    g = back(net.head, dY)
    skip = [None] * len(net.ch)
    for k in reversed(range(len(net.dec))):
        c1, c2 = net.dec[k]
        l = len(net.ch) - 2 - k
        g = back(c1, back(c2, g))
        skip[l], du = g[..., :net.ch[l]], g[..., net.ch[l]:]
        nb, D, H, Wd, c = du.shape
        g = du.reshape(nb, D // 2, 2, H // 2, 2, Wd // 2, 2, c).sum((2, 4, 6))
    for l in range(len(net.ch) - 1, -1, -1):
        c1, c2 = net.enc[l]
        g = g + skip[l] if skip[l] is not None else g
        g = back(c1, back(c2, g), need=l > 0)
        if l > 0:
            g = _up64(g) / 8.0
    return {"Y": Y, "grads": [grads[c] for c in net.layers()]}


def _jump_exact(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    T, row, p = _window(seed, nx, ny, nz)
    T3 = T.double().reshape(nz, ny, nx)
    inside = torch.zeros((nz, ny, nx), dtype=torch.bool, device="cuda")
    inside[1:, 1:-1, 1:-1] = True  # faces x, y and z = 0 are held
    X = torch.zeros((1, nz, ny, nx, 16), dtype=torch.float64, device="cuda")
    X[0, ..., 0] = (T3 - 300.0) / T_SCALE
    X[0, ..., 2] = _intensity(row, nx, ny, nz)
    X[0, ..., 3] = row[6] / P_SCALE
    X = X.to(torch.bfloat16).double()
    Y = _net64(_net(case, seed), X)
    Tn = torch.where(inside, (T3 + T_SCALE * Y[0, ..., 0]).clamp_min(300.0),
                     torch.full_like(T3, 300.0))
    return {"T": Tn.reshape(-1), "Y": Y}
