"""The work that a program has this library do, as measurable cases.

A case is one call (or one training step) through the package's public entry
points: the FFT matvec (`Context.matvec`, `matvec_batched`, `matvec_c128`),
the tile inverses (`tiles.Tiles.apply`), the learned network
(`fno.Preconditioner.forward` / `backward`) and the solvers (`Context.gmres`,
`Context.fgmres`, `block.solve_map`).  Sizes are those of the benchmark
workloads (N = 512 binary maps, N = 1024 in FP64, 16 right-hand sides per
map), of the tests' small grids, and odd ones between them.
"""
import math

import numpy as np
import torch

from cugmres_amd import _lib, block, fno, problems, solver, sweep
from cugmres_amd.tiles import Tiles

_MODES = {"forward": _lib.OP_FORWARD, "adjoint": _lib.OP_ADJOINT, "green": _lib.OP_GREEN}


def listed():
    return [
        # the smallest call: one product on the CPU workload's 64 x 64 grid (latency and launches)
        {"name": "matvec_n64", "op": "matvec", "N": 64, "batch": 1, "mode": "forward"},
        # an odd grid (embedding 3 * 2^8) and the transposed product of gradient solves
        {"name": "matvec_adjoint_n301_b2", "op": "matvec", "N": 301, "batch": 2, "mode": "adjoint"},
        # the batched workload's product: 16 plane waves on one map at the benchmark size
        {"name": "matvec_n512_b16", "op": "matvec", "N": 512, "batch": 16, "mode": "forward"},
        # the FP64 product of the mixed-precision refinement workload
        {"name": "matvec_c128_n1024", "op": "matvec_c128", "N": 1024, "mode": "forward"},
        # the reference's own problem (eps = 2.25 disk, x0 = b) solved to 1e-6 with GMRES(30)
        {"name": "gmres_disk_n512", "op": "gmres", "N": 512, "restart": 30},
        # one Krylov step's tile inverses on the benchmark map: 128 x 128 tiles, one vector
        {"name": "tiles_t128_n512", "op": "tiles", "N": 512, "T": 128, "batch": 1},
        # the same for the 16 right-hand sides of one map (block GMRES)
        {"name": "tiles_t128_n512_b16", "op": "tiles", "N": 512, "T": 128, "batch": 16},
        # the default tile side (dense inverses), four right-hand sides
        {"name": "tiles_t16_n256_b4", "op": "tiles", "N": 256, "T": 16, "batch": 4},
        # one Krylov step's network pass at the benchmark size
        {"name": "network_n512", "op": "network", "N": 512, "batch": 1},
        # one training step of the network at the trainer's default size: forward, backward
        {"name": "network_train_n256_b8", "op": "network_train", "N": 256, "batch": 8},
        # block GMRES over 16 plane waves of one map to 1e-6
        {"name": "block_n256_s16", "op": "block", "N": 256, "T": 64, "s": 16},
        # one system to 1e-6 with the tile inverses and a long recurrence, the whole basis in HBM
        {"name": "fgmres_n512_t128", "op": "fgmres", "N": 512, "T": 128, "restart": 400},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["matvec", "matvec", "matvec_c128", "gmres", "tiles", "tiles", "network", "network_train",
                     "block", "fgmres"])
    if op == "matvec":
        N = _log_int(rng, 24, 1100)
        batch = min(_log_int(rng, 1, 32), max(1, 16 * 512 * 512 // (N * N)))
        return {"op": op, "N": N, "batch": batch, "mode": rng.choice(["forward", "adjoint", "green"])}
    if op == "matvec_c128":
        return {"op": op, "N": _log_int(rng, 24, 1024), "mode": rng.choice(["forward", "adjoint", "green"])}
    if op == "gmres":
        return {"op": op, "N": rng.choice([64, 96, 128, 192, 256, 384, 512, 150, 333]),
                "restart": rng.choice([20, 30, 49])}
    if op == "tiles":
        T = rng.choice([8, 16, 32, 64, 128])
        top = {8: 512, 16: 512, 32: 256, 64: 512, 128: 512}[T]
        N = T * rng.randint(max(1, 64 // T), top // T)
        return {"op": op, "N": N, "T": T, "batch": _log_int(rng, 1, 16)}
    if op == "network":
        N = 64 * rng.randint(1, 8)
        return {"op": op, "N": N, "batch": min(_log_int(rng, 1, 16), max(1, 4 * 512 * 512 // (N * N)))}
    if op == "network_train":
        N = 64 * rng.randint(1, 6)
        return {"op": op, "N": N, "batch": min(_log_int(rng, 1, 12), max(1, 8 * 256 * 256 // (N * N)))}
    if op == "block":
        T = rng.choice([32, 64])
        return {"op": op, "N": rng.choice([64, 128, 192, 256]), "T": T, "s": rng.randint(2, 16)}
    T = rng.choice([64, 128])
    return {"op": op, "N": T * rng.randint(2, 512 // T), "T": T, "restart": rng.randint(300, 400)}


# ---- inputs ----------------------------------------------------------------


def _map(N, blk, seed, eps_hi=problems.EPS_HI):
    """The benchmark's binary map: blk x blk cells over the central 75 %."""
    return problems.block_eps_map(N, blk, 0.5, 0.75, seed=seed, eps_hi=eps_hi) - 1.0


def _angles(count, seed):
    r = np.random.default_rng(seed)
    return 2.0 * math.pi * r.random(count)


def _waves(N, count, seed):
    """`count` plane waves on the map's grid, complex128 (count, N*N)."""
    i = np.arange(N, dtype=np.float64)
    return np.stack([np.outer(np.exp(-1j * problems.KH * math.cos(t) * i),
                              np.exp(-1j * problems.KH * math.sin(t) * i)).reshape(-1) for t in _angles(count, seed)])


def _residuals(N, count, seed):
    """Krylov vectors as the solvers hand them on: unit-norm complex noise."""
    r = np.random.default_rng(seed)
    v = r.standard_normal((count, N * N, 2)).astype(np.float32)
    v = (v[..., 0] + 1j * v[..., 1]).astype(np.complex64)
    return (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.complex64)


def _disk(N):
    """The reference's problem: k, chi on the eps = 2.25 disk."""
    k = 2.0 * 3.14 / (N / 6.0)
    return k, sweep.reference_mask(N).reshape(-1) * (1.25 * k * k)


def _inputs(case, seed):
    """The case's numbers on the host, the same for prepare() and exact()."""
    op, N = case["op"], case["N"]
    if op == "matvec":
        return {"chi": _map(N, 8, seed).reshape(-1).astype(np.float32), "x": _residuals(N, case["batch"], seed)}
    if op == "matvec_c128":
        return {"chi": _map(N, 8, seed).reshape(-1), "x": _residuals(N, 1, seed)[0].astype(np.complex128)}
    if op == "gmres":
        k, chi = _disk(N)
        i = np.exp(-1j * (k * np.arange(N, dtype=np.float64) + _angles(1, seed)[0]))
        return {"k": k, "chi": chi.astype(np.float32), "b": np.repeat(i, N).astype(np.complex64)}
    if op == "tiles":
        return {"chi": _map(N, 8, seed).reshape(-1).astype(np.float32), "x": _residuals(N, case["batch"], seed)}
    if op in ("network", "network_train"):
        B = case["batch"]
        v = _residuals(N, B, seed)
        r = np.random.default_rng(seed + 1)
        dz = (r.standard_normal((B, N * N)) + 1j * r.standard_normal((B, N * N))).astype(np.complex64) / np.float32(N * B)
        return {"chi": np.stack([_map(N, 8, seed * 100 + b).reshape(-1) for b in range(B)]).astype(np.float32),
                "v": v, "dz": dz, "params": fno.init_params(seed, zero_out=False)}
    if op == "block":
        return {"chi": _map(N, 8, seed, eps_hi=2.25).reshape(-1).astype(np.float32),
                "b": _waves(N, case["s"], seed).astype(np.complex64)}
    return {"chi": _map(N, 8, seed, eps_hi=2.25).reshape(-1).astype(np.float32),
            "b": _waves(N, 1, seed)[0].astype(np.complex64)}


def prepare(case, seed):
    op, N = case["op"], case["N"]
    d = _inputs(case, seed)
    ctx = solver.Context(N)
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).to(ctx.device) for k, v in d.items()
           if isinstance(v, np.ndarray)}
    s = {"case": case, "ctx": ctx, **dev}
    if op == "gmres":
        s["gamma"] = ctx.spectrum_reference(d["k"], 0.5, 0.0)
        s["out"] = torch.empty_like(s["b"])
    elif op in ("matvec_c128", "fgmres"):
        s["gamma"], s["gamma64"] = ctx.spectrum_helmholtz(problems.KH, fp64=True)
    elif op not in ("network", "network_train"):
        s["gamma"] = ctx.spectrum_helmholtz(problems.KH)
    if op in ("matvec", "matvec_c128", "tiles"):
        s["out"] = torch.empty_like(s["x"])
    if op in ("tiles", "block", "fgmres"):
        s["tiles"] = Tiles(ctx, case["T"], 1).factor(ctx.block_helmholtz(problems.KH), s["chi"])
    if op == "fgmres":
        ctx.set_flexible_fp64(s["gamma64"])
    if op in ("network", "network_train"):
        s["net"] = fno.Preconditioner(ctx, batch=case["batch"], params=d["params"])
    if op == "network_train":
        s["grad"] = torch.empty(fno.NUM_PARAMS, dtype=torch.float32, device=ctx.device)
    return s


def run(state):
    case, ctx = state["case"], state["ctx"]
    op = case["op"]
    if op == "matvec":
        x, mode = state["x"], _MODES[case["mode"]]
        if case["batch"] == 1:
            return ctx.matvec(state["gamma"], state["chi"], x, mode, out=state["out"])
        return ctx.matvec_batched(state["gamma"], state["chi"], x, mode, out=state["out"])
    if op == "matvec_c128":
        return ctx.matvec_c128(state["gamma64"], state["chi"], state["x"], _MODES[case["mode"]], out=state["out"])
    if op == "gmres":  # x0 = b, as the reference starts
        x = state["out"].copy_(state["b"])
        return ctx.gmres(state["gamma"], state["chi"], state["b"], x, restart=case["restart"], tol=1e-6,
                         max_cycles=100)[0]
    if op == "tiles":
        return state["tiles"].apply(state["x"], out=state["out"])
    if op == "network":
        return state["net"].forward(state["chi"], state["v"])
    if op == "network_train":
        z = state["net"].forward(state["chi"], state["v"], train=True)
        return z, state["net"].backward(state["dz"], grad=state["grad"])
    if op == "block":
        return block.solve_map(ctx, state["gamma"], state["chi"], state["b"], tiles=state["tiles"], restart=64,
                               tol=1e-6, max_cycles=6)[0]
    return ctx.fgmres(state["gamma"], state["chi"], state["b"], precond=state["tiles"], restart=case["restart"],
                      tol=1e-6, max_cycles=1, stall_ratio=0.0)[0]


def _cells(chi):
    return int(np.count_nonzero(chi))


def work(case):
    """Bytes and operations of one pass that no implementation can leave out."""
    op, N = case["op"], case["N"]
    n = N * N
    fft = 2 * 5.0 * (2 * N) ** 2 * math.log2(4 * n)   # forward and inverse on the embedding
    if op == "matvec":
        b = case["batch"]
        return {"bytes": 16 * n * b + 4 * n + 8 * (N + 1) ** 2, "flops": b * fft}
    if op == "matvec_c128":
        return {"bytes": 32 * n + 8 * n + 16 * (N + 1) ** 2, "flops": fft}
    if op == "gmres":  # the reference problem takes about 58 steps; x, b in, x out, the basis written once
        return {"bytes": 8 * n * 58 + 24 * n, "flops": 58 * fft}
    if op == "tiles":
        T, b = case["T"], case["batch"]
        if T <= 32:
            e = (N // T) ** 2 * T ** 4
            return {"bytes": 8 * e + 16 * n * b, "flops": 8.0 * e * b}
        # W of the cells with chi != 0, its lower triangle in FP16 complex
        m = _map(N, 8, 0).reshape(N // T, T, N // T, T).transpose(0, 2, 1, 3).reshape(-1, T * T)
        c = np.count_nonzero(m, axis=1).astype(np.float64)
        e = float((c * (c + 1) / 2).sum())
        return {"bytes": 4 * e + 16 * n * b, "flops": 16.0 * e * b}
    if op in ("network", "network_train"):
        b = case["batch"]
        f = b * n * 4 * (2.0 * 32 * 32 + 4 * 16 * 32)   # dense channel products and the row transforms
        w = 4 * fno.NUM_PARAMS
        if op == "network":
            return {"bytes": 20 * n * b + w, "flops": f}
        return {"bytes": 28 * n * b + 2 * w, "flops": 3 * f}
    if op == "block":
        s = case["s"]
        return {"bytes": 16 * n * s * 16, "flops": 16.0 * s * fft}
    k = 0.53 * N   # steps to 1e-6 on these maps; each reads the basis twice
    return {"bytes": 8.0 * n * k * (k + 1), "flops": k * fft}


# ---- the same in 64 bits -----------------------------------------------------


def _hankel(z, order):
    """H_n^(1)(z), n = 0 or 1, complex128: Hankel's integral
    sqrt(2 / (pi z)) e^{i (z - n pi/2 - pi/4)} / Gamma(n + 1/2) int_0^inf e^{-u} u^{n-1/2} (1 + i u / 2z)^{n-1/2} du
    with u = s^2, by the trapezoidal rule (its error falls as exp(-2 pi sqrt(z) / h))."""
    z = z.to(torch.complex128)
    h = min(0.1, math.sqrt(float(z.real.min())) / 8.0)
    total = torch.zeros_like(z)
    for j in range(int(6.5 / h) + 1):
        q = (j * h) ** 2
        f = torch.sqrt(1.0 + 0.5j * q / z)
        w = h * (1.0 if j else 0.5) * 2.0 * math.exp(-q)
        total = total + (w / f if order == 0 else w * q * f)
    norm = math.gamma(order + 0.5)
    return torch.sqrt(2.0 / (math.pi * z)) * torch.exp(1j * (z - (order * 0.5 + 0.25) * math.pi)) * total / norm


def _generator(N, k, sr=None, sc=None):
    """g[|di|, |dj|] (N, N) complex128: the benchmark's operator for sr = None,
    else the reference's with its half-cell shift."""
    i = torch.arange(N, dtype=torch.float64)
    if sr is None:
        r = k * torch.sqrt(i[:, None] ** 2 + i[None, :] ** 2)
        r[0, 0] = k
        g = k * k * 0.25j * _hankel(r.to(_device()), 0)
        ka = torch.tensor(k / math.sqrt(math.pi), dtype=torch.float64)
        g[0, 0] = 0.5j * math.pi * ka * _hankel(ka, 1) - 1.0
        return g
    r = k * torch.sqrt((i[:, None] - sr) ** 2 + (i[None, :] - sc) ** 2)
    return 0.25j * _hankel(r.to(_device()), 0)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Operator:
    """x - G(chi x), x - chi G(x) and G(x) through a 2N x 2N embedding."""

    def __init__(self, g, chi, device):
        N = self.N = g.shape[0]
        t = torch.arange(2 * N, device=g.device)
        d = torch.where(t < N, t, 2 * N - t) % N          # offset N is zeroed: the cropped product never uses it
        E = g[d[:, None], d[None, :]]
        E[N, :] = 0
        E[:, N] = 0
        self.hat = torch.fft.fft2(E.to(device))
        self.chi = torch.as_tensor(np.asarray(chi, np.float64)).to(device).reshape(N, N)

    def green(self, x):
        N = self.N
        u = torch.fft.fft2(x.reshape(-1, N, N), s=(2 * N, 2 * N))
        return torch.fft.ifft2(u * self.hat)[:, :N, :N].reshape(x.shape)

    def __call__(self, x, mode="forward"):
        c = self.chi.reshape(-1)
        if mode == "forward":
            return x - self.green(x * c)
        return x - c * self.green(x) if mode == "adjoint" else self.green(x)


def _solve(op, b, tol=1e-11, m=1200):
    """Unrestarted GMRES in 64 bits for one right-hand side."""
    n = b.numel()
    beta = torch.linalg.vector_norm(b)
    V = torch.empty((m + 1, n), dtype=torch.complex128, device=b.device)
    H = np.zeros((m + 1, m), np.complex128)
    V[0] = b / beta
    for j in range(m):
        w = op(V[j])
        h = V[:j + 1].conj() @ w
        w = w - h @ V[:j + 1]
        h2 = V[:j + 1].conj() @ w
        w = w - h2 @ V[:j + 1]
        nw = float(torch.linalg.vector_norm(w))
        H[:j + 1, j] = (h + h2).cpu().numpy()
        H[j + 1, j] = nw
        V[j + 1] = w / nw
        if j % 32 == 31:
            e = np.zeros(j + 2, np.complex128)
            e[0] = float(beta)
            y = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)[0]
            if np.linalg.norm(e - H[:j + 2, :j + 1] @ y) <= tol * float(beta):
                return torch.as_tensor(y).to(b.device) @ V[:j + 1]
    return None


def _tiles_exact(g, chi, x, T, device):
    """(I - G_t diag(chi_t))^{-1} x_t on every tile, through the cells with chi != 0."""
    N = g.shape[0]
    gd = g.to(device)
    y = x.clone().reshape(-1, N, N)
    r = torch.arange(T, device=device).repeat_interleave(T)
    c = torch.arange(T, device=device).repeat(T)
    chi = torch.as_tensor(np.asarray(chi, np.float64)).to(device).reshape(N, N)
    corner = g[:T, :T]
    for a in range(N // T):
        for b in range(N // T):
            at = chi[a * T:(a + 1) * T, b * T:(b + 1) * T].reshape(-1)
            S = torch.nonzero(at).reshape(-1)
            if not S.numel():
                continue
            A = -gd[(r[S][:, None] - r[S][None, :]).abs(), (c[S][:, None] - c[S][None, :]).abs()]
            A.diagonal().add_(1.0 / at[S])
            v = x.reshape(-1, N, N)[:, a * T:(a + 1) * T, b * T:(b + 1) * T].reshape(-1, T * T)
            u = torch.zeros_like(v)
            u[:, S] = torch.linalg.solve(A, v[:, S].T.contiguous()).T
            y[:, a * T:(a + 1) * T, b * T:(b + 1) * T] += \
                _Operator(corner, np.zeros((T, T)), device).green(u).reshape(-1, T, T)
    return y.reshape(x.shape)


def _network(p, chi, v, N):
    """The network's definition on (B, N, N) inputs in 64 bits."""
    w = fno.unpack(p)
    a = torch.stack([chi * fno.CHI_SCALE, N * v.real, N * v.imag], dim=-1)
    h = a @ w["W_in"] + w["b_in"]
    rows = list(range(16)) + list(range(N - 16, N))
    for l in range(fno.LAYERS):
        hf = torch.fft.rfft2(h, dim=(1, 2))
        S = torch.view_as_complex(w[f"S{l}"].contiguous())
        sel = hf[:, rows][:, :, :fno.KY].permute(1, 2, 0, 3)                  # (kx, ky, B, c)
        mixed = torch.matmul(sel.contiguous(), S).permute(2, 0, 1, 3)
        full = torch.zeros_like(hf)
        full[:, :16, :fno.KY] = mixed[:, :16]
        full[:, N - 16:, :fno.KY] = mixed[:, 16:]
        pre = h @ w[f"W{l}"] + w[f"b{l}"] + torch.fft.irfft2(full, s=(N, N), dim=(1, 2))
        h = torch.nn.functional.gelu(pre, approximate="tanh") if l < fno.LAYERS - 1 else pre
    out = h @ w["W_out"] + w["b_out"]
    return w["s_id"] * v + torch.complex(out[..., 0], out[..., 1]) / N


def exact(case, seed):
    op, N = case["op"], case["N"]
    d = _inputs(case, seed)
    dev = _device()

    def up(a, dt):
        return torch.from_numpy(np.ascontiguousarray(a)).to(device=dev, dtype=dt)

    if op in ("matvec", "matvec_c128"):
        A = _Operator(_generator(N, problems.KH), d["chi"], dev)
        x = up(d["x"], torch.complex128)
        return A(x, case["mode"])
    if op == "gmres":
        A = _Operator(_generator(N, d["k"], 0.5, 0.0), d["chi"], dev)
        return _solve(A, up(d["b"], torch.complex128))
    if op == "tiles":
        if case["T"] == 128 and N > 512:
            return None
        return _tiles_exact(_generator(N, problems.KH), d["chi"], up(d["x"], torch.complex128), case["T"], dev)
    if op in ("network", "network_train"):
        p = up(d["params"], torch.float64).requires_grad_(op == "network_train")
        B = case["batch"]
        z = _network(p, up(d["chi"], torch.float64).reshape(B, N, N), up(d["v"], torch.complex128).reshape(B, N, N), N)
        if op == "network":
            return z.reshape(B, -1)
        dz = up(d["dz"], torch.complex128).reshape(B, N, N)
        g, = torch.autograd.grad((z.real * dz.real + z.imag * dz.imag).sum(), p)
        return z.detach().reshape(B, -1), g
    A = _Operator(_generator(N, problems.KH), d["chi"], dev)
    if op == "block":
        xs = [_solve(A, b) for b in up(d["b"], torch.complex128)]
        return None if any(x is None for x in xs) else torch.stack(xs)
    if N > 256:
        return None   # over 1200 unpreconditioned steps
    return _solve(A, up(d["b"], torch.complex128))
