"""Performance cases: the work a user of neon_amd has it do, through its public
entry points.

A case is a dict of plain values; `family` names the path:

  dense    DenseLattice.run: the lid-driven cavity on a dense grid, with
           bounce-back boxes and, as a convergence loop has it, the residual
  duct     DenseLattice.run_zouhe: a pressure-driven duct, Zou-He ends
  porous   BlockLattice.run: body-forced flow through a sphere pack on 8^3 blocks
  batch    CavityBatch.run: many uneven cavities with the convergence check
  refined  mgrid.MGrid.run and the read-back of every level's populations
  train    surrogate.UNet.train_step, the loss, the gradients and the weights
  predict  surrogate.UNet.forward
  conv     surrogate.conv3d_{fwd,bwd_data,bwd_weight}: one layer, both directions

`exact` evaluates the same passes in binary64 with plain torch: collide and
stream by rolled arrays, convolutions by shifted matrix products.
"""
import math

import numpy as np
import torch

import neon_amd as nx
from neon_amd import mgrid, surrogate
from neon_amd.abi import NX_CELL_BOUNCEBACK, NX_CELL_BULK, NX_CELL_MOVINGWALL, NX_CELL_UNDEFINED, NX_ZH_XMAX, NX_ZH_XMIN

BYTES = {"f64": 8, "f32": 4, "f32dev": 4, "f16dev": 2}
DTYPE = {"f64": torch.float64, "f32": torch.float32, "f32dev": torch.float32, "f16dev": torch.float16}
TYPESTR = {torch.float64: "<f8", torch.float32: "<f4", torch.float16: "<f2", torch.int16: "<i2"}
ULB = 0.05
_stream = None


def stream():
    """The one created stream that the flow solvers step on."""
    global _stream
    nx.init()
    if _stream is None:
        _stream = nx.Stream()
    return _stream.handle


class _Span:
    """Device memory that `owner` keeps, for torch.as_tensor."""

    def __init__(self, owner, ptr, count, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": (int(count),), "typestr": TYPESTR[dtype],
                                         "strides": None, "version": 3}


def span(owner, ptr, count, dtype):
    if dtype is torch.bfloat16:
        return span(owner, ptr, count, torch.int16).view(torch.bfloat16)
    return torch.as_tensor(_Span(owner, ptr, count, dtype), device="cuda")


def buffer_of(t):
    """A DeviceBuffer holding the tensor's values, and a tensor over it."""
    b = nx.DeviceBuffer(t.numel() * t.element_size())
    v = span(b, b.ptr, t.numel(), t.dtype)
    v.copy_(t.reshape(-1))
    return b, v


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


# ---- lattices -----------------------------------------------------------------

# D3Q19 population order of the library's fields (x, y, z)
C19 = [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (-1, -1, 0), (-1, 1, 0), (-1, 0, -1), (-1, 0, 1), (0, -1, -1), (0, -1, 1),
       (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, -1, 0), (1, 0, 1), (1, 0, -1), (0, 1, 1), (0, 1, -1)]
W19 = [1 / 3 if c == (0, 0, 0) else 1 / 18 if sum(map(abs, c)) == 1 else 1 / 36 for c in C19]
# D3Q27 order of the refined grid's KBC lattice: z fastest, each axis over 0, -1, 1
C27 = [(x, y, z) for x in (0, -1, 1) for y in (0, -1, 1) for z in (0, -1, 1)]
W27 = [(8 / 27, 2 / 27, 1 / 54, 1 / 216)[sum(map(abs, c))] for c in C27]


def opposite(C):
    return [C.index((-x, -y, -z)) for x, y, z in C]


def at_upstream(a, c):
    """a[..., z, y, x] taken at x - c (wrapping)."""
    return torch.roll(a, (c[2], c[1], c[0]), (-3, -2, -1))


def moments(f, C):
    rho = f.sum(0)
    u = [sum(c[a] * f[q] for q, c in enumerate(C) if c[a]) / rho for a in range(3)]
    return rho, u


def equilibrium(rho, u, C, W):
    usqr = 1.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    out = rho.new_empty((len(C),) + tuple(rho.shape))
    for q, c in enumerate(C):
        cu = 3.0 * (c[0] * u[0] + c[1] * u[1] + c[2] * u[2])
        out[q] = W[q] * rho * (1.0 + cu + 0.5 * cu * cu - usqr)
    return out


def pull(f, bulk, C):
    """Pull streaming; a link from a non-bulk cell returns the own opposite
    population plus the wall's (0 where there is no cell)."""
    opp, out = opposite(C), torch.empty_like(f)
    for q, c in enumerate(C):
        if c == (0, 0, 0):
            out[q] = f[q]
        else:
            out[q] = torch.where(at_upstream(bulk, c), at_upstream(f[q], c), f[opp[q]] + at_upstream(f[opp[q]], c))
    return out


def step19(f, bulk, omega, g=(0.0, 0.0, 0.0), ends=None):
    """One BGK step (Guo forcing g); ends = (x, density, sign) prescribes the
    density on planes of x by non-equilibrium bounce back, the unknown
    populations having c_x = sign."""
    p = pull(f, bulk, C19)
    rho, u = moments(p, C19)
    opp = opposite(C19)
    for x, value, sign in ends or ():
        s = p[..., x]
        m = sum(s[q] for q, c in enumerate(C19) if c[0] == 0)
        k = sum(s[q] for q, c in enumerate(C19) if c[0] == -sign)
        r = torch.full_like(m, value)
        un = [sign * (1.0 - (m + 2.0 * k) / r), torch.zeros_like(m), torch.zeros_like(m)]
        eq = equilibrium(r, un, C19, W19)
        for q, c in enumerate(C19):
            if c[0] == sign:
                s[q] = s[opp[q]] + eq[q] - eq[opp[q]]
        rho[..., x] = r
        for a in range(3):
            u[a][..., x] = un[a]
    if any(g):
        u = [u[a] + 0.5 * g[a] for a in range(3)]
    usqr = 1.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    ug = u[0] * g[0] + u[1] * g[1] + u[2] * g[2]
    for q, c in enumerate(C19):
        cu = c[0] * u[0] + c[1] * u[1] + c[2] * u[2]
        new = p[q] + omega * (W19[q] * rho * (1.0 + 3.0 * cu + 4.5 * cu * cu - usqr) - p[q])
        if any(g):
            cg = c[0] * g[0] + c[1] * g[1] + c[2] * g[2]
            new = new + (1.0 - 0.5 * omega) * W19[q] * rho * (3.0 * (cg - ug) + 9.0 * cu * cg)
        p[q] = torch.where(bulk, new, f[q])
    return p


# ---- geometry and starting flow -----------------------------------------------


def cavity(dim, boxes, geometry):
    """Classes [z, y, x] of a closed box with the lid at the last y plane and
    seeded bounce-back boxes with edges of 4 to 16 cells."""
    X, Y, Z = dim
    c = np.full((Z, Y, X), NX_CELL_BULK, np.uint8)
    rng = np.random.default_rng(geometry)
    for _ in range(boxes):
        lo, hi = [], []
        for n in (Z, Y, X):
            e = int(min(rng.integers(4, 17), max(1, n // 3)))
            s = int(rng.integers(1, max(2, n - 1 - e)))
            lo.append(s)
            hi.append(s + e)
        c[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] = NX_CELL_BOUNCEBACK
    c[:, :, [0, -1]] = c[:, [0, -1], :] = c[[0, -1]] = NX_CELL_BOUNCEBACK
    c[:, -1, :] = NX_CELL_MOVINGWALL
    return c


def sphere_pack(dim, spheres, geometry):
    """Solid mask [z, y, x] of seeded spheres of radius 6 to 20, periodic in x."""
    X, Y, Z = dim
    solid = torch.zeros((Z, Y, X), dtype=torch.bool, device="cuda")
    rng = np.random.default_rng(geometry)
    for _ in range(spheres):
        cx, cy, cz = (rng.uniform(0, n) for n in dim)
        r = rng.uniform(6.0, 20.0)
        ys = torch.arange(max(0, int(cy - r)), min(Y, int(cy + r) + 2), device="cuda")
        zs = torch.arange(max(0, int(cz - r)), min(Z, int(cz + r) + 2), device="cuda")
        xs = torch.arange(int(math.floor(cx - r)), int(cx + r) + 2, device="cuda")
        inside = ((zs - cz)[:, None, None] ** 2 + (ys - cy)[None, :, None] ** 2 + (xs - cx)[None, None, :] ** 2) < r * r
        for k in (-1, 0, 1):
            a, b = max(int(xs[0]), k * X), min(int(xs[0]) + xs.numel(), (k + 1) * X)
            if a < b:
                o = int(xs[0])
                solid[int(zs[0]):int(zs[0]) + zs.numel(), int(ys[0]):int(ys[0]) + ys.numel(), a - k * X:b - k * X] |= \
                    inside[:, :, a - o:b - o]
    return solid


def smooth_flow(dim, seed, scale):
    """(rho, u) of a few seeded sine modes: density near 1, speeds up to about `scale`."""
    X, Y, Z = dim
    gen = generator(seed)
    axes = [torch.arange(n, device="cuda", dtype=torch.float64) * (2.0 * math.pi / n) for n in (Z, Y, X)]
    fields = []
    for k in range(4):
        v = torch.zeros((Z, Y, X), device="cuda", dtype=torch.float64)
        for _ in range(3):
            r = torch.rand(7, generator=gen, device="cuda", dtype=torch.float64).tolist()
            m = [1 + int(3 * r[a]) for a in range(3)]
            w = [torch.sin(m[a] * axes[a] + 6.2832 * r[3 + a]) for a in range(3)]
            v += (r[6] - 0.5) * (w[0][:, None, None] * w[1][None, :, None] * w[2][None, None, :])
        fields.append(v)
    return 1.0 + 0.2 * scale * fields[0], [scale * v for v in fields[1:]]


def stored(full, bulk, storage):
    """Populations as the library stores them: f - w in bulk cells of the
    deviation types, f elsewhere."""
    if storage.endswith("dev"):
        w = torch.tensor(W19, device=full.device, dtype=torch.float64).view(-1, 1, 1, 1)
        full = torch.where(bulk, full - w, full)
    return (full.float() if storage == "f16dev" else full).to(DTYPE[storage])


def decoded(value, bulk, storage):
    full = value.double()
    if storage.endswith("dev"):
        w = torch.tensor(W19, device=full.device, dtype=torch.float64).view(-1, 1, 1, 1)
        full = torch.where(bulk, full + w, full)
    return full


def encoded(full, bulk, storage):
    """stored() without the rounding: what exact() returns."""
    if storage.endswith("dev"):
        w = torch.tensor(W19, device=full.device, dtype=torch.float64).view(-1, 1, 1, 1)
        full = torch.where(bulk, full - w, full)
    return full.reshape(-1)


def wall_values(cls, ulb, storage):
    """Populations of wall cells: 0, and the moving wall's -6 w c.u."""
    lid = torch.from_numpy(cls == NX_CELL_MOVINGWALL).cuda()
    f = torch.zeros((19,) + cls.shape, device="cuda", dtype=torch.float64)
    for q, c in enumerate(C19):
        f[q] = torch.where(lid, -6.0 * W19[q] * ulb * c[0], 0.0)
    return (f.float() if storage == "f16dev" else f).to(DTYPE[storage])


def flow_start(cls, seed, storage, scale, ulb=0.0):
    """Stored populations [19, z, y, x]: a smooth flow off equilibrium by a
    little noise in the bulk, the walls' values elsewhere."""
    Z, Y, X = cls.shape
    bulk = torch.from_numpy(cls == NX_CELL_BULK).cuda()
    rho, u = smooth_flow((X, Y, Z), seed, scale)
    f = equilibrium(rho, u, C19, W19)
    gen = generator(seed + 1)
    for q in range(19):
        f[q] *= 1.0 + 1e-4 * (torch.rand(f[q].shape, generator=gen, device="cuda", dtype=torch.float64) - 0.5)
    return torch.where(bulk, stored(f, bulk, storage), wall_values(cls, ulb, storage)), bulk


def cavity_omega(dim):
    nu = ULB * dim[1] / min(1000.0, 4.0 * min(dim))
    return 1.0 / (3.0 * nu + 0.5)


# ---- the refined cavity ---------------------------------------------------------


def shells(case):
    """Level lambdas of the refined cavity: level 0 within t0 cells of the
    walls, level 1 within t1, level 2 the rest; [z, y, x] masks."""
    N, out = case["edge"], []
    bounds = (0, N // 8, 3 * (N // 8), N)
    for l in range(3):
        a = np.arange((N + (1 << l) - 1) >> l) << l
        d = np.minimum(a, N - 1 - a)
        d = np.minimum(np.minimum(d[:, None, None], d[None, :, None]), d[None, None, :])
        out.append((d >= bounds[l]) & (d < bounds[l + 1]))
    return out


def refined_omega(case):
    return 1.0 / (3.0 * (0.04 * (case["edge"] // 4) / 100.0) + 0.5)


def refined_speed(seed):
    return 0.03 + 0.02 * float(np.random.default_rng(seed).random())


def collide_kbc(f, omega):
    """KBC with the shear / trace split on D3Q27 and entropic gamma."""
    beta = 0.5 * omega
    rho, u = moments(f, C27)
    eq = equilibrium(rho, u, C27, W27)
    neq = f - eq
    pi = {(a, b): sum(c[a] * c[b] * neq[q] for q, c in enumerate(C27) if c[a] * c[b]) for a in range(3)
          for b in range(a, 3)}
    nxz, nyz = pi[0, 0] - pi[2, 2], pi[1, 1] - pi[2, 2]
    face = [(2.0 * nxz - nyz) / 6.0, (2.0 * nyz - nxz) / 6.0, (-nxz - nyz) / 6.0]
    ds = torch.zeros_like(f)
    for q, c in enumerate(C27):
        axes = [a for a in range(3) if c[a]]
        if len(axes) == 1:
            ds[q] = rho * face[axes[0]]
        elif len(axes) == 2:
            ds[q] = rho * pi[axes[0], axes[1]] * (c[axes[0]] * c[axes[1]] / 4.0)
    dh = neq - ds
    gamma = 1.0 / beta - (2.0 - 1.0 / beta) * (ds * dh / eq).sum(0) / (1e-7 + (dh * dh / eq).sum(0))
    return f - beta * (2.0 * ds + gamma * dh)


def collide_bgk(f, omega):
    return f + omega * (equilibrium(*moments(f, C19), C19, W19) - f)


class RefinedExact:
    """Three-level refined cavity on dense level arrays [q, z, y, x]."""

    def __init__(self, case, ulb):
        self.C, W = (C27, W27) if case["lattice"] == "kbc27" else (C19, W19)
        self.collision = collide_kbc if case["lattice"] == "kbc27" else collide_bgk
        self.opp, self.D = opposite(self.C), 3
        lam = shells(case)
        act = [np.zeros(a.shape, bool) for a in lam]
        for l in range(3):      # whole 2^3 groups, an active group activates its parent
            on = act[l] | lam[l]
            s = on.shape
            g = on.reshape(s[0] // 2, 2, s[1] // 2, 2, s[2] // 2, 2).any((1, 3, 5))
            act[l] = np.repeat(np.repeat(np.repeat(g, 2, 0), 2, 1), 2, 2)
            if l < 2:
                act[l + 1] |= g
        for l in (2, 1):        # a refined voxel stays only beside an unrefined one
            ref = self.children(act[l - 1])
            pad = np.pad(ref, 1, constant_values=True)
            near = np.zeros(ref.shape, bool)
            for k in np.ndindex(3, 3, 3):
                near |= ~pad[k[0]:k[0] + ref.shape[0], k[1]:k[1] + ref.shape[1], k[2]:k[2] + ref.shape[2]]
            act[l] &= ~(ref & ~near)
        N = case["edge"]
        self.act = [torch.from_numpy(a).cuda() for a in act]
        self.ref = [torch.from_numpy(a & (self.children(act[l - 1]) if l else False)).cuda() for l, a in enumerate(act)]
        self.leaf = [a & ~r for a, r in zip(self.act, self.ref)]
        i = torch.arange(N, device="cuda")
        edge = (i == 0) | (i == N - 1)
        wall = (edge[:, None, None] | edge[None, :, None] | edge[None, None, :]) & self.leaf[0]
        lid = wall & (i == N - 1)[None, :, None]
        self.bulk = [self.leaf[0] & ~wall, self.leaf[1], self.leaf[2]]
        self.fin = []
        for l in range(3):
            f = torch.zeros((len(self.C),) + tuple(self.act[l].shape), device="cuda", dtype=torch.float64)
            for q, c in enumerate(self.C):
                f[q][self.bulk[l]] = W[q]
                if l == 0:
                    f[q][lid] = -6.0 * W[q] * c[0] * ulb
            self.fin.append(f)
        self.fout = [f.clone() for f in self.fin]
        self.wall0 = wall
        self.links()

    @staticmethod
    def children(fine):
        s = fine.shape
        return fine.reshape(s[0] // 2, 2, s[1] // 2, 2, s[2] // 2, 2).any((1, 3, 5))

    def inside(self, p, l):
        s = self.act[l].shape[0]
        return ((p >= 0) & (p < s)).all(1)

    def active(self, p, l):
        ok = self.inside(p, l)
        p = p.clamp(0, self.act[l].shape[0] - 1)
        return ok & self.act[l][p[:, 2], p[:, 1], p[:, 0]]

    def flat(self, p, l):
        s = self.act[l].shape[0]
        return (p[:, 2] * s + p[:, 1]) * s + p[:, 0]

    def has_parent(self, p, l):
        """The 8^3 block of the next level that holds the parent exists."""
        if l == 2:
            return torch.zeros(p.shape[0], dtype=torch.bool, device="cuda")
        a = self.act[l + 1]
        n = a.shape[0]
        nb = (n + 7) // 8
        pad = torch.zeros((8 * nb,) * 3, dtype=torch.bool, device="cuda")
        pad[:n, :n, :n] = a
        blocks = pad.view(nb, 8, nb, 8, nb, 8).any(5).any(3).any(1)
        b = p >> 4
        return blocks[b[:, 2], b[:, 1], b[:, 0]]

    def links(self):
        """Index lists per level and population: (kind, voxel, source)."""
        vox = [torch.nonzero(b)[:, [2, 1, 0]] for b in self.bulk]
        self.link, self.send = [], []
        for l in range(3):
            p, per_q = vox[l], []
            parent = self.has_parent(p, l)
            for c in self.C:
                d = torch.tensor(c, device="cuda")
                n = p - d
                on = self.active(n, l)
                m = self.flat(n.clamp(0, self.act[l].shape[0] - 1), l)
                refined = on & self.ref[l].reshape(-1)[m]
                wall = on & (self.wall0.reshape(-1)[m] if l == 0 else False)
                lists = {"plain": on & ~refined & ~wall, "wall": wall, "coal": refined}
                per = {k: (self.flat(p[s], l), m[s]) for k, s in lists.items()}
                if l < 2:
                    s = ~on & parent
                    s = s & self.active(torch.div(n, 2, rounding_mode="floor"), l + 1)
                    per["expl"] = (self.flat(p[s], l), self.flat(torch.div(n[s], 2, rounding_mode="floor"), l + 1))
                per_q.append(per)
            self.link.append(per_q)
        self.weight = [None]
        for l in range(2):
            p = torch.nonzero(self.act[l])[:, [2, 1, 0]]
            p = p[self.has_parent(p, l)]
            leaf = self.leaf[l].reshape(-1)[self.flat(p, l)]
            count = torch.zeros_like(self.fin[l + 1]).view(len(self.C), -1)
            per_q = []
            for q, c in enumerate(self.C):
                d = torch.tensor(c, device="cuda")
                s = (p & 1) + d
                un = torch.where(s <= 0, s, s - 1)     # from the parent of x to the parent of x + c
                keep = ~self.active(p + un, l) & self.active((p >> 1) + un, l + 1) & bool(any(c))
                back = un - d
                keep &= self.active((p >> 1) + back, l + 1)
                t = self.flat(((p >> 1) + back)[keep], l + 1)
                count[q].index_add_(0, t, torch.ones(t.numel(), device="cuda", dtype=torch.float64))
                give = leaf[keep] & self.active((p + back)[keep], l)
                per_q.append((t[give], self.flat(p[keep], l)[give]))
            self.send.append(per_q)
            w = torch.where(count > 0, 1.0 / (2.0 * count.clamp(min=1.0)), count)
            self.weight.append(w.float().double())

    def omega(self, l, w0):
        k = 2 - l
        return 2.0 * w0 / (2.0 ** (k + 1) + (1.0 - 2.0 ** k) * w0)

    def collide(self, l, w0):
        new = self.collision(torch.where(self.bulk[l], self.fin[l], 1.0), self.omega(l, w0))
        self.fout[l] = torch.where(self.bulk[l], new, torch.where(self.ref[l], 0.0, self.fout[l]))

    def store(self, l):
        for q, (t, s) in enumerate(self.send[l]):
            self.fout[l + 1].view(len(self.C), -1)[q].index_add_(0, t, self.fout[l].view(len(self.C), -1)[q][s])

    def stream(self, l):
        out, new = self.fout[l].view(len(self.C), -1), self.fin[l].view(len(self.C), -1)
        for q, per in enumerate(self.link[l]):
            v, m = per["plain"]
            new[q][v] = out[q][m]
            v, m = per["wall"]
            new[q][v] = out[self.opp[q]][v] + out[self.opp[q]][m]
            v, m = per["coal"]
            if l:
                new[q][v] = out[q][m] * self.weight[l][q][m]
            if "expl" in per:
                v, m = per["expl"]
                new[q][v] = self.fout[l + 1].view(len(self.C), -1)[q][m]

    def step(self, w0, l=2):
        for _ in range(1 if l == 2 else 2):
            self.collide(l, w0)
            if l < 2:
                self.store(l)
            if l:
                self.step(w0, l - 1)
            self.stream(l)


# ---- the network ------------------------------------------------------------------


def widths_of(case):
    return [int(w) for w in case["widths"].split(",")]


def net_convs(case):
    """(cin, cout, ksize, level) of every convolution in parameter order."""
    w = widths_of(case)
    L, out = len(w), []
    for l in range(L):
        out += [(16 if l == 0 else w[l - 1], w[l], 3, l), (w[l], w[l], 3, l)]
    for l in range(L - 1):
        out += [(w[l + 1] + w[l], w[l], 3, l), (w[l], w[l], 3, l)]
    return out + [(w[0], 16, 1, 0)]


def net_params(case, seed):
    """He-normal weights (W[co][tap][ci], then the biases) with zeros in the
    padded channels of the first and last layer."""
    rng, out, convs = np.random.default_rng(seed), [], net_convs(case)
    for k, (ci, co, ks, _) in enumerate(convs):
        real_i, real_o = (3 if k == 0 else ci), (4 if k == len(convs) - 1 else co)
        w = rng.standard_normal((co, ks ** 3, ci), np.float32) * np.float32(math.sqrt(2.0 / (ks ** 3 * real_i)))
        w[real_o:], w[:, :, real_i:] = 0.0, 0.0
        b = 0.05 * rng.standard_normal(co, np.float32)
        b[real_o:] = 0.0
        out += [w.reshape(-1), b.astype(np.float32)]
    return np.concatenate(out)


def net_inputs(case, seed):
    """Features [n, S^3, 3] (solid, lid, Re / 1000), smooth targets [n, S^3, 4]
    and loss weights [n, S^3] (bulk cells)."""
    S, n = case["size"], case["batch"]
    x, t, w = [], [], []
    for k in range(n):
        cls = torch.from_numpy(cavity((S, S, S), k % 5 if S >= 16 else 0, case["geometry"] + 1000 * seed + k)).cuda()
        f = torch.stack([(cls == NX_CELL_BOUNCEBACK).float(), (cls == NX_CELL_MOVINGWALL).float(),
                         torch.full(cls.shape, 0.05 + 0.9 * ((37 * seed + 11 * k) % 100) / 100, device="cuda")], -1)
        rho, u = smooth_flow((S, S, S), 7919 * seed + k, 1.0)
        bulk = (cls == NX_CELL_BULK)
        y = torch.stack([rho - 1.0] + u, -1).float() * bulk[..., None]
        x.append(f)
        t.append(y)
        w.append(bulk.float() / (4.0 * bulk.sum()))
    return torch.stack(x).view(n, -1, 3), torch.stack(t).view(n, -1, 4), torch.stack(w).view(n, -1)


class Conv64(torch.autograd.Function):
    """Same-size 3D convolution of [n, z, y, x, c] by shifted matrix products."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return Conv64.shifted(x, w)

    @staticmethod
    def offsets(T):
        r = 1 if T == 27 else 0
        return [(z, y, x) for z in range(-r, r + 1) for y in range(-r, r + 1) for x in range(-r, r + 1)]

    @staticmethod
    def window(x, o):
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        n = x.shape
        return p[:, 1 + o[0]:1 + o[0] + n[1], 1 + o[1]:1 + o[1] + n[2], 1 + o[2]:1 + o[2] + n[3]].reshape(-1, n[4])

    @staticmethod
    def shifted(x, w):
        y = 0.0
        for t, o in enumerate(Conv64.offsets(w.shape[1])):
            y = y + Conv64.window(x, o) @ w[:, t].t().contiguous()
        return y.view(tuple(x.shape[:4]) + (w.shape[0],))

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        dx = Conv64.shifted(g, w.flip(1).permute(2, 1, 0).contiguous()) if ctx.needs_input_grad[0] else None
        flat = g.reshape(-1, g.shape[-1]).t().contiguous()
        dw = torch.stack([flat @ Conv64.window(x, o) for o in Conv64.offsets(w.shape[1])], 1)
        return dx, dw


def net_forward64(case, params, x):
    """The U-Net on [n, S^3, 3] in binary64; params the flat vector."""
    w, S = widths_of(case), case["size"]
    L, parts, at = len(w), [], 0
    for ci, co, ks, _ in net_convs(case):
        n = co * ks ** 3 * ci
        parts.append((params[at:at + n].view(co, ks ** 3, ci), params[at + n:at + n + co]))
        at += n + co

    def conv(k, v, relu=True):
        y = Conv64.apply(v, parts[k][0]) + parts[k][1]
        return torch.relu(y) if relu else y

    def pooled(v):
        n, z, y, c = v.shape[0], v.shape[1] // 2, v.shape[2] // 2, v.shape[4]
        return v.view(n, z, 2, y, 2, v.shape[3] // 2, 2, c).mean((2, 4, 6))

    def up(v):
        return v.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    v = torch.nn.functional.pad(x.view(-1, S, S, S, x.shape[-1]), (0, 16 - x.shape[-1]))
    e = []
    for l in range(L):
        e.append(conv(2 * l + 1, conv(2 * l, v)))
        v = pooled(e[l]) if l < L - 1 else e[l]
    for l in range(L - 2, -1, -1):
        v = conv(2 * L + 2 * l + 1, conv(2 * L + 2 * l, torch.cat([up(v), e[l]], -1)))
    return conv(len(parts) - 1, v, relu=False)[..., :4].reshape(x.shape[0], -1, 4)


# ---- the cases ----------------------------------------------------------------------


def listed():
    return [
        # smallest calls: a few steps of a small cavity between a program's own looks at it
        dict(name="cavity32_f32", family="dense", X=32, Y=32, Z=32, storage="f32", boxes=0, geometry=1, steps=8, check=False),
        # the validation run's grid and type (64^3 binary64), one replayed stretch of steps
        dict(name="cavity64_f64", family="dense", X=64, Y=64, Z=64, storage="f64", boxes=0, geometry=1, steps=64, check=False),
        # the headline grid in the default type and in 16-bit deviation storage
        dict(name="cavity256_f32", family="dense", X=256, Y=256, Z=256, storage="f32", boxes=0, geometry=1, steps=10, check=False),
        dict(name="cavity256_f16dev", family="dense", X=256, Y=256, Z=256, storage="f16dev", boxes=0, geometry=1, steps=10, check=False),
        # an odd-sized box with obstacles, stepped to the next look at its residual
        dict(name="obstacles_f32dev", family="dense", X=175, Y=131, Z=97, storage="f32dev", boxes=4, geometry=3, steps=50, check=True),
        # the pressure-driven duct
        dict(name="duct512_f32", family="duct", X=512, Y=128, Z=128, storage="f32", steps=10),
        # sphere pack on sparse blocks, 16-bit storage
        dict(name="porous320_f16dev", family="porous", X=320, Y=320, Z=320, storage="f16dev", spheres=1157, geometry=5, steps=8),
        # a sweep of uneven cavities iterated with the convergence check
        dict(name="batch96_f32", family="batch", members=96, emin=32, emax=96, storage="f32", geometry=7, steps=20),
        # refined lid-driven cavity, the refinement's default collision, stepped and read back
        dict(name="refined128_kbc_f32", family="refined", edge=128, lattice="kbc27", storage="f32", steps=200),
        # training the warm-start network at its configured size
        dict(name="train64_b8", family="train", size=64, batch=8, widths="16,32,64,64", geometry=11, steps=2),
        # prediction with the wide three-level network
        dict(name="predict32_b16", family="predict", size=32, batch=16, widths="64,128,128", geometry=13),
        # the widest-input full-resolution layer of the network, forward and backward
        dict(name="conv64_48to16", family="conv", n=8, size=64, cin=48, cout=16, ksize=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    family = rng.choice(["dense", "dense", "dense", "duct", "porous", "porous", "batch", "batch", "refined", "train",
                         "predict", "conv", "conv"])
    g = rng.randrange(1 << 20)
    if family == "dense":
        X, Y, Z = (_log(rng, 24, 256) for _ in range(3))
        steps = max(4, min(64, int(rng.uniform(0.2, 1.0) * 1.5e8 / (X * Y * Z))))
        return dict(family=family, X=X, Y=Y, Z=Z, storage=rng.choice(["f64", "f32", "f32dev", "f16dev"]),
                    boxes=rng.randrange(5), geometry=g, steps=steps, check=rng.random() < 0.4)
    if family == "duct":
        return dict(family=family, X=_log(rng, 64, 512), Y=_log(rng, 24, 128), Z=_log(rng, 24, 128),
                    storage=rng.choice(["f32", "f64"]), steps=rng.randrange(4, 11))
    if family == "porous":
        X, Y, Z = 8 * _log(rng, 8, 40), _log(rng, 64, 320), _log(rng, 64, 320)
        return dict(family=family, X=X, Y=Y, Z=Z, storage=rng.choice(["f64", "f32", "f32dev", "f16dev"]),
                    spheres=max(4, int(X * Y * Z * 3.5e-5)), geometry=g, steps=rng.randrange(4, 9))
    if family == "batch":
        return dict(family=family, members=_log(rng, 4, 96), emin=32, emax=rng.choice([48, 64, 96]),
                    storage=rng.choice(["f32", "f32dev", "f16dev"]), geometry=g, steps=4 * rng.randrange(2, 6))
    if family == "refined":
        return dict(family=family, edge=16 * rng.randrange(4, 9), lattice=rng.choice(["kbc27", "bgk19"]),
                    storage=rng.choice(["f32", "f64"]), steps=rng.randrange(20, 101))
    if family in ("train", "predict"):
        size = rng.choice([16, 32, 64])
        d = dict(family=family, size=size, batch=rng.randrange(1, 9),
                 widths=rng.choice(["16,32,64,64", "32,64,64", "16,48", "64,128,128"] if size < 64 else ["16,32,64,64", "16,32"]),
                 geometry=g)
        return dict(d, steps=2) if family == "train" else d
    size = rng.choice([8, 16, 32, 64])
    cap = 128 if size < 64 else 48
    return dict(family=family, n=rng.randrange(1, 9), size=size, cin=16 * rng.randrange(1, cap // 16 + 1),
                cout=16 * rng.randrange(1, (cap if size < 64 else 32) // 16 + 1), ksize=rng.choice([3, 3, 3, 1]))


# ---- prepare ---------------------------------------------------------------------------


def _lattice_state(lat, start, steps, **more):
    """Both population buffers hold the start; the views are the outputs."""
    dtype = start.dtype
    views = [span(b, b.ptr, start.numel(), dtype) for b in lat.pop]
    for v in views:
        v.copy_(start.reshape(-1))
    torch.cuda.synchronize()
    return dict(lat=lat, views=views, steps=steps, stream=stream(), **more)


def _prepare_dense(case, seed):
    dim = (case["X"], case["Y"], case["Z"])
    cls = cavity(dim, case["boxes"], case["geometry"])
    start, _ = flow_start(cls, seed, case["storage"], ULB, ULB)
    lat = nx.DenseLattice(dim, case["storage"])
    lat.set_classes(cls.astype(np.uint32), ULB)
    u_prev = None
    if case["check"]:
        u_prev = buffer_of(torch.zeros(3 * cls.size, device="cuda"))
    return _lattice_state(lat, start, case["steps"], omega=cavity_omega(dim), u_prev=u_prev)


def duct_classes(case):
    cls = np.full((case["Z"], case["Y"], case["X"]), NX_CELL_BULK, np.uint8)
    cls[:, [0, -1]] = cls[[0, -1]] = NX_CELL_BOUNCEBACK
    return cls


DUCT_VALUES = (1.0005, 0.9995, 0.0, 0.0, 0.0, 0.0)
OMEGA_002 = 1.0 / (3.0 * 0.02 + 0.5)     # nu = 0.02
FORCE = (1e-6, 0.0, 0.0)


def _prepare_duct(case, seed):
    cls = duct_classes(case)
    zh = np.zeros(cls.shape, np.uint32)
    zh[:, :, 0], zh[:, :, -1] = NX_ZH_XMIN, NX_ZH_XMAX
    zh[cls != NX_CELL_BULK] = 0
    start, _ = flow_start(cls, seed, case["storage"], 0.01)
    lat = nx.DenseLattice((case["X"], case["Y"], case["Z"]), case["storage"])
    lat.set_classes(cls.astype(np.uint32), zouhe=zh)
    return _lattice_state(lat, start, case["steps"])


def to_blocks(dense, mask):
    """[k, z, y, x] to the 8^3-block order [block, k, voxel] of the blocks that
    hold a set voxel of the mask; unset voxels 0."""
    Z, Y, X = mask.shape
    b = [(n + 7) // 8 for n in (Z, Y, X)]
    pad = (0, 8 * b[2] - X, 0, 8 * b[1] - Y, 0, 8 * b[0] - Z)
    cut = lambda a: torch.nn.functional.pad(a, pad).view(-1, b[0], 8, b[1], 8, b[2], 8)  # noqa: E731
    on = cut(mask.to(torch.uint8)[None]).amax((0, 2, 4, 6)).reshape(-1) > 0
    v = cut(torch.where(mask, dense, torch.zeros((), dtype=dense.dtype, device=dense.device)))
    return v.permute(1, 3, 5, 0, 2, 4, 6).reshape(-1, dense.shape[0], 512)[on]


def porous_classes(case):
    solid = sphere_pack((case["X"], case["Y"], case["Z"]), case["spheres"], case["geometry"])
    return ~solid


def _prepare_porous(case, seed):
    dim = (case["X"], case["Y"], case["Z"])
    fluid = porous_classes(case)
    cls = torch.where(fluid, NX_CELL_BULK, NX_CELL_BOUNCEBACK).to(torch.uint8).cpu().numpy()
    grid = nx.BlockGrid(dim, fluid.to(torch.uint8).cpu().numpy(), periodic=1)
    lat = nx.BlockLattice(grid, case["storage"])
    on = np.unpackbits(grid.masks.view(np.uint8), bitorder="little").astype(bool)
    lat.set_classes(np.where(on, NX_CELL_BULK, NX_CELL_UNDEFINED).astype(np.uint32))
    start, bulk = flow_start(cls, seed, case["storage"], 0.002)
    return _lattice_state(lat, to_blocks(start, fluid), case["steps"])


def batch_members(case):
    rng = np.random.default_rng(case["geometry"])
    edges = np.arange(case["emin"], case["emax"] + 1, 8)
    out = []
    for k in range(case["members"]):
        e = int(rng.choice(edges))
        nu = ULB * e / float(rng.uniform(50.0, 4.0 * e))
        cls = cavity((e, e, e), int(rng.integers(0, 5)), int(rng.integers(0, 1 << 30)))
        out.append({"dim": (e, e, e), "classes": cls, "omega": 1.0 / (3.0 * nu + 0.5), "ulb": ULB})
    return out


def batch_flow(members, seed):
    flows = [smooth_flow(m["dim"], seed + 31 * k, ULB) for k, m in enumerate(members)]
    return [(r.float(), [v.float() for v in u]) for r, u in flows]


def _prepare_batch(case, seed):
    members = batch_members(case)
    flows = batch_flow(members, seed)
    b = nx.CavityBatch(members, case["storage"])
    rho, _ = buffer_of(torch.cat([r.reshape(-1) for r, _ in flows]))
    u, _ = buffer_of(torch.cat([v.reshape(-1) for _, us in flows for v in us]))
    torch.cuda.synchronize()
    b.init(rho, u)
    return dict(batch=b, steps=case["steps"], view=span(b, b.member(0)[1], 19 * b.n_cells, DTYPE[case["storage"]]))


def _prepare_refined(case, seed):
    N = case["edge"]
    g = mgrid.MGrid((N, N, N), [a.astype(np.uint8) for a in shells(case)], case["storage"], lattice=case["lattice"])
    g.setup_cavity(refined_speed(seed))
    return dict(grid=g, steps=case["steps"], omega=refined_omega(case), stream=stream())


def _prepare_net(case, seed):
    w = widths_of(case)
    net = surrogate.UNet(case["size"], len(w), w, case["batch"], seed=1)
    net.set_params(net_params(case, seed))
    x, t, wt = net_inputs(case, seed)
    y, out = buffer_of(torch.zeros_like(t))
    return dict(net=net, x=buffer_of(x)[0], t=buffer_of(t)[0], w=buffer_of(wt)[0], y=y, out=out,
                batch=case["batch"], steps=case.get("steps", 0))


def conv_inputs(case, seed):
    gen, S, T = generator(seed), case["size"], case["ksize"] ** 3
    V = case["n"] * S ** 3
    x = torch.relu(torch.randn((V, case["cin"]), generator=gen, device="cuda")).bfloat16()
    w = (torch.randn((case["cout"], T, case["cin"]), generator=gen, device="cuda") * math.sqrt(2.0 / (T * case["cin"]))).bfloat16()
    b = 0.05 * torch.randn(case["cout"], generator=gen, device="cuda")
    dy = (torch.randn((V, case["cout"]), generator=gen, device="cuda") * 1e-3).bfloat16()
    return x, w, b, dy


def _prepare_conv(case, seed):
    x, w, b, dy = conv_inputs(case, seed)
    s = {k: buffer_of(v) for k, v in dict(x=x, w=w, b=b, dy=dy, y=torch.zeros_like(dy), dx=torch.zeros_like(x),
                                          dw=torch.zeros(w.shape, device="cuda"), db=torch.zeros_like(b)).items()}
    torch.cuda.synchronize()
    S = case["size"]
    return dict(s, shape=(case["n"], S, S, S), cin=case["cin"], cout=case["cout"], ksize=case["ksize"])


def prepare(case, seed):
    nx.init()
    fam = case["family"]
    state = {"dense": _prepare_dense, "duct": _prepare_duct, "porous": _prepare_porous, "batch": _prepare_batch,
             "refined": _prepare_refined, "train": _prepare_net, "predict": _prepare_net, "conv": _prepare_conv}[fam](case, seed)
    state["family"] = fam
    return state


# ---- run -------------------------------------------------------------------------------


def run(s):
    fam = s["family"]
    if fam == "dense":
        lat = s["lat"]
        lat.run(s["steps"], s["omega"], stream=s["stream"])
        if s["u_prev"] is None:
            return s["views"][lat.parity]
        return {"f": s["views"][lat.parity], "residual": lat.residual(s["u_prev"][0], s["stream"]), "u": s["u_prev"][1]}
    if fam == "duct":
        s["lat"].run_zouhe(s["steps"], OMEGA_002, DUCT_VALUES, stream=s["stream"])
        return s["views"][s["lat"].parity]
    if fam == "porous":
        s["lat"].run(s["steps"], OMEGA_002, force=FORCE, stream=s["stream"])
        return s["views"][s["lat"].parity]
    if fam == "batch":
        steps, residual, left = s["batch"].run(s["steps"], s["steps"] // 2, 1e-12)
        return {"f": s["view"], "steps": steps, "residual": residual, "left": left}
    if fam == "refined":
        s["grid"].run(s["steps"], s["omega"], stream=s["stream"])
        return [s["grid"].fields(l) for l in range(s["grid"].depth)]
    net = s.get("net")
    if fam == "train":
        for k in range(s["steps"]):
            loss = net.train_step(s["x"], s["t"], s["w"], s["batch"], 5e-4, want_loss=k == s["steps"] - 1)
        return {"loss": loss, "grads": net.grads(), "params": net.params()}
    if fam == "predict":
        net.forward(s["x"], s["batch"], s["y"])
        return s["out"]
    at = (s["shape"], s["cin"], s["cout"], s["ksize"])
    surrogate.conv3d_fwd(s["x"][0], s["w"][0], s["b"][0], s["y"][0], *at, relu=True)
    surrogate.conv3d_bwd_data(s["dy"][0], s["w"][0], s["dx"][0], *at)
    surrogate.conv3d_bwd_weight(s["x"][0], s["dy"][0], s["dw"][0], s["db"][0], *at)
    return {k: s[k][1] for k in ("y", "dx", "dw", "db")}


# ---- work and tolerance ------------------------------------------------------------------


def conv_flops(voxels, cin, cout, ks):
    return 2.0 * voxels * cin * cout * ks ** 3


def work(case):
    """Each population read and written once per fluid cell and step; each
    layer's multiply-adds over its real channels, its tensors once each way."""
    fam, b = case["family"], BYTES.get(case.get("storage"), 0)
    if fam == "dense":
        cls = cavity((case["X"], case["Y"], case["Z"]), case["boxes"], case["geometry"])
        n = float((cls == NX_CELL_BULK).sum())
        return {"bytes": n * (case["steps"] * 38 * b + (19 * b + 24 if case["check"] else 0)), "flops": n * case["steps"] * 250}
    if fam == "duct":
        n = float((case["Y"] - 2) * (case["Z"] - 2) * case["X"])
        return {"bytes": n * case["steps"] * 38 * b, "flops": n * case["steps"] * 250}
    if fam == "porous":
        n = float(porous_classes(case).sum())
        return {"bytes": n * case["steps"] * 38 * b, "flops": n * case["steps"] * 350}
    if fam == "batch":
        n = float(sum((m["classes"] == NX_CELL_BULK).sum() for m in batch_members(case)))
        return {"bytes": n * (case["steps"] * 38 * b + 2 * (19 * b + 24)), "flops": n * case["steps"] * 250}
    if fam == "refined":
        q = 27 if case["lattice"] == "kbc27" else 19
        lam = shells(case)
        updates = float(sum(int(a.sum()) * (4 >> l) for l, a in enumerate(lam)))
        values = float(sum(a.size for a in lam))
        return {"bytes": updates * case["steps"] * 2 * q * b + values * q * b,
                "flops": updates * case["steps"] * (1200 if q == 27 else 250)}
    if fam in ("train", "predict"):
        S, n, bts, fl = case["size"], case["batch"], 0.0, 0.0
        convs = net_convs(case)
        for k, (ci, co, ks, l) in enumerate(convs):
            v = n * (S >> l) ** 3
            ri, ro = (3 if k == 0 else ci), (4 if k == len(convs) - 1 else co)
            once = conv_flops(v, ri, ro, ks)
            if fam == "predict":
                fl += once
                bts += 2.0 * v * (ci + co)
            else:
                fl += (3 if k else 2) * once
                bts += 2.0 * v * 3 * (ci + co)
        return {"bytes": bts * case.get("steps", 1), "flops": fl * case.get("steps", 1)}
    v = float(case["n"] * case["size"] ** 3)
    w = case["cin"] * case["cout"] * case["ksize"] ** 3
    return {"bytes": 2.0 * v * 3 * (case["cin"] + case["cout"]) + 8.0 * w,
            "flops": 3.0 * conv_flops(v, case["cin"], case["cout"], case["ksize"])}


def tolerance(case):
    """Four times the distance from binary64 that was measured over these
    ranges; velocities of raw binary32 populations carry the rounding of w,
    and the velocity kept for the residual is binary32 for every storage."""
    fam, st = case["family"], case.get("storage")
    if fam in ("dense", "duct", "porous", "batch"):
        if case.get("check"):
            return {"f64": {"rel": 1e-7}, "f32": {"rel": 5e-5}, "f32dev": {"rel": 5e-6}, "f16dev": {"rel": 1e-2}}[st]
        return {"f64": {"rel": 1e-14}, "f32": {"rel": 3e-6}, "f32dev": {"rel": 5e-6}, "f16dev": {"rel": 4e-3}}[st]
    if fam == "refined":
        return {"rel": 1e-12 if st == "f64" else 6e-6}
    if fam == "conv":
        return {"rel": 7e-3, "max": 0.05}
    return {"rel": 0.03, "max": 0.99}


# ---- exact --------------------------------------------------------------------------------


def _exact_dense(case, seed):
    dim, st = (case["X"], case["Y"], case["Z"]), case["storage"]
    cls = cavity(dim, case["boxes"], case["geometry"])
    start, bulk = flow_start(cls, seed, st, ULB, ULB)
    f = decoded(start, bulk, st)
    for _ in range(case["steps"]):
        f = step19(f, bulk, cavity_omega(dim))
    if not case["check"]:
        return encoded(f, bulk, st)
    _, u = moments(pull(f, bulk, C19), C19)
    u = torch.stack([torch.where(bulk, v, 0.0) for v in u])
    total = float(u.square().sum())
    return {"f": encoded(f, bulk, st), "residual": (total, total), "u": u.reshape(-1)}


def _exact_duct(case, seed):
    cls = duct_classes(case)
    start, bulk = flow_start(cls, seed, case["storage"], 0.01)
    pad = torch.nn.functional.pad
    f, on = pad(start.double(), (1, 1)), pad(bulk, (1, 1))
    for _ in range(case["steps"]):
        f = step19(f, on, OMEGA_002, ends=((1, DUCT_VALUES[0], 1), (case["X"], DUCT_VALUES[1], -1)))
    return f[..., 1:-1].reshape(-1)


def _exact_porous(case, seed):
    st, fluid = case["storage"], porous_classes(case)
    cls = torch.where(fluid, NX_CELL_BULK, NX_CELL_BOUNCEBACK).to(torch.uint8).cpu().numpy()
    start, bulk = flow_start(cls, seed, st, 0.002)
    pad = torch.nn.functional.pad
    f, on = pad(decoded(start, bulk, st), (0, 0, 1, 1, 1, 1)), pad(bulk, (0, 0, 1, 1, 1, 1))
    for _ in range(case["steps"]):
        f = step19(f, on, OMEGA_002, g=FORCE)
    f = f[:, 1:-1, 1:-1].contiguous()
    return to_blocks(encoded(f, bulk, st).view(f.shape), fluid).reshape(-1)


def _exact_batch(case, seed):
    st, members = case["storage"], batch_members(case)
    out, residual, half = [], [], case["steps"] // 2
    for m, (rho, u) in zip(members, batch_flow(members, seed)):
        cls = m["classes"]
        bulk = torch.from_numpy(cls == NX_CELL_BULK).cuda()
        full = equilibrium(rho.double(), [v.double() for v in u], C19, W19)
        f = decoded(torch.where(bulk, stored(full, bulk, st), wall_values(cls, ULB, st)), bulk, st)
        seen = []
        for k in range(case["steps"]):
            f = step19(f, bulk, m["omega"])
            if (k + 1) % half == 0:
                _, v = moments(pull(f, bulk, C19), C19)
                seen.append(torch.stack([torch.where(bulk, a, 0.0) for a in v]))
        out.append(encoded(f, bulk, st))
        residual.append(math.sqrt(float((seen[-1] - seen[-2]).square().sum() / seen[-1].square().sum())))
    return {"f": torch.cat(out), "steps": None, "residual": np.array(residual), "left": None}


def _exact_refined(case, seed):
    u = refined_speed(seed)
    g = RefinedExact(case, float(np.float32(u)) if case["storage"] == "f32" else u)
    for _ in range(case["steps"]):
        g.step(refined_omega(case))
    return [f.reshape(-1) for f in g.fin]


def _exact_train(case, seed):
    p = torch.from_numpy(net_params(case, seed)).double().cuda()
    x, t, w = (v.double() for v in net_inputs(case, seed))
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for k in range(1, case["steps"] + 1):
        q = p.clone().requires_grad_(True)
        loss = (w[..., None] * (net_forward64(case, q, x) - t) ** 2).sum()
        (g,) = torch.autograd.grad(loss, q)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - 5e-4 * (m / (1 - 0.9 ** k)) / ((v / (1 - 0.999 ** k)).sqrt() + 1e-8)
    return {"loss": float(loss.detach()), "grads": g, "params": p}


def exact(case, seed):
    fam = case["family"]
    if fam == "dense":
        return _exact_dense(case, seed)
    if fam == "duct":
        return _exact_duct(case, seed)
    if fam == "porous":
        return _exact_porous(case, seed)
    if fam == "batch":
        return _exact_batch(case, seed)
    if fam == "refined":
        return _exact_refined(case, seed)
    if fam == "train":
        return _exact_train(case, seed)
    if fam == "predict":
        p = torch.from_numpy(net_params(case, seed)).double().cuda()
        with torch.no_grad():
            return net_forward64(case, p, net_inputs(case, seed)[0].double()).reshape(-1)
    x, w, b, dy = conv_inputs(case, seed)
    S = case["size"]
    x5 = x.double().view(case["n"], S, S, S, -1)
    g5 = dy.double().view(case["n"], S, S, S, -1)
    y = torch.relu(Conv64.shifted(x5, w.double()) + b.double())
    dx = Conv64.shifted(g5, w.double().flip(1).permute(2, 1, 0).contiguous())
    flat = dy.double().t().contiguous()
    dw = torch.stack([flat @ Conv64.window(x5, o) for o in Conv64.offsets(w.shape[1])], 1)
    return {"y": y.reshape(-1), "dx": dx.reshape(-1), "dw": dw.reshape(-1), "db": dy.double().sum(0)}
