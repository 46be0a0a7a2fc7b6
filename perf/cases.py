"""Workloads whose speed matters to users of grid_amd.

Each case is one call (or one short sequence of calls) of the public binding, on synthetic gauge
links near the unit matrix and Gaussian spinors.  The paths:

  apply     the full Dirac operator M or Mdag on a whole lattice (propagator checks, Krylov methods
            on the full system, residuals)
  hop       the even-odd hop DhopEO / DhopOE, the benchmark of the library
  schur     the normal operator MpcDagMpc of the red-black system: one call per Krylov step of a
            solver or eigensolver that a user writes on top of the operator
  solve     a red-black solve of the full system, FP64 or mixed precision
  shifts    the multishift solve of rational HMC
  slices    the slice matrices of block Krylov solvers: two inner-product matrices, one update
  force     the fermion force DhopDeriv of HMC, delivered to host memory
  transfer  a source uploaded and a solution downloaded, host arrays on both sides

A field's values are returned where the library keeps them, on the GPU, as tensors over its memory
(see `views`): a program that goes on computing on the GPU copies nothing to the host either.
"""
import ctypes
import math

import numpy as np
import torch

import grid_amd as gx

PRECS = {'f64': gx.F64, 'f32': gx.F32, 'f16': gx.F16}
SIZE = {'f64': 16, 'f32': 8, 'f16': 4}       # bytes of a complex number
M5, B, C = 1.8, 1.5, 0.5                     # Mobius parameters of the repository's benchmark
EPS = 0.3                                    # spread of the links around the unit matrix


def listed():
    return [
        # latency: the operator on the smallest lattice that is used in earnest
        case('wilson_m_small', 'apply', (8, 8, 8, 8), kind='wilson', Ls=1, prec='f64', mass=0.1),
        # a whole solve where every kernel is short (tuning runs, small-volume ensembles)
        case('wilson_solve_small', 'solve', (8, 8, 8, 8), kind='wilson', Ls=1, prec='f64', mass=0.1, mixed=0),
        # the library's headline: the 5D hop in FP64
        case('mobius_hop_f64', 'hop', (16, 16, 16, 16), kind='mobius', Ls=16, prec='f64', mass=0.01),
        # the 12 spin-colour sources of a propagator in one hop, FP32 (inner solves of defect correction)
        case('wilson_hop_12rhs_f32', 'hop', (32, 32, 32, 64), kind='wilson', Ls=12, prec='f32', mass=0.05, dag=1),
        # the adjoint 5D operator on a production-like lattice
        case('mobius_mdag_f64', 'apply', (24, 24, 24, 24), kind='mobius', Ls=12, prec='f64', mass=0.005, dag=1),
        # the Krylov operator of the FP32 inner solves, on a lattice of unequal extents
        case('mobius_schur_f32', 'schur', (20, 12, 18, 28), kind='mobius', Ls=10, prec='f32', mass=0.01),
        # the same in FP16 storage with many right-hand sides
        case('wilson_schur_12rhs_f16', 'schur', (24, 24, 24, 48), kind='wilson', Ls=12, prec='f16', mass=0.05),
        # the mixed-precision light-quark solve
        case('mobius_solve_mixed', 'solve', (16, 16, 16, 16), kind='mobius', Ls=16, prec='f64', mass=0.01, mixed=1),
        # rational HMC: twelve poles of one light operator
        case('mobius_shifts', 'shifts', (12, 12, 12, 24), kind='mobius', Ls=8, prec='f64', mass=0.05, nshift=12),
        # one orthogonalisation step of a block of twelve
        case('block_slices', 'slices', (16, 16, 16, 32), Ls=12, prec='f64'),
        # molecular dynamics force of a 5D fermion
        case('mobius_force', 'force', (16, 16, 16, 32), kind='mobius', Ls=8, prec='f64', mass=0.05),
        # a 4D source in, a 4D solution out
        case('propagator_transfer', 'transfer', (24, 20, 14, 36), Ls=1, prec='f64'),
    ]


def case(name, path, dims, **kw):
    c = {'name': name, 'path': path, 'lx': dims[0], 'ly': dims[1], 'lz': dims[2], 'lt': dims[3]}
    c.update(kw)
    return c


# ---------------- drawn cases ----------------

SPREAD = {  # path: smallest and largest entries V4 * Ls, and the weight it is drawn with
    'apply': (4096, 4.2e6, 3), 'hop': (4096, 2.6e7, 4), 'schur': (4096, 8.0e6, 4), 'solve': (4096, 5.0e5, 2),
    'shifts': (1.6e4, 3.4e5, 1), 'slices': (2.0e4, 1.6e6, 2), 'force': (8192, 1.1e6, 1),
    'transfer': (4096, 4.0e5, 1),
}


def draw(rng):
    path = rng.choice([p for p, (_, _, n) in SPREAD.items() for _ in range(n)])
    kind = rng.choice(['wilson', 'mobius'])
    lo, hi, _ = SPREAD[path]
    if path == 'transfer':
        Ls = rng.choice([1, 1, 2, 8, 12])
    elif path == 'slices':
        Ls = rng.choice([2, 3, 4, 6, 8, 12, 12, 16])
    elif kind == 'mobius':
        Ls = rng.choice([6, 8, 8, 10, 12, 12, 14, 16, 16, 20, 24])
    elif path in ('force', 'shifts'):
        Ls = 1
    else:
        Ls = rng.choice([1, 1, 1, 2, 3, 4, 5, 6, 8, 12, 12, 16])
    vol = math.exp(rng.uniform(math.log(lo), math.log(hi))) / Ls
    vol = min(max(vol, 8 * 6 * 6 * 6), 32 ** 3 * 64)
    c = {'path': path}
    c.update(zip(('lx', 'ly', 'lz', 'lt'), extents(rng, vol)))
    c['Ls'] = Ls
    c['prec'] = 'f64'
    if path in ('hop', 'schur', 'apply'):
        c['prec'] = rng.choice(['f64', 'f32', 'f32', 'f16'] if path != 'apply' else ['f64', 'f64', 'f32'])
    if path == 'transfer':
        c['prec'] = rng.choice(['f64', 'f32'])
    if path not in ('slices', 'transfer'):
        c['kind'] = kind
        c['mass'] = round(rng.uniform(0.05, 0.2), 4)
    if path in ('hop', 'apply', 'force'):
        c['dag'] = rng.randint(0, 1)
    if path == 'solve':
        c['mixed'] = rng.choice([0, 1, 2] if kind == 'wilson' and Ls > 1 else [0, 1, 2, 3])
    if path == 'shifts':
        c['nshift'] = rng.randint(3, 12)
    return c


def extents(rng, vol):
    """Four even extents, 6 at least, with a product near vol and at most 1.1 of it or the smallest."""
    side = vol ** 0.25
    d = [max(6, 2 * round(side * rng.uniform(0.7, 1.35) / 2)) for _ in range(3)]
    d[0] = max(8, d[0])
    return d + [max(6, 2 * round(vol / (d[0] * d[1] * d[2]) / 2))]


# ---------------- inputs ----------------

_context = None


def context():
    """One context for the process, as a program on one GPU has."""
    global _context
    if _context is None:
        _context = gx.Context(0)
    return _context


def extent(c):
    return c['lx'], c['ly'], c['lz'], c['lt']


def generator(seed, stream):
    g = torch.Generator(device='cuda')
    g.manual_seed((seed * 1000003 + stream) % (1 << 62))
    return g


def links(c, seed):
    """(Lt, Lz, Ly, Lx, 4, 3, 3) complex128 SU(3) matrices, Gaussian around the unit matrix."""
    lx, ly, lz, lt = extent(c)
    x = torch.randn((lt, lz, ly, lx, 4, 2, 3, 2), generator=generator(seed, 1), device='cuda', dtype=torch.float64)
    x = torch.view_as_complex(x) * EPS
    r0, r1 = x[..., 0, :], x[..., 1, :]
    r0[..., 0] += 1
    r1[..., 1] += 1
    r0 /= r0.abs().square().sum(-1, keepdim=True).sqrt()
    r1 -= (r0.conj() * r1).sum(-1, keepdim=True) * r0
    r1 /= r1.abs().square().sum(-1, keepdim=True).sqrt()
    r2 = torch.stack([r0[..., 1] * r1[..., 2] - r0[..., 2] * r1[..., 1],
                      r0[..., 2] * r1[..., 0] - r0[..., 0] * r1[..., 2],
                      r0[..., 0] * r1[..., 1] - r0[..., 1] * r1[..., 0]], -1).conj()
    return torch.stack([r0, r1, r2], -2)


def spinor(c, seed, stream, halves):
    """(halves, H4, Ls, 12) complex128 Gaussian numbers, one set of 4D half-lattice sites per half,
    rounded to the case's precision (FP16 storage rounds further when it stores them)."""
    n = c['lx'] * c['ly'] * c['lz'] * c['lt'] // 2
    x = torch.randn((halves, n, c['Ls'], 12, 2), generator=generator(seed, stream), device='cuda',
                    dtype=torch.float64 if c['prec'] == 'f64' else torch.float32)
    if c['prec'] == 'f16':
        val, scale = stored(torch.view_as_complex(x.double()), 'f16')
        x = torch.view_as_real(unstored(c, val.half().double(), scale.float().double()))
    return torch.view_as_complex(x.double())


def stored(x, prec):
    """(halves, H4, Ls, 12) numbers in the order in which the library keeps them: blocks of 64
    entries (site, s), padded with zeros, and in a block the components in groups of 16 bytes.  FP16
    storage: the values over their entry's largest part, and those."""
    halves, n = x.shape[0], x.shape[1] * x.shape[2]
    x = x.reshape(halves, n, 12)
    pad = -n % 64
    if pad:
        x = torch.cat([x, torch.zeros((halves, pad, 12), device=x.device, dtype=x.dtype)], 1)
    x = torch.view_as_real(x)
    vw = 16 // SIZE[prec]
    scale = None
    if prec == 'f16':
        scale = x.abs().amax((-1, -2))
        x = x / torch.where(scale > 0, scale, 1.0)[..., None, None]
        scale = scale.reshape(halves, -1, 64)
    x = x.reshape(halves, -1, 64, 12 // vw, vw, 2).transpose(2, 3).reshape(halves, -1, 64 * 24)
    return (x, scale) if prec == 'f16' else (x,)


def unstored(c, val, scale):
    """The inverse of `stored` for FP16 values and scales."""
    halves, n = val.shape[0], c['lx'] * c['ly'] * c['lz'] * c['lt'] // 2 * c['Ls']
    x = val.reshape(halves, -1, 3, 64, 4, 2).transpose(2, 3) * scale[:, :, :, None, None, None]
    return torch.view_as_complex(x.reshape(halves, -1, 12, 2)[:, :n].contiguous()).reshape(halves, -1, c['Ls'], 12)


class _Memory:
    def __init__(self, field, at, words):
        self.field = field  # keeps the memory while a tensor looks at it
        self.__cuda_array_interface__ = {'shape': (words,), 'typestr': '<i4', 'data': (at, False), 'version': 2}


def views(field):
    """A field's memory as tensors, one tuple for its halves together: (halves, blocks, values), and
    for FP16 storage the (halves, blocks, 64) scales.  The binding hands out no device address: it
    is the ninth 8-byte word of the object behind a field's handle, its size in bytes the next."""
    at, size = (ctypes.c_uint64 * 2).from_address(field.h.value + 64)
    halves = 2 if field.subset == gx.FULL else 1
    mem = torch.as_tensor(_Memory(field, at, size // 4), device='cuda')
    if field.prec == gx.F16:
        mem = mem.view(halves, -1, 64 * 13)
        return mem[..., :64 * 12].view(torch.float16), mem[..., 64 * 12:].view(torch.float32)
    return (mem.view(halves, -1).view(torch.float64 if field.prec == gx.F64 else torch.float32).view(halves, -1, 64 * 24),)


def filled(field, c, seed, stream):
    context().sync()
    x = spinor(c, seed, stream, 2 if field.subset == gx.FULL else 1)
    for to, v in zip(views(field), stored(x, c['prec'])):
        to.copy_(v)
    torch.cuda.synchronize()
    return field


class State(dict):
    def __del__(self):
        if 'op' in self:
            self['op'].close()


def prepare(c, seed):
    ctx, dims, path, Ls = context(), extent(c), c['path'], c['Ls']
    st = State(case=dict(c))
    prec = PRECS[c['prec']]
    if path == 'transfer':
        shape = dims[::-1] + (Ls, 4, 3)
        st['host'] = torch.view_as_complex(torch.randn(
            shape + (2,), generator=generator(seed, 2), device='cuda', dtype=torch.float64)).cpu().numpy()
        st['f'] = gx.Field(ctx, dims, Ls, prec, gx.FULL)
        return st
    if path == 'slices':
        x, y, r = (gx.Field(ctx, dims, Ls, prec, gx.ODD) for _ in range(3))
        st['x'], st['y'], st['r'] = filled(x, c, seed, 2), filled(y, c, seed, 3), r
        st['a'] = coefficients(c, seed)
        st['out'] = views(r)
        return st
    U = links(c, seed).cpu().numpy()
    op = gx.FermionOp(ctx, U, dims, Ls, c['kind'], mass=c['mass'], M5=M5, b=B, c=C)
    st['op'] = op
    if path in ('apply', 'solve', 'force'):
        st['in'] = filled(op.field(prec), c, seed, 2)
        st['to'] = op.field(prec)
        if path == 'force':
            filled(st['to'], c, seed, 3)
    elif path == 'shifts':
        st['in'] = filled(op.field(prec, gx.ODD), c, seed, 2)
        st['to'] = [op.field(prec, gx.ODD) for _ in range(c['nshift'])]
        st['shifts'] = shifts(c)
    else:
        st['in'] = filled(op.field(prec, gx.ODD), c, seed, 2)
        st['to'] = op.field(prec, gx.EVEN if path == 'hop' else gx.ODD)
    if path != 'force':
        st['out'] = [views(f) for f in (st['to'] if path == 'shifts' else [st['to']])]
    ctx.sync()
    return st


def coefficients(c, seed):
    a = np.random.default_rng(seed).standard_normal((c['Ls'], c['Ls'], 2)) / c['Ls']
    return np.ascontiguousarray(a[..., 0] + 1j * a[..., 1])


def shifts(c):
    """Poles of a rational approximation: spread evenly over the logarithm from 1e-4 to 3."""
    n = c['nshift']
    return [1e-4 * (3e4 ** (k / (n - 1))) for k in range(n)]


def tolerance(c):
    """The normal equations' tolerance at which the full system's residual is below 1e-10."""
    return 1e-11 if c['kind'] == 'wilson' else 1e-12


def run(st):
    c = st['case']
    path = c['path']
    if path == 'transfer':
        return st['f'].upload(st['host']).download()
    if path == 'slices':
        m = gx.slice_inner_product_matrix(st['x'], st['y'])
        g = gx.slice_inner_product_matrix(st['x'], st['x'])
        gx.slice_madd_matrix(st['r'], st['a'], st['x'], st['y'], -1.0)
        return m, g, st['out']
    op = st['op']
    if path == 'apply':
        (op.Mdag if c.get('dag') else op.M)(st['in'], st['to'])
    elif path == 'hop':
        op.DhopEO(st['in'], st['to'], c.get('dag', 0))
    elif path == 'schur':
        op.MpcDagMpc(st['in'], st['to'])
    elif path == 'solve':
        st['to'].zero()
        op.schur_solve(st['in'], st['to'], tol=tolerance(c), mixed=c['mixed'])
    elif path == 'shifts':
        op.cg_multishift(st['in'], st['to'], st['shifts'], [1e-11] * c['nshift'])
    else:
        return op.DhopDeriv(st['in'], st['to'], c.get('dag', 0))
    return st['out']


# ---------------- what a pass cannot do without ----------------

def iterations(c):
    """Krylov steps of a solve: of the order that the mass and the precision make necessary."""
    if c['path'] == 'shifts' or c['kind'] == 'mobius':
        return round(40 / max(c['mass'], 0.1) if c['mass'] >= 0.05 else 460)
    return round(65 * (0.05 / c['mass']) ** 0.4)


def work(c):
    lx, ly, lz, lt = extent(c)
    H, Ls, z = lx * ly * lz * lt // 2, c['Ls'], SIZE[c['prec']]
    path = c['path']
    field, link = H * Ls * 12 * z, H * 72 * z          # a half field; the links of one checkerboard
    if c['prec'] == 'f16':
        field += H * Ls * 4
    hop = H * Ls * 1320
    fifth = 0 if c.get('kind') != 'mobius' else H * Ls * 12 * 8 * 2   # a bidiagonal matrix per half field
    if path == 'transfer':
        return {'bytes': 2 * 2 * H * Ls * 12 * 16 + 2 * 2 * field, 'flops': 0}
    if path == 'slices':
        return {'bytes': 3 * field, 'flops': 3 * H * 12 * Ls * Ls * 8}
    if path == 'hop':
        return {'bytes': 2 * field + link, 'flops': hop}
    if path == 'apply':
        return {'bytes': 2 * (2 * field + link), 'flops': 2 * (hop + 2 * fifth)}
    if path == 'force':
        return {'bytes': 2 * (2 * field + H * 36 * 16) + 2 * H * 36 * 16, 'flops': 2 * 4 * H * Ls * (132 + 4 * 72)}
    # Mpc and MpcDag: four hops; the links of both checkerboards, the field in, the field out
    step = {'bytes': 2 * field + 2 * link, 'flops': 4 * hop + 6 * fifth}
    if path == 'schur':
        return step
    n = iterations(c)
    if path == 'solve' and c['mixed']:     # the steps run in FP32, or in FP16 storage
        step['bytes'] *= 0.5 if c['mixed'] != 2 else 0.27
    extra = 0 if path == 'solve' else 4 * c['nshift'] / 2 * field   # half the poles stay to the end
    return {'bytes': n * (step['bytes'] + extra), 'flops': n * step['flops']}


# ---------------- the same in plain torch, 64 bits ----------------

# gamma_mu psi in the library's basis: component i is phase[i] * psi[source[i]]
GAMMA = (((3, 2, 1, 0), (1j, 1j, -1j, -1j)), ((3, 2, 1, 0), (-1, 1, 1, -1)),
         ((2, 3, 0, 1), (1j, -1j, -1j, 1j)), ((2, 3, 0, 1), (1, 1, 1, 1)))


def whole(c, x, cb):
    """Half-lattice numbers (H4, Ls, 12) of checkerboard cb on the whole lattice (Lt, Lz, Ly, Lx, Ls,
    4, 3), zero on the other one."""
    lx, ly, lz, lt = extent(c)
    full = torch.zeros((lt, lz, ly, lx, c['Ls'], 4, 3), device='cuda', dtype=torch.complex128)
    full.view(-1, c['Ls'] * 12)[sites(c, cb)] = x.reshape(-1, c['Ls'] * 12)
    return full


def half(c, full, cb):
    return full.reshape(-1, c['Ls'], 12)[sites(c, cb)]


def sites(c, cb):
    """Lexicographic numbers of a checkerboard's sites in the order of the half lattice."""
    lx, ly, lz, lt = extent(c)
    t, z, y, x = torch.meshgrid(*(torch.arange(n, device='cuda') for n in (lt, lz, ly, lx // 2)), indexing='ij')
    x = 2 * x + (cb + t + z + y) % 2
    return (x + lx * (y + ly * (z + lz * t))).reshape(-1)


def times(u, psi, dag):
    """u (.., 3, 3) or its adjoint on the colours of psi (.., Ls, 4, 3)."""
    out = []
    for a in range(3):
        v = 0
        for b in range(3):
            w = u[..., b, a].conj() if dag else u[..., a, b]
            v = v + w[..., None, None] * psi[..., b]
        out.append(v)
    return torch.stack(out, -1)


def gamma(mu, psi):
    src, phase = GAMMA[mu]
    return psi[..., list(src), :] * torch.tensor(phase, device='cuda', dtype=torch.complex128)[:, None]


def exact_hop(U, psi, dag):
    sign = -1.0 if dag else 1.0
    out = torch.zeros_like(psi)
    for mu in range(4):
        ax = 3 - mu
        f = torch.roll(psi, -1, ax)
        out += times(U[..., mu, :, :], f - sign * gamma(mu, f), False)
        b = torch.roll(times(U[..., mu, :, :], psi, True), 1, ax)
        out += b + sign * gamma(mu, b)
    return -0.5 * out


def band(c, diag, off, corner):
    """Real Ls x Ls matrices of the two chiralities: diag, off towards s - 1 (spins 0, 1) or s + 1
    (spins 2, 3), `corner` where that wraps."""
    n = c['Ls']
    p = torch.eye(n, dtype=torch.float64, device='cuda') * diag
    for s in range(n):
        p[s, (s - 1) % n] += off if s else corner
    m = torch.eye(n, dtype=torch.float64, device='cuda') * diag
    for s in range(n):
        m[s, (s + 1) % n] += off if s < n - 1 else corner
    return p, m


def fifth(mats, psi):
    out = torch.empty_like(psi)
    for mat, sp in zip(mats, (slice(0, 2), slice(2, 4))):
        v = torch.view_as_real(psi[..., sp, :].contiguous())
        n = v.shape[-4]
        w = torch.matmul(mat, v.reshape(-1, n, 12))
        out[..., sp, :] = torch.view_as_complex(w.reshape(v.shape))
    return out


class Exact:
    def __init__(self, c, U):
        self.c, self.U, self.mob = c, U, c['kind'] == 'mobius'
        m = c['mass']
        if self.mob:
            bee, cee = B * (4 - M5) + 1, 1 - C * (4 - M5)
            self.eo5 = band(c, B, C, -m * C)
            self.ee = band(c, bee, -cee, m * cee)
            self.inv = tuple(torch.linalg.inv(a) for a in self.ee)
        else:
            one = torch.eye(c['Ls'], dtype=torch.float64, device='cuda')
            self.eo5, self.ee, self.inv = (one, one), ((4 + m) * one,) * 2, (one / (4 + m),) * 2

    def dag(self, mats, d):
        return tuple(a.T.contiguous() for a in mats) if d else mats

    def eo(self, psi, d=False):
        if not d:
            return exact_hop(self.U, fifth(self.eo5, psi) if self.mob else psi, False)
        out = exact_hop(self.U, psi, True)
        return fifth(self.dag(self.eo5, True), out) if self.mob else out

    def m(self, psi, d=False):
        return self.eo(psi, d) + fifth(self.dag(self.ee, d), psi)

    def mpc(self, psi, d=False):
        return fifth(self.dag(self.ee, d), psi) - self.eo(fifth(self.dag(self.inv, d), self.eo(psi, d)), d)


def solved(apply, b, tol=1e-14, most=1000):
    """Conjugate gradients on apply, a Hermitian positive map."""
    x, r, p = torch.zeros_like(b), b.clone(), b.clone()
    rr = first = r.abs().square().sum()
    for _ in range(most):
        q = apply(p)
        a = rr / (p.conj() * q).sum().real
        x += a * p
        r -= a * q
        new = r.abs().square().sum()
        if new <= tol * tol * first:
            break
        p = r + new / rr * p
        rr = new
    return x


def exact(c, seed):
    path, Ls = c['path'], c['Ls']
    if path == 'transfer':
        x = torch.view_as_complex(torch.randn(extent(c)[::-1] + (Ls, 4, 3, 2), generator=generator(seed, 2), device='cuda',
                                              dtype=torch.float64))
        return x.cpu().numpy()
    if path == 'slices':
        x, y = (spinor(c, seed, k, 1)[0].transpose(0, 1).reshape(Ls, -1) for k in (2, 3))
        a = torch.from_numpy(coefficients(c, seed)).cuda()
        r = (y - a.T.contiguous() @ x).reshape(Ls, -1, 12).transpose(0, 1)
        adj = x.conj().resolve_conj()
        m, g = (adj @ v.T.contiguous() for v in (y, x))
        return m.cpu().numpy(), g.cpu().numpy(), stored(r[None], 'f64')
    # the plain solves of light 5D systems and of the poles take minutes
    if path == 'shifts' or (path == 'solve' and (c['kind'] == 'mobius' or c['lx'] * c['ly'] * c['lz'] * c['lt'] * Ls > 2e5)):
        return None
    U = links(c, seed)
    E = Exact(c, U)
    dag = bool(c.get('dag'))

    def put(*halves):
        return [stored(torch.stack(halves), c['prec'])]

    if path == 'hop':
        psi = whole(c, spinor(c, seed, 2, 1)[0], gx.ODD)
        return put(half(c, exact_hop(U, psi, dag), gx.EVEN))
    if path == 'schur':
        psi = whole(c, spinor(c, seed, 2, 1)[0], gx.ODD)
        return put(half(c, E.mpc(E.mpc(psi), True), gx.ODD))
    x = spinor(c, seed, 2, 2)
    psi = whole(c, x[0], 0) + whole(c, x[1], 1)
    if path == 'force':
        y = spinor(c, seed, 3, 2)
        chi = whole(c, y[0], 0) + whole(c, y[1], 1)
        sign = -1.0 if dag else 1.0
        mats = []
        for mu in range(4):
            f = torch.roll(chi, -1, 3 - mu)
            f = -0.5 * times(U[..., mu, :, :], f - sign * gamma(mu, f), False)
            mats.append(torch.stack([torch.stack([(f[..., a] * psi[..., b].conj()).sum((-1, -2)) for b in range(3)], -1)
                                     for a in range(3)], -2))
        return torch.stack(mats, 4).cpu().numpy()
    if path == 'solve':
        out = solved(lambda v: E.m(E.m(v), True), E.m(psi, True))
    else:
        out = E.m(psi, dag)
    return put(half(c, out, 0), half(c, out, 1))
