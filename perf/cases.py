"""Timed cases of the framework's public entry points.

Twelve listed cases and, with ``draw``, more of the same ranges: linear
systems (one small system, a batch on one workgroup each, a batch on the mixed
schedule, a large system on a gang in FP64 and in FP32 with FP64 refinement),
eigenproblems (one chain, a batch of chains), the rank-adaptive solver, an
implicit time integration, the residual check of a batch, and the two TT
operations that a solver's user spends time in: operator times vector, and
rounding.

Inputs.  ``-Laplacian`` and TFIM operators as in ``scikit_tt_amd.workloads``;
batches have the sizes of the uneven batch of the benchmark (order 8..24,
modes 4, 8 or 16, rank 4..48; operator ``d I`` plus a rank-3 perturbation) in
the form of one implicit time step of an ensemble: the right-hand side is the
previous state, a train of the solution's rank, and the solve starts from it.
Outputs are compared number by number, so they are quantities that do not
depend on an arbitrary choice of basis: the full tensor where it fits, the
cores where every bond has full numerical rank (the QR is then unique),
eigenvalues of chains whose Schmidt values decay below rounding.
"""
import math

import numpy as np
import torch

from scikit_tt_amd import tensor_train as tt
from scikit_tt_amd import workloads as W
from scikit_tt_amd.solvers import evp, ode, sle
from scikit_tt_amd.tensor_train import TT


def listed():
    return [
        # one small system as a script solves it: latency of one call (the rank-5 Laplacian with an all-ones
        # right-hand side of the small configuration, at an order whose full tensor can be returned)
        {'name': 'als_small', 'kind': 'als', 'd': 6, 'n': 8, 'r': 5, 'sweeps': 4},
        # implicit Euler on the heat equation: many short calls, local systems of at most 96 unknowns (dense LU),
        # TT sums, products and norms between the solves
        {'name': 'heat_steps', 'kind': 'heat', 'd': 8, 'n': 4, 'r': 4, 'steps': 4},
        # rank-adaptive two-site solve, driven from the host piece by piece
        {'name': 'mals', 'kind': 'mals', 'd': 6, 'n': 8, 'r': 4, 'cap': 8},
        # one chain's ground state
        {'name': 'evp_small', 'kind': 'evp', 'd': 12, 'r': 8, 'sweeps': 3},
        # an ensemble of uneven systems, one workgroup each (the default schedule)
        {'name': 'batch_one', 'kind': 'batch', 'count': 192, 'dmax': 24, 'rmax': 32, 'schedule': 'one', 'sweeps': 1},
        # the benchmark's batch size and ranges on the mixed schedule
        {'name': 'batch_auto', 'kind': 'batch', 'count': 512, 'dmax': 24, 'rmax': 48, 'schedule': 'auto', 'sweeps': 1},
        # a large system on a gang of workgroups: the large Laplacian's modes and ranks, FP64
        {'name': 'gang_fp64', 'kind': 'gang', 'd': 4, 'n': 32, 'r': 32, 'precision': 'fp64', 'sweeps': 2},
        # the same engine with FP32 Krylov steps and FP64 refinement, at an odd mode size
        {'name': 'gang_mixed', 'kind': 'gang', 'd': 4, 'n': 21, 'r': 40, 'precision': 'mixed', 'sweeps': 1},
        # the eigenproblem batch of the benchmark: TFIM chains, 32 sites, rank 16, adaptive local tolerance
        {'name': 'evp_batch', 'kind': 'evps', 'count': 1024, 'd': 32, 'r': 16, 'sweeps': 4, 'adaptive': True},
        # residual check of a batch of approximate solutions in one launch
        {'name': 'residuals', 'kind': 'resid', 'count': 96, 'dmax': 24, 'rmax': 32},
        # operator times vector, then rounding back
        {'name': 'round', 'kind': 'round', 'd': 10, 'n': 4, 'r': 20},
        # operator times a large-rank vector: memory traffic
        {'name': 'matvec', 'kind': 'matvec', 'd': 8, 'n': 16, 'r': 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['als', 'heat', 'mals', 'evp', 'batch', 'batch', 'gang', 'gang', 'evps', 'resid', 'round',
                       'matvec'])
    if kind in ('als', 'heat'):
        n = rng.randint(3, 12)
        d = rng.randint(3, max(3, int(math.log(3e5) / math.log(n))))
        if kind == 'als':
            return {'kind': kind, 'd': d, 'n': n, 'r': rng.randint(2, 9), 'sweeps': rng.randint(1, 4)}
        return {'kind': kind, 'd': d, 'n': n, 'r': rng.randint(2, 7), 'steps': rng.randint(1, 5)}
    if kind == 'mals':
        n = rng.randint(4, 9)
        return {'kind': kind, 'd': rng.randint(4, 6 if n <= 7 else 5), 'n': n, 'r': rng.randint(2, 5),
                'cap': rng.randint(5, 9)}
    if kind == 'evp':
        return {'kind': kind, 'd': rng.randint(6, 16), 'r': rng.randint(4, 14), 'sweeps': rng.randint(2, 4)}
    if kind == 'batch':
        return {'kind': kind, 'count': _log(rng, 4, 400), 'dmax': rng.randint(9, 24), 'rmax': rng.randint(6, 48),
                'schedule': rng.choice(['one', 'auto']), 'sweeps': 1}
    if kind == 'gang':
        return {'kind': kind, 'd': 4, 'n': _log(rng, 9, 32), 'r': _log(rng, 10, 48),
                'precision': rng.choice(['fp64', 'mixed']), 'sweeps': 1}
    if kind == 'evps':
        return {'kind': kind, 'count': _log(rng, 16, 1024), 'd': rng.randint(8, 32), 'r': rng.randint(5, 16),
                'sweeps': rng.randint(2, 4), 'adaptive': rng.random() < 0.5}
    if kind == 'resid':
        return {'kind': kind, 'count': _log(rng, 4, 96), 'dmax': rng.randint(9, 24), 'rmax': rng.randint(6, 32)}
    if kind == 'round':
        n = rng.randint(2, 5)
        return {'kind': kind, 'd': rng.randint(6, {2: 14, 3: 10, 4: 9, 5: 8}[n]), 'n': n, 'r': _log(rng, 5, 20)}
    return {'kind': 'matvec', 'd': rng.randint(3, 8), 'n': rng.choice([2, 3, 4, 7, 8, 11, 16]), 'r': _log(rng, 6, 128)}


# -- inputs ---------------------------------------------------------------------------------------


def _ranks(d, n, r):
    """The rank profile of a train of rank r: no bond above what its modes allow."""
    return [min(r, n ** min(i, 24), n ** min(d - i, 24)) for i in range(d + 1)]


def _states(gen, shapes):
    """Trains of N(0, 1) cores scaled to a norm near 1, made on the device in one buffer.

    ``shapes``: (d, n, rank profile) per train."""
    dev = tt.device()
    total = sum(rs[i] * n * rs[i + 1] for d, n, rs in shapes for i in range(d))
    flat = torch.randn(total, dtype=torch.float64, device=dev, generator=gen)
    out, at = [], 0
    for d, n, rs in shapes:
        cores = []
        for i in range(d):
            size = rs[i] * n * rs[i + 1]
            cores.append(flat[at:at + size].view(rs[i], n, 1, rs[i + 1]))
            cores[-1] *= 1.0 / math.sqrt(n * rs[i + 1])
            at += size
        out.append(TT(cores))
    return out


def _gen(seed):
    return torch.Generator(device=tt.device()).manual_seed(int(seed))


def _systems(case):
    """(d, n, r) of each system of an uneven batch: part of the case, not of its seed."""
    rng = np.random.default_rng(case['count'] * 1000003 + case['dmax'] * 1009 + case['rmax'])
    return [(int(rng.integers(8, case['dmax'] + 1)), int(rng.choice((4, 8, 16))),
             int(rng.integers(4, case['rmax'] + 1))) for _ in range(case['count'])]


def _chains(case, seed):
    """Couplings and right-orthonormal starts of `count` chains (host, all at once)."""
    count, d, r = case.get('count', 1), case['d'], case['r']
    rng = np.random.default_rng(seed)
    J, g = rng.uniform(0.5, 1.5, (count, d - 1)), rng.uniform(0.5, 1.5, (count, d))
    rs = _ranks(d, 2, r)
    cores, push = [None] * d, np.ones((count, 1, 1))
    for i in range(d - 1, -1, -1):
        c = rng.standard_normal((count, rs[i], 2, rs[i + 1])) @ push[:, None]
        if i > 0:
            q, f = np.linalg.qr(c.reshape(count, rs[i], -1).transpose(0, 2, 1))
            cores[i] = np.ascontiguousarray(q.transpose(0, 2, 1)).reshape(count, rs[i], 2, 1, rs[i + 1])
            push = f.transpose(0, 2, 1)
        else:
            cores[i] = (c / np.sqrt((c * c).sum(axis=(1, 2, 3), keepdims=True)))[:, :, :, None, :]
    return [W.tfim_operator(J[s], g[s]) for s in range(count)], [[c[s] for c in cores] for s in range(count)]


def _laplace(case, seed):
    """Operator, start and right-hand side of a Laplacian system, on the host."""
    d, n, r = case['d'], case['n'], case['r']
    rng = np.random.default_rng(seed)
    x0 = W.right_orthonormal(W.random_tt(rng, [n] * d, _ranks(d, n, r)))
    if case['kind'] == 'gang':
        b = W.random_tt(rng, [n] * d, _ranks(d, n, (r + 1) // 2), scale=0.5 / math.sqrt(n))
    else:
        b = W.ones_tt([n] * d)
        b[0] = b[0] * rng.uniform(0.5, 1.5, (1, n, 1, 1))  # a source that varies along the first mode
    return W.laplace_operator(d, n), x0, b


def prepare(case, seed):
    kind = case['kind']
    state = {'case': case}
    if kind in ('als', 'mals', 'gang'):
        A, x0, b = _laplace(case, seed)
        state.update(A=TT(A), x0=TT(x0), b=TT(b))
    elif kind == 'heat':
        d, n = case['d'], case['n']
        A, x0, v = _heat(case, seed)
        state.update(A=TT(A), x0=TT(x0), v=TT(v), steps=[0.5 / (n + 1) ** 2 * (k + 1) for k in range(case['steps'])])
    elif kind in ('evp', 'evps'):
        A, x0 = _chains(case, seed)
        state.update(A=tt.from_host_batch(A), x0=tt.from_host_batch(x0))
    elif kind in ('batch', 'resid'):
        sys_ = _systems(case)
        rng = np.random.default_rng(seed)
        state['A'] = tt.from_host_batch([W.shifted_operator(rng, d, n) for d, n, r in sys_])
        gen = _gen(seed)
        state['x'] = _states(gen, [(d, n, _ranks(d, n, r)) for d, n, r in sys_])
        if kind == 'resid':
            state['b'] = _states(gen, [(d, n, _ranks(d, n, 4)) for d, n, r in sys_])
    else:
        d, n, r = case['d'], case['n'], case['r']
        state['A'] = TT(W.shifted_operator(np.random.default_rng(seed), d, n))
        state['x'] = _states(_gen(seed), [(d, n, _ranks(d, n, r))])[0]
    return state


def _heat(case, seed):
    """-Laplacian generator, starting guess and initial state (two bumps) of the heat equation."""
    d, n, r = case['d'], case['n'], case['r']
    rng = np.random.default_rng(seed)
    A = W.laplace_operator(d, n)
    A[0] = -A[0]
    for i in range(1, d):  # core 0 carries D and I, the others pass one of the two on: the sign goes to every D
        A[i] = A[i].copy()
        A[i][1, :, :, 0] = -A[i][1, :, :, 0]
    A[0][0, :, :, 1] = np.eye(n)
    grid = (np.arange(n) + 1.0) / (n + 1)
    bumps = [[np.exp(-(grid - c) ** 2 / 0.08).reshape(1, n, 1, 1) for c in rng.uniform(0.2, 0.8, d)] for _ in range(2)]
    x0 = W.right_orthonormal(W.random_tt(rng, [n] * d, _ranks(d, n, r)))
    return A, x0, W.tt_sum(bumps[0], bumps[1])


# -- one pass -------------------------------------------------------------------------------------


def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'als':
        return sle.als(state['A'], state['x0'], state['b'], repeats=case['sweeps']).full()
    if kind == 'heat':
        steps = ode.implicit_euler(state['A'], state['v'], state['x0'], state['steps'], repeats=2, normalize=2)
        return [s.full() for s in steps[1:]]
    if kind == 'mals':
        return sle.mals(state['A'], state['x0'], state['b'], repeats=1, threshold=1e-10, max_rank=case['cap']).full()
    if kind == 'gang':
        x = sle.als_gang([state['A']], [state['x0']], [state['b']], repeats=case['sweeps'],
                         precision=case['precision'])[0]
        return x.full()
    if kind == 'evp':
        value, x, iterations = evp.als(state['A'][0], state['x0'][0], repeats=case['sweeps'], conv_eps=0, sigma=-100)
        return {'value': value, 'vector': x.full(), 'iterations': iterations}
    if kind == 'evps':
        out = evp.als_batch(state['A'], state['x0'], repeats=case['sweeps'], conv_eps=0, sigma=-100,
                            adaptive_tol=case['adaptive'])
        return out.eigenvalues
    if kind == 'batch':
        xs = sle.als_batch(state['A'], state['x'], state['x'], repeats=case['sweeps'], schedule=case['schedule'])
        # the cores of a batch are views of one device buffer: every solution, whole
        return xs[0].device_cores[0]._base
    if kind == 'resid':
        return tt.residual_norms(state['A'], state['x'], state['b'])
    if kind == 'round':
        return state['A'].dot(state['x']).ortho(threshold=1e-10, max_rank=2 * case['r']).full()
    return state['A'].dot(state['x']).device_cores


# -- what one pass cannot do without --------------------------------------------------------------


def _cores(ra, rs, n, i):
    """Entries of operator core, state core."""
    return ra[i] * n * n * ra[i + 1], rs[i] * n * rs[i + 1]


def _sweep_flops(ra, rs, n, d, matvecs):
    """One forward and backward sweep: per position a stack update, `matvecs` local products and a QR."""
    total = 0.0
    for i in range(d):
        a, b, P, Q = rs[i], rs[i + 1], ra[i], ra[i + 1]
        op = 2.0 * a * b * n * (a * P + P * n * Q + b * Q)
        total += (2 if i < d - 1 else 1) * (op * (1 + matvecs) + 4.0 * a * n * b * min(a, b))
    return total


def _bytes(ra, rs, rb, n, d):
    return 8.0 * sum(ra[i] * n * n * ra[i + 1] + 2 * rs[i] * n * rs[i + 1] + rb[i] * n * rb[i + 1] for i in range(d))


def work(case):
    kind = case['kind']

    def inner(r, d):
        return [1] + [r] * (d - 1) + [1]

    if kind in ('als', 'heat', 'mals', 'gang'):
        d, n = case['d'], case['n']
        rs, ra = _ranks(d, n, case.get('cap', case['r'])), inner(2, d)
        rb = _ranks(d, n, (case['r'] + 1) // 2) if kind == 'gang' else inner(1, d)
        reps = case.get('sweeps', 1) if kind != 'heat' else 2 * case['steps']
        nn = n * n if kind == 'mals' else n
        return {'bytes': _bytes(ra, rs, rb, n, d) * (case['steps'] if kind == 'heat' else 1) + 8.0 * n ** d,
                'flops': reps * _sweep_flops(ra, rs, nn, d, 8)}
    if kind in ('evp', 'evps'):
        d, count = case['d'], case.get('count', 1)
        rs, ra = _ranks(d, 2, case['r']), inner(3, d)
        return {'bytes': count * _bytes(ra, rs, [0] * (d + 1), 2, d),
                'flops': count * case['sweeps'] * _sweep_flops(ra, rs, 2, d, 8)}
    if kind in ('batch', 'resid'):
        nbytes = flops = 0.0
        for d, n, r in _systems(case):
            rs, ra = _ranks(d, n, r), inner(4, d)
            rb = rs if kind == 'batch' else _ranks(d, n, 4)
            nbytes += _bytes(ra, rs, rb, n, d)
            if kind == 'batch':
                flops += case['sweeps'] * _sweep_flops(ra, rs, n, d, 2)
            else:
                # the norm of the residual train from its transfer matrices: rank rho on every bond
                for i in range(d):
                    r0, r1 = ra[i] * rs[i] + rb[i], ra[i + 1] * rs[i + 1] + rb[i + 1]
                    flops += 2.0 * n * r0 * r1 * (r0 + r1) / 2
        return {'bytes': nbytes, 'flops': flops}
    d, n, r = case['d'], case['n'], case['r']
    rs, ra = _ranks(d, n, r), inner(4, d)
    out = [ra[i] * rs[i] for i in range(d)] + [1]
    prod = sum(2.0 * out[i] * n * n * out[i + 1] for i in range(d))
    nbytes = 8.0 * sum(sum(_cores(ra, rs, n, i)) + out[i] * n * out[i + 1] for i in range(d))
    if kind == 'matvec':
        return {'bytes': nbytes, 'flops': prod}
    return {'bytes': 8.0 * (sum(sum(_cores(ra, rs, n, i)) for i in range(d)) + n ** d),
            'flops': prod + sum(8.0 * out[i] * n * out[i + 1] * min(out[i], out[i + 1]) for i in range(d))}


# -- the same results by plain numpy / torch in 64 bits -------------------------------------------


def _full(cores):
    t = np.ones((1, 1))
    for c in cores:
        t = (t @ c.reshape(c.shape[0], -1)).reshape(-1, c.shape[-1])
    return t.reshape([c.shape[1] for c in cores])


def _kron_solve(L, op, R, f):
    """(L0 x I x I + I x D x I + I x I x R1) v = f: the local problem of a Laplacian train between orthonormal
    interfaces, by three eigenbases."""
    a, n, e = f.shape
    l0 = L[:, 0, :] if L.shape[1] == 2 else np.zeros((a, a))
    r1 = R[:, 1, :] if R.shape[1] == 2 else np.zeros((e, e))
    parts = [np.linalg.eigh((m + m.T) / 2) for m in (l0, op[-1, :, :, 0], r1)]
    (wl, vl), (wd, vd), (wr, vr) = parts

    def turn(t, u, v, w):
        return np.tensordot(u, np.tensordot(np.tensordot(t, w, 1), v, (1, 0)), 1).transpose(0, 2, 1)

    t = turn(f, vl.T, vd, vr) / (wl[:, None, None] + wd[None, :, None] + wr[None, None, :])
    return turn(t, vl, vd.T, vr.T)


def _svd(m, threshold, cap):
    u, s, w = np.linalg.svd(m, full_matrices=False)
    k = min(int(np.sum(s / s[0] > threshold)), cap)
    return u[:, :k], s[:k], w[:k]


class _Als:
    """ALS with direct local solves: b None for the lowest eigenpair; `laplace` takes the Kronecker-sum solve."""

    def __init__(self, A, x0, b, laplace=False):
        self.A, self.d, self.laplace = A, len(A), laplace
        self.x = [c[:, :, 0, :].copy() for c in x0]
        self.B = None if b is None else [c[:, :, 0, :] for c in b]
        self.L, self.R, self.Lb, self.Rb = ({0: np.ones((1,) * k), self.d: np.ones((1,) * k)} for k in (3, 3, 2, 2))
        for i in range(self.d - 1, 0, -1):
            self.keep(i, self.x[i], False, push=True)
            self.right(i)

    def left(self, i):  # interface left of site i + 1
        x = self.x[i]
        t = np.tensordot(np.tensordot(self.L[i], x, (0, 0)), self.A[i], ((0, 2), (0, 2)))  # c b m q
        self.L[i + 1] = np.tensordot(t, x, ((0, 2), (0, 1)))
        if self.B:
            self.Lb[i + 1] = np.einsum('pc,pmq,cmd->qd', self.Lb[i], self.B[i], x, optimize=True)

    def right(self, i):  # interface right of site i - 1
        x = self.x[i]
        t = np.tensordot(np.tensordot(self.R[i + 1], x, (0, 2)), self.A[i], ((0, 3), (3, 2)))  # d a p m
        self.R[i] = np.tensordot(t, x, ((0, 3), (2, 1)))
        if self.B:
            self.Rb[i] = np.einsum('qd,pmq,cmd->pc', self.Rb[i + 1], self.B[i], x, optimize=True)

    def keep(self, i, v, forward, push=False):
        """Core i from the local solution: its left (forward) or right orthonormal factor."""
        a, n, e = v.shape
        if forward:
            self.x[i] = np.linalg.qr(v.reshape(a * n, e))[0].reshape(a, n, -1)
        elif i > 0:
            q, f = np.linalg.qr(v.reshape(a, n * e).T)
            self.x[i] = q.T.reshape(-1, n, e)
            if push:
                self.x[i - 1] = self.x[i - 1] @ f.T
        else:
            self.x[i] = v

    def local(self, i, j):
        """Solution over the sites i..j-1 (one or two)."""
        op, L, R = self.A[i], self.L[i], self.R[j]
        f = self.B[i] if self.B else None
        if j == i + 2:
            o = self.A[i + 1]
            op = np.einsum('pmns,sklq->pmknlq', op, o).reshape(op.shape[0], op.shape[1] * o.shape[1], -1, o.shape[3])
            f = np.tensordot(f, self.B[i + 1], 1).reshape(f.shape[0], -1, self.B[i + 1].shape[2])
        a, n, e = L.shape[0], op.shape[1], R.shape[0]
        if self.B:
            f = np.tensordot(np.tensordot(self.Lb[i], f, (0, 0)), self.Rb[j], 1)
            if self.laplace:
                return _kron_solve(L, op, R, f)
        M = np.einsum('apc,pmnq,bqd->cmdanb', L, op, R, optimize=True).reshape(a * n * e, -1)
        if self.B:
            return np.linalg.solve(M, f.ravel()).reshape(a, n, e)
        w, v = np.linalg.eigh((M + M.T) / 2)
        self.value = float(w[0])
        return v[:, 0].reshape(a, n, e)

    def sweep(self):
        for i in range(self.d - 1):
            self.keep(i, self.local(i, i + 1), True)
            self.left(i)
        for i in range(self.d - 1, -1, -1):
            self.keep(i, self.local(i, i + 1), False)
            if i:
                self.right(i)
        return self

    def sweep_two(self, threshold, cap):
        def split(i):
            v = self.local(i, i + 2)
            a, e, n = v.shape[0], v.shape[2], self.A[i].shape[1]
            u, s, w = _svd(v.reshape(a * n, -1), threshold, cap)
            return u, s, w, lambda m: m.reshape(a, n, -1), lambda m: m.reshape(len(s), -1, e)

        for i in range(self.d - 2):
            u, s, w, first, second = split(i)
            self.x[i], self.x[i + 1] = first(u), second(s[:, None] * w)
            self.left(i)
        for i in range(self.d - 2, -1, -1):
            u, s, w, first, second = split(i)
            self.x[i], self.x[i + 1] = first(u * s), second(w)
            self.right(i + 1)
        return self


def _inner(x, y):
    """<x, y> of two trains of device cores (r, n, r'), in 64 bits."""
    E = torch.ones((1, 1), dtype=torch.float64, device=x[0].device)
    for p, q in zip(x, y):
        t = torch.tensordot(E, p, dims=([0], [0]))  # s n r'
        E = torch.tensordot(t, q, dims=([0, 1], [0, 1]))
    return E


def _product(A, x):
    """Operator times vector, core by core: (P a, n, Q b)."""
    out = []
    for p, q in zip(A, x):
        t = torch.tensordot(p, q[:, :, 0, :], dims=([2], [1]))  # P m Q a b
        t = t.permute(0, 3, 1, 2, 4)
        out.append(t.reshape(t.shape[0] * t.shape[1], t.shape[2], -1))
    return out


def exact(case, seed):
    kind = case['kind']
    if kind in ('als', 'mals', 'gang'):
        A, x0, b = _laplace(case, seed)
        solve = _Als(A, x0, b, laplace=True)
        if kind == 'mals':
            return _full(solve.sweep_two(1e-10, case['cap']).x)
        for _ in range(case['sweeps']):
            solve.sweep()
        return _full(solve.x)
    if kind == 'heat':
        d, n = case['d'], case['n']
        A, x, v = _heat(case, seed)
        out = []
        for k in range(case['steps']):
            h = 0.5 / (n + 1) ** 2 * (k + 1)
            op = W.tt_sum(W.identity_operator([n] * d), [-h * A[0]] + A[1:])
            x = _Als(op, x, v).sweep().sweep().x
            x = [x[0] / np.linalg.norm(_full(x))] + x[1:]
            out.append(_full(x))
            x = v = [c[:, :, None, :] for c in x]
        return out
    if kind == 'evp':
        A, x0 = _chains(case, seed)
        solve, best = _Als(A[0], x0[0], None), math.inf
        for _ in range(case['sweeps']):
            best = min(best, solve.sweep().value)
        return {'value': best, 'vector': None, 'iterations': case['sweeps']}  # (the vector's sign is arbitrary)
    if kind == 'resid':
        state = prepare(case, seed)
        res, rhs = [], []
        for A, x, b in zip(state['A'], state['x'], state['b']):
            y, z = _product(A.device_cores, x.device_cores), [c[:, :, 0, :] for c in b.device_cores]
            yy, yz, zz = (float(_inner(*p)) for p in ((y, y), (y, z), (z, z)))
            res.append(math.sqrt(yy - 2 * yz + zz))
            rhs.append(math.sqrt(zz))
        return np.array(res), np.array(rhs)
    if kind == 'matvec':
        state = prepare(case, seed)
        return [c[:, :, None, :] for c in _product(state['A'].device_cores, state['x'].device_cores)]
    if kind == 'round':
        state = prepare(case, seed)
        y = [c.cpu().numpy() for c in _product(state['A'].device_cores, state['x'].device_cores)]
        for i in range(len(y) - 1):
            r, n, e = y[i].shape
            u, s, w = _svd(y[i].reshape(r * n, e), 1e-10, 1 << 30)
            y[i], y[i + 1] = u.reshape(r, n, -1), np.tensordot(s[:, None] * w, y[i + 1], 1)
        for i in range(len(y) - 1, 0, -1):
            r, n, e = y[i].shape
            u, s, w = _svd(y[i].reshape(r, n * e), 1e-10, 2 * case['r'])
            y[i], y[i - 1] = w.reshape(-1, n, e), np.tensordot(y[i - 1], u * s, 1)
        return _full(y)
    return None  # the batches: dense local solves of up to 36864 unknowns, thousands of local eigenproblems
