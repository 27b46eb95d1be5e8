"""Timed cases of the engine: the calls a sampling program makes, from one
chain on a thousand rows to 4096 chains on a million.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges,
``prepare(case, seed)`` makes what a program holds before the call (data
bound, chains' start points, weights), ``run(state)`` makes the call,
``work(case)`` counts the bytes and operations it needs, and
``exact(case, seed)`` gives its outputs in float64 from plain torch / numpy.

Accept uniforms fed to the multi-chain cases lie in (0, 2e-4): with log
ratios of a few nats every proposal is taken, and no accept decision hangs on
the last digits of a log joint of 1e5 nats.
"""

import math

import numpy as np
import torch

from edward_amd import diagnostics, readout
from edward_amd.engine import Context, GLMEngine
from edward_amd.hier import HierEngine
from edward_amd.surrogate import Surrogate

_DEV = 'cuda'
_CHUNK = 32768          # rows per float64 block of the exact values
_LLC = 32 << 20         # data above this size is read anew by every evaluation


def listed():
  return [
      # One chain on a small table, twenty transitions in one call: Edward's
      # logistic-regression example; nothing but latency.
      dict(name='one_chain_small', kind='run', N=1000, D=10, C=1, L=10, T=20,
           precision='fp32', lik='bernoulli'),
      # One chain on a table of Covertype's size (581,012 x 54): the HMC
      # program of Edward's own paper, ten leapfrog steps a transition.
      dict(name='one_chain_covertype', kind='run', N=581012, D=54, C=1, L=10, T=3,
           precision='fp32', lik='bernoulli'),
      # A workstation run: a few dozen chains, sizes that divide nothing.
      dict(name='chains_ragged', kind='chains', N=100003, D=101, C=50, L=10,
           precision='fp32', lik='bernoulli'),
      # The mid configuration of the benchmark, one transition from a fresh
      # state, fp32.
      dict(name='chains_mid', kind='chains', N=100000, D=256, C=1024, L=20,
           precision='fp32', lik='bernoulli'),
      # The large configuration in bf16: a short descent transition as the
      # warm-up makes them.
      dict(name='chains_large', kind='chains', N=1000000, D=512, C=4096, L=4,
           precision='bf16', lik='bernoulli'),
      # Surrogate-driven sampling of the large configuration: 32 network
      # steps and one exact forward pass a transition, four transitions.
      dict(name='surrogate_sampling', kind='sur_sample', N=1000000, D=512, C=4096, H=1024, L=32,
           T=4),
      # Start of surrogate training on recorded pairs: normalisation from
      # the column statistics, least-squares linear skip.
      dict(name='surrogate_start', kind='sur_start', P=196608, D=512, H=1024),
      # Loss and parameter gradient of one training batch.
      dict(name='surrogate_gradient', kind='sur_grad', B=4096, D=512, H=1024),
      # Hierarchical regression with 2048 groups, one transition of 512
      # chains.
      dict(name='hier_groups', kind='hier', G=2048, mean=400, D=64, C=512, L=16),
      # Criticism: the posterior predictive of evaluate()'s 500 draws.
      dict(name='predictive', kind='predict', N=200000, D=100, S=500, precision='fp32',
           lik='bernoulli'),
      # Readout of a sample store: effective sample sizes, means, variances.
      dict(name='readout', kind='readout', T=1000, C=1024, D=256),
      # Newton terms at one position (log joint, gradient, Hessian): a step
      # of the Laplace warm start on the large configuration.
      dict(name='newton', kind='newton', N=1000000, D=512, precision='bf16', lik='bernoulli'),
  ]


# -- drawn cases ---------------------------------------------------------------

def _log_int(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  kind = rng.choice(['run', 'run', 'chains', 'chains', 'chains', 'sur_sample', 'sur_start',
                     'sur_grad', 'hier', 'predict', 'readout', 'newton'])
  prec = rng.choice(['fp32', 'bf16'])
  lik = rng.choice(['bernoulli', 'bernoulli', 'bernoulli', 'normal'])
  if kind == 'run':
    return dict(kind=kind, N=_log_int(rng, 100, 1000000), D=_log_int(rng, 1, 128),
                C=rng.choice([1, 1, 2, 4]), L=rng.randint(2, 12), T=rng.randint(2, 6),
                precision=prec, lik=lik)
  if kind == 'chains':
    N, D, C = _log_int(rng, 500, 1000000), _log_int(rng, 2, 512), _log_int(rng, 8, 4096)
    L = rng.randint(2, 12)
    # at most the work of chains_large in bf16, of chains_mid in fp32
    cap = 5 * 1e6 * 512 * 4096 if prec == 'bf16' else 21 * 1e5 * 256 * 1024
    while (L + 1) * N * D * float(C) > cap:
      N = max(500, int(0.7 * N))
      C = max(8, int(0.8 * C))
    return dict(kind=kind, N=N, D=D, C=C, L=L, precision=prec, lik=lik)
  if kind == 'sur_sample':
    return dict(kind=kind, N=_log_int(rng, 10000, 1000000), D=_log_int(rng, 16, 512),
                C=_log_int(rng, 128, 4096), H=_log_int(rng, 64, 1024), L=rng.randint(4, 32),
                T=rng.randint(1, 4))
  if kind == 'sur_start':
    return dict(kind=kind, P=_log_int(rng, 4000, 196608), D=_log_int(rng, 8, 512),
                H=_log_int(rng, 64, 1024))
  if kind == 'sur_grad':
    return dict(kind=kind, B=_log_int(rng, 128, 4096), D=_log_int(rng, 8, 512),
                H=_log_int(rng, 64, 1024))
  if kind == 'hier':
    return dict(kind=kind, G=_log_int(rng, 8, 2048), mean=_log_int(rng, 5, 400),
                D=_log_int(rng, 1, 64), C=_log_int(rng, 4, 512), L=rng.randint(2, 16))
  if kind == 'predict':
    return dict(kind=kind, N=_log_int(rng, 500, 200000), D=_log_int(rng, 2, 100),
                S=_log_int(rng, 50, 500), precision=prec, lik=lik)
  if kind == 'readout':
    return dict(kind=kind, T=_log_int(rng, 100, 1000), C=_log_int(rng, 1, 1024),
                D=_log_int(rng, 2, 256))
  return dict(kind=kind, N=_log_int(rng, 1000, 1000000), D=_log_int(rng, 2, 512),
              precision=prec, lik=lik)


# -- inputs --------------------------------------------------------------------

def _gen(seed):
  return torch.Generator(device=_DEV).manual_seed(int(seed))


def _randn(g, *shape):
  return torch.randn(*shape, generator=g, device=_DEV)


def _data(case, g):
  """Design matrix with column scales in (0.5, 2), coefficients, and
  observations drawn from the model; bf16 cases hand X over in bf16."""
  N, D = case['N'], case['D']
  scale = 0.5 + 1.5 * torch.rand(D, generator=g, device=_DEV)
  w = 0.1 * _randn(g, D)
  X = _randn(g, N, D) * scale
  if case.get('precision', 'bf16') == 'bf16':
    X = X.to(torch.bfloat16)
  eta = torch.empty(N, device=_DEV)
  for s in range(0, N, _CHUNK):
    eta[s:s + _CHUNK] = X[s:s + _CHUNK].float() @ w
  if case.get('lik', 'bernoulli') == 'bernoulli':
    y = (torch.rand(N, generator=g, device=_DEV) < torch.sigmoid(eta)).float()
  else:
    y = eta + _randn(g, N)
  return X, y, w


def _starts(case, g, w):
  """Chains within a posterior standard deviation or so of the generating
  coefficients, momenta and accept uniforms."""
  D, C = case['D'], case['C']
  W0 = w + _width(case) * _randn(g, C, D)
  r0 = _randn(g, C, D)
  u = 2e-4 * torch.rand(C, generator=g, device=_DEV, dtype=torch.float64) + 1e-12
  return W0, r0, u


def _width(case):
  """A posterior standard deviation or so of one coefficient."""
  return ((0.2 if case.get('lik', 'bernoulli') == 'bernoulli' else 1.0) * case['N']) ** -0.5


def _eps(case):
  """Step size, as float32: 0.3 over the square root of the largest
  curvature (a Normal row's is 1, a Bernoulli row's at most 1/4, times the
  column's scale of at most 2 squared)."""
  c = 0.3 if case.get('lik', 'bernoulli') == 'bernoulli' else 0.15
  return float(np.float32(c / math.sqrt(case['N'] + 1.0)))


def _sur_net(D, H, g, skip=None):
  """Flat surrogate parameters [W1 b1 W2 b2 W3 b3]: Glorot hidden layers, a
  small hidden output part, and the linear skip."""
  def glorot(o, i):
    a = math.sqrt(6.0 / (i + o))
    return a * (2.0 * torch.rand(o, i, generator=g, device=_DEV) - 1.0)
  b = lambda n: 0.05 * _randn(g, n)
  W1, b1, W2, b2 = glorot(H, D), b(H), glorot(H, H), b(H)
  Wh = 0.01 * glorot(D, H)
  Wx = torch.zeros(D, D, device=_DEV) if skip is None else skip
  b3 = torch.zeros(D, device=_DEV)
  return torch.cat([W1.reshape(-1), b1, W2.reshape(-1), b2,
                    torch.cat([Wh, Wx], 1).reshape(-1), b3])


def _newton_point(X, y, w):
  """One float32 Newton step of the logistic posterior from w: the mode to
  within the data's rounding, and the negative Hessian."""
  D = X.shape[1]
  g = torch.zeros(D, device=_DEV)
  Hm = torch.zeros(D, D, device=_DEV)
  for s in range(0, X.shape[0], _CHUNK):
    x = X[s:s + _CHUNK].float()
    p = torch.sigmoid(x @ w)
    g += x.t() @ (y[s:s + _CHUNK] - p)
    Hm += (x * (p * (1 - p))[:, None]).t() @ x
  g -= w
  Hm += torch.eye(D, device=_DEV)
  return w + torch.linalg.solve(Hm, g), Hm


def _sur_inputs(case, seed):
  g = _gen(seed)
  X, y, w = _data(case, g)
  mode, Hm = _newton_point(X, y, w)
  dg = Hm.diagonal().sqrt()
  norm = (mode, dg.clone(), torch.zeros_like(mode), dg.clone())
  flat = _sur_net(case['D'], case['H'], g, -Hm / dg[:, None] / dg[None, :])
  C, D, T = case['C'], case['D'], case['T']
  W0 = mode + _randn(g, C, D) / dg
  r0 = _randn(g, T, C, D)
  u = 2e-4 * torch.rand(T, C, generator=g, device=_DEV, dtype=torch.float64) + 1e-12
  return X, y, norm, flat, W0, r0, u


def _pairs(P, D, g):
  """(position, gradient) pairs like recorded ones: correlated positions a
  posterior width around a mode, gradients linear in them with a cubic bend."""
  sd = 0.002 * (0.5 + torch.rand(D, generator=g, device=_DEV))
  mode = 0.1 * _randn(g, D)
  mix = torch.eye(D, device=_DEV) + 0.2 * _randn(g, D, D) / math.sqrt(D)
  x = _randn(g, P, D) @ mix
  gr = -(x + 0.02 * x ** 3) / sd + 0.05 * _randn(g, P, D) / sd
  return mode + x * sd, gr


def _hier_inputs(case, seed):
  G, D, C = case['G'], case['D'], case['C']
  rng = np.random.default_rng(seed)
  sizes = 1 + rng.poisson(case['mean'], size=G)
  offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
  N = int(offsets[-1])
  g = _gen(seed)
  X = _randn(g, N, D)
  group = torch.as_tensor(np.repeat(np.arange(G), sizes), device=_DEV)
  ls = -0.5
  a = 0.3 + math.exp(ls) * _randn(g, G)
  w = 0.5 * _randn(g, D)
  y = (torch.rand(N, generator=g, device=_DEV) < torch.sigmoid(a[group] + X @ w)).float()
  truth = torch.cat([a, torch.tensor([0.3, ls], device=_DEV), w])
  theta = truth + 0.5 * (0.2 * N) ** -0.5 * _randn(g, C, G + 2 + D)
  r0 = _randn(g, C, G + 2 + D)
  u = 2e-4 * torch.rand(C, generator=g, device=_DEV, dtype=torch.float64) + 1e-12
  return X, y, offsets, group, theta, r0, u


def _hier_eps(case):
  return float(np.float32(0.4 / math.sqrt(case['G'] * (case['mean'] + 1.0))))


def _store(case, seed):
  """AR(1) chains with coordinate-wise correlations and spread-out means."""
  g = _gen(seed)
  T, C, D = case['T'], case['C'], case['D']
  rho = 0.9 * torch.rand(D, generator=g, device=_DEV)
  s = _randn(g, T, C, D)
  s[1:] *= torch.sqrt(1.0 - rho ** 2)
  for t in range(1, T):
    s[t].addcmul_(s[t - 1], rho.expand(C, D))
  s += 0.1 * _randn(g, 1, C, D) + _randn(g, D)
  return s


def prepare(case, seed):
  kind = case['kind']
  st = dict(case=case)
  if kind in ('run', 'chains'):
    g = _gen(seed)
    X, y, w = _data(case, g)
    st['eng'] = GLMEngine(X, y, likelihood=case['lik'], precision=case['precision'])
    st['W0'], st['r0'], st['u'] = _starts(case, g, w)
    st['eps'] = _eps(case)
    st['seed'] = int(seed) & 0xffff
  elif kind == 'sur_sample':
    X, y, norm, flat, st['W0'], st['r0'], st['u'] = _sur_inputs(case, seed)
    st['eng'] = GLMEngine(X, y, precision='bf16')
    st['sur'] = Surrogate(st['eng'], hidden=case['H'], max_batch=case['C'])
    st['sur'].set_params(flat)
    st['sur'].set_normalisation(*norm)
    st['eps'] = _eps(case)
  elif kind in ('sur_start', 'sur_grad'):
    g = _gen(seed)
    D, n = case['D'], case['P'] if kind == 'sur_start' else case['B']
    st['W'], st['G'] = _pairs(n, D, g)
    flat = _sur_net(D, case['H'], g)
    st['eng'] = GLMEngine(_randn(g, 512, D), torch.ones(512, device=_DEV), precision='bf16')
    st['sur'] = Surrogate(st['eng'], hidden=case['H'], max_batch=min(n, 4096))
    st['sur'].set_params(flat)
    if kind == 'sur_grad':
      st['sur'].normalise_from(st['W'], st['G'])
  elif kind == 'hier':
    X, y, off, _, st['theta'], st['r0'], st['u'] = _hier_inputs(case, seed)
    st['eng'] = HierEngine(X, y, off)
    st['eps'] = _hier_eps(case)
  elif kind in ('predict', 'newton'):
    g = _gen(seed)
    X, y, w = _data(case, g)
    st['eng'] = GLMEngine(X, y, likelihood=case['lik'], precision=case['precision'])
    if kind == 'predict':
      st['W'] = w + _width(case) * _randn(g, case['S'], case['D'])
    else:
      st['w'] = (w + _width(case) * _randn(g, case['D'])).cpu().numpy()
  else:
    st['eng'] = Context()
    st['s'] = _store(case, seed)
  torch.cuda.synchronize()
  return st


# -- the calls -----------------------------------------------------------------

def run(st):
  case = st['case']
  kind = case['kind']
  eng = st['eng']
  if kind == 'run':
    params = torch.empty(case['T'], case['C'], case['D'], device=_DEV)
    acc = torch.zeros(case['C'], dtype=torch.int32, device=_DEV)
    eng.set_state(st['W0'])
    eng.run(params, st['eps'], case['L'], seed=st['seed'], n_accept=acc)
    return dict(params=params, n_accept=acc)
  if kind == 'chains':
    sample = torch.empty(case['C'], case['D'], device=_DEV)
    acc = torch.empty(case['C'], dtype=torch.int32, device=_DEV)
    eng.set_state(st['W0'])
    eng.transition(st['eps'], case['L'], momenta=st['r0'], uniforms=st['u'], sample_out=sample,
                   accepted_out=acc)
    _, logp, grad = eng.get_state()
    return dict(sample=sample, accepted=acc, ratio=eng.last_ratio(), logp=logp, grad=grad)
  if kind == 'sur_sample':
    T = case['T']
    samples = torch.empty(T, case['C'], case['D'], device=_DEV)
    acc = torch.zeros(case['C'], dtype=torch.int32, device=_DEV)
    eng.set_state(st['W0'])
    for t in range(T):
      st['sur'].transition(st['eps'], case['L'], momenta=st['r0'][t], uniforms=st['u'][t],
                           sample_out=samples[t], n_accept=acc)
    return dict(samples=samples, n_accept=acc, ratio=eng.last_ratio())
  if kind == 'sur_start':
    st['sur'].normalise_from(st['W'], st['G'])
    st['sur'].init_skip_least_squares(st['W'], st['G'])
    return st['sur'].get_params()
  if kind == 'sur_grad':
    return st['sur'].loss_grad(st['W'], st['G'])
  if kind == 'hier':
    theta = torch.empty(case['C'], eng.dim, device=_DEV)
    acc = torch.empty(case['C'], dtype=torch.int32, device=_DEV)
    eng.set_state(st['theta'])
    eng.transition(st['eps'], case['L'], momenta=st['r0'], uniforms=st['u'], sample_out=theta,
                   accepted_out=acc)
    return dict(theta=theta, accepted=acc, ratio=eng.last_ratio())
  if kind == 'predict':
    mean, loglik, _ = eng.predict(st['W'])
    return mean, loglik
  if kind == 'newton':
    return eng.newton_terms(st['w'])
  ess = diagnostics.ess(eng, st['s'])
  mean, var = readout.empirical_moments(st['s'])
  return ess, mean, var


# -- work ----------------------------------------------------------------------

def work(case):
  kind = case['kind']
  if kind in ('run', 'chains'):
    N, D, C = case['N'], case['D'], case['C']
    evals = case.get('T', 1) * case['L'] + 1
    x = N * D * (2 if case['precision'] == 'bf16' else 4)
    out = case.get('T', 1) * C * D * 4
    return dict(bytes=(x + 4 * N) * (evals if x > _LLC else 1) + 12 * C * D + out,
                flops=4.0 * N * D * C * evals)
  if kind == 'sur_sample':
    N, D, C, H, T = case['N'], case['D'], case['C'], case['H'], case['T']
    x = N * D * 2 + 4 * N
    net = 2.0 * (H * D + H * H + D * (H + D))
    return dict(bytes=x * (T + 1 if x > _LLC else 1) + 8 * C * D * (T + 1),
                flops=2.0 * N * D * C * (T + 2) + C * net * (T * case['L'] + 1))
  if kind == 'sur_start':
    P, D, H = case['P'], case['D'], case['H']
    n = min(P, 32768)
    return dict(bytes=2 * P * D * 4 + 4 * (H * D + H * H + D * (H + D)),
                flops=8.0 * P * D + 4.0 * n * D * D + 2.0 / 3 * D ** 3)
  if kind == 'sur_grad':
    B, D, H = case['B'], case['D'], case['H']
    n = H * D + H * H + D * (H + D)
    return dict(bytes=2 * B * D * 4 + 2 * 4 * n, flops=6.0 * B * n - 2.0 * B * (H * D + D * D))
  if kind == 'hier':
    N, D, C = case['G'] * (case['mean'] + 1), case['D'], case['C']
    x = N * D * 4
    return dict(bytes=(x + 8 * N) * (case['L'] + 1 if x > _LLC else 1)
                + 3 * 4 * C * (case['G'] + 2 + D),
                flops=(4.0 * N * D * C + 2.0 * N * C) * (case['L'] + 1))
  if kind == 'predict':
    N, D, S = case['N'], case['D'], case['S']
    return dict(bytes=N * D * (2 if case['precision'] == 'bf16' else 4) + 8 * N + 4 * S * D,
                flops=2.0 * N * D * S)
  if kind == 'newton':
    N, D = case['N'], case['D']
    return dict(bytes=N * D * (2 if case['precision'] == 'bf16' else 4) + 4 * N + 8 * D * D,
                flops=1.0 * N * D * D + 4.0 * N * D)
  T, C, D = case['T'], case['C'], case['D']
  return dict(bytes=4 * T * C * D + 16 * C * D,
              flops=(2.0 * min(65, T) + 6.0) * T * C * D)


# -- exact values --------------------------------------------------------------

def _glm_terms(case, X, y, W, grad=True):
  """Log joint [C] and gradient [C, D] in float64; standard normal prior."""
  C, D = W.shape
  lp = -0.5 * (W * W).sum(1) - 0.5 * D * math.log(2 * math.pi)
  g = -W.clone() if grad else None
  for s in range(0, X.shape[0], _CHUNK):
    x = X[s:s + _CHUNK].double()
    yv = y[s:s + _CHUNK].double()
    eta = W @ x.t()
    if case.get('lik', 'bernoulli') == 'bernoulli':
      lp += (yv * eta - torch.nn.functional.softplus(eta, threshold=800.0)).sum(1)
      if grad:
        g += (yv - torch.sigmoid(eta)) @ x
    else:
      lp += (-0.5 * (yv - eta) ** 2).sum(1) - 0.5 * yv.numel() * math.log(2 * math.pi)
      if grad:
        g += (yv - eta) @ x
  return lp, g


def _hmc(terms, z, lp, g, r, u, eps, L, force=None):
  """One transition; terms(z) -> (log joint, gradient), or with ``force``
  the leapfrog follows force(z) and terms only weighs the end point."""
  z0, lp0, g0 = z, lp, g
  k0 = 0.5 * (r * r).sum(1)
  for k in range(L):
    r = r + 0.5 * eps * g
    z = z + eps * r
    if force is None:
      lp, g = terms(z)
    else:
      g = force(z)
    r = r + 0.5 * eps * g
  if force is not None:
    lp, _ = terms(z)
  ratio = k0 - 0.5 * (r * r).sum(1) + lp - lp0
  acc = torch.log(u) < ratio
  sel = acc[:, None]
  return (torch.where(sel, z, z0), torch.where(acc, lp, lp0), torch.where(sel, g, g0), ratio,
          acc)


def _philox(seed, counter, a, chain, stream):
  """Philox4x32-10 (Salmon et al. 2011) words of counters (a, chain, counter
  low, counter high | stream << 31); a and chain are uint64 arrays."""
  mask = np.uint64(0xffffffff)
  c = [np.asarray(a, np.uint64), np.asarray(chain, np.uint64),
       np.uint64(counter & 0xffffffff) + np.zeros_like(a),
       np.uint64(((counter >> 32) & 0x7fffffff) | (0x80000000 if stream else 0))
       + np.zeros_like(a)]
  k0, k1 = seed & 0xffffffff, seed >> 32
  for _ in range(10):
    p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
    c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & mask,
         (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & mask]
    k0, k1 = (k0 + 0x9E3779B9) & 0xffffffff, (k1 + 0xBB67AE85) & 0xffffffff
  return c


def _momenta(seed, t, C, D):
  nb = (D + 3) // 4
  ch, j = np.meshgrid(np.arange(C, dtype=np.uint64), np.arange(nb, dtype=np.uint64),
                      indexing='ij')
  x = _philox(seed, t, j, ch, 0)
  out = np.empty((C, nb, 4))
  for h in (0, 1):
    u1 = ((x[2 * h] >> np.uint64(8)).astype(np.float64) + 1.0) * 2.0 ** -24
    th = (x[2 * h + 1] >> np.uint64(8)).astype(np.float64) * (2.0 ** -24 * 2 * math.pi)
    rad = np.sqrt(-2.0 * np.log(u1))
    out[:, :, 2 * h] = rad * np.cos(th)
    out[:, :, 2 * h + 1] = rad * np.sin(th)
  return torch.as_tensor(out.reshape(C, 4 * nb)[:, :D].copy(), device=_DEV)


def _uniforms(seed, t, C):
  ch = np.arange(C, dtype=np.uint64)
  x = _philox(seed, t, np.zeros_like(ch), ch, 1)
  m = (x[0] << np.uint64(21)) | (x[1] >> np.uint64(11))
  return torch.as_tensor(m.astype(np.float64) * 2.0 ** -53, device=_DEV)


def _net_parts(flat, D, H):
  sizes = [H * D, H, H * H, H, D * (H + D), D]
  W1, b1, W2, b2, W3, b3 = torch.split(flat.double(), sizes)
  return W1.view(H, D), b1, W2.view(H, H), b2, W3.view(D, H + D), b3


def _net(parts, x):
  W1, b1, W2, b2, W3, b3 = parts
  gelu = lambda a: torch.nn.functional.gelu(a, approximate='tanh')
  h = gelu(x @ W1.t() + b1)
  h = gelu(h @ W2.t() + b2)
  return torch.cat([h, x], 1) @ W3.t() + b3


def _col_stats(W):
  n = W.shape[0]
  m = sum(W[s:s + _CHUNK].double().sum(0) for s in range(0, n, _CHUNK)) / n
  v = sum(((W[s:s + _CHUNK].double() - m) ** 2).sum(0) for s in range(0, n, _CHUNK)) / n
  return m, v.sqrt()


def _hier_terms(X, y, offsets, group, th, G):
  C, D = th.shape[0], X.shape[1]
  a, mu, ls, w = th[:, :G], th[:, G], th[:, G + 1], th[:, G + 2:]
  h = 0.5 * math.log(2 * math.pi)
  z = (a - mu[:, None]) * torch.exp(-ls)[:, None]
  lp = ((-0.5 * z * z - ls[:, None] - h).sum(1) - 0.5 * mu ** 2 - h - 0.5 * ls ** 2 - h
        - 0.5 * (w * w).sum(1) - D * h)
  ga = -z * torch.exp(-ls)[:, None]
  gmu = -ga.sum(1) - mu
  gls = (z * z).sum(1) - G - ls
  gw = -w.clone()
  off = torch.as_tensor(offsets, device=_DEV)
  for s in range(0, X.shape[0], _CHUNK):
    x, yv = X[s:s + _CHUNK].double(), y[s:s + _CHUNK].double()
    eta = a[:, group[s:s + _CHUNK]] + w @ x.t()
    lp = lp + (yv * eta - torch.nn.functional.softplus(eta, threshold=800.0)).sum(1)
    r = yv - torch.sigmoid(eta)
    gw = gw + r @ x
    cs = torch.nn.functional.pad(r.cumsum(1), (1, 0))
    o = (off - s).clamp(0, x.shape[0])
    ga = ga + cs[:, o[1:]] - cs[:, o[:-1]]
  return lp, torch.cat([ga, gmu[:, None], gls[:, None], gw], 1)


def exact(case, seed):
  kind = case['kind']
  if kind in ('run', 'chains'):
    g = _gen(seed)
    X, y, w = _data(case, g)
    W0, r0, u = _starts(case, g, w)
    terms = lambda q: _glm_terms(case, X, y, q)
    z = W0.double()
    lp, gr = terms(z)
    if kind == 'chains':
      z, lp, gr, ratio, acc = _hmc(terms, z, lp, gr, r0.double(), u, _eps(case), case['L'])
      # in bf16 a chain's own trajectory, and with it the small ratio of two
      # log joints, differs from the exact trajectory's by its rounding
      return dict(sample=z, accepted=acc.int(),
                  ratio=ratio if case['precision'] == 'fp32' else None, logp=lp, grad=gr)
    rows, n = [], 0
    s = int(seed) & 0xffff
    for t in range(case['T']):
      z, lp, gr, _, acc = _hmc(terms, z, lp, gr, _momenta(s, t, case['C'], case['D']),
                               _uniforms(s, t, case['C']), _eps(case), case['L'])
      rows.append(z)
      n = n + acc.int()
    return dict(params=torch.stack(rows), n_accept=n)
  if kind == 'sur_sample':
    X, y, norm, flat, W0, r0, u = _sur_inputs(case, seed)
    mode, isc, _, osc = [v.double() for v in norm]
    parts = _net_parts(flat, case['D'], case['H'])
    force = lambda q: _net(parts, (q - mode) * isc) * osc
    terms = lambda q: _glm_terms(case, X, y, q, grad=False)
    z = W0.double()
    lp, _ = terms(z)
    gr = force(z)
    rows, n = [], 0
    for t in range(case['T']):
      z, lp, gr, ratio, acc = _hmc(terms, z, lp, gr, r0[t].double(), u[t], _eps(case),
                                   case['L'], force)
      rows.append(z)
      n = n + acc.int()
    return dict(samples=torch.stack(rows), n_accept=n, ratio=None)
  if kind in ('sur_start', 'sur_grad'):
    g = _gen(seed)
    D, H = case['D'], case['H']
    W, G = _pairs(case['P'] if kind == 'sur_start' else case['B'], D, g)
    flat = _sur_net(D, H, g)
    (wm, ws), (gm, gs) = _col_stats(W), _col_stats(G)
    if kind == 'sur_start':
      sel = np.linspace(0, W.shape[0] - 1, min(W.shape[0], 32768)).astype(np.int64)
      x = (W[torch.as_tensor(sel, device=_DEV)].double() - wm) / ws
      t = (G[torch.as_tensor(sel, device=_DEV)].double() - gm) / gs
      A = torch.linalg.solve(x.t() @ x + 1e-6 * len(sel) * torch.eye(D, device=_DEV).double(),
                             x.t() @ t)
      out = flat.double().clone()
      o3 = H * D + H + H * H + H
      out[o3:o3 + D * (H + D)].view(D, H + D)[:, H:] = A.t()
      out[o3 + D * (H + D):] = 0.0
      return out
    p = flat.double().requires_grad_(True)
    o = _net(_net_parts(p, D, H), (W.double() - wm) / ws)
    loss = ((o - (G.double() - gm) / gs) ** 2).mean()
    loss.backward()
    return loss.detach().reshape(1), p.grad
  if kind == 'hier':
    X, y, off, group, th, r0, u = _hier_inputs(case, seed)
    terms = lambda q: _hier_terms(X, y, off, group, q, case['G'])
    z = th.double()
    lp, gr = terms(z)
    z, _, _, ratio, acc = _hmc(terms, z, lp, gr, r0.double(), u, _hier_eps(case), case['L'])
    return dict(theta=z, accepted=acc.int(), ratio=ratio)
  if kind == 'predict':
    g = _gen(seed)
    X, y, w = _data(case, g)
    W = (w + _width(case) * _randn(g, case['S'], case['D'])).double()
    mean = torch.empty(case['N'], dtype=torch.float64, device=_DEV)
    ll = 0.0
    for s in range(0, case['N'], _CHUNK):
      eta = W @ X[s:s + _CHUNK].double().t()
      yv = y[s:s + _CHUNK].double()
      if case['lik'] == 'bernoulli':
        mean[s:s + _CHUNK] = torch.sigmoid(eta).mean(0)
        ll = ll + (yv * eta - torch.nn.functional.softplus(eta, threshold=800.0)).sum(1)
      else:
        mean[s:s + _CHUNK] = eta.mean(0)
        ll = ll + (-0.5 * (yv - eta) ** 2 - 0.5 * math.log(2 * math.pi)).sum(1)
    return mean, ll
  if kind == 'newton':
    g = _gen(seed)
    X, y, w = _data(case, g)
    D = case['D']
    q = (w + _width(case) * _randn(g, D)).double()
    lp, gr = _glm_terms(case, X, y, q[None])
    P = torch.eye(D, device=_DEV).double()
    for s in range(0, case['N'], _CHUNK):
      x = X[s:s + _CHUNK].double()
      p = torch.sigmoid(x @ q)
      v = p * (1 - p) if case['lik'] == 'bernoulli' else torch.ones_like(p)
      P += (x * v[:, None]).t() @ x
    return float(lp[0]), gr[0].cpu().numpy(), P.cpu().numpy()
  return _exact_readout(_store(case, seed))


def _exact_readout(s):
  """Multi-chain effective sample sizes (Gelman et al., BDA3, sec. 11.5, with
  Geyer's initial monotone sequence), means and variances per coordinate."""
  T, C, D = s.shape
  x = s.double()
  mean = x.mean(0)
  x -= mean
  var = (x * x).mean(0)
  m = mean.cpu().numpy()
  acov = []
  W = var.sum(0).cpu().numpy() / C * T / (T - 1.0)
  vp = W * (T - 1.0) / T + (m.var(axis=0, ddof=1) if C > 1 else 0.0)
  total, prev = np.zeros(D), np.full(D, np.inf)
  live = vp > 0
  k = 0
  while live.any() and 2 * k + 1 < T:
    pair = np.zeros(D)
    for lag in (2 * k, 2 * k + 1):
      a = sum((x[i:min(i + 128, T - lag)] * x[i + lag:min(i + 128, T - lag) + lag]).sum((0, 1))
              for i in range(0, T - lag, 128)) / T
      pair += 1.0 if lag == 0 else 1.0 - (W - a.cpu().numpy() / C) / vp
    live = live & (pair > 0)
    pair = np.minimum(pair, prev)
    total = np.where(live, total + pair, total)
    prev = pair
    k += 1
  tau = np.maximum(-1.0 + 2.0 * total, 1.0 / math.log10(C * T))
  return np.where(vp > 0, C * T / tau, 0.0), mean, var
