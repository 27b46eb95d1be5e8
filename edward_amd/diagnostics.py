"""Effective sample size from device sample stores (no reference counterpart:
Edward reports only the acceptance rate, ``monte_carlo.py:152-158``).

The lag sums run on the GPU (``edhmc_autocov``); the truncation is done here.
``between=True`` (the default) is the multi-chain estimator of Gelman et al.
(BDA3, sec. 11.5): rho_t = 1 - (W - mean_m acov_m(t)) / var+, with var+ the
within-chain variance plus the spread of the chain means, summed with Geyer's
(1992) initial positive, monotone sequence, tau floored at 1/log10(M n),
ESS = M n / tau.  ``between=False`` leaves the spread of the chain means out,
so it credits only what the transitions themselves decorrelate: chains that
never move score 0 even when their starting points are spread over the
posterior."""

import math

import numpy as np
import torch

from edward_amd import _lib as L


_ALL_LAGS = 2048   # draws up to which edhmc_autocov sums every lag at once


def autocov(engine, samples, max_lag):
  """Sum over chains of each chain's biased autocovariance at lags
  0..max_lag, [max_lag+1, D] fp64, plus chain means [C, D]."""
  s = samples.contiguous()
  T, C, D = s.shape
  max_lag = int(min(max_lag, T - 1))
  acov = torch.empty(max_lag + 1, D, dtype=torch.float64, device=s.device)
  cmean = torch.empty(C, D, dtype=torch.float64, device=s.device)
  engine.check(engine.lib.edhmc_autocov(engine.h, L.ptr(s), T, C, D, max_lag, L.ptr(acov),
                                        L.ptr(cmean), engine.stream))
  return acov, cmean


def autocov_lags(engine, samples, lag0, n_lags, chain_means):
  """The sums of :func:`autocov` at lags lag0 .. lag0 + n_lags - 1 only,
  [n_lags, D] fp64, from the chain means it returned."""
  s = samples.contiguous()
  T, C, D = s.shape
  acov = torch.empty(n_lags, D, dtype=torch.float64, device=s.device)
  engine.check(engine.lib.edhmc_autocov_lags(engine.h, L.ptr(s), T, C, D, int(lag0), int(n_lags),
                                             L.ptr(chain_means), L.ptr(acov), engine.stream))
  return acov


def ess_from_acov(acov_sum, chain_means, n, between=False):
  """ESS per coordinate from summed autocovariances [lags, D] and chain means
  [M, D] of n draws per chain."""
  chain_means = np.asarray(chain_means, np.float64)
  M = chain_means.shape[0]
  spread = chain_means.var(axis=0, ddof=1) if between and M > 1 else 0.0
  return _ess_from_spread(np.asarray(acov_sum, np.float64), spread, M, n)


def _ess_from_spread(acov_sum, spread, M, n):
  """:func:`ess_from_acov` from the variance of the chain means over the
  chains (0 where the spread is left out)."""
  lags, D = acov_sum.shape
  acov_mean = acov_sum / M
  W = acov_mean[0] * n / (n - 1.0)
  var_plus = W * (n - 1.0) / n + spread
  moved = var_plus > 0               # no movement: nothing was sampled
  rho = 1.0 - (W - acov_mean) / np.where(moved, var_plus, 1.0)
  rho[0] = 1.0
  pairs = lags // 2
  p = rho[0:2 * pairs:2] + rho[1:2 * pairs:2]
  # Geyer's initial sequence: the pairs before the first that is not
  # positive, made non-increasing
  stop = np.concatenate([p <= 0, np.ones((1, D), bool)])
  k = stop.argmax(axis=0)
  truncated = k < pairs
  total = np.zeros((pairs + 1, D))
  np.cumsum(np.minimum.accumulate(p, axis=0), axis=0, out=total[1:])
  tau = np.maximum(-1.0 + 2.0 * total[k, np.arange(D)], 1.0 / math.log10(M * n))
  out = np.where(moved, M * n / tau, 0.0)
  if lags < n:                       # lag window too short: caller widens it
    out[moved & ~truncated] = np.nan
  return out


def ess(engine, samples, max_lag=64, between=True):
  """Per-coordinate ESS of samples [T, C, D] (device, fp32).  Up to 2048
  draws all lags come from one transform per pair of chains and are summed
  on the device (``edhmc_ess``); beyond, the lag window doubles until every
  coordinate's Geyer sequence is truncated (each lag is summed once)."""
  T, M, D = (int(v) for v in samples.shape)
  if T < 4:
    return np.full(D, np.nan)   # too few draws to estimate
  s = samples.contiguous()
  if T <= _ALL_LAGS:
    out = torch.empty(D, dtype=torch.float64, device=s.device)
    engine.check(engine.lib.edhmc_ess(engine.h, L.ptr(s), T, M, D, int(bool(between)), L.ptr(out),
                                      engine.stream))
    return out.cpu().numpy()
  lag = min(max_lag, T - 1)
  acov, cmean = autocov(engine, s, lag)
  acov = acov.cpu().numpy()
  spread = cmean.cpu().numpy().var(axis=0, ddof=1) if between and M > 1 else 0.0
  while True:
    e = _ess_from_spread(acov, spread, M, T)
    if not np.any(np.isnan(e)) or lag >= T - 1:
      return np.where(np.isnan(e), 0.0, e)
    wider = min(2 * lag + 1, T - 1)
    more = autocov_lags(engine, s, lag + 1, wider - lag, cmean)
    acov = np.concatenate([acov, more.cpu().numpy()])
    lag = wider


def min_ess(engine, samples, max_lag=64, between=True):
  return float(np.min(ess(engine, samples, max_lag, between)))
