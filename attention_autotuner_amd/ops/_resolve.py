"""Shared by the two operator front ends: pick the configuration to launch."""
import os

import torch

from ..autotuner import base_tunner, gfx950_space
from ..autotuner.runtime import Runtime

_PKG = os.path.normpath(os.path.join(os.path.dirname(os.path.abspath(__file__)), ".."))
DEFAULT_LOG_DIR = os.environ.get("AAT_LOG_DIR", os.path.join(_PKG, "logs"))


# Octaves (BaseTunner.nearest_cached) within which a tuned problem's entry is taken before a built-in default that looks at the
# whole problem (gfx950_space.covered_by_rule).
# Attention forward, random problems: entries up to 3 octaves away run within 1 % of what the rule picks, entries 4 ... 12
# octaves away are 9 % slower on the mean and up to 32 % (256-row blocks on 256 rows of 60 heads: 10.5 against 8.1 us).  The other
# operators' rules were compared with the best of five to eight shapes (1 to 4 % slower on the mean, gfx950_space.py), not with
# entries by distance; half the distance that is safe in the forward keeps an entry where it was tuned, one length or row count
# off by less than a factor of three.
NEAR_ENOUGH = 1.5


def tune_on_miss():
    """The reference tunes whenever its cache has no entry; set AAT_TUNE_ON_MISS=0 to launch the
    configuration tuned for the nearest problem of the same head sizes instead, or the built-in default
    where there is none (no compile storm on first use)."""
    return os.environ.get("AAT_TUNE_ON_MISS", "1") != "0"


def resolve(tuner, default_factory, near=None):
    """``near``: how far away (octaves) a tuned problem may be for its entry to be taken before the built-in default."""
    cfg = tuner.check_cache()
    if cfg is not None:
        return cfg
    if tune_on_miss():
        return tuner.tune(log_path=DEFAULT_LOG_DIR)
    return tuner.nearest_cached(near) or default_factory()


def planned(key, make_tuner, default_factory):
    """``(configuration, Runtime)`` for the problem ``key`` (operator, device type, batch, heads, lengths, head sizes, mask
    walk): resolved through a tuner the
    first time this process meets the problem and kept in the tuners' own memo, so that every later call costs one
    dictionary lookup instead of a tuner, a cache-file name and a library path (the reference reads its JSON cache,
    python/autotuner/base_tunner.py:197-206, and opens the library, python/autotuner/runtime.py:74-82, on every call;
    its README.md:113 lists "the performance of python interface?" as open)."""
    k = ("plan", base_tunner.DEFAULT_CACHE_DIR, tune_on_miss()) + key
    plan = base_tunner._memo.get(k)
    if plan is None:
        tuner = make_tuner()
        op, key_dim, head_dim = key[0].replace("_decay", ""), key[6], key[7]
        near = NEAR_ENOUGH if gfx950_space.covered_by_rule(op, key_dim, head_dim) else None
        if op == "attn" and gfx950_space.few_blocks_config(key_dim, head_dim, *key[2:6], key[8]) is not None:
            near = -1                                      # no other problem's entry
        cc = resolve(tuner, default_factory, near)
        plan = base_tunner._memo[k] = (cc, Runtime(tuner.arch, cc))
    return plan


class NoGraph:
    """Stands in for the autograd context when no input of a call requires a gradient: the operators then run their
    forward directly (an inference call skips the ~15 us a ``torch.autograd.Function.apply`` costs on the host)."""
    needs_input_grad = (False,) * 8

    def save_for_backward(self, *tensors):
        pass


def wants_graph(*tensors):
    return torch.is_grad_enabled() and any(t.requires_grad for t in tensors)
