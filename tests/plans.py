"""The launches' plans (csrc/attn_plan.h) compiled for the host, so that tests can see which build runs and
how many workgroups share a tile."""

import ctypes
import functools
import os
import subprocess
import tempfile
from collections import namedtuple

import torch

from fa4_ring import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_SOURCE = """
#include "%s"
using namespace fa4cp;
static void put(const Shares& s, int* o) { o[0] = s.k; o[1] = s.k2; o[2] = s.chunk; o[3] = s.top2; o[4] = s.chunk2; }
extern "C" void split(const fa4cp_sweep_args* a, int* o) {
  const SplitPlan pl = split_plan(a);
  o[0] = pl.ns_back; o[1] = pl.ns_front; o[2] = pl.shares.chunk; o[3] = pl.n_front; o[4] = pl.n_row;
}
extern "C" int sweep_two(const fa4cp_sweep_args* a) { return sweep_two_per_cu(a); }
extern "C" int attn_two(const fa4cp_attn_args* a) { return attn_two_per_cu(a); }
extern "C" int shares(const int* s, int n) { return shares_of(s[0], s[2], s[3], s[4], n); }
extern "C" int turned(int i, int tile, int ns) { return turned_share(i, tile, ns); }
extern "C" void backward(const fa4cp_sweep_bwd_args* a, int* o) {
  const BwdPlan pl = bwd_plan(*a);
  put(pl.dq, o);
  put(pl.kv, o + 5);
}
"""

Split = namedtuple("Split", "back front chunk n_front n_row")  # workgroups per row tile, key tiles each; row tiles
Shares = namedtuple("Shares", "k k2 chunk top2 chunk2")        # as share_model.h


@functools.lru_cache(maxsize=None)
def _probe():
    with tempfile.TemporaryDirectory() as td:
        src, lib = os.path.join(td, "p.cpp"), os.path.join(td, "p.so")
        with open(src, "w") as f:
            f.write(_SOURCE % os.path.join(ROOT, "fa4-cp_amd", "csrc", "attn_plan.h"))
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", lib, src], check=True)
        return ctypes.CDLL(lib)


def _shape(a, lens, h, h_kv, d, cp, rank):
    a.total, a.h_q, a.h_kv, a.d, a.cp_rank, a.cp_size, a.nseq = sum(lens), h, h_kv, d, rank, cp, 1
    if len(lens) > 1:
        a.cu, a.nseq, a.max_seqlen = 1 << 20, len(lens), max(lens)  # (the plans look only at whether cu is NULL)
    return a


def sweep_args(lens, h, h_kv, d, cp, rank, dtype):
    a = _shape(_lib.SweepArgs(), lens, h, h_kv, d, cp, rank)
    a.dtype = _lib.dtype_code(dtype)
    return a


def split_plan(lens, h, h_kv, d, cp, rank, dtype):
    out = (ctypes.c_int * 5)()
    _probe().split(ctypes.byref(sweep_args(lens, h, h_kv, d, cp, rank, dtype)), out)
    return Split(*out)


def heads_per_wg(group):
    return 4 if group % 4 == 0 else 2 if group % 2 == 0 else 1


def sweep_two_per_cu(lens, h, h_kv, d):
    return bool(_probe().sweep_two(ctypes.byref(sweep_args(lens, h, h_kv, d, 4, 1, torch.bfloat16))))


def attn_two_per_cu(lens, h, h_kv, d, q_sel=0):
    a = _lib.AttnArgs()
    a.total_q, a.h_q, a.h_kv, a.d, a.nseq, a.q_sel = sum(lens), h, h_kv, d, 1, q_sel
    if len(lens) > 1:
        a.cu_q, a.nseq, a.max_seqlen_q = 1 << 20, len(lens), max(lens)
    return bool(_probe().attn_two(ctypes.byref(a)))


def backward_args(lens, h, h_kv, d, cp, rank):
    return _shape(_lib.SweepBwdArgs(), lens, h, h_kv, d, cp, rank)


def backward_plan(lens, h, h_kv, d, cp, rank):
    """(dq's, dk / dv's) Shares."""
    out = (ctypes.c_int * 10)()
    _probe().backward(ctypes.byref(backward_args(lens, h, h_kv, d, cp, rank)), out)
    return Shares(*out[:5]), Shares(*out[5:])


def shares_of(plan, n):
    """Workgroups that share a tile of n steps under a Shares plan."""
    return _probe().shares((ctypes.c_int * 5)(*plan), n)


def turned_share(i, tile, ns):
    return _probe().turned(i, tile, ns)
