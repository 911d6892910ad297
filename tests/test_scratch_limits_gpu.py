"""Calls at the limit of device memory: where a faster form wants more scratch memory than can be
had, the call takes the form that needs less and gives the same results.

A shared object whose hipMalloc fails past a budget of live bytes is loaded ahead of the library
in a child process (symbol lookup finds it first); no memory is really used up.
"""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>

static int (*real_malloc)(void**, size_t);
static int (*real_free)(void*);
static size_t budget, live;       /* budget 0: none */
static struct { void* p; size_t n; } held[4096];

int shim_init(const char* hip) {
    void* h = dlopen(hip, RTLD_NOW | RTLD_NOLOAD);
    if (!h) return -1;
    real_malloc = (int (*)(void**, size_t))dlsym(h, "hipMalloc");
    real_free = (int (*)(void*))dlsym(h, "hipFree");
    return real_malloc && real_free ? 0 : -2;
}
void shim_budget(size_t n) { budget = n; live = 0; for (int i = 0; i < 4096; ++i) held[i].p = 0; }
size_t shim_live(void) { return live; }

int hipMalloc(void** p, size_t n) {
    if (budget && live + n > budget) return 2;  /* hipErrorOutOfMemory */
    const int rc = real_malloc(p, n);
    if (rc == 0 && budget)
        for (int i = 0; i < 4096; ++i)
            if (!held[i].p) {
                held[i].p = *p;
                held[i].n = n;
                live += n;
                break;
            }
    return rc;
}
int hipFree(void* p) {
    for (int i = 0; p && i < 4096; ++i)
        if (held[i].p == p) {
            held[i].p = 0;
            live -= held[i].n;
            break;
        }
    return real_free(p);
}
"""

PROLOGUE = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.shim_budget.argtypes = [ctypes.c_size_t]
shim.shim_live.restype = ctypes.c_size_t
import numpy as np
import torch
torch.zeros(1, device="cpu")
hip = [l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64.so" in l][0]
assert shim.shim_init(hip.encode()) == 0, hip
from cortexsdr_amd import _lib, encode, synth
from cortexsdr_amd._lib import CsdrError
torch.cuda.init()
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    so = d / "shim.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(d / "shim.c"), "-o", str(so), "-ldl"],
                   check=True)
    return so


def run(shim, body):
    r = subprocess.run([sys.executable, "-c", PROLOGUE + body, str(shim)], cwd=ROOT, text=True,
                       env=dict(os.environ, PYTHONPATH=ROOT), capture_output=True, timeout=100)
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0 and "OK" in r.stdout


def test_prefill_without_room_for_the_planes(shim):
    """The pass's fp32 buffers exactly: no room for the split form's planes. The scores are the
    split form's within 1e-4, as the forms of the passes are compared elsewhere. One byte less:
    an error, and the decoder still prefills once there is memory."""
    run(shim, r"""
from cortexsdr_amd.decoder import Decoder, DecoderSpec, synthetic_weights
H, F, kvw, n = 512, 2048, 128, 39
w = synthetic_weights(DecoderSpec(2, H, 8, 2, 64, F, 300, 64), n_atoms=128, nnz=8, seed=3, sigma=0.1)
prompt = ((np.arange(n + 1) * 7919 + 11) % 300).astype(np.int32)
dec = Decoder(w)
dec.prefill(prompt, 0.0, 0.0)
want = dec.logits()
dec.close()
need = 4 * (n * (3 * H + 2 * kvw + max(H, F) + 2 * F + 1) + F * H)
dec = Decoder(w)
dec.prefill(prompt[:1], 0.0, 0.0)      # no pass: everything but its buffers
shim.shim_budget(need - 1)
try:
    dec.prefill(prompt, 0.0, 0.0)
    raise SystemExit("prefilled in less memory than its buffers")
except CsdrError:
    pass
assert shim.shim_live() == 0
for budget in (need, 0):
    shim.shim_budget(budget)
    dec.prefill(prompt, 0.0, 0.0)
    got = dec.logits()
    assert np.linalg.norm(got - want) < 1e-4 * np.linalg.norm(want), budget
print("OK")
""")


COMPRESS = r"""
R, C, K, S, k, iters = 2048, 64, 512, 2, 3, %d
w = synth.normal(7, R * C, sigma=0.02).astype(np.float32).reshape(R, C)
def go():
    a = encode.compress(w, 1, C, K, S, k, ksvd_iters=iters)
    b, skipped = encode.hsda_build({"a": w, "b": w[:600]}, 1, C, K, S, k, ksvd_iters=iters)
    assert not skipped
    return a, b
want = go()
n = R + 600                       # the archive's pool is the larger of the two
codes = n * S * k
need = n * C * 4 + K * C * 4 + codes * 2                   # tiles, dictionary, codes
init = n * 8 + K * 12                                      # the initialisation's norms
refine = n * C * 4 + (K + 1) * 4 + codes * 12 + K * 9      # residuals, user lists, flags
shim.shim_budget(need + (refine if iters else init))
assert go() == want
assert shim.shim_live() == 0
print("OK")
"""


def test_compress_without_room_for_the_scores(shim):
    """Tiles, dictionary and codes, and no room for the Gram form's scores: the same bytes by
    projections, for a matrix and for an archive of two."""
    run(shim, COMPRESS % 0)


def test_refinement_in_the_memory_of_its_results(shim):
    """Two refinement passes in the tiles, dictionary, codes, residuals and user lists, the
    buffers that the passes cannot do without."""
    run(shim, COMPRESS % 2)
