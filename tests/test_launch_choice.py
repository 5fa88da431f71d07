"""Split choices of the fixed-split decode on the CPU: the host library runs in
a child process over a recording stand-in of the HIP runtime (no GPU, no
kernel), so every launch a call would make can be read back."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_HIP = r"""
#include <stddef.h>
#include <stdint.h>
#include <string.h>
static char names[1024][64];
static int n_fn;
int n_launch;
char name[16][64];
uint32_t grid[16][3];
uint32_t tps[16], max_splits[16];
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int d) { return 0; }
int hipMalloc(void **p, size_t n) { *p = (void *)0x100000; return 0; }
int hipFree(void *p) { return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { *v = 256; return 0; }
int hipGetSymbolAddress(void **p, const void *s) { *p = (void *)0x200000; return 0; }
int hipModuleLoad(void **m, const char *f) { *m = (void *)1; return 0; }
int hipModuleUnload(void *m) { return 0; }
int hipModuleGetFunction(void **f, void *m, const char *n) {
    if (n_fn == 1023) return 1;
    strncpy(names[++n_fn], n, 63);
    *f = (void *)(uintptr_t)n_fn;
    return 0;
}
int hipModuleLaunchKernel(void *f, unsigned x, unsigned y, unsigned z, unsigned bx, unsigned by,
                          unsigned bz, unsigned lds, void *stream, void **a, void **extra) {
    const int i = n_launch++ & 15;
    strcpy(name[i], names[(uintptr_t)f]);
    grid[i][0] = x, grid[i][1] = y, grid[i][2] = z;
    const int split = !strncmp(name[i], "eh_decode_rows", 14) || !strncmp(name[i], "eh_decode_split", 15);
    tps[i] = split ? *(uint32_t *)a[16] : 0, max_splits[i] = split ? *(uint32_t *)a[17] : 0;
    return 0;
}
"""

_CHILD = r"""
import ctypes as C, json, sys
sys.path.insert(0, sys.argv[2])
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
from titan_amd import _lib
L = _lib.load()
ctx = C.c_void_p()
assert L.eh_create(0, None, C.byref(ctx)) == 0
P = C.c_void_p(1 << 28)   # never dereferenced
n_launch = C.c_int.in_dll(hip, "n_launch")
names = ((C.c_char * 64) * 16).in_dll(hip, "name")
grids = ((C.c_uint32 * 3) * 16).in_dll(hip, "grid")
tps_of = (C.c_uint32 * 16).in_dll(hip, "tps")
splits_of = (C.c_uint32 * 16).in_dll(hip, "max_splits")

def launches():
    n, n_launch.value = n_launch.value, 0
    return [(names[i].value.decode(), list(grids[i]), tps_of[i], splits_of[i]) for i in range(n)]

out = []
for case in json.load(sys.stdin):
    dt, batch, nh, nkv, hd, bt, ctx_len, how = case
    elt = 4 if dt == 0 else 2
    pages = -(-ctx_len // bt)
    qb, pool = batch * nh * hd * 4, pages * bt * 2 * nkv * hd * elt
    if how.startswith("pool"):   # a pool of one page, less the named bytes
        pool, how = bt * 2 * nkv * hd * elt - int(how.split()[1]), how.split()[2]
    if how == "plan":
        t, m, w = C.c_uint32(), C.c_uint32(), C.c_uint64()
        st = L.eh_decode_plan(dt, batch, nh, nkv, hd, bt, ctx_len, 0, C.byref(t), C.byref(m), C.byref(w))
        if st == 0:
            st = L.eh_paged_decode_batched(ctx, None, dt, P, qb, P, pool, P, batch * pages * 4, pages, P,
                                           batch, P, qb, nh, nkv, hd, bt, t.value, m.value, P, w.value)
    elif how == "fused":    # device position, the table's capacity is ctx_len
        row = nkv * hd * elt
        st = L.eh_append_flash_decoding(ctx, None, dt, P, row, P, row, P, qb, P, pool, P, pages * 4, P, qb,
                                        nh, nkv, hd, bt, 100, P)
    else:                   # host position ctx_len - 1
        st = L.eh_flash_decoding(ctx, None, dt, P, qb, P, pool, P, pages * 4, P, qb, nh, nkv, hd, bt,
                                 ctx_len, ctx_len - 1, 1, None)
    name = C.create_string_buffer(64)
    assert L.eh_decode_kernel_name(dt, nh, nkv, hd, bt, name, 64) == 0
    out.append((st, launches(), name.value.decode()))
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    """cases [(dtype, batch, n_head, n_kv, head_dim, block_tokens, context, how)] -> [(status, launches,
    name of the batched split kernel)]."""
    d = tmp_path_factory.mktemp("hip")
    (d / "hip.c").write_text(_HIP)
    so = str(d / "hip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(d / "hip.c"), "-o", so], check=True)

    def run(cases):
        r = subprocess.run([sys.executable, "-c", _CHILD, so, ROOT], input=json.dumps(cases),
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout.strip().splitlines()[-1])
    return run


HEADS = ((14, 2), (32, 8), (32, 32), (64, 8), (64, 64), (12, 3))


@pytest.mark.parametrize("how", ["plan", "fused", "host"])
def test_splits_near_the_largest(choose, how):
    """Automatic splits that reach the largest one (1022 pages, in whole tiles) are
    accepted by the calls they are made for and cover the context, for every type,
    page size and head count; contexts where no rule holds it back are among them."""
    cases = []
    for dt in (0, 1, 3):  # f32, f16, bf16
        for hd in (64, 128):
            for nh, nkv in HEADS:
                for bt in (8, 16, 24, 32, 64):
                    most = 1022 * bt // 16 * 16  # no kernel's largest split is shorter
                    for ctx in (4096, 32768, 131072, 262144, 1 << 20):
                        if ctx <= 256 * most:
                            cases += [(dt, b, nh, nkv, hd, bt, ctx, how)
                                      for b in ((2, 16, 32, 128, 256) if how == "plan" else (1,))]
    at_limit = 0
    for case, (st, launches, _) in zip(cases, choose(cases)):
        assert st == 0, case
        name, _, tps, splits = launches[0]
        if not name.startswith(("eh_decode_rows", "eh_decode_split")):
            continue                             # token-balanced
        dt, bt, ctx = case[0], case[5], case[6]
        assert tps * splits >= ctx and splits <= 256, case
        tile = 16 if dt == 0 else 32
        largest = -(-1022 * bt // tile) * tile
        assert tps <= largest and (name.startswith("eh_decode_split") or tps % tile == 0), case
        at_limit += tps > largest - 4 * tile
    assert at_limit > 20


@pytest.mark.parametrize("how", ["fused", "host"])
def test_a_pool_below_one_page_is_refused(choose, how):
    """Masked keys read page 0, so a pool that holds no whole page launches nothing."""
    shapes = [(dt, 1, 14, 2, hd, 16, 500) for dt in (0, 1, 3) for hd in (32, 64, 128)]
    for st, launches, _ in choose([(*s, f"pool 1 {how}") for s in shapes]):
        assert st == 1 and launches == []
    for st, launches, _ in choose([(*s, f"pool 0 {how}") for s in shapes]):
        assert st == 0 and launches


def test_kernel_name_is_the_batched_launch(choose):
    """eh_decode_kernel_name names what a batch launches."""
    cases = [(dt, b, nh, nkv, hd, bt, 32768, "plan") for dt in (0, 1, 3) for hd in (32, 64, 128)
             for nh, nkv in HEADS for bt in (4, 8, 16, 24) for b in (2, 16)
             if b == 2 or (bt >= 8 and dt != 0)]   # (the length and number count for the others)
    for case, (st, launches, name) in zip(cases, choose(cases)):
        assert st == 0 and launches[0][0] == name, case


def test_kernel_by_page_size_and_heads(choose):
    """Pages under 8 tokens and up to 4 q heads per kv head: the per-token kernel from
    98304 tokens over the batch's kv heads on (196608 at 3 and 4 heads) and for fused
    steps up to 384; f32 batches at head_dim 64 with 1 or 2: from 131072 on; and back
    to the row kernels where the per-token kernel's largest split (992 tokens of
    pages of one) is too short."""
    def kernels(cases):
        return [launches[0][0].split("_hd")[0] for st, launches, _ in choose(cases) if st == 0]
    small, want = [], []
    for dt in (1, 3):
        for hd in (64, 128):
            for bt in (1, 2, 4):
                for g in (1, 2, 3, 4, 5, 16):
                    for ctx in (384, 23040, 25600, 46080, 51200):   # 4 kv heads; whole splits of either
                        small.append((dt, 2, 2 * g, 2, hd, bt, ctx, "plan"))
                        split = g <= 4 and 4 * ctx >= (98304 if g <= 2 else 196608)
                        want.append("eh_decode_" + ("split" if split else "rows") + ("_f16" if dt == 1 else "_bf16"))
    assert kernels(small) == want
    step = [(1, 1, 3 * g, 3, 64, 4, ctx, "fused") for g in (1, 2, 4, 5) for ctx in (384, 512, 49152, 81920)]
    names = ["split", "rows", "split", "split"] * 2 + ["split", "rows", "rows", "split"] + ["rows"] * 4
    assert kernels(step) == [f"eh_decode_{n}_f16" for n in names]
    f32 = [(0, b, nkv * g, nkv, 64, 16, ctx, "plan") for b, nkv, ctx in ((1, 64, 4096), (2, 32, 1024), (2, 32, 3072),
                                                                         (16, 4, 1792), (16, 4, 2304)) for g in (1, 2, 3)]
    want = ["eh_decode_" + ("split" if c[1] > 1 and c[1] * c[3] * c[6] >= 131072 and c[2] <= 2 * c[3] else "rows") + "_f32"
            for c in f32]
    assert kernels(f32) == want
    far = [(1, 1, 3, 3, 64, 1, ctx, how) for ctx in (256 * 992, 256 * 992 + 1) for how in ("fused", "host", "plan")]
    assert kernels(far) == ["eh_decode_split_f16"] * 3 + ["eh_decode_rows_f16"] * 3
