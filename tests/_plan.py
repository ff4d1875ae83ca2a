"""The decode launch plan (csrc/p1a_plan.hpp, host arithmetic) as a function: compiled by itself, no library and no GPU."""
import ctypes
import functools
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FIELDS = ("mfma", "NW", "NT", "RG", "nsplit", "sb", "list", "loop", "RPS", "GPS", "x", "y", "direct", "deal_sh")
SHIM = '''
#include <cstring>
#include "p1a_plan.hpp"
extern "C" void plan(uint32_t type, int Hq, int Hkv, int D, int n_ctx, int T, int rows_per_seq, int pos_rows, int nsplit_req, int cus, int host_n, int partials, long long * o) {
    p1a_kv c;
    memset(&c, 0, sizeof c);
    c.type = type; c.Hkv = Hkv; c.D = D; c.n_ctx = n_ctx; c.k = c.v = (void *) 4096;
    const int rps = rows_per_seq < 1 ? 1 : rows_per_seq;
    int rg = p1a::make_plan(c, Hq, pos_rows ? rps : T, 0, 256).RG;
    while (pos_rows && rps > 1 && rps % rg) --rg;             // (as decode_call does)
    p1a::dec_plan p = p1a::make_plan(c, Hq, rg, nsplit_req, cus);
    p.RG = rg;
    p1a::finish_plan(p);
    const p1a::decode_grid g = p1a::plan_grid(p, type, D, Hkv, n_ctx, T, pos_rows ? rps : 1 << 30, pos_rows, cus, host_n, partials);
    const long long v[] = {p.mfma, p.NW, p.NT, p.RG, p.nsplit, g.sb, g.list, g.loop, g.RPS, g.GPS, g.x, g.y, g.direct, g.deal_sh};
    memcpy(o, v, sizeof v);
}
'''


@functools.lru_cache(maxsize=1)
def _lib():
    d = tempfile.mkdtemp(prefix="p1a_plan_")
    with open(os.path.join(d, "plan.cpp"), "w") as f:
        f.write(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "p100e-engine_amd", "csrc"),
                    os.path.join(d, "plan.cpp"), "-o", os.path.join(d, "plan.so")], check=True, capture_output=True, timeout=100)
    L = ctypes.CDLL(os.path.join(d, "plan.so"))
    L.plan.argtypes = [ctypes.c_uint32] + [ctypes.c_int] * 11 + [ctypes.POINTER(ctypes.c_longlong)]
    L.plan.restype = None
    return L


def plan(kv_type, Hq, Hkv, D, n_ctx, T, rows_per_seq=1, pos_rows=True, nsplit=0, cus=256, host_n=0, partials=False):
    """a cache whose memory is aligned, on a device of `cus` compute units -> {field: number}; host_n: positions seen where the call
    says them, partials: a call that leaves them unmerged"""
    o = (ctypes.c_longlong * len(FIELDS))()
    _lib().plan(kv_type, Hq, Hkv, D, n_ctx, T, rows_per_seq, pos_rows, nsplit, cus, host_n, partials, o)
    return dict(zip(FIELDS, o))
