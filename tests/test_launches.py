"""Which kernels a forward call launches, on the CPU: the built library runs against hip_recorder.c instead of the HIP
runtime. All launch shapes are bit-identical by design, so no output tells which of them ran."""
import json
import os
import re
import subprocess
import sys

import pytest

from conftest import PKG

DRIVER = r"""
import ctypes as C, json, sys
rec = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
rec.hip_recorder_log.restype = C.c_char_p
rec.hip_recorder_limit.argtypes = [C.c_size_t]
import _native
lib, job, h = _native.load(), json.load(sys.stdin), C.c_void_p()
_native.check(lib.gfl_ctx_create(0, C.byref(h)))
if job["limit"] is not None:
    rec.hip_recorder_limit(job["limit"])
E, H, I, Ks = job["layer"]
rc = lib.gfl_register_layer(h, 0, E, H, I, *Ks, (C.c_uint64 * (9 * E))(*[1 << 20] * (9 * E)))
out = [[rc, lib.gfl_last_error().decode(), ""]]
rec.hip_recorder_limit(C.c_size_t(-1).value)
lib.gfl_ctx_set_shared(h, job["shared"])
for M, topk, mode, offset in job["calls"]:
    rec.hip_recorder_clear()
    if mode == "grouped":
        rc = lib.gfl_grouped_forward(h, 0, 1 << 21, 1 << 22, 1 << 23, 1, M, topk, 1 << 24, 0.0, None)
    elif mode == "reserve":
        rc = lib.gfl_grouped_reserve(h, M * topk)
    else:
        rc = lib.gfl_moe_forward(h, 0, 1 << 21, 1 << 22, 1 << 23, 1, M, topk, (1 << 24) + offset, mode, 0.0, None)
    out.append([rc, lib.gfl_last_error().decode(), rec.hip_recorder_log().decode()])
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """launches(layer, calls, limit, env): [(rc, error, [kernel names])] of the registration and of each call
    (M, topk, mode, offset of out), on a context created with env and `limit` bytes of device memory left after that;
    launches.lds has each launch's dynamic LDS bytes."""
    import _native
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    so = str(tmp_path_factory.mktemp("rec") / "hip_recorder.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", so,
                    os.path.join(os.path.dirname(__file__), "hip_recorder.c")], check=True)

    def run(layer, calls, limit=None, env=(), shared=0):
        r = subprocess.run([sys.executable, "-c", DRIVER, so], capture_output=True, text=True,
                           input=json.dumps(dict(layer=layer, calls=calls, limit=limit, shared=shared)), env=dict(os.environ, PYTHONPATH=PKG, **dict(env)))
        assert r.returncode == 0, r.stderr[-2000:]
        got = json.loads(r.stdout.strip().split("\n")[-1])
        names = subprocess.run(["c++filt"], input="\n".join(g[2].replace("\n", " ") for g in got), capture_output=True,
                               text=True, check=True).stdout.split("\n")
        run.lds = [[int(v) for v in re.findall(r"\) (\d+)", n)] for n in names]
        return [(rc, err, re.findall(r"(?:gfl::)(\w+(?:<[^(]*>)?)\(", n)) for (rc, err, _), n in zip(got, names)]
    return run


EXACT, MFMA = 1, 3
B, S = (5120, 1536, (3, 3, 3)), (512, 256, (3, 3, 3))   # the benchmark's layer, the GPU tests' small one


@pytest.mark.parametrize("layer,call,env,first", [
    # the calls of tests/test_gpu_parity.py that name their launches
    ((108, *B), (16, 8, EXACT, 0), {}, "gp_plan"), ((169, *B), (32, 8, EXACT, 0), {}, "gp_plan"),
    ((249, *B), (64, 8, EXACT, 0), {}, "gp_plan"),
    ((288, *B), (16, 8, EXACT, 0), {}, "plan"), ((249, *B), (64, 8, EXACT, 4), {}, "plan"),
    ((32, *S), (128, 8, EXACT, 0), {}, "gp_plan"), ((32, *S), (128, 8, EXACT, 4), {}, "plan"),
    ((8, *S), (16, 8, EXACT, 0), {}, "gp_plan"), ((8, *S), (16, 8, EXACT, 4), {}, "plan"),
    ((20, 512, 256, (3, 4, 3)), (8, 16, EXACT, 0), {}, "gp_plan"),
    ((288, 512, 256, (3, 4, 3)), (8, 16, EXACT, 0), {}, "plan"),
    ((20, 512, 256, (3, 4, 3)), (8, 16, EXACT, 0), {"GFL_RELAY": "1,1"}, "plan"),
    ((6, *S), (12, 8, EXACT, 0), {"GFL_SLOTS_PER_PASS": "2"}, "plan"),
    # either side of each line: 64 picks; half a pick per expert, three quarters where gate and up differ; mode; 1,024 picks
    ((16, *S), (64, 1, EXACT, 0), {}, "gu"), ((16, *S), (8, 8, EXACT, 0), {}, "gu_relay"),
    ((16, *S), (65, 1, EXACT, 0), {}, "gp_plan"),
    ((130, *S), (65, 1, EXACT, 0), {}, "gp_plan"), ((131, *S), (65, 1, EXACT, 0), {}, "plan"),
    ((88, 512, 256, (3, 4, 3)), (66, 1, EXACT, 0), {}, "gp_plan"), ((89, 512, 256, (3, 4, 3)), (66, 1, EXACT, 0), {}, "plan"),
    ((16, *S), (65, 1, MFMA, 0), {}, "plan"),
    ((1024, *S), (1025, 1, EXACT, 0), {}, "gp_rank"), ((16, *S), (4, 16, "grouped", 0), {}, "gp_plan"),
])
def test_launch_choice(launches, layer, call, env, first):
    """The first kernel of a call: relay or per-slot / per-entry decode launches (plan_kernel above 64 picks), or the grouped
    plan of the chains and the grouped path."""
    (rc, err, _), (crc, cerr, names) = launches(layer, [call], env=env)
    assert (rc, err, crc, cerr) == (0, "", 0, "") and names[0].split("<")[0] == first + "_kernel", names


def test_registration_without_memory_for_the_chains(launches):
    """Room for the decode workspace (28 MB at H = 4096, I = 256) but not for the chains' (44 MB): the layer is registered
    and its calls run on the decode launches, none of them reporting the refused allocation; with memory they take the
    chains."""
    got = launches((8, 4096, 256, (3, 3, 3)), [(65, 1, EXACT, 0), (4, 4, EXACT, 0), (16, 16, "reserve", 0),
                                              (65, 1, EXACT, 0), (256, 1, EXACT, 0), (512, 1, EXACT, 0)], limit=40 << 20)
    assert [(rc, err) for rc, err, _ in got] == [(0, "")] * len(got)
    assert got[1][2] == ["plan_kernel", "gu_kernel<3, 4, false>", "down_kernel<3, 4, false>"]
    assert got[2][2] == ["gu_relay_kernel<3, 4>", "dn_relay_kernel<3, 1>"]
    for k, slots in ((4, 32), (5, 64)):
        assert got[k][2] == ["gp_plan_kernel", "gp_prep_kernel<true, false>", "xg_gemm_kernel<3, %d>" % slots,
                             "gp_act_kernel<true, 1>", "xg_gemm_kernel<3, %d>" % slots, "gp_comb_kernel"]
    assert got[6][2] == ["plan_kernel", "gu_kernel<3, 4, false>", "down_kernel<3, 4, false>"]   # beyond what was reserved


@pytest.mark.parametrize("Ks,M,slots", [
    ((3, 3, 3), 7, 16), ((3, 3, 3), 8, 32), ((3, 3, 3), 27, 32), ((3, 3, 3), 28, 64), ((5, 3, 4), 28, 64),
    ((3, 3, 5), 200, 64), ((5, 5, 5), 7, 16), ((5, 5, 2), 27, 32), ((5, 5, 2), 28, 32), ((5, 2, 5), 47, 32),
    ((4, 5, 5), 48, 64), ((5, 5, 5), 60, 32), ((5, 5, 5), 200, 32),
])
def test_chain_pass_sizes(launches, Ks, M, slots):
    """16, 32 and 64 slots per pass by picks per expert; with matrices of 5 bits, whose 64-slot pass leaves a CU one
    workgroup, 32 for longer. Calls within 1,024 picks and above take the same sizes."""
    for E in (16, 288):
        (rc, err, _), call = launches((E, 512, 256, Ks), [(M * E // 16, 16, EXACT, 0)])
        assert (rc, err, call[0], call[1]) == (0, "", 0, "")
        gemms = [n for n in call[2] if n.startswith("xg_gemm_kernel")]
        want = ["xg_gemm_kernel<%d, %d>" % (k, slots) for k in (Ks if Ks[0] != Ks[1] else Ks[1:])]
        assert gemms == want, call[2]


@pytest.mark.parametrize("layer,M,shared,per_cu", [
    (B, 2, 0, (3, 5)), (B, 3, 0, (5, 4)), (B, 4, 0, (6, 4)), (B, 8, 0, (4, 4)), (B, 2, 1, (3, 5)), (B, 4, 1, (4, 4)),
    ((4096, 2048, (3, 3, 3)), 3, 0, (6, 6)), ((4096, 2048, (3, 3, 3)), 4, 0, (4, 4)),
])
def test_relay_workgroups_per_cu(launches, layer, M, shared, per_cu):
    """The one-wave relay launches' LDS lets a CU (160 KB) hold the launch's share of workgroups where the registers take
    that many (6; on a context told of other work beside it 5), else 4."""
    _, (rc, err, names) = launches((288, *layer), [(M, 8, EXACT, 0)], shared=shared)
    assert (rc, err, names) == (0, "", ["gu_relay_kernel<3, 1>", "dn_relay_kernel<3, 1>"])
    assert tuple(163840 // lds for lds in launches.lds[1]) == per_cu
