"""Host paths of the library without a GPU: the HIP runtime is replaced by tests/cpp/host_hip.cpp,
which keeps device memory on the host under a limit and counts kernels instead of running them.
Each case runs in a process of its own, where the replacement is loaded before the library."""
import ctypes
import json
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
L16 = (16, 16, 16, 16)


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    so = str(tmp_path_factory.mktemp("host") / "host_hip.so")
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-w", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "cpp", "host_hip.cpp"), "-o", so], check=True, timeout=300)
    return so


# ---------------------------------------------------------------- the cases, in a process of their own

def check_memory(h, la, call):
    """A context that keeps a smearing buffer gives it back to the call that needs its memory."""
    ctx = la.Context(0)
    a, b = la.GaugeField(ctx, L16), la.GaugeField(ctx, L16)
    before = h.host_used()
    la.StoutSmearingN(a, b, 2, 0.12)
    kept = h.host_used() - before
    spare = 0
    if call == "scratch":
        run = lambda: la.TopChargeCloverDensity(a)
    elif call == "read_rate":
        run = lambda: ctx.read_rate(1 << 16)
    elif call == "tune_sweep":
        run, spare = lambda: a.autotune("sweep"), kept // 2
    elif call == "tune_flow":
        run, spare = lambda: a.autotune("flow"), 3 * kept // 2
    elif call == "update":
        run = lambda: la.UpdateSweeps(a, 6.0, 1, 1, 2)
    elif call == "checksum":
        run = lambda: a.bmw_checksum()
    h.host_limit(h.host_used() + spare)
    run()


def check_tune_sweep(h, la):
    """Tuning the sweeps sets the tile of the plaquette pass alone, tuning the flow that of the
    other link kernels; nothing comes to the host while the pass is timed."""
    ctx = la.Context(0)
    a, b = la.GaugeField(ctx, L16), la.GaugeField(ctx, L16)
    cache = os.path.join(os.path.dirname(sys.argv[1]), "tiles.json")

    def blocks():
        la.StoutSmearingN(a, b, 1, 0.12)
        la.PlaquetteSum(a)
        la.UpdateSweeps(a, 6.0, 1, 1, 1, 4)
        return [h.host_block(k) for k in (b"stout_kernel", b"upd_plaq_kernel", b"cb4_plaq_kernel")]

    assert blocks() == [128, 128, 128]
    with open(cache, "w") as f:
        json.dump({"gfx950|16x16x16x16|sweep": [2, 2, 4, 4, 1.0], "gfx950|16x16x16x16|flow": [1, 2, 16, 8, 1.0]}, f)
    assert a.autotune("sweep", cache)[0] == a.get_tile() == (2, 2, 4, 4)
    assert blocks() == [128, 64, 64]
    assert a.autotune("flow", cache)[0] == a.get_tile() == (1, 2, 16, 8)
    assert blocks() == [256, 64, 64]
    a.set_tile(1, 1, 8, 8)
    assert a.get_tile() == (1, 1, 8, 8) and blocks() == [64, 64, 64]
    n = h.host_copies_to_host()
    a.autotune("sweep")
    assert h.host_copies_to_host() == n


def check_batch_views(h, la):
    """Tuning a batch leaves the tiles of its replicas' fields alone: it tries only blocks of the
    batch's own size, the single-lattice kernels have another on large lattices."""
    b = la.ReplicaBatch(la.Context(0), [L16, (8, 8, 8, 8)], 2, 0.12)
    before = [b.field(r).get_tile() for r in range(2)]
    b.autotune()
    assert [b.field(r).get_tile() for r in range(2)] == before


def check_batch_cache(h, la):
    """A cached tile of more threads than the batch launches is not taken: its kernels would reach
    past the LDS of their block."""
    cache = os.path.join(os.path.dirname(sys.argv[1]), "batch.json")
    key = "gfx950|2x2x2x2|batch64"
    for entry in ([0, 0, 0, 128, 1.0], [0, 0, 0, 256, 1.0]):
        with open(cache, "w") as f:
            json.dump({key: entry}, f)
        b = la.ReplicaBatch(la.Context(0), [(2, 2, 2, 2)], 2, 0.12)
        b.autotune(cache)
        with open(cache) as f:
            tile = json.load(f)[key][:4]
        assert tile == [0, 0, 0, 64], tile


def check_momenta(h, la, call):
    """A trajectory that runs out of memory leaves its momenta as whole matrices, as one that ends:
    in the 8 reals that it keeps them in, a caller that goes on with them would read other ones."""
    ctx = la.Context(0)
    U, V, P, F = la.GaugeField(ctx, L16), la.GaugeField(ctx, L16), la.MatrixField(ctx, L16), la.MatrixField(ctx, L16)
    cv = la.CollectiveVariable(ctx, L16, 1, 0.12)
    bias = la.MetaBiasPotential(-8.0, 8.0, 80, 1.5, 0.3, 10.0, 1000.0, well_tempered=False)
    run = {"hmc": lambda: la.HMCKernel(U, V, P, "omf2", 6.0, 1.0)(2, False),
           "hmc_reversibility": lambda: la.HMCKernel(U, V, P, "omf2", 6.0, 1.0).ReversibilityTest(2),
           "metad": lambda: la.HMCMetaDKernel(U, V, P, F, bias, cv, "omf2", 6.0, 1.0)(2, False),
           "metad_reversibility": lambda: la.HMCMetaDKernel(U, V, P, F, bias, cv, "omf2", 6.0, 1.0).ReversibilityTest(2)}[call]
    h.host_limit(h.host_used())
    try:
        run()
    except la.LettuceError as e:
        assert "allocation failed" in str(e), e
    else:
        raise AssertionError("no scratch to be had, and no error")
    assert h.host_launches(b"15momentum_kernelILb1E") == 1 and h.host_launches(b"momentum_entry_kernelILb1E") == 1


CASES = {f"memory_{c}": (lambda h, la, c=c: check_memory(h, la, c))
         for c in ("scratch", "read_rate", "tune_sweep", "tune_flow", "update", "checksum")}
CASES.update({f"momenta_{c}": (lambda h, la, c=c: check_momenta(h, la, c))
              for c in ("hmc", "hmc_reversibility", "metad", "metad_reversibility")})
CASES["tune_sweep"] = check_tune_sweep
CASES["batch_views"] = check_batch_views
CASES["batch_cache"] = check_batch_cache


@pytest.mark.parametrize("case", sorted(CASES))
def test_host_path(host_hip, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), host_hip, case], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    h = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    h.host_used.restype = ctypes.c_size_t
    h.host_limit.argtypes = [ctypes.c_size_t]
    h.host_copies_to_host.restype = ctypes.c_long
    h.host_launches.restype = ctypes.c_long
    sys.path.insert(0, ROOT)
    import lettuce_amd
    CASES[sys.argv[2]](h, lettuce_amd)
