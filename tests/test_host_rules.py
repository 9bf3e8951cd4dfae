"""Rules of the launchers that no result shows (which variant a call takes), compiled for the host."""
import glob
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "universal-lm-trainer_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")
OBJDUMP = os.path.join(ROCM, "llvm", "bin", "llvm-objdump")
LIB = os.path.join(os.path.dirname(CSRC), "lib", "libfa2_mi355x.so")


@pytest.fixture(scope="module")
def evaluate(tmp_path_factory):
    """evaluate(expressions) -> their values as integers, with namespace fa2 open and `args` / `rope_args` at hand."""
    def run(expressions):
        d = tmp_path_factory.mktemp("rules")
        src = d / "rules.cpp"
        src.write_text('#include "%s/fa2_kernels.h"\n#include <cstdio>\nusing namespace fa2;\n' % CSRC + """
static FwdArgs args(int B, int H, int Sk, int coff, int64_t sb, int64_t sh, int64_t ss, bool v_only = false) {
    FwdArgs a = {};
    a.B = B; a.H = H; a.S = 1; a.Sk = Sk; a.coff = coff;
    a.vsb = sb; a.vsh = sh; a.vss = ss;
    a.ksb = v_only ? (int64_t)H * Sk * 64 : sb; a.ksh = v_only ? (int64_t)Sk * 64 : sh; a.kss = v_only ? 64 : ss;
    return a;
}
static RopeArgs rope_args(int B, int H, int S, int64_t k_head) {
    RopeArgs a = {};
    a.B = B; a.H = H; a.S = S;
    a.qsb = a.ksb = (int64_t)S * 3 * H * 64; a.qss = a.kss = 3 * H * 64; a.qsh = 64; a.ksh = k_head;
    return a;
}
int main() {
""" + "\n".join(f'printf("%lld\\n", (long long)({e}));' for e in expressions) + "\n}\n")
        exe = d / "rules"
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", str(src), "-o", str(exe)], check=True,
                       capture_output=True)
        return [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    return run


def test_decode_streams_large_caches_read_once(evaluate):
    """80 MiB of K and V is B*H*keys = 327680."""
    n = 16384
    dense = (12 * n * 64, n * 64, 64)
    cases = [
        (1, "args(8, 12, %d, %d, %d, %d, %d), true" % (n, n - 1, *dense)),
        (1, "args(8, 12, %d, %d, %d, %d, %d), false" % (n, 0, *dense)),
        (0, "args(8, 12, %d, %d, %d, %d, %d), true" % (n, 3000, *dense)),        # 3001 keys seen
        (0, "args(8, 12, %d, %d, %d, %d, %d), true" % (n, -1, *dense)),
        (1, "args(8, 12, %d, %d, %d, 64, 768), true" % (n, n - 1, n * 768)),     # [B, S, H, D]
        (1, "args(8, 12, %d, %d, %d, %d, 64), true" % (n, n - 1, 12 * (n + 128) * 64, (n + 128) * 64)),   # spare keys
        (0, "args(8, 12, %d, %d, %d, 0, 64), true" % (n, n - 1, n * 64)),        # one head for all
        (0, "args(8, 12, %d, %d, 0, %d, 64), true" % (n, n - 1, n * 64)),        # one batch for all
        (0, "args(8, 12, %d, %d, %d, 0, 64, true), true" % (n, n - 1, n * 64)),  # V alone
        (0, "args(8, 12, %d, %d, %d, %d, 8), true" % (n, n - 1, 12 * n * 8, n * 8)),   # rows overlap
        (1, "args(1, 1, 400000, 399999, 0, 0, 64), true"),                       # strides of single heads don't count
        (0, "args(1, 20, 16384, 16383, %d, %d, 64), true" % (20 * n * 64, n * 64)),    # exactly 80 MiB
    ]
    got = evaluate(["decode_streams(%s)" % c for _, c in cases])
    assert got == [e for e, _ in cases]


def test_rope_streams_large_tensors(evaluate):
    """88 MiB of q and k is B*H*S = 360448; a k expanded over the heads is read from the caches."""
    cases = [
        (1, "rope_args(8, 12, 4096, 64)"), (0, "rope_args(8, 12, 2048, 64)"), (0, "rope_args(8, 11, 4096, 64)"),
        (1, "rope_args(8, 11, 4097, 64)"), (0, "rope_args(16, 12, 4096, 0)"),
    ]
    assert evaluate(["rope_streams(%s)" % c for _, c in cases]) == [e for e, _ in cases]


def test_head_groups(evaluate):
    """Multiples of eight heads in groups as ever; rounded head numbers under the causal mask only where
    the last, partial group does not set the time (768 dQ workgroups resident)."""
    cases = [
        (1, "fwd_groups(8, true, 8)"), (1, "fwd_groups(136, true, 8)"), (0, "fwd_groups(127, false, 8)"),
        (0, "fwd_groups(132, true, 8)"), (1, "fwd_groups(132, false, 8)"), (0, "fwd_groups(372, true, 5)"),
        (1, "fwd_groups(372, true, 4)"), (0, "fwd_groups(428, true, 8)"), (1, "fwd_groups(444, true, 8)"),
        (0, "fwd_groups((1 << 20) + 1, true, 2)"), (0, "fwd_groups(1024, true, 1)"), (1, "fwd_groups(1024, true, 2)"),
        (0, "dq_groups(1024, true, 1024, 768)"), (0, "dq_groups(1500, true, 1504, 768)"),
        (1, "dq_groups(128, true, 512, 768)"), (0, "dq_groups(132, true, 544, 768)"),
        (1, "dq_groups(132, false, 544, 768)"), (0, "dq_groups(188, true, 768, 768)"),
        (1, "dq_groups(196, true, 800, 768)"), (0, "dq_groups(100, true, 800, 768)"),
    ]
    assert evaluate([c for _, c in cases]) == [e for e, _ in cases]


def test_kernels_access_memory_by_address_space(tmp_path):
    """No flat loads or stores (they count as LDS accesses too, and every wait for an LDS read would wait
    for them) and no scratch in the kernels as built."""
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    objects = glob.glob(str(tmp_path / "lib.so.*gfx950"))
    assert len(objects) >= 3
    count = {"flat_": 0, "scratch_": 0, "global_": 0}
    for o in objects:
        for line in subprocess.run([OBJDUMP, "-d", o], check=True, capture_output=True, text=True).stdout.splitlines():
            for kind in count:
                count[kind] += line.strip().startswith(kind)
    assert count["global_"] > 100 and count["flat_"] == 0 and count["scratch_"] == 0, count
