"""CPU check of the rules that choose a quantised projection's kernel and tiles
(engine-mlx_amd/csrc/qmatmul_plan.hpp, the definitions that the launches use): every case of the
GPU tests whose kernel its comment names runs that kernel on 256 CUs, every kernel and tile has
such a case, and a call's arithmetic (exact products, or weights dequantised into the activation
type) depends on its rows and K alone."""
import os
import subprocess

import pytest

import test_gpu_qmatmul as cases

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.fixture(scope="module")
def routes():
    subprocess.run(["make", "-s", "-C", CPP, "test_qmm_route"], check=True)

    def run(calls):
        """calls: (M, N, K, group, bits, ldx, bytes of scales past 16, CUs)"""
        text = "\n".join(" ".join(str(v) for v in c) for c in calls) + "\n"
        r = subprocess.run([os.path.join(CPP, "test_qmm_route")], input=text, capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        out = r.stdout.strip().split("\n")
        assert len(out) == len(calls)
        return out

    return run


def test_gpu_cases_run_the_kernel_they_name(routes):
    listed = [(c[:5], 0, c[6]) for c in cases.KSPLIT_TILES + cases.KSPLIT_DECODE + cases.DQ_TILES]
    listed += [(c[:5], c[6], c[7]) for c in cases.OFF_ALIGNMENT]
    got = routes([(*c, c[2], past, 256) for c, past, _ in listed])
    for (c, past, want), r in zip(listed, got):
        assert r == want, f"{c}, scales {past} bytes past 16: {r}, not {want}"


def units(K):
    return K // 128


def test_every_tile_has_a_case_of_its_main_loop(routes):
    """Each tile of the K-split GEMM that the rules can choose is tested with several units per
    wave, at 4 and at 8 bits."""
    calls = [(M, N, K, 32, bits, K, 0, 256) for M in range(33, 700, 9) for N in range(64, 9000, 331)
             for K in (1152, 4096) for bits in (4, 8)]
    chosen = {(c[4], r) for c, r in zip(calls, routes(calls)) if r.startswith("qgemm_ks")}
    tested = {(c[4], c[6]) for c in cases.KSPLIT_TILES if units(c[2]) > 8}
    assert chosen == tested, chosen ^ tested


def test_arithmetic_depends_on_rows_and_k_alone(routes):
    """More than 32 rows and K a multiple of 64: dequantised weights whatever the tile, up to the
    row stride at which 256 rows pass the 2 GiB of a buffer range; beyond it exact products."""
    strides = (0, 72, 4_000_000, 4_186_000, 4_194_304, 5_000_000, 8_000_000, 13_000_000, 30_000_000)
    calls = [(M, N, K, gs, bits, max(K, s), past, 256) for M in (33, 157, 300, 1531) for N in (100, 4096, 6144)
             for K in (256, 320, 4096) for gs, bits in ((32, 8), (64, 4)) for s in strides for past in (0, 2)]
    for c, r in zip(calls, routes(calls)):
        dequantised = 256 * c[5] * 2 + c[2] * 2 < 1 << 31
        assert (r.split()[0] in ("qgemm_ks", "qgemm_dq", "qgemm_dq_staged")) == dequantised, (c, r)


def test_many_columns_of_short_rows_keep_the_staged_kernels(routes):
    """Up to 32 rows, K of 2048 to 3072 and more columns than one round of workgroups: calls that
    the K-split kernel took 1.1 to 1.5 times as long for (measured on 256 CUs), and neighbours
    that it is faster for."""
    staged = [(2, 8208, 2048, 64, 4), (2, 151936, 2048, 64, 4), (3, 18944, 2048, 128, 4), (8, 151936, 2048, 64, 4),
              (8, 10240, 2048, 64, 4), (16, 151936, 2048, 128, 4), (24, 9216, 2048, 32, 4), (24, 151936, 2048, 64, 8),
              (32, 32768, 2048, 32, 8), (32, 32768, 2560, 64, 8), (24, 32768, 3072, 32, 4), (2, 9216, 3072, 128, 4)]
    split = [(2, 8192, 2048, 64, 4), (8, 10240, 2048, 32, 4), (16, 10240, 2048, 64, 4), (24, 9216, 2048, 64, 4),
             (2, 18944, 2560, 64, 4), (8, 151936, 2560, 64, 4), (16, 151936, 3072, 64, 4), (32, 9216, 2560, 64, 8),
             (32, 9216, 3072, 64, 8), (2, 151936, 4096, 64, 4), (32, 151936, 4096, 64, 8), (20, 9216, 2816, 64, 8)]
    got = routes([(*c, c[2], 0, 256) for c in staged + split])
    for c, r in zip(staged + split, got):
        assert r.split()[0] in (("qmv", "qmvx") if c in staged else ("qmv_ks",)), (c, r)
