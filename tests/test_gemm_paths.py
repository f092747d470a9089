"""The rules that send a product to the special GEMM kernels and share it out:
no 32-bit offset of a kernel wraps for any product it is given, products a
kernel is meant for are not turned away, and a split sum leaves nothing out."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CXX = shutil.which("g++") or shutil.which("c++")


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    if CXX is None:
        pytest.skip("no host compiler")
    exe = tmp_path_factory.mktemp("paths") / "gemm_paths"
    subprocess.run([CXX, "-O1", "-std=c++17", f"-I{ROOT / 'namsa_amd' / 'csrc'}", str(ROOT / "tests" / "gemm_paths.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, timeout=300)

    def run(rows):
        text = "\n".join(" ".join(map(str, r)) for r in rows)
        out = subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout
        return [tuple(map(int, ln.split())) for ln in out.splitlines()]
    return run


def test_pointwise_offsets_do_not_wrap(ask):
    """The largest byte offsets of gemm_pointwise_kernel, restated: row 16 KS - 1
    of B at the last column its workgroups cover, row 32 MT - 1 of C at the last
    column."""
    rows = []
    for M in (1, 2, 8, 13, 31, 32, 33, 64):
        for K in (1, 2, 8, 15, 16, 17, 32, 33, 64):
            for e in range(13, 31):
                for N in (2 ** e - 1, 2 ** e, 5 * 2 ** (e - 2) + 1):
                    if N < 2 ** 31:
                        rows += [(M, N, K, N, N), (M, N, K, N + 7, N), (M, N, K, N, N + 1)]
            for pitch in (2 ** 31, 2 ** 40, 2 ** 62):
                rows += [(M, 8192, K, pitch, 8192), (M, 8192, K, 8192, pitch)]
            N = (2 ** 31 - 1) // 128                       # around the limits themselves
            rows += [(M, N // d + i, K, N // d + i, N // d + i) for d in (1, 2) for i in range(-40, 41)]
    answers = ask([("p", *r) for r in rows])
    assert len(answers) == len(rows)
    taken = 0
    for (M, N, K, sB, sC), (fits, mt, ks) in zip(rows, answers):
        if not fits:
            continue
        taken += 1
        cols = (N + 511) // 512 * 512
        assert 4 * ((16 * ks - 1) * sB + cols - 1) < 2 ** 31, (M, N, K, sB, sC)
        assert 4 * ((32 * mt - 1) * sC + N - 1) < 2 ** 31, (M, N, K, sB, sC)
        assert 32 * mt >= M and 16 * ks >= K
    assert taken > 1000


def test_pointwise_keeps_the_layers_it_is_for(ask):
    """Layers of 32 and 64 channels over the pixels of 16 to 256 samples of 170 x 170."""
    rows = [("p", M, B * 28900, K, B * 28900, B * 28900) for B in (16, 64, 256) for M, K in ((32, 32), (32, 7), (64, 32), (2, 64))]
    assert all(fits for fits, _, _ in ask(rows))


@pytest.mark.parametrize("cus", [1, 256, 304])
@pytest.mark.parametrize("batch", [1, 2, 300, 65535])
def test_split_shares_cover_k(ask, cus, batch):
    """Every k belongs to one workgroup, no workgroup is empty, and a
    wavefront's last step of 128 stays in 31 bits, up to the largest K taken."""
    top = 2 ** 31 - 256
    Ks = [1, 31, 127, 128, 129, 4099, 462400, 2 ** 24 + 1, 2 ** 30, top // 2 + 1, top - 1000, top - 1, top]
    for K, (groups, k_per, total, most, least) in zip(Ks, ask([("s", K, batch, cus) for K in Ks])):
        assert total == K and least >= 1 and most <= k_per, (K, groups, k_per, total, least)
        assert groups <= max(1, -(-cus // batch)) and k_per % 128 == 0
        assert groups * k_per < 2 ** 32 and most - 1 + 128 < 2 ** 31
