"""Which launches of the many-row GEMM the GPU tests cover: the shape and the
K-slices that csrc/wide_shape.h picks for their sizes, from the header itself
(tests/c/wide_shapes.cpp), so that new costs there cannot drop one unseen."""
import os
import subprocess

import pytest
import test_gpu_gemm
import test_gpu_prefill

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def pick(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("wide") / "wide_shapes")
    rocm = os.environ.get("ROCM", "/opt/rocm")
    r = subprocess.run([rocm + "/llvm/bin/clang++", "-std=c++17", "-O1", "-o", exe,
                        os.path.join(ROOT, "tests", "c", "wide_shapes.cpp")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]

    def run(split, rope, scheme, m, k, part, rows):
        line = " ".join(str(int(v)) for v in (split, rope, scheme, m, k, part, len(rows), *rows))
        out = subprocess.run([exe], input=line, capture_output=True, text=True).stdout.split()
        return int(out[0]), int(out[1])
    return run


def part_floats(rows, nb):
    """The linear's workspace for K-slices (csrc/capi_gemm.cpp, part_floats)."""
    def whole(k):
        return -(-nb // -(-nb // k))
    kg = whole(max(1, min(-(-512 // -(-rows // 128)), nb // 15)))
    small = whole(min(nb, max(min(-(-240 // -(-rows // 64)), max(1, nb // 4)), -(-nb // 30))))
    return max(kg * 64, small * 16) * (-(-rows // 16) * 16) if kg > 1 or small > 1 else 0


def test_every_shape_is_covered(pick):
    seen = {(split, scheme, pick(split, 0, scheme, m, cols, part_floats(rows, cols // 128), [rows])[0])
            for scheme, rows, cols, m in test_gpu_gemm.MANY_ROWS for split in (0, 1)}
    assert seen == {(p, s, h) for p in (0, 1) for s in (3, 4) for h in range(5)}
    # the q/k/v epilogue's forms, each with both schemes
    qkv = [[nh * 128, nkv * 128, nkv * 128] for nh, nkv, _ in test_gpu_prefill.QKV_SHAPES]
    for scheme in (3, 4):
        assert {pick(1, 1, scheme, n, 256, 0, rows)[0] for rows, (_, _, n) in zip(qkv, test_gpu_prefill.QKV_SHAPES)} \
            == {0, 1, 2}


def test_k_slices_where_the_chip_has_room(pick):
    """The sliced cases of the GPU tests are sliced (both shapes, both
    schemes, both kinds of X), the others are not; no slice is empty; nothing
    is sliced without the workspace for it."""
    seen = set()
    for scheme, rows, cols, m in test_gpu_gemm.MANY_ROWS + test_gpu_gemm.K_SLICED:
        for split in (0, 1):
            part = part_floats(rows, cols // 128)
            shape, k = pick(split, 0, scheme, m, cols, part, [rows])
            assert (k > 1) == ((scheme, rows, cols, m) in test_gpu_gemm.K_SLICED), (scheme, rows, cols, m, split, k)
            nbk = -(-(cols // 128) // k)
            assert (k - 1) * nbk < cols // 128 and k * m * (-(-rows // 16) * 16) <= max(part, m * (-(-rows // 16) * 16))
            assert pick(split, 0, scheme, m, cols, 0, [rows])[1] == 1
            if k > 1:
                seen.add((split, scheme, shape))
    assert seen == {(p, s, h) for s in (3, 4) for p, h in ((0, 3), (0, 4), (1, 1), (1, 3))}
    # q, k and v together, or gate and up, have no slices
    assert pick(1, 1, 4, 24, 2560, 1 << 22, [4096, 1024, 1024])[1] == 1
    assert pick(1, 0, 4, 24, 12288, 1 << 22, [512, 512])[1] == 1
