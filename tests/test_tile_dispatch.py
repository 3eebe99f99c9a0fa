"""The 16-bit dispatch by rows per touched expert: kernel codes on both sides of
each line, and workspaces past a line that do for the batches before it."""
import pytest

import candle_moe as cm

# (H, I, E, k, pairs per expert) -> kernel code (moe_type 0, bf16, 256 CUs)
EDGES = [
    (4096, 1536, 8, 2, 32, 18),        # decode kernels: 256 pairs
    (4096, 1536, 8, 2, 33, 5),         # 128x128 up to 136 rows
    (4096, 1536, 8, 2, 136, 5),
    (4096, 1536, 8, 2, 137, 7),        # above: one 256-row tile per expert
    (2048, 768, 128, 8, 32, 12),
    (2048, 768, 128, 8, 33, 14),       # more than 1.5 128x128 tiles per CU
    (2048, 768, 128, 8, 136, 14),
    (2048, 768, 128, 8, 137, 7),
    (2048, 768, 128, 8, 231, 7),
    (2048, 768, 128, 8, 232, 14),      # a 256-row tile often spills over
    (2048, 768, 128, 8, 1023, 14),
    (2048, 768, 128, 8, 1024, 7),
    (1024, 1024, 16, 2, 128, 12),      # few down tiles: f32 atomics kept
    (1024, 1024, 16, 2, 129, 5),
    (1024, 1024, 16, 2, 255, 5),       # short gate/up K loops, few 256x256 tiles
    (1024, 1024, 16, 2, 256, 7),
]


@pytest.mark.parametrize("H,I,E,k,rows,code", EDGES)
def test_kernel_at_the_lines(H, I, E, k, rows, code):
    T = rows * E // k
    assert T * k == rows * E
    assert cm.fused_moe_kernel(T, H, I, E, k, cm.DT_BF16) == code


@pytest.mark.parametrize("dt", [cm.DT_BF16, cm.DT_F16, cm.DT_F32])
@pytest.mark.parametrize("H,I,E,k", [(4096, 1536, 8, 2), (2048, 768, 128, 8), (768, 3072, 8, 2), (1024, 2048, 16, 2),
                                     (520, 264, 5, 3)])
def test_workspace_past_a_line(H, I, E, k, dt):
    """Past a line the workspace still holds the largest batch before it. (The
    lines that lie at a number of rows; the next test has all batches.)"""
    size = cm.lib().candle_moe_fused_moe_workspace_size
    lines = sorted({256 // k} | {r * E // k for r in (32, 64, 128, 136)} | {(256 * E - 1) // k})
    for i, T in enumerate(lines):
        for larger in [T + 1] + lines[i + 1:] + [2 * lines[-1]]:
            assert size(larger, H, I, E, k, dt) >= size(T, H, I, E, k, dt) > 0, (T, larger)


@pytest.mark.parametrize("dt", [cm.DT_BF16, cm.DT_F16, cm.DT_F32])
@pytest.mark.parametrize("H,I,E,k", [(4096, 1536, 8, 2), (2048, 768, 128, 8), (768, 3072, 8, 2), (4096, 4096, 128, 1),
                                     (1280, 1888, 64, 2), (8192, 2048, 8, 1), (4096, 512, 128, 8), (520, 264, 5, 3),
                                     (1536, 2048, 256, 4), (4096, 4096, 1, 1), (516, 260, 6, 2), (257, 129, 4, 2)])
def test_workspace_never_shrinks(H, I, E, k, dt):
    """A workspace for a batch does for every smaller one: its size never falls
    from one number of tokens to the next (decode slices, K splits, the pairs'
    rows and the expert sets all come and go on the way)."""
    size = cm.lib().candle_moe_fused_moe_workspace_size
    last = 0
    for T in list(range(1, 1200)) + list(range(1200, 6000, 7)) + list(range(6000, 40000, 211)):
        n = size(T, H, I, E, k, dt)
        assert n >= last > 0 or (T == 1 and n > 0), (T, last, n)
        last = n


def test_tail_parts(tmp_path):
    """K parts of the tiles of a 256x256 launch's last round (tests/cpp/tail_parts.cpp)."""
    import os
    import shutil
    import subprocess

    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = str(tmp_path / "tail_parts")
    subprocess.run([cxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                    os.path.join(root, "tests", "cpp", "tail_parts.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
