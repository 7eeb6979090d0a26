"""The device-wide scan's choice of form by size (scan_layout::spread_u, large_tiles), replayed on the
CPU: coverage, slot counts and workspace at the edges between the forms, powers of two and random sizes."""
import os
import random
import subprocess

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def test_every_form_covers_its_sizes_and_fits_the_workspace():
    subprocess.run(["make", "-C", NATIVE, "scan_forms_check"], check=True, capture_output=True)
    edges = [64 * vec * u * tiles for vec in (2, 4) for u in (2, 4, 8, 16) for tiles in (1, 2, 64, 256, 512)]
    edges += [64 * vec * u * w * t for t in (128, 255, 256, 383, 384) for vec in (2, 4) for u in (16, 32, 64) for w in (4, 8)]
    sizes = {e + d for e in edges for d in (-3, -1, 0, 1, 2, 5)} | {1 << k for k in range(36)}
    rng = random.Random(11)
    sizes |= {int(2 ** rng.uniform(0, 33)) for _ in range(3000)}
    r = subprocess.run([os.path.join(NATIVE, "scan_forms_check")] + [str(n) for n in sorted(sizes)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
