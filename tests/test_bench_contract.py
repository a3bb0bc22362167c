"""The benchmark's command-line contract on the CPU: more than one GPU is
refused with a message before any device work, and the argument parser
accepts the driver's flags (--gpus, --steps, --warmup)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2",
                        "--steps", "3", "--warmup", "1"],
                       stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode != 0
    msg = r.stdout + r.stderr
    assert "one GPU" in msg and "--gpus 2" in msg


def test_help_lists_the_driver_flags():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--help"],
                       stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == 0
    for flag in ("--gpus", "--steps", "--warmup", "--workload"):
        assert flag in r.stdout


def test_bytes_follow_the_launches():
    """What the record's rates are made of: a gauge-fixing iteration reads and
    writes every link once in one launch and twice in two, and a_f once either
    way; renorm adds its writes to a launch that reads the links anyway."""
    sys.path.insert(0, ROOT)
    import bench
    links, higgs = 3 * 32, 24  # bytes a site
    assert bench.GFIX_BYTES_PER_SITE == {1: 2 * links + 2 * higgs, 2: 4 * links + 2 * higgs}
    assert bench.REF_SWEEP_BYTES_PER_SITE == 4 * bench.HIGGS_PASS_BYTES_PER_SITE \
        + 6 * bench.LINK_PASS_BYTES_PER_SITE + links
