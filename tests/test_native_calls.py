"""The parts of the native callers (csrc_torch) that need no GPU, compiled by themselves."""
import os
import shutil
import subprocess
import sys
import sysconfig

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "bladedisc_amd", "csrc_torch")
INCLUDE = sysconfig.get_paths()["include"]

pytestmark = pytest.mark.skipif(
    shutil.which("g++") is None or not os.path.exists(os.path.join(INCLUDE, "Python.h")),
    reason="needs g++ and Python's headers")


def _compile(tmp_path, source, target, *flags):
    out = str(tmp_path / target)
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-I" + SRC, "-isystem", INCLUDE,
           os.path.join(ROOT, "tests", "native", source), "-o", out] + list(flags)
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


def test_the_interpreter_lock_is_held_again_after_an_exception(tmp_path):
    """A launch runs without the lock; an exception from it, or from reading its arguments, comes
    out as an ordinary Python exception (in a process of its own: the fault is a crash)."""
    _compile(tmp_path, "unlocked_module.cc", "unlocked_module.so", "-shared", "-fPIC")
    script = ("import unlocked_module as m\n"
              "assert m.call(0) == 42\n"
              "for where, text in ((1, 'without'), (2, 'with the')) * 3:\n"
              "    try:\n"
              "        m.call(where)\n"
              "    except RuntimeError as e:\n"
              "        assert text in str(e), e\n"
              "    else:\n"
              "        raise SystemExit('no exception')\n"
              "print('ok')\n")
    r = subprocess.run([sys.executable, "-c", script], cwd=str(tmp_path), capture_output=True,
                       text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr)


def test_a_status_word_with_an_answer_outstanding_is_not_lent_again(tmp_path):
    """An answer that comes after its call has failed must not reach the next borrower."""
    exe = _compile(tmp_path, "status_words_check.cc", "status_words_check", "-pthread")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
