"""What calls of the library launch, asked on the CPU: the library in a process of its own behind launch_recorder.c, which takes the
place of the HIP runtime, with addresses in place of tensors (nothing reads or writes what they point to)."""
import ctypes
import os
import subprocess
import sys
import types

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(body, tmp_path):
    """Runs the function `body` of a test module in such a process and returns the lines that it prints."""
    so = os.path.join(str(tmp_path), 'launch_recorder.so')
    subprocess.run(['gcc', '-O1', '-shared', '-fPIC', os.path.join(ROOT, 'tests', 'launch_recorder.c'), '-o', so], check=True)
    code = f'import tests.launches as l\nl.begin({so!r})\nimport importlib\nimportlib.import_module({body.__module__!r}).{body.__name__}()'
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT] + os.environ.get('PYTHONPATH', '').split(os.pathsep)).rstrip(os.pathsep))
    r = subprocess.run([sys.executable, '-c', code], cwd=ROOT, env=env, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    return r.stdout.splitlines()


recorder = None


def begin(so):
    """The recorder and then the library, without the package's __init__ (which loads torch, and torch the HIP runtime)."""
    global recorder
    recorder = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    recorder.recorder_text.restype = ctypes.c_char_p
    recorder.recorder_events.restype = ctypes.c_long
    package = types.ModuleType('substation_amd')
    package.__path__ = [os.path.join(ROOT, 'substation_amd')]
    sys.modules['substation_amd'] = package


def launched(call):
    """[(kernel, grid)] of a call."""
    recorder.recorder_clear()
    call()
    lines = [line.split() for line in recorder.recorder_text().decode().splitlines()]
    return [(name, tuple(int(x) for x in grid)) for name, *grid in lines]


def tensors(count, first=1):
    """Addresses that stand for tensors, far apart."""
    return [(first + i) << 36 for i in range(count)]
