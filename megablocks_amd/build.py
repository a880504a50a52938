"""Builds libmbx.so (the HIP kernels + C ABI) and libmbx_probe.so (measurement aids for bench.py) in-tree for
gfx950 with hipcc.

    python megablocks_amd/build.py            # compile what is out of date
    python megablocks_amd/build.py --force    # recompile everything

(run it as a script: `python -m megablocks_amd.build` would import the package, which needs the
library to exist already)
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
BUILD = os.path.join(HERE, 'build')
LIB = os.path.join(HERE, 'libmbx.so')
PROBE_LIB = os.path.join(HERE, 'libmbx_probe.so')
# the library with per-tile time stamps in the grouped-GEMM kernels (csrc/gmm_dma.h, MBX_TICKS), for bench.py --tile-ticks
TICKS_LIB = os.path.join(HERE, 'libmbx_ticks.so')
PROBE_SOURCE = 'probe.hip'
SOURCES = ['routing.hip', 'permute.hip', 'gmm.hip', 'gmm_rows.hip', 'gmm_rows_tail.hip', 'gmm_few.hip', 'gmm_f32.hip', 'gmm_mid.hip', 'gmm_pair.hip', 'gmm_tn_short.hip', 'elementwise.hip', 'router.hip', 'experts.hip']
TICKS_SOURCES = ['gmm.hip', 'gmm_rows.hip', 'gmm_rows_tail.hip']
HEADERS = [os.path.join(CSRC, 'common.h'), os.path.join(CSRC, 'gmm_dma.h'), os.path.join(CSRC, 'gmm_common.h'), os.path.join(CSRC, 'gmm_rows.h'),
           os.path.join(os.path.dirname(HERE), 'include', 'mbx.h'), os.path.join(os.path.dirname(HERE), 'include', 'mbx_probe.h')]
ARCH = 'gfx950'
# -packed-fp32-ops is switched off: hipcc must not form v_pk_*_f32 from scalar float code.
FLAGS = ['-O3', '-fPIC', '-std=c++17', f'--offload-arch={ARCH}', '-Xclang', '-target-feature', '-Xclang',
         '-packed-fp32-ops', '-Wno-unused-command-line-argument']


def _hipcc():
    for cand in (os.environ.get('HIPCC'), '/opt/rocm/bin/hipcc', 'hipcc'):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    return 'hipcc'


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = '\n'.join(l for l in proc.stdout.splitlines() if "is not a recognized feature for this target" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f'command failed: {" ".join(cmd)}\n{out}')
    return out


def build(force: bool = False, verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    hipcc = _hipcc()
    objs = []
    newest_header = max(os.path.getmtime(h) for h in HEADERS)
    procs = []
    for src in SOURCES:
        s = os.path.join(CSRC, src)
        o = os.path.join(BUILD, src.replace('.hip', '.o'))
        objs.append(o)
        stale = force or not os.path.exists(o) or os.path.getmtime(o) < max(os.path.getmtime(s), newest_header)
        if stale:
            cmd = [hipcc] + FLAGS + ['-c', s, '-o', o]
            if verbose:
                print(' '.join(cmd), flush=True)
            procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    # the 16-bit grouped-GEMM sources a second time with the time stamps compiled in
    ticks_objs = {}
    for src in TICKS_SOURCES:
        s, o = os.path.join(CSRC, src), os.path.join(BUILD, src.replace('.hip', '_ticks.o'))
        ticks_objs[os.path.join(BUILD, src.replace('.hip', '.o'))] = o
        if force or not os.path.exists(o) or os.path.getmtime(o) < max(os.path.getmtime(s), newest_header):
            cmd = [hipcc] + FLAGS + ['-DMBX_TICKS', '-c', s, '-o', o]
            if verbose:
                print(' '.join(cmd), flush=True)
            procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    probe_src = os.path.join(CSRC, PROBE_SOURCE)
    probe_cmd = None
    if force or not os.path.exists(PROBE_LIB) or os.path.getmtime(PROBE_LIB) < max(os.path.getmtime(probe_src), newest_header):
        probe_cmd = [hipcc] + FLAGS + ['-shared', probe_src, '-o', PROBE_LIB]
        if verbose:
            print(' '.join(probe_cmd), flush=True)
        procs.append((probe_cmd, subprocess.Popen(probe_cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    for cmd, p in procs:
        out, _ = p.communicate()
        if p.returncode != 0:
            raise RuntimeError(f'command failed: {" ".join(cmd)}\n{out}')
    if [c for c, _ in procs if c is not probe_cmd] or force or not os.path.exists(LIB) or not os.path.exists(TICKS_LIB):
        _run([hipcc, '-shared', '-fPIC', f'--offload-arch={ARCH}', '-o', LIB] + objs)
        _run([hipcc, '-shared', '-fPIC', f'--offload-arch={ARCH}', '-o', TICKS_LIB] +
             [ticks_objs.get(o, o) for o in objs])
    return LIB


if __name__ == '__main__':
    print(build(force='--force' in sys.argv, verbose=True))
