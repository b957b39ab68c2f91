"""Rings of direct global-to-LDS loads (CPU, from the sources): a wave passes a
raw barrier only once its LDS reads are done, because the loads that the other
waves issue behind it overwrite what was read, and the compiler orders no read
before a barrier by itself.  So every s_barrier written in asm stands in the
statement that waits, which only common.h has."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'qwen3_dspark_amd', 'csrc')


def test_every_asm_barrier_waits_for_the_lds_reads():
    found = {}
    for path in sorted(glob.glob(os.path.join(CSRC, '*.h*'))):
        code = re.sub(r'//[^\n]*', '', open(path).read())
        for statement in re.findall(r'asm volatile\((.*?)\);', code, re.S):
            if 's_barrier' in statement:
                assert re.search(r's_waitcnt[^"]*lgkmcnt\(0\)[^"]*s_barrier', statement), (path, statement)
                found[os.path.basename(path)] = found.get(os.path.basename(path), 0) + 1
        assert 'builtin_amdgcn_s_barrier' not in code
    assert found == {'common.h': 1}
