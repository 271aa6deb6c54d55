"""Registers and scratch of the built library's kernels, from the AMDGPU metadata
notes the compiler writes into each code object."""
import struct
import subprocess

import msgpack

from sde_mc_amd import build

_BUNDLE = b'__CLANG_OFFLOAD_BUNDLE__'
_NT_AMDGPU_METADATA = 32
_SHT_NOTE = 7


def _code_objects(data):
    """The device ELF images of every offload bundle in the library."""
    pos = data.find(_BUNDLE)
    while pos >= 0:
        entry = pos + 32
        for _ in range(struct.unpack_from('<Q', data, pos + 24)[0]):
            off, size, n = struct.unpack_from('<QQQ', data, entry)
            if size and b'amdgcn' in data[entry + 24:entry + 24 + n]:
                yield data[pos + off:pos + off + size]
            entry += 24 + n
        pos = data.find(_BUNDLE, entry)


def _notes(elf):
    shoff = struct.unpack_from('<Q', elf, 40)[0]
    width, count = struct.unpack_from('<HH', elf, 58)
    for i in range(count):
        kind, = struct.unpack_from('<I', elf, shoff + i * width + 4)
        off, size = struct.unpack_from('<QQ', elf, shoff + i * width + 24)
        p = off
        while kind == _SHT_NOTE and p < off + size:
            name, desc, what = struct.unpack_from('<III', elf, p)
            p += 12 + (name + 3) // 4 * 4
            if what == _NT_AMDGPU_METADATA:
                yield msgpack.unpackb(elf[p:p + desc], strict_map_key=False)
            p += (desc + 3) // 4 * 4


def kernels():
    """{kernel name as written in the source, e.g. 'k_batch<0, 1>': metadata}."""
    with open(build.lib_path(), 'rb') as f:
        data = f.read()
    found = {k['.name']: k for elf in _code_objects(data) for n in _notes(elf)
             for k in n['amdhsa.kernels']}
    names = list(found)
    plain = subprocess.run(['c++filt', '-p'], input='\n'.join(names), capture_output=True,
                           text=True, check=True).stdout.split('\n')
    return {p.replace('sdemc::', '').replace('(int)', ''): found[n] for p, n in zip(plain, names)}


def waves_per_simd(kernel):
    """Wavefronts its vector registers let a SIMD hold (512 registers a lane, in
    steps of 8, at most 8 wavefronts)."""
    used = max(8, (kernel['.vgpr_count'] + 7) // 8 * 8)
    return min(8, 512 // used)
