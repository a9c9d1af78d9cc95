"""What the compiler gave the kernels of libaqtx.so, read from the library's own metadata (no GPU needed)."""
import struct

import msgpack

from aqt_amd import _lib as L
from aqt_amd import build


def _gfx950_objects(data):
  """The gfx950 code objects of a library's offload bundles."""
  magic = b'__CLANG_OFFLOAD_BUNDLE__'
  at = data.find(magic)
  while at >= 0:
    p = at + 32
    for _ in range(struct.unpack_from('<Q', data, at + 24)[0]):
      off, size, length = struct.unpack_from('<QQQ', data, p)
      if b'gfx950' in data[p + 24:p + 24 + length]:
        yield data[at + off:at + off + size]
      p += 24 + length
    at = data.find(magic, at + 24)


def _kernels():
  """The metadata of every kernel (the AMDGPU note of each object, a msgpack map)."""
  L.lib()  # built if it is not there
  with open(build.LIB_PATH, 'rb') as f:
    data = f.read()
  for elf in _gfx950_objects(data):
    shoff, = struct.unpack_from('<Q', elf, 40)
    size, count = struct.unpack_from('<HH', elf, 58)
    for i in range(count):
      kind, = struct.unpack_from('<I', elf, shoff + i * size + 4)
      if kind == 7:  # SHT_NOTE
        off, = struct.unpack_from('<Q', elf, shoff + i * size + 24)
        name, desc, _ = struct.unpack_from('<III', elf, off)
        start = off + 12 + (name + 3) // 4 * 4
        yield from msgpack.unpackb(elf[start:start + desc])['amdhsa.kernels']


def test_row_quantizers_use_no_scratch():
  """A row's values live in registers between its two passes; a launch bound that makes them spill costs more than the
  waves it wins."""
  rows = [k for k in _kernels() if 'quant_rows_kernel' in k['.name']]
  assert len(rows) > 40
  spilled = {k['.name']: k['.private_segment_fixed_size'] for k in rows if k['.private_segment_fixed_size']}
  assert not spilled
