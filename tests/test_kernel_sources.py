"""What the kernel sources must keep where no run can show it: how the lanes of a wave hand each other LDS data. A bare
wave barrier orders no memory, and an access through another type than the object's may pass the object's own accesses, so
either can be reordered by a compiler that is right to do so."""

import os
import re

import pytest

from vgr import build


def source(name):
	with open(os.path.join(build.CSRC, name)) as f:
		return re.sub(r'//[^\n]*', '', f.read())


@pytest.mark.parametrize('name', sorted(f for f in os.listdir(build.CSRC) if f.endswith(('.hip', '.h'))))
def test_wave_barriers_order_memory(name):
	"""Every wave barrier is wave_sync's, between a release and an acquire fence."""
	bare = source(name).count('__builtin_amdgcn_wave_barrier')
	assert bare == (1 if name == 'vgr_device.h' else 0)
	if bare:
		body = source(name).split('void wave_sync()')[1].split('}')[0]
		calls = re.findall(r'__builtin_amdgcn_(?:fence\(__ATOMIC_(\w+), "wavefront"\)|(wave_barrier))', body)
		assert [a or b for a, b in calls] == ['RELEASE', 'wave_barrier', 'ACQUIRE']


def test_queue_is_accessed_through_its_own_types():
	"""foam_tile.hip's LDS queue is cast to nothing but a vector type that may alias its elements."""
	text = source('foam_tile.hip')
	casts = re.findall(r'reinterpret_cast<([^>]+)>\(Q\.', text)
	alias = set(re.findall(r'typedef \w+ (\w+) __attribute__\(\([^;]*may_alias', text))
	assert all(c.rstrip('* ') in alias for c in casts)
