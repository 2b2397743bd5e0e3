"""Sixteen lanes per particle, which the size rule (lanes 0) gives contexts as
small as these, in the cases that force one lane and four: the pair terms at the
edges of their common form, impulses that are no number, nudges of coincident
particles, dense and overfull lattices, caps inside a cell, frozen scenes."""
import pytest

from tests import test_gpu_lanes as forced
from tests import test_gpu_pairs as pairs
from tests import test_gpu_reference_scenes as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h", [1.0, 1.3])
def test_pairs_at_the_edges(h):
    pairs.test_pairs_at_the_edges(h, lanes=0)


def test_impulse_that_is_no_number():
    pairs.test_impulse_that_is_no_number(lanes=0)


def test_coincident_particles_nudge_owner():
    ref.test_coincident_particles_nudge_owner(lanes=0)


def test_c1_dam_break():
    forced.test_c1_dam_break(lanes=0)


@pytest.mark.parametrize("cap", [0, 40])
def test_dense_lattice(cap):
    forced.test_dense_lattice(lanes=0, cap=cap)


def test_overfull_lattice():
    forced.test_overfull_lattice(lanes=0)


def test_batch_with_a_frozen_scene():
    forced.test_batch_with_a_frozen_scene(lanes=0)
