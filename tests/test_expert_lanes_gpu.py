"""Routing with an expert a lane: 64 experts, one fewer and one more, as many choices as experts."""
import pytest

from test_few_rows_experts_gpu import test_routes_and_their_tiles as routes_and_their_tiles
from test_few_rows_experts_gpu import test_routes_of_logits_that_are_not_numbers as routes_of_odd_logits

pytestmark = pytest.mark.gpu
FORMS = ["softmax", "over all", "sigmoid"]


@pytest.mark.parametrize("T,E,top", [(4, 64, 8), (3, 64, 11), (16, 63, 2), (11, 40, 3), (8, 65, 4), (1, 64, 64), (2, 3, 3)])
@pytest.mark.parametrize("form", FORMS)
def test_places_and_tiles(T, E, top, form):
    routes_and_their_tiles(T, E, top, form)


@pytest.mark.parametrize("T,E,top", [(4, 63, 8), (5, 64, 6), (16, 64, 2), (40, 64, 8)])
@pytest.mark.parametrize("form", FORMS)
def test_odd_logits(T, E, top, form):
    routes_of_odd_logits(T, E, top, form)
