"""The device face loops on a randomly numbered mesh whose cells the lists
reorder and one of whose cells has more faces than a slice has slots for."""
import pytest

import test_gpu_faces as faces_tests
from test_gpu_faces import S  # noqa: F401  (fixture)
from test_layout_face_tails import with_hub

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def hub_mesh(monkeypatch):
    # just over the sizes from which cells are reordered
    monkeypatch.setitem(faces_tests.MESHES, "assembly reordered, hub",
                        lambda: with_hub((61, 67, 65), 45)[:2])
    monkeypatch.setitem(faces_tests.MESHES, "reordered, hub",
                        lambda: with_hub((81, 83, 79), 70)[:2])


@pytest.mark.parametrize("kinds", [(0, 1, 2), (0, 1, 2, 3)])
def test_gradients_and_velocity(S, oracle, kinds):  # noqa: F811
    faces_tests.test_gradients_and_velocity(S, oracle, "reordered, hub", kinds)


@pytest.mark.parametrize("name", ["assembly reordered, hub", "reordered, hub"])
def test_pressure_and_assembly(S, oracle, name):  # noqa: F811
    faces_tests.test_pressure_and_assembly(S, oracle, name)
