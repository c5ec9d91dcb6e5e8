"""The output kernel's quick colour forms where they hand over to the general
ones, byte for byte against the host path, which has only those: chromaticities
on and about the gamut's edges, its corners' rays from the white point and the
white point's vertical; values about the steps of 8 and 16 bits and about the
ends of the sRGB curve; black, negative and huge pixels; and an output address
of every alignment."""
import numpy as np
import pytest
import torch

from rise_amd.output import output_desc, resolve, write_image
from tests.conftest import log_case
from tests.test_output import _png_rgba

pytestmark = pytest.mark.gpu

V = np.array([[0.64, 0.33], [0.30, 0.60], [0.15, 0.06], [0.3127, 0.3290]])  # red, green, blue, white
M = np.linalg.inv([[3.240479, -1.537150, -0.498535], [-0.969256, 1.875992, 0.041556], [0.055648, -0.204043, 1.057311]])


@pytest.fixture(scope="module")
def film():
    g = np.random.default_rng(5)
    n = 40_000
    a, b = V[g.integers(0, 4, n)], V[g.integers(0, 4, n)]
    t = np.where(g.random(n) < 0.5, g.uniform(-2, 2, n), g.integers(0, 3, n))[:, None]
    xy = a + t * (b - a) + g.normal(size=(n, 2)) * np.where(g.random((n, 1)) < 0.3, 0.0, np.exp(g.uniform(-36, -2, (n, 1))))
    xy[::16, 0] = V[3, 0]
    xy[:, 1] = np.where(np.abs(xy[:, 1]) < 1e-3, 1e-3, xy[:, 1])
    Y = np.exp(g.uniform(-8, 1, n))
    clip = np.stack([xy[:, 0] / xy[:, 1] * Y, Y, (1 - xy.sum(1)) / xy[:, 1] * Y], 1)
    step = np.concatenate([np.arange(256) / 255.0, g.integers(0, 65536, 20_000) / 65535.0])
    lin = np.where(step <= 0.0392857, step / 12.92, ((step + 0.055) / 1.055) ** 2.4)
    lin = np.concatenate([lin, np.full(64, 0.003040247678), np.full(64, 1.0), np.full(64, 1.01)])
    gray = (lin[:, None] * M.sum(1)) * (1.0 + g.integers(-3, 4, (len(lin), 1)) * 2.0 ** -23)
    odd = np.array([[0, 0, 0], [0, 1, 0], [1, -1, 0], [-1, -1, -1], [1e30, 1e30, 1e30], [1e-38, 1e-38, 1e-38], [2, -1, 3]])
    px = np.concatenate([clip, gray, odd]).astype(np.float32)
    h = len(px) // 251
    return np.ascontiguousarray(px[len(px) - 251 * h:].reshape(h, 251, 3))


@pytest.mark.parametrize("bpp", [8, 16])
@pytest.mark.parametrize("display,ev", [("none", 0.0), ("aces", 0.0), ("reinhard", 1.5)])
@pytest.mark.parametrize("space", ["sRGB", "Rec709RGB_Linear"])
def test_gpu_output_edges(cuda, tmp_path, film, bpp, display, ev, space):
    log_case(f"{bpp} {display} {ev} {space}")
    d = output_desc("PNG", bpp, space, display, ev)
    write_image(film, tmp_path / "h.png", d)
    write_image(torch.from_numpy(film).to(cuda), tmp_path / "g.png", d)
    assert (tmp_path / "g.png").read_bytes() == (tmp_path / "h.png").read_bytes()


def test_gpu_output_alignment(cuda, tmp_path, film):
    d = output_desc("PNG", 8)
    write_image(film, tmp_path / "h.png", d)
    want = np.asarray(_png_rgba((tmp_path / "h.png").read_bytes())).reshape(-1)
    dev = torch.from_numpy(film).to(cuda)
    for off in range(5):
        log_case(f"output address + {off}")
        buf = torch.full((want.size + 16,), 7, dtype=torch.uint8, device=cuda)
        resolve(dev, buf[off:], d)
        got = buf.cpu().numpy()
        assert np.array_equal(got[off:off + want.size], want)
        assert np.all(got[:off] == 7) and np.all(got[off + want.size:] == 7)
