"""Batch creation's host part: what it accepts (no GPU needed: an ordinal that no machine has makes
creation end at the device, after the lists are counted)."""
import numpy as np
import pytest


def test_window_with_more_pairs_than_an_int_counts(sg):
    """30 cameras that see one point 2,222 times each: 435 * 2222^2 > 2^31 pairs of observations that two
    cameras share.  The counts and positions of pairs are 64 bits wide, so nothing is refused."""
    cams, times = 31, 2222
    assert (cams - 1) * (cams - 2) // 2 * times * times > 2**31
    cam = np.repeat(np.arange(1, cams), times)
    poses = np.zeros((cams, 7))
    poses[:, 0] = 1.0
    point = np.array([[0.0, 0.0, 5.0]])
    idx = np.stack([np.zeros_like(cam), cam, np.zeros_like(cam)], axis=1)
    w = sg.BaProblem(np.array([[500.0, 500.0, 320.0, 240.0]]), poses, poses, point, point, idx, np.zeros((len(cam), 2)))
    with pytest.raises(sg.DeviceError):
        sg.Batch([w], sg.OptParams(device=99))
