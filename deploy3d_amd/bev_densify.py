"""Sparse-to-dense operator with the calling convention of the reference's
``bev_densify`` (deploy3d/symfun/ops/spconv/bev_densify.py:18-45), executed by
the HIP engine: the reference's torch-side ``forward`` returns zeros of the
right shape, this one returns the map.
"""
import numpy as np
import torch

from .plugin import Launch, LaunchCache, Plugin, TensorDesc, current_stream, scratch

_plugins = {}
_launches = LaunchCache()


def densify_blob(out_channels):
    """BEVDensifyPluginParam (trt/spconv/bev_densify_trt.cu:43-47; writer: bev_densify.py:38)."""
    return np.array([out_channels], dtype=np.int32).tobytes()


def bev_densify(in_feats, in_coors, num_act_in, in_spatial_shape, out_channels, out=None):
    """out[B, C*Z, Y, X]: zero everywhere except out[b, c*Z + z, y, x] = in_feats[i, c] for the live rows.

    in_feats          [cap, C] float32 / float16 / bfloat16 / int8, device
    in_coors          int32 [cap, 4] rows (b, z, y, x), device
    num_act_in        int32 [1], device (never read on the host)
    in_spatial_shape  zero-element tensor of shape [B, 0, Z, Y, X]
    out_channels      C*Z
    """
    if in_coors.dtype != torch.int32 or num_act_in.dtype != torch.int32:
        raise TypeError("coordinates and counts must be int32")
    in_feats = in_feats.contiguous()
    in_coors = in_coors.contiguous()
    # the tensors' devices and types decide nothing else: shape inference and descriptors are made once per signature
    key = (int(out_channels), in_feats.shape, in_feats.dtype, in_coors.shape, num_act_in.shape, in_spatial_shape.shape)
    launch = _launches.get(key)
    if launch is None:
        plugin = _plugins.get(key[0])
        if plugin is None:
            plugin = _plugins[key[0]] = Plugin("BEVDensify", densify_blob(out_channels))
        launch = _launches.put(key, Launch(plugin, [
            TensorDesc.of_tensor(in_feats), TensorDesc.of_tensor(in_coors), TensorDesc.of_tensor(num_act_in),
            TensorDesc.of(tuple(in_spatial_shape.shape), torch.int32)]))
    dev = in_feats.device
    stream = current_stream(dev)
    if out is None:
        out = torch.empty(launch.shapes[0], dtype=in_feats.dtype, device=dev)
    launch((in_feats, in_coors, num_act_in, None), (out,), scratch(launch.nbytes, dev, stream), stream)
    return out


class BEVDensify:
    """Name-compatible handle: ``BEVDensify.apply(...)`` as in the reference."""
    apply = staticmethod(bev_densify)
