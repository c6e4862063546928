"""Voxeliser with the calling convention of the reference's ``simple_mean_encoder``
(deploy3d/symfun/ops/voxel_encoder/simple_mean.py:6-52), executed by the HIP
engine: the reference's torch-side ``forward`` returns zero tensors of the right
shape, this one returns the voxels.
"""
import numpy as np
import torch

from .plugin import Launch, LaunchCache, Plugin, TensorDesc, current_stream, scratch

_plugins = {}
_launches = LaunchCache()


def simple_mean_blob(max_num_act_out):
    """SimpleMeanEncoderPluginParam (trt/voxel_encoder/simple_mean_trt.cu:176-180; writer: simple_mean.py:44)."""
    return np.array([max_num_act_out], dtype=np.int32).tobytes()


def simple_mean_encoder(batch_point_feats, batch_indices, voxel_config, in_spatial_shape, max_num_act_out):
    """Points to voxels: mean of the features of the points in every occupied cell.

    batch_point_feats  float32 [N, C], x y z first; rows with a non-finite feature are skipped
    batch_indices      int32 [N]; negative = skip the point
    voxel_config       float32 [6] on the device: xMin yMin zMin xSize ySize zSize
    in_spatial_shape   zero-element tensor of shape [B, 0, Z, Y, X]
    Returns (out_feats [max_num_act_out, C], out_coors int32 [max_num_act_out, 4] rows (b, z, y, x),
    num_act_out int32 [1]); voxels come in order of first appearance among the points.
    """
    if batch_point_feats.dtype != torch.float32 or voxel_config.dtype != torch.float32:
        raise TypeError("point features and voxel config must be float32")
    if batch_indices.dtype != torch.int32:
        raise TypeError("batch indices must be int32")
    batch_point_feats = batch_point_feats.contiguous()
    batch_indices = batch_indices.contiguous()
    dev = batch_point_feats.device
    if voxel_config.device != dev:
        voxel_config = voxel_config.to(dev)
    voxel_config = voxel_config.contiguous()
    key = (int(max_num_act_out), batch_point_feats.shape, batch_indices.shape, voxel_config.shape, in_spatial_shape.shape)
    launch = _launches.get(key)
    if launch is None:
        plugin = _plugins.get(key[0])
        if plugin is None:
            plugin = _plugins[key[0]] = Plugin("SimpleMeanEncoder", simple_mean_blob(max_num_act_out))
        launch = _launches.put(key, Launch(plugin, [
            TensorDesc.of_tensor(batch_point_feats), TensorDesc.of_tensor(batch_indices),
            TensorDesc.of_tensor(voxel_config), TensorDesc.of(tuple(in_spatial_shape.shape), torch.int32)]))
    feats_shape, coors_shape, num_shape = launch.shapes
    outs = (torch.empty(feats_shape, dtype=torch.float32, device=dev),
            torch.empty(coors_shape, dtype=torch.int32, device=dev),
            torch.empty(num_shape, dtype=torch.int32, device=dev))
    stream = current_stream(dev)
    launch((batch_point_feats, batch_indices, voxel_config, None), outs, scratch(launch.nbytes, dev, stream), stream)
    return outs


class SimpleMeanEncoder:
    """Name-compatible handle: ``SimpleMeanEncoder.apply(...)`` as in the reference."""
    apply = staticmethod(simple_mean_encoder)
