"""MSD network for segmentation (reference msd_segmentation_model.py:10-119)."""
import torch
import torch.nn as nn

from . import _native
from .msd_model import MSDModel, _moments, scaling_module_set_bias, scaling_module_set_scale


class MSDSegmentationModel(MSDModel):
    def __init__(self, c_in, num_labels, depth, width, *, dilations=[1, 2, 3, 4, 5, 6, 7, 8, 9, 10],
                 parallel=False, ndim=2):
        """``num_labels`` output classes; log-softmax over channels + NLL loss."""
        self.num_labels = num_labels
        super().__init__(c_in, num_labels, depth, width, dilations, ndim=ndim)
        self.criterion = nn.NLLLoss()

        net_trained = nn.Sequential(self.msd, nn.LogSoftmax(dim=1))
        self.net = nn.Sequential(self.scale_in, net_trained)
        self.net.cuda()
        if parallel:
            self.net = nn.DataParallel(self.net)
        self.init_optimizer(net_trained)

    def set_normalization(self, dataloader):
        """Only the input is normalised; the targets are labels."""
        mean, std, _, _ = _moments(dataloader)
        if std == 0:
            raise ValueError("set_normalization: the input data has zero variance")
        scaling_module_set_scale(self.scale_in, 1 / std)
        scaling_module_set_bias(self.scale_in, -mean / std)

    def set_target(self, target):
        """Labels in [0, num_labels), checked here as msd_segmentation_model.py:105-119 does (for
        a tensor on the GPU that read-back waits for the device; ``train`` defers it)."""
        target = target.long()
        lo, hi = target.min(), target.max()
        if lo < 0 or self.num_labels <= hi:
            raise ValueError(
                f"Target invalid: expected values in range {[0, self.num_labels - 1]}, but got {[lo, hi]}")
        # NLLLoss takes (B, *spatial) class indices: drop the channel axis
        self.target = target.squeeze(1).cuda()

    _label_range = None

    def _set_target_deferred(self, target):
        if not target.is_cuda:
            return self.set_target(target)      # a host tensor is checked on the host: no device wait
        # lowest and highest label seen since the last verdict, kept on the device; the step
        # itself runs on labels clamped into range, so no loss kernel ever sees an invalid one
        target = target.long().contiguous()
        seen = self._label_range
        if seen is None:
            limits = torch.iinfo(torch.int64)
            seen = torch.full((2,), limits.min, dtype=torch.int64, device=target.device)
            seen[0] = limits.max
        clamped = _native.host().label_check(target, self.num_labels, seen)
        if clamped is None:                     # an empty batch, another device than the batch before
            return self.set_target(target)
        self._label_range = seen
        self.target = clamped.squeeze(1)

    def _raise_deferred_target_error(self):
        seen, self._label_range = self._label_range, None
        if seen is None:
            return
        lo, hi = seen.tolist()
        if lo < 0 or self.num_labels <= hi:
            raise ValueError(
                f"Target invalid: expected values in range {[0, self.num_labels - 1]}, but got {[lo, hi]}")

    def _fused_parts(self):
        if self._loss_kind() != "nll" or not isinstance(self.net, nn.Sequential) or len(self.net) != 2:
            return None
        trained = self.net[1]
        if not isinstance(trained, nn.Sequential) or len(trained) != 2 or trained[0] is not self.msd \
                or type(trained[1]) is not nn.LogSoftmax or trained[1].dim != 1:
            return None
        return "nll", None
