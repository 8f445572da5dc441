"""One attention row in 64 bits, with what the kernels' roundings may move it by."""
import torch


class Row:
    """q [16, 256] over all rows of k, v [S, 2, 256]: ``ref`` and ``tol`` [4096], and
    ``without(keys)``, the row with those keys left out.

    The kernels keep scores, sums and O in fp32 and round only P to bf16, by at most
    2^-8 of each p.  So the row is off by at most 2^-8 sum p |v|, and, as the
    roundings of different keys are independent with a root mean square of at most
    2^-8 / sqrt(3), by 4 x 2^-8 sqrt(sum p^2 v^2) at seven standard deviations.
    5e-5 covers the fp32 scores and sums."""

    def __init__(self, q, k, v):
        self.s = k.shape[0]
        qg, kg = q.double().view(2, 8, 256), k.double().transpose(0, 1)
        self.v = v.double().transpose(0, 1)
        self.p = torch.softmax(qg @ kg.transpose(1, 2) / 16, -1)
        self.ref = (self.p @ self.v).reshape(4096)
        spread = (self.p ** 2 @ self.v ** 2).sqrt()
        most = self.p @ self.v.abs()
        self.tol = (torch.minimum(4 * spread, most) * 2.0 ** -8 + 5e-5).reshape(4096)

    def without(self, keys):
        p = self.p.clone()
        p[:, :, keys] = 0
        return (p / p.sum(-1, keepdim=True) @ self.v).reshape(4096)

    def sees(self, keys):
        """Whether a kernel that left these keys out would be told from a right one."""
        return bool(((self.without(keys) - self.ref).abs() > 2 * self.tol).any())
