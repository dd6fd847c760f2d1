"""Measured tile / split-K choices for convolution shapes of the benchmark networks
(ResNet-152, DenseNet-201, Inception-v3, MobileNetV2).

Key: (M = Cout, N = Ho*Wo, K = Cin*kh*kw, 1 if the filter is 1x1 else 0) -> (tile, split_k, microseconds).
Each entry is the fastest of every compiled tile x split-K factor for that shape, timed on an
MI355X as device durations (kernel trace) of the convolution plus its split-K reduce, inside one
long model whose weights are never reused, i.e. with cold caches as in a batch-1 inference;
the figure of a candidate is the median of three such sweeps (each itself a median over runs).
A negative split_k means: that split, folded inside the convolution launch (direct family), no
reduce launch; the sweeps are plain launches, so a split of two is folded through the pair slots
(one atomic exchange per element), the way a real-time model runs it.
Tiles named g<G>[m2] are the row form of the 3x3 / stride 1 / padding 1 convolution.
Shapes that are not listed fall back to the cost model in tiling.py.
Three entries of DenseNet-201 at 56x56 -- (32, 3136, 1152, 0) and (128, 3136, 160 / 224, 1) --
deliberately keep a tile that is 0.5-1.2 us slower when the network runs alone: with the faster
ones (row form g2 split in two, 16x32k4) four best-effort clients together were 1.5 % slower and
a preemption took 5-8 us longer at the 99th percentile.
(128, 3136, 64 / 96, 1) name 32x32d4 although 16x64k4 is 1 us faster as a kernel: in DenseNet-201
these layers read their input through a BN + ReLU, which the 32x32d4 and 16x32k4 tiles apply as
they load (reef_conv2d_p1_*) and 16x64k4 cannot -- a launch less each, 1145 -> 1131 us per pass.
"""
TUNED = {
    (16, 12544, 32, 1): ("16x64k4", 1, 4.7),
    (24, 3136, 96, 1): ("16x32k4", 1, 3.8),
    (24, 3136, 144, 1): ("16x16k4", 1, 3.5),
    (32, 49, 1152, 0): ("g1", -2, 6.0),
    (32, 196, 1152, 0): ("g1", -2, 5.4),
    (32, 784, 144, 1): ("16x16k4", 1, 3.8),
    (32, 784, 192, 1): ("16x16k4", 1, 3.9),
    (32, 784, 1152, 0): ("16x16k4", -2, 5.6),
    (32, 3136, 1152, 0): ("16x32k4", 1, 7.9),
    (32, 12544, 27, 0): ("32x32d4", 1, 7.0),
    (32, 21609, 288, 0): ("32x32d4", 1, 11.2),
    (32, 22201, 27, 0): ("32x32d4", 1, 8.8),
    (64, 196, 192, 1): ("16x16k4", 1, 4.3),
    (64, 196, 384, 1): ("16x16k4", 1, 4.9),
    (64, 1225, 288, 1): ("16x32k4", 1, 5.4),
    (64, 1225, 1200, 0): ("16x16k4", 1, 9.4),
    (64, 3136, 256, 1): ("16x32k4", 1, 5.3),
    (64, 3136, 576, 0): ("g2", 1, 9.8),
    (64, 12544, 147, 0): ("64x32k2", 1, 16.3),
    (64, 21609, 288, 0): ("32x32d4", 1, 18.2),
    (80, 5329, 64, 1): ("16x64k4", 1, 6.3),
    (96, 196, 384, 1): ("16x16k4", 1, 4.8),
    (96, 196, 576, 1): ("16x16k4", 1, 5.3),
    (96, 289, 864, 0): ("16x16k4", -2, 6.2),
    (96, 1225, 576, 0): ("16x32k4", 1, 6.4),
    (96, 1225, 864, 0): ("16x16k4", 1, 6.4),
    (96, 12544, 16, 1): ("32x64k2", 1, 7.7),
    (128, 49, 896, 1): ("16x16k4", -2, 5.6),
    (128, 49, 928, 1): ("16x16k4", -2, 6.2),
    (128, 49, 960, 1): ("16x16k4", -2, 6.0),
    (128, 49, 992, 1): ("16x16k4", -2, 6.0),
    (128, 49, 1024, 1): ("16x16k4", -2, 6.2),
    (128, 49, 1056, 1): ("16x16k4", -2, 6.3),
    (128, 49, 1088, 1): ("16x16k4", -2, 6.4),
    (128, 49, 1120, 1): ("16x16k4", -2, 6.3),
    (128, 49, 1152, 1): ("16x16k4", -2, 6.3),
    (128, 49, 1184, 1): ("16x16k4", -2, 6.1),
    (128, 49, 1216, 1): ("16x16k4", -2, 6.4),
    (128, 49, 1248, 1): ("16x16k4", -2, 6.4),
    (128, 49, 1280, 1): ("16x16k4", -2, 6.4),
    (128, 49, 1312, 1): ("16x16k4", -4, 6.4),
    (128, 49, 1344, 1): ("16x16k4", -4, 6.4),
    (128, 49, 1376, 1): ("16x16k4", -4, 6.4),
    (128, 49, 1408, 1): ("16x16k4", -4, 6.4),
    (128, 49, 1440, 1): ("16x16k4", -4, 6.3),
    (128, 49, 1472, 1): ("16x16k4", -4, 6.4),
    (128, 49, 1504, 1): ("16x16k4", -4, 6.5),
    (128, 49, 1536, 1): ("16x16k4", -4, 6.5),
    (128, 49, 1568, 1): ("16x16k4", -4, 6.8),
    (128, 49, 1600, 1): ("16x16k4", -4, 6.7),
    (128, 49, 1632, 1): ("16x16k4", -4, 6.8),
    (128, 49, 1664, 1): ("16x16k4", -4, 6.9),
    (128, 49, 1696, 1): ("16x16k4", -4, 6.8),
    (128, 49, 1728, 1): ("16x16k4", -4, 6.8),
    (128, 49, 1760, 1): ("16x16k4", -4, 6.7),
    (128, 49, 1792, 1): ("16x16k4", -4, 6.9),
    (128, 49, 1824, 1): ("16x16k4", -4, 6.8),
    (128, 49, 1856, 1): ("16x16k4", -4, 6.8),
    (128, 49, 1888, 1): ("16x16k4", -4, 6.8),
    (128, 196, 256, 1): ("16x16k4", 1, 4.8),
    (128, 196, 288, 1): ("16x16k4", 1, 5.0),
    (128, 196, 320, 1): ("16x16k4", 1, 4.6),
    (128, 196, 352, 1): ("16x16k4", 1, 4.8),
    (128, 196, 384, 1): ("16x16k4", 1, 5.0),
    (128, 196, 416, 1): ("16x16k4", 1, 5.0),
    (128, 196, 448, 1): ("16x16k4", 1, 5.0),
    (128, 196, 480, 1): ("16x16k4", 1, 5.2),
    (128, 196, 512, 1): ("16x16k4", 1, 5.4),
    (128, 196, 544, 1): ("16x16k4", 1, 5.3),
    (128, 196, 576, 1): ("16x16k4", 1, 5.2),
    (128, 196, 608, 1): ("16x16k4", 1, 5.4),
    (128, 196, 640, 1): ("16x16k4", -2, 5.4),
    (128, 196, 672, 1): ("16x16k4", -2, 5.6),
    (128, 196, 704, 1): ("16x16k4", -2, 5.6),
    (128, 196, 736, 1): ("16x16k4", -2, 5.7),
    (128, 196, 768, 1): ("16x16k4", -2, 5.8),
    (128, 196, 800, 1): ("16x16k4", -2, 5.8),
    (128, 196, 832, 1): ("16x16k4", -2, 5.8),
    (128, 196, 864, 1): ("16x16k4", -2, 5.8),
    (128, 196, 896, 1): ("16x16k4", -2, 5.8),
    (128, 196, 928, 1): ("16x16k4", -2, 5.9),
    (128, 196, 960, 1): ("16x16k4", -2, 6.0),
    (128, 196, 992, 1): ("16x16k4", -2, 6.0),
    (128, 196, 1024, 1): ("16x16k4", -2, 6.0),
    (128, 196, 1056, 1): ("16x16k4", -2, 6.1),
    (128, 196, 1088, 1): ("16x16k4", -2, 6.0),
    (128, 196, 1120, 1): ("16x16k4", -2, 6.0),
    (128, 196, 1152, 1): ("16x16k4", -2, 6.1),
    (128, 196, 1184, 1): ("16x16k4", -2, 6.1),
    (128, 196, 1216, 1): ("16x16k4", -2, 6.2),
    (128, 196, 1248, 1): ("16x16k4", -2, 6.2),
    (128, 196, 1280, 1): ("16x16k4", -2, 6.1),
    (128, 196, 1312, 1): ("16x16k4", -2, 7.2),
    (128, 196, 1344, 1): ("16x16k4", -2, 7.3),
    (128, 196, 1376, 1): ("16x16k4", -2, 7.1),
    (128, 196, 1408, 1): ("16x16k4", -2, 7.4),
    (128, 196, 1440, 1): ("16x16k4", -2, 7.5),
    (128, 196, 1472, 1): ("16x16k4", -2, 7.4),
    (128, 196, 1504, 1): ("16x16k4", -2, 7.5),
    (128, 196, 1536, 1): ("16x16k4", -2, 7.4),
    (128, 196, 1568, 1): ("16x16k4", -2, 7.4),
    (128, 196, 1600, 1): ("16x16k4", -2, 7.5),
    (128, 196, 1632, 1): ("16x16k4", -2, 7.4),
    (128, 196, 1664, 1): ("16x16k4", -2, 7.6),
    (128, 196, 1696, 1): ("16x16k4", -2, 7.6),
    (128, 196, 1728, 1): ("16x16k4", -2, 7.6),
    (128, 196, 1760, 1): ("16x16k4", -2, 7.6),
    (128, 289, 896, 0): ("16x16k4", 1, 5.3),
    (128, 784, 128, 1): ("16x32k4", 1, 4.4),
    (128, 784, 160, 1): ("16x32k4", 1, 4.7),
    (128, 784, 192, 1): ("16x32k4", 1, 4.7),
    (128, 784, 224, 1): ("16x32k4", 1, 4.8),
    (128, 784, 256, 1): ("16x32k4", 1, 4.6),
    (128, 784, 288, 1): ("16x32k4", 1, 5.2),
    (128, 784, 320, 1): ("16x32k4", 1, 5.2),
    (128, 784, 352, 1): ("16x32k4", 1, 5.0),
    (128, 784, 384, 1): ("16x32k4", 1, 5.2),
    (128, 784, 416, 1): ("16x32k4", 1, 5.0),
    (128, 784, 448, 1): ("16x32k4", 1, 5.4),
    (128, 784, 480, 1): ("16x32k4", 1, 5.5),
    (128, 784, 512, 1): ("16x32k4", 1, 5.4),
    (128, 784, 1152, 0): ("g2", 1, 9.6),
    (128, 3136, 64, 1): ("32x32d4", 1, 6.8),
    (128, 3136, 96, 1): ("32x32d4", 1, 7.0),
    (128, 3136, 128, 1): ("16x32k4", 1, 6.2),
    (128, 3136, 160, 1): ("32x32d4", 1, 7.4),
    (128, 3136, 192, 1): ("16x32k4", 1, 7.7),
    (128, 3136, 224, 1): ("32x32d4", 1, 7.8),
    (128, 3136, 256, 1): ("32x32d4", 1, 7.9),
    (144, 3136, 24, 1): ("32x32k4", 1, 5.7),
    (160, 49, 576, 1): ("16x16k4", 1, 5.6),
    (160, 49, 960, 1): ("16x16k4", -2, 6.1),
    (160, 289, 1120, 0): ("16x16k4", 1, 5.8),
    (192, 64, 1728, 0): ("16x16k4", -3, 6.9),
    (192, 289, 896, 0): ("16x16k4", 1, 5.4),
    (192, 289, 1120, 0): ("16x16k4", 1, 6.8),
    (192, 289, 1344, 0): ("16x16k4", 1, 6.1),
    (192, 784, 32, 1): ("16x64k4", 1, 4.6),
    (192, 5041, 720, 0): ("32x32d4", 1, 21.5),
    (208, 1225, 192, 1): ("16x32k4", 1, 6.3),
    (240, 1225, 256, 1): ("16x32k4", 1, 7.4),
    (240, 1225, 288, 1): ("16x32k4", 1, 9.2),
    (256, 196, 1024, 1): ("16x32k4", -2, 6.8),
    (256, 196, 2304, 0): ("g2", -2, 9.1),
    (256, 784, 512, 1): ("16x32k4", 1, 7.8),
    (256, 3136, 64, 1): ("16x32k4", 1, 5.4),
    (320, 49, 960, 1): ("16x16k4", -2, 6.2),
    (320, 64, 1728, 0): ("16x16k4", -3, 7.0),
    (320, 3136, 64, 1): ("64x32k2", 1, 7.1),
    (384, 64, 1152, 0): ("16x16k4", -2, 5.6),
    (384, 64, 4032, 0): ("16x16k4", -2, 9.1),
    (384, 196, 64, 1): ("16x32k4", 1, 3.8),
    (384, 289, 768, 1): ("16x32k4", 1, 7.5),
    (384, 289, 2592, 0): ("32x32d4", -2, 13.7),
    (512, 49, 2048, 1): ("16x16k4", -2, 7.9),
    (512, 49, 4608, 0): ("16x16k4", -2, 10.4),
    (512, 784, 128, 1): ("16x32k4", 1, 5.4),
    (576, 196, 96, 1): ("16x32k4", 1, 4.1),
    (640, 289, 768, 1): ("16x32k4", 1, 10.6),
    (640, 784, 256, 1): ("32x32d4", 1, 10.2),
    (704, 289, 768, 1): ("16x64k4", 1, 10.9),
    (768, 289, 768, 1): ("16x64k4", 1, 10.8),
    (896, 196, 1792, 1): ("32x32d4", 1, 16.8),
    (960, 49, 160, 1): ("16x32k4", 1, 4.6),
    (1024, 196, 256, 1): ("16x32k4", 1, 5.8),
    (1280, 49, 320, 1): ("16x32k4", 1, 5.9),
    (1280, 196, 512, 1): ("32x32d4", 1, 14.0),
    (1344, 64, 1280, 1): ("16x32k4", 1, 8.9),
    (1344, 64, 2048, 1): ("16x32k4", 1, 11.5),
    (2048, 49, 512, 1): ("16x32k4", 1, 6.2),
    (2560, 49, 1024, 1): ("32x32d4", 1, 15.0),
    (256, 196, 512, 1): ("16x16k4", 1, 5.3),
    (896, 49, 1792, 1): ("16x32k4", -2, 8.4),
}

# Entries that replace TUNED's when a network is generated to run as a best-effort model beside
# others (GraphBuilder(under_load=True); the DenseNet-201 of the benchmark configurations is one).
# TUNED holds what is fastest for a model that has the device to itself.  With four clients of the
# same network on four streams a finer split of K is better for these shapes: measured as
# inferences per second of four DenseNet-201 clients alone (three runs of two seconds each per
# candidate, same process) 1722 -> 1774 with these entries together, each group worth 1.2-1.9 % on
# its own; splitting twice as fine again, or less than TUNED does, loses 2-10 %.  In the headline
# pair (real-time ResNet-152 beside the four clients) 1612-1617 -> 1667-1685 inferences per second,
# preemption and real-time latency unchanged.  Alone, the network is about 3 % slower with them.
# Two 128-wide 1x1 layers on the 56x56 image are the other way round: 32x32d4 (392 workgroups)
# instead of 16x32k4 (784) -- 1768-1780 -> 1780-1799 inferences per second in two sweeps (the same
# sweeps gave 1799-1818 for the two neighbouring layers, whose change to 32x32d4 also pays for a
# model alone and is in TUNED).
# Key as in TUNED -> (tile, split_k).
TUNED_UNDER_LOAD = {
    (128, 3136, 128, 1): ("32x32d4", 1),
    (128, 3136, 192, 1): ("32x32d4", 1),
    (32, 49, 1152, 0): ("g1", -4),
    (32, 196, 1152, 0): ("g1", -4),
    (128, 49, 896, 1): ("16x16k4", -4),
    (128, 49, 928, 1): ("16x16k4", -4),
    (128, 49, 960, 1): ("16x16k4", -4),
    (128, 49, 992, 1): ("16x16k4", -4),
    (128, 49, 1024, 1): ("16x16k4", -4),
    (128, 49, 1056, 1): ("16x16k4", -4),
    (128, 49, 1088, 1): ("16x16k4", -4),
    (128, 49, 1120, 1): ("16x16k4", -4),
    (128, 49, 1152, 1): ("16x16k4", -4),
    (128, 49, 1184, 1): ("16x16k4", -4),
    (128, 49, 1216, 1): ("16x16k4", -4),
    (128, 49, 1248, 1): ("16x16k4", -4),
    (128, 49, 1280, 1): ("16x16k4", -4),
    (128, 49, 1312, 1): ("16x16k4", -8),
    (128, 49, 1344, 1): ("16x16k4", -8),
    (128, 49, 1376, 1): ("16x16k4", -8),
    (128, 49, 1408, 1): ("16x16k4", -8),
    (128, 49, 1440, 1): ("16x16k4", -8),
    (128, 49, 1472, 1): ("16x16k4", -8),
    (128, 49, 1504, 1): ("16x16k4", -8),
    (128, 49, 1536, 1): ("16x16k4", -8),
    (128, 49, 1568, 1): ("16x16k4", -8),
    (128, 49, 1600, 1): ("16x16k4", -8),
    (128, 49, 1632, 1): ("16x16k4", -8),
    (128, 49, 1664, 1): ("16x16k4", -8),
    (128, 49, 1696, 1): ("16x16k4", -8),
    (128, 49, 1728, 1): ("16x16k4", -8),
    (128, 49, 1760, 1): ("16x16k4", -8),
    (128, 49, 1792, 1): ("16x16k4", -8),
    (128, 49, 1824, 1): ("16x16k4", -8),
    (128, 49, 1856, 1): ("16x16k4", -8),
    (128, 49, 1888, 1): ("16x16k4", -8),
}

# The same for the K-contiguous matrix products (tiling.choose_gemm(under_load=True)):
# (M, N, K) -> (direct tile, split of K folded inside the launch).  BERT-base's FFN-down product in four,
# which is the choice for a model alone as well.  Two clients of the network on two streams, inferences
# per second of both (five runs of 1.2 s per candidate in turn, same process): in four 1695-1722, in three
# 1641-1673, with the output projection (768 x 768) in two beside it 1686-1714, in three 1602-1613.
# Beside a real-time Inception-v3 (900 requests, two runs each): in four 1662-1666 inferences per second
# and 0.587 / 0.975-0.977 ms real-time p50 / p99, in three 1606-1607 and 0.587-0.590 / 0.987-1.033 -- the
# 64 workgroups fewer buy the real-time model nothing.
# On packed weights these are taken for a model alone too: a graph for one use and for the other is the same then, as
# the checks of nets.bert ask.  They cost: the cost table would run the product unsplit on 16x16k4, a pass of twelve layers
# 594 us instead of 634 alone, of six layers as a best-effort model 308 instead of 329; two clients 2380
# inferences per second instead of 2308.
GEMM_UNDER_LOAD = {
    (128, 768, 3072): ("32x48d4", 4),
}
