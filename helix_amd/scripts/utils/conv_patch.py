"""Host model of the convolutions whose input stays in LDS (src_template/common/helix_conv_patch.h), shared by both backends:
what a configuration reserves and launches for a layer (the arithmetic of make_plan there), and the prediction that ranks the
configurations.  They have no profile: the model's first PATCH_TOP are timed with the profiled candidates of a layer, once."""
from utils.roofline import NUM_CU

LDS_BYTES = 160 * 1024
K_TILE_BYTES = 128
PATCH_TOP = 4
LARGE_WAVE_TILES = 8       # 16 x 16 tiles of a wave beyond which its registers leave a compute unit 8 waves instead of 16
LARGEST_WAVE_TILES_F32 = 10    # and in FP32, with two sets of accumulators, 4


class PatchFamily:
    """One backend's family.  A point is (BLOCK_ROWS, BLOCK_COLS, WAVE_ROWS, WAVE_COLS, K_GROUPS).

    The constants are clocks at 2.4 GHz (bytes per clock and compute unit for the rates), fitted to the times of all points on
    50 layers each: FP16 318 pairs, 8 % rms; FP32 420 pairs, 14 % rms.  What decides is the order: the fastest of the first
    four by the model is 0.24 % (FP16, 29 layers, 3.8 % at worst) and 0.3 % (FP32, 34 layers, 2.7 %) behind the fastest point, the
    first alone 4.6 and 2 %."""

    def __init__(self, element_bytes, whole_chunks, points, fixed, stage_rate, multiply, lds_rate, weight_rate, tile, add):
        self.element_bytes, self.whole_chunks, self.points = element_bytes, whole_chunks, points
        self.fixed = fixed                 # launch, first loads, last stores
        self.stage_rate = stage_rate       # input into LDS
        self.multiply = multiply           # the products of one 16 x 16 tile in a K tile
        self.lds_rate, self.weight_rate = lds_rate, weight_rate
        self.tile = tile                   # of a K tile at least, whatever is in it
        self.add = add                     # adding one part of K of one 16 x 16 tile; about the same to store a tile

    def layout(self, point, batch, IC, H, W, OC, kH, kW, stride, pad):
        """(bytes of LDS, of which staged input, workgroups) of a layer, None where the point cannot run it."""
        rows, cols, wave_rows, wave_cols, groups = point
        per_chunk = 16 // self.element_bytes
        OH, OW = (H + 2 * pad - kH) // stride + 1, (W + 2 * pad - kW) // stride + 1
        pixel, M = IC * self.element_bytes, batch * OH * OW
        filter_bytes = kH * kW * pixel
        if (OH < 1 or OW < 1 or (self.whole_chunks and IC % per_chunk) or filter_bytes > 0x1000000
                or batch * H * W * pixel >= 0x40000000 or OC * filter_bytes >= 0x40000000):
            return None
        image_rows, row_pixels = (OH - 1) * stride + kH, (OW - 1) * stride + kW
        blocks = -(-M // rows) * -(-OC // cols)
        if (M > 0x7fffff or W * pixel > 0x7fffff or batch * H > 0x7fffff or batch * image_rows > 0x7fffff or blocks > 0x3fffffff
                or row_pixels - pad < 1):
            return None
        pixels = min(rows, M)
        if pixels % OW == 0:
            n = pixels // OW
            crossings = n // OH - 1 if n % OH == 0 else 0 if OH % n == 0 else (n - 2) // OH + 1
        else:
            n = (pixels - 2) // OW + 2
            crossings = (n - 2) // OH + 1
        staged_rows = (n - 1) * stride + kH + crossings * max(kH - stride, 0)
        group = -(-IC // per_chunk)
        pixel_bytes = 16 * (group + (6 - group % 4) % 4 if stride % 2 else group | 1)
        waves = rows // wave_rows * (cols // wave_cols) * groups
        patch = staged_rows * row_pixels * pixel_bytes
        offset = 16 + waves * wave_cols * K_TILE_BYTES + 8 * (self.k_tiles(IC, kH, kW) + 1) * 4
        lds = max(offset + patch, waves * wave_rows * wave_cols * 4 if groups > 1 else 0)
        return (lds, patch, blocks) if lds <= LDS_BYTES else None

    def k_tiles(self, IC, kH, kW):
        return -(-kH * kW * -(-IC * self.element_bytes // 16) // (K_TILE_BYTES // 16))

    def seconds(self, point, batch, IC, H, W, OC, kH, kW, stride, pad):
        """Predicted time of a layer; inf where the point cannot run it."""
        layout = self.layout(point, batch, IC, H, W, OC, kH, kW, stride, pad)
        if layout is None:
            return float("inf")
        lds, patch, blocks = layout
        rows, cols, wave_rows, wave_cols, groups = point
        waves = rows // wave_rows * (cols // wave_cols) * groups
        tm, tn = wave_rows // 16, wave_cols // 16
        of_registers = 4 if self.element_bytes == 4 and tm * tn > LARGEST_WAVE_TILES_F32 else 16 if tm * tn <= LARGE_WAVE_TILES else 8
        resident = max(1, min(LDS_BYTES // lds, of_registers // waves))
        part = -(-self.k_tiles(IC, kH, kW) // groups)

        def round_clocks(share):             # workgroups of one round on a compute unit
            walk = max(part * tm * tn * self.multiply * max(1.0, waves * share / 4),
                       share * waves * part * (2 * tm + 4 * tn) * 1024 / self.lds_rate,
                       share * waves * part * tn * 2048 / self.weight_rate, part * self.tile)
            return (patch * share / self.stage_rate + walk + (self.add * groups * tm * tn if groups > 1 else 0)
                    + self.add * share * tm * tn * waves / groups)

        rounds = -(-blocks // (NUM_CU * resident))
        last = blocks - (rounds - 1) * NUM_CU * resident
        return (self.fixed + (rounds - 1) * round_clocks(resident) + round_clocks(min(resident, -(-last // NUM_CU)))) / 2.4e9

    def ranked(self, layer, top=PATCH_TOP):
        """The `top` points with the lowest predicted time that can run the layer, best first."""
        costs = sorted((self.seconds(point, *layer), point) for point in self.points)
        return [point for cost, point in costs[:top] if cost < float("inf")]
