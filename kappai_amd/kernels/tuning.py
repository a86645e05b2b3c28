"""The numbers by which the parts and the kernels' faces choose between forms of a kernel.

They were measured on LFM2-sized layers (widths of 1024 to 4096) on one MI355X and decide speed
only: every form gives the same result for the shapes it takes.  They live here, not in the
parts, so that a part holds no size of any particular model; the C side of a step gets the same
numbers in its model description.
"""

# A projection whose consumer can add partial sums asks for them only above this many rows:
# 6144 x 2048 plus the conv step takes 13.0 us unsplit and 13.3 us in two K ranges at 8 rows, 18 us
# and 12 us at 64 rows.
PARTIAL_SUMS_MIN_ROWS = 16
# ... and in steps of up to this many rows whatever their segments (short prompt portions): with
# few rows the products of in_proj and qkv have too few blocks to fill the chip unless K is cut
# (in_proj of 128 rows of the 1.2B shape: 9-12 us in four ranges against 22 us whole).  Above it only steps of
# single rows (decode at large batches) hand on partial sums.  us a prompt step, whole / in sums, 1.2B shape (width
# 2,048): 64 rows 1,043 / 1,014, 128 rows 1,295 / 1,247, 256 rows 1,466 / 1,422, 320 rows 1,540 / 1,563, 417 rows of
# three prompts 1,646 / 1,628; but 24 rows 848 / 890.  At the 350M shape (width 1,024) sums are behind, 64 rows
# 706 / 756, 128 rows 838 / 881, 256 rows 916 / 926: their convolution is two kernels, 13.9 us a layer, that of whole
# products one of 4.3.
PARTIAL_SUMS_MAX_ROWS = 256


def takes_partial_sums(rows: int, single_rows: bool) -> bool:
    """Whether in_proj / qkv of a step of ``rows`` rows hand their consumer partial sums."""
    return rows > PARTIAL_SUMS_MIN_ROWS and (rows <= PARTIAL_SUMS_MAX_ROWS or single_rows)

# Every bfloat16 matrix whose shape allows it (rows a multiple of 16, columns of 32) is kept in
# the order in which the product kernels load it (``ops.fragment_order``), and only so: decode
# steps stream it 10-20 % faster than rows (a step at batch 8: about a tenth), the block kernels
# of prompt steps are faster over it, and the matrices' memory is needed once.  False keeps the
# matrices as the checkpoint has them.
FRAGMENT_ORDER = True

# The norm kernel hands its rows on in fragment order from this many rows on (up to 16): a step of
# the 1.2B shape takes 1.06 against 1.08 ms at 16 rows, 0.994 against 1.000 at 12, even at 8; with
# fewer rows the ordinary order is as fast or faster.
FRAGMENT_ROWS = True
FRAGMENT_ROWS_MIN = 8

# The conv layer's fused decode kernel (in_proj, gates, FIR, state shift in one) gives one block 16
# channels (8 below a width of 4096, where 16 would leave CUs without a block), one block a CU.  It beats
# the separate product (which may split K) with the small step kernel behind it while all its blocks run
# at once: up to a width of FUSED_STEP_NARROW_WIDTH with up to FUSED_STEP_NARROW_ROWS rows, and from
# FUSED_STEP_MIN_WIDTH on.  us fused / separate, W in fragment order from memory: width 128, 1 row 3.0 / 3.9;
# 1024, 1 row 4.3 / 5.4, 16 rows 6.1 / 6.4, 24 rows 6.6 / 7.6, 48 rows 8.1 / 10.0; 2048, 8 rows 8.8 / 10.2, 48 rows
# 12.1 / 13.5, 64 rows 14.6 / 14.0; 2560, 1 row 13.0 / 11.7; 3072, 8 rows 18.5 / 16.8; 4096, 1 row 21.0 / 22.1, 64 rows
# 28.3 / 31.1.  Over W as rows: from FUSED_STEP_NARROW_WIDTH on with up to 16 rows.
FUSED_STEP_MIN_WIDTH = 4096
FUSED_STEP_NARROW_WIDTH = 2048
FUSED_STEP_NARROW_ROWS = 48
FUSED_STEP_ROWS_OVER_ROWS = 16


def fused_conv_step(width: int, rows: int, in_fragments: bool) -> bool:
    """Whether a conv layer's decode step of ``rows`` rows runs as one kernel."""
    if width >= FUSED_STEP_MIN_WIDTH:
        return True
    if in_fragments:
        return width <= FUSED_STEP_NARROW_WIDTH and rows <= FUSED_STEP_NARROW_ROWS
    return width >= FUSED_STEP_NARROW_WIDTH and rows <= FUSED_STEP_ROWS_OVER_ROWS

# A decode step's attention kernel normalises and rotates q and the row's own key itself and
# stores key and value (head sizes 64 and 128, rotate-half over the whole head, a projection that
# comes as bfloat16 rows, more than 512 keys or head size 64) for steps of up to FUSED_QK_MAX_ROWS rows and
# no more than the kernel itself says (``ops.decode_qk_rows``: 16 at head size 64, 4 at 128): every wave of the
# kernel does that work again, beside its first keys' way.  A layer's kernels, 5 to 16 rows of 60 to 12,000 keys, of
# one length and of mixed ones, 8 to 64 heads of 64 on 1 to 32 kv heads: 0 to 7 us less in place of 6 to 100, a
# tenth on average (``ops.QK_BLOCKS`` and ``ops.QK_LONG_BLOCKS`` are the exceptions).  0 switches it off.
FUSED_QK = True
FUSED_QK_MAX_ROWS = 16

# In a step that holds prompt portions, a single decoded token is one tile for the tiled attention
# kernel, and the block that gets it walks all its keys alone: 0.9 ms at 32 k keys, however short
# the portions beside it are.  From this many keys on such rows go to the decode kernel (keys
# split over blocks) instead: a second kernel and its merge against that walk.  16 requests with 32 k-token
# prompts: prompt steps 19 -> 14 ms.  Tiled kernel alone / with the decode kernel behind it, us a layer beside a
# portion of 512, 16 heads of 64 on 8 kv heads: 63 rows of up to 2300 keys 44 / 48, of 4000 68 / 69, of 6000 93 / 94; 8
# rows of up to 3000 keys 20 / 21, of 4000 26 / 24, of 6000 37 / 29; 32 heads on 8, 63 rows of up to 4000 keys 64 / 76, 8
# rows of up to 2300 27 / 23, of 4000 45 / 27.
LONE_ROWS_FROM = 4096

# The minGRU recurrence over a segment: one thread a channel walks the rows in order, which is the
# whole of a decode step and fine for short portions; a segment of more than SCAN_CHUNKS_FROM_ROWS
# rows is cut into chunks of SCAN_CHUNK_ROWS rows that are scanned side by side in three passes
# (chunk sums, carry over the chunks, outputs).
SCAN_CHUNK_ROWS = 32
SCAN_CHUNKS_FROM_ROWS = 64

# The state-space recurrence: segments of up to this many rows are walked token by token, longer
# ones (in bfloat16) worked in chunks on the matrix cores.
STATE_SPACE_CHUNKS_FROM_ROWS = 16

# The gated sum and the delta rule (a matrix of state a head, a decay per key channel) walk the tokens
# at 0.26 to 0.45 us each, however many segments walk side by side; in chunks of 16 rows a token takes
# 0.03 to 0.08 us, but a segment of any length costs at least one chunk, 0.1 to 0.8 us of the whole
# chip.  Hence chunks from a longest segment of 24 rows and 2 more a segment on.  Walk / chunks in us
# with 16 heads of 64 x 64, delta rule: one segment of 24 rows 16.1 / 16.1, of 64 29.2 / 17.5, of 2,048
# 743 / 121; 8 segments of 32 22.2 / 22.0, of 48 29.1 / 24.8; 64 of 32 75 / 85; 60 single rows beside
# one of 128 51 / 44.  Of 128 x 128: 60 single rows beside one of 128 68.5 / 74.8, of 160 80.3 / 75.2.
# The gated sum gains more at every one of these.  bfloat16 only: in float32 the tokens are walked.
MATRIX_STATE_CHUNKS_FROM_ROWS = 24
MATRIX_STATE_CHUNKS_FROM_ROWS_A_SEGMENT = 2
