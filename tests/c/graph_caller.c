/* A caller of the device ABI (aspen_hip.h) that builds its own graph: three matmul layers, one per way the weights are laid out
   for the kernels (64 x 64, 32 x 32 and 128 x 32 tiles), from plain row-major weights.  Runs it with either engine, writes
   other weights into the same buffers, runs it again; every result against sums in double precision. */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "aspen.h"
#include "aspen_hip.h"

#define LAYERS 4
#define COLUMNS 70
static const unsigned int rows[LAYERS] = {96, 100, 72, 130}, stride[LAYERS] = {96, 128, 96, 160};
static const int variant[LAYERS] = {0, ASPEN_HIP_GEMM_SMALL, ASPEN_HIP_GEMM_NARROW, ASPEN_HIP_GEMM_TALL};
static const unsigned int tile_m[LAYERS] = {0, 64, 32, 128}, tile_n[LAYERS] = {0, 64, 32, 32};
static float *weight[LAYERS], *bias[LAYERS], *d_weight[LAYERS], *d_bias[LAYERS], *d_out[LAYERS], *input;

static unsigned int up (unsigned int a, unsigned int to) { return (a + to - 1) / to * to; }
static float noise (void) { return (float)rand () / (float)RAND_MAX - 0.5f; }
#define CHECK(x) do { if (x) { fprintf (stderr, "%s: %s\n", #x, aspen_hip_last_error ()); return 1; } } while (0)

static int new_weights (void)
{
    for (int l = 1; l < LAYERS; l++)
    {
        const unsigned int kp = up (rows[l - 1], 32);
        for (unsigned int m = 0; m < rows[l]; m++)
        {
            for (unsigned int k = 0; k < rows[l - 1]; k++) weight[l][m * kp + k] = noise ();
            bias[l][m] = noise ();
        }
        CHECK (aspen_hip_h2d (d_weight[l], weight[l], (size_t)up (rows[l], 128) * kp * sizeof (float)));
        CHECK (aspen_hip_h2d (d_bias[l], bias[l], rows[l] * sizeof (float)));
    }
    return 0;
}

static int compare (const char *what)
{
    static double x[2][COLUMNS][256];
    for (unsigned int n = 0; n < COLUMNS; n++) for (unsigned int k = 0; k < rows[0]; k++) x[0][n][k] = input[n * stride[0] + k];
    for (int l = 1; l < LAYERS; l++)
    {
        float *got = calloc ((size_t)COLUMNS * stride[l], sizeof (float));
        CHECK (got == NULL || aspen_hip_d2h (got, d_out[l], (size_t)COLUMNS * stride[l] * sizeof (float)));
        double diff = 0, norm = 0;
        for (unsigned int n = 0; n < COLUMNS; n++)
            for (unsigned int m = 0; m < rows[l]; m++)
            {
                double s = bias[l][m];
                for (unsigned int k = 0; k < rows[l - 1]; k++) s += (double)weight[l][m * up (rows[l - 1], 32) + k] * x[(l - 1) & 1][n][k];
                x[l & 1][n][m] = s;
                diff += (s - got[n * stride[l] + m]) * (s - got[n * stride[l] + m]);
                norm += s * s;
            }
        free (got);
        printf ("%s layer %d: relative error %.3g\n", what, l, sqrt (diff / norm));
        if (!(diff <= 1e-10 * norm)) { fprintf (stderr, "%s layer %d: relative error %.3g\n", what, l, sqrt (diff / norm)); return 1; }
        CHECK (aspen_hip_zero (d_out[l], (size_t)COLUMNS * stride[l] * sizeof (float)));
    }
    return 0;
}

int main (void)
{
    aspen_hip_layer_t L[LAYERS];
    uint32_t ninst_layer[64], num_parents[64], child_off[65], child_idx[1024], roots[64], n = 0, edges = 0, num_roots = 0;
    CHECK (aspen_hip_init ());
    memset (L, 0, sizeof (L));
    input = calloc ((size_t)COLUMNS * stride[0], sizeof (float));
    for (unsigned int c = 0; c < COLUMNS; c++) for (unsigned int k = 0; k < rows[0]; k++) input[c * stride[0] + k] = noise ();
    for (int l = 0; l < LAYERS; l++)
    {
        d_out[l] = aspen_hip_alloc ((size_t)COLUMNS * stride[l] * sizeof (float));
        L[l].type = l ? MATMUL_LAYER : INPUT_LAYER;
        L[l].M = rows[l]; L[l].N = COLUMNS; L[l].ld = stride[l]; L[l].out = d_out[l];
        if (l == 0) { CHECK (d_out[0] == NULL || aspen_hip_h2d (d_out[0], input, (size_t)COLUMNS * stride[0] * sizeof (float))); continue; }
        const unsigned int kp = up (rows[l - 1], 32), mp = up (rows[l], 128);
        weight[l] = calloc ((size_t)mp * kp, sizeof (float)); bias[l] = calloc (rows[l], sizeof (float));
        d_weight[l] = aspen_hip_alloc ((size_t)mp * kp * sizeof (float)); d_bias[l] = aspen_hip_alloc (rows[l] * sizeof (float));
        CHECK (!d_out[l] || !d_weight[l] || !d_bias[l] || !weight[l] || !bias[l]);
        L[l].act = NO_ACTIVATION; L[l].variant = variant[l]; L[l].direct = ASPEN_HIP_OPERAND_DIRECT;
        L[l].tile_m = tile_m[l]; L[l].tile_n = tile_n[l];
        L[l].tiles_m = (rows[l] + tile_m[l] - 1) / tile_m[l]; L[l].tiles_n = (COLUMNS + tile_n[l] - 1) / tile_n[l];
        L[l].splits = 1; L[l].num_ninst = L[l].tiles_m * L[l].tiles_n; L[l].ninst_start = n;
        L[l].K = rows[l - 1]; L[l].Kp = kp; L[l].ld0 = stride[l - 1]; L[l].in0 = d_out[l - 1];
        L[l].weight = d_weight[l]; L[l].bias = d_bias[l];
        n += L[l].num_ninst;
    }
    /* every tile waits for all tiles of the layer before */
    for (int l = 1; l < LAYERS; l++)
        for (uint32_t t = L[l].ninst_start; t < L[l].ninst_start + L[l].num_ninst; t++)
        {
            ninst_layer[t] = (uint32_t)l;
            num_parents[t] = l == 1 ? 0 : L[l - 1].num_ninst;
            if (l == 1) roots[num_roots++] = t;
            child_off[t] = edges;
            for (uint32_t c = 0; l + 1 < LAYERS && c < L[l + 1].num_ninst; c++) child_idx[edges++] = L[l + 1].ninst_start + c;
        }
    child_off[n] = edges;
    CHECK (new_weights ());
    aspen_hip_graph_t *g = aspen_hip_graph_create (L, LAYERS, ninst_layer, num_parents, child_off, child_idx, n, roots, num_roots);
    CHECK (g == NULL);
    for (int round = 0; round < 3; round++)
    {
        if (round) CHECK (new_weights ());
        CHECK (aspen_hip_run_dataflow (g, 0, 0) || aspen_hip_graph_sync (g) || compare ("dataflow"));
        if (round) CHECK (new_weights ());
        CHECK (aspen_hip_run_layers (g, 1, LAYERS - 1) || aspen_hip_graph_sync (g) || compare ("layers"));
    }
    aspen_hip_graph_destroy (g);
    printf ("ok\n");
    return 0;
}
