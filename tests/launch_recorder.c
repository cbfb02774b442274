/* The HIP runtime calls by which libach.so launches a kernel, recorded
 * instead of run: loaded globally before the library, these definitions are
 * the ones it resolves, so its launch decisions can be tested without a GPU. */
#include <stddef.h>

typedef struct { unsigned x, y, z; } dim3_t;
typedef struct {
    const void *kernel;
    unsigned grid[3], block[3];
    size_t lds;
    int lds_limit; /* of the kernel when it was launched; 0: never set */
} launch_t;

enum { MAX = 4096 };
static launch_t launches[MAX];
static int nlaunch;
static const void *limit_of[MAX];
static int limit[MAX], nlimit;
static dim3_t cfg_grid, cfg_block;
static size_t cfg_lds;

int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void *stream)
{
    (void)stream;
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    return 0;
}

int __hipPopCallConfiguration(dim3_t *grid, dim3_t *block, size_t *lds, void **stream)
{
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *stream = NULL;
    return 0;
}

int hipFuncSetAttribute(const void *f, int attr, int value)
{
    (void)attr; /* the library sets the dynamic LDS limit only */
    if (nlimit < MAX) {
        limit_of[nlimit] = f;
        limit[nlimit++] = value;
    }
    return 0;
}

int hipLaunchKernel(const void *f, dim3_t grid, dim3_t block, void **args, size_t lds, void *stream)
{
    (void)args;
    (void)stream;
    if (nlaunch < MAX) {
        launch_t *l = &launches[nlaunch++];
        l->kernel = f;
        l->grid[0] = grid.x, l->grid[1] = grid.y, l->grid[2] = grid.z;
        l->block[0] = block.x, l->block[1] = block.y, l->block[2] = block.z;
        l->lds = lds;
        l->lds_limit = 0;
        for (int i = 0; i < nlimit; ++i)
            if (limit_of[i] == f) l->lds_limit = limit[i];
    }
    return 0;
}

int hipGetLastError(void) { return 0; }

int rec_count(void) { return nlaunch; }
const launch_t *rec_launch(int i) { return &launches[i]; }
void rec_reset(void) { nlaunch = 0; }
