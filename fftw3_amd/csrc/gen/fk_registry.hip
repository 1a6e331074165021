// generated by fftw3_amd/gen_kernels.py -- do not edit
#include <stdlib.h>
#include <string.h>
#include "../fk_args.h"

extern "C" const fk_kernel *fk_registry_part0(int *n);
extern "C" const fk_kernel *fk_registry_part1(int *n);
extern "C" const fk_kernel *fk_registry_part2(int *n);
extern "C" const fk_kernel *fk_registry_part3(int *n);
extern "C" const fk_kernel *fk_registry_part4(int *n);
extern "C" const fk_kernel *fk_registry_part5(int *n);
extern "C" const fk_kernel *fk_registry_part6(int *n);
extern "C" const fk_kernel *fk_registry_part7(int *n);

extern "C" const fk_kernel *fk_registry(int *count)
{
    static fk_kernel *all = 0;
    static int total = 0;
    if (!all) {
        int n, off = 0;
        const fk_kernel *t;
        fk_kernel *buf = (fk_kernel *)malloc(sizeof(fk_kernel) * 2571);
        t = fk_registry_part0(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part1(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part2(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part3(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part4(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part5(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part6(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part7(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        total = off;
        all = buf;
    }
    *count = total;
    return all;
}
