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
extern "C" const fk_kernel *fk_registry_part8(int *n);
extern "C" const fk_kernel *fk_registry_part9(int *n);
extern "C" const fk_kernel *fk_registry_part10(int *n);
extern "C" const fk_kernel *fk_registry_part11(int *n);
extern "C" const fk_kernel *fk_registry_part12(int *n);
extern "C" const fk_kernel *fk_registry_part13(int *n);
extern "C" const fk_kernel *fk_registry_part14(int *n);
extern "C" const fk_kernel *fk_registry_part15(int *n);
extern "C" const fk_kernel *fk_registry_part16(int *n);
extern "C" const fk_kernel *fk_registry_part17(int *n);
extern "C" const fk_kernel *fk_registry_part18(int *n);
extern "C" const fk_kernel *fk_registry_part19(int *n);
extern "C" const fk_kernel *fk_registry_part20(int *n);
extern "C" const fk_kernel *fk_registry_part21(int *n);
extern "C" const fk_kernel *fk_registry_part22(int *n);
extern "C" const fk_kernel *fk_registry_part23(int *n);
extern "C" const fk_kernel *fk_registry_part24(int *n);
extern "C" const fk_kernel *fk_registry_part25(int *n);
extern "C" const fk_kernel *fk_registry_part26(int *n);
extern "C" const fk_kernel *fk_registry_part27(int *n);
extern "C" const fk_kernel *fk_registry_part28(int *n);
extern "C" const fk_kernel *fk_registry_part29(int *n);
extern "C" const fk_kernel *fk_registry_part30(int *n);
extern "C" const fk_kernel *fk_registry_part31(int *n);

extern "C" const fk_kernel *fk_registry(int *count)
{
    static fk_kernel *all = 0;
    static int total = 0;
    if (!all) {
        int n, off = 0;
        const fk_kernel *t;
        fk_kernel *buf = (fk_kernel *)malloc(sizeof(fk_kernel) * 2615);
        t = fk_registry_part0(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part1(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part2(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part3(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part4(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part5(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part6(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part7(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part8(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part9(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part10(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part11(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part12(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part13(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part14(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part15(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part16(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part17(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part18(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part19(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part20(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part21(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part22(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part23(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part24(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part25(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part26(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part27(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part28(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part29(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part30(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        t = fk_registry_part31(&n); memcpy(buf + off, t, sizeof(fk_kernel) * n); off += n;
        total = off;
        all = buf;
    }
    *count = total;
    return all;
}
