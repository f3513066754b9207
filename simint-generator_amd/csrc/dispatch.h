// Class dispatch: (la lb | lc ld) -> kernel launcher.  The tables are
// generated (gen/dispatch.cpp): one lane-per-quartet and one wave-per-quartet
// launcher per class where built, and the family in use for each class.
#pragma once
#include <hip/hip_runtime.h>
#include "device_types.h"

typedef hipError_t (*simint_launch_fn)(const EriArgs *, hipStream_t);

typedef hipError_t (*simint_list_launch_fn)(const EriListArgs *, hipStream_t);

simint_launch_fn simint_dispatch(int la, int lb, int lc, int ld);
// staging doubles per lane the selected kernel needs in EriArgs::scratch
// (split lane-per-quartet family), 0 for the others
int simint_dispatch_staging(int la, int lb, int lc, int ld);
// The family of a launch of `items` work items of up to `depth` primitive
// quartets: the selected one or, where the build chose it, the class's family
// for large launches of deep contractions.  Its launcher and staging doubles.
int simint_range_family(int la, int lb, int lc, int ld, long long items, long long depth);
simint_launch_fn simint_family_launch(int family, int la, int lb, int lc, int ld);
int simint_family_staging(int family, int la, int lb, int lc, int ld);
// quartet-list launcher of the class's selected family (or the other family
// when the selected one has no list kernel); null if the class is not built
simint_list_launch_fn simint_dispatch_list(int la, int lb, int lc, int ld);
// the lane-per-quartet list launcher where the build chose the component-lane
// one for the class and a list of n quartets, all of about `depth` primitive
// quartets, is large enough to run faster there; null otherwise
simint_list_launch_fn simint_dispatch_list_even(int la, int lb, int lc, int ld, long long n, long long depth);
// FP32-VRR/HRR prefix kernel of the class (lane-per-quartet family only);
// null where the class has none or runs the wave-per-quartet family
simint_launch_fn simint_dispatch_mixed(int la, int lb, int lc, int ld);
