// Chip-resident time loop, FDORDER 8.
#define DN_F 4
#include "dn_resident_inst.inc"
