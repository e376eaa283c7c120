// Chip-resident time loop, FDORDER 2, acoustic, VTI, TTI and SH.
#define DN_F 1
#define DN_GROUP 1
#include "dn_resident_inst.inc"
